"""A key that outweighs the rest by far, and later ones above it: once the probabilities of a wave's tiles are small the flash kernel stops
forming row maxima until a sum of probabilities says that one may have grown.  Row maxima, exact here, and outputs against float64; scores and
bound as in test_growing_scores.py."""
import pytest
import torch

from test_growing_scores import LOG2E, _causal, _check, _reference

pytestmark = pytest.mark.gpu


def _inputs(n, d, dtype, risers):
    g = torch.Generator().manual_seed(n + d)
    q, k = torch.zeros(1, 4, n, d, dtype=dtype), torch.zeros(1, 2, n, d, dtype=dtype)
    q[..., 0] = 8.0
    k[..., 0] = torch.randint(-30, -10, (1, 2, n), generator=g).float()
    k[..., 0, 0] = 8.0
    for i, at in enumerate(risers):
        k[:, i % 2:, at, 0] = 8.0 + 4.0 * (i // 2)  # (the first two tie with the sink)
    v = torch.randn(1, 2, n, d, generator=g).to(dtype)
    return q.cuda(), k.cuda(), v.cuda()


# first and last keys of tiles, of their halves and of a lane's runs of four, both tiles of an unrolled pair
RISERS = [200, 260, 448, 511, 543, 544, 580, 639, 640, 775, 899, 900, 1000, 1023]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_keys_above_a_sink(d, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, dense_causal_attention
    from anchor_attn.src.ops.anchor_step_1_2_v2 import anchor_attn_step_1
    unit = float(torch.tensor(LOG2E).to(dtype))
    for n, risers in ((1024, RISERS), (1152, RISERS[::2]), (1152, [])):
        q, k, v = _inputs(n, d, dtype, risers)
        _check(dense_causal_attention(q, k, v, sm_scale=0.125), _reference(q, k, v, 0.125 * unit / LOG2E, _causal(n)), v)
        k[:, :, 900, 1] = float("nan")
        got = dense_causal_attention(q, k, v, sm_scale=0.125)
        assert bool(torch.isfinite(got[:, :, :900]).all()) and bool(got[:, :, 900:].isnan().all())
    # the operator's window and its sparse stage: the third big block takes the second's keys there, with risers above all that its rows have seen
    n = 3072
    q, k, v = _inputs(n, d, dtype, RISERS + [1024 + x for x in RISERS] + [2048 + x for x in RISERS[:3]])
    k[:, :, 1024:2048:97, 0] = 100.0
    got = anchor_attn(q, k, v, sm_scale=0.125, block_size=64, difference=1e4, strict_reference=False)[0]
    _check(got, _reference(q, k, v, 0.125 * unit / LOG2E, _causal(n)), v)
    M = anchor_attn_step_1(q, k, v, 1, 1, 64, 16, 1, 4, n, d, 0.125)[1].reshape(1, 4, n)
    rows = torch.arange(n, device="cuda")
    seen = _causal(n) & ((rows[None, :] < 1024) | (rows[None, :] >= rows[:, None] // 1024 * 1024))
    want = (k[..., 0].float() * unit)[:, :, None, :].masked_fill(~seen, float("-inf")).amax(-1).repeat_interleave(2, 1)
    assert torch.equal(M, want)
