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
    # the operator's window and its sparse stage: the third big block takes the second's keys there, of which the first is above all that its rows have seen
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


def _multiplicity(n, block, big):
    """How often a row takes a key with every candidate selected: window and list of the operator as it runs, which share keys and leave some out."""
    rows, keys = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
    own = rows // big * big
    window = (keys < big) | (keys >= own)
    listed = (own > 0) & (keys >= block) & (keys < own - block)
    return ((window & (keys <= rows)).double() + listed.double())[None, None]


def _weighted(q, k, v, scale, times):
    group = q.shape[1] // k.shape[1]
    s = (q.double()[..., :1] @ k.double()[..., :1].repeat_interleave(group, 1).transpose(2, 3).contiguous()) * scale
    p = (s - s.masked_fill(times == 0, float("-inf")).amax(-1, keepdim=True)).clamp(max=0).exp() * times
    return p / p.sum(-1, keepdim=True) @ v.double().repeat_interleave(group, 1)


def _quiet_but(risers, batch, n, hq, hkv, d, dtype, seed):
    """A sink, and per batch element and KV head ``risers`` [batch, hkv, m]: keys that are each a nat (rows of half the size: half a nat) above the one
    before, so that sink and risers all have weight at the end; the others score 18 nats and more (9) less."""
    g = torch.Generator().manual_seed(seed)
    q, k = torch.zeros(batch, hq, n, d, dtype=dtype), torch.zeros(batch, hkv, n, d, dtype=dtype)
    q[..., 0] = 8.0 / 2.0 ** torch.randint(0, 2, (batch, hq, n), generator=g)
    k[..., 0] = torch.randint(-30, -10, (batch, hkv, n), generator=g).to(dtype)
    k[..., 0, 0] = 8.0
    up = 9.0 + torch.arange(risers.shape[2]).to(dtype).expand_as(risers)
    k[..., 0].scatter_(2, risers, up)
    v = torch.randn(batch, hkv, n, d, generator=g).to(dtype)
    return q.cuda(), k.cuda(), v.cuda()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_keys_above_the_sink_in_a_list(d, dtype):
    """Lists of 15, 23, 31 and 39 tiles of which the first are quiet, with two risers in later ones: in both halves of tiles, both buffers, the first and a
    later window of the list, a single one and ones that are walked by two query blocks in turn; elsewhere the same risers are keys of the rows' own big block."""
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    n, batch, hkv, block, big = 3072, 40, 2, 32, 512
    g = torch.Generator().manual_seed(d)
    first = torch.randint(big, 2300, (batch, hkv, 1), generator=g)
    risers = torch.cat((first, first + torch.randint(1, 200, (batch, hkv, 1), generator=g)), 2)
    q, k, v = _quiet_but(risers, batch, n, 4, hkv, d, dtype, d)
    got = anchor_attn(q, k, v, sm_scale=0.125, block_size=block, difference=1e4)[0]
    scale, times = 0.125 * float(torch.tensor(LOG2E).to(dtype)) / LOG2E, _multiplicity(n, block, big)
    for b in range(batch):
        _check(got[b:b + 1], _weighted(q[b:b + 1], k[b:b + 1], v[b:b + 1], scale, times), v[b:b + 1])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch", [3, 16])  # (head dimension 64: 108 and 576 work-groups, of two teams of waves and of one)
def test_keys_above_the_sink_in_dense_rows(d, dtype, batch):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_causal_attention
    n, hkv = 1152, 2
    first = torch.randint(128, 900, (batch, hkv, 1), generator=torch.Generator().manual_seed(batch))
    q, k, v = _quiet_but(torch.cat((first, first + 101), 2), batch, n, 4, hkv, d, dtype, batch)
    scale = 0.125 * float(torch.tensor(LOG2E).to(dtype)) / LOG2E
    _check(dense_causal_attention(q, k, v, sm_scale=0.125), _weighted(q, k, v, scale, _causal(n).double()[None, None]), v)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_maximum_that_grows_again_and_again(d, dtype):
    """More leavings of the loops without maxima than rows of 98 tiles pay for, one after the other and again after stretches without."""
    from anchor_attn.src.ops.anchor_attn_v4 import dense_causal_attention
    n = 6272
    at = torch.cat([torch.arange(start, start + 800, 77) for start in (130, 3300, 5400)])
    q, k, v = _quiet_but(at.expand(1, 2, -1), 1, n, 8, 2, d, dtype, d)
    k[0, :, at, 0] = (8.0 + 0.25 * torch.arange(1, len(at) + 1)).to(dtype).cuda()
    scale = 0.125 * float(torch.tensor(LOG2E).to(dtype)) / LOG2E
    _check(dense_causal_attention(q, k, v, sm_scale=0.125), _weighted(q, k, v, scale, _causal(n).double()[None, None]), v)
