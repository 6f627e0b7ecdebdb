"""Scores that grow along the keys, by less and by far more than a probability's range, against float64: the flash kernel's
reference is the row max of the first 32 keys until the probabilities of a half-tile sum to too much.

Scores are whole numbers of nats times the 16-bit rounding of log2(e) that the kernels scale queries with (the rows mode
scales in float32), so they are exact.  Bound as in test_dense_rows.py: probabilities rounded to the 16-bit type (unit roundoff
u), u * max|v|, the result's rounding u * |out|, and five per cent for the float32 sums and exp2."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LOG2E = 1.44269504


def _inputs(n, d, dtype, seed, batch=1, hq=4, hkv=2):
    """Key scores of row-dependent size (1, 1/2 or 1/4 of them): low at first, then rising by steps between keys that are no
    multiple of a tile's, the largest of them past exp2's range, with stretches that stay level or fall."""
    g = torch.Generator().manual_seed(seed)
    level, scores = -100.0, []
    while len(scores) < n:
        level += (0.0, 4.0, 8.0, -12.0, 16.0, 104.0)[int(torch.randint(0, 6, (1,), generator=g))]
        level = min(level, 120.0) if len(scores) > n // 3 else min(level, -40.0)
        scores += [level] * int(torch.randint(9, 47, (1,), generator=g))
    q, k = torch.zeros(batch, hq, n, d, dtype=dtype), torch.zeros(batch, hkv, n, d, dtype=dtype)
    q[..., 0] = 8.0 / 2.0 ** torch.randint(0, 3, (batch, hq, n), generator=g)
    k[..., 0] = torch.tensor(scores[:n]) + torch.randint(-3, 4, (batch, hkv, n), generator=g) * 4.0
    v = torch.randn(batch, hkv, n, d, generator=g).to(dtype)
    return q.cuda(), k.cuda(), v.cuda()


def _reference(q, k, v, scale, keep):
    group = q.shape[1] // k.shape[1]
    s = (q.double()[..., :1] @ k.double()[..., :1].repeat_interleave(group, 1).transpose(2, 3).contiguous()) * scale
    return s.masked_fill(~keep, float("-inf")).softmax(-1).nan_to_num() @ v.double().repeat_interleave(group, 1)


def _check(out, want, v):
    u = 2.0 ** -8 if out.dtype == torch.bfloat16 else 2.0 ** -11
    past = (out.double() - want).abs() - 1.05 * u * (v.double().abs().max() + want.abs())
    assert bool((past <= 0).all()), float(past.max())


def _causal(n, rows=None):
    keys = torch.arange(n, device="cuda")
    return keys[None, :] <= keys[n - (rows or n):, None]


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_rows_masked_and_operator(d, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, dense_causal_attention, dense_rows_attention
    scaled = 0.125 * float(torch.tensor(LOG2E).to(dtype)) / LOG2E  # what the pre-scaled queries stand for
    for seed, n in ((1, 640), (2, 1664)):
        q, k, v = _inputs(n, d, dtype, seed)
        _check(dense_causal_attention(q, k, v, sm_scale=0.125), _reference(q, k, v, scaled, _causal(n)), v)
        for rows in (77, n):
            want = _reference(q[:, :, n - rows:], k, v, 0.125, _causal(n, rows))
            _check(dense_rows_attention(q[:, :, n - rows:], k, v, n - rows, sm_scale=0.125), want, v)
        keep = _causal(n) & (torch.arange(n, device="cuda") % 97 >= 40)[None, :]  # (rows that see nothing, tiles that start unseen)
        keep[n // 2:, : n // 3] = False
        got = dense_rows_attention(q, k, v, sm_scale=0.125, mask=keep[None, None])
        _check(got, _reference(q, k, v, 0.125, keep), v)
    # the operator: a single big block, and three of which the last takes all keys of the second in its sparse stage
    for n_big in (1, 3):
        q, k, v = _inputs(1024 * n_big, d, dtype, 3 + n_big)
        got = anchor_attn(q, k, v, sm_scale=0.125, block_size=64, difference=1e4, strict_reference=False)[0]
        _check(got, _reference(q, k, v, scaled, _causal(1024 * n_big)), v)
    # scores of the sparse stage's keys far above all that stage 1 has seen
    k[:, :, 1024:2048, 0] += 112.0
    got = anchor_attn(q, k, v, sm_scale=0.125, block_size=64, difference=1e4, strict_reference=False)[0]
    _check(got, _reference(q, k, v, scaled, _causal(3072)), v)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n,rows", [(900, 900), (6000, 77)])  # (teams of waves at head dimension 64; chunks that are merged)
def test_values_that_sums_of_larger_probabilities_would_overflow_with(n, rows, d):
    """Every second 32 keys score 6.75 nats above the others, so that probabilities relative to a part's first 32 keys are up to 2^9.7 and
    none is redone for it; values from what n probabilities of 1 hold without overflow downwards, past 1024 times smaller."""
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    g = torch.Generator().manual_seed(n + d)
    q, k = torch.zeros(1, 4, rows, d, dtype=torch.bfloat16), torch.zeros(1, 2, n, d, dtype=torch.bfloat16)
    q[..., 0] = 8.0
    k[..., 0] = (torch.arange(n) // 32 % 2) * 6.75
    unit = torch.rand(1, 2, n, d, generator=g) * 0.5 + 0.5
    unit[..., 1::2] *= -1.0
    q, k, keep = q.cuda(), k.cuda(), _causal(n, rows)
    for power in range(0, 20, 2):
        v = (unit * (3.4e38 / n / 2.0 ** power)).bfloat16().cuda()
        want = _reference(q, k, v, 0.125, keep)
        _check(dense_rows_attention(q, k, v, n - rows, sm_scale=0.125), want, v)
        _check(dense_rows_attention(q, k, v, sm_scale=0.125, mask=keep[None, None]), want, v)
    v[:, :, 5, 0] = float("inf")  # (and infinities stay what they are)
    got = dense_rows_attention(q, k, v, n - rows, sm_scale=0.125)
    assert bool((got[:, :, 5:, 0] == float("inf")).all()) and bool(torch.isfinite(got[..., 1:]).all())
