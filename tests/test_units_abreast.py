"""More KV heads (of all batch elements) than XCDs, or fewer that share them unevenly: work-groups take them side by side.  Every row must still be computed, once, at
numbers of units that do and do not divide the XCDs and their CUs, against float64 (bound as in test_dense_rows.py)."""
import pytest
import torch

from test_dense_rows import _check, _qkv, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,hq,hkv,n,d", [
    (2, 16, 8, 333, 128),   # two units an XCD
    (4, 8, 8, 200, 64),     # four, a CU's share of 32 work-groups and fewer
    (3, 16, 8, 300, 64),    # three: not a divisor of 32
    (3, 8, 4, 190, 128),    # twelve units: all XCDs take all units
    (5, 4, 2, 129, 64),     # ten, and a number of work-groups that 8 does not divide
    (9, 8, 8, 257, 64),
    (1, 28, 4, 333, 128),   # fewer than XCDs, with rows that the XCDs of a unit cannot share evenly
    (1, 14, 2, 333, 64),
    (2, 2, 1, 700, 64),
])
def test_rows_masked_dense_and_operator(batch, hq, hkv, n, d):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, dense_causal_attention, dense_rows_attention
    q, k, v = _qkv(batch, hq, hkv, n, n, d, torch.bfloat16, n)
    rows = torch.arange(n, device="cuda")
    causal = (rows[None, :] <= rows[:, None]).expand(batch, -1, -1)
    nan = torch.full((batch, n, hq, d), float("nan"), dtype=q.dtype, device="cuda").transpose(1, 2)
    _check(dense_rows_attention(q, k, v, 0, out=nan.clone()), _reference(q, k, v, d ** -0.5, causal), v, q.dtype)
    pads = torch.arange(batch, device="cuda") * (n // (batch + 1))
    keep = causal & (rows[None, None, :] >= pads[:, None, None])
    got = dense_rows_attention(q, k, v, mask=keep[:, None], out=nan.clone())
    _check(got, _reference(q, k, v, d ** -0.5, keep), v, q.dtype)
    n = 256
    q, k, v = _qkv(batch, hq, hkv, n, n, d, torch.bfloat16, 7)
    q = q * 0.25  # (queries are rounded once more when they are scaled: smaller scores)
    causal = torch.ones(n, n, dtype=torch.bool, device="cuda").tril().expand(batch, -1, -1)
    want = _reference(q, k, v, d ** -0.5, causal)
    for got in (dense_causal_attention(q, k, v), anchor_attn(q, k, v, block_size=16, return_computational_ratio=False)):
        assert bool(torch.isfinite(got).all()) and float((got.double() - want).norm() / want.norm()) < 1e-2
