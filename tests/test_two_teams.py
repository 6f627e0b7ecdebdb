"""Head dimension 64 in launches that leave a work-group alone on its CU: two teams of waves share its tiles and are merged.  Even and odd
numbers of tiles, tiles that only one team has, and rows whose keys all belong to one team, against float64 (bound as in test_dense_rows.py)."""
import pytest
import torch

from test_dense_rows import _check, _qkv, _reference

pytestmark = pytest.mark.gpu
D = 64


def _causal(n, batch=1):
    return torch.ones(n, n, dtype=torch.bool, device="cuda").tril().expand(batch, -1, -1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n", [(32, 8, 769), (32, 8, 900), (32, 8, 992), (4, 4, 1600), (28, 4, 833)])
def test_rows(hq, hkv, n, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    q, k, v = _qkv(1, hq, hkv, n, n, D, dtype, n)
    out = torch.full((1, n, hq, D), float("nan"), dtype=dtype, device="cuda").transpose(1, 2)
    _check(dense_rows_attention(q, k, v, 0, out=out), _reference(q, k, v, D ** -0.5, _causal(n)), v, dtype)
    v[:, :, 321, 3] = float("inf")  # in a tile of the second team
    got = dense_rows_attention(q, k, v, 0)
    assert bool((got[:, :, 321:, 3] == float("inf")).all()) and bool(torch.isfinite(got[:, :, :256]).all())
    other = [c for c in range(D) if c != 3]
    assert bool(torch.isfinite(got[..., other]).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_masked(dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    batch, hq, hkv, n = 2, 14, 2, 900
    q, k, v = _qkv(batch, hq, hkv, n, n, D, dtype, 5)
    tile = torch.arange(n, device="cuda") // 64
    keep = _causal(n, batch).clone()
    keep[0, :300, tile != 2] = False           # one tile, the first team's
    keep[0, 300:500, (tile != 1) & (tile != 2)] = False
    keep[0, 500:600] = False                   # nothing at all
    keep[1, :, tile % 2 == 0] = False          # tiles that are not visited
    keep[1, 800:, tile > 4] = False
    got = dense_rows_attention(q, k, v, mask=keep[:, None])
    _check(got, _reference(q, k, v, D ** -0.5, keep), v, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,n,block", [(14, 2, 2048, 128), (4, 2, 1024, 64), (32, 8, 1024, 64), (2, 1, 4096, 256)])
def test_dense_and_single_big_blocks(hq, hkv, n, block, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, anchor_attn_without_anchor, dense_causal_attention
    q, k, v = _qkv(1, hq, hkv, n, n, D, dtype, n)
    q = q * 0.25  # (queries are rounded once more when they are scaled: smaller scores)
    want = _reference(q, k, v, D ** -0.5, _causal(n))
    bound = 1e-2 if dtype == torch.bfloat16 else 1.5e-3
    out, ratio = anchor_attn(q, k, v, block_size=block)
    assert float(ratio) == 0.0 and torch.equal(out, anchor_attn_without_anchor(q, k, v, block_size=block)[0])
    for got in (out, dense_causal_attention(q, k, v)):
        assert float((got.double() - want).norm() / want.norm()) < bound
