"""The operator against its own stages run one by one, at context lengths where the one-call path takes other routes: the
first big block is finished by stage 1, a single one has nothing to select, and the work-groups of stage 3 take one, two or
four query blocks.  The arithmetic is the same, so the results are the same bit for bit."""
import pytest
import torch

from anchor_attn.synthetic import make_qkv


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_big,d,block,step,theta,dtype", [
    (1, 14, 2, 1, 64, 128, 16, 12.0, torch.bfloat16),   # one big block
    (2, 4, 4, 1, 128, 64, 32, 12.0, torch.float16),
    (1, 7, 1, 2, 128, 16, 16, 2.0, torch.bfloat16),     # big blocks of two query blocks
    (1, 8, 2, 3, 64, 256, 16, 12.0, torch.float16),     # pooling as a pass of its own
    (1, 32, 8, 3, 128, 128, 16, 100.0, torch.bfloat16), # every key: two query blocks to a work-group would not fill the chip
    (1, 32, 8, 10, 64, 64, 32, 2.0, torch.bfloat16),    # two to a work-group
    (1, 32, 8, 9, 128, 128, 16, 2.0, torch.bfloat16),   # four
])
def test_operator_equals_its_stages(batch, hq, hkv, n_big, d, block, step, theta, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, anchor_attn_without_anchor
    n = n_big * block * step
    q, k, v, _ = make_qkv(n, hq, hkv, n_stripes=max(4, n // 100), seed=n + hq, head_dim=d)
    q, k, v = (x.expand(batch, -1, -1, -1).to("cuda", dtype).contiguous() for x in (q, k, v))
    out = torch.full((batch, n, hq, d), float("nan"), dtype=dtype, device="cuda").transpose(1, 2)
    got, ratio = anchor_attn(q, k, v, block_size=block, step=step, difference=theta, out=out)
    want, want_ratio = anchor_attn_without_anchor(q, k, v, block_size=block, step=step, difference=theta)
    assert got is out and torch.equal(out, want) and torch.equal(ratio, want_ratio)
    assert n_big > 1 or float(ratio) == 0.0


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_ctx", [(1, 2048), (255, 6144), (256, 10240), (8192, 131072), (70001, 126976)])
def test_ratio_equals_the_expression_in_torch(n, n_ctx):
    """The same operations on the same whole numbers, so the same float; sums beyond 2^31 among them."""
    from anchor_attn.src.ops.anchor_attn_v4 import _ratio
    counts = torch.randint(0, n_ctx, (n, 1, 1, 1), dtype=torch.int32, generator=torch.Generator().manual_seed(n)).cuda()
    got = _ratio(counts, 3, 7, n_ctx, 128, 16)
    want = counts.sum() / (3 * 7 * n_ctx * n_ctx / (128 * 16) // 2)
    assert got.dtype == want.dtype and got.shape == want.shape and torch.equal(got, want)
