"""Stage 2's thresholds: the smallest float32 dot product that passes the selection test, found by search, against the test itself
evaluated in numpy at the threshold and at the float32 below it (exact: no tolerance)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _round16(x, scale2, dtype):
    """(x * scale2).to(dtype) as the operator's definition compiles: bf16 rounds the float32 product, fp16 the exact one."""
    if dtype == torch.bfloat16:
        return torch.from_numpy((x * scale2).astype(np.float32)).bfloat16().float().numpy()
    return (x.astype(np.float64) * float(scale2)).astype(np.float16).astype(np.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("theta", [0.0, 17.3, -17.3, 1e30, float("inf"), float("-inf")])
def test_thresholds_are_the_smallest_numbers_that_pass(dtype, theta):
    from anchor_attn.src.ops import _hip
    lib, bs, step, heads, d = _hip.lib(), 16, 16, 7, 64
    n = 512  # two big blocks, 32 pooled rows a head: 224 rows, no multiple of a wave's or a work-group's
    g = torch.Generator().manual_seed(5)
    anchors = (torch.randn(heads, n // bs, generator=g) * 20).to(dtype)
    tiny = 1e-30 if dtype == torch.bfloat16 else 6e-8
    special = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), 6e4, -6e4, tiny, -tiny])
    anchors[0, : special.numel()] = special.to(dtype)
    abar = anchors.cuda()
    qbar, k = torch.zeros(heads, n // bs, d, dtype=dtype, device="cuda"), torch.zeros(heads, n, d, dtype=dtype, device="cuda")
    words = lib.aa_mask_words(1, heads, n, bs, step)
    ws = torch.zeros(words, dtype=torch.int32, device="cuda")
    coords = torch.zeros(heads * lib.aa_coords_entries_per_head(n, bs, step), dtype=torch.int32, device="cuda")
    counts = torch.zeros(heads * 2, dtype=torch.int32, device="cuda")
    _hip.check(lib.aa_stage2_select(qbar.data_ptr(), abar.data_ptr(), k.data_ptr(), heads * n * d, n * d, d, ws.data_ptr(), coords.data_ptr(),
                                    counts.data_ptr(), 1, heads, heads, n, d, bs, step, d ** -0.5, theta, 0, _hip.dtype_code(k),
                                    torch.cuda.current_stream().cuda_stream))
    thr = ws[words - heads * (n // bs):].view(torch.float32).cpu().numpy()
    a, scale2 = anchors.float().numpy().ravel(), np.float32(d ** -0.5 * 1.44269504)

    def passes(x):
        with np.errstate(all="ignore"):
            return (_round16(x, scale2, dtype) + np.float32(theta)).astype(np.float32) >= a
    none = np.isnan(thr)
    assert np.array_equal(none, ~passes(np.full_like(thr, np.inf)))
    assert passes(thr)[~none].all()
    lowest = thr == -np.inf
    assert not passes(np.nextafter(thr, np.float32(-np.inf)))[~none & ~lowest].any()
