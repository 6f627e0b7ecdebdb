"""Stage 2's index lists where a list is formed in several ways: one wave or eight, few or many keys to a wave, the ends of a
candidate range inside a mask word - against the keys that were made to pass (whole numbers: no tolerance)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (tokens, block size, step): rows of 1 to 4 words; 60 words; 64 (one wave's last size) and more; 512 words and 4096 (a turn, all turns) crossed
SIZES = [(1024, 16, 16), (4096, 128, 16), (6144, 128, 16), (4608, 16, 32), (20480, 64, 32), (139264, 256, 16)]


@pytest.mark.parametrize("n,bs,step", SIZES)
@pytest.mark.parametrize("geometry", [0, 1])
def test_lists_hold_the_keys_that_pass(n, bs, step, geometry):
    from anchor_attn.src.ops import _hip
    lib, big, heads, d = _hip.lib(), bs * step, 5, 64  # (each head another share of keys: none, few, half a word, mixed, all)
    g = torch.Generator().manual_seed(n)
    share = torch.tensor([0.0, 0.01, 0.4, 0.0, 1.0])[:, None].repeat(1, n)
    share[3] = (torch.arange(n) // 2048 % 3 == 1).float() * 0.97 + 0.01  # a wave's words dense, the next ones' not
    on = torch.rand(heads, n, generator=g) < share
    k = torch.zeros(heads, n, d, dtype=torch.bfloat16)
    k[..., 0] = on * 2.0 - 1.0
    k, qbar = k.cuda(), torch.zeros(heads, n // bs, d, dtype=torch.bfloat16, device="cuda")
    qbar[..., 0] = 64.0
    abar = torch.zeros(heads, n // bs, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(lib.aa_mask_words(1, heads, n, bs, step), dtype=torch.int32, device="cuda").fill_(-1)
    per_head = lib.aa_coords_entries_per_head(n, bs, step)
    coords = torch.full((heads, per_head), -7, dtype=torch.int32, device="cuda")
    counts = torch.full((heads, n // big), -7, dtype=torch.int32, device="cuda")
    _hip.check(lib.aa_stage2_select(qbar.data_ptr(), abar.data_ptr(), k.data_ptr(), heads * n * d, n * d, d, ws.data_ptr(), coords.data_ptr(),
                                    counts.data_ptr(), 1, heads, heads, n, d, bs, step, d ** -0.5, 0.0, geometry, _hip.dtype_code(k),
                                    torch.cuda.current_stream().cuda_stream))
    lo, slack = (bs, bs) if geometry == 0 else (big, 0)
    coords, counts = coords.cpu(), counts.cpu()
    written = torch.zeros_like(coords, dtype=torch.bool)
    for bb in range(n // big):
        at = 0 if bb <= 1 else big * (bb - 1) * bb // 2 - 2 * bs * (bb - 1)
        for h in range(heads):
            want = lo + on[h, lo:max(lo, bb * big - slack)].nonzero()[:, 0]
            assert int(counts[h, bb]) == want.numel(), (h, bb)
            assert torch.equal(coords[h, at:at + want.numel()].long(), want), (h, bb)
            written[h, at:at + want.numel()] = True
    assert (coords[~written] == -7).all()
