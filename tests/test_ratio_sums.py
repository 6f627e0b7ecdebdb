"""The share of selected keys where the scores' work-groups form it, against the counts of the lists: on both sides of the line between the two, with
candidate ranges that begin and end inside a word of key bits, and on every replay of a captured graph."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(n, hq, hkv, seed, dtype=torch.bfloat16, batch=1, d=64):
    from anchor_attn.synthetic import make_qkv
    sets = [make_qkv(n, hq, hkv, head_dim=d, n_stripes=24, seed=seed + b)[:3] for b in range(batch)]
    return [torch.cat(x).to(dtype).cuda() for x in zip(*sets)]


def _by_lists(q, k, v, block, step, theta, geometry):
    """The same call with counts, whose sum the framework divides."""
    from anchor_attn.src.ops import _hip
    from anchor_attn.src.ops.anchor_attn_v4 import LOG2E, _anchor_attn, _ratio_denominator
    torch.set_default_dtype(torch.float64)  # (the route with counts)
    try:
        out, ratio = _anchor_attn(q, k, v, q.shape[-1] ** -0.5, block, step, theta * LOG2E, True, geometry=geometry)
    finally:
        torch.set_default_dtype(torch.float32)
    denominator = _ratio_denominator(*q.shape[:3], block, step)
    return out, round(float(ratio) * denominator), torch.tensor(float(denominator), dtype=torch.float32)


# work-groups of the scores: KV heads x batch x n / 256
@pytest.mark.parametrize("n,hq,hkv,block,step,theta,dtype,batch", [
    (512, 2, 1, 16, 16, 1e4, torch.bfloat16, 1),     # two big blocks of 256 keys, candidates 16 .. 239
    (1024, 4, 2, 16, 16, 12.3, torch.bfloat16, 2),   # ranges inside words
    (1536, 4, 4, 16, 32, 1e4, torch.float16, 1),
    (2048, 4, 2, 64, 16, -1e4, torch.bfloat16, 1),   # nothing selected
    (4096, 14, 2, 64, 32, 11.0, torch.float16, 1),
    (16384, 4, 2, 128, 16, 12.0, torch.bfloat16, 1),  # 128
    (8192, 5, 5, 64, 16, 12.0, torch.bfloat16, 1),    # 160: by the lists
])
@pytest.mark.parametrize("strict", [True, False])
def test_ratio_is_the_sum_of_the_counts(n, hq, hkv, block, step, theta, dtype, batch, strict):
    from anchor_attn.src.ops import _hip
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    q, k, v = _inputs(n, hq, hkv, 3, dtype, batch)
    want_out, total, denominator = _by_lists(q, k, v, block, step, theta, _hip.AA_GEOMETRY_AS_RUN if strict else _hip.AA_GEOMETRY_INTENDED)
    out, ratio = anchor_attn(q, k, v, block_size=block, step=step, difference=theta, strict_reference=strict)
    assert torch.equal(out, want_out)
    # (a whole number below 2^24 times a rounded reciprocal: three roundings of 2^-24)
    assert abs(float(ratio) * float(denominator) - total) <= 4 * 2.0 ** -24 * total
    if theta == 1e4 and strict:  # (without it two big blocks have no candidates)
        assert total > 0


@pytest.mark.parametrize("hq", [44, 48])  # 11 * 2^20 elements of stage 3's output: the last that the scores sum for, and more
def test_ratio_at_the_output_s_size_where_the_scores_stop_summing(hq):
    from anchor_attn.src.ops import _hip
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    q, k, v = _inputs(3072, hq, 4, 5, d=128)
    want_out, total, denominator = _by_lists(q, k, v, 64, 16, 12.0, _hip.AA_GEOMETRY_AS_RUN)
    out, ratio = anchor_attn(q, k, v, block_size=64, difference=12.0)
    assert torch.equal(out, want_out) and total > 0
    assert abs(float(ratio) * float(denominator) - total) <= 4 * 2.0 ** -24 * total


def test_ratio_on_every_replay_of_a_graph(monkeypatch):
    import my_utils
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn
    monkeypatch.setattr(my_utils.Logger, "enabled", False)  # (a line waits for the number, which a capture does not allow)
    given = [_inputs(2048, 4, 2, seed) for seed in (3, 11, 20)]
    want = [[x.clone() for x in anchor_attn(q, k, v, block_size=64)] for q, k, v in given]
    assert len({float(ratio) for _, ratio in want}) > 1
    q, k, v = [x.clone() for x in given[0]]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, ratio = anchor_attn(q, k, v, block_size=64)
    for i in (1, 0, 2, 2):
        for x, y in zip((q, k, v), given[i]):
            x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i][0]) and float(ratio) == float(want[i][1])
