"""Prompts that end in part of a big block: the operator on the whole big blocks and dense attention of the rows that remain, in one call.
Against the two calls that it takes the place of, over what both accept, and the remaining rows against float64 (bound as in test_dense_rows.py)."""
import ctypes
from types import SimpleNamespace

import pytest
import torch

from test_dense_rows import _check, _qkv, _reference


def _module(block, step, theta):
    return SimpleNamespace(config=SimpleNamespace(block_size_M=block, step=step, theta=theta))


def _two_calls(q, k, v, block, step, theta, scale=None):
    from anchor_attn.src.ops.anchor_attn_v4 import anchor_attn, dense_rows_attention
    main = q.shape[2] - q.shape[2] % (block * step)
    first = anchor_attn(q[:, :, :main], k[:, :, :main], v[:, :, :main], sm_scale=scale, block_size=block, step=step, difference=theta,
                        return_computational_ratio=False)
    return torch.cat([first, dense_rows_attention(q[:, :, main:], k, v, main, sm_scale=scale)], 2)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n,d,block,step,dtype,storage", [
    (1, 32, 8, 2049, 128, 128, 16, torch.bfloat16, "model"),   # one row: the decode kernel
    (1, 28, 4, 2053, 128, 128, 16, torch.float16, "model"),    # the fewest rows that a column block takes
    (1, 8, 2, 4095, 128, 128, 16, torch.bfloat16, "heads"),    # the most rows beside one big block
    (2, 7, 1, 2100, 128, 128, 16, torch.bfloat16, "cache"),    # chunks that are merged
    (1, 14, 2, 2400, 64, 128, 16, torch.bfloat16, "model"),    # two teams of waves in both parts
    (1, 14, 2, 2400, 64, 128, 16, torch.float16, "cache"),
    (3, 16, 16, 2061, 64, 128, 16, torch.bfloat16, "heads"),   # more units than XCDs, no groups
    (1, 4, 2, 7167, 64, 64, 16, torch.bfloat16, "model"),      # six big blocks of 1024 and all but one row of a seventh
    (2, 4, 1, 4500, 128, 64, 32, torch.float16, "model"),
    (1, 4, 2, 9001, 128, 256, 16, torch.bfloat16, "heads"),    # queries pooled by a launch of their own
])
def test_against_two_calls(batch, hq, hkv, n, d, block, step, dtype, storage):
    from anchor_attn.src.modules.llama.anchor_attention import anchor_attention_forward
    q, k, v = _qkv(batch, hq, hkv, n, n, d, dtype, n + d)
    q *= 0.25  # (the operator's queries are rounded once more when they are scaled: smaller scores)
    if storage == "heads":
        q = q.contiguous()
    elif storage == "cache":  # the filled part of a larger cache, keys and values interleaved
        kv = torch.full((batch, hkv, n + 64, 2, d), float("nan"), dtype=dtype, device="cuda")
        kv[:, :, :n, 0], kv[:, :, :n, 1] = k, v
        k, v = kv[:, :, :n, 0], kv[:, :, :n, 1]
    main = n - n % (block * step)
    out, _ = anchor_attention_forward(_module(block, step, 2.0), q, k, v, None)
    got, want = out.transpose(1, 2), _two_calls(q, k, v, block, step, 2.0)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # (each within 1.05 u (max|v| + |out|) of the attention of the same rounded queries, from another reference for the exponentials)
    assert bool(((got - want).double().abs() <= 2.1 * u * (v.double().abs().max() + want.double().abs())).all())
    if not (d == 64 and main == block * step):  # (a single big block's teams of waves depend on what else is in the launch)
        assert torch.equal(got[:, :, :main], want[:, :, :main])
    keep = (torch.arange(n, device="cuda")[None, :] <= torch.arange(main, n, device="cuda")[:, None]).expand(batch, -1, -1)
    _check(got[:, :, main:], _reference(q[:, :, main:], k, v, d ** -0.5, keep), v, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2300, 6500])
def test_captured_and_on_another_stream(n):
    from anchor_attn.src.modules.llama.anchor_attention import anchor_attention_forward
    module = _module(128, 16, 12.0)
    q, k, v = _qkv(1, 8, 2, n, n, 128, torch.bfloat16, 3)
    want = anchor_attention_forward(module, q, k, v, None)[0]
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        assert torch.equal(anchor_attention_forward(module, q, k, v, None)[0], want)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        got = anchor_attention_forward(module, q, k, v, None)[0]
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.gpu
def test_who_keeps_the_two_calls(monkeypatch):
    from anchor_attn.src.modules.llama import anchor_attention as plug
    q, k, v = _qkv(1, 4, 2, 2300, 2300, 64, torch.bfloat16, 9)
    module, beside = _module(128, 16, 12.0), []
    want = plug.anchor_attention_forward(module, q, k, v, None)[0]
    inner = plug.anchor_attn
    monkeypatch.setattr(plug, "anchor_attn", lambda *a, **kw: (beside.append("rows" in kw), inner(*a, **kw))[1])
    plug.anchor_attention_forward(module, q, k, v, None, scaling=1e-31)  # (a scale that the rows kernel does not take)
    got = plug.anchor_attention_forward(module, q.requires_grad_(True), k, v, None)[0]
    assert beside == [False, False] and float((got - want).detach().float().abs().max()) < 0.05
    with torch.no_grad():
        assert torch.equal(plug.anchor_attention_forward(module, q, k, v, None)[0], want)
    assert beside == [False, False, True]


def test_sizes_that_are_refused():
    from anchor_attn.src.ops import _hip
    lib = _hip.lib()
    p = ctypes.create_string_buffer(1 << 16)
    base = (ctypes.addressof(p) + 255) & ~255

    def run(n=2048, rows=300, hq=4, hkv=2, d=64, block=128, step=16, nbytes=1 << 40, scale=0.1, workspace=base, dtype=0, offset=2048, ratio=None):
        t3 = (base, 0, 0, d)
        rc = lib.aa_anchor_attn_rows_fwd(*t3 * 8, rows, 2348, offset, scale, workspace, nbytes, None, ratio, None, 0.0, 1, hq, hkv, n, d, block, step, 0.1,
                                         12.0, _hip.AA_SCALE_BF16_CHAIN, 0, dtype, None)
        return rc, lib.aa_last_error().decode()

    for bad in (dict(n=2047), dict(n=0), dict(n=-1), dict(block=0), dict(step=-16), dict(hkv=3), dict(d=96), dict(nbytes=1), dict(scale=0.0),
                dict(workspace=None), dict(dtype=7), dict(rows=0), dict(offset=-1), dict(rows=1 << 21), dict(ratio=base)):
        rc, message = run(**bad)
        assert rc != 0 and "aa_anchor_attn_rows_fwd" in message, (bad, message)
    assert lib.aa_anchor_attn_rows_workspace_bytes(1, 4, 2, 2047, 64, 128, 16, 300, 2347, 2047) == 0
    for n in (2049, 2300, 4095, 40001):  # the operator's scratch, and the rows' where they are cut into chunks
        main = n - n % 2048
        whole = lib.aa_anchor_attn_rows_workspace_bytes(1, 4, 2, main, 64, 128, 16, n - main, n, main)
        assert whole >= lib.aa_workspace_bytes(1, 4, main, 64, 128, 16) > 0
