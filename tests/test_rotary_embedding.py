"""The rotary embedding of queries and keys as one kernel, which rounds as the framework's single operations do: the same bits."""
import copy
import inspect
import pickle
import types

import pytest
import torch

from test_between_products import _tiny

FAMILIES = ("Llama", "Qwen2")


def _modeling(family):
    from transformers.models.llama import modeling_llama
    from transformers.models.qwen2 import modeling_qwen2
    return modeling_llama if family == "Llama" else modeling_qwen2


def _attentions(model, family):
    return [m for m in model.modules() if type(m).__name__ == f"{family}Attention"]


@pytest.mark.parametrize("family", FAMILIES)
def test_attentions_run_their_class_s_code(family, monkeypatch):
    from anchor_attn import patch_model
    from anchor_attn.src.modules import model_forward
    plain = patch_model(_tiny(family), "flash", {"fuse_between_products": False})
    m = patch_model(_tiny(family), "flash")
    tokens = torch.randint(0, 100, (2, 9))
    assert all("forward" in a.__dict__ for a in _attentions(m, family)) and not any("forward" in a.__dict__ for a in _attentions(plain, family))
    with torch.no_grad():
        want = plain(tokens).logits
        assert torch.equal(m(tokens).logits, want)
        other = copy.deepcopy(m.model.layers[0].self_attn)
        assert other.forward.module is other and type(pickle.loads(pickle.dumps(other))) is type(other)
        assert torch.equal(torch.compile(m, backend="eager", fullgraph=True)(tokens, use_cache=False).logits, plain(tokens).logits)
        # what a program puts in the places later
        taken = []
        monkeypatch.setattr(model_forward, "_rope_tensors", lambda *args: taken.append(args))
        m(tokens)
        assert len(taken) == 2
        with monkeypatch.context() as later:
            later.setattr(_modeling(family), "apply_rotary_pos_emb", lambda q, k, cos, sin: (q, k))
            assert torch.equal(m(tokens).logits, plain(tokens).logits) and not torch.equal(m(tokens).logits, want)
            assert model_forward.fuse_between_products(_tiny(family).model.layers[0].self_attn) == 0
        with monkeypatch.context() as later:
            cls = getattr(_modeling(family), f"{family}Attention")
            later.setattr(cls, "forward", lambda self, hidden_states, **kwargs: (hidden_states, None))
            assert torch.equal(m(tokens).logits, plain(tokens).logits)
        assert len(taken) == 2


@pytest.mark.parametrize("family", FAMILIES)
def test_a_patched_forward_names_its_module_and_function(family):
    from anchor_attn import patch_model
    m = patch_model(_tiny(family), "flash")
    hidden = torch.randn(1, 5, m.config.hidden_size)
    embeddings = m.model.rotary_emb(hidden, torch.arange(5)[None])
    for a in _attentions(m, family):
        for bound in (a.forward, copy.copy(a.forward), copy.deepcopy(a).forward):
            assert bound.__name__ == "forward"
            assert inspect.signature(bound) == inspect.signature(type(a).forward.__get__(a))
            with torch.no_grad():
                want = type(a).forward(a, hidden, position_embeddings=embeddings, attention_mask=None)[0]
                assert torch.equal(types.MethodType(bound.__func__, bound.__self__)(hidden, position_embeddings=embeddings, attention_mask=None)[0], want)
        assert a.forward.__self__ is a and copy.copy(a.forward).__self__ is a


@pytest.mark.parametrize("change,message", [
    ({"batch": 0}, "must be positive"), ({"n_kv_heads": -1}, "must be positive"), ({"n_tokens": 0}, "must be positive"),
    ({"head_dim": 24}, "not supported"), ({"head_dim": 1040}, "not supported"), ({"head_dim": 0}, "not supported"),
    ({"batch": 1 << 20, "n_tokens": 1 << 12}, "not supported"),  # 2^32 pieces
    ({"dtype": 2}, "dtype"), ({"q": 0}, "q is NULL"), ({"k_out": 0}, "k_out is NULL"), ({"cos": 0}, "cos is NULL"), ({"sin": 4104}, "sin must be 16-byte aligned"),
    ({"k": 4104}, "k must be 16-byte aligned"), ({"q_sh": 60}, "q must be 16-byte aligned with strides"), ({"ko_sn": 56}, "smaller than head_dim"),
    ({"qo_sn": 16392}, "larger than 16384"), ({"n_tokens": 1 << 20, "k_sn": 4096}, "32-bit byte offsets"), ({"cs_sb": 20}, "batch stride"),
])
def test_what_the_c_interface_refuses(change, message):
    """Before anything is launched: the addresses are never read."""
    from anchor_attn.src.ops import _hip
    args = {"q": 4096, "q_sb": 2048, "q_sh": 64, "q_sn": 256, "k": 4096, "k_sb": 1024, "k_sh": 64, "k_sn": 128,
            "q_out": 4096, "qo_sb": 2048, "qo_sh": 64, "qo_sn": 256, "k_out": 4096, "ko_sb": 1024, "ko_sh": 512, "ko_sn": 64,
            "cos": 4096, "sin": 4096, "cs_sb": 0, "batch": 1, "n_q_heads": 4, "n_kv_heads": 2, "n_tokens": 8, "head_dim": 64, "dtype": 0, "stream": None}
    assert len(args) == len(_hip.lib().aa_rope.argtypes) and set(change) <= set(args)
    with pytest.raises(_hip.AnchorAttnHipError, match=message):
        _hip.check(_hip.lib().aa_rope(*{**args, **change}.values()))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,n,hq,hkv,d,own_angles", [(1, 1, 32, 8, 64, False), (1, 37, 14, 2, 64, False), (3, 65, 28, 4, 128, False),
                                                        (2, 130, 5, 1, 128, True), (2, 7, 1, 1, 16, True), (1, 300, 32, 8, 128, False), (1, 9, 3, 3, 256, False)])
def test_against_the_single_operations(batch, n, hq, hkv, d, own_angles, dtype):
    from transformers.models.llama.modeling_llama import apply_rotary_pos_emb

    from anchor_attn.src.modules.model_forward import _rope_tensors
    from anchor_attn.src.ops import _hip
    from anchor_attn.src.ops.anchor_step_1_2_v2 import _stream
    g = torch.Generator(device="cuda").manual_seed(n + d)
    make = lambda *shape: (4.0 * torch.randn(shape, generator=g, device="cuda")).to(dtype)  # noqa: E731
    angles = torch.rand(batch if own_angles else 1, n, d, generator=g, device="cuda") * 100.0
    cos, sin = angles.cos().to(dtype), angles.sin().to(dtype)
    layouts = (make(batch, n, hq, d).transpose(1, 2), make(batch, n, hkv, d).transpose(1, 2)), (make(batch, hq, n, d), make(batch, hkv, n, d)), \
        tuple(make(batch, n, hq + hkv, d).transpose(1, 2).split((hq, hkv), 1))  # (as projected; contiguous; parts of one projection)
    with torch.no_grad():
        for q, k in layouts:
            q[0, 0, 0, 0], k[0, 0, 0, -1] = float("inf"), -0.0
            (q_out, k_out), numbers = _rope_tensors(q, k, cos, sin)
            _hip.check(_hip.lib().aa_rope(*numbers, _stream()))
            want = apply_rotary_pos_emb(q, k, cos, sin)
            assert q_out.stride() == torch.empty_like(q).stride() and k_out.is_contiguous()
            for got, w in zip((q_out, k_out), want):
                assert torch.equal(got.isnan(), w.isnan()) and torch.equal(got.nan_to_num(7.0), w.nan_to_num(7.0))


@pytest.mark.gpu
def test_calls_that_stay_with_the_single_operations():
    from anchor_attn.src.modules.model_forward import _rope_tensors
    q, k = (torch.randn(1, h, 6, 64, device="cuda").bfloat16() for h in (4, 2))
    cos, sin = (torch.randn(1, 6, 64, device="cuda").bfloat16() for _ in range(2))
    assert _rope_tensors(q, k, cos, sin) is not None
    wide = torch.randn(1, 4, 6, 128, device="cuda").bfloat16()
    for args in ((q.float(), k.float(), cos.float(), sin.float()), (q, k, cos.float(), sin.float()), (q.cpu(), k.cpu(), cos.cpu(), sin.cpu()), (q, k, cos[:, :5], sin[:, :5]),
                 (wide[..., ::2], k, cos, sin), (wide[..., 1:65], k, cos, sin), (q[:, :, :0], k[:, :, :0], cos[:, :0], sin[:, :0]), (q, k, cos[0], sin[0]),
                 (q[..., :40], k[..., :40], cos[..., :40], sin[..., :40]), (q.clone().requires_grad_(), k, cos, sin), (q, k[:, :, :5], cos, sin),
                 (torch.nn.Parameter(q), k, cos, sin), (q, k, cos.expand(2, 6, 64), sin.expand(2, 6, 64))):
        assert _rope_tensors(*args) is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert _rope_tensors(q, k, cos, sin) is None


@pytest.mark.gpu
@pytest.mark.parametrize("family", FAMILIES)
def test_patched_model_gives_the_same_bits(family, monkeypatch):
    from anchor_attn import patch_model
    from anchor_attn.src.ops import _hip
    m = patch_model(_tiny(family).to("cuda", torch.bfloat16), "flash")
    calls, inner = [], _hip.lib().aa_rope
    monkeypatch.setattr(_hip.lib(), "aa_rope", lambda *a: (calls.append(a), inner(*a))[1])
    mask = torch.ones(2, 33, dtype=torch.long, device="cuda")
    mask[1, :5] = 0
    tokens = torch.randint(1, 100, (2, 33), device="cuda")
    with torch.no_grad():
        got = m(tokens, attention_mask=mask, position_ids=(mask.cumsum(-1) - 1).clamp(min=0))  # (a batch element's own angles)
        step = m(tokens[:, :1], attention_mask=torch.cat((mask, mask[:, :1]), 1), past_key_values=copy.deepcopy(got.past_key_values))
        assert len(calls) == 4
        for a in _attentions(m, family):
            del a.__dict__["forward"]
        want = m(tokens, attention_mask=mask, position_ids=(mask.cumsum(-1) - 1).clamp(min=0))
        assert torch.equal(got.logits, want.logits)
        assert torch.equal(step.logits, m(tokens[:, :1], attention_mask=torch.cat((mask, mask[:, :1]), 1), past_key_values=want.past_key_values).logits)
        assert len(calls) == 4
