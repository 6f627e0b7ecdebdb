"""The norms and gated activations of patched models as single kernels, against the framework's single operations.

Bound: both round to the 16-bit type twice (unit roundoff u), from float32 numbers that differ in their last bits (order of the sum of
squares, exponential), so a result may differ by one unit for either rounding: 4 u |want|."""
import copy
import pickle
import types

import pytest
import torch


def _close(got, want):
    u = 2.0 ** -8 if want.dtype == torch.bfloat16 else 2.0 ** -11
    assert got.dtype == want.dtype and got.shape == want.shape
    assert bool(((got.double() - want.double()).abs() <= 4 * u * want.double().abs() + 2.0 ** -23).all())


def _tiny(family="Llama", **kw):
    import transformers
    torch.manual_seed(0)
    cfg = getattr(transformers, f"{family}Config")(hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=4,
                                                   num_key_value_heads=2, vocab_size=100, max_position_embeddings=512, **kw)
    return getattr(transformers, f"{family}ForCausalLM")(cfg).eval()


@pytest.mark.parametrize("family", ["Llama", "Qwen2"])
def test_which_modules_are_fused_and_that_copies_keep_their_own(family):
    from anchor_attn import patch_model
    m = patch_model(_tiny(family), "flash")
    fused = [x for x in m.modules() if isinstance(x.__dict__.get("forward"), types.MethodType)]
    assert sorted({type(x).__name__ for x in fused}) == [f"{family}RMSNorm"] and len(fused) == 5  # (MLPs: the chunking wrapper is outside)
    assert all(x.forward.__self__ is x for x in fused)
    norm = copy.deepcopy(m.model.norm)
    assert norm.forward.__self__ is norm
    with torch.no_grad():
        norm.weight.fill_(2.0)
        x = torch.randn(3, 256)
        assert torch.equal(norm(x), 2.0 * m.model.norm(x))  # (on the CPU: the class's own)
    again = pickle.loads(pickle.dumps(m.model.norm))
    assert torch.equal(again(x), m.model.norm(x))
    before = [x.forward for x in fused]
    assert [x.forward for x in fused if patch_model(m, "dense")] == before


def test_other_activations_keep_their_own_forward(monkeypatch):
    from anchor_attn.src.modules import model_forward
    gelu, silu = _tiny(hidden_act="gelu").model.layers[0].mlp.bfloat16(), _tiny().model.layers[0].mlp.bfloat16()
    assert model_forward.fuse_between_products(gelu) == 0 and "forward" not in gelu.__dict__
    # an MLP that is given another activation after it was fused
    assert model_forward.fuse_between_products(silu) == 1
    x = torch.randn(1, 5, 256).bfloat16()
    monkeypatch.setattr(model_forward, "_kernel_takes", lambda *tensors: True)
    monkeypatch.setattr(model_forward, "_launch", lambda *args: pytest.fail("the kernel"))
    silu.act_fn = gelu.act_fn
    assert torch.equal(silu(x), type(silu).forward(silu, x))


@pytest.mark.parametrize("pattern", ["flash", "dense", "anchor_attn"])
def test_the_config_declines_the_fusion(pattern):
    from anchor_attn import patch_model
    m = patch_model(_tiny(), pattern, {"fuse_between_products": False})
    assert not any(isinstance(x.__dict__.get("forward"), types.MethodType) for x in m.modules()) and not hasattr(m.config, "fuse_between_products")
    assert sum(isinstance(x.__dict__.get("forward"), types.MethodType) for x in patch_model(m, pattern).modules()) == 5


def test_classes_that_compute_something_else_are_left_alone():
    from anchor_attn.src.modules.model_forward import fuse_between_products

    class LlamaRMSNorm(torch.nn.Module):  # a norm whose weight is an offset from one
        def __init__(self):
            super().__init__()
            self.weight, self.variance_epsilon = torch.nn.Parameter(torch.zeros(16)), 1e-3

        def forward(self, x):
            y = x.float()
            return ((1.0 + self.weight.float()) * y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + self.variance_epsilon)).to(x.dtype)
    m = torch.nn.Sequential(LlamaRMSNorm())
    assert fuse_between_products(m) == 0 and "forward" not in m[0].__dict__


def test_a_forward_that_a_class_is_given_later_is_used(monkeypatch):
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaMLP, LlamaRMSNorm

    from anchor_attn.src.modules import model_forward
    norm, mlp = LlamaRMSNorm(16), LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1))
    x = torch.randn(2, 16).bfloat16()
    assert model_forward.fuse_between_products(torch.nn.Sequential(norm, mlp).bfloat16()) == 2
    monkeypatch.setattr(model_forward, "_kernel_takes", lambda *tensors: True)
    monkeypatch.setattr(model_forward, "_launch", lambda *args: pytest.fail("the kernel"))
    with pytest.raises(pytest.fail.Exception):
        norm(x)
    with monkeypatch.context() as m:
        m.setattr(LlamaRMSNorm, "forward", lambda self, t: t + 1)
        m.setattr(LlamaMLP, "forward", lambda self, t: t + 2)
        assert torch.equal(norm(x), x + 1) and torch.equal(mlp(x), x + 2)
    with monkeypatch.context() as m:
        m.setattr(type(mlp.act_fn), "forward", lambda self, t: t * 3)
        assert torch.equal(mlp(x), mlp.down_proj(mlp.gate_proj(x) * 3 * mlp.up_proj(x)))
        assert model_forward.fuse_between_products(torch.nn.Sequential(LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1)))) == 0


@pytest.mark.parametrize("kind", ["norm", "mlp"])
def test_tracers_see_the_single_operations(kind):
    """Symbolic tracing, and export with a size that stays open, meet the class's own forward: no branch on a size or a device."""
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaMLP, LlamaRMSNorm

    from anchor_attn.src.modules.model_forward import fuse_between_products
    m = LlamaRMSNorm(16) if kind == "norm" else LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1))
    outer, x, longer = torch.nn.Sequential(m), torch.randn(2, 3, 16), torch.randn(2, 5, 16)
    assert fuse_between_products(outer) == 1
    with torch.no_grad():
        want = type(m).forward(m, longer)
        assert torch.equal(torch.fx.symbolic_trace(outer)(longer), want)
        for strict in (False, True):
            exported = torch.export.export(outer, (x,), dynamic_shapes=({1: torch.export.Dim("tokens")},), strict=strict)
            assert torch.equal(exported.module()(longer), want)


def test_other_activations_of_that_name_are_left_alone():
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaMLP

    from anchor_attn.src.modules.model_forward import _is_silu, fuse_between_products

    class SiLU(torch.nn.Module):  # a cheaper curve
        def forward(self, x):
            return x * torch.nn.functional.hardsigmoid(x)
    m = LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1))
    m.act_fn = SiLU()
    assert fuse_between_products(m) == 0
    for act in (torch.nn.SiLU(), LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1)).act_fn):
        assert _is_silu(act)
        act.forward = lambda x: x  # (a forward of the instance's own)
        assert not _is_silu(act)
    assert fuse_between_products(torch.nn.Sequential(LlamaMLP(LlamaConfig(hidden_size=16, intermediate_size=16, num_attention_heads=1)))) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 64), (257, 896), (5, 2048), (2, 2056), (66, 4096), (3, 8192), (2, 16384), (1, 16376)])
def test_norm_against_the_single_operations(rows, hidden, dtype):
    from transformers.models.llama.modeling_llama import LlamaRMSNorm

    from anchor_attn.src.modules.model_forward import fuse_between_products
    g = torch.Generator(device="cuda").manual_seed(hidden)
    m = LlamaRMSNorm(hidden, 1e-5).to("cuda", dtype)
    with torch.no_grad():
        m.weight.copy_(1.0 + 0.2 * torch.randn(hidden, generator=g, device="cuda"))
        x = (torch.randn(1, rows, hidden, generator=g, device="cuda") * torch.linspace(0.01, 30.0, rows, device="cuda")[None, :, None]).to(dtype)
        assert fuse_between_products(m) == 1
        _close(m(x), LlamaRMSNorm.forward(m, x))
        x[0, 0, 0] = float("inf")
        assert torch.equal(m(x).isnan(), LlamaRMSNorm.forward(m, x).isnan())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1, 8), (1, 3, 24), (2, 77, 512), (1, 300, 1000)])
def test_gated_activation_against_the_single_operations(shape, dtype):
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaMLP

    from anchor_attn.src.modules.model_forward import fuse_between_products
    g = torch.Generator(device="cuda").manual_seed(shape[1])
    m = LlamaMLP(LlamaConfig(hidden_size=shape[2], intermediate_size=shape[2], num_attention_heads=1)).to("cuda", dtype)
    for name in ("gate_proj", "up_proj", "down_proj"):
        setattr(m, name, torch.nn.Identity())
    x = (8.0 * torch.randn(shape, generator=g, device="cuda")).to(dtype)
    assert fuse_between_products(m) == 1
    with torch.no_grad():
        _close(m(x), LlamaMLP.forward(m, x))


@pytest.mark.gpu
def test_calls_that_stay_with_the_single_operations(monkeypatch):
    from transformers.models.llama.modeling_llama import LlamaRMSNorm

    from anchor_attn.src.modules.model_forward import fuse_between_products
    from anchor_attn.src.ops import _hip
    m = LlamaRMSNorm(64).to("cuda", torch.bfloat16)
    fuse_between_products(m)
    monkeypatch.setattr(_hip.lib(), "aa_rms_norm", lambda *a: pytest.fail("the kernel"))
    x = torch.randn(4, 64, device="cuda", dtype=torch.bfloat16)
    y = m(x)  # gradients are enabled and the weight wants one
    y.sum().backward()
    assert m.weight.grad is not None
    with torch.no_grad():
        wide = torch.randn(4, 128, device="cuda", dtype=torch.bfloat16)
        for t in (x.float(), wide[:, ::2], wide[:, :64], torch.randn(4 * 64 + 1, device="cuda").bfloat16()[1:].view(4, 64), x[:0], x.cpu().cuda().requires_grad_(False).double()):
            assert torch.equal(m(t), LlamaRMSNorm.forward(m, t))
        with torch.autocast("cuda", dtype=torch.float16):
            assert torch.equal(m(x), LlamaRMSNorm.forward(m, x))
        assert torch.equal(torch.func.vmap(m)(x[None]), LlamaRMSNorm.forward(m, x[None]))
    monkeypatch.undo()


@pytest.mark.gpu
@pytest.mark.parametrize("act,mlps", [("silu", 2), ("gelu", 0)])
def test_patched_model_gives_the_logits_of_the_unfused_one(monkeypatch, act, mlps):
    from anchor_attn import patch_model
    from anchor_attn.src.ops import _hip
    m = patch_model(_tiny(hidden_act=act).to("cuda", torch.bfloat16), "flash")
    tokens = torch.randint(0, 100, (2, 33), device="cuda")
    calls = []
    with torch.no_grad():
        with monkeypatch.context() as watched:
            for name in ("aa_rms_norm", "aa_silu_mul"):
                inner = getattr(_hip.lib(), name)
                watched.setattr(_hip.lib(), name, lambda *a, inner=inner, name=name: (calls.append(name), inner(*a))[1])
            got = m(tokens).logits
        assert calls.count("aa_rms_norm") == 5 and calls.count("aa_silu_mul") == mlps
        for x in m.modules():
            if isinstance(x.__dict__.get("forward"), types.MethodType):
                del x.__dict__["forward"]
        for layer in m.model.layers:
            del layer.mlp.__dict__["forward"]
        want = m(tokens).logits
    assert float((got - want).norm() / want.norm()) < 1e-2
