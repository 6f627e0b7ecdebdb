"""The two model-level patches that the reference applies next to the attention forward, for every pattern but
"default" (anchor_attn/src/modules/patch.py:146-157): logits for the last position only, and the MLP evaluated in
chunks of the sequence.  Both exist to keep a 128k-token prefill small in memory - full logits are
131072 x 128256 values (33 GB in bf16 before the float32 copy), the MLP's intermediate 131072 x 14336 x 3.

The reference replaces ``LlamaForCausalLM.forward`` and ``LlamaMLP.forward`` wholesale with edited copies of the
transformers 4.45 sources (modules/llama/causal_model_forward.py:100-126, modules/llama/llama_mlp_forward.py:46-58).
Here both are thin wrappers around whatever forward the installed transformers has, so nothing is tied to one
release: the causal-LM wrapper asks the model's own ``logits_to_keep`` mechanism for one position, the MLP wrapper
calls the module's own forward on slices.

``fuse_between_products`` runs the norms, the MLPs' activation and product and the rotary embedding of queries and keys, single operations of
the framework with a pass over memory each, as one kernel where nothing watches the single operations.  The 16-bit roundings are
theirs, but the sum of squares has another order, so a norm may differ in the last 16-bit unit (of 6001 x 2048 random elements, 4 in a
million in bf16, 27 in fp16; the activation and product and the embedding in none), and what a model computes from it by as much as
its own roundings make out.
"""
import copy
import functools
import types

import torch

from anchor_attn.src.ops import _hip
from anchor_attn.src.ops.anchor_attn_v4 import _called_plainly
from anchor_attn.src.ops.anchor_step_1_2_v2 import _stream

MLP_CHUNK_TOKENS = 32768  # the reference's chunk (llama_mlp_forward.py:52)


def keep_last_token_logits(model) -> None:
    """After this, ``model(input_ids)`` returns float32 logits of the last position only, ``[B, 1, vocab]`` - what the
    reference's patched forward returns (causal_model_forward.py:124-125: ``lm_head(hidden_states[:, -1:, :])``, then
    ``.float()``).  A caller that passes ``logits_to_keep`` itself, or ``labels`` (a loss needs every position), gets
    what it asked for."""
    inner = model.forward
    if getattr(inner, "_keeps_last_token_logits", False):
        return

    @functools.wraps(inner)
    def forward(*args, **kwargs):
        if "logits_to_keep" not in kwargs and kwargs.get("labels") is None:
            kwargs["logits_to_keep"] = 1
        out = inner(*args, **kwargs)
        logits = out.get("logits") if isinstance(out, dict) else None
        if logits is not None and logits.dtype != torch.float32:
            out["logits"] = logits.float()
        return out

    forward._keeps_last_token_logits = True
    model.forward = forward


def chunk_mlp_over_tokens(model, chunk_tokens: int = MLP_CHUNK_TOKENS) -> int:
    """Every MLP of the model (a module named ``mlp`` with gate/up/down projections) is evaluated ``chunk_tokens``
    positions at a time per batch element, into a preallocated output, as llama_mlp_forward.py:46-58 does.  Rows of
    a linear layer do not interact, so the result is that of the unchunked forward.  Returns how many modules were
    wrapped; calling it again only updates the chunk size."""
    n = 0
    for _, m in model.named_modules():
        if not all(hasattr(m, a) for a in ("gate_proj", "up_proj", "down_proj")):
            continue
        n += 1
        m._mlp_chunk_tokens = int(chunk_tokens)
        if getattr(m.forward, "_chunks_tokens", False):
            continue
        inner = m.forward

        def forward(x, _inner=inner, _m=m):
            chunk = _m._mlp_chunk_tokens
            if chunk <= 0 or x.dim() != 3 or x.shape[1] <= chunk:
                return _inner(x)
            out = torch.empty_like(x)
            for b in range(x.shape[0]):
                for i in range(0, x.shape[1], chunk):
                    out[b:b + 1, i:i + chunk] = _inner(x[b:b + 1, i:i + chunk])
            return out

        forward._chunks_tokens = True
        m.forward = forward
    return n


def _kernel_takes(*tensors) -> bool:
    """Plain 16-bit tensors on one GPU, contiguous on 16-byte boundaries, in an eager call that nothing differentiates or watches.
    (What a tracer puts in the place of a tensor is not asked for its sizes: the answer would end the trace or tie it to them.)"""
    if not (all(type(t) in (torch.Tensor, torch.nn.Parameter) for t in tensors) and _called_plainly()):
        return False
    first = tensors[0]
    if not first.is_cuda or first.dtype not in (torch.bfloat16, torch.float16) or torch.is_autocast_enabled("cuda"):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if t.dtype != first.dtype or t.device != first.device or not t.is_contiguous():
            return False
        if (grad and t.requires_grad) or not 0 < t.numel() < 1 << 35 or t.data_ptr() & 15:
            return False
    return True


def _launch(fn, device, *args) -> None:
    if device.index == torch.cuda.current_device():
        _hip.check(fn(*args, _stream()))
    else:
        with torch.cuda.device(device):
            _hip.check(fn(*args, _stream()))


def _rms_norm_forward(own):
    """A norm's forward in the place of its class's, ``own``.  (One that a program gives the class later is used instead; and by its
    name the bound method is pickled as the class's.)"""
    def forward(self, hidden_states):
        if type(self).forward is not own or not _kernel_takes(hidden_states, self.weight):
            return type(self).forward(self, hidden_states)
        weight, n = self.weight, self.weight.numel()
        if not (hidden_states.shape[-1:] == weight.shape and n % 8 == 0 and n <= 16384 and hidden_states.numel() // n < 1 << 24):
            return own(self, hidden_states)
        out = torch.empty_like(hidden_states)
        _launch(_hip.lib().aa_rms_norm, out.device, hidden_states.data_ptr(), weight.data_ptr(), out.data_ptr(), out.numel() // n, n,
                float(self.variance_epsilon), _hip.dtype_code(out))
        return out

    return forward


def _is_silu(act) -> bool:
    """The framework's or transformers' SiLU module (another class of that name may compute something else), and nothing that sees it called."""
    kind = type(act)
    return ((kind is torch.nn.SiLU or (kind.__module__, kind.__name__) == ("transformers.activations", "SiLUActivation"))
            and not (act._forward_hooks or act._forward_pre_hooks or "forward" in act.__dict__)
            and not (torch.nn.modules.module._global_forward_hooks or torch.nn.modules.module._global_forward_pre_hooks))


def _gated_mlp_forward(own, own_act):
    """An MLP's forward in the place of its class's, ``own``, with an activation whose class has the forward ``own_act``."""
    def forward(self, x):
        act = self.act_fn
        if not (type(self).forward is own and _kernel_takes(x) and _is_silu(act) and type(act).forward is own_act):
            return type(self).forward(self, x)
        gate, up = self.gate_proj(x), self.up_proj(x)
        if gate.shape == up.shape and gate.numel() % 8 == 0 and _kernel_takes(gate, up):
            h = torch.empty_like(gate)
            _launch(_hip.lib().aa_silu_mul, h.device, gate.data_ptr(), up.data_ptr(), h.data_ptr(), h.numel(), _hip.dtype_code(h))
        else:
            h = act(gate) * up
        return self.down_proj(h)

    return forward


_ROPE = "apply_rotary_pos_emb"


def _rope_tensors(q, k, cos, sin):
    """What the kernel is given of these tensors, with new ones for its results (the keys' contiguous, as a cache lays them out); None where
    it does not take them."""
    tensors = (q, k, cos, sin)
    if not (all(type(t) is torch.Tensor for t in tensors) and _called_plainly()):
        return None
    if not q.is_cuda or q.dtype not in (torch.bfloat16, torch.float16) or torch.is_autocast_enabled("cuda"):
        return None
    if not (q.dim() == k.dim() == 4 and cos.dim() == sin.dim() == 3 and cos.shape == sin.shape):
        return None
    (B, H, N, D), kv_heads = q.shape, k.shape[1]
    if not (k.shape == (B, kv_heads, N, D) and cos.shape in ((B, N, D), (1, N, D)) and D % 16 == 0 and D <= 256 and 0 < q.numel() < 1 << 35 and 0 < k.numel() < 1 << 35):
        return None
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return None
    if any(t.dtype != q.dtype or t.device != q.device or t.data_ptr() & 15 for t in tensors) or not (cos.is_contiguous() and sin.is_contiguous()):
        return None
    outs = torch.empty_like(q), torch.empty(k.shape, dtype=k.dtype, device=k.device)
    for t in (q, k, *outs):
        sb, sh, sn, sd = t.stride()
        if sd != 1 or (sb | sh | sn) & 7 or not D <= sn <= 1 << 14 or N > 1 << 20 or N * sn * 2 >= 1 << 32:
            return None
    return outs, (*_hip.t3(q), *_hip.t3(k), *_hip.t3(outs[0]), *_hip.t3(outs[1]), cos.data_ptr(), sin.data_ptr(), N * D if cos.shape[0] > 1 else 0,
                  B, H, kv_heads, N, D, _hip.dtype_code(q))


class _Names(dict):
    """The global names of a function, as they are at any time, but for one."""

    def __init__(self, names, rope):
        super().__init__({_ROPE: rope, "__builtins__": names["__builtins__"]})
        self.names = names

    def __missing__(self, name):
        return self.names[name]


class _Bound:
    """A forward bound to its module, which copies and pickles as a bound method does, the copy's and by its name, and names its module and
    function as one.  (It is none: those mark the modules whose kernels take over the whole forward.)"""

    __self__ = property(lambda self: self.module)
    __func__ = property(lambda self: self.forward)

    def __init__(self, module, forward):
        self.module, self.forward = module, forward
        functools.update_wrapper(self, types.MethodType(type(module).forward, module))

    def __call__(self, *args, **kwargs):
        return self.forward(self.module, *args, **kwargs)

    def __deepcopy__(self, memo):
        return _Bound(copy.deepcopy(self.module, memo), self.forward)

    def __reduce__(self):
        return getattr, (self.module, "forward")


def _attention_forward(own):
    """An attention's forward in the place of its class's, ``own``: the same code, in which one name, the rotary embedding of its
    queries and keys, means the kernel where that takes the tensors.  (Of a forward or an embedding that a program puts in their
    places later, that is used.)"""
    single_operations = own.__globals__[_ROPE]

    def rope(*args, **kwargs):
        taken = _rope_tensors(*args) if len(args) == 4 and not kwargs else None
        if taken is None:
            return single_operations(*args, **kwargs)
        outs, numbers = taken
        _launch(_hip.lib().aa_rope, outs[0].device, *numbers)
        return outs

    fused = types.FunctionType(own.__code__, _Names(own.__globals__, rope), own.__name__, own.__defaults__, own.__closure__)
    fused.__kwdefaults__ = own.__kwdefaults__

    def forward(self, *args, **kwargs):
        if not _called_plainly() or type(self).forward is not own or own.__globals__.get(_ROPE) is not single_operations:
            return type(self).forward(self, *args, **kwargs)
        return fused(self, *args, **kwargs)

    return forward


def _rotates(own) -> bool:
    """Whether an attention's forward is a plain function that embeds by that name, bit for bit as the kernel does on a few numbers."""
    if type(own) is not types.FunctionType or _ROPE not in own.__code__.co_names or type(own.__globals__.get(_ROPE)) is not types.FunctionType:
        return False
    x = torch.linspace(-3.0, 3.0, 2 * 3 * 2 * 16, dtype=torch.float32, device="cpu").reshape(2, 3, 2, 16).bfloat16()
    cos, sin = (x[:, 0] * 0.3).cos(), (x[:, 1] * 0.7).sin()  # (halves that differ)
    want = [t * cos[:, None] + torch.cat((-t[..., 8:], t[..., :8]), -1) * sin[:, None] for t in (x, x[:, :1] + 1)]
    try:
        got = own.__globals__[_ROPE](x, x[:, :1] + 1, cos, sin)
        return len(got) == 2 and all(torch.equal(a, b) for a, b in zip(got, want))
    except Exception:  # noqa: BLE001 - one that works otherwise
        return False


def _computes(cls, stub, x, want) -> bool:
    """Whether the class's own forward does what the kernel would take over, bit for bit on a few numbers."""
    try:
        return torch.equal(cls.forward(stub, x.clone()), want)  # (an activation may work in place)
    except Exception:  # noqa: BLE001 - a class that works otherwise
        return False


def fuse_between_products(model) -> int:
    """RMS norms, gated MLPs and attentions of the model's family whose classes compute what the kernels do, and whose instances have no
    ``forward`` of their own, get one that uses the kernels.  Returns how many; calling it again changes nothing."""
    x = torch.linspace(-3.0, 3.0, 32, dtype=torch.float32, device="cpu").reshape(2, 16).bfloat16()
    norm = types.SimpleNamespace(weight=x[0] + 1.0, variance_epsilon=1e-3)
    scaled = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-3)
    normed = norm.weight * scaled.to(x.dtype)
    mlp = types.SimpleNamespace(gate_proj=lambda t: t * 3, up_proj=lambda t: t + 1, down_proj=lambda t: t * 0.5, act_fn=torch.nn.functional.silu)
    silu = torch.nn.functional.silu(x)
    gated = torch.nn.functional.silu(x * 3) * (x + 1) * 0.5
    n = 0
    with torch.no_grad():
        for m in model.modules():
            name, fused, act = type(m).__name__, None, getattr(m, "act_fn", None)
            if "forward" in m.__dict__:
                continue
            if name in ("LlamaRMSNorm", "Qwen2RMSNorm") and _computes(type(m), norm, x, normed):
                fused = _rms_norm_forward(type(m).forward)
            elif (name in ("LlamaMLP", "Qwen2MLP") and _is_silu(act) and _computes(type(act), act, x, silu)
                  and _computes(type(m), mlp, x, gated)):
                fused = _gated_mlp_forward(type(m).forward, type(act).forward)
            elif name in ("LlamaAttention", "Qwen2Attention") and _rotates(type(m).forward):
                m.forward = _Bound(m, _attention_forward(type(m).forward))
                n += 1
            if fused is not None:
                m.forward = types.MethodType(fused, m)
                n += 1
    return n
