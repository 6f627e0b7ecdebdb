"""Dense attention of any query rows over any keys (``dense_rows_attention``: ragged tails, short prompts, continued prompts)
against float64 attention, at the sizes where tiles, column blocks and key chunks end.

Bound (loose; the tight one is with the test of the probabilities' precision): probabilities rounded to the 16-bit type (unit
roundoff u) before the second product would put the sum off by at most u * max|v|, and the result is rounded once more,
u * |out|; five per cent on top covers the float32 sums and exp2."""
import pytest
import torch


def _reference(q, k, v, scale, keep):
    """float64 attention, head by head; ``keep`` [B,n_rows,n_keys] says which keys a row sees (a row without any gives 0)."""
    group = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for h in range(q.shape[1]):
        kt = k[:, h // group].double().transpose(1, 2).contiguous()
        s = torch.matmul(q[:, h].double(), kt) * scale
        p = torch.nan_to_num(s.masked_fill(~keep, float("-inf")).softmax(-1))
        out[:, h] = torch.matmul(p, v[:, h // group].double())
    return out


def _check(out, want, v, dtype):
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err, bound = (out.double() - want).abs(), 1.05 * u * (v.double().abs().max() + want.abs())
    assert bool((err <= bound).all()), float((err - bound).max())


def _qkv(batch, hq, hkv, n_rows, n_keys, d, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    # queries in the [B,N,H,D] storage a model hands over, keys and values as a cache holds them; large scores (a spread of
    # about 4) so that single keys matter
    q = (4.0 * torch.randn(batch, n_rows, hq, d, generator=g, device="cuda")).to(dtype).transpose(1, 2)
    k = torch.randn(batch, hkv, n_keys, d, generator=g, device="cuda").to(dtype)
    v = torch.randn(batch, hkv, n_keys, d, generator=g, device="cuda").to(dtype)
    return q, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,offset,d,dtype", [
    (1, 4, 2, 77, 4096, 128, torch.bfloat16),     # a tail: several chunks, the last of them ragged
    (1, 32, 8, 127, 0, 128, torch.bfloat16),      # a short prompt: fewer keys in the early column blocks
    (2, 14, 2, 65, 0, 64, torch.bfloat16),        # a group of seven: column blocks that cut a row's heads
    (1, 28, 4, 64, 12345, 128, torch.float16),    # many chunks; rows whose last chunk holds no key of theirs
    (3, 8, 8, 130, 63, 64, torch.float16),        # no groups, two column blocks, chunk and tile edges
    (1, 7, 1, 33, 0, 128, torch.bfloat16),        # fewer keys than a tile
    (1, 2, 1, 2047, 2048, 64, torch.bfloat16),    # the longest tail
    # at most 32 (row, head) columns: the decode kernel
    (1, 32, 8, 1, 33000, 128, torch.bfloat16),    # a decode step: a chunk per CU, the last tile ragged
    (3, 14, 2, 1, 0, 64, torch.float16),          # one key
    (2, 8, 1, 4, 61, 128, torch.float16),         # all 32 columns, rows that end in the same tile
    (5, 4, 4, 3, 1021, 64, torch.bfloat16),       # no groups
    (40, 16, 8, 1, 300, 128, torch.bfloat16),     # more units than CUs: one wave to a unit, written without a merge
    (40, 32, 16, 2, 190, 64, torch.float16),      # the same, two rows
    (40, 16, 8, 1, 512, 128, torch.float16),      # and its largest cache; one key more and four waves share a unit
    (40, 16, 8, 1, 513, 128, torch.float16),      # (513 + 1 keys: the last tile holds two)
    (300, 2, 1, 1, 31, 128, torch.bfloat16),      # a single full tile
    (300, 2, 1, 1, 32, 128, torch.bfloat16),      # and a second one of one key
    (2, 8, 2, 1, 639, 128, torch.bfloat16),       # the most keys of a single chunk
    (2, 8, 2, 1, 640, 64, torch.bfloat16),        # and the fewest of several
    (1, 4, 4, 9, 500, 64, torch.bfloat16),        # nine columns
    (1, 33, 1, 1, 700, 64, torch.bfloat16),       # one column too many for it
])
def test_dense_rows_against_float64(batch, hq, hkv, n_rows, offset, d, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention, dense_rows_supported
    n_keys = offset + n_rows
    q, k, v = _qkv(batch, hq, hkv, n_rows, n_keys, d, dtype, n_rows + offset)
    assert dense_rows_supported(q, k, v)
    out = torch.full((batch, n_rows, hq, d), float("nan"), dtype=dtype, device="cuda").transpose(1, 2)
    got = dense_rows_attention(q, k, v, offset, out=out)
    assert got is out
    keys, rows = torch.arange(n_keys, device="cuda"), torch.arange(n_rows, device="cuda") + offset
    keep = (keys[None, :] <= rows[:, None]).expand(batch, -1, -1)
    _check(out, _reference(q, k, v, d ** -0.5, keep), v, dtype)
    again = dense_rows_attention(q.contiguous(), k, v, offset, sm_scale=d ** -0.5)
    assert torch.equal(again, out)


SINK_CASES = [(77, 1000, 128, False), (130, 63, 64, False), (129, 0, 128, True), (65, 0, 64, True), (1, 3000, 128, False), (2, 517, 64, False),
              (1, 777, 128, True), (1, 901, 64, True)]  # rows, masked, decode and masked decode kernels


def _as_kept(p, dtype, how):
    """What is left of probabilities kept as one 16-bit number, as two, or as two formed as 2^15 p (fp16's subnormals)."""
    factor = 2.0 ** 15 if how != "plain pair" and dtype == torch.float16 else 1.0
    x = (p * factor).float()
    hi = x.to(dtype).float()
    return (hi if how == "one" else hi + (x - hi).to(dtype).float()).double() / factor


def _sink_scores(gap, dtype):
    """The number of nats in [gap, gap + 1), a multiple of 1/16, whose exp(-x) the poorer ways of keeping it hit worst."""
    x = gap + torch.arange(16, dtype=torch.float64) / 16
    p = torch.exp(-x)
    worst = (_as_kept(p, dtype, "one") / p - 1).abs()
    if dtype == torch.float16 and gap >= 10:
        worst = torch.minimum(worst, (_as_kept(p, dtype, "plain pair") / p - 1).abs())
    return float(x[worst.argmax()])


def _sink_inputs(n_rows, n_keys, d, dtype, gap, device):
    """An attention sink: key 0 with a value of 0, and all others ``gap`` nats below it with values of one sign, so that the
    output is their sum and a probability's error shows in full.  Scores are exact (one product of whole sixteenths, scale 1/8)."""
    g = torch.Generator().manual_seed(n_rows + n_keys + d)
    q, k = torch.zeros(2, 4, n_rows, d, dtype=dtype), torch.zeros(2, 2, n_keys, d, dtype=dtype)
    q[..., 0] = 8.0
    k[:, :, 1:, 0] = -_sink_scores(gap, dtype)
    v = (0.5 + torch.rand(2, 2, n_keys, d, generator=g)).to(dtype)
    v[:, :, 0] = 0.0
    keys, rows = torch.arange(n_keys), torch.arange(n_rows) + n_keys - n_rows
    return [x.to(device) for x in (q, k, v, (keys[None, :] <= rows[:, None]).expand(2, -1, -1))]


def _beyond_rounding(out, want, n_keys):
    """How far ``out`` is past the bound: half a unit of the 16-bit result, and of the result 2^-16 for a probability kept as two
    numbers (bf16: 2^-17, fp16: 2^-22) with its score's exponential, and n_keys * 2^-24 for the float32 sums."""
    digits, smallest = (8, -133) if out.dtype == torch.bfloat16 else (11, -24)
    exponent = torch.frexp(want)[1].double()
    half_unit = 0.5 * torch.exp2((exponent - digits).clamp(min=smallest))
    return (out.double() - want).abs() - half_unit - (2.0 ** -16 + n_keys * 2.0 ** -24) * want.abs()


@pytest.mark.gpu
@pytest.mark.parametrize("n_rows,offset,d,masked", SINK_CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_probabilities_keep_float32_precision(n_rows, offset, d, masked, dtype):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    n_keys = offset + n_rows
    for gap in (1, 10, 12, 14):
        q, k, v, keep = _sink_inputs(n_rows, n_keys, d, dtype, gap, "cuda")
        how = {"mask": keep[:, None]} if masked else {"causal_offset": offset}
        out = dense_rows_attention(q, k, v, sm_scale=0.125, **how)
        past = _beyond_rounding(out, _reference(q, k, v, 0.125, keep), n_keys)
        assert bool((past <= 0).all()), (gap, float(past.max()))


@pytest.mark.parametrize("n_rows,offset,d,masked", SINK_CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_poorer_probabilities_are_seen(n_rows, offset, d, masked, dtype):
    """The bound above lets two numbers pass and, on the same inputs, neither a single 16-bit number nor - fp16 - a pair whose
    small members fall among the subnormals."""
    n_keys = offset + n_rows
    for gap in (1, 10, 12, 14):
        q, k, v, keep = _sink_inputs(n_rows, n_keys, d, dtype, gap, "cpu")
        s = torch.matmul(q.double(), k.double().repeat_interleave(2, 1).transpose(2, 3)) * 0.125
        p = torch.exp(s.masked_fill(~keep[:, None], float("-inf")))
        want = _reference(q, k, v, 0.125, keep)
        fails = {}
        for how in ("one", "pair", "plain pair"):
            out = (torch.matmul(_as_kept(p, dtype, how), v.double().repeat_interleave(2, 1)) / p.sum(-1, keepdim=True)).to(dtype)
            fails[how] = bool((_beyond_rounding(out, want, n_keys) > 0).any())
        assert fails["one"] and not fails["pair"], (gap, fails)
        assert fails["plain pair"] == (dtype == torch.float16 and gap >= 10), (gap, fails)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,offset,d,masked", [
    (1, 8, 2, 77, 9000, 128, False),   # chunks, a ragged last tile
    (1, 4, 4, 150, 0, 64, False),      # one chunk
    (2, 4, 2, 129, 0, 128, True), (1, 2, 1, 5, 67000, 64, True),
    (1, 8, 2, 1, 3000, 128, False), (2, 8, 1, 4, 61, 64, False),
    (2, 8, 2, 1, 777, 64, True), (1, 4, 4, 1, 2500, 128, True),
    (40, 8, 8, 1, 70, 128, False), (80, 8, 8, 1, 27, 64, True),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_values_that_are_not_finite(batch, hq, hkv, n_rows, offset, d, masked, dtype):
    """A row that sees an infinite value gives that infinity, NaN for infinities of both signs and for NaN, in the columns of
    these values and in no other.  (A row that does not see the key gives NaN there too or what it would without: 0 times
    infinity is NaN where its tile is multiplied.)  A key that is NaN makes every row NaN that sees it."""
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    n_keys = offset + n_rows
    q, k, v = _qkv(batch, hq, hkv, n_rows, n_keys, d, dtype, 7 * n_rows + offset)
    q /= 4.0
    inf, mid, last = float("inf"), n_keys // 2, n_keys - 1
    spots = [(0, 1, inf), (mid, 3, -inf), (last, 5, inf), (mid, 40, inf), (last, 40, -inf), (mid, 41, float("nan")), (0, d - 1, -inf)]
    for key, col, x in spots:
        v[:, :, key, col] = x
    rows, keys = torch.arange(n_rows, device="cuda") + offset, torch.arange(n_keys, device="cuda")
    keep = (keys[None, :] <= rows[:, None]).expand(batch, -1, -1)
    if masked:
        keep = keep & ((keys % 5 != 3) | (keys == 0) | (keys == mid) | (keys == last))
    how = {"mask": keep[:, None]} if masked else {"causal_offset": offset}
    out = dense_rows_attention(q, k, v, **how).double()
    finite = torch.where(v.isfinite(), v, torch.zeros_like(v))
    want = _reference(q, k, finite, d ** -0.5, keep)
    special = torch.zeros(batch, n_rows, d, dtype=torch.float64, device="cuda")
    unseen = torch.zeros(batch, n_rows, d, dtype=torch.bool, device="cuda")
    for key, col, x in spots:
        special[:, :, col] += torch.where(keep[:, :, key], x, 0.0)
        unseen[:, :, col] |= ~keep[:, :, key]
    want = want + special[:, None]
    same = (out == want) | (out.isnan() & want.isnan()) | (want.isfinite() & ((out - want).abs() <= 1.05 * 2.0 ** -7 * (6 + want.abs())))
    assert bool((same | (out.isnan() & unseen[:, None])).all())
    assert bool(out[..., :1].isfinite().all()) and bool((out[:, :, -1, 1] == inf).all()) and bool((out[:, :, -1, 5] == inf).all())
    k[:, :, mid] = float("nan")
    out = dense_rows_attention(q, k, finite, **how)
    sees = keep[:, None, :, mid, None]
    assert bool((out.isnan() == sees).all())
    q[:, 1, 0] = float("nan")
    out = dense_rows_attention(q, torch.nan_to_num(k), finite, **how)
    assert bool(out[:, 1, 0].isnan().all()) and bool(out[:, 0].isfinite().all()) and bool(out[:, 1, 1:].isfinite().all())


def _mask(kind, batch, n_rows, n_keys):
    rows, keys = torch.arange(n_rows, device="cuda") + max(n_keys - n_rows, 0), torch.arange(n_keys, device="cuda")
    causal = keys[None, :] <= rows[:, None]
    if kind == "padded":  # left-padded prompts: whole tiles nobody sees, rows without any key
        pads = torch.tensor([(37 * b) % n_keys + 70 * b for b in range(batch)], device="cuda")
        return (causal[None] & (keys[None, None, :] >= pads[:, None, None]))[:, None]
    if kind == "causal":
        return causal[None, None]
    if kind == "window":  # one mask for the whole batch
        return (causal & (keys[None, :] > rows[:, None] - 100))[None, None]
    g = torch.Generator(device="cuda").manual_seed(n_keys)
    return torch.rand(batch, 1, n_rows, n_keys, generator=g, device="cuda") < 0.4


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,n_keys,d,dtype,kind", [
    (3, 8, 2, 333, 333, 128, torch.bfloat16, "padded"),
    (2, 7, 1, 129, 1025, 64, torch.float16, "random"),   # a group of seven; one key past a tile
    (2, 4, 4, 65, 4161, 128, torch.bfloat16, "padded"),  # more keys than one work-group of the mask kernel packs; chunks
    (2, 4, 2, 300, 300, 64, torch.bfloat16, "window"),
    (1, 2, 1, 5, 67000, 128, torch.bfloat16, "random"),  # more tiles than one chunk may list
    (2, 4, 2, 40, 13, 64, torch.bfloat16, "random"),     # fewer keys than a lane of the mask kernel packs
    (1, 2, 2, 150, 16, 128, torch.float16, "random"),    # and as many; more rows than it loads at once
    (2, 3, 1, 30, 1023, 64, torch.bfloat16, "padded"),   # a ragged end of one work-group's keys
    (4, 28, 4, 1, 2501, 128, torch.bfloat16, "padded"),  # a padded batch's decode step: tiles that are skipped
    (1, 2, 2, 1, 9000, 64, torch.float16, "random"),
    (40, 16, 8, 1, 70, 128, torch.float16, "padded"),    # one wave to a unit; prompts of a few keys, one of none
    (80, 8, 8, 1, 25, 64, torch.bfloat16, "random"),
    (40, 16, 8, 1, 8193, 64, torch.bfloat16, "window"),  # a second chunk of one key, since the first may hold no more
])
def test_masked_rows_against_float64(batch, hq, hkv, n_rows, n_keys, d, dtype, kind):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    q, k, v = _qkv(batch, hq, hkv, n_rows, n_keys, d, dtype, n_rows + n_keys)
    mask = _mask(kind, batch, n_rows, n_keys)
    out = dense_rows_attention(q, k, v, mask=mask)
    _check(out, _reference(q, k, v, d ** -0.5, mask[:, 0].expand(batch, -1, -1)), v, dtype)


def test_own_kernels_are_left_out_of_transformed_and_traced_calls():
    """Their work is invisible to vmap, forward-mode differentiation, tracing, dispatch and function modes."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    from anchor_attn.src.ops.anchor_attn_v4 import _called_plainly
    assert _called_plainly()
    seen = []

    def probe(x):
        seen.append(_called_plainly())
        return x * 2

    x = torch.ones(2, 3)
    torch.func.vmap(probe)(x)
    torch.func.jvp(probe, (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        probe(torch.autograd.forward_ad.make_dual(x, x))
    make_fx(probe)(x)
    torch.jit.trace(probe, (x,), check_trace=False)
    with FlopCounterMode(display=False):
        probe(x)
    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Watch():
        probe(x)
    with Watch(), torch.device("cpu"):
        probe(x)
    assert len(seen) >= 8 and not any(seen)
    with torch.device("cpu"):  # (says where new tensors go, no more)
        assert _called_plainly()
    assert _called_plainly()


def _layouts(q, k, v):
    """The same keys and values in other storage: [B,N,H,D], slices of a longer and wider cache, rows of different pitch."""
    batch, hkv, n_keys, d = k.shape
    yield "as they are", q, k, v
    yield "B,N,H,D", q, *[x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v)]
    cache = torch.full((2, batch + 1, hkv + 1, n_keys + 77, d), float("nan"), dtype=k.dtype, device=k.device)
    cache[0, 1:, 1:, 5:5 + n_keys], cache[1, 1:, 1:, 5:5 + n_keys] = k, v
    yield "a sliced cache", q, cache[0, 1:, 1:, 5:5 + n_keys], cache[1, 1:, 1:, 5:5 + n_keys]
    wide = torch.full((batch, n_keys, hkv, 3 * d), float("nan"), dtype=k.dtype, device=k.device)
    wide[..., d:2 * d] = k.transpose(1, 2)
    yield "different pitches", q, wide[..., d:2 * d].transpose(1, 2), v.transpose(1, 2).contiguous().transpose(1, 2)
    packed = torch.full((batch, q.shape[2], q.shape[1], 2 * d), float("nan"), dtype=q.dtype, device=q.device)
    packed[..., d:] = q.transpose(1, 2)
    yield "queries of a packed projection", packed[..., d:].transpose(1, 2), k, v


KERNELS = [(2, 8, 2, 77, 1300, 128, False), (1, 4, 4, 130, 130, 64, False), (2, 8, 2, 129, 1301, 64, True), (2, 6, 2, 65, 65, 128, True),
           (2, 8, 2, 1, 1301, 128, False), (40, 8, 8, 2, 90, 64, False), (2, 8, 2, 1, 1301, 64, True), (40, 8, 8, 1, 90, 128, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,n_keys,d,masked", KERNELS)
def test_storage_of_keys_values_and_queries(batch, hq, hkv, n_rows, n_keys, d, masked):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention, dense_rows_supported
    mask = _mask("padded", batch, n_rows, n_keys) if masked else None
    first = None
    for name, q, k, v in _layouts(*_qkv(batch, hq, hkv, n_rows, n_keys, d, torch.bfloat16, n_keys)):
        assert dense_rows_supported(q, k, v, mask), name
        out = dense_rows_attention(q, k, v, n_keys - n_rows, mask=mask)
        first = out if first is None else first
        assert torch.equal(out, first), name
    keep = mask[:, 0] if masked else _mask("causal", batch, n_rows, n_keys)[:, 0].expand(batch, -1, -1)
    _check(first, _reference(q, k, v, d ** -0.5, keep), v, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,n_keys,d,masked", [x for x in KERNELS if x[-1]])
def test_storage_of_masks(batch, hq, hkv, n_rows, n_keys, d, masked):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    q, k, v = _qkv(batch, hq, hkv, n_rows, n_keys, d, torch.bfloat16, n_keys)

    def strided(mask):  # rows wider than the mask, from an odd byte on; last dimension not the fastest; every second byte
        wide = torch.ones(batch, 1, n_rows, n_keys + 39, dtype=torch.bool, device="cuda")
        wide[..., 3:3 + n_keys] = mask
        return [wide[..., 3:3 + n_keys], mask.transpose(2, 3).contiguous().transpose(2, 3), torch.repeat_interleave(mask, 2, dim=3)[..., ::2]]

    mask = _mask("padded", batch, n_rows, n_keys)
    want = dense_rows_attention(q, k, v, mask=mask)
    _check(want, _reference(q, k, v, d ** -0.5, mask[:, 0]), v, torch.bfloat16)
    for m in strided(mask):
        assert torch.equal(dense_rows_attention(q, k, v, mask=m), want)
    # one row for all rows, one mask for the whole batch (strides of 0), and both
    for m in (mask[:, :, -1:].expand(-1, -1, n_rows, -1), mask[:1].expand(batch, -1, -1, -1), mask[:1], mask[:1, :, -1:].expand(batch, -1, n_rows, -1)):
        assert torch.equal(dense_rows_attention(q, k, v, mask=m), dense_rows_attention(q, k, v, mask=m.expand(batch, 1, n_rows, n_keys).clone()))


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n_rows,n_keys,d,masked", KERNELS)
def test_rows_on_other_streams_in_graphs_and_from_another_device(monkeypatch, batch, hq, hkv, n_rows, n_keys, d, masked):
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    sets = [(*_qkv(batch, hq, hkv, n_rows, n_keys, d, torch.bfloat16, seed),
             _mask(kind, batch, n_rows, n_keys).expand(batch, -1, -1, -1) if masked else None)
            for seed, kind in ((1, "padded"), (2, "random"), (3, "window"))]
    offset = n_keys - n_rows
    eager = [dense_rows_attention(q, k, v, offset, mask=m) for q, k, v, m in sets]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for (q, k, v, m), want in zip(sets, eager):
            assert torch.equal(dense_rows_attention(q, k, v, offset, mask=m), want)
    torch.cuda.synchronize()
    fixed = [x.clone() if x is not None else None for x in sets[0]]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dense_rows_attention(*fixed[:3], offset, mask=fixed[3])
    for i in (1, 2, 0, 1):  # every replay against the eager result, with eager work between
        for dst, src in zip(fixed, sets[i]):
            if dst is not None:
                dst.copy_(src)
        out.fill_(float("nan"))
        graph.replay()
        q, k, v, m = sets[(i + 1) % 3]
        assert torch.equal(dense_rows_attention(q, k, v, offset, mask=m), eager[(i + 1) % 3])
        torch.cuda.synchronize()
        assert torch.equal(out, eager[i]), i
    # with another device current than that of the tensors (a pipeline's later layers): pretended, there is one
    entered = []

    class Device(torch.cuda.device):
        def __init__(self, device):
            entered.append(device)
            super().__init__(device)

    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0 if entered else 1)
    monkeypatch.setattr(torch.cuda, "device", Device)
    q, k, v, m = sets[0]
    got = dense_rows_attention(q, k, v, offset, mask=m)
    assert entered == [q.device]
    monkeypatch.undo()
    assert torch.equal(got, eager[0])


def _spy_on_library_attention(monkeypatch):
    from anchor_attn.src.modules.llama import anchor_attention
    calls, library = [], torch.nn.functional.scaled_dot_product_attention
    monkeypatch.setattr(anchor_attention.F, "scaled_dot_product_attention", lambda *a, **kw: calls.append(a[0].dtype) or library(*a, **kw))
    return calls


def _plug(q, k, v, mask=None, scaling=0.125):
    import types

    from anchor_attn.src.modules.llama.anchor_attention import anchor_attention_forward
    module = types.SimpleNamespace(config=types.SimpleNamespace(block_size_M=128, step=16, theta=12.0))
    return anchor_attention_forward(module, q, k, v, mask, scaling=scaling)[0].transpose(1, 2)


@pytest.mark.gpu
def test_a_chosen_backend_of_library_attention_is_used(monkeypatch):
    from torch.nn.attention import SDPBackend, sdpa_kernel
    calls = _spy_on_library_attention(monkeypatch)
    q, k, v = _qkv(1, 4, 2, 5, 40, 64, torch.bfloat16, 1)
    own = _plug(q, k, v)
    assert not calls
    with sdpa_kernel(SDPBackend.MATH):
        got = _plug(q, k, v)
    assert len(calls) == 1
    _check(got, own.double(), 2 * v, torch.bfloat16)
    _plug(q, k, v)
    assert len(calls) == 1


@pytest.mark.gpu
def test_autocast_says_which_type_attention_is_computed_in(monkeypatch):
    calls = _spy_on_library_attention(monkeypatch)
    q, k, v = _qkv(1, 4, 2, 5, 40, 64, torch.bfloat16, 1)
    with torch.autocast("cuda", torch.float16):
        assert _plug(q, k, v).dtype == torch.bfloat16
    assert len(calls) == 1
    with torch.autocast("cuda", torch.bfloat16):
        _plug(q, k, v)
    assert len(calls) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("scaling", [0.0, -0.125, 1e-46, 1e-40, 1e-20])
def test_scales_beyond_the_kernels_range(scaling):
    """0 and negative ones, and one that is 0 or not normal as a float32; the last is computed by the kernels.  The result but
    for the negative one is the mean of the values that a row sees."""
    q, k, v = _qkv(2, 4, 2, 5, 40, 64, torch.bfloat16, 1)
    rows, keys = torch.arange(5, device="cuda") + 35, torch.arange(40, device="cuda")
    keep = (keys[None, :] <= rows[:, None]).expand(2, -1, -1)
    _check(_plug(q, k, v, scaling=scaling), _reference(q, k, v, scaling, keep), v, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,hq,hkv,n,library", [(65, 32, 32, 31, True), (64, 32, 32, 31, False), (65, 32, 32, 32, False), (65, 32, 16, 31, False)])
def test_many_padded_prompts_of_a_few_tokens(monkeypatch, batch, hq, hkv, n, library):
    calls = _spy_on_library_attention(monkeypatch)
    q, k, v = _qkv(batch, hq, hkv, n, n, 64, torch.bfloat16, n)
    pads, pos = torch.arange(batch, device="cuda") % (n // 2), torch.arange(n, device="cuda")
    mask = (pos[None, None, :] >= pads[:, None, None]) & (pos[None, None, :] <= pos[None, :, None])
    got = _plug(q, k, v, mask[:, None])
    assert bool(calls) == library
    rows = mask.any(-1)[:, None, :, None]  # (what a row that sees nothing gives is not looked at here)
    _check(torch.where(rows, got, 0.0), _reference(q, k, v, 0.125, mask), v, torch.bfloat16)


def test_own_kernels_are_left_out_where_the_framework_lacks_a_name(monkeypatch):
    from anchor_attn.src.ops.anchor_attn_v4 import _called_plainly
    assert _called_plainly()
    monkeypatch.delattr(torch._C, "_len_torch_dispatch_stack")
    assert not _called_plainly()


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,n_rows,n_keys", [(160, 8, 1, 300), (136, 136, 40, 40), (128, 8, 1, 300)])
def test_plug_with_an_output_too_wide_for_the_kernels(hq, hkv, n_rows, n_keys):
    """The plug's output has rows of all heads, n_heads * D elements, also where the queries' rows are D apart (every one-token
    step); beyond 16384 the kernels do not address them (the last case is the widest that they do)."""
    q, k, v = _qkv(2, hq, hkv, n_rows, n_keys, 128, torch.bfloat16, hq)
    out = _plug(q.clone(memory_format=torch.contiguous_format), k, v, scaling=128 ** -0.5)
    rows, keys = torch.arange(n_rows, device="cuda") + n_keys - n_rows, torch.arange(n_keys, device="cuda")
    keep = (keys[None, :] <= rows[:, None]).expand(2, -1, -1)
    _check(out, _reference(q, k, v, 128 ** -0.5, keep), v, torch.bfloat16)


@pytest.mark.gpu
def test_tensors_that_the_kernels_would_misread_are_refused():
    """On the host, before anything is launched: nothing behind this call looks at shapes again."""
    from anchor_attn.src.ops._hip import AnchorAttnHipError
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_attention
    q, k, v = _qkv(2, 4, 2, 3, 40, 64, torch.bfloat16, 1)
    mask = torch.ones(2, 1, 3, 40, dtype=torch.bool, device="cuda")
    dense_rows_attention(q, k, v, 37)
    for bad in [dict(V=v[:, :, :39]), dict(K=k[:1], V=v[:1]), dict(K=k.half()), dict(K=k.cpu(), V=v.cpu()), dict(Q=q.cpu()), dict(Q=q[0]),
                dict(K=k[..., :32], V=v[..., :32]), dict(out=torch.empty_like(q)[:, :, :2]), dict(out=torch.empty_like(q).half()),
                dict(out=torch.empty_like(q).cpu()), dict(mask=mask[..., :39]), dict(mask=mask[:, :, :2]), dict(mask=mask.to(torch.uint8)),
                dict(mask=mask.cpu()), dict(mask=mask.expand(2, 4, 3, 40))]:
        with pytest.raises(AnchorAttnHipError, match="unsupported tensors"):
            dense_rows_attention(**{"Q": q, "K": k, "V": v, "causal_offset": 37, **bad})


@pytest.mark.gpu
def test_calls_that_stay_with_library_attention():
    from anchor_attn.src.ops.anchor_attn_v4 import dense_rows_supported
    q, k, v = _qkv(2, 4, 2, 1, 40, 64, torch.bfloat16, 1)
    assert dense_rows_supported(q, k, v)
    assert not dense_rows_supported(q[:0], k[:0], v[:0])  # an empty batch
    many = [x[:1, :2].expand(1 << 23, -1, -1, -1) for x in (q, k, v)]
    assert not dense_rows_supported(*many)  # more work-groups than a launch takes
    assert dense_rows_supported(*[x[1:] for x in many])
    mask = torch.ones(2, 1, 1, 40, dtype=torch.bool, device="cuda")
    assert dense_rows_supported(q, k, v, mask)
    assert not dense_rows_supported(q, k, v, mask.cpu()) and not dense_rows_supported(q, k.cpu(), v.cpu())
