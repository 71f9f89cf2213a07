"""The eager calls in one step (tqamd_fastcall) against the general path behind them, over the forms that either may be given."""
import ctypes

import pytest
import torch

from test_gpu_parity import DEV, bits16, outlier_kv, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


class _Declines:
    """An extension module that takes nothing."""
    def __getattr__(self, name):
        return lambda *args: None


def _general(pkg, monkeypatch, f):
    with monkeypatch.context() as m:
        m.setattr(pkg._native, "fast", lambda: _Declines())
        return f()


def _flat(x):
    if isinstance(x, torch.Tensor):
        yield x
    elif isinstance(x, dict):
        for k in sorted(x):
            yield from _flat(x[k])
    elif isinstance(x, (list, tuple)):
        for y in x:
            yield from _flat(y)
    else:
        yield x


def _same(a, b):
    a, b = list(_flat(a)), list(_flat(b))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        if isinstance(x, torch.Tensor):
            assert x.shape == y.shape and x.dtype == y.dtype and x.device == y.device and x.requires_grad == y.requires_grad and torch.equal(x, y)
        else:
            assert x == y and type(x) is type(y)


def _forms(dim, dtype):
    x = outlier_kv((2, 3, 41, dim), seed=dim, dtype=dtype).to(DEV)
    yield "dense", x
    yield "one token", x[:, :, :1]
    yield "one row", x[:1, :1]
    yield "token slice", x[:, :, 3:35]
    yield "heads last", outlier_kv((2, 41, 3, dim), seed=dim, dtype=dtype).to(DEV).transpose(1, 2)
    yield "every other token", x[:, :, ::2]
    yield "every other head", x[:, ::2]
    yield "broadcast", x[:1].expand(3, 3, 41, dim)
    yield "wider rows", outlier_kv((2, 3, 41, 2 * dim), seed=dim, dtype=dtype).to(DEV)[..., :dim]
    yield "odd address", torch.empty(x.numel() + 1, dtype=dtype, device=DEV)[1:].view(x.shape).copy_(x)
    yield "parameter", torch.nn.Parameter(x.clone())
    yield "subclass", x.as_subclass(type("Sub", (torch.Tensor,), {}))
    yield "empty", x[:, :, :0]


@pytest.mark.parametrize("dim,bits,dtype", [(128, 4, torch.bfloat16), (128, 6, torch.float32), (64, 3, torch.float16), (80, 2, torch.bfloat16), (256, 8, torch.float16), (45, 1, torch.float32)])
def test_one_step_codec_calls_equal_the_general_path(pkg, monkeypatch, dim, bits, dtype):
    comp = pkg.MSECompressor(dim, bits, seed=3, device=DEV)
    layer = pkg.TurboQuantV3(dim, key_bits=bits, value_bits=2, residual_window=7, layer_idx=8, device=DEV)
    for name, x in _forms(dim, dtype):
        if name in ("empty", "subclass"):
            packed = comp.compress(x)
            _same([packed[k] for k in ("shape", "idx_pad")], [tuple(x.shape), -dim % (8 // bits)])
            continue
        if name == "odd address" and dim % 32 == 0:        # the kernels of these load 16 bytes at a time
            with pytest.raises((TypeError, RuntimeError)):
                comp.compress(x)
            continue
        packed = comp.compress(x)
        _same(packed, _general(pkg, monkeypatch, lambda: comp.compress(x)))
        _same(comp.decompress(packed), _general(pkg, monkeypatch, lambda: comp.decompress(packed)))
        strided = dict(packed, idx_bytes=packed["idx_bytes"].repeat(1, 1, 1, 2)[..., :packed["idx_bytes"].shape[-1]])
        _same(comp.decompress(strided), comp.decompress(packed))
        if x.shape[2] > 7:
            both = layer.compress_kv(x, x)
            _same(both, _general(pkg, monkeypatch, lambda: layer.compress_kv(x, x)))
            _same(layer.decompress_kv(*both), _general(pkg, monkeypatch, lambda: layer.decompress_kv(*both)))
            other = layer.compress_kv(x, x.contiguous().clone())       # laid out differently where x is not dense
            _same([c["compressed"] for c in other], [c["compressed"] for c in both])


@pytest.mark.parametrize("dim,dtype", [(64, torch.float16), (96, torch.bfloat16), (128, torch.bfloat16), (128, torch.float32), (256, torch.float16), (80, torch.float16)])
def test_one_step_decode_calls_equal_the_general_path(pkg, monkeypatch, dim, dtype):
    """update, append and attend over steps that fill the window, move it back and grow the store, new tokens in every layout."""
    B, H = 2, 2
    caches = [pkg.V3Cache(6, 2, residual_window=5, n_layers=40) for _ in range(2)]
    x = outlier_kv((B, H, 300, dim), seed=1, dtype=dtype).to(DEV)
    swapped = x.transpose(1, 2).contiguous().transpose(1, 2)
    q = torch.randn(B, 2 * H, 40, dim, generator=torch.Generator().manual_seed(2)).to(dtype).to(DEV)
    for c in caches:
        c.append(x[:, :, :260], x[:, :, :260], 8)
    for t in range(260, 300):
        src = (x, swapped, x.repeat(1, 1, 1, 2)[..., :dim])[t % 3]
        k, v = src[:, :, t:t + 1], src[:, :, t - 1:t]
        qt = q[:, :, t - 260:t - 259]                  # not dense: copied
        qt = qt.contiguous() if t % 2 else qt
        step = lambda c: (c.update(k, v, 8) if t % 4 else c.append(k, v, 8), c.attend(qt, 8), c.attend(qt, 8, scale=0.25))  # noqa: E731
        _same(step(caches[0]), _general(pkg, monkeypatch, lambda: step(caches[1])))
    a, b = (c._stores[8] for c in caches)
    assert (a.n_compressed, a.n_recent, a.w0, a.total_seq) == (b.n_compressed, b.n_recent, b.w0, b.total_seq)


def test_one_step_calls_refuse_what_the_general_path_refuses(pkg):
    comp = pkg.MSECompressor(128, 4, seed=3, device=DEV)
    x = torch.randn(1, 2, 5, 128, device=DEV)
    packed = comp.compress(x)
    with pytest.raises(pkg._native.TqError):
        comp.compress(x.double())
    with pytest.raises(pkg._native.TqError):
        comp.compress(x.cpu())
    comp.bits = 2                                      # the table was built for four
    with pytest.raises(pkg._native.TqError):
        comp.compress(x)
    comp.bits = 4
    with pytest.raises((RuntimeError, ValueError)):
        comp.decompress(dict(packed, shape=(1, 2, 6, 128)))
    cache = pkg.V3Cache(4, 2, residual_window=4, n_layers=40)
    y = x.bfloat16()
    cache.append(y, y, 8)
    for bad in (y[:, :, :2], y[:, :, :1].repeat(2, 1, 1, 1), torch.zeros(1, 3, 1, 128, device=DEV).bfloat16(), y[:, :, :1, :64]):
        with pytest.raises(ValueError):
            cache.attend(bad, 8)
    with pytest.raises(ValueError):
        cache.append(y[:, :1, :1], y[:, :1, :1], 8)
    assert cache._stores[8].total_seq == 5


@pytest.mark.parametrize("bits,dtype", [(3, torch.bfloat16), (5, torch.float32)])
def test_one_step_v2_calls_equal_the_general_path(pkg, monkeypatch, bits, dtype):
    """The codes bit for bit; scores of few queries come from another kernel than the general path's (bound as in
    test_v2_scores_of_few_queries_equal_those_of_many)."""
    comp = pkg.TurboQuantCompressorV2(128, bits, seed=5, device=DEV)
    for name, x in _forms(128, dtype):
        if name in ("empty", "subclass"):
            continue
        packed = comp.compress(x)
        _same(packed, _general(pkg, monkeypatch, lambda: comp.compress(x)))
        q = torch.randn(*x.shape[:2], 3, 128, device=DEV)
        for queries in (q, q.transpose(1, 2).contiguous().transpose(1, 2), q.to(torch.bfloat16), q[:, :, :1], torch.cat((q.new_zeros(1), q.reshape(-1)))[1:].view(q.shape)):
            a, b = comp.asymmetric_attention_scores(queries, packed), _general(pkg, monkeypatch, lambda: comp.asymmetric_attention_scores(queries, packed))
            assert a.shape == b.shape and a.dtype == b.dtype
            scale = queries.double().norm(dim=-1)[..., None] * x.detach().double().norm(dim=-1)[:, :, None, :]
            assert float(((a.double() - b.double()).abs() / scale.clamp_min(1e-30)).max()) < 3e-5, name


def test_allocations_that_fail_raise_torchs_own_error(pkg):
    """A caller that frees memory and tries again on torch.cuda.OutOfMemoryError gets that error from every call."""
    comp = pkg.MSECompressor(128, 1, seed=3, device=DEV)
    layer = pkg.TurboQuantV3(128, key_bits=1, value_bits=1, residual_window=0, layer_idx=8, device=DEV)
    x = torch.zeros(1, 8, 1 << 16, 128, dtype=torch.bfloat16, device=DEV)
    packed, both = comp.compress(x), layer.compress_kv(x, x)
    big = torch.zeros(1, 8, 1 << 20, 16, dtype=torch.uint8, device=DEV)
    many = {"idx_bytes": big, "vec_norms": torch.zeros(big.shape[:3], dtype=torch.float16, device=DEV), "shape": (*big.shape[:3], 128), "idx_pad": 0}
    wide = tuple(dict(b, compressed=many, shape=(1, 8, 1 << 20, 128), split_at=1 << 20) for b in both)
    torch.cuda.empty_cache()
    try:
        torch.cuda.set_per_process_memory_fraction(1e-6)        # nothing can be added to what is held
        for call in (lambda: comp.decompress(many), lambda: layer.decompress_kv(*wide)):
            with pytest.raises(torch.cuda.OutOfMemoryError):
                call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert comp.decompress(packed).shape == x.shape


def test_v2_scores_of_a_negated_view(pkg):
    """A tensor whose sign torch keeps as a flag is read with that sign."""
    comp = pkg.TurboQuantCompressorV2(128, 3, seed=5, device=DEV)
    x = outlier_kv((1, 2, 70, 128), seed=1, dtype=torch.bfloat16).to(DEV)
    packed = comp.compress(x)
    q = torch.randn(1, 2, 3, 128, generator=torch.Generator().manual_seed(2)).to(DEV)
    got, want = comp.asymmetric_attention_scores(torch._neg_view(q), packed), comp.asymmetric_attention_scores(-q, packed)
    scale = q.double().norm(dim=-1)[..., None] * x.double().norm(dim=-1)[:, :, None, :]
    assert float(((got.double() - want.double()).abs() / scale).max()) < 3e-5      # (two kernels: as in test_v2_scores_of_few_queries_equal_those_of_many)


def test_outputs_are_seen_by_those_who_listen(pkg):
    """Outputs come from the allocator directly, and through torch's dispatcher where a mode or deterministic algorithms want to see them; inference
    mode makes inference tensors either way."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    comp = pkg.MSECompressor(128, 4, seed=42, device=DEV)
    x = outlier_kv((1, 2, 70, 128), seed=3, dtype=torch.bfloat16).to(DEV)
    want = comp.compress(x)
    full = comp.decompress(want)
    with Seen() as seen:
        _same(comp.compress(x), want)
        _same(comp.decompress(want), full)
    assert sum("empty" in n for n in seen.names) >= 3
    torch.use_deterministic_algorithms(True)
    try:
        _same(comp.compress(x), want)
        _same(comp.decompress(want), full)
    finally:
        torch.use_deterministic_algorithms(False)
    with torch.inference_mode():
        got = comp.compress(x)
        out = comp.decompress(got)
    assert out.is_inference() and got["idx_bytes"].is_inference() and torch.equal(out, full)


def test_decompress_kv_with_shapes_that_are_not_the_tensors(pkg):
    """Dictionaries whose shapes are lists, or numbers of another type, restore as tuples of integers do; shapes of other tensors are not taken."""
    comp = pkg.TurboQuantV3(128, key_bits=4, value_bits=2, residual_window=16, layer_idx=8, device=DEV)
    k = outlier_kv((1, 2, 70, 128), seed=4, dtype=torch.float16).to(DEV)
    pair = comp.compress_kv(k, k)
    want = comp.decompress_kv(*pair)
    for form in (list, lambda t: tuple(float(i) for i in t), torch.Size):
        if form is list or form is torch.Size:
            other = [dict(c, shape=form(c["shape"]), compressed=dict(c["compressed"], shape=form(c["compressed"]["shape"]))) for c in pair]
            _same(comp.decompress_kv(*other), want)
        else:
            assert pkg._native.fast().restore_dicts(*[pair[i]["compressed"][n] for i in (0, 1) for n in ("idx_bytes", "vec_norms")], 54, comp.key_compressor.table(k.device),
                                                    comp.val_compressor.table(k.device), 4, 2, pair[0]["fp16"], pair[1]["fp16"], form(pair[0]["shape"]),
                                                    pair[0]["compressed"]["shape"]) is None
    assert comp._restore(*[dict(c, shape=(1, 2, 71, 128)) for c in pair]) is None


def test_outputs_are_recorded_for_the_profiler(pkg):
    """torch's profiler (and any other observer of operators) sees the outputs being made, on the calling thread and by name."""
    comp = pkg.MSECompressor(128, 4, seed=42, device=DEV)
    layer = pkg.TurboQuantV3(128, key_bits=4, value_bits=2, residual_window=16, layer_idx=8, device=DEV)
    x = outlier_kv((1, 2, 70, 128), seed=3, dtype=torch.bfloat16).to(DEV)
    want = (comp.compress(x), layer.compress_kv(x, x))
    for call, outputs in ((lambda: comp.compress(x), 2), (lambda: comp.decompress(want[0]), 1), (lambda: layer.compress_kv(x, x), 4), (lambda: layer.decompress_kv(*want[1]), 2)):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], acc_events=True) as prof:
            call()
        assert sum(e.name.startswith("aten::empty") for e in prof.events()) == outputs, [e.name for e in prof.events()]


def test_outputs_are_filled_for_deterministic_algorithms(pkg):
    """torch fills new memory while algorithms have to be deterministic: a kernel more for every output, seen as nodes of a captured graph."""
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipGraphGetNodes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_size_t)]
    comp = pkg.MSECompressor(128, 4, seed=42, device=DEV)
    x = outlier_kv((1, 2, 70, 128), seed=3, dtype=torch.bfloat16).to(DEV)
    want = comp.decompress(comp.compress(x))
    nodes, before = [], torch.are_deterministic_algorithms_enabled()
    try:
        for on in (False, True):
            torch.use_deterministic_algorithms(on)
            graph = torch.cuda.CUDAGraph(keep_graph=True)
            with torch.cuda.graph(graph):
                out = comp.decompress(comp.compress(x))
            n = ctypes.c_size_t()
            assert hip.hipGraphGetNodes(graph.raw_cuda_graph(), None, ctypes.byref(n)) == 0
            nodes.append(n.value)
            torch.use_deterministic_algorithms(before)
            for _ in range(3):
                out.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, want)
    finally:
        torch.use_deterministic_algorithms(before)
    assert nodes == [2, 2 + 3], nodes


def test_decompress_kv_with_shapes_of_floats(pkg):
    """Shapes whose numbers are floats of the same value: what shapes of integers restore, or what the general path says to them."""
    comp = pkg.TurboQuantV3(128, key_bits=4, value_bits=2, residual_window=16, layer_idx=8, device=DEV)
    k = outlier_kv((1, 2, 70, 128), seed=4, dtype=torch.float16).to(DEV)
    pair = comp.compress_kv(k, k)
    floats = lambda t: tuple(float(i) for i in t)  # noqa: E731
    other = [dict(c, shape=floats(c["shape"]), compressed=dict(c["compressed"], shape=floats(c["compressed"]["shape"]))) for c in pair]
    _same(comp.decompress_kv(*other), comp.decompress_kv(*pair))
