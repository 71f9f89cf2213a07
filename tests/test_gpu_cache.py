"""GPU tests of the append-in-place packed store (packed_row_stride of the C ABI) and of the
streaming cache built on it, against the dense kernels, the CPU oracle and the bookkeeping of
the reference's generation-time cache (generation_test_v2.py:80-165)."""
import copy

import ctypes

import numpy as np
import pytest
import torch

from test_gpu_parity import DEV, bits16, outlier_kv, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("these tests need a HIP device; there is no CPU fallback to test")


@pytest.mark.parametrize("bits", [2, 4, 8])
def test_append_to_packed_store_equals_dense(pkg, bits):
    """Chunks compressed into consecutive token slots of a [B,H,capacity,G] store give the bytes of
    one dense call over the concatenated tokens; de-quantising a slice of the store gives the dense
    result; slots outside the written range stay untouched."""
    B, H, cap, D = 2, 3, 192, 128
    comp = pkg.MSECompressor(D, bits, seed=5, device=DEV)
    G = D // (8 // bits)
    x = outlier_kv((B, H, 150, D), seed=bits, dtype=torch.bfloat16).to(DEV)
    store = torch.full((B, H, cap, G), 0xEE, dtype=torch.uint8, device=DEV)
    norms = torch.full((B, H, cap), -7.0, dtype=torch.float16, device=DEV)
    pos = 3                                   # start away from slot 0: pointers are advanced, not rows
    for lo, hi in ((0, 70), (70, 71), (71, 150)):          # many tokens, a single one, a ragged rest
        n = hi - lo
        comp.compress_into(x[:, :, lo:hi], store[:, :, pos:pos + n], norms[:, :, pos:pos + n])
        pos += n
    dense = comp.compress(x)
    assert torch.equal(store[:, :, 3:153], dense["idx_bytes"])
    assert torch.equal(norms[:, :, 3:153], dense["vec_norms"])
    assert bool((store[:, :, :3] == 0xEE).all()) and bool((store[:, :, 153:] == 0xEE).all())
    assert bool((norms[:, :, :3] == -7).all()) and bool((norms[:, :, 153:] == -7).all())
    want = torch.empty(B, H, 150, D, dtype=torch.bfloat16, device=DEV)
    comp.decompress_into(dense, want)
    out = torch.zeros(B, H, 160, D, dtype=torch.bfloat16, device=DEV)
    comp.decompress_packed(store[:, :, 3:153], norms[:, :, 3:153], out[:, :, :150])
    assert torch.equal(out[:, :, :150], want) and not bool(out[:, :, 150:].any())
    # one row, one token: the smallest append
    one = torch.zeros(1, 1, 8, G, dtype=torch.uint8, device=DEV)
    onen = torch.zeros(1, 1, 8, dtype=torch.float16, device=DEV)
    comp.compress_into(x[:1, :1, 4:5], one[:, :, 6:7], onen[:, :, 6:7])
    assert torch.equal(one[0, 0, 6], dense["idx_bytes"][0, 0, 4]) and not bool(one[0, 0, :6].any())


def test_batched_jobs_with_packed_row_stride(pkg):
    native = pkg._native
    comps = [pkg.MSECompressor(128, 4, seed=100 + l, device=DEV) for l in range(3)]
    xs = [outlier_kv((2, 2, 90 + l, 128), seed=40 + l, dtype=torch.float16).to(DEV) for l in range(3)]
    stores = [torch.zeros(2, 2, 128, 64, dtype=torch.uint8, device=DEV) for _ in range(3)]
    norms = [torch.zeros(2, 2, 128, dtype=torch.float16, device=DEV) for _ in range(3)]
    jobs = [{"states": x, "idx_bytes": s[:, :, 10:10 + x.shape[2]], "vec_norms": n[:, :, 10:10 + x.shape[2]],
             "table": c.table(), "bits": 4} for x, s, n, c in zip(xs, stores, norms, comps)]
    native.JobList(jobs, DEV).compress()
    torch.cuda.synchronize()
    for x, s, n, c in zip(xs, stores, norms, comps):
        d = c.compress(x)
        assert torch.equal(s[:, :, 10:10 + x.shape[2]], d["idx_bytes"]) and torch.equal(n[:, :, 10:10 + x.shape[2]], d["vec_norms"])
        assert not bool(s[:, :, :10].any()) and not bool(s[:, :, 10 + x.shape[2]:].any())
    outs = [torch.zeros_like(x) for x in xs]
    native.JobList([dict(j, states=o) for j, o in zip(jobs, outs)], DEV).decompress()
    torch.cuda.synchronize()
    for x, o, c in zip(xs, outs, comps):
        want = torch.empty_like(x)
        c.decompress_into(c.compress(x), want)
        assert torch.equal(o, want)


@pytest.mark.parametrize("rw", [0, 16, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_v3cache_stream_equals_one_shot_codec(pkg, oracle, rw, dtype):
    """Prefill, single-token decode steps and a multi-token step through V3Cache.update.  After every
    call: length and bookkeeping as the reference's cache computes them, the uncompressed tail
    bit-identical to the incoming tokens, the de-quantised part bit-identical to one dense
    compress + decompress over the same tokens (codes do not depend on the chunking), and within
    tolerance of the CPU oracle's decode of the stored bytes."""
    B, H, D, L = 2, 2, 128, 2
    cache = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=rw, protected_layers=0, n_layers=L)
    steps = [150, 1, 1, 1, 7, 1, 40, 1]
    keys = [outlier_kv((B, H, sum(steps), D), seed=300 + l, dtype=dtype).to(DEV) for l in range(L)]
    vals = [outlier_kv((B, H, sum(steps), D), seed=400 + l, dtype=dtype).to(DEV) for l in range(L)]
    seen = 0
    for n_new in steps:
        for l in range(L):
            fk, fv = cache.update(keys[l][:, :, seen:seen + n_new], vals[l][:, :, seen:seen + n_new], l)
            total = seen + n_new
            n_c = total if rw == 0 else max(total - rw, 0)
            assert fk.shape == (B, H, total, D) and fv.shape == fk.shape and fk.dtype == dtype
            assert cache.get_seq_length(l) == total
            assert torch.equal(fk[:, :, n_c:], keys[l][:, :, n_c:total]), (rw, total)
            assert torch.equal(fv[:, :, n_c:], vals[l][:, :, n_c:total])
            if n_c:
                tq = cache._get_compressor(l, D, DEV)
                assert tq.residual_window == 0
                ck, cv = tq.compress_kv(keys[l][:, :, :n_c], vals[l][:, :, :n_c])
                dk, dv = tq.decompress_kv(ck, cv)
                assert torch.equal(fk[:, :, :n_c], dk) and torch.equal(fv[:, :, :n_c], dv), (rw, total)
        seen += n_new
    total = sum(steps)
    n_c = total if rw == 0 else total - rw
    assert cache.get_compression_info() == f"{n_c} compressed, {total - n_c} fp16, {total} total"
    # stored bytes decoded by the oracle
    st = cache._stores[1]
    tq = cache._get_compressor(1, D, DEV)
    for comp, idx, nrm, full in ((tq.key_compressor, st.k_idx, st.k_nrm, fk), (tq.val_compressor, st.v_idx, st.v_nrm, fv)):
        orc = oracle.COracle(comp.Pi.cpu().numpy(), comp.centroids.cpu().numpy(), comp.bits, True)
        packed = idx[:, :, :n_c].contiguous().cpu().numpy().reshape(-1, idx.shape[-1])
        ref = orc.decompress(packed, bits16(nrm[:, :, :n_c].contiguous()).reshape(-1))
        err, _ = rel_l2(full[:, :, :n_c].float().cpu().numpy().reshape(-1, D), ref)
        assert err < 5e-3, err               # bf16 / fp16 rounding of the output on top of the 1e-3 bar
    assert cache.stored_bytes() == L * B * H * (n_c * (64 + 32 + 4) + 2 * (total - n_c) * D * 2)


def test_config5_shape_decode_streaming(pkg, oracle):
    """The decode-streaming workload at its real shape, one layer: 64 sequences x 8 KV heads, 16 384 compressed +
    128 window tokens prefilled (bf16, K4/V2, residual_window=128), then three single-token decode steps.
    Everything is checked on all 512 rows against the one-shot codec on the device (bit for bit), and on a sample
    of rows (first and last sequence) against the CPU oracle: stored codes and norms, the de-quantised history
    `update` returns, and `attend` against float64 attention over the oracle-decoded cache."""
    B, H, D, S0, rw, G = 64, 8, 128, 16384, 128, 4
    from test_gpu_parity import _device_kv, check_codes, check_norms
    cache = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=rw, protected_layers=0, n_layers=32, capacity=S0 + 16)
    total = S0 + rw + 3
    keys = _device_kv((B, H, total, D), 5_000_000, torch.bfloat16)
    vals = _device_kv((B, H, total, D), 5_000_001, torch.bfloat16)
    layer = 0
    fk, fv = cache.update(keys[:, :, :S0 + rw], vals[:, :, :S0 + rw], layer)
    assert fk.shape == (B, H, S0 + rw, D) and cache.get_compression_info() == f"{S0} compressed, {rw} fp16, {S0 + rw} total"
    del fk, fv
    for t in range(S0 + rw, total):
        fk, fv = cache.update(keys[:, :, t:t + 1], vals[:, :, t:t + 1], layer)
        if t + 1 < total:
            del fk, fv
    n_c = total - rw
    st = cache._stores[layer]
    assert cache.get_seq_length(layer) == total and st.n_compressed == n_c == S0 + 3
    assert fk.shape == (B, H, total, D) and fk.dtype == torch.bfloat16
    # all rows: the window verbatim, the history equal to the one-shot codec over the same tokens
    assert torch.equal(fk[:, :, n_c:], keys[:, :, n_c:]) and torch.equal(fv[:, :, n_c:], vals[:, :, n_c:])
    tq = cache._get_compressor(layer, D, DEV)
    ck, cv = tq.compress_kv(keys[:, :, :n_c], vals[:, :, :n_c])
    assert torch.equal(st.k_idx[:, :, :n_c], ck["compressed"]["idx_bytes"]) and torch.equal(st.k_nrm[:, :, :n_c], ck["compressed"]["vec_norms"])
    assert torch.equal(st.v_idx[:, :, :n_c], cv["compressed"]["idx_bytes"]) and torch.equal(st.v_nrm[:, :, :n_c], cv["compressed"]["vec_norms"])
    dk, dv = tq.decompress_kv(ck, cv)
    assert torch.equal(fk[:, :, :n_c], dk) and torch.equal(fv[:, :, :n_c], dv)
    del dk, dv, ck, cv
    # the query step on all rows; sampled sequences against the oracle
    q = _device_kv((B, H * G, 1, D), 5_000_003, torch.bfloat16) * 0.05
    out = cache.attend(q, layer)
    assert out.shape == q.shape and bool(torch.isfinite(out.float()).all())
    for b in (0, B - 1):
        dec = {}
        for comp, idx, nrm, x, full, name in ((tq.key_compressor, st.k_idx, st.k_nrm, keys, fk, "K4"),
                                              (tq.val_compressor, st.v_idx, st.v_nrm, vals, fv, "V2")):
            Pi, cent = comp.Pi.cpu().numpy(), comp.centroids.cpu().numpy()
            flat = x[b, :, :n_c].float().cpu().numpy().reshape(-1, D)
            ref, _ = check_codes(oracle, idx[b, :, :n_c].contiguous().cpu().numpy(), flat, Pi, cent, comp.bits, f"config 5 seq {b} {name}")
            check_norms(oracle, bits16(nrm[b, :, :n_c].contiguous()), ref["vec_norms"], f"config 5 seq {b} {name}")
            orc = oracle.COracle(Pi, cent, comp.bits, True)
            stored = orc.decompress(idx[b, :, :n_c].contiguous().cpu().numpy().reshape(-1, idx.shape[-1]),
                                    bits16(nrm[b, :, :n_c].contiguous()).reshape(-1))
            err, _ = rel_l2(full[b, :, :n_c].float().cpu().numpy().reshape(-1, D), stored)
            assert err < 4e-3, (name, err)                 # bf16 output rounding on top of the 1e-3 bar
            dec[name] = np.concatenate([stored.reshape(H, n_c, D), x[b, :, n_c:].float().cpu().numpy()], axis=1)
        _, want = oracle.attention_decode(q[b:b + 1, :, 0].float().cpu().numpy(), dec["K4"][None], dec["V2"][None], D ** -0.5)
        got = out[b, :, 0].float().cpu().numpy()
        err = float(np.linalg.norm(got - want[0]) / np.linalg.norm(want[0]))
        print(f"[config 5] seq {b}: attend vs float64 attention over the oracle-decoded cache: {err:.2e}")
        assert err < 6e-3, err                             # bf16 output rounding of `attend`
    assert cache.stored_bytes() == B * H * (n_c * (64 + 32 + 4) + 2 * rw * D * 2)


def test_v3cache_grows_and_protects_layers(pkg):
    """Capacity doubles without losing history; protected layers store 8-bit codes for K and V."""
    cache = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=8, protected_layers=1, n_layers=3)
    x = outlier_kv((1, 2, 700, 128), seed=9, dtype=torch.bfloat16).to(DEV)
    out = None
    for lo in range(0, 700, 100):
        for l in range(3):
            out = cache.update(x[:, :, lo:lo + 100], x[:, :, lo:lo + 100], l)
    assert cache._stores[0].k_idx.shape[-1] == 128 and cache._stores[0].v_idx.shape[-1] == 128
    assert cache._stores[1].k_idx.shape[-1] == 64 and cache._stores[1].v_idx.shape[-1] == 32
    assert cache._stores[2].k_idx.shape[-1] == 128
    assert cache._stores[1].capacity >= 692 and cache._stores[1].n_compressed == 692
    tq = cache._get_compressor(2, 128, DEV)
    ck, cv = tq.compress_kv(x[:, :, :692], x[:, :, :692])
    dk, _ = tq.decompress_kv(ck, cv)
    assert torch.equal(out[0][:, :, :692], dk) and torch.equal(out[0][:, :, 692:], x[:, :, 692:])
    with pytest.raises(ValueError):
        cache.update(x[:, :1, :1], x[:, :1, :1], 0)          # head count changed


def test_hf_dynamic_cache_subclass(pkg):
    """The transformers-facing subclass keeps DynamicCache's interface alive around update()."""
    transformers = pytest.importorskip("transformers")
    cls = pkg.hf_cache_class()
    cache = cls(key_bits=4, value_bits=2, residual_window=4, n_layers=2)
    assert isinstance(cache, transformers.DynamicCache) and isinstance(cache, pkg.V3Cache)
    x = outlier_kv((1, 2, 12, 128), seed=1, dtype=torch.float16).to(DEV)
    for l in range(2):
        k, v = cache.update(x, x, l)
        assert k.shape == (1, 2, 12, 128)
    assert cache.get_seq_length() == 12 and cache.get_seq_length(1) == 12
    assert cache.get_compression_info() == "8 compressed, 4 fp16, 12 total"


# ---------------------------------------------------------------------------------------------
# attention straight from the packed store
# ---------------------------------------------------------------------------------------------
def _oracle_decode(oracle, comp, idx, nrm, shape):
    orc = oracle.COracle(comp.Pi.cpu().numpy(), comp.centroids.cpu().numpy(), comp.bits, True)
    flat = orc.decompress(idx.contiguous().cpu().numpy().reshape(-1, idx.shape[-1]), bits16(nrm.contiguous()).reshape(-1))
    return flat.reshape(shape)


@pytest.mark.parametrize("bits,group,S", [(4, 4, 1000), (2, 8, 333), (8, 1, 64), (3, 2, 31), (1, 16, 257), (6, 32, 96)])
def test_packed_scores_against_oracle(pkg, oracle, bits, group, S):
    """scale * q . k_hat from packed keys (query rotated once, codes never expanded to vectors) equals the
    float64 scores over the oracle's de-quantised keys; tolerance: the fp16 rounding of the centroid
    table the decode kernels share (2^-11 relative per coordinate), i.e. 1e-3 of scale*|q|*|k|."""
    B, H, D = 2, 3, 128
    comp = pkg.MSECompressor(D, bits, seed=77 + bits, device=DEV)
    keys = outlier_kv((B, H, S, D), seed=bits * 10 + group, dtype=torch.bfloat16).to(DEV)
    store = torch.zeros(B, H, S + 40, D // (8 // bits), dtype=torch.uint8, device=DEV)
    norms = torch.zeros(B, H, S + 40, dtype=torch.float16, device=DEV)
    comp.compress_into(keys, store[:, :, 7:7 + S], norms[:, :, 7:7 + S])
    g = torch.Generator(device="cpu")
    g.manual_seed(group)
    q = (torch.randn(B, H * group, 1, D, generator=g) * torch.exp(torch.randn(B, H * group, 1, 1, generator=g))).to(DEV)
    scale = D ** -0.5
    out = torch.full((B, H * group, S + 5), 123.0, dtype=torch.float32, device=DEV)
    got = comp.packed_scores(store[:, :, 7:7 + S], norms[:, :, 7:7 + S], q, scale, out=out[:, :, :S])
    assert got.data_ptr() == out.data_ptr() and bool((out[:, :, S:] == 123.0).all())
    k_hat = _oracle_decode(oracle, comp, store[:, :, 7:7 + S], norms[:, :, 7:7 + S], (B, H, S, D))
    ref, _ = oracle.attention_decode(q.squeeze(2).cpu().numpy(), k_hat, k_hat, scale)
    bound = scale * np.linalg.norm(q.squeeze(2).cpu().numpy().astype(np.float64), axis=-1)[:, :, None] \
        * np.repeat(np.linalg.norm(k_hat.astype(np.float64), axis=-1), group, axis=1)
    err = np.abs(got.cpu().numpy() - ref) / np.maximum(bound, 1e-30)
    print(f"[scores] b{bits} G{group} S{S}: max error {err.max():.2e} of scale*|q|*|k|")
    assert err.max() < 1e-3
    # and the definition the reference uses: scores over the product's own de-quantised keys
    deq = torch.empty(B, H, S, D, dtype=torch.float32, device=DEV)
    comp.decompress_packed(store[:, :, 7:7 + S], norms[:, :, 7:7 + S], deq)
    same = pkg.attention_scores(q, deq.repeat_interleave(group, dim=1)) * scale
    assert float((got - same).abs().max()) < 1e-3 * float(bound.max())
    dense = comp.packed_scores(store[:, :, 7:7 + S].contiguous(), norms[:, :, 7:7 + S].contiguous(), q.squeeze(2), scale)
    assert torch.equal(dense, got)


@pytest.mark.parametrize("bits,group,S", [(2, 4, 1000), (4, 8, 333), (8, 1, 64), (3, 2, 31), (1, 16, 257)])
def test_packed_weighted_values_against_oracle(pkg, oracle, bits, group, S):
    B, H, D = 2, 3, 128
    comp = pkg.MSECompressor(D, bits, seed=177 + bits, device=DEV)
    vals = outlier_kv((B, H, S, D), seed=bits * 10 + group + 1, dtype=torch.float16).to(DEV)
    store = torch.zeros(B, H, S + 9, D // (8 // bits), dtype=torch.uint8, device=DEV)
    norms = torch.zeros(B, H, S + 9, dtype=torch.float16, device=DEV)
    comp.compress_into(vals, store[:, :, 2:2 + S], norms[:, :, 2:2 + S])
    g = torch.Generator(device="cpu")
    g.manual_seed(S)
    w_full = torch.softmax(3 * torch.randn(B, H * group, S + 16, generator=g), dim=-1).to(DEV)
    w = w_full[:, :, :S]                                         # a strided slice, as the cache passes it
    got = comp.packed_weighted_values(store[:, :, 2:2 + S], norms[:, :, 2:2 + S], w)
    v_hat = _oracle_decode(oracle, comp, store[:, :, 2:2 + S], norms[:, :, 2:2 + S], (B, H, S, D)).astype(np.float64)
    ref = np.einsum("bhgs,bhsd->bhgd", w.cpu().numpy().astype(np.float64).reshape(B, H, group, S), v_hat).reshape(B, H * group, D)
    err = np.linalg.norm(got.cpu().numpy() - ref) / np.linalg.norm(ref)
    print(f"[weighted values] b{bits} G{group} S{S}: relative L2 error {err:.2e}")
    assert got.shape == (B, H * group, D) and err < 1e-3
    again = comp.packed_weighted_values(store[:, :, 2:2 + S], norms[:, :, 2:2 + S], w)
    assert torch.equal(again, got)                               # fixed summation order


@pytest.mark.parametrize("rw,dtype,D", [(128, torch.bfloat16, 128), (0, torch.float16, 128), (16, torch.bfloat16, 128),
                                         (16, torch.bfloat16, 64), (128, torch.float16, 256), (0, torch.bfloat16, 96),
                                         (16, torch.float16, 80), (8, torch.bfloat16, 45)])
def test_v3cache_attend_equals_attention_over_the_cache(pkg, oracle, rw, dtype, D):
    """append() leaves the cache in the state update() leaves it in, and attend() equals one-query
    attention over (oracle-decoded packed tokens ++ window) in float64; it also agrees with attention
    over the bf16 / fp16 tensors update() hands to the model within their rounding.  128-wide heads are read
    straight from the packed codes; other head dimensions are de-quantised by the codec kernels first."""
    B, H, G, L = 2, 2, 4, 2
    a = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=rw, n_layers=L)
    b = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=rw, n_layers=L)
    steps = [300, 1, 1, 5, 1] + [1] * 20
    total = sum(steps)
    keys = [outlier_kv((B, H, total, D), seed=600 + l, dtype=dtype).to(DEV) for l in range(L)]
    vals = [outlier_kv((B, H, total, D), seed=700 + l, dtype=dtype).to(DEV) for l in range(L)]
    g = torch.Generator(device="cpu")
    g.manual_seed(9)
    seen = 0
    for i, n_new in enumerate(steps):
        for l in range(L):
            fk, fv = a.update(keys[l][:, :, seen:seen + n_new], vals[l][:, :, seen:seen + n_new], l)
            b.append(keys[l][:, :, seen:seen + n_new], vals[l][:, :, seen:seen + n_new], l)
            sa, sb = a._stores[l], b._stores[l]
            assert (sa.n_compressed, sa.n_recent, sa.total_seq) == (sb.n_compressed, sb.n_recent, sb.total_seq)
            if i in (0, 3, len(steps) - 1):
                n_c = sb.n_compressed
                assert torch.equal(sa.k_idx[:, :, :n_c], sb.k_idx[:, :, :n_c]) and torch.equal(sa.v_nrm[:, :, :n_c], sb.v_nrm[:, :, :n_c])
                assert all(torch.equal(x, y) for x, y in zip(sa.window(), sb.window()))
                q = (4 * torch.randn(B, H * G, 1, D, generator=g)).to(dtype).to(DEV)
                out = b.attend(q, l)
                assert out.shape == (B, H * G, 1, D) and out.dtype == dtype
                three = b.attend(q, l, fused=False)              # scores / softmax / weighted values as separate steps
                assert float((out.float() - three.float()).norm() / three.float().norm()) < 4e-3
                tq = b._get_compressor(l, D, DEV)
                kw, vw = sb.window()
                parts_k, parts_v = [], []
                if n_c:
                    parts_k.append(_oracle_decode(oracle, tq.key_compressor, sb.k_idx[:, :, :n_c], sb.k_nrm[:, :, :n_c], (B, H, n_c, D)))
                    parts_v.append(_oracle_decode(oracle, tq.val_compressor, sb.v_idx[:, :, :n_c], sb.v_nrm[:, :, :n_c], (B, H, n_c, D)))
                parts_k.append(kw.float().cpu().numpy())
                parts_v.append(vw.float().cpu().numpy())
                _, ref = oracle.attention_decode(q.squeeze(2).float().cpu().numpy(), np.concatenate(parts_k, 2),
                                                 np.concatenate(parts_v, 2), D ** -0.5)
                got = out.squeeze(2).float().cpu().numpy()
                err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
                # what the model would compute from update()'s tensors
                model = torch.nn.functional.scaled_dot_product_attention(
                    q.float(), fk.float().repeat_interleave(G, dim=1), fv.float().repeat_interleave(G, dim=1)).squeeze(2)
                err_model = float((out.squeeze(2).float() - model).norm() / model.norm())
                print(f"[attend] rw={rw} step {i} layer {l}: vs oracle {err:.2e}, vs attention over update() tensors {err_model:.2e}")
                # output rounded to bf16 / fp16: 2^-9 / 2^-11.  (The tensors update() returns are rounded to 16 bits; with 64-wide
                # heads the softmax scale is 1/8 and the same rounding of a key moves a weight further.)
                assert err < 6e-3 and err_model < (2e-2 if D >= 128 else 4e-2)
        seen += n_new
    with pytest.raises(ValueError):
        b.attend(torch.zeros(B, H * G, 2, D, device=DEV), 0)


@pytest.mark.parametrize("kb,vb,G,S", [(4, 2, 4, 1500), (8, 8, 8, 200), (2, 4, 1, 77), (3, 1, 2, 640), (6, 2, 8, 33), (4, 2, 16, 900), (8, 4, 13, 150)])
def test_fused_attention_partials_against_oracle(pkg, oracle, kb, vb, G, S):
    """The one-pass kernel (scores, online softmax, weighted values per split) merged by the log-sum-exp rule
    equals float64 attention over the oracle-decoded packed keys and values; its records are consistent
    (reference score within the documented distance of the largest score, sums taken against it)."""
    B, H, D = 2, 3, 128
    kc = pkg.MSECompressor(D, kb, seed=11 + kb, device=DEV)
    vc = pkg.MSECompressor(D, vb, seed=511 + vb, device=DEV)
    keys = outlier_kv((B, H, S, D), seed=kb * 100 + S, dtype=torch.bfloat16).to(DEV)
    vals = outlier_kv((B, H, S, D), seed=vb * 100 + S + 1, dtype=torch.bfloat16).to(DEV)
    cap = S + 24
    k_idx = torch.zeros(B, H, cap, D // (8 // kb), dtype=torch.uint8, device=DEV)
    v_idx = torch.zeros(B, H, cap, D // (8 // vb), dtype=torch.uint8, device=DEV)
    k_nrm = torch.zeros(B, H, cap, dtype=torch.float16, device=DEV)
    v_nrm = torch.zeros(B, H, cap, dtype=torch.float16, device=DEV)
    kc.compress_into(keys, k_idx[:, :, :S], k_nrm[:, :, :S])
    vc.compress_into(vals, v_idx[:, :, :S], v_nrm[:, :, :S])
    g = torch.Generator(device="cpu")
    g.manual_seed(S)
    q = (3 * torch.randn(B, H * G, D, generator=g) * torch.exp(0.5 * torch.randn(B, H * G, 1, generator=g))).to(DEV)
    q[0, 0] = 0                                              # a zero query: uniform attention
    scale = D ** -0.5
    q_rot = torch.matmul(q, kc.Pi.T) * scale
    part = torch.ops.tqamd.attend_partials(k_idx[:, :, :S], k_nrm[:, :, :S], v_idx[:, :, :S], v_nrm[:, :, :S],
                                           kc.table(), vc.table(), kb, vb, q_rot)
    assert part.shape[:2] == (B, H * G) and part.shape[3] == D + 2
    m_s, l_s, a_s = part[..., 0], part[..., 1], part[..., 2:]
    m_all = m_s.amax(dim=-1, keepdim=True)
    f = torch.exp(m_s - m_all)
    got = (torch.matmul((f.unsqueeze(-1) * a_s).sum(2), vc.Pi) / (f * l_s).sum(-1, keepdim=True)).cpu().numpy()
    k_hat = _oracle_decode(oracle, kc, k_idx[:, :, :S], k_nrm[:, :, :S], (B, H, S, D))
    v_hat = _oracle_decode(oracle, vc, v_idx[:, :, :S], v_nrm[:, :, :S], (B, H, S, D))
    ref_scores, ref = oracle.attention_decode(q.cpu().numpy(), k_hat, v_hat, scale)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    # the record's reference score is at most the largest score and at most 8 binary orders below it ...
    gap = ref_scores.max(-1) - m_all.squeeze(-1).cpu().numpy()
    tol = 1e-3 * np.abs(ref_scores).max() + 1e-6
    assert gap.min() > -tol and gap.max() < 8 * np.log(2.0) + tol
    # ... and the sum of exponentials is taken against exactly that reference
    l_got = (f * l_s).sum(-1).cpu().numpy()
    l_ref = np.exp(ref_scores - m_all.cpu().numpy().astype(np.float64)).sum(-1)
    # (a score error ds changes exp(score) by the factor e^ds: fp16 keys and queries put ds near 1e-4 of the largest |score|)
    assert np.abs(l_got / l_ref - 1).max() < 3e-3 + 4e-4 * np.abs(ref_scores).max()
    print(f"[fused attention] K{kb} V{vb} G{G} S{S}: relative L2 error {err:.2e}")
    # queries and decoded keys enter the score product as fp16 (2^-12 relative per coordinate), probabilities times
    # value norms as fp16 as well; the queries here are scaled up to logits beyond 100, where that shows most
    assert err < 3e-3


def test_attend_with_window_only_and_without_window(pkg, oracle):
    """Decode-step attention when nothing is compressed yet (window tokens only) and when there is no window."""
    B, H, G, D = 2, 2, 4, 128
    for rw, n in ((128, 50), (0, 90)):
        cache = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=rw, n_layers=1)
        k = outlier_kv((B, H, n, D), seed=800 + rw, dtype=torch.bfloat16).to(DEV)
        v = outlier_kv((B, H, n, D), seed=801 + rw, dtype=torch.bfloat16).to(DEV)
        fk, fv = cache.update(k, v, 0)
        g = torch.Generator(device="cpu")
        g.manual_seed(rw)
        q = (2 * torch.randn(B, H * G, 1, D, generator=g)).to(torch.bfloat16).to(DEV)
        out = cache.attend(q, 0)
        ref = torch.nn.functional.scaled_dot_product_attention(
            q.float(), fk.float().repeat_interleave(G, dim=1), fv.float().repeat_interleave(G, dim=1))
        err = float((out.float() - ref).norm() / ref.norm())
        print(f"[attend] rw={rw}, {n} tokens: vs attention over update() tensors {err:.2e}")
        assert out.shape == q.shape and err < (4e-3 if rw else 2e-2)
        assert float((out.float() - cache.attend(q, 0, fused=False).float()).norm() / ref.norm()) < 4e-3


@pytest.mark.parametrize("wdtype,qdtype,G,W,splits", [(torch.bfloat16, torch.bfloat16, 4, 128, 3), (torch.float16, torch.float16, 8, 512, 1),
                                                      (torch.float32, torch.float32, 1, 37, 2), (torch.bfloat16, torch.float32, 7, 1, 0),
                                                      (torch.float16, torch.bfloat16, 3, 0, 4), (torch.bfloat16, torch.bfloat16, 16, 300, 2), (torch.float32, torch.float16, 11, 70, 1)])
@pytest.mark.parametrize("B", [2, 50])       # 6 rows: one merge block per (row, head); 150 rows: one per row, all heads
def test_attend_prepare_and_merge_against_float64(pkg, wdtype, qdtype, G, W, splits, B):
    """tq_attend_prepare / tq_attend_merge through the C-ABI against the same arithmetic in float64:
    rotated queries to 1e-5, window records to 1e-5, merged output to the output type's rounding."""
    nat = pkg._native
    L = nat.lib()
    H, D, cap = 3, 128, 520
    rows = B * H
    g = torch.Generator(device="cpu")
    g.manual_seed(1000 + G * 7 + W + B)
    q = (3 * torch.randn(B, H * G, 1, D, generator=g)).to(qdtype).to(DEV)
    kbuf = torch.randn(B, H, cap, D, generator=g).to(wdtype).to(DEV)
    vbuf = torch.randn(B, H, cap, D, generator=g).to(wdtype).to(DEV)
    kw, vw = kbuf[:, :, 8:8 + W], vbuf[:, :, 8:8 + W]                # token-axis slices of a larger buffer
    pi_k = pkg.generate_rotation_matrix(D, seed=11).contiguous().to(DEV)
    pi_v = pkg.generate_rotation_matrix(D, seed=12).contiguous().to(DEV)
    scale = 0.11
    q_rot = torch.empty(B, H * G, D, dtype=torch.float32, device=DEV)
    part_w = torch.full((rows, G, D + 2), float("nan"), dtype=torch.float32, device=DEV)
    rc = L.tq_attend_prepare(q.data_ptr(), nat.dtype_code(q.dtype), rows, G, scale, pi_k.t().contiguous().data_ptr(),
                             kw.data_ptr() if W else None, vw.data_ptr() if W else None, nat.dtype_code(wdtype), W, cap * D,
                             q_rot.data_ptr(), part_w.data_ptr() if W else None, None)
    assert rc == 0
    torch.cuda.synchronize()
    q64 = q.double().reshape(B, H, G, D) * scale
    ref_rot = torch.matmul(q64, pi_k.double().T).reshape(B, H * G, D)
    assert float((q_rot.double() - ref_rot).norm() / ref_rot.norm()) < 1e-5
    if W:
        s = torch.matmul(q64, kw.double().transpose(-2, -1))
        m = s.amax(-1)
        p = torch.exp(s - m.unsqueeze(-1))
        l = p.sum(-1)
        a = torch.matmul(p, vw.double())
        pw = part_w.double().reshape(B, H, G, D + 2)
        assert float((pw[..., 0] - m).abs().max()) < 1e-4 and float(((pw[..., 1] - l) / l).abs().max()) < 1e-5
        assert float(((pw[..., 2:] - a).norm(dim=-1) / a.norm(dim=-1)).max()) < 1e-5
    # split records as the one-pass kernel would leave them: random maxima, sums, rotated value sums
    part = None
    if splits:
        part = torch.randn(rows, splits, G, D + 2, generator=g).to(DEV)
        part[..., 0] = part[..., 0] * 3 + (float(m.mean()) if W else 0.0)
        part[..., 1] = part[..., 1].abs() + 0.5
    for odtype in (torch.float32, qdtype):
        out = torch.empty(B, H * G, 1, D, dtype=odtype, device=DEV)
        rc = L.tq_attend_merge(part.data_ptr() if splits else None, splits, part_w.data_ptr() if W else None, pi_v.data_ptr(),
                               rows, G, out.data_ptr(), nat.dtype_code(odtype), None)
        assert rc == 0
        torch.cuda.synchronize()
        m_all = torch.full((rows, G), -float("inf"), dtype=torch.float64, device=DEV)
        if splits:
            p64 = part.double()
            m_all = torch.maximum(m_all, p64[..., 0].amax(dim=1))
        if W:
            w64 = part_w.double()
            m_all = torch.maximum(m_all, w64[..., 0])
        num = torch.zeros(rows, G, D, dtype=torch.float64, device=DEV)
        den = torch.zeros(rows, G, dtype=torch.float64, device=DEV)
        if splits:
            f = torch.exp(p64[..., 0] - m_all.unsqueeze(1))
            num = torch.matmul((f.unsqueeze(-1) * p64[..., 2:]).sum(1), pi_v.double())
            den = (f * p64[..., 1]).sum(1)
        if W:
            f = torch.exp(w64[..., 0] - m_all)
            num = num + f.unsqueeze(-1) * w64[..., 2:]
            den = den + f * w64[..., 1]
        ref = (num / den.unsqueeze(-1)).reshape(B, H * G, 1, D)
        err = float((out.double() - ref).norm() / ref.norm())
        tol = {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 6e-3}[odtype]
        print(f"[prepare/merge] window {W} x {wdtype}, {G} heads, {splits} splits -> {odtype}: {err:.2e}")
        assert err < tol


def test_hf_model_runs_on_the_cache(pkg):
    """A small randomly initialised Llama (transformers, no download) runs prefill + decode and `generate` with the
    cache as `past_key_values`, the way generation_test_v2.py:178-201 drives the reference's cache.  With 8-bit keys
    and values the logits stay close to those of the stock DynamicCache; with K4/V2 the run completes and the cache
    holds what the model fed it."""
    transformers = pytest.importorskip("transformers")
    from transformers import DynamicCache, LlamaConfig, LlamaForCausalLM
    torch.manual_seed(0)
    cfg = LlamaConfig(vocab_size=256, hidden_size=512, intermediate_size=1024, num_hidden_layers=3, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, max_position_embeddings=512)
    model = LlamaForCausalLM(cfg).to(DEV, dtype=torch.bfloat16).eval()
    cls = pkg.hf_cache_class()
    ids = torch.randint(0, 256, (2, 40), device=DEV)
    mask = torch.ones_like(ids)
    with torch.no_grad():
        cache = cls(key_bits=8, value_bits=8, residual_window=8, n_layers=3)
        ref_cache = DynamicCache()
        out = model(ids, attention_mask=mask, past_key_values=cache, use_cache=True)
        ref = model(ids, attention_mask=mask, past_key_values=ref_cache, use_cache=True)
        # prefill attends over what update() returned: the de-quantised prompt (all but the window)
        rel = float((out.logits.float() - ref.logits.float()).norm() / ref.logits.float().norm())
        print(f"[hf] prefill logits, 8-bit cache vs DynamicCache: {rel:.2e}")
        assert rel < 3e-2
        for step in range(6):
            nxt = torch.randint(0, 256, (2, 1), device=DEV)
            mask = torch.cat([mask, torch.ones_like(nxt)], dim=1)
            out = model(nxt, attention_mask=mask, past_key_values=cache, use_cache=True)
            ref = model(nxt, attention_mask=mask, past_key_values=ref_cache, use_cache=True)
            rel = float((out.logits.float() - ref.logits.float()).norm() / ref.logits.float().norm())
            assert rel < 3e-2, (step, rel)
        print(f"[hf] decode step logits, 8-bit cache vs DynamicCache: {rel:.2e}")
        assert cache.get_seq_length() == 46 and ref_cache.get_seq_length() == 46
        assert cache.get_compression_info() == "38 compressed, 8 fp16, 46 total"
        small = cls(key_bits=4, value_bits=2, residual_window=16, n_layers=3)
        gen = model.generate(ids, attention_mask=torch.ones_like(ids), past_key_values=small, max_new_tokens=12, do_sample=False)
        assert gen.shape == (2, 52) and torch.equal(gen[:, :40], ids)
        assert small.get_seq_length() == 51            # the last generated token has not been fed back
        assert small.get_compression_info() == "35 compressed, 16 fp16, 51 total"
        assert sorted(small._stores) == [0, 1, 2]


def test_hf_model_decodes_through_packed_attention(pkg):
    """The same small Llama with the registered attention function: decode steps are answered from the packed
    store (`attend`) and never de-quantise the history.  Same tokens fed to both, the logits equal those of the
    ordinary `update` path of an identically configured cache up to rounding; `generate` runs on it."""
    transformers = pytest.importorskip("transformers")
    from transformers import LlamaConfig, LlamaForCausalLM
    torch.manual_seed(0)
    cfg = LlamaConfig(vocab_size=256, hidden_size=512, intermediate_size=1024, num_hidden_layers=3, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, max_position_embeddings=512)
    model = LlamaForCausalLM(cfg).to(DEV, dtype=torch.bfloat16).eval()
    name = pkg.register_packed_attention()
    cls = pkg.hf_cache_class()
    ids = torch.randint(0, 256, (2, 70), device=DEV)
    steps = [torch.randint(0, 256, (2, 1), device=DEV) for _ in range(8)]
    logits = {}
    with torch.no_grad():
        for packed in (False, True):
            model.config._attn_implementation = name if packed else "sdpa"
            cache = cls(key_bits=4, value_bits=2, residual_window=16, n_layers=3, packed_attention=packed)
            mask = torch.ones_like(ids)
            out = [model(ids, attention_mask=mask, past_key_values=cache, use_cache=True).logits[:, -1:].float()]
            for nxt in steps:
                mask = torch.cat([mask, torch.ones_like(nxt)], dim=1)
                out.append(model(nxt, attention_mask=mask, past_key_values=cache, use_cache=True).logits.float())
            logits[packed] = torch.cat(out, dim=1)
            assert cache.get_seq_length() == 78 and cache.get_compression_info() == "62 compressed, 16 fp16, 78 total"
        a, b = logits[False], logits[True]
        assert torch.equal(a[:, 0], b[:, 0])                       # prefill takes the same path in both
        rel = float((a[:, 1:] - b[:, 1:]).norm() / a[:, 1:].norm())
        print(f"[hf] decode logits, packed attention vs update path (K4/V2): {rel:.2e}")
        assert rel < 2e-2
        model.config._attn_implementation = name
        cache = cls(key_bits=4, value_bits=2, residual_window=16, n_layers=3, packed_attention=True)
        gen = model.generate(ids, attention_mask=torch.ones_like(ids), past_key_values=cache, max_new_tokens=10, do_sample=False)
        assert gen.shape == (2, 80) and cache.get_seq_length() == 79
        # a padded batch is refused in that mode: attention from the packed store counts every cached token
        cache = cls(key_bits=4, value_bits=2, residual_window=16, n_layers=3, packed_attention=True)
        mask = torch.ones_like(ids)
        model(ids, attention_mask=mask, past_key_values=cache, use_cache=True)
        mask = torch.cat([mask, torch.ones_like(steps[0])], dim=1)
        mask[1, :3] = 0
        with pytest.raises(RuntimeError, match="hides cached tokens"):
            model(steps[0], attention_mask=mask, past_key_values=cache, use_cache=True)
        # a cache in packed mode under a model whose attention is not the registered function: the step of layer 0
        # would be attention over one token; the next call on the cache says so instead
        model.config._attn_implementation = "sdpa"
        cache = cls(key_bits=4, value_bits=2, residual_window=16, n_layers=3, packed_attention=True)
        mask = torch.ones_like(ids)
        model(ids, attention_mask=mask, past_key_values=cache, use_cache=True)
        mask = torch.cat([mask, torch.ones_like(steps[0])], dim=1)
        with pytest.raises(RuntimeError, match="never answered"):
            model(steps[0], attention_mask=mask, past_key_values=cache, use_cache=True)


def test_fused_attention_over_extreme_value_norms(pkg, oracle):
    """Value norms spanning twelve decimal orders inside one history (tiny, ordinary, huge, exactly zero) and keys
    with zero vectors: the kernel scales value norms relative to the largest one it has seen, so the result follows
    float64 attention over the oracle-decoded cache wherever the huge-norm tokens carry weight, and rows whose
    values are all tiny or all zero come out tiny or zero, never NaN."""
    B, H, G, S, D = 1, 4, 4, 700, 128
    kc = pkg.MSECompressor(D, 4, seed=21, device=DEV)
    vc = pkg.MSECompressor(D, 2, seed=521, device=DEV)
    g = torch.Generator(device="cpu")
    g.manual_seed(77)
    keys = torch.randn(B, H, S, D, generator=g)
    vals = torch.randn(B, H, S, D, generator=g)
    vals[:, 0] *= 1e-6                                   # a row of tiny values
    vals[:, 1, :300] *= 1e-6                             # tiny first, then huge: the reference exponent has to move
    vals[:, 1, 300:] *= 3e3
    vals[:, 2] = 0                                       # all zero
    vals[:, 3, ::7] *= 3e3                               # mixed within every run (norms stay below the fp16 limit of 65504)
    keys[:, 3, 100:140] = 0                              # zero keys score 0
    keys, vals = keys.to(torch.bfloat16).to(DEV), vals.to(torch.bfloat16).to(DEV)
    ck, cv = kc.compress(keys), vc.compress(vals)
    k_idx, k_nrm = ck["idx_bytes"].reshape(B, H, S, -1), ck["vec_norms"].reshape(B, H, S)
    v_idx, v_nrm = cv["idx_bytes"].reshape(B, H, S, -1), cv["vec_norms"].reshape(B, H, S)
    q = torch.randn(B, H * G, D, generator=g).to(DEV)
    scale = D ** -0.5
    q_rot = torch.matmul(q, kc.Pi.T) * scale
    part = torch.ops.tqamd.attend_partials(k_idx, k_nrm, v_idx, v_nrm, kc.table(), vc.table(), 4, 2, q_rot)
    assert bool(torch.isfinite(part).all())
    m_s, l_s, a_s = part[..., 0], part[..., 1], part[..., 2:]
    f = torch.exp(m_s - m_s.amax(dim=-1, keepdim=True))
    got = (torch.matmul((f.unsqueeze(-1) * a_s).sum(2), vc.Pi) / (f * l_s).sum(-1, keepdim=True)).cpu().numpy()
    k_hat = _oracle_decode(oracle, kc, k_idx, k_nrm, (B, H, S, D))
    v_hat = _oracle_decode(oracle, vc, v_idx, v_nrm, (B, H, S, D))
    _, ref = oracle.attention_decode(q.cpu().numpy(), k_hat, v_hat, scale)
    got, ref = got.reshape(H, G, D), ref.reshape(H, G, D)
    for h in (0, 1, 3):
        err = np.linalg.norm(got[h] - ref[h]) / np.linalg.norm(ref[h])
        print(f"[fused attention] value-norm case {h}: relative L2 error {err:.2e}, |out| = {np.linalg.norm(ref[h]):.2e}")
        assert err < 3e-3
    assert np.all(got[2] == 0) and np.all(ref[2] == 0)


def test_attend_with_sixteen_query_heads_per_kv_head(pkg, oracle):
    """The widest group the one-pass path takes (128 query heads over 8 kv heads): same result as the three-step
    form and as attention over the tensors update() returns."""
    B, H, G, D = 1, 2, 16, 128
    a = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=32, n_layers=1)
    b = pkg.V3Cache(key_bits=4, value_bits=2, residual_window=32, n_layers=1)
    k = outlier_kv((B, H, 700, D), seed=900, dtype=torch.bfloat16).to(DEV)
    v = outlier_kv((B, H, 700, D), seed=901, dtype=torch.bfloat16).to(DEV)
    fk, fv = a.update(k, v, 0)
    b.append(k, v, 0)
    g = torch.Generator(device="cpu")
    g.manual_seed(16)
    q = (2 * torch.randn(B, H * G, 1, D, generator=g)).to(torch.bfloat16).to(DEV)
    out = b.attend(q, 0)
    three = b.attend(q, 0, fused=False)
    ref = torch.nn.functional.scaled_dot_product_attention(
        q.float(), fk.float().repeat_interleave(G, dim=1), fv.float().repeat_interleave(G, dim=1))
    e1 = float((out.float() - three.float()).norm() / three.float().norm())
    e2 = float((out.float() - ref).norm() / ref.norm())
    print(f"[attend] 16 heads per kv head: vs three-step {e1:.2e}, vs attention over update() tensors {e2:.2e}")
    assert e1 < 4e-3 and e2 < 1.5e-2


@pytest.mark.parametrize("dtype,layout", [(torch.bfloat16, "bhsd"), (torch.float16, "bshd"), (torch.float32, "bhsd")])
def test_single_call_decode_step_equals_the_general_path(pkg, dtype, layout):
    """Steady-state decode steps go through tq_append_token / tq_attend_step (one library call each).  Two
    caches fed the same tokens, one of them forced onto the general path, must hold the same bytes after every
    step and give the same attention output; the run crosses several compactions of the window buffer and a
    growth of the packed store."""
    kvc = pkg.kv_cache
    B, H, G, D, rw = 2, 3, 4, 128, 16
    fast = pkg.V3Cache(4, 2, residual_window=rw, n_layers=4)
    slow = pkg.V3Cache(4, 2, residual_window=rw, n_layers=4)
    g = torch.Generator().manual_seed(5)

    def tokens(n):
        if layout == "bshd":                      # what a model's projections give: [B,S,H,D] storage
            return (torch.randn(B, n, H, D, generator=g) * 1.5).to(dtype).to(DEV).transpose(1, 2)
        return (torch.randn(B, H, n, D, generator=g) * 1.5).to(dtype).to(DEV)

    calls = {"append": 0, "attend": 0}
    real_append, real_attend = kvc._LayerStore.append_one, kvc.V3Cache._attend_step

    def counted_append(self, k, v):
        done = real_append(self, k, v)
        calls["append"] += bool(done)
        return done

    def counted_attend(st, q, G_, scale):
        out = real_attend(st, q, G_, scale)
        calls["attend"] += out is not None
        return out

    k0, v0 = tokens(40), tokens(40)
    for c in (fast, slow):
        c.append(k0, v0, 1)
    steps = 300
    for i in range(steps):
        k, v = tokens(1), tokens(1)
        q = (torch.randn(B, H * G, 1, D, generator=g)).to(dtype).to(DEV)
        kvc._LayerStore.append_one, kvc.V3Cache._attend_step = counted_append, staticmethod(counted_attend)
        try:
            fast.append(k, v, 1)
            a = fast.attend(q, 1)
        finally:
            kvc._LayerStore.append_one, kvc.V3Cache._attend_step = real_append, staticmethod(real_attend)
        kvc._LayerStore.append_one = lambda self, k_, v_: False
        kvc.V3Cache._attend_step = staticmethod(lambda st, q_, G_, s_: None)
        try:
            slow.append(k, v, 1)
            b = slow.attend(q, 1)
        finally:
            kvc._LayerStore.append_one, kvc.V3Cache._attend_step = real_append, staticmethod(real_attend)
        assert torch.equal(a, b), i
    sf, ss = fast._stores[1], slow._stores[1]
    assert (sf.n_compressed, sf.n_recent, sf.total_seq) == (ss.n_compressed, ss.n_recent, ss.total_seq) == (40 + steps - rw, rw, 40 + steps)
    n = sf.n_compressed
    for name in ("k_idx", "k_nrm", "v_idx", "v_nrm"):
        assert torch.equal(getattr(sf, name)[:, :, :n], getattr(ss, name)[:, :, :n]), name
    for x, y in zip(sf.window(), ss.window()):
        assert torch.equal(x, y)
    # the single-call path really ran: every step attends through it, and every append except those that
    # first have to move the window back to the front of its buffer or to grow the packed store
    assert calls["attend"] == steps and calls["append"] >= steps - steps // rw - 6, calls


def test_append_token_and_attend_step_through_the_c_abi(pkg, oracle):
    """The two per-step entry points called by hand: the evicted window token lands in the packed slot with the
    bytes tq_compress gives, the new token in the window slot, and tq_attend_step returns what the three
    separate calls return."""
    nat = pkg._native
    L = nat.lib()
    rows, D, G, win_cap, cap = 6, 128, 4, 32, 64
    kc, vc = pkg.MSECompressor(D, 4, seed=1, device=DEV), pkg.MSECompressor(D, 2, seed=2, device=DEV)
    g = torch.Generator().manual_seed(9)
    k_win = torch.randn(rows, win_cap, D, generator=g).to(torch.bfloat16).to(DEV)
    v_win = torch.randn(rows, win_cap, D, generator=g).to(torch.bfloat16).to(DEV)
    k_new = torch.randn(rows, 2, D, generator=g).to(torch.bfloat16).to(DEV)[:, 1]      # rows 2*D elements apart
    v_new = torch.randn(rows, D, generator=g).to(torch.bfloat16).to(DEV)
    k_idx = torch.full((rows, cap, 64), 0xEE, dtype=torch.uint8, device=DEV)
    v_idx = torch.full((rows, cap, 32), 0xEE, dtype=torch.uint8, device=DEV)
    k_nrm = torch.full((rows, cap), -3.0, dtype=torch.float16, device=DEV)
    v_nrm = torch.full((rows, cap), -3.0, dtype=torch.float16, device=DEV)
    want_k, want_v = k_win.clone(), v_win.clone()
    stream = torch.cuda.current_stream().cuda_stream
    evict, put, slot = 5, 21, 7
    rc = L.tq_append_token(k_new.data_ptr(), v_new.data_ptr(), 2, 2 * D, D, k_win.data_ptr(), v_win.data_ptr(), win_cap * D,
                           evict, put, kc.table().data_ptr(), vc.table().data_ptr(), D, 4, 2,
                           k_idx.data_ptr(), k_nrm.data_ptr(), v_idx.data_ptr(), v_nrm.data_ptr(), cap, slot, rows, stream)
    assert rc == 0, L.tq_status_string(rc)
    torch.cuda.synchronize()
    want_k[:, put], want_v[:, put] = k_new, v_new
    assert torch.equal(k_win, want_k) and torch.equal(v_win, want_v)
    ck = kc.compress(want_k[:, evict].reshape(1, rows, 1, D))
    cv = vc.compress(want_v[:, evict].reshape(1, rows, 1, D))
    assert torch.equal(k_idx[:, slot], ck["idx_bytes"].reshape(rows, 64)) and torch.equal(k_nrm[:, slot], ck["vec_norms"].reshape(rows))
    assert torch.equal(v_idx[:, slot], cv["idx_bytes"].reshape(rows, 32)) and torch.equal(v_nrm[:, slot], cv["vec_norms"].reshape(rows))
    untouched = torch.ones(cap, dtype=torch.bool)
    untouched[slot] = False
    assert bool((k_idx[:, untouched] == 0xEE).all()) and bool((v_nrm[:, untouched] == -3).all())
    # evict = -1: only the window is written
    rc = L.tq_append_token(k_new.data_ptr(), v_new.data_ptr(), 2, 2 * D, D, k_win.data_ptr(), v_win.data_ptr(), win_cap * D,
                           -1, 0, None, None, D, 4, 2, None, None, None, None, cap, 0, rows, stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(k_win[:, 0], k_new) and bool((k_idx[:, untouched] == 0xEE).all())
    # attend over 40 packed tokens + 9 window tokens: one call against three
    x = outlier_kv((1, rows, 40, D), seed=3, dtype=torch.bfloat16).to(DEV)
    pk, pv = kc.compress(x), vc.compress(x * 0.7)
    q = torch.randn(rows, G, D, generator=g).to(torch.bfloat16).to(DEV)
    n_w, splits, scale = 9, 2, D ** -0.5
    outs = []
    for single in (True, False):
        q_rot = torch.empty(rows, G, D, device=DEV)
        part_w = torch.empty(rows, G, D + 2, device=DEV)
        part = torch.empty(rows, splits, G, D + 2, device=DEV)
        out = torch.empty(rows, G, D, dtype=torch.bfloat16, device=DEV)
        kw, vw = k_win[:, 3:], v_win[:, 3:]
        packed = (pk["idx_bytes"].data_ptr(), pk["vec_norms"].data_ptr(), pv["idx_bytes"].data_ptr(), pv["vec_norms"].data_ptr())
        if single:
            rc = L.tq_attend_step(q.data_ptr(), 2, rows, G, scale, kc.pi_transposed().data_ptr(), vc.Pi.data_ptr(),
                                  kw.data_ptr(), vw.data_ptr(), 2, n_w, win_cap * D, *packed, 0, 40,
                                  kc.table().data_ptr(), vc.table().data_ptr(), D, 4, 2,
                                  q_rot.data_ptr(), part_w.data_ptr(), part.data_ptr(), splits, out.data_ptr(), 2, stream)
            assert rc == 0, L.tq_status_string(rc)
        else:
            assert L.tq_attend_prepare(q.data_ptr(), 2, rows, G, scale, kc.pi_transposed().data_ptr(), kw.data_ptr(), vw.data_ptr(),
                                       2, n_w, win_cap * D, q_rot.data_ptr(), part_w.data_ptr(), stream) == 0
            assert L.tq_attend_partials(*packed, 0, rows, 40, kc.table().data_ptr(), vc.table().data_ptr(), D, 4, 2,
                                        q_rot.data_ptr(), G, splits, part.data_ptr(), stream) == 0
            assert L.tq_attend_merge(part.data_ptr(), splits, part_w.data_ptr(), vc.Pi.data_ptr(), rows, G, out.data_ptr(), 2, stream) == 0
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    # and against float64 attention over the de-quantised history and the window
    kd = kc.decompress(pk).double().reshape(rows, 40, D)
    vd = vc.decompress(pv).double().reshape(rows, 40, D)
    K = torch.cat([kd, k_win[:, 3:3 + n_w].double()], 1)
    V = torch.cat([vd, v_win[:, 3:3 + n_w].double()], 1)
    ref = torch.softmax(torch.einsum("rgd,rtd->rgt", q.double(), K) * scale, -1) @ V
    err = float((outs[0].double() - ref).norm() / ref.norm())
    assert err < 6e-3, err


def _codes(idx_bytes, bits, dim):
    """[.., G] packed bytes -> [.., dim] codes (most significant code of a byte first)."""
    ipb = 8 // bits
    shifts = torch.arange(ipb - 1, -1, -1, device=idx_bytes.device, dtype=torch.uint8) * bits
    return ((idx_bytes.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)).flatten(-2)[..., :dim].long()


@pytest.mark.parametrize("dim,bits,group,dtype", [(64, (6, 4), 4, torch.float16), (64, (4, 2), 1, torch.bfloat16), (96, (4, 2), 7, torch.bfloat16),
                                                  (96, (8, 8), 2, torch.float16), (96, (2, 3), 16, torch.bfloat16), (128, (4, 2), 4, torch.bfloat16),
                                                  (128, (1, 1), 3, torch.float16), (128, (8, 4), 16, torch.bfloat16), (256, (4, 2), 5, torch.bfloat16),
                                                  (256, (8, 8), 12, torch.float16), (256, (2, 4), 2, torch.bfloat16)])
def test_one_launch_decode_step_against_float64(pkg, dim, bits, group, dtype):
    """tq_decode_attend at the edges of its tiles: histories of 0, 1, 31 ... tokens (partial runs, one and several splits of a
    row), windows of 1 to 512 tokens, one and many rows; float64 attention over the decoded store and the window.  The result
    is rounded to the element type (2^-9 or 2^-12 relative, 0.29 of that in the mean square per ulp) and carries the 2^-12
    roundings of the query term (times logits of about 10 here) and of the weights: 6e-3 and 3e-3 leave a factor of two."""
    dec = lambda comp, idx, nrm, n: ((comp.centroids.double()[_codes(idx[:, :, :n].contiguous(), comp.bits, dim)] @ comp.Pi.double())
                                     * nrm[:, :, :n].double().unsqueeze(-1))
    g = torch.Generator().manual_seed(dim + group)
    for rows, tokens, window in ((1, 0, 1), (2, 1, 16), (3, 31, 33), (1, 64, 128), (5, 513, 7), (1, 3001, 512), (40, 700, 64), (300, 90, 8)):
        cache = pkg.V3Cache(bits[0], bits[1], residual_window=window, n_layers=40)
        k = (torch.randn(1, rows, tokens + window, dim, generator=g) * torch.exp(0.5 * torch.randn(dim, generator=g))).to(dtype).to(DEV)
        v = torch.randn(1, rows, tokens + window, dim, generator=g).to(dtype).to(DEV)
        cache.append(k, v, 8)
        for step in range(2):
            q = torch.randn(1, rows * group, 1, dim, generator=g).to(dtype).to(DEV)
            out = cache.attend(q, 8).double().reshape(rows, group, dim)
            st = cache._stores[8]
            n = st.n_compressed
            kw, vw = (t.double() for t in st.window())
            K = (torch.cat([dec(st.comp.key_compressor, st.k_idx, st.k_nrm, n), kw], 2) if n else kw).reshape(rows, -1, dim)
            V = (torch.cat([dec(st.comp.val_compressor, st.v_idx, st.v_nrm, n), vw], 2) if n else vw).reshape(rows, -1, dim)
            ref = torch.softmax(torch.matmul(q.double().reshape(rows, group, dim), K.transpose(1, 2).contiguous()) * dim ** -0.5, -1) @ V
            err = float((out - ref).norm() / ref.norm())
            assert err < (6e-3 if dtype == torch.bfloat16 else 3e-3), (rows, tokens, window, step, err)
            cache.append(k[:, :, :1].contiguous(), v[:, :, :1].contiguous(), 8)


@pytest.mark.parametrize("dim,bits", [(64, (4, 4)), (64, (8, 2)), (96, (4, 2)), (96, (8, 8)), (128, (4, 2)), (128, (2, 1)), (128, (8, 8)), (256, (4, 2)), (256, (8, 4))])
def test_decode_attention_with_heads_side_by_side(pkg, dim, bits):
    """Up to 4 and up to 8 query heads of a row share the columns of the matrix products with 4 and 2 blocks of 16 tokens: every group
    size around those bounds, histories that end inside each block of a run, against float64 over the store as the kernel holds it.
    float16 results round to 2^-11 / sqrt(12) of a value (1.4e-4, twice that at the lower end of a binade); at 128 the 2^-12 roundings of
    query and weight come on top (times logits of about 3 here): 3.5e-4 and 1.5e-3."""
    g = torch.Generator().manual_seed(dim + bits[0])
    for rows, tokens in ((2, 15), (1, 17), (3, 47), (1, 63), (2, 65), (1, 545), (1, 4099)):
        cache = pkg.V3Cache(bits[0], bits[1], residual_window=3, n_layers=40)
        k, v = (torch.randn(1, rows, tokens + 3, dim, generator=g).half().to(DEV) for _ in range(2))
        cache.append(k, v, 8)
        for group in (1, 2, 4, 5, 8, 9, 16):
            q = torch.randn(1, rows * group, 1, dim, generator=g).half().to(DEV)
            ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
            err = float((cache.attend(q, 8).double().reshape(ref.shape) - ref).norm() / ref.norm())
            assert err < (1.5e-3 if dim == 128 else 3.5e-4), (rows, tokens, group, err)


def test_decode_attention_with_scratch_at_any_float(pkg):
    """Scratch that begins at an odd multiple of 4 bytes gives the same bytes, and nothing is written outside of it."""
    native = pkg._native
    cache = pkg.V3Cache(4, 2, residual_window=40, n_layers=40)
    x = torch.randn(2, 2, 1500, 128, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
    cache.append(x, x, 8)
    st, q = cache._stores[8], torch.randn(2, 8, 1, 128, generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
    floats = native.lib().tq_decode_scratch_floats(4, 4, 128, st.n_compressed, st.n_recent)
    counters, want = torch.zeros(4, dtype=torch.int32, device=DEV), cache.attend(q, 8)
    for start in (4, 5):
        scratch, out = torch.full((floats + 16,), 7.0, device=DEV), torch.empty_like(q)
        assert (scratch.data_ptr() + 4 * start) % 8 == 4 * (start % 2)
        native.check(native.lib().tq_decode_attend(ctypes.addressof(st.record()), q.data_ptr(), 4, 128 ** -0.5, st.w0, st.n_recent, st.n_compressed, scratch.data_ptr() + 4 * start,
                                                   floats, counters.data_ptr(), out.data_ptr(), native._stream_handle(q.device)), "tq_decode_attend")
        assert torch.equal(out, want) and bool((scratch[:start] == 7).all()) and bool((scratch[start + floats:] == 7).all())


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (64, (2, 8)), (96, (4, 2)), (96, (8, 8)), (128, (4, 2)), (128, (1, 1)), (128, (8, 8)), (256, (4, 2)), (256, (8, 4))])
def test_decode_attention_of_a_layer_on_either_side_of_streaming(pkg, dim, bits):
    """A layer of 8 MiB of packed codes and norms is read with other loads than one a token short of it: one row, the last tokens of a run
    and of the store among them.  Against float64 over the store as the kernel holds it, bounds as in test_decode_attention_with_heads_side_by_side; the
    many tokens of about equal weight leave results of 0.01, where float16 still rounds to 2^-11 of a value."""
    g = torch.Generator().manual_seed(dim + bits[0])
    per_token = dim // (8 // bits[0]) + dim // (8 // bits[1]) + 4
    least = -(-(8 << 20) // (2 * per_token))          # tokens of two rows from which on a layer is streamed
    for tokens in (least - 1, least, least + 33):
        cache = pkg.V3Cache(bits[0], bits[1], residual_window=3, n_layers=40)
        k, v = (torch.randn(1, 2, tokens + 3, dim, generator=g).half().to(DEV) for _ in range(2))
        cache.append(k, v, 8)
        for group in (1, 5, 16):
            q = 2 * torch.randn(1, 2 * group, 1, dim, generator=g).half().to(DEV)
            ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
            err = float((cache.attend(q, 8).double().reshape(ref.shape) - ref).norm() / ref.norm())
            assert err < (1.5e-3 if dim == 128 else 3.5e-4), (tokens, group, err)


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (64, (2, 8)), (64, (4, 4)), (96, (2, 2)), (96, (4, 2)), (96, (8, 8)), (128, (4, 2)), (128, (1, 1)), (128, (2, 4)), (128, (8, 8)),
                                      (256, (4, 2)), (256, (2, 8)), (256, (8, 4))])
def test_decode_attention_gives_the_same_bytes_streamed(pkg, monkeypatch, dim, bits):
    """A history read with the non-temporal hint and without it: the same products and sums in the same order.  One row and several, histories
    that end inside a run, groups of every number of blocks; eager steps, captured ones and the C ABI's calls for a cache whose size is not known."""
    native = pkg._native
    g = torch.Generator().manual_seed(dim + bits[0])
    fits, large = 1, 1 << 40
    asked = []
    real = native.fast()

    class Spy:
        def __getattr__(self, name):
            if name != "decode_attend":
                return getattr(real, name)
            return lambda *args: asked.append(args[-1]) or real.decode_attend(*args)

    for rows, tokens in ((1, 33), (2, 4099), (5, 1025)):
        cache = pkg.V3Cache(bits[0], bits[1], residual_window=20, n_layers=40)
        k, v = (torch.randn(1, rows, tokens + 20, dim, generator=g).half().to(DEV) for _ in range(2))
        cache.append(k, v, 8)
        st = cache._stores[8]
        for group in (1, 5, 16):
            q = torch.randn(1, rows * group, 1, dim, generator=g).half().to(DEV)
            want = cache.attend(q, 8)
            for size in (fits, large):
                st.cache_slot_bytes, st.cache_window_bytes = 0, size
                with monkeypatch.context() as m:
                    m.setattr(native, "fast", Spy)
                    assert torch.equal(cache.attend(q, 8), want), (rows, tokens, group, size)
                assert asked[-1] == size and native.lib().tq_decode_streams(ctypes.addressof(st.record()), tokens, 20, size) == (size == large)
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph):
                    out = cache.attend(q, 8)
                for _ in range(2):
                    out.zero_()
                    graph.replay()
                    torch.cuda.synchronize()
                    assert torch.equal(out, want), (rows, tokens, group, size)


@pytest.mark.parametrize("n_arrived", [5, 9, 10, 63, 64, 159, 160, 1000])
def test_decode_attention_with_counters_at_any_spread(pkg, n_arrived):
    """5 rows whose arrival counters lie 1 to 32 apart, by how many there are: the same bytes, all counters zero again, none touched past the last."""
    native = pkg._native
    cache = pkg.V3Cache(4, 2, residual_window=40, n_layers=40)
    x = torch.randn(1, 5, 1500, 128, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
    cache.append(x, x, 8)
    st, q = cache._stores[8], torch.randn(1, 20, 1, 128, generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
    floats = native.lib().tq_decode_scratch_floats(5, 4, 128, st.n_compressed, st.n_recent)
    scratch, counters, out, want = torch.empty(floats, device=DEV), torch.zeros(n_arrived + 8, dtype=torch.int32, device=DEV), torch.empty_like(q), cache.attend(q, 8)
    counters[n_arrived:] = 7
    for _ in range(2):
        native.check(native.lib().tq_decode_attend_spread(ctypes.addressof(st.record()), q.data_ptr(), 4, 128 ** -0.5, st.w0, st.n_recent, st.n_compressed, scratch.data_ptr(), floats,
                                                          counters.data_ptr(), n_arrived, out.data_ptr(), native._stream_handle(q.device)), "tq_decode_attend_spread")
        assert torch.equal(out, want) and not bool(counters[:n_arrived].any()) and bool((counters[n_arrived:] == 7).all())


@pytest.mark.parametrize("dim,tokens,window", [(64, 34000, 260), (96, 17000, 40), (128, 70000, 128), (256, 20000, 5)])
def test_decode_attention_merges_many_splits(pkg, dim, tokens, window):
    """One row over many blocks: more records than a lane has under way at a time (32) and than a wave has lanes, several windows' tiles
    among them, against float64 over the store as the kernel holds it.  Bounds as in test_decode_attention_with_heads_side_by_side; the many
    tokens of about equal weight leave results of 0.01, where float16 still rounds to 2^-11 of a value."""
    g = torch.Generator().manual_seed(dim)
    cache = pkg.V3Cache(4, 2, residual_window=window, n_layers=40)
    k, v = (torch.randn(1, 1, tokens + window, dim, generator=g).half().to(DEV) for _ in range(2))
    cache.append(k, v, 8)
    for group in (1, 8, 16):
        q = 2 * torch.randn(1, group, 1, dim, generator=g).half().to(DEV)
        ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
        err = float((cache.attend(q, 8).double() - ref).norm() / ref.norm())
        assert err < (1.5e-3 if dim == 128 else 3.5e-4), (group, err)


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (96, (4, 2)), (128, (4, 2)), (256, (8, 4)), (256, (4, 2))])
@pytest.mark.parametrize("rows,tokens,window", [(1, 200, 128), (2, 400, 33), (1, 700, 512), (3, 1500, 128), (1, 6000, 128), (1, 9000, 128), (40, 1300, 100), (300, 70, 128)])
def test_decode_attention_deals_out_window_and_history(pkg, dim, bits, rows, tokens, window):
    """Tiles of the window against splits of the history: fewer, as many and more of them, splits with and without a tile, groups on both
    sides of what is merged in one go, against float64 over the store as the kernel holds it.  Bounds as in test_decode_attention_merges_many_splits."""
    g = torch.Generator().manual_seed(dim + tokens)
    cache = pkg.V3Cache(bits[0], bits[1], residual_window=window, n_layers=40)
    k, v = (torch.randn(1, rows, tokens + window, dim, generator=g).half().to(DEV) for _ in range(2))
    cache.append(k, v, 8)
    for group in (1, 4, 7, 16):
        q = 2 * torch.randn(1, rows * group, 1, dim, generator=g).half().to(DEV)
        ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
        err = float((cache.attend(q, 8).double().reshape(ref.shape) - ref).norm() / ref.norm())
        assert err < (1.5e-3 if dim == 128 else 3.5e-4), (group, err)


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (96, (4, 2)), (128, (4, 2)), (128, (8, 4)), (256, (4, 2))])
@pytest.mark.parametrize("rows,tokens,window", [(1, 150, 32), (2, 1500, 128), (1, 9000, 128), (1, 16000, 160)])
def test_decode_attention_of_any_number_of_heads(pkg, dim, bits, rows, tokens, window):
    """Heads that end at every place of what a wave weighs, a pass merges and is rotated back, against float64 over the store as the kernel
    holds it; one split, up to 32, 64 and more records.  Bounds as in test_decode_attention_merges_many_splits."""
    g = torch.Generator().manual_seed(dim + tokens)
    cache = pkg.V3Cache(bits[0], bits[1], residual_window=window, n_layers=40)
    k, v = (torch.randn(1, rows, tokens + window, dim, generator=g).half().to(DEV) for _ in range(2))
    cache.append(k, v, 8)
    for group in (2, 3, 5, 6, 8, 9, 10, 11, 12, 13, 15, 16):
        q = 2 * torch.randn(1, rows * group, 1, dim, generator=g).half().to(DEV)
        ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
        err = float((cache.attend(q, 8).double().reshape(ref.shape) - ref).norm() / ref.norm())
        assert err < (1.5e-3 if dim == 128 else 3.5e-4), (group, err)


@pytest.mark.parametrize("dim", [64, 96, 128, 256])
@pytest.mark.parametrize("rows,tokens", [(2, 1000), (4, 6000), (8, 20000), (40, 1300)])
def test_decode_attention_sums_the_history_alike_whatever_the_window_holds(pkg, dim, rows, tokens):
    """Windows of no weight at all, logits below -1000: bit for bit what the history gives without one, whatever their size.  (Histories cut
    by what the window takes came out rounded another way: 8e-4 at 128.)"""
    g = torch.Generator().manual_seed(dim + tokens)
    k, v = (torch.randn(1, rows, tokens, dim, generator=g).half().to(DEV) for _ in range(2))
    q = torch.randn(1, rows * 8, 1, dim, generator=g)
    q[..., 0] = 8.0
    q = q.half().to(DEV)
    want = None
    for window in (0, 16, 100, 128, 500):
        far = torch.zeros(1, rows, window, dim)
        far[..., 0] = -250.0 * dim ** 0.5
        part = torch.randn(1, rows, window, dim, generator=g).half().to(DEV)
        cache = pkg.V3Cache(4, 2, residual_window=window, n_layers=40)
        cache.append(torch.cat([k, far.half().to(DEV)], 2), torch.cat([v, part], 2), 8)
        got = cache.attend(q, 8)
        want = got if want is None else want
        assert torch.equal(got, want), (window, float((got.double() - want.double()).norm() / want.double().norm()))


@pytest.mark.parametrize("dim", [64, 96, 128, 256])
@pytest.mark.parametrize("bits", [(4, 2), (8, 3), (6, 4)])
def test_one_launch_append_stores_the_bytes_of_compress(pkg, dim, bits):
    """tq_decode_append against MSECompressor.compress on the evicted tokens (1 to 70 rows: full and partial tiles of rows)."""
    for rows, dtype in ((1, torch.bfloat16), (31, torch.float16), (32, torch.bfloat16), (70, torch.float16)):
        cache = pkg.V3Cache(bits[0], bits[1], residual_window=4, n_layers=40, capacity=64)
        k = outlier_kv((1, rows, 30, dim), seed=dim + rows, dtype=dtype).to(DEV)
        v = outlier_kv((1, rows, 30, dim), seed=dim + rows + 1, dtype=dtype).to(DEV)
        cache.append(k[:, :, :4], v[:, :, :4], 8)
        for t in range(4, 30):
            cache.append(k[:, :, t:t + 1], v[:, :, t:t + 1], 8)
        st = cache._stores[8]
        assert (st.n_compressed, st.n_recent) == (26, 4)
        for comp, x, idx, nrm in ((st.comp.key_compressor, k, st.k_idx, st.k_nrm), (st.comp.val_compressor, v, st.v_idx, st.v_nrm)):
            for t in range(26):
                want = comp.compress(x[:, :, t:t + 1])
                assert torch.equal(nrm[:, :, t:t + 1], want["vec_norms"]) and torch.equal(idx[:, :, t:t + 1], want["idx_bytes"]), (rows, t)
        assert torch.equal(st.window()[0], k[:, :, 26:]) and torch.equal(st.window()[1], v[:, :, 26:])


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (96, (4, 2)), (256, (8, 8)), (256, (4, 4))])
def test_decode_attention_of_other_head_dims_keeps_float32_weights(pkg, dim, bits):
    """At 64, 96 and 256 queries enter the matrix products as two fp16 terms (22 bits) and softmax weights as three.  Against float64
    over the centroids as the kernel holds them (float16) what is left is the rounding of the float16 result, 2^-11 / sqrt(12) = 1.4e-4
    of a value on average over a binade at its lower end (2.4e-4 seen); single-term queries alone add 5e-4 at the logits here."""
    g = torch.Generator().manual_seed(dim)
    tokens, heads, group = 2000, 2, 4
    cache = pkg.V3Cache(bits[0], bits[1], residual_window=32, n_layers=40)
    k = (torch.randn(1, heads, tokens, dim, generator=g) * torch.exp(torch.randn(dim, generator=g))).half().to(DEV)
    v = torch.randn(1, heads, tokens, dim, generator=g).half().to(DEV)
    cache.append(k, v, 8)
    q = (2 * torch.randn(1, heads * group, 1, dim, generator=g)).half().to(DEV)
    out = cache.attend(q, 8).double().reshape(heads, group, dim)
    st = cache._stores[8]
    n = st.n_compressed
    dec = lambda comp, idx, nrm: ((comp.centroids.half().double()[_codes(idx[:, :, :n].contiguous(), comp.bits if comp.bits < 5 else 8, dim)] @ comp.Pi.double())
                                  * nrm[:, :, :n].double().unsqueeze(-1))
    K = torch.cat([dec(st.comp.key_compressor, st.k_idx, st.k_nrm), st.window()[0].double()], 2).reshape(heads, -1, dim)
    V = torch.cat([dec(st.comp.val_compressor, st.v_idx, st.v_nrm), st.window()[1].double()], 2).reshape(heads, -1, dim)
    ref = torch.softmax(torch.matmul(q.double().reshape(heads, group, dim), K.transpose(1, 2).contiguous()) * dim ** -0.5, -1) @ V
    err = float((out - ref).norm() / ref.norm())
    assert err < 3.5e-4, err


def _exact_attention(st, q, scale):
    """float64 attention over a layer's store and window, the centroids rounded to float16 as the kernels hold them."""
    B, Hq, _, D = q.shape
    n = st.n_compressed
    dec = lambda comp, idx, nrm: ((comp.centroids.half().double()[_codes(idx[:, :, :n].contiguous(), comp.bits if comp.bits < 5 else 8, D)] @ comp.Pi.double())  # noqa: E731
                                  * nrm[:, :, :n].double().unsqueeze(-1))
    K = torch.cat([dec(st.comp.key_compressor, st.k_idx, st.k_nrm), st.window()[0].double()], 2)
    V = torch.cat([dec(st.comp.val_compressor, st.v_idx, st.v_nrm), st.window()[1].double()], 2)
    s = torch.matmul(q.double().reshape(B, st.H, Hq // st.H, D), K.transpose(-2, -1).contiguous()) * scale
    return torch.matmul(torch.softmax(s, -1), V).reshape(q.shape)


def _one_heavy_token(pkg, dim, bits, at, orders, norm):
    """A cache of 30 tokens (one wave takes them all) and a window of 32, one head, in which the token `at` has a zero value and 2^orders[g] times the weight
    of every other token for query head g; the others of its part (history or window) share one value of this norm."""
    g = torch.Generator().manual_seed(dim)
    k, v = torch.zeros(1, 1, 62, dim), torch.zeros(1, 1, 62, dim)
    u, val = torch.randn(2, dim, generator=g)
    lo, hi = (0, 30) if at < 30 else (30, 62)
    v[:, :, lo:hi] = val * (norm / val.norm())
    v[:, :, at] = 0
    k[:, :, at] = 40 * u / u.norm()
    q = torch.stack([u / u.norm() * (o * np.log(2.0) / 40 * dim ** 0.5) for o in orders])
    cache = pkg.V3Cache(bits[0], bits[1], residual_window=32, n_layers=40)
    cache.append(k.half().to(DEV), v.half().to(DEV), 8)
    return cache, q.half().reshape(1, len(orders), 1, dim).to(DEV)


@pytest.mark.parametrize("dim,bits", [(64, (6, 4)), (96, (6, 2)), (256, (8, 8)), (256, (6, 4))])
def test_decode_attention_keeps_the_bits_of_small_weights(pkg, dim, bits):
    """One packed token takes nearly all the weight, the others 2^-21 to 2^-22.5 of it each (as float32: 24 bits).  A weight's terms lie on a
    grid of 2^-34 of the largest one, which is 2^-11.5 of the smallest here; the result is rounded to float16, 2^-11 / sqrt(3) in the
    mean square at most: 4.5e-4 in all.  Terms on a grid of 2^-30 gave 4.6e-4 to 6.5e-4."""
    cache, q = _one_heavy_token(pkg, dim, bits, 7, [21 + 1.5 * i / 15 for i in range(16)], 3e4)
    out = cache.attend(q, 8).double()
    ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
    err = float((out - ref).norm() / ref.norm())
    assert err < 4.5e-4, err


@pytest.mark.parametrize("dim", [64, 96, 128, 256])
def test_window_attention_keeps_the_bits_of_small_weights(pkg, dim):
    """The same inside the window of a float16 cache, 2^-28 to 2^-31: nothing but the rounding of the result is left (5 % for single
    elements that round the other way).  Probabilities as two float16 terms are off by twice to three times that."""
    cache, q = _one_heavy_token(pkg, dim, (6, 4), 40, [28 + 3 * i / 15 for i in range(16)], 5e4)
    out = cache.attend(q, 8).double()
    ref = _exact_attention(cache._stores[8], q, dim ** -0.5)
    rounding = float((ref.half().double() - ref).norm())
    assert float((out - ref).norm()) < 1.05 * rounding


@pytest.mark.parametrize("dim", [64, 96, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_infinite_window_values_stay_in_their_coordinate(pkg, dim, dtype):
    """Infinities and a NaN among the values of the window come out in their own coordinate as attention in float32 gives them, for tokens of
    every part of a tile, the last token of a partial tile (which is read again for the rest of it) and the token of weight one."""
    g = torch.Generator().manual_seed(dim)
    for window in (1, 45):
        k = torch.randn(1, 2, 50 + window, dim, generator=g).to(dtype)
        v = torch.randn(1, 2, 50 + window, dim, generator=g).to(dtype)
        q = torch.randn(1, 8, 1, dim, generator=g).to(dtype)
        k[:, :, -1] = q[:, ::4, 0] * 4                 # (the largest probability is exactly one)
        v[:, :, -1, 1], v[:, :, -1, dim - 2] = float("inf"), -float("inf")
        if window > 1:
            v[:, :, 50, 3], v[:, :, 50 + 20, 5], v[:, :, 50 + 31, 6], v[:, :, 50 + 33, 9] = float("inf"), -float("inf"), float("nan"), float("inf")
            v[:, :, 50 + 2, 10], v[:, :, 50 + 3, 10] = float("inf"), -float("inf")
        cache = pkg.V3Cache(4, 2, residual_window=window, n_layers=40)
        cache.append(k.to(DEV), v.to(DEV), 8)
        out = cache.attend(q.to(DEV), 8).double()
        ref = _exact_attention(cache._stores[8], q.to(DEV), dim ** -0.5)
        fin = ref.isfinite()
        assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out[ref.isinf()], ref[ref.isinf()])
        assert float((out[fin] - ref[fin]).norm() / ref[fin].norm()) < (6e-3 if dtype == torch.bfloat16 else 3e-3)


@pytest.mark.parametrize("dim,bits", [(64, 4), (64, 8), (96, 4), (128, 8), (256, 4), (256, 8)])
def test_logits_that_cancel_are_as_exact_as_float32(pkg, dim, bits):
    """Queries almost orthogonal to a packed key, scaled up until the roundings of rotation and score show in the result: it is no
    further from float64 than rotation and score in float32 are (queries and, in float16 caches, Pi enter as two float16 terms)."""
    g = torch.Generator().manual_seed(dim + bits)
    heads, group = 32, 8
    cache = pkg.V3Cache(bits, 4, residual_window=1, n_layers=40)
    k = torch.zeros(1, heads, 3, dim)
    k[:, :, 0] = torch.randn(1, heads, dim, generator=g)
    v = torch.randn(1, heads, 3, dim, generator=g)
    v[:, :, 2] = 0
    cache.append(k.half().to(DEV), v.half().to(DEV), 8)
    st = cache._stores[8]
    kc = st.comp.key_compressor
    codes = kc.centroids.half().double()[_codes(st.k_idx[0, :, :1].contiguous(), bits, dim)][:, 0]       # the keys' directions, rotated
    unit = codes @ kc.Pi.double()
    q = torch.randn(heads, 2048, dim, generator=g).double().to(DEV)
    q = (q - (q @ unit.unsqueeze(-1)) * unit.unsqueeze(1) / (unit * unit).sum(-1)[:, None, None]).half()
    nearest = (q.double() @ unit.unsqueeze(-1)).squeeze(-1).abs().argsort(dim=1)[:, :group]
    q = torch.gather(q, 1, nearest.unsqueeze(-1).expand(-1, -1, dim)).reshape(1, heads * group, 1, dim).contiguous()
    scale = 2.0 ** 17 / (float(st.k_nrm[0, :, 0].float().mean()) * dim ** 0.5)
    ref = _exact_attention(st, q, scale)
    err = float((cache.attend(q, 8, scale=scale).double() - ref).norm())
    rot = torch.matmul(q.float().reshape(heads, group, dim), kc.Pi.t().contiguous()) * scale
    first = (torch.matmul(rot, codes.float().unsqueeze(-1)) * st.k_nrm[0, :, :1].float().unsqueeze(-1)).double()
    vc = st.comp.val_compressor
    vals = (vc.centroids.half().double()[_codes(st.v_idx[0, :, :2].contiguous(), 4, dim)] @ vc.Pi.double()) * st.v_nrm[0, :, :2, None].double()
    probs = torch.softmax(torch.cat([first, torch.zeros_like(first), torch.zeros_like(first)], -1), -1)
    f32 = torch.matmul(probs[..., :2], vals).reshape(q.shape)
    assert err <= float((f32 - ref).norm()), (err, float((f32 - ref).norm()))


@pytest.mark.parametrize("dim", [64, 128])
def test_attend_takes_queries_at_any_element_address(pkg, dim):
    """Contiguous queries that start in the middle of a buffer, on no 16-byte boundary."""
    cache = pkg.V3Cache(4, 2, residual_window=16, n_layers=40)
    k, v = (outlier_kv((1, 2, 100, dim), seed=s, dtype=torch.float16).to(DEV) for s in (1, 2))
    cache.append(k, v, 8)
    q = torch.randn(1, 4, 1, dim, dtype=torch.float16, generator=torch.Generator().manual_seed(3)).to(DEV)
    odd = torch.empty(4 * dim + 1, dtype=torch.float16, device=DEV)[1:].view(1, 4, 1, dim)
    odd.copy_(q)
    assert torch.equal(cache.attend(odd, 8), cache.attend(q, 8))


@pytest.mark.parametrize("dim", [64, 128])
def test_attend_replayed_from_a_graph(pkg, dim):
    """A captured decode step brings its own scratch and clears its arrival counters itself: replays between eager steps of another
    shape on the same stream give the bytes of the eager call (several splits a row: the last block of a row finishes it)."""
    cache, other = (pkg.V3Cache(4, 2, residual_window=16, n_layers=40) for _ in range(2))
    k, v = (outlier_kv((1, 2, 5000, dim), seed=s, dtype=torch.bfloat16).to(DEV) for s in (1, 2))
    cache.append(k, v, 8)
    other.append(k[:, :, :700].expand(3, 2, 700, dim), v[:, :, :700].expand(3, 2, 700, dim), 8)
    qs = torch.randn(6, 1, 8, 1, dim, generator=torch.Generator().manual_seed(dim)).to(torch.bfloat16).to(DEV)
    q3 = qs[:1, 0].expand(3, 8, 1, dim).contiguous()
    want = [cache.attend(q, 8) for q in qs]
    want_other = other.attend(q3, 8)
    q = qs[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        cache.attend(q, 8)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = cache.attend(q, 8)
    for i, expected in enumerate(want):
        q.copy_(qs[i])
        assert torch.equal(other.attend(q3, 8), want_other)
        graph.replay()
        assert torch.equal(out, expected), i
        torch.cuda.synchronize()
        assert torch.equal(cache.attend(qs[i], 8), expected), i


def test_decode_steps_on_two_streams(pkg):
    """Steps of two caches queued on two streams without waiting for each other: scratch and counters are each stream's own."""
    caches, q = [], torch.randn(1, 8, 1, 128, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(DEV)
    for tokens in (6000, 9000):
        cache = pkg.V3Cache(4, 2, residual_window=16, n_layers=40, capacity=tokens + 64)
        k, v = (outlier_kv((1, 2, tokens, 128), seed=tokens + s, dtype=torch.bfloat16).to(DEV) for s in (1, 2))
        cache.append(k, v, 8)
        caches.append((cache, k, v))
    runs = []
    for streams in ((torch.cuda.current_stream(),) * 2, (torch.cuda.Stream(), torch.cuda.Stream())):
        torch.cuda.synchronize()
        outs, copies = ([], []), [copy.deepcopy(c) for c, _, _ in caches]
        torch.cuda.synchronize()
        for step in range(20):
            for i, (_, k, v) in enumerate(caches):
                with torch.cuda.stream(streams[i]):
                    copies[i].append(k[:, :, step:step + 1], v[:, :, step:step + 1], 8)
                    outs[i].append(copies[i].attend(q, 8))
        torch.cuda.synchronize()
        runs.append(outs)
    for i in range(2):
        assert all(torch.equal(a, b) for a, b in zip(runs[0][i], runs[1][i]))


def _layer_forms(dim, dtype, g):
    """[B,H,S,D] tensors laid out in the ways a caller's may be: dense, one row, one head, token slices of a longer buffer, heads
    and tokens exchanged, a broadcast batch; where vectors are moved element by element also an address on no 16-byte boundary."""
    mk = lambda *shape: (torch.randn(shape, generator=g) * 2).to(dtype).to(DEV)
    yield "dense", mk(2, 3, 70, dim)
    yield "one row", mk(1, 1, 33, dim)
    yield "one head", mk(3, 1, 40, dim)
    yield "slice", mk(2, 3, 90, dim)[:, :, 5:77]
    yield "heads last", mk(2, 50, 3, dim).transpose(1, 2)
    if dim % 32:
        yield "odd address", torch.empty(2 * 2 * 40 * dim + 1, dtype=dtype, device=DEV)[1:].view(2, 2, 40, dim).copy_(mk(2, 2, 40, dim))
    yield "broadcast", mk(1, 2, 40, dim).expand(3, 2, 40, dim)


@pytest.mark.parametrize("dim,bits", [(64, (4, 2)), (80, (4, 4)), (96, (6, 3)), (128, (4, 2)), (128, (8, 1)), (256, (3, 2))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_calls_equal_the_calls_per_tensor(pkg, monkeypatch, dim, bits, dtype):
    """compress_kv / decompress_kv through tq_compress_layer and tq_restore_layer against the same methods tensor by tensor: the same
    bytes and values for every layout, with windows of none, one and most of the tokens."""
    g = torch.Generator().manual_seed(dim)
    for window in (0, 1, 32):
        comp = pkg.TurboQuantV3(dim, key_bits=bits[0], value_bits=bits[1], residual_window=window, layer_idx=8, device=DEV)
        for name, k in _layer_forms(dim, dtype, g):
            v = k.flip(0).contiguous() if name in ("dense", "one row") else (k * 1 if name == "slice" else k)
            got = comp.compress_kv(k, v)
            got_full = comp.decompress_kv(*got)
            with monkeypatch.context() as m:
                m.setattr(pkg._native, "compress_layer", lambda *a: None)
                m.setattr(pkg._native, "restore_layer", lambda *a: None)
                want = comp.compress_kv(k, v)
                want_full = comp.decompress_kv(*want)
            for a, b in zip(got, want):
                assert a["compressed"]["shape"] == b["compressed"]["shape"] and a["compressed"]["idx_pad"] == b["compressed"]["idx_pad"]
                assert torch.equal(a["compressed"]["idx_bytes"], b["compressed"]["idx_bytes"]), (name, window)
                assert torch.equal(a["compressed"]["vec_norms"], b["compressed"]["vec_norms"]), (name, window)
            for a, b in zip(got_full, want_full):
                assert a.is_contiguous() and a.dtype == b.dtype and torch.equal(a, b), (name, window)


@pytest.mark.parametrize("dim,dtype", [(128, torch.bfloat16), (64, torch.float16), (80, torch.bfloat16), (256, torch.float16)])
def test_large_layers_equal_the_calls_per_tensor(pkg, dim, dtype):
    """Layers large enough for blocks to draw their tiles from counters (64 and 128: keys and values have a pair of counters each in one
    record of the workspace), with keys and values of different widths, twice in a row: the counters are zero again behind a call."""
    g = torch.Generator().manual_seed(dim)
    tokens = 26003 if dim == 128 else 52007 if dim == 64 else 9001
    k, v = (torch.randn(1, 16, tokens, dim, generator=g).to(dtype).to(DEV) for _ in range(2))
    comp = pkg.TurboQuantV3(dim, key_bits=6, value_bits=2, residual_window=77, layer_idx=8, device=DEV)
    want = [c.compress(x[:, :, :-77].contiguous()) for c, x in ((comp.key_compressor, k), (comp.val_compressor, v))]
    full = [torch.cat([c.decompress(w).to(dtype), x[:, :, -77:]], 2) for c, w, x in zip((comp.key_compressor, comp.val_compressor), want, (k, v))]
    for _ in range(2):
        packed = comp.compress_kv(k, v)
        for got, w in zip(packed, want):
            assert torch.equal(got["compressed"]["idx_bytes"], w["idx_bytes"]) and torch.equal(got["compressed"]["vec_norms"], w["vec_norms"])
        assert all(torch.equal(a, b) for a, b in zip(comp.decompress_kv(*packed), full))


@pytest.mark.parametrize("dim,dtype,tokens", [(128, torch.bfloat16, 2048), (128, torch.float16, 4096), (128, torch.bfloat16, 4097), (128, torch.bfloat16, 8191),
                                              (128, torch.float32, 3000), (64, torch.float16, 8193), (64, torch.bfloat16, 6001), (96, torch.bfloat16, 4500), (256, torch.float16, 1027)])
def test_layers_of_a_few_tiles_a_block_equal_the_calls_per_tensor(pkg, dim, dtype, tokens):
    """Sizes about those at which the blocks of a layer launch, a few tiles each, are dealt out to keys and values by bytes or in halves."""
    g = torch.Generator().manual_seed(tokens)
    k, v = (torch.randn(1, 16, tokens, dim, generator=g).to(dtype).to(DEV) for _ in range(2))
    comp = pkg.TurboQuantV3(dim, key_bits=8, value_bits=2, residual_window=0, layer_idx=8, device=DEV)
    packed = comp.compress_kv(k, v)
    full = comp.decompress_kv(*packed)
    for c, x, got, out in zip((comp.key_compressor, comp.val_compressor), (k, v), packed, full):
        want = c.compress(x)
        assert torch.equal(got["compressed"]["idx_bytes"], want["idx_bytes"]) and torch.equal(got["compressed"]["vec_norms"], want["vec_norms"])
        assert torch.equal(out, c.decompress(want).to(out.dtype))


@pytest.mark.parametrize("dim", [64, 128])
def test_update_restores_the_layer_as_the_calls_per_tensor_do(pkg, monkeypatch, dim):
    """V3Cache.update from a per-row store (packed slots between the rows) and a window that moves through its buffer."""
    full = []
    for fast in (True, False):
        with monkeypatch.context() as m:
            if not fast:
                m.setattr(pkg._native, "restore_layer", lambda *a: None)
            cache = pkg.V3Cache(4, 2, residual_window=8, n_layers=40)
            x = outlier_kv((2, 3, 60, dim), seed=dim, dtype=torch.float16).to(DEV)
            steps = [cache.update(x[:, :, :40], x[:, :, :40], 8)]
            steps += [cache.update(x[:, :, t:t + 1], x[:, :, t:t + 1], 8) for t in range(40, 60)]
            full.append(steps)
    for a, b in zip(*full):
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
