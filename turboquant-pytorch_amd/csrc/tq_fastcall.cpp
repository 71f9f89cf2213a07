// The eager calls of the package from Python to the C ABI in one step each: arguments checked, outputs allocated and the library called
// without going through torch's Python bindings and ctypes for every tensor and address.  A call of the codec is a launch of a few
// microseconds; the interpreter took 13 us around compress, 23 around compress_kv, 12 around attend (launch included, of which the
// runtime's own part is 2.5), so that small calls were bound by the host.
// Every function answers None where the arguments are not plain tensors laid out as its kernel reads them (other types and subclasses, a
// device that is not the current one, strides, alignment, a stream that is being captured where that matters): the caller then takes its
// general path, which copies, falls back or raises.  A status other than 0 comes back as an integer.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include "../../include/tqamd.h"

namespace {

constexpr int INTERFACE = 3;      // of this module to _native.py (FAST_INTERFACE there): raised with any change of what init or a function takes or answers

PyObject *g_workspace = nullptr, *g_drop_workspace = nullptr;      // _native's: ticket counters of (device, stream)
PyObject *g_scratch = nullptr, *g_arrived = nullptr;               // _native's: (device index, stream) -> tensor
PyObject *g_tag = nullptr, *g_device = nullptr;                    // attribute names

// entry points of the library, as _native has loaded it
struct Entries {
    decltype(&tq_compress) compress;
    decltype(&tq_decompress) decompress;
    decltype(&tq_compress_layer) compress_layer;
    decltype(&tq_restore_layer) restore_layer;
    decltype(&tq_decode_append) decode_append;
    decltype(&tq_decode_attend_cached) decode_attend;
    decltype(&tq_qjl_compress) qjl_compress;
    decltype(&tq_qjl_query_scores) qjl_query_scores;
} lib{};

struct Raised {};        // a Python exception is set

// Not taken: the function answers None.  A return and no exception: unwinding through torch's libraries takes 2 us and more, which the
// caller's general path would pay on every call (head dimension 90 with a window, decompress_kv of 700 tokens: 47.7 us without the
// extension, 51.4 with a throw).
#define NEED(ok) do { if (!(ok)) Py_RETURN_NONE; } while (0)
#define TENSOR(name, o) const at::Tensor *const name##_at = tensor(o); NEED(name##_at); const at::Tensor &name = *name##_at
#define TABLE(name, o, like, dim, bits) const at::Tensor *const name##_at = table(o, like, dim, bits); NEED(name##_at); const at::Tensor &name = *name##_at

inline const at::Tensor *tensor(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.has_storage() && t.layout() == at::kStrided && t.is_cuda() && !t.is_neg() ? &t : nullptr;      // (neg: memory holds the values without their sign)
}
inline long long integer(PyObject *o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}
inline int dtype_code(const at::Tensor &t) {      // -1: none
    switch (t.scalar_type()) {
        case at::kFloat: return TQ_F32;
        case at::kHalf: return TQ_F16;
        case at::kBFloat16: return TQ_BF16;
        default: return -1;
    }
}
inline uint8_t *address(const at::Tensor &t) { return static_cast<uint8_t *>(t.data_ptr()); }
inline bool aligned(const void *p, long long bytes) { return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)bytes) == 0; }
inline long long packed_width(long long dim, long long bits) { const long long ipb = 8 / bits; return (dim + ipb - 1) / ipb; }
inline long long vector_alignment(long long dim, long long elem) { return dim % 32 ? elem : 16; }

// A codec table that fits (head_dim, bits): tables carry the pair they were built for.
inline const at::Tensor *table(PyObject *o, const at::Tensor &like, long long dim, long long bits) {
    const at::Tensor *t = tensor(o);
    if (!t || t->device() != like.device() || bits < 1 || bits > 8) return nullptr;
    PyObject *tag = PyObject_GetAttr(o, g_tag);
    if (!tag) { PyErr_Clear(); return nullptr; }
    const bool fits = PyTuple_CheckExact(tag) && PyTuple_GET_SIZE(tag) == 2 && PyLong_AsLongLong(PyTuple_GET_ITEM(tag, 0)) == dim &&
                      PyLong_AsLongLong(PyTuple_GET_ITEM(tag, 1)) == bits;
    Py_DECREF(tag);
    if (PyErr_Occurred()) PyErr_Clear();
    return fits ? t : nullptr;
}

// The current stream of the tensor's device, which has to be the current device (`ok`).
struct Stream {
    int dev;
    unsigned long long handle = 0;
    bool ok = false;
    explicit Stream(const at::Tensor &t) : dev(t.device().index()) {
        int current = -1;
        if (hipGetDevice(&current) != hipSuccess || current != dev) return;
        handle = (unsigned long long)reinterpret_cast<uintptr_t>(c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
        ok = true;
    }
    void *raw() const { return reinterpret_cast<void *>(handle); }
    bool capturing() const {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(static_cast<hipStream_t>(raw()), &status) != hipSuccess) {
            (void)hipGetLastError();      // (the next launch does not answer for it)
            return true;
        }
        return status != hipStreamCaptureStatusNone;
    }
};

// Ticket counters of (device, stream), kept by _native; only calls of many vectors draw tickets.
struct Workspace {
    PyObject *owner;
    const Stream &s;
    void *address = nullptr;
    Workspace(PyObject *any_tensor, const Stream &stream, long long vectors, long long dim) : owner(any_tensor), s(stream) {
        if (vectors < 65536 || (dim != 64 && dim != 128)) return;
        address = reinterpret_cast<void *>(PyLong_AsUnsignedLongLong(call(g_workspace)));
        if (PyErr_Occurred()) throw Raised{};
    }
    void drop() { if (address) call(g_drop_workspace); }      // counters of a launch that did not complete are not trusted

  private:
    PyObject *held = nullptr;
    PyObject *call(PyObject *f) {
        PyObject *device = PyObject_GetAttr(owner, g_device), *h = device ? PyLong_FromUnsignedLongLong(s.handle) : nullptr;
        PyObject *r = h ? PyObject_CallFunctionObjArgs(f, device, h, nullptr) : nullptr;
        Py_XDECREF(device);
        Py_XDECREF(h);
        if (!r) throw Raised{};
        Py_XDECREF(held);
        return held = r;
    }

  public:
    ~Workspace() { Py_XDECREF(held); }
};

// From the allocator, without the dispatcher (which takes about as long again) unless somebody listens there: modes of torch, its function
// transforms, its profiler and other observers of operators, algorithms that have to be deterministic (torch fills new memory then).
inline at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Tensor &like) {
    constexpr c10::DispatchKeySet always({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
    if ((c10::impl::tls_local_dispatch_key_set().included_ - always).empty() && !at::globalContext().deterministicAlgorithms() && !at::hasCallbacks())
        return at::Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
    return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}

template <typename... A> int launch(int (*f)(A...), A... a) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(a...);
    Py_END_ALLOW_THREADS
    return rc;
}

// What the arguments' layout is to the codec: rows of tokens, in elements.
struct Rows {
    long long rows, tokens, row_stride, token_stride;
};
// [B,H,S,D] with a dense last dimension whose other strides merge into two levels
bool two_levels(const at::Tensor &t, Rows &l) {
    const auto size = t.sizes(), stride = t.strides();
    const long long elem = (long long)t.element_size(), align = vector_alignment(size[3], elem);
    if ((size[3] != 1 && stride[3] != 1) || !aligned(t.data_ptr(), align)) return false;
    long long e[3], st[3];
    int n = 0;
    for (int i = 0; i < 3; ++i) {
        if ((stride[i] * elem) % align || size[i] <= 0) return false;
        if (size[i] == 1) continue;
        if (n && st[n - 1] == size[i] * stride[i]) { e[n - 1] *= size[i]; st[n - 1] = stride[i]; }
        else { e[n] = size[i]; st[n] = stride[i]; ++n; }
    }
    if (n > 2) return false;
    if (n == 0) l = {1, 1, 0, size[3]};
    else if (n == 1) l = {1, e[0], 0, st[0]};
    else l = {e[0], e[1], st[0], st[1]};
    return true;
}
inline bool shape_is(const at::Tensor &t, std::initializer_list<long long> want) {
    if (t.dim() != (long long)want.size()) return false;
    int i = 0;
    for (long long w : want) if (t.size(i++) != w) return false;
    return true;
}

PyObject *wrapped(std::initializer_list<at::Tensor> out) {
    PyObject *tuple = PyTuple_New((Py_ssize_t)out.size());
    if (!tuple) throw Raised{};
    Py_ssize_t i = 0;
    for (const at::Tensor &t : out) {
        PyObject *o = THPVariable_Wrap(t);
        if (!o) { Py_DECREF(tuple); throw Raised{}; }
        PyTuple_SET_ITEM(tuple, i++, o);
    }
    return tuple;
}

// compress(states, table, bits) -> (idx_bytes, vec_norms)
PyObject *compress(PyObject *const *a) {
    TENSOR(x, a[0]);
    NEED(x.dim() == 4);
    const int dt = dtype_code(x);
    NEED(dt >= 0);
    const long long bits = integer(a[2]), B = x.size(0), H = x.size(1), S = x.size(2), D = x.size(3), n = B * H * S;
    NEED(n > 0);
    TABLE(tb, a[1], x, D, bits);
    Rows l;
    NEED(two_levels(x, l));
    const Stream s(x);
    NEED(s.ok);
    at::Tensor idx = empty({B, H, S, packed_width(D, bits)}, at::kByte, x), nrm = empty({B, H, S}, at::kHalf, x);
    Workspace ws(a[0], s, n, D);
    const int rc = launch(lib.compress, (const void *)address(x), dt, l.rows, l.tokens, l.row_stride, l.token_stride, (const void *)address(tb), (int)D, (int)bits,
                          address(idx), (uint16_t *)address(nrm), 0ll, ws.address, s.raw());
    if (rc) { ws.drop(); return PyLong_FromLong(rc); }
    return wrapped({idx, nrm});
}

// decompress(idx_bytes, vec_norms, table, bits, shape) -> float32 [B,H,S,D] = shape; dense packed buffers of that shape
PyObject *decompress(PyObject *const *a) {
    TENSOR(idx, a[0]); TENSOR(nrm, a[1]);
    const long long bits = integer(a[3]);
    NEED(idx.dim() == 4 && PyTuple_Check(a[4]) && PyTuple_GET_SIZE(a[4]) == 4);
    for (int i = 0; i < 3; ++i) NEED(integer(PyTuple_GET_ITEM(a[4], i)) == idx.size(i));
    const long long D = integer(PyTuple_GET_ITEM(a[4], 3));
    TABLE(tb, a[2], idx, D, bits);
    NEED(idx.scalar_type() == at::kByte && nrm.scalar_type() == at::kHalf && nrm.device() == idx.device());
    const long long B = idx.size(0), H = idx.size(1), S = idx.size(2), n = B * H * S;
    NEED(n > 0 && idx.size(3) == packed_width(D, bits) && shape_is(nrm, {B, H, S}) && idx.is_contiguous() && nrm.is_contiguous());
    const Stream s(idx);
    NEED(s.ok);
    at::Tensor out = empty({B, H, S, D}, at::kFloat, idx);
    Workspace ws(a[0], s, n, D);
    const int rc = launch(lib.decompress, (const uint8_t *)address(idx), (const uint16_t *)address(nrm), 0ll, 1ll, n, (const void *)address(tb), (int)D, (int)bits,
                          (void *)address(out), (int)TQ_F32, 0ll, D, ws.address, s.raw());
    if (rc) { ws.drop(); return PyLong_FromLong(rc); }
    return THPVariable_Wrap(out);
}

// compress_layer(keys, values, tokens, table_k, table_v, bits_k, bits_v) -> ((k_idx, k_norms, keys[:, :, tokens:]), (v_idx, v_norms, values[:, :, tokens:]))
PyObject *compress_layer(PyObject *const *a) {
    TENSOR(k, a[0]); TENSOR(v, a[1]);
    const int dt = dtype_code(k);
    NEED(dt >= 0);
    NEED(k.dim() == 4 && v.sizes() == k.sizes() && v.strides() == k.strides() && v.scalar_type() == k.scalar_type() && v.device() == k.device());
    const long long tokens = integer(a[2]), bk = integer(a[5]), bv = integer(a[6]);
    const long long B = k.size(0), H = k.size(1), S = k.size(2), D = k.size(3), rows = B * H, elem = (long long)k.element_size();
    const long long sb = k.stride(0), sh = k.stride(1), ss = k.stride(2), align = vector_alignment(D, elem);
    NEED(tokens >= 1 && tokens <= S && rows >= 1 && k.stride(3) == 1 && ss >= D && !(B > 1 && H > 1 && sb != H * sh));
    long long n_rows = rows, n_tokens = tokens, row_stride = H > 1 ? sh : sb;
    NEED(!(rows > 1 && row_stride < D) && aligned(k.data_ptr(), align) && aligned(v.data_ptr(), align));
    NEED((sb * elem) % align == 0 && (sh * elem) % align == 0 && (ss * elem) % align == 0);
    if (rows == 1) row_stride = 0;
    else if (row_stride == tokens * ss) { n_rows = 1; n_tokens = rows * tokens; row_stride = 0; }
    TABLE(tk, a[3], k, D, bk); TABLE(tv, a[4], k, D, bv);
    const Stream s(k);
    NEED(s.ok);
    at::Tensor ki = empty({B, H, tokens, packed_width(D, bk)}, at::kByte, k), kn = empty({B, H, tokens}, at::kHalf, k);
    at::Tensor vi = empty({B, H, tokens, packed_width(D, bv)}, at::kByte, k), vn = empty({B, H, tokens}, at::kHalf, k);
    Workspace ws(a[0], s, rows * tokens, D);
    const int rc = launch(lib.compress_layer, (const void *)address(k), (const void *)address(v), dt, n_rows, n_tokens, row_stride, ss, (const void *)address(tk),
                          (const void *)address(tv), (int)D, (int)bk, (int)bv, address(ki), (uint16_t *)address(kn), address(vi), (uint16_t *)address(vn), ws.address, s.raw());
    if (rc) { ws.drop(); return PyLong_FromLong(rc); }
    PyObject *first = wrapped({ki, kn, k.slice(2, tokens)}), *second = nullptr, *both = nullptr;
    try {
        second = wrapped({vi, vn, v.slice(2, tokens)});
        if (!(both = PyTuple_Pack(2, first, second))) throw Raised{};
    } catch (...) {
        Py_DECREF(first);
        Py_XDECREF(second);
        throw;
    }
    Py_DECREF(first);
    Py_DECREF(second);
    return both;
}

// the windows [B,H,n_win,D] behind `tokens` packed tokens a row: shared by the two callers below
PyObject *restore(PyObject *any, const at::Tensor &ki, const at::Tensor &kn, const at::Tensor &vi, const at::Tensor &vn, long long row_slots, long long B, long long H,
                  long long D, long long tokens, const at::Tensor &tk, const at::Tensor &tv, long long bk, long long bv, const at::Tensor &like, uint8_t *kw, uint8_t *vw,
                  long long n_win, long long sb, long long sh) {
    const int dt = dtype_code(like);
    NEED(dt >= 0);
    const long long elem = (long long)like.element_size();
    NEED(tokens >= 1 && B * H >= 1 && B * H <= 65535);
    if (n_win && (D * elem) % 16) Py_RETURN_FALSE;      // not in the general form either: nothing there has to look again
    if (n_win) NEED(sb >= 0 && sh >= 0 && (sb * elem) % 16 == 0 && (sh * elem) % 16 == 0 && aligned(kw, 16) && aligned(vw, 16));
    else kw = vw = nullptr;
    const Stream s(like);
    NEED(s.ok);
    at::Tensor k = empty({B, H, tokens + n_win, D}, like.scalar_type(), like), v = empty({B, H, tokens + n_win, D}, like.scalar_type(), like);
    Workspace ws(any, s, B * H * tokens, D);
    const int rc = launch(lib.restore_layer, (const uint8_t *)address(ki), (const uint16_t *)address(kn), (const uint8_t *)address(vi), (const uint16_t *)address(vn), row_slots, B, H,
                          tokens, (const void *)address(tk), (const void *)address(tv), (int)D, (int)bk, (int)bv, (const void *)kw, (const void *)vw, n_win, B > 1 ? sb : 0ll,
                          H > 1 ? sh : 0ll, (void *)address(k), (void *)address(v), dt, ws.address, s.raw());
    if (rc) { ws.drop(); return PyLong_FromLong(rc); }
    return wrapped({k, v});
}

inline bool tuple_is(PyObject *o, std::initializer_list<long long> want) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != (Py_ssize_t)want.size()) return false;
    Py_ssize_t i = 0;
    for (long long w : want) {
        PyObject *const v = PyTuple_GET_ITEM(o, i++);
        if (!PyLong_Check(v) || integer(v) != w) return false;
    }
    return true;
}

// restore_dicts(k_idx, k_norms, v_idx, v_norms, tokens, table_k, table_v, bits_k, bits_v, k_win, v_win, shape, packed_shape): restore_layer where the
// shapes of the two dictionaries are those of the tensors, None otherwise
PyObject *restore_layer(PyObject *const *a);
PyObject *restore_dicts(PyObject *const *a) {
    TENSOR(kw, a[9]);
    NEED(kw.dim() == 4);
    const long long tokens = integer(a[4]), B = kw.size(0), H = kw.size(1), D = kw.size(3);
    NEED(tuple_is(a[11], {B, H, tokens + kw.size(2), D}) && tuple_is(a[12], {B, H, tokens, D}));
    return restore_layer(a);
}

// restore_layer(k_idx, k_norms, v_idx, v_norms, tokens, table_k, table_v, bits_k, bits_v, k_win, v_win) -> (keys, values); dense packed buffers
PyObject *restore_layer(PyObject *const *a) {
    TENSOR(ki, a[0]); TENSOR(kn, a[1]); TENSOR(vi, a[2]); TENSOR(vn, a[3]); TENSOR(kw, a[9]); TENSOR(vw, a[10]);
    const long long tokens = integer(a[4]), bk = integer(a[7]), bv = integer(a[8]);
    NEED(kw.dim() == 4 && vw.sizes() == kw.sizes() && vw.strides() == kw.strides() && vw.scalar_type() == kw.scalar_type() && vw.device() == kw.device());
    const long long B = kw.size(0), H = kw.size(1), n_win = kw.size(2), D = kw.size(3);
    TABLE(tk, a[5], kw, D, bk); TABLE(tv, a[6], kw, D, bv);
    for (const at::Tensor *t : {&ki, &kn, &vi, &vn}) NEED(t->is_contiguous() && t->device() == kw.device());
    NEED(shape_is(ki, {B, H, tokens, packed_width(D, bk)}) && shape_is(vi, {B, H, tokens, packed_width(D, bv)}) && shape_is(kn, {B, H, tokens}) && shape_is(vn, {B, H, tokens}));
    NEED(ki.scalar_type() == at::kByte && vi.scalar_type() == at::kByte && kn.scalar_type() == at::kHalf && vn.scalar_type() == at::kHalf);
    NEED(!n_win || (kw.stride(3) == 1 && (n_win == 1 || kw.stride(2) == D)));
    return restore(a[9], ki, kn, vi, vn, 0, B, H, D, tokens, tk, tv, bk, bv, kw, n_win ? address(kw) : nullptr, n_win ? address(vw) : nullptr, n_win, kw.stride(0), kw.stride(1));
}

// restore_store(k_idx, k_norms, v_idx, v_norms, k_win, v_win, table_k, table_v, bits_k, bits_v, tokens, w0, n_win): the same for the first `tokens`
// slots of a cache layer's stores [B,H,capacity,..] and the tokens [w0, w0 + n_win) of its window buffers, all dense
PyObject *restore_store(PyObject *const *a) {
    TENSOR(ki, a[0]); TENSOR(kn, a[1]); TENSOR(vi, a[2]); TENSOR(vn, a[3]); TENSOR(kw, a[4]); TENSOR(vw, a[5]);
    const long long bk = integer(a[8]), bv = integer(a[9]), tokens = integer(a[10]), w0 = integer(a[11]), n_win = integer(a[12]);
    NEED(ki.dim() == 4 && kw.dim() == 4);
    const long long B = kw.size(0), H = kw.size(1), win_cap = kw.size(2), D = kw.size(3), cap = ki.size(2);
    TABLE(tk, a[6], kw, D, bk); TABLE(tv, a[7], kw, D, bv);
    for (const at::Tensor *t : {&ki, &kn, &vi, &vn, &kw, &vw}) NEED(t->is_contiguous() && t->device() == kw.device());
    NEED(tokens <= cap && shape_is(ki, {B, H, cap, packed_width(D, bk)}) && shape_is(vi, {B, H, cap, packed_width(D, bv)}) && shape_is(kn, {B, H, cap}) && shape_is(vn, {B, H, cap}));
    NEED(ki.scalar_type() == at::kByte && vi.scalar_type() == at::kByte && kn.scalar_type() == at::kHalf && vn.scalar_type() == at::kHalf);
    NEED(vw.sizes() == kw.sizes() && vw.scalar_type() == kw.scalar_type() && w0 >= 0 && n_win >= 0 && w0 + n_win <= win_cap);
    const long long off = w0 * D * (long long)kw.element_size();
    return restore(a[4], ki, kn, vi, vn, tokens == cap || B * H == 1 ? 0 : cap, B, H, D, tokens, tk, tv, bk, bv, kw, address(kw) + off, address(vw) + off, n_win, H * win_cap * D, win_cap * D);
}

// decode_append(record, keys, values, k_win, evict, put, slot) -> status; record = address of the layer's tq_decode_layer
PyObject *decode_append(PyObject *const *a) {
    TENSOR(win, a[3]);
    NEED(win.dim() == 4 && win.size(0) * win.size(1) <= 65535);
    const long long B = win.size(0), H = win.size(1), D = win.size(3);
    const uint8_t *p[2];
    long long stride[2];
    for (int i = 0; i < 2; ++i) {
        TENSOR(t, a[1 + i]);
        NEED(t.scalar_type() == win.scalar_type() && t.device() == win.device() && shape_is(t, {B, H, 1, D}));
        NEED(t.stride(3) == 1 && !(B > 1 && H > 1 && t.stride(0) != H * t.stride(1)));
        stride[i] = H > 1 ? t.stride(1) : t.stride(0);
        NEED(!(B * H > 1 && stride[i] < D));           // broadcast views: the general path copies them
        p[i] = address(t);
    }
    const Stream s(win);
    NEED(s.ok);
    const int rc = launch(lib.decode_append, reinterpret_cast<const tq_decode_layer *>(integer(a[0])), (const void *)p[0], (const void *)p[1], stride[0], stride[1],
                          integer(a[4]), integer(a[5]), integer(a[6]), s.raw());
    NEED(rc != TQ_ERR_ALIGN);
    return PyLong_FromLong(rc);
}

// decode_attend(record, queries, k_win, scale, win_first, n_win, tokens, cache_bytes) -> output; scratch and counters of the stream as _native keeps them
PyObject *decode_attend(PyObject *const *a) {
    TENSOR(q, a[1]); TENSOR(win, a[2]);
    NEED(win.dim() == 4 && q.dim() == 4 && q.scalar_type() == win.scalar_type() && q.device() == win.device());
    const long long B = win.size(0), H = win.size(1), D = win.size(3), Hq = q.size(1), rows = B * H, n_win = integer(a[5]);
    NEED(q.size(0) == B && q.size(2) == 1 && q.size(3) == D && Hq > 0 && Hq % H == 0 && Hq / H <= 16 && n_win <= 512 && rows <= 65535);
    NEED(q.is_contiguous() && aligned(q.data_ptr(), 16));
    const Stream s(q);
    NEED(s.ok);
    NEED(!s.capturing());
    const double scale = PyFloat_AsDouble(a[3]);
    if (scale == -1.0 && PyErr_Occurred()) throw Raised{};
    PyObject *key = Py_BuildValue("(iK)", s.dev, s.handle);
    if (!key) throw Raised{};
    PyObject *scratch = PyDict_GetItem(g_scratch, key), *arrived = PyDict_GetItem(g_arrived, key);      // borrowed; this frame keeps them through the call
    Py_XINCREF(scratch);
    Py_XINCREF(arrived);
    Py_DECREF(key);
    struct Held { PyObject *a, *b; ~Held() { Py_XDECREF(a); Py_XDECREF(b); } } held{scratch, arrived};
    NEED(scratch && arrived);
    TENSOR(buf, scratch); TENSOR(counters, arrived);
    NEED(counters.numel() >= rows);
    at::Tensor out = empty(q.sizes(), q.scalar_type(), q);
    const int rc = launch(lib.decode_attend, reinterpret_cast<const tq_decode_layer *>(integer(a[0])), (const void *)address(q), (int)(Hq / H), (float)scale, integer(a[4]), n_win,
                          integer(a[6]), (float *)address(buf), (long long)buf.numel(), (uint32_t *)address(counters), (long long)counters.numel(), integer(a[7]), (void *)address(out), s.raw());
    NEED(rc == 0);           // (a buffer that is too small, or an argument the library refuses: nothing was launched)
    return THPVariable_Wrap(out);
}

// qjl_compress(states, table, qjl_table, mse_bits) -> (idx_bytes, vec_norms, sign_bytes, residual_norm)
PyObject *qjl_compress(PyObject *const *a) {
    TENSOR(x, a[0]); TENSOR(qt, a[2]);
    const int dt = dtype_code(x);
    NEED(dt >= 0);
    NEED(x.dim() == 4 && x.is_contiguous() && aligned(x.data_ptr(), 16) && qt.device() == x.device());
    const long long bits = integer(a[3]), B = x.size(0), H = x.size(1), S = x.size(2), D = x.size(3), n = B * H * S;
    NEED(n > 0 && D == 128);
    TABLE(tb, a[1], x, D, bits);
    const Stream s(x);
    NEED(s.ok);
    at::Tensor idx = empty({B, H, S, packed_width(D, bits)}, at::kByte, x), nrm = empty({B, H, S}, at::kHalf, x);
    at::Tensor sign = empty({B, H, S, D / 8}, at::kByte, x), rn = empty({B, H, S}, at::kHalf, x);
    const int rc = launch(lib.qjl_compress, (const void *)address(x), dt, n, D, (const void *)address(tb), (const void *)address(qt), (int)D, (int)bits, address(idx),
                          (uint16_t *)address(nrm), address(sign), (uint16_t *)address(rn), s.raw());
    if (rc) return PyLong_FromLong(rc);
    return wrapped({idx, nrm, sign, rn});
}

// qjl_scores(queries, idx_bytes, vec_norms, sign_bytes, residual_norm, table, both, mse_bits) -> float32 [B,H,S_q,S_k]
PyObject *qjl_scores(PyObject *const *a) {
    TENSOR(given, a[0]); TENSOR(idx, a[1]); TENSOR(nrm, a[2]); TENSOR(sign, a[3]); TENSOR(rn, a[4]); TENSOR(both, a[6]);
    NEED(given.dim() == 4 && given.size(2) >= 1 && given.size(2) <= 8);
    const at::Tensor q = given.contiguous();
    const int dt = dtype_code(q);
    NEED(dt >= 0);
    NEED(idx.dim() == 4);
    const long long bits = integer(a[7]), B = idx.size(0), H = idx.size(1), S = idx.size(2), D = 128, n_q = q.size(2);
    TABLE(tb, a[5], q, D, bits);
    for (const at::Tensor *t : {&idx, &nrm, &sign, &rn, &both}) NEED(t->is_contiguous() && t->device() == q.device());
    NEED(shape_is(q, {B, H, n_q, D}) && B * H >= 1 && B * H <= 65535 && S >= 1);
    NEED(shape_is(idx, {B, H, S, packed_width(D, bits)}) && shape_is(nrm, {B, H, S}) && shape_is(sign, {B, H, S, D / 8}) && shape_is(rn, {B, H, S}) && shape_is(both, {2, D, D}));
    NEED(idx.scalar_type() == at::kByte && sign.scalar_type() == at::kByte && nrm.scalar_type() == at::kHalf && rn.scalar_type() == at::kHalf && both.scalar_type() == at::kFloat);
    const Stream s(q);
    NEED(s.ok);
    at::Tensor out = empty({B, H, n_q, S}, at::kFloat, q);
    const int rc = launch(lib.qjl_query_scores, (const uint8_t *)address(idx), (const uint16_t *)address(nrm), (const uint8_t *)address(sign), (const uint16_t *)address(rn), B * H, S,
                          (const void *)address(tb), (const float *)address(both), (int)D, (int)bits, (const void *)address(q), dt, n_q, (float *)address(out), s.raw());
    NEED(rc != TQ_ERR_ALIGN);
    if (rc) return PyLong_FromLong(rc);
    return THPVariable_Wrap(out);
}

// No exception leaves a function, and none records gradients.  Errors of torch's (no memory, a device error) become the Python exceptions
// that its own functions raise.
template <PyObject *(*F)(PyObject *const *), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    HANDLE_TH_ERRORS
    try {
        c10::NoGradGuard no_grad;
        return F(args);
    } catch (const Raised &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// init(addresses of the entry points in the order of Entries, workspace, drop_workspace, scratch, arrived, tag)
PyObject *init(PyObject *, PyObject *args) {
    PyObject *addresses, *tag;
    if (!PyArg_ParseTuple(args, "O!OOO!O!U", &PyTuple_Type, &addresses, &g_workspace, &g_drop_workspace, &PyDict_Type, &g_scratch, &PyDict_Type, &g_arrived, &tag))
        return nullptr;
    void *p[sizeof(Entries) / sizeof(void *)];
    if (PyTuple_GET_SIZE(addresses) != (Py_ssize_t)(sizeof(p) / sizeof(p[0]))) {
        PyErr_SetString(PyExc_ValueError, "entry points");
        return nullptr;
    }
    for (size_t i = 0; i < sizeof(p) / sizeof(p[0]); ++i) {
        p[i] = reinterpret_cast<void *>(PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(addresses, (Py_ssize_t)i)));
        if (PyErr_Occurred()) return nullptr;
    }
    static_assert(sizeof(lib) == sizeof(p), "one address each");
    memcpy(&lib, p, sizeof(p));
    for (PyObject *o : {g_workspace, g_drop_workspace, g_scratch, g_arrived}) Py_INCREF(o);      // kept for the life of the process
    Py_INCREF(tag);
    g_tag = tag;
    g_device = PyUnicode_InternFromString("device");
    Py_RETURN_NONE;
}

#define TQ_ENTRY(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"init", &init, METH_VARARGS, nullptr},
    TQ_ENTRY(compress, 3), TQ_ENTRY(decompress, 5), TQ_ENTRY(compress_layer, 7), TQ_ENTRY(restore_layer, 11), TQ_ENTRY(restore_dicts, 13), TQ_ENTRY(restore_store, 13),
    TQ_ENTRY(decode_append, 7), TQ_ENTRY(decode_attend, 8), TQ_ENTRY(qjl_compress, 4), TQ_ENTRY(qjl_scores, 8),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "tqamd_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tqamd_fastcall(void) {
    PyObject *m = PyModule_Create(&module);
    if (m && (PyModule_AddIntConstant(m, "abi_version", TQ_ABI_VERSION) < 0 || PyModule_AddIntConstant(m, "interface", INTERFACE) < 0)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
