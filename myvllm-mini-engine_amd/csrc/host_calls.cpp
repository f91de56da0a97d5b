// Native call path of the Python entry points.
//
// A small decode or prefill call runs 4-10 us on the GPU; checking its
// tensors, allocating its output and workspace and marshalling two dozen
// arguments in Python costs more than that.  These functions do the same for
// the plain form of a call -- ordinary dense CUDA tensors on the current
// device, no caller-supplied buffers, no host-synchronising validation -- and
// return None for anything else, also for everything the entry points refuse:
// the Python code then runs its checks in full and raises what it always
// raised.  Nothing is kept between calls.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <cmath>
#include <cstdint>
#include <cstring>

#include "mvme_paged.h"

namespace {

// Entry points of libmvme_paged, bound once by the loader.
struct Library {
    decltype(&mvme_last_error) last_error;
    decltype(&mvme_paged_attention_workspace_size) decode_workspace;
    decltype(&mvme_paged_attention) decode;
    decltype(&mvme_paged_attention_decode_write) decode_write;
    decltype(&mvme_paged_prefill_workspace_size) prefill_workspace;
    decltype(&mvme_paged_prefill_attention) prefill;
    decltype(&mvme_prefill_attention_workspace_size) dense_workspace;
    decltype(&mvme_prefill_attention) dense;
    decltype(&mvme_write_kv_cache_slots) write_slots;
    decltype(&mvme_linear_rows) linear;
    decltype(&mvme_qk_norm_rope_write_kv) rope;
} lib;
PyObject* current_raw_stream = nullptr;  // torch's getter: device index -> hipStream_t

constexpr int64_t kMaxCapacity = 1048576;
constexpr int64_t kMaxBatchHeads = 2147483647;

// The tensor behind an exact torch.Tensor / Parameter with dense CUDA storage
// of the process's current device; nullptr for anything else (subclasses,
// functorch wrappers, fake or sparse tensors).
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
    if (t.unsafeGetTensorImpl()->is_python_dispatch() || t.is_conj() || t.is_neg()) return nullptr;
    return &t;
}

// Ordinary eager state: no function or dispatch mode wants to see the calls
// that the Python path would make.
bool eager() { return !at::impl::torch_function_mode_enabled() && !c10::impl::dispatch_mode_enabled(); }

bool as_int(PyObject* o, int64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

bool half_type(const at::Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
int dtype_code(const at::Tensor& t) { return t.scalar_type() == at::kHalf ? MVME_FP16 : MVME_BF16; }
bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
bool on_current_device(const at::Tensor& t) {
    return c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA)->getDevice().index() == t.device().index();
}

// torch's current stream on the tensor's device; false with an error set.
bool stream_of(const at::Tensor& t, void*& stream) {
    PyObject* index = PyLong_FromLong(t.device().index());
    PyObject* raw = index ? PyObject_CallOneArg(current_raw_stream, index) : nullptr;
    Py_XDECREF(index);
    if (!raw) return false;
    stream = PyLong_AsVoidPtr(raw);
    Py_DECREF(raw);
    return !PyErr_Occurred();
}

at::Tensor bytes_like(const at::Tensor& t, size_t bytes) {
    return at::empty({static_cast<int64_t>(bytes)}, t.options().dtype(at::kByte).requires_grad(false));
}

PyObject* raise_status(const char* name, int status) {
    const char* message = lib.last_error();
    PyErr_Format(PyExc_RuntimeError, "%s: %s (status %d)", name, message ? message : "", status);
    return nullptr;
}

// Token stride of [T, H, D] rows the kernels can read in place, or -1.
int64_t row_stride(const at::Tensor& t) {
    const int64_t tokens = t.size(0), heads = t.size(1), dim = t.size(2);
    if ((dim != 1 && t.stride(2) != 1) || (heads != 1 && t.stride(1) != dim)) return -1;
    if (tokens <= 1) return heads * dim;
    return t.stride(0) >= heads * dim ? t.stride(0) : -1;
}

// What decode needs of the cache, the tables and the lengths beside a query
// of [batch, q_heads, head_dim] (which may be a strided view).
struct DecodeShape {
    int64_t batch, q_heads, kv_heads, head_dim, num_blocks, block, width;
};
bool decode_shape(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& tables,
                  const at::Tensor& lens, int64_t block, DecodeShape& s) {
    if (q.dim() != 3 || k.dim() != 4 || v.dim() != 4 || tables.dim() != 2 || lens.dim() != 1) return false;
    const auto device = q.device();
    if (k.device() != device || v.device() != device || tables.device() != device || lens.device() != device) return false;
    if (!half_type(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
        tables.scalar_type() != at::kLong || lens.scalar_type() != at::kLong)
        return false;
    if (!k.is_contiguous() || !v.is_contiguous() || !tables.is_contiguous() || !lens.is_contiguous()) return false;
    if (v.sizes() != k.sizes()) return false;
    s = {q.size(0), q.size(1), k.size(2), q.size(2), k.size(0), block, tables.size(1)};
    if (s.batch <= 0 || s.q_heads <= 0 || s.num_blocks <= 0 || s.kv_heads <= 0 || block <= 0 || k.size(1) != block ||
        k.size(3) != s.head_dim || s.q_heads % s.kv_heads != 0)
        return false;
    switch (s.head_dim) {
        case 16: case 32: case 64: case 80: case 96: case 128: case 192: case 256: break;
        default: return false;
    }
    return tables.size(0) == s.batch && s.width > 0 && lens.size(0) == s.batch && block <= kMaxCapacity &&
           s.width <= kMaxCapacity / block && s.batch <= kMaxBatchHeads / s.q_heads;
}

// decode(query, key_cache, value_cache, block_tables, context_lens, block_size, partition_tokens)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t block = 0, partition = 0;
    if (n != 7 || !as_int(args[5], block) || !as_int(args[6], partition)) Py_RETURN_NONE;
    const at::Tensor* t[5];
    for (int i = 0; i < 5; ++i)
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &tables = *t[3], &lens = *t[4];
    DecodeShape s;
    if (!eager() || !on_current_device(q) || !decode_shape(q, k, v, tables, lens, block, s) || !q.is_contiguous())
        Py_RETURN_NONE;
    void* stream = nullptr;
    if (!stream_of(q, stream)) return nullptr;
    at::Tensor out = at::empty(q.sizes(), q.options().requires_grad(false));
    const size_t need = lib.decode_workspace(s.batch, s.q_heads, s.kv_heads, s.head_dim, block, s.width, partition);
    at::Tensor workspace;
    if (need) workspace = bytes_like(q, need);
    void* ws = need ? workspace.data_ptr() : nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.decode(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                        static_cast<const int64_t*>(tables.data_ptr()), static_cast<const int64_t*>(lens.data_ptr()),
                        s.batch, s.q_heads, s.kv_heads, s.head_dim, s.num_blocks, block, s.width, partition,
                        dtype_code(q), ws, need, stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_paged_attention", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// decode_write(query, key_cache, value_cache, block_tables, context_lens, block_size, new_key, new_value,
//              q_weight, k_weight, cos, sin, eps, partition_tokens): the fused form with norm and RoPE
// (or, with None for the four, the plain write) for rows the one launch can read in place.
PyObject* decode_write(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t block = 0, partition = 0;
    if (n != 14 || !as_int(args[5], block) || !as_int(args[13], partition) || !PyFloat_CheckExact(args[12]))
        Py_RETURN_NONE;
    const bool rope = args[8] != Py_None;
    const double eps = PyFloat_AS_DOUBLE(args[12]);
    const at::Tensor* t[12] = {};
    for (int i = 0; i < 12; ++i) {
        if (i == 5 || (i >= 8 && !rope)) continue;
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    }
    // Without q_weight the Python path does not look at the other three.
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &tables = *t[3], &lens = *t[4], &nk = *t[6], &nv = *t[7];
    DecodeShape s;
    if (!eager() || !on_current_device(q) || !decode_shape(q, k, v, tables, lens, block, s)) Py_RETURN_NONE;
    switch (s.head_dim) {
        case 16: case 32: case 64: case 128: case 256: break;
        default: Py_RETURN_NONE;
    }
    const auto device = q.device();
    for (const at::Tensor* r : {&nk, &nv})
        if (r->dim() != 3 || r->size(0) != s.batch || r->size(1) != s.kv_heads || r->size(2) != s.head_dim ||
            r->scalar_type() != q.scalar_type() || r->device() != device || !aligned16(*r))
            Py_RETURN_NONE;
    const int64_t qs = rope ? row_stride(q) : s.q_heads * s.head_dim, ks = row_stride(nk), vs = row_stride(nv);
    if ((!rope && !q.is_contiguous()) || qs < 0 || ks < 0 || vs < 0 || qs % 8 || ks % 8 || vs % 8 || !aligned16(q) ||
        !aligned16(k) || !aligned16(v))
        Py_RETURN_NONE;
    if (rope) {
        for (int i = 8; i < 10; ++i)
            if (t[i]->scalar_type() != q.scalar_type() || t[i]->dim() != 1 || t[i]->size(0) != s.head_dim ||
                !t[i]->is_contiguous() || t[i]->device() != device || !aligned16(*t[i]))
                Py_RETURN_NONE;
        for (int i = 10; i < 12; ++i)
            if (t[i]->dim() != 2 || t[i]->size(0) != s.batch || t[i]->size(1) * 2 != s.head_dim ||
                !t[i]->is_contiguous() || t[i]->scalar_type() != q.scalar_type() || t[i]->device() != device ||
                !aligned16(*t[i]))
                Py_RETURN_NONE;
    }
    void* stream = nullptr;
    if (!stream_of(q, stream)) return nullptr;
    at::Tensor out = at::empty(q.sizes(), q.options().requires_grad(false));
    const size_t need = lib.decode_workspace(s.batch, s.q_heads, s.kv_heads, s.head_dim, block, s.width, partition);
    at::Tensor workspace;
    if (need) workspace = bytes_like(q, need);
    void* ws = need ? workspace.data_ptr() : nullptr;
    auto ptr = [&](int i) -> const void* { return rope ? t[i]->data_ptr() : nullptr; };
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.decode_write(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                              static_cast<const int64_t*>(tables.data_ptr()),
                              static_cast<const int64_t*>(lens.data_ptr()), s.batch, s.q_heads, s.kv_heads, s.head_dim,
                              s.num_blocks, block, s.width, partition, dtype_code(q), nk.data_ptr(), nv.data_ptr(), ks,
                              vs, ptr(8), ptr(9), ptr(10), ptr(11), static_cast<float>(eps), qs, nullptr, ws, need,
                              stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_paged_attention_decode_write", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// prefill(q, key_cache, value_cache, cu_seqlens_q, query_starts, block_tables, context_lens, block_size, chunk_tokens)
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t block = 0, chunk = 0;
    if (n != 9 || !as_int(args[7], block) || !as_int(args[8], chunk)) Py_RETURN_NONE;
    const at::Tensor* t[7];
    for (int i = 0; i < 7; ++i)
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &cu = *t[3], &starts = *t[4], &tables = *t[5], &lens = *t[6];
    if (!eager() || !on_current_device(q)) Py_RETURN_NONE;
    if (q.dim() != 3 || k.dim() != 4 || v.sizes() != k.sizes() || k.size(1) != block || block <= 0 || k.numel() <= 0 ||
        !k.is_contiguous() || !v.is_contiguous() || !q.is_contiguous() || !half_type(q) ||
        k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
        Py_RETURN_NONE;
    const int64_t tokens = q.size(0), q_heads = q.size(1), head_dim = q.size(2), kv_heads = k.size(2);
    if (tokens <= 0 || q_heads <= 0 || head_dim != k.size(3) || head_dim > 1024 || q_heads % kv_heads != 0) Py_RETURN_NONE;
    if (cu.dim() != 1 || starts.dim() != 1 || lens.dim() != 1 || tables.dim() != 2) Py_RETURN_NONE;
    const int64_t seqs = starts.size(0), width = tables.size(1);
    if (tables.size(0) != seqs || lens.size(0) != seqs || cu.size(0) != seqs + 1) Py_RETURN_NONE;
    for (int i = 1; i < 7; ++i) {
        if (t[i]->device() != q.device()) Py_RETURN_NONE;
        if (i >= 3 && (t[i]->scalar_type() != at::kLong || !t[i]->is_contiguous())) Py_RETURN_NONE;
    }
    void* stream = nullptr;
    if (!stream_of(q, stream)) return nullptr;
    at::Tensor out = at::empty(q.sizes(), q.options().requires_grad(false));
    const size_t need = lib.prefill_workspace(seqs, tokens, q_heads, kv_heads, head_dim, block, width, chunk,
                                              dtype_code(q));
    at::Tensor workspace;
    if (need) workspace = bytes_like(q, need);
    void* ws = need ? workspace.data_ptr() : nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.prefill(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                         static_cast<const int64_t*>(cu.data_ptr()), static_cast<const int64_t*>(starts.data_ptr()),
                         static_cast<const int64_t*>(tables.data_ptr()), static_cast<const int64_t*>(lens.data_ptr()),
                         seqs, tokens, q_heads, kv_heads, head_dim, k.size(0), block, width, chunk, dtype_code(q), ws,
                         need, stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_paged_prefill_attention", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// dense(q, k, v, query_start): [batch, heads, tokens, head_dim] views whose layout needs no copy, head
// dims of the MFMA path.
PyObject* dense(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t start = 0;
    if (n != 4 || !as_int(args[3], start)) Py_RETURN_NONE;
    const at::Tensor* t[3];
    for (int i = 0; i < 3; ++i)
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2];
    if (!eager() || !on_current_device(q) || q.dim() != 4 || k.dim() != 4 || v.sizes() != k.sizes() ||
        v.strides() != k.strides() || !half_type(q) || k.scalar_type() != q.scalar_type() ||
        v.scalar_type() != q.scalar_type() || k.device() != q.device() || v.device() != q.device())
        Py_RETURN_NONE;
    const int64_t batch = q.size(0), q_heads = q.size(1), tokens = q.size(2), d = q.size(3);
    const int64_t kv_heads = k.size(1), kv_tokens = k.size(2);
    if (batch <= 0 || q_heads <= 0 || tokens <= 0 || d <= 0 || d % 8 != 0 || d > 256 || kv_heads <= 0 ||
        q_heads % kv_heads != 0 || k.size(0) != batch || k.size(3) != d || start < 0 || start > kMaxCapacity ||
        start + tokens > kv_tokens || start + tokens > kMaxCapacity)
        Py_RETURN_NONE;
    // (batch, head, token) strides as the kernels read them: 0 for dimensions of size 1.
    int64_t st[3][3];
    for (int i = 0; i < 3; ++i) {
        if (t[i]->stride(3) != 1 || !aligned16(*t[i])) Py_RETURN_NONE;
        for (int j = 0; j < 3; ++j) {
            st[i][j] = t[i]->size(j) > 1 ? t[i]->stride(j) : 0;
            if (st[i][j] % 8 != 0) Py_RETURN_NONE;
        }
    }
    void* stream = nullptr;
    if (!stream_of(q, stream)) return nullptr;
    at::Tensor out = at::empty({batch, tokens, q_heads, d}, q.options().requires_grad(false)).transpose(1, 2);
    int64_t so[3];
    for (int j = 0; j < 3; ++j) so[j] = out.size(j) > 1 ? out.stride(j) : 0;
    const size_t need = lib.dense_workspace(batch, tokens, q_heads, kv_heads, d, start, dtype_code(q));
    at::Tensor workspace;
    if (need) workspace = bytes_like(q, need);
    void* ws = need ? workspace.data_ptr() : nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.dense(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), batch, q_heads, kv_heads, tokens,
                       kv_tokens, d, start, st[0][0], st[0][1], st[0][2], st[1][0], st[1][1], st[1][2], so[0], so[1],
                       so[2], dtype_code(q), ws, need, stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_prefill_attention", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// write_slots(key_cache, value_cache, slot_mapping, key, value): True when the rows were written.
PyObject* write_slots(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) Py_RETURN_NONE;
    const at::Tensor* t[5];
    for (int i = 0; i < 5; ++i)
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    const at::Tensor &kc = *t[0], &vc = *t[1], &slots = *t[2], &key = *t[3], &value = *t[4];
    if (!eager() || !on_current_device(kc) || kc.dim() != 4 || vc.sizes() != kc.sizes() || kc.numel() <= 0 ||
        !kc.is_contiguous() || !vc.is_contiguous() || key.dim() != 3 || value.sizes() != key.sizes() ||
        key.size(1) != kc.size(2) || key.size(2) != kc.size(3) || slots.dim() != 1 || slots.size(0) != key.size(0) ||
        key.size(0) <= 0 || slots.scalar_type() != at::kLong || !slots.is_contiguous() || !half_type(kc))
        Py_RETURN_NONE;
    for (int i = 1; i < 5; ++i)
        if (t[i]->device() != kc.device() || (i != 2 && t[i]->scalar_type() != kc.scalar_type())) Py_RETURN_NONE;
    const int64_t ks = row_stride(key), vs = row_stride(value);
    if (ks < 0 || vs < 0) Py_RETURN_NONE;
    void* stream = nullptr;
    if (!stream_of(kc, stream)) return nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.write_slots(kc.data_ptr(), vc.data_ptr(), kc.size(0), kc.size(1), kc.size(2), kc.size(3),
                             static_cast<const int64_t*>(slots.data_ptr()), key.data_ptr(), value.data_ptr(),
                             key.size(0), ks, vs, dtype_code(kc), stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_write_kv_cache_slots", status);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// linear(x, weight, bias or None) for x of [..., in_features] with dense rows.
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]), *w = plain(args[1]);
    const at::Tensor* bias = args[2] == Py_None ? nullptr : plain(args[2]);
    if (!x || !w || (args[2] != Py_None && !bias) || !eager() || !on_current_device(*x)) Py_RETURN_NONE;
    if (x->dim() != 2 || w->dim() != 2 || !half_type(*x) || w->scalar_type() != x->scalar_type() ||
        w->device() != x->device() || !w->is_contiguous())
        Py_RETURN_NONE;
    const int64_t rows = x->size(0), in = x->size(1), out_features = w->size(0);
    if (rows < 1 || rows > 64 || w->size(1) != in || in <= 0 || in % 32 != 0 || out_features <= 0 ||
        out_features % 16 != 0 || x->stride(1) != 1 || x->stride(0) < in || x->stride(0) % 8 != 0 || !aligned16(*x) ||
        !aligned16(*w))
        Py_RETURN_NONE;
    if (bias && (bias->dim() != 1 || bias->size(0) != out_features || bias->scalar_type() != x->scalar_type() ||
                 !bias->is_contiguous() || bias->device() != x->device()))
        Py_RETURN_NONE;
    void* stream = nullptr;
    if (!stream_of(*x, stream)) return nullptr;
    at::Tensor out = at::empty({rows, out_features}, x->options().requires_grad(false));
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.linear(out.data_ptr(), x->data_ptr(), w->data_ptr(), bias ? bias->data_ptr() : nullptr, rows, in,
                        out_features, x->stride(0), dtype_code(*x), stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_linear_rows", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// rope_slots(q, k, v, q_weight, k_weight, cos, sin, key_cache, value_cache, slot_mapping, eps): the
// rotated queries of the slot-mapping (prefill) form.
PyObject* rope_slots(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 11 || !PyFloat_CheckExact(args[10])) Py_RETURN_NONE;
    const double eps = PyFloat_AS_DOUBLE(args[10]);
    const at::Tensor* t[10];
    for (int i = 0; i < 10; ++i)
        if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
    const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &cos = *t[5], &sin = *t[6], &kc = *t[7], &vc = *t[8];
    if (!eager() || !on_current_device(q) || !half_type(q) || q.dim() != 3 || k.dim() != 3 || v.sizes() != k.sizes() ||
        kc.dim() != 4 || vc.sizes() != kc.sizes() || kc.numel() <= 0 || !kc.is_contiguous() || !vc.is_contiguous())
        Py_RETURN_NONE;
    // What the entry point and the library refuse as too small stays with the Python checks.
    const float eps32 = static_cast<float>(eps);
    if (!(eps32 > 0.f) || !(eps32 < HUGE_VALF)) Py_RETURN_NONE;
    const int64_t tokens = q.size(0), q_heads = q.size(1), d = q.size(2), kv_heads = k.size(1);
    if (tokens <= 0 || k.size(0) != tokens || k.size(2) != d || kv_heads <= 0 || q_heads < kv_heads ||
        q_heads % kv_heads != 0 || d % 2 != 0 || d <= 0 || d > 512 || kc.size(2) != kv_heads || kc.size(3) != d)
        Py_RETURN_NONE;
    for (int i = 1; i < 10; ++i) {
        if (t[i]->device() != q.device()) Py_RETURN_NONE;
        if (i < 9 && t[i]->scalar_type() != q.scalar_type()) Py_RETURN_NONE;
    }
    for (int i = 3; i < 5; ++i)
        if (t[i]->dim() != 1 || t[i]->size(0) != d || !t[i]->is_contiguous()) Py_RETURN_NONE;
    if (cos.dim() != 2 || sin.sizes() != cos.sizes() || cos.size(0) != tokens || cos.size(1) * 2 != d ||
        !cos.is_contiguous() || !sin.is_contiguous())
        Py_RETURN_NONE;
    const at::Tensor& slots = *t[9];
    if (slots.dim() != 1 || slots.size(0) != tokens || slots.scalar_type() != at::kLong || !slots.is_contiguous())
        Py_RETURN_NONE;
    const int64_t qs = row_stride(q), ks = row_stride(k), vs = row_stride(v);
    if (qs < 0 || ks < 0 || vs < 0) Py_RETURN_NONE;
    void* stream = nullptr;
    if (!stream_of(q, stream)) return nullptr;
    at::Tensor out = at::empty(q.sizes(), q.options().requires_grad(false));
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = lib.rope(out.data_ptr(), kc.data_ptr(), vc.data_ptr(), kc.size(0), kc.size(1), kv_heads, d,
                      static_cast<const int64_t*>(slots.data_ptr()), nullptr, 0, nullptr, q.data_ptr(), k.data_ptr(),
                      v.data_ptr(), qs, ks, vs, t[3]->data_ptr(), t[4]->data_ptr(), cos.data_ptr(), sin.data_ptr(),
                      tokens, q_heads, eps32, dtype_code(q), stream);
    Py_END_ALLOW_THREADS
    if (status != MVME_OK) return raise_status("mvme_qk_norm_rope_write_kv", status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// bind(raw_stream_getter, (address, ...)): the library's entry points in the order of Library.
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *getter = nullptr, *addresses = nullptr;
    if (!PyArg_ParseTuple(args, "OO!", &getter, &PyTuple_Type, &addresses)) return nullptr;
    constexpr Py_ssize_t kCount = sizeof(Library) / sizeof(void*);
    if (PyTuple_GET_SIZE(addresses) != kCount) {
        PyErr_SetString(PyExc_ValueError, "wrong number of entry points");
        return nullptr;
    }
    void* found[kCount];
    for (Py_ssize_t i = 0; i < kCount; ++i) {
        found[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i));
        if (PyErr_Occurred()) return nullptr;
        if (!found[i]) {
            PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    static_assert(sizeof(Library) == sizeof(found), "one address per member");
    memcpy(&lib, found, sizeof(lib));
    Py_INCREF(getter);
    Py_XSETREF(current_raw_stream, getter);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"decode", reinterpret_cast<PyCFunction>(decode), METH_FASTCALL, nullptr},
    {"decode_write", reinterpret_cast<PyCFunction>(decode_write), METH_FASTCALL, nullptr},
    {"prefill", reinterpret_cast<PyCFunction>(prefill), METH_FASTCALL, nullptr},
    {"dense", reinterpret_cast<PyCFunction>(dense), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(linear), METH_FASTCALL, nullptr},
    {"rope_slots", reinterpret_cast<PyCFunction>(rope_slots), METH_FASTCALL, nullptr},
    {"write_slots", reinterpret_cast<PyCFunction>(write_slots), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "mvme_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mvme_host(void) { return PyModule_Create(&module); }
