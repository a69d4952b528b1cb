// Native front-end of the Python binding (module nntile_amd._front): what
// hip_sdpa.py and kv_cache.py do on every call - look at the tensors, fill the
// argument block, find the stream, call the C ABI - without the interpreter
// and without ctypes.
//
// What bounds it: the call is host work in front of a kernel of a few
// microseconds, and a launch alone costs the host 2.3 us.  Through ctypes a
// generation step cost 13 us of host time, a rotary embedding or a transpose
// 8 us, a backward of one tile pair 20 us - more than the kernels of most
// small calls - nearly all of it attribute look-ups on tensors, ctypes
// structures and torch.cuda.current_stream().  Here a tensor is read through
// its C++ object (a few ns) and the stream through c10.
//
// Conventions: every function takes its arguments by position (the Python
// wrappers own names and defaults) and returns the C ABI's code as an int;
// what is wrong with the Python objects themselves raises, with the
// exceptions and messages the wrappers document.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/nntile_hip_sdpa.h"

namespace
{

enum Type { BF16 = 0, FP16 = 1, FP32 = 2, OTHER = -1 };

// Not a code of the C ABI: the call does not fit the one-launch form.
constexpr int kOtherWay = -100;

struct Bad {};      // a Python exception is set

const at::Tensor &tensor(PyObject *o)
{
    if(!THPVariable_Check(o))
    {
        PyErr_Format(PyExc_TypeError, "a torch tensor is expected, got %.100s",
                Py_TYPE(o)->tp_name);
        throw Bad();
    }
    return THPVariable_Unpack(o);
}

// a tile: a contiguous device tensor
const at::Tensor &tile(PyObject *o)
{
    const at::Tensor &t = tensor(o);
    if(!t.is_cuda() || !t.is_contiguous())
    {
        PyErr_SetString(PyExc_ValueError, "tiles must be contiguous device tensors");
        throw Bad();
    }
    return t;
}

// ... or None
const at::Tensor *maybe_tile(PyObject *o)
{
    return o == Py_None ? nullptr : &tile(o);
}

void *ptr(const at::Tensor *t)
{
    return t == nullptr ? nullptr : t->data_ptr();
}

size_t nbytes(const at::Tensor *t)
{
    return t == nullptr ? 0 : (size_t)t->numel() * t->element_size();
}

Type type_of(PyObject *o, const at::Tensor &t, bool fp32 = true)
{
    switch(t.scalar_type())
    {
        case at::kBFloat16: return BF16;
        case at::kHalf: return FP16;
        case at::kFloat:
            if(fp32)
            {
                return FP32;
            }
            break;
        default: break;
    }
    PyObject *name = PyObject_GetAttrString(o, "dtype");
    PyErr_Format(PyExc_TypeError, "unsupported tile dtype %S", name ? name : Py_None);
    Py_XDECREF(name);
    throw Bad();
}

int64_t integer(PyObject *o)
{
    const long long v = PyLong_AsLongLong(o);
    if(v == -1 && PyErr_Occurred())
    {
        throw Bad();
    }
    return v;
}

void *stream_of(PyObject *o)
{
    if(o == Py_None)
    {
        return c10::hip::getCurrentHIPStream().stream();
    }
    PyObject *v = PyObject_GetAttrString(o, "cuda_stream");
    if(v == nullptr)
    {
        throw Bad();
    }
    void *s = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    if(s == nullptr && PyErr_Occurred())
    {
        throw Bad();
    }
    return s;
}

void rank3(const at::Tensor &t)
{
    if(t.dim() != 3)
    {
        PyErr_Format(PyExc_ValueError, "a tile of three axes is expected, got %d", (int)t.dim());
        throw Bad();
    }
}

// The wrapped body of a function: converts exceptions.
template<typename F>
PyObject *guarded(Py_ssize_t given, Py_ssize_t wanted, F body)
{
    if(given != wanted)
    {
        PyErr_Format(PyExc_TypeError, "%zd arguments are expected, got %zd", wanted, given);
        return nullptr;
    }
    try
    {
        return PyLong_FromLong(body());
    }
    catch(const Bad &)
    {
        return nullptr;
    }
    catch(const std::exception &e)
    {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// The C call itself, without the interpreter's lock: a launch into a full queue
// blocks, and neither the other threads nor a host function ahead of it in the
// stream that wants the lock may wait for it.
// The arguments have been worked out by then, so nothing in here needs Python.
template<typename F, typename... A>
int unlocked(F fn, A... args)
{
    struct Released
    {
        PyThreadState *state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    return fn(args...);
}

typedef int (*tile_fn)(void *, const nntile_hip_sdpa_tile_args *);
typedef int (*tile_cache_fn)(void *, const nntile_hip_sdpa_tile_args *, int64_t);
typedef int (*decode_fn)(void *, const nntile_hip_sdpa_tile_args *, void *, size_t);
typedef int (*decode_cache_fn)(void *, const nntile_hip_sdpa_tile_args *, int64_t, void *, size_t);
typedef int (*append_fn)(void *, const nntile_hip_sdpa_tile_args *, int64_t, const void *,
        const void *, int64_t, void *, size_t);
typedef int (*bwd_fn)(void *, const nntile_hip_sdpa_bwd_args *);

const tile_fn tile_fns[] = {nntile_hip_sdpa_fwd_tile_bf16, nntile_hip_sdpa_fwd_tile_fp16,
    nntile_hip_sdpa_fwd_tile_fp32};
const tile_cache_fn tile_cache_fns[] = {nntile_hip_sdpa_fwd_tile_cache_bf16,
    nntile_hip_sdpa_fwd_tile_cache_fp16, nntile_hip_sdpa_fwd_tile_cache_fp32};
const decode_cache_fn tile_cache_ws_fns[] = {nntile_hip_sdpa_fwd_tile_cache_ws_bf16,
    nntile_hip_sdpa_fwd_tile_cache_ws_fp16, nntile_hip_sdpa_fwd_tile_cache_ws_fp32};
const decode_fn decode_fns[] = {nntile_hip_sdpa_fwd_decode_bf16, nntile_hip_sdpa_fwd_decode_fp16,
    nntile_hip_sdpa_fwd_decode_fp32};
const decode_cache_fn decode_cache_fns[] = {nntile_hip_sdpa_fwd_decode_cache_bf16,
    nntile_hip_sdpa_fwd_decode_cache_fp16, nntile_hip_sdpa_fwd_decode_cache_fp32};
const bwd_fn bwd_fns[] = {nntile_hip_sdpa_bwd_tile_bf16, nntile_hip_sdpa_bwd_tile_fp16};

int append_call(Type ty, void *s, const nntile_hip_sdpa_tile_args *a, int64_t capacity,
        const at::Tensor &k_new, const at::Tensor &v_new, const at::Tensor *ws)
{
    const int64_t rows = k_new.size(1);
    if(ty == FP32)
    {
        return unlocked(nntile_hip_sdpa_fwd_decode_append_cache_fp32, s, a, capacity,
                static_cast<const float *>(k_new.data_ptr()),
                static_cast<const float *>(v_new.data_ptr()), rows, ptr(ws), nbytes(ws));
    }
    return unlocked(ty == BF16 ? nntile_hip_sdpa_fwd_decode_append_cache_bf16
            : nntile_hip_sdpa_fwd_decode_append_cache_fp16, s, a, capacity,
                static_cast<const uint16_t *>(k_new.data_ptr()),
                static_cast<const uint16_t *>(v_new.data_ptr()), rows, ptr(ws), nbytes(ws));
}

size_t decode_workspace(Type ty, const nntile_hip_sdpa_tile_args *a)
{
    return ty == FP32 ? nntile_hip_sdpa_fwd_decode_workspace_bytes_fp32(a)
        : nntile_hip_sdpa_fwd_decode_workspace_bytes(a);
}

// K, Q, V: [entries, rows, head]; n_batch may be None (the whole batch)
void fill_tile_args(nntile_hip_sdpa_tile_args &a, const at::Tensor &K, const at::Tensor &Q,
        const at::Tensor *mask, const at::Tensor &lse, const at::Tensor &V, const at::Tensor &A,
        int64_t mask_mode, PyObject *n_batch, int64_t kv_group, int64_t q_pos0, int64_t k_pos0,
        int64_t causal_offset, int64_t flags)
{
    rank3(Q);
    rank3(K);
    a.batch = Q.size(0);
    a.q_seq = Q.size(1);
    a.head = Q.size(2);
    a.k_seq = K.size(1);
    a.n_batch = n_batch == Py_None ? a.batch : integer(n_batch);
    a.kv_group = kv_group;
    a.mask_mode = (int32_t)mask_mode;
    a.flags = (int32_t)flags;
    a.q_pos0 = q_pos0;
    a.k_pos0 = k_pos0;
    a.causal_offset = causal_offset;
    a.K = K.data_ptr();
    a.Q = Q.data_ptr();
    a.V = V.data_ptr();
    a.mask = ptr(mask);
    a.lse = static_cast<float *>(lse.data_ptr());
    a.A = A.data_ptr();
}

// (K, Q, mask, lse, V, A, mask_mode, n_batch, kv_group, q_pos0, k_pos0,
// causal_offset, flags) at v[0..12]
Type read_tile_call(nntile_hip_sdpa_tile_args &a, PyObject *const *v)
{
    const at::Tensor &K = tile(v[0]), &Q = tile(v[1]);
    const at::Tensor *mask = maybe_tile(v[2]);
    const at::Tensor &lse = tile(v[3]), &V = tile(v[4]), &A = tile(v[5]);
    fill_tile_args(a, K, Q, mask, lse, V, A, integer(v[6]), v[7], integer(v[8]), integer(v[9]),
            integer(v[10]), integer(v[11]), integer(v[12]));
    return type_of(v[1], Q);
}

PyObject *fwd_tile(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 14, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const Type ty = read_tile_call(a, v);
        return unlocked(tile_fns[ty], stream_of(v[13]), &a);
    });
}

// ... + k_seq, stream: K, V are caches
PyObject *fwd_tile_cache(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 15, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const Type ty = read_tile_call(a, v);
        const int64_t capacity = a.k_seq;
        if(tensor(v[0]).sizes() != tensor(v[4]).sizes())
        {
            return NNTILE_HIP_EINVAL;
        }
        a.k_seq = integer(v[13]);
        return unlocked(tile_cache_fns[ty], stream_of(v[14]), &a, capacity);
    });
}

// ... + k_seq, workspace, stream: K, V are caches
PyObject *fwd_tile_cache_ws(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 16, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const at::Tensor *ws = maybe_tile(v[14]);
        const Type ty = read_tile_call(a, v);
        const int64_t capacity = a.k_seq;
        if(tensor(v[0]).sizes() != tensor(v[4]).sizes())
        {
            return NNTILE_HIP_EINVAL;
        }
        a.k_seq = integer(v[13]);
        return unlocked(tile_cache_ws_fns[ty], stream_of(v[15]), &a, capacity, ptr(ws), nbytes(ws));
    });
}

// (Q, k_seq, mask_mode) -> bytes
PyObject *tile_cache_workspace(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 3, [&]() -> long
    {
        const at::Tensor &Q = tensor(v[0]);
        rank3(Q);
        nntile_hip_sdpa_tile_args a = {};
        a.batch = Q.size(0);
        a.q_seq = Q.size(1);
        a.head = Q.size(2);
        a.k_seq = integer(v[1]);
        a.mask_mode = (int32_t)integer(v[2]);
        return (long)(type_of(v[0], Q) == FP32
                ? nntile_hip_sdpa_fwd_tile_cache_workspace_bytes_fp32
                : nntile_hip_sdpa_fwd_tile_cache_workspace_bytes)(&a);
    });
}

// ... + workspace, stream
PyObject *fwd_decode(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 15, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const at::Tensor *ws = maybe_tile(v[13]);
        const Type ty = read_tile_call(a, v);
        return unlocked(decode_fns[ty], stream_of(v[14]), &a, ptr(ws), nbytes(ws));
    });
}

// ... + k_seq, workspace, stream: K, V are caches
PyObject *fwd_decode_cache(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 16, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const at::Tensor *ws = maybe_tile(v[14]);
        const Type ty = read_tile_call(a, v);
        const int64_t capacity = a.k_seq;
        if(tensor(v[0]).sizes() != tensor(v[4]).sizes())
        {
            return NNTILE_HIP_EINVAL;
        }
        a.k_seq = integer(v[13]);
        return unlocked(decode_cache_fns[ty], stream_of(v[15]), &a, capacity, ptr(ws), nbytes(ws));
    });
}

// the new rows fit the caches they are to join
bool rows_fit(const at::Tensor &k_new, const at::Tensor &v_new, const at::Tensor &K,
        const at::Tensor &V)
{
    return k_new.dim() == 3 && K.dim() == 3 && v_new.sizes() == k_new.sizes()
        && K.sizes() == V.sizes() && K.size(0) == k_new.size(0) && K.size(2) == k_new.size(2);
}

// ... + k_seq, k_new, v_new, workspace, stream
PyObject *fwd_decode_append_cache(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 18, [&]() -> int
    {
        nntile_hip_sdpa_tile_args a;
        const at::Tensor &k_new = tile(v[14]), &v_new = tile(v[15]);
        const at::Tensor *ws = maybe_tile(v[16]);
        const Type ty = read_tile_call(a, v);
        const int64_t capacity = a.k_seq, k_seq = integer(v[13]);
        const at::Tensor &K = tensor(v[0]), &V = tensor(v[4]);
        if(!rows_fit(k_new, v_new, K, V) || k_new.size(1) > k_seq
                || k_new.scalar_type() != K.scalar_type())
        {
            return NNTILE_HIP_EINVAL;
        }
        a.k_seq = k_seq;
        return append_call(ty, stream_of(v[17]), &a, capacity, k_new, v_new, ws);
    });
}

// A generation step of KVCache: (k_cache, v_cache, k_new, v_new, Q, lse, A,
// filled, max_cache_size, n_batch, kv_group, mask_mode, flags, workspace or
// None, stream).  kOtherWay when the one-launch form does not take the call,
// EWORKSPACE when the workspace is missing or too small.
PyObject *cache_step(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 15, [&]() -> int
    {
        if(v[0] == Py_None)
        {
            return kOtherWay;       // nothing in the cache yet
        }
        const at::Tensor &k_new = tensor(v[2]), &v_new = tensor(v[3]), &Qt = tensor(v[4]);
        rank3(k_new);
        rank3(Qt);
        const int64_t filled = integer(v[7]), most = integer(v[8]), kv_group = integer(v[10]);
        const int64_t rows = k_new.size(1);
        if(v_new.dim() != 3 || v_new.size(1) != rows || kv_group * Qt.size(1) > 64
                || (Qt.size(2) != 64 && Qt.size(2) != 128) || rows + filled > most
                || !k_new.is_contiguous() || !v_new.is_contiguous())
        {
            return kOtherWay;
        }
        const at::Tensor &K = tile(v[0]), &V = tile(v[1]), &Q = tile(v[4]), &lse = tile(v[5]),
              &A = tile(v[6]);
        tile(v[2]);
        tile(v[3]);
        const int64_t k_seq = filled + rows;
        nntile_hip_sdpa_tile_args a;
        fill_tile_args(a, K, Q, nullptr, lse, V, A, integer(v[11]), v[9], kv_group, 0, 0,
                k_seq - Q.size(1), integer(v[12]));
        const Type ty = type_of(v[4], Q);
        const int64_t capacity = a.k_seq;
        if(!rows_fit(k_new, v_new, K, V) || k_new.scalar_type() != K.scalar_type())
        {
            return NNTILE_HIP_EINVAL;
        }
        a.k_seq = k_seq;
        const at::Tensor *ws = maybe_tile(v[13]);
        if(nbytes(ws) < decode_workspace(ty, &a))
        {
            return NNTILE_HIP_EWORKSPACE;
        }
        return append_call(ty, stream_of(v[14]), &a, capacity, k_new, v_new, ws);
    });
}

// (k_new, v_new, k_cache, v_cache, filled, stream)
PyObject *kv_append(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 6, [&]() -> int
    {
        const at::Tensor &k_new = tile(v[0]), &v_new = tile(v[1]), &K = tile(v[2]),
              &V = tile(v[3]);
        rank3(k_new);
        if(!rows_fit(k_new, v_new, K, V))
        {
            return NNTILE_HIP_EINVAL;
        }
        const Type ty = type_of(v[2], K);
        void *s = stream_of(v[5]);
        const int64_t head = k_new.size(2), rows = k_new.size(1), entries = k_new.size(0),
              capacity = K.size(1), filled = integer(v[4]);
        switch(ty)
        {
            case BF16:
                return unlocked(nntile_hip_kv_cache_append_bf16, s, head, rows, entries, capacity, filled,
                        static_cast<const uint16_t *>(k_new.data_ptr()),
                        static_cast<const uint16_t *>(v_new.data_ptr()),
                        static_cast<uint16_t *>(K.data_ptr()),
                        static_cast<uint16_t *>(V.data_ptr()));
            case FP16:
                return unlocked(nntile_hip_kv_cache_append_fp16, s, head, rows, entries, capacity, filled,
                        static_cast<const uint16_t *>(k_new.data_ptr()),
                        static_cast<const uint16_t *>(v_new.data_ptr()),
                        static_cast<uint16_t *>(K.data_ptr()),
                        static_cast<uint16_t *>(V.data_ptr()));
            default:
                return unlocked(nntile_hip_kv_cache_append_fp32, s, head, rows, entries, capacity, filled,
                        static_cast<const float *>(k_new.data_ptr()),
                        static_cast<const float *>(v_new.data_ptr()),
                        static_cast<float *>(K.data_ptr()), static_cast<float *>(V.data_ptr()));
        }
    });
}

// (K, Q, mask, lse, V, A, scratch_lse, scratch_A, stream)
PyObject *flash_fwd(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 9, [&]() -> int
    {
        const at::Tensor &K = tile(v[0]), &Q = tile(v[1]);
        const at::Tensor *mask = maybe_tile(v[2]);
        const at::Tensor &lse = tile(v[3]), &V = tile(v[4]), &A = tile(v[5]);
        const at::Tensor *s_lse = maybe_tile(v[6]), *s_A = maybe_tile(v[7]);
        rank3(Q);
        const int64_t batch = Q.size(0), seq = Q.size(1), head = Q.size(2);
        if(s_lse != nullptr && nbytes(s_lse) < 4 * (size_t)batch * (size_t)seq)
        {
            PyErr_SetString(PyExc_ValueError, "scratch_lse is smaller than a logsumexp tile");
            throw Bad();
        }
        const Type ty = type_of(v[1], Q);
        void *s = stream_of(v[8]);
        float *l = static_cast<float *>(lse.data_ptr()), *sl = static_cast<float *>(ptr(s_lse));
        if(ty == FP32)
        {
            return unlocked(nntile_hip_flash_sdpa_fwd_fp32, s, seq, head, batch,
                    static_cast<const float *>(K.data_ptr()),
                    static_cast<const float *>(Q.data_ptr()),
                    static_cast<const float *>(ptr(mask)), sl,
                    static_cast<const float *>(V.data_ptr()), static_cast<float *>(ptr(s_A)), l,
                    static_cast<float *>(A.data_ptr()));
        }
        return unlocked(ty == BF16 ? nntile_hip_flash_sdpa_fwd_bf16 : nntile_hip_flash_sdpa_fwd_fp16,
                s, seq, head, batch, static_cast<const uint16_t *>(K.data_ptr()),
                static_cast<const uint16_t *>(Q.data_ptr()),
                static_cast<const uint16_t *>(ptr(mask)), sl,
                static_cast<const uint16_t *>(V.data_ptr()), static_cast<uint16_t *>(ptr(s_A)), l,
                static_cast<uint16_t *>(A.data_ptr()));
    });
}

// (K, Q, V, A, dA, mask, lse, scratch_dQ, dK, dQ, dV, stream)
PyObject *flash_bwd(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 12, [&]() -> int
    {
        const at::Tensor *t[11];
        for(int i = 0; i < 11; ++i)
        {
            t[i] = maybe_tile(v[i]);
        }
        const at::Tensor &Q = tile(v[1]);
        rank3(Q);
        const Type ty = type_of(v[1], Q, false);
        auto p = [&](int i) { return static_cast<uint16_t *>(ptr(t[i])); };
        return unlocked(ty == BF16 ? nntile_hip_flash_sdpa_bwd_bf16 : nntile_hip_flash_sdpa_bwd_fp16,
                stream_of(v[11]), Q.size(1), Q.size(2), Q.size(0), p(0), p(1), p(2), p(3), p(4),
                p(5), static_cast<const float *>(ptr(t[6])), nullptr, p(7), nullptr, p(8), p(9),
                p(10));
    });
}

// (K, Q, V, A, dA, mask, lse, dK, dQ, dV, workspace, mask_mode, n_batch,
// kv_group, q_pos0, k_pos0, causal_offset, flags, stream)
PyObject *bwd_tile(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 19, [&]() -> int
    {
        const at::Tensor *t[11];
        for(int i = 0; i < 11; ++i)
        {
            t[i] = (i == 5) ? maybe_tile(v[i]) : &tile(v[i]);
        }
        const at::Tensor &K = *t[0], &Q = *t[1];
        rank3(Q);
        rank3(K);
        nntile_hip_sdpa_bwd_args a;
        a.batch = Q.size(0);
        a.q_seq = Q.size(1);
        a.head = Q.size(2);
        a.k_seq = K.size(1);
        a.mask_mode = (int32_t)integer(v[11]);
        a.n_batch = v[12] == Py_None ? a.batch : integer(v[12]);
        a.kv_group = integer(v[13]);
        a.q_pos0 = integer(v[14]);
        a.k_pos0 = integer(v[15]);
        a.causal_offset = integer(v[16]);
        a.flags = (int32_t)integer(v[17]);
        a.K = ptr(t[0]);
        a.Q = ptr(t[1]);
        a.V = ptr(t[2]);
        a.A = ptr(t[3]);
        a.dA = ptr(t[4]);
        a.mask = ptr(t[5]);
        a.lse = static_cast<const float *>(ptr(t[6]));
        a.dK = ptr(t[7]);
        a.dQ = ptr(t[8]);
        a.dV = ptr(t[9]);
        a.workspace = ptr(t[10]);
        a.workspace_bytes = nbytes(t[10]);
        return unlocked(bwd_fns[type_of(v[1], Q, false)], stream_of(v[18]), &a);
    });
}

// (src_lse, src_attn, dst_lse, dst_attn, stream)
PyObject *accumulate(PyObject *, PyObject *const *v, Py_ssize_t n)
{
    return guarded(n, 5, [&]() -> int
    {
        const at::Tensor &sl = tile(v[0]), &sa = tile(v[1]), &dl = tile(v[2]), &da = tile(v[3]);
        rank3(da);
        const Type ty = type_of(v[3], da);
        void *s = stream_of(v[4]);
        const int64_t batch = da.size(0), seq = da.size(1), head = da.size(2);
        const float *src_lse = static_cast<const float *>(sl.data_ptr());
        float *dst_lse = static_cast<float *>(dl.data_ptr());
        if(ty == FP32)
        {
            return unlocked(nntile_hip_accumulate_attn_output_fp32, s, head, seq, batch, src_lse,
                    static_cast<const float *>(sa.data_ptr()), dst_lse,
                    static_cast<float *>(da.data_ptr()));
        }
        return unlocked(ty == BF16 ? nntile_hip_accumulate_attn_output_bf16
                : nntile_hip_accumulate_attn_output_fp16, s, head, seq, batch, src_lse,
                    static_cast<const uint16_t *>(sa.data_ptr()), dst_lse,
                    static_cast<uint16_t *>(da.data_ptr()));
    });
}

// (sin, cos, src, dst, backward, stream)
PyObject *rope(PyObject *, PyObject *const *v, Py_ssize_t n_args)
{
    return guarded(n_args, 6, [&]() -> int
    {
        const at::Tensor &sin = tile(v[0]), &cos = tile(v[1]), &src = tile(v[2]),
              &dst = tile(v[3]);
        const int64_t m = sin.numel();
        if(cos.numel() != m || src.numel() != dst.numel()
                || (m != 0 && src.numel() % (2 * m) != 0))
        {
            return NNTILE_HIP_EINVAL;
        }
        const int64_t n = m != 0 ? src.numel() / (2 * m) : 0;
        const int backward = PyObject_IsTrue(v[4]);
        if(backward < 0)
        {
            throw Bad();
        }
        const Type ty = type_of(v[2], src);
        void *s = stream_of(v[5]);
        if(ty == FP32)
        {
            return unlocked(backward ? nntile_hip_rope_backward_fp32 : nntile_hip_rope_fp32, s, m, n,
                    static_cast<const float *>(sin.data_ptr()),
                    static_cast<const float *>(cos.data_ptr()),
                    static_cast<const float *>(src.data_ptr()),
                    static_cast<float *>(dst.data_ptr()));
        }
        const auto fn = ty == BF16
            ? (backward ? nntile_hip_rope_backward_bf16 : nntile_hip_rope_bf16)
            : (backward ? nntile_hip_rope_backward_fp16 : nntile_hip_rope_fp16);
        return unlocked(fn, s, m, n, static_cast<const uint16_t *>(sin.data_ptr()),
                static_cast<const uint16_t *>(cos.data_ptr()),
                static_cast<const uint16_t *>(src.data_ptr()),
                static_cast<uint16_t *>(dst.data_ptr()));
    });
}

// (alpha, src, dst, m, n, stream)
PyObject *transpose(PyObject *, PyObject *const *v, Py_ssize_t n_args)
{
    return guarded(n_args, 6, [&]() -> int
    {
        const at::Tensor &src = tile(v[1]), &dst = tile(v[2]);
        const int64_t m = integer(v[3]), n = integer(v[4]);
        if(src.numel() != m * n || dst.numel() != m * n)
        {
            return NNTILE_HIP_EINVAL;
        }
        const double alpha = PyFloat_AsDouble(v[0]);
        if(alpha == -1.0 && PyErr_Occurred())
        {
            throw Bad();
        }
        const Type ty = type_of(v[1], src);
        void *s = stream_of(v[5]);
        if(ty == FP32)
        {
            return unlocked(nntile_hip_transpose_fp32, s, m, n, (float)alpha,
                    static_cast<const float *>(src.data_ptr()),
                    static_cast<float *>(dst.data_ptr()));
        }
        return unlocked(ty == BF16 ? nntile_hip_transpose_bf16 : nntile_hip_transpose_fp16, s, m, n,
                (float)alpha, static_cast<const uint16_t *>(src.data_ptr()),
                static_cast<uint16_t *>(dst.data_ptr()));
    });
}

// ---- calls prepared once ------------------------------------------------------
// Launch(function address, argument block address, extras): `call(stream)` is
// the C call and nothing else.  extras: the arguments behind the block, as
// integers (addresses, sizes); their number says which of the C ABI's shapes
// the function has.
struct Launch
{
    PyObject_HEAD
    void *fn;
    const void *args;
    int n_extra;
    int64_t extra[6];
};

int launch_init(PyObject *self_, PyObject *args, PyObject *)
{
    Launch *self = reinterpret_cast<Launch *>(self_);
    PyObject *fn, *block, *extra;
    if(!PyArg_ParseTuple(args, "O!O!O!", &PyLong_Type, &fn, &PyLong_Type, &block, &PyTuple_Type,
                &extra))
    {
        return -1;
    }
    self->fn = PyLong_AsVoidPtr(fn);
    self->args = PyLong_AsVoidPtr(block);
    const Py_ssize_t n = PyTuple_GET_SIZE(extra);
    if(n != 0 && n != 2 && n != 3 && n != 6)
    {
        PyErr_SetString(PyExc_ValueError, "no call of the C ABI has that many extra arguments");
        return -1;
    }
    self->n_extra = (int)n;
    for(Py_ssize_t i = 0; i < n; ++i)
    {
        PyObject *e = PyTuple_GET_ITEM(extra, i);
        self->extra[i] = (int64_t)PyLong_AsUnsignedLongLongMask(e);
    }
    return PyErr_Occurred() ? -1 : 0;
}

PyObject *launch_call(PyObject *self_, PyObject *stream)
{
    Launch *self = reinterpret_cast<Launch *>(self_);
    return guarded(1, 1, [&]() -> int
    {
        void *s = stream_of(stream);
        auto p = [&](int i) { return reinterpret_cast<void *>(self->extra[i]); };
        const auto *ta = static_cast<const nntile_hip_sdpa_tile_args *>(self->args);
        switch(self->n_extra)
        {
            case 0:
                // tile, grid and backward calls: (stream, block)
                return unlocked(reinterpret_cast<int (*)(void *, const void *)>(self->fn), s, self->args);
            case 2:
                return unlocked(reinterpret_cast<decode_fn>(self->fn), s, ta, p(0), (size_t)self->extra[1]);
            case 3:
                return unlocked(reinterpret_cast<decode_cache_fn>(self->fn), s, ta, self->extra[0], p(1),
                        (size_t)self->extra[2]);
            default:
                return unlocked(reinterpret_cast<append_fn>(self->fn), s, ta, self->extra[0], p(1), p(2),
                        self->extra[3], p(4), (size_t)self->extra[5]);
        }
    });
}

PyMethodDef launch_methods[] = {
    {"call", launch_call, METH_O, "call(stream or None) -> code"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject launch_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), \
    METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FAST(fwd_tile), FAST(fwd_tile_cache), FAST(fwd_tile_cache_ws), FAST(tile_cache_workspace), FAST(fwd_decode), FAST(fwd_decode_cache),
    FAST(fwd_decode_append_cache), FAST(cache_step), FAST(kv_append), FAST(flash_fwd),
    FAST(flash_bwd), FAST(bwd_tile), FAST(accumulate), FAST(rope), FAST(transpose),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front", nullptr, -1, methods, nullptr, nullptr,
    nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__front()
{
    launch_type.tp_name = "nntile_amd._front.Launch";
    launch_type.tp_basicsize = sizeof(Launch);
    launch_type.tp_flags = Py_TPFLAGS_DEFAULT;
    launch_type.tp_new = PyType_GenericNew;
    launch_type.tp_init = launch_init;
    launch_type.tp_methods = launch_methods;
    if(PyType_Ready(&launch_type) < 0)
    {
        return nullptr;
    }
    PyObject *m = PyModule_Create(&module);
    if(m == nullptr)
    {
        return nullptr;
    }
    Py_INCREF(&launch_type);
    PyModule_AddObject(m, "Launch", reinterpret_cast<PyObject *>(&launch_type));
    PyModule_AddIntConstant(m, "OTHER_WAY", kOtherWay);
    // the builds of torch and Python that this file was compiled against; the
    // loader compares them, and the build looks for them in the file
    static const char tag[] = "nntile_front for " NNTILE_FRONT_TAG ";";
    PyModule_AddStringConstant(m, "TAG", tag);
    return m;
}
