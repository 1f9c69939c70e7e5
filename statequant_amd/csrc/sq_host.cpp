// The Python side's calls into libsqhip.so, in native code: argument checks, the C ABI's structs and the launch of one
// decode step (or state hand-over) without an interpreted instruction in between.
//
// What it is for: a decode step calls the library once per layer, and reading some twenty tensors' pointers, strides and
// dtypes through Python took 16 to 19 us per call -- four times as long as the kernel itself runs for one sequence, so small
// batches waited for the host.  Host time of a call: GDN step on slots, gates from a, b 18.9 -> 6 to 7 us, KDA step on plain
// tensors 16.5 -> 3.8; a layer of one GDN sequence, int8, launched so 18.1 -> 6 (its kernel alone 4.8, in a graph).
//
// Every function here takes exactly the calls that the Python code around it accepts in its ordinary form -- plain dense
// tensors on one GPU, the documented shapes -- and answers None to anything else (another tensor class, a tensor under a
// function transform, a CPU tensor, a wrong dtype or stride, a dict entry that is missing): the Python code then does the
// whole call itself, so what is refused, and with which message, is decided in one place.  Nothing is kept between calls.
//
// The extension uses torch's C++ classes, so it belongs to the torch it was built against: SQ_TORCH, the module's TORCH,
// names that version, and the Python side leaves a module of another one alone (every call then goes the Python way).
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>

#include <limits>

#include "../../include/statequant_hip.h"

namespace {

struct Library {
    int (*gdn_step)(const sq_gdn_args*, void*);
    int (*kda_step)(const sq_kda_args*, void*);
    int (*mamba2_step)(const sq_mamba2_args*, void*);
    int (*gga_step)(const sq_gga_args*, void*);
    int (*pack_vk)(const sq_pack_args*, void*);
    int (*read)(const sq_read_args*, void*);
} lib = {};

// The field names of a state dict, interned once.
enum Field { F_S, F_SC, F_KB, F_KBS, F_UB, F_UBS, F_GB, F_GCUR, F_NPTR, F_COUNT };
const char* const FIELD_NAMES[F_COUNT] = {"S", "SC", "KB", "KBS", "UB", "UBS", "GB", "GCUR", "NPTR"};
PyObject* field_name[F_COUNT];
PyObject* blob_name;

// "Not an ordinary call": the function returns false (or null, or a negative number) and the call ends as None.  Return
// values and no C++ exception: unwinding took 3.6 us of a call, a fifth of what the Python path behind it takes; now 0.15.
#define SQ_WANT(ok)                 \
    do {                            \
        if (!(ok)) return false;    \
    } while (0)

// A dense GPU tensor that is nothing else: no subclass, no wrapper of a transform, no lazy conjugate or negative.
const at::Tensor* plain(PyObject* o) {
    const PyTypeObject* const t = Py_TYPE(o);
    if (reinterpret_cast<const PyObject*>(t) != THPVariableClass && reinterpret_cast<const PyObject*>(t) != ParameterClass)
        return nullptr;
    static const uint64_t ordinary =
        (c10::DispatchKeySet(c10::BackendComponent::CUDABit) | c10::DispatchKeySet(c10::DispatchKey::Dense) |
         c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutogradFunctionality) |
         c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA)).raw_repr();
    const at::Tensor& x = THPVariable_Unpack(o);
    return x.defined() && (x.key_set().raw_repr() & ~ordinary) == 0 && x.is_cuda() ? &x : nullptr;
}
// ... on the GPU `dev`.
const at::Tensor* on(PyObject* o, c10::Device dev) {
    const at::Tensor* const x = plain(o);
    return x && x->device() == dev ? x : nullptr;
}
// `const at::Tensor& name`: the plain tensor `o` on `dev`, or the end of the function.
#define SQ_TENSOR(name, o, dev)                         \
    const at::Tensor* const name##_p = on((o), (dev));  \
    SQ_WANT(name##_p);                                  \
    const at::Tensor& name = *name##_p
int dtype_code(const at::Tensor& x) {
    switch (x.scalar_type()) {
        case at::kFloat: return SQ_F32;
        case at::kBFloat16: return SQ_BF16;
        case at::kHalf: return SQ_F16;
        default: return -1;
    }
}
// [rows, heads, d] with contiguous rows of heads: the row stride (else -1).
int64_t rows_of(const at::Tensor& x, int64_t d) {
    return x.dim() == 3 && x.stride(2) == 1 && x.stride(1) == d ? x.stride(0) : -1;
}
// [rows, heads]
int64_t rows_of(const at::Tensor& x) { return x.dim() == 2 && x.stride(1) == 1 ? x.stride(0) : -1; }
bool number(PyObject* o, double* v) {
    if (PyFloat_CheckExact(o)) {
        *v = PyFloat_AS_DOUBLE(o);
        return true;
    }
    SQ_WANT(PyLong_CheckExact(o));
    *v = PyLong_AsDouble(o);
    return !(*v == -1.0 && PyErr_Occurred());
}
bool number(PyObject* o, float* v) {
    double d;
    SQ_WANT(number(o, &d));
    *v = float(d);
    return true;
}
bool integer(PyObject* o, int32_t* out) {
    SQ_WANT(PyLong_CheckExact(o));
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    SQ_WANT(!overflow && v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max());
    *out = int32_t(v);
    return true;
}
// A ctypes struct's bytes.
template <class T>
bool struct_of(PyObject* o, T* v) {
    Py_buffer b;
    SQ_WANT(PyObject_CheckBuffer(o) && PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) == 0);
    const bool fits = b.len == Py_ssize_t(sizeof(T));
    if (fits) memcpy(v, b.buf, sizeof(T));
    PyBuffer_Release(&b);
    return fits;
}
// The slot indices and their number.
bool index_of(PyObject* o, c10::Device dev, const int32_t** idx, int32_t* rows) {
    SQ_TENSOR(x, o, dev);
    SQ_WANT(x.scalar_type() == at::kInt && x.dim() == 1 && x.is_contiguous() && x.size(0) > 0 &&
            x.size(0) <= std::numeric_limits<int32_t>::max());
    *idx = static_cast<const int32_t*>(x.data_ptr());
    *rows = int32_t(x.size(0));
    return true;
}
bool order_of(PyObject* o, int rows, c10::Device dev, const int32_t** order) {
    *order = nullptr;
    if (o == Py_None) return true;
    SQ_TENSOR(x, o, dev);
    SQ_WANT(x.scalar_type() == at::kInt && x.is_contiguous() && x.dim() >= 1 && x.size(0) >= rows);
    *order = static_cast<const int32_t*>(x.data_ptr());
    return true;
}

// The nine tensors of a state, and their per-sequence strides: the tensors' own (`strides` None: slot views) or the
// given ones (lockstep states: eight of them, and `counters` for the fill counters).
bool state_of(PyObject* fields, PyObject* strides, int64_t counters, sq_state* st, c10::Device* dev) {
    SQ_WANT(PyDict_CheckExact(fields));
    const at::Tensor* t[F_COUNT];
    for (int f = 0; f < F_COUNT; ++f) {
        PyObject* const o = PyDict_GetItemWithError(fields, field_name[f]);
        if (!o) {
            SQ_WANT(!PyErr_Occurred() && (f == F_SC || f == F_KBS || f == F_UBS));      // absent: no scales of that kind
            t[f] = nullptr;
        } else {
            t[f] = plain(o);
            SQ_WANT(t[f] && t[f]->dim() >= 1);
        }
    }
    *dev = t[F_S]->device();
    int64_t s[F_COUNT];
    if (strides == Py_None) {
        for (int f = 0; f < F_COUNT; ++f) s[f] = t[f] ? t[f]->stride(0) : 0;
    } else {
        SQ_WANT(PyTuple_CheckExact(strides) && PyTuple_GET_SIZE(strides) == F_COUNT - 1);
        for (int f = 0; f < F_NPTR; ++f) {
            int32_t v;
            SQ_WANT(integer(PyTuple_GET_ITEM(strides, f), &v));
            s[f] = v;
        }
        s[F_NPTR] = counters;
    }
    auto ptr = [&](int f) { return (t[f] ? t[f] : t[F_GB])->data_ptr(); };
    st->S = ptr(F_S);                               st->sS = s[F_S];
    st->SC = ptr(F_SC);                             st->sSC = s[F_SC];
    st->KB = ptr(F_KB);                             st->sKB = s[F_KB];
    st->KBS = ptr(F_KBS);                           st->sKBS = s[F_KBS];
    st->UB = ptr(F_UB);                             st->sUB = s[F_UB];
    st->UBS = ptr(F_UBS);                           st->sUBS = s[F_UBS];
    st->GB = static_cast<float*>(ptr(F_GB));        st->sGB = s[F_GB];
    st->GCUR = static_cast<float*>(ptr(F_GCUR));    st->sGC = s[F_GCUR];
    st->NPTR = static_cast<int32_t*>(ptr(F_NPTR));  st->sN = s[F_NPTR];
    return true;
}

// The call itself, on the current stream; the interpreter is free meanwhile (a full queue makes a launch wait).
template <class Args>
bool launch(int (*fn)(const Args*, void*), const Args& a, c10::Device dev, PyObject** result) {
    SQ_WANT(fn != nullptr);
    void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(&a, stream);
    Py_END_ALLOW_THREADS
    *result = PyLong_FromLong(rc);
    return true;
}

// A float operand: pointer, row stride and dtype of x.
#define SQ_VEC(a, name, x, stride)                                          \
    do {                                                                    \
        (a).name = (x).data_ptr();                                          \
        (a).s_##name = (stride);                                            \
        (a).name##_dtype = dtype_code(x);                                   \
        SQ_WANT((a).s_##name >= 0 && (a).name##_dtype >= 0);                \
    } while (0)
// The same without a stride.
#define SQ_FLAT(a, name, x)                                                 \
    do {                                                                    \
        (a).name = (x).data_ptr();                                          \
        (a).name##_dtype = dtype_code(x);                                   \
        SQ_WANT((a).name##_dtype >= 0);                                     \
    } while (0)

// gate = (a, b, A_log, dt_bias), or g and beta
template <class Args>
bool gate_of(Args& a, PyObject* g, PyObject* beta, PyObject* gate, c10::Device dev) {
    if (gate != Py_None) {
        SQ_WANT(g == Py_None && beta == Py_None && PyTuple_CheckExact(gate) && PyTuple_GET_SIZE(gate) == 4);
        SQ_TENSOR(ga, PyTuple_GET_ITEM(gate, 0), dev);
        SQ_TENSOR(gb, PyTuple_GET_ITEM(gate, 1), dev);
        SQ_TENSOR(A_log, PyTuple_GET_ITEM(gate, 2), dev);
        SQ_TENSOR(dt_bias, PyTuple_GET_ITEM(gate, 3), dev);
        SQ_WANT(A_log.is_contiguous() && dt_bias.is_contiguous());
        a.gate = 1;
        SQ_VEC(a, a, ga, rows_of(ga));
        SQ_VEC(a, b, gb, rows_of(gb));
        SQ_FLAT(a, A_log, A_log);
        SQ_FLAT(a, dt_bias, dt_bias);
    } else {
        SQ_TENSOR(tg, g, dev);
        SQ_TENSOR(tb, beta, dev);
        a.gate = 0;
        SQ_VEC(a, g, tg, rows_of(tg));
        SQ_VEC(a, beta, tb, rows_of(tb));
    }
    return true;
}

// gdn_step(lay, views, idx, q, k, v, out, scale, g, beta, gate, order)
bool gdn_step(PyObject* const* v, PyObject** result) {
    sq_gdn_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], Py_None, 0, &a.st, &dev));
    SQ_WANT(index_of(v[2], dev, &a.idx, &a.rows));
    SQ_TENSOR(q, v[3], dev);
    SQ_TENSOR(k, v[4], dev);
    SQ_TENSOR(vv, v[5], dev);
    SQ_TENSOR(out, v[6], dev);
    SQ_VEC(a, q, q, rows_of(q, a.lay.dk));
    SQ_VEC(a, k, k, rows_of(k, a.lay.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.lay.dv));
    a.qk_per_key_head = 1;
    SQ_WANT(out.is_contiguous() && out.dim() >= 1 && out.size(0) >= a.rows);
    SQ_FLAT(a, out, out);
    SQ_WANT(number(v[7], &a.scale));
    SQ_WANT(gate_of(a, v[8], v[9], v[10], dev));
    SQ_WANT(order_of(v[11], a.rows, dev, &a.order));
    return launch(lib.gdn_step, a, dev, result);
}

// gdn_lockstep(lay, fields, strides, rows, q, k, v, g, beta, out, scale): contiguous tensors, q and k per key head or
// per value head
bool gdn_lockstep(PyObject* const* v, PyObject** result) {
    sq_gdn_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    SQ_WANT(integer(v[3], &a.rows));
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], v[2], a.lay.hv, &a.st, &dev));
    SQ_TENSOR(q, v[4], dev);
    SQ_TENSOR(k, v[5], dev);
    SQ_TENSOR(vv, v[6], dev);
    SQ_TENSOR(g, v[7], dev);
    SQ_TENSOR(beta, v[8], dev);
    SQ_TENSOR(out, v[9], dev);
    SQ_WANT(q.is_contiguous() && k.is_contiguous() && vv.is_contiguous() && g.is_contiguous() && beta.is_contiguous());
    SQ_WANT(q.dim() >= 1 && k.dim() >= 1);
    const int64_t heads = int64_t(a.rows) * a.lay.hv, keys = int64_t(a.rows) * a.lay.hk;
    a.qk_per_key_head = q.size(0) != heads;
    SQ_WANT(!a.qk_per_key_head || (q.size(0) == keys && k.size(0) == keys));
    const int64_t sqk = int64_t(a.qk_per_key_head ? a.lay.hk : a.lay.hv) * a.lay.dk;
    SQ_VEC(a, q, q, sqk);
    SQ_VEC(a, k, k, sqk);
    SQ_VEC(a, v, vv, int64_t(a.lay.hv) * a.lay.dv);
    SQ_VEC(a, g, g, a.lay.hv);
    SQ_VEC(a, beta, beta, a.lay.hv);
    SQ_FLAT(a, out, out);
    SQ_WANT(number(v[10], &a.scale));
    return launch(lib.gdn_step, a, dev, result);
}

// kda_step(lay, views, idx, q, k, v, g, beta, out, scale, order)
bool kda_step(PyObject* const* v, PyObject** result) {
    sq_kda_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], Py_None, 0, &a.st, &dev));
    SQ_WANT(index_of(v[2], dev, &a.idx, &a.rows));
    SQ_TENSOR(q, v[3], dev);
    SQ_TENSOR(k, v[4], dev);
    SQ_TENSOR(vv, v[5], dev);
    SQ_TENSOR(g, v[6], dev);
    SQ_TENSOR(beta, v[7], dev);
    SQ_TENSOR(out, v[8], dev);
    SQ_VEC(a, q, q, rows_of(q, a.lay.dk));
    SQ_VEC(a, k, k, rows_of(k, a.lay.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.lay.dv));
    SQ_VEC(a, g, g, rows_of(g, a.lay.dk));
    SQ_VEC(a, beta, beta, rows_of(beta));
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    SQ_WANT(number(v[9], &a.scale));
    SQ_WANT(order_of(v[10], a.rows, dev, &a.order));
    return launch(lib.kda_step, a, dev, result);
}

// A tensor that flattens to rows x n as a view (what `reshape` of a contiguous tensor gives).
const at::Tensor* flat(PyObject* o, c10::Device dev, int64_t numel) {
    const at::Tensor* const x = on(o, dev);
    return x && x->is_contiguous() && x->numel() == numel ? x : nullptr;
}
#define SQ_ROWS(a, name, o, dev, per_row)                                   \
    do {                                                                    \
        const at::Tensor* const x_ = flat((o), (dev), (a).rows * (per_row)); \
        SQ_WANT(x_);                                                        \
        SQ_VEC(a, name, *x_, (per_row));                                    \
    } while (0)

// kda_lockstep(lay, fields, strides, rows, q, k, v, g, beta, out, scale)
bool kda_lockstep(PyObject* const* v, PyObject** result) {
    sq_kda_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    SQ_WANT(integer(v[3], &a.rows));
    SQ_WANT(a.rows > 0);
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], v[2], a.lay.hv, &a.st, &dev));
    const int64_t nk = int64_t(a.lay.hv) * a.lay.dk, nv = int64_t(a.lay.hv) * a.lay.dv;
    SQ_ROWS(a, q, v[4], dev, nk);
    SQ_ROWS(a, k, v[5], dev, nk);
    SQ_ROWS(a, v, v[6], dev, nv);
    SQ_ROWS(a, g, v[7], dev, nk);
    SQ_ROWS(a, beta, v[8], dev, int64_t(a.lay.hv));
    SQ_TENSOR(out, v[9], dev);
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    SQ_WANT(number(v[10], &a.scale));
    return launch(lib.kda_step, a, dev, result);
}

bool mamba2_model(sq_mamba2_args& a, PyObject* A, PyObject* D, PyObject* dt_bias, PyObject* softplus, PyObject* limit,
                  c10::Device dev) {
    SQ_TENSOR(tA, A, dev);
    SQ_WANT(tA.is_contiguous());
    SQ_FLAT(a, A, tA);
    if (D != Py_None) {
        SQ_TENSOR(t, D, dev);
        SQ_WANT(t.is_contiguous());
        SQ_FLAT(a, D, t);
    }
    if (dt_bias != Py_None) {
        SQ_TENSOR(t, dt_bias, dev);
        SQ_WANT(t.is_contiguous());
        SQ_FLAT(a, dt_bias, t);
    }
    SQ_WANT(PyBool_Check(softplus));
    a.dt_softplus = softplus == Py_True;
    if (limit != Py_None) {
        double lo, hi;
        SQ_WANT(PyTuple_CheckExact(limit) && PyTuple_GET_SIZE(limit) == 2 && number(PyTuple_GET_ITEM(limit, 0), &lo) &&
                number(PyTuple_GET_ITEM(limit, 1), &hi));
        if (!(lo == 0.0 && hi == std::numeric_limits<double>::infinity())) {
            a.dt_clamp = 1;
            a.dt_min = float(lo);
            a.dt_max = float(hi);
        }
    }
    return true;
}

// mamba2_step(lay, views, idx, x, dt, B, C, out, A, D, dt_bias, dt_softplus, dt_limit, order)
bool mamba2_step(PyObject* const* v, PyObject** result) {
    sq_mamba2_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], Py_None, 0, &a.st, &dev));
    SQ_WANT(index_of(v[2], dev, &a.idx, &a.rows));
    SQ_TENSOR(x, v[3], dev);
    SQ_TENSOR(dt, v[4], dev);
    SQ_TENSOR(B, v[5], dev);
    SQ_TENSOR(C, v[6], dev);
    SQ_TENSOR(out, v[7], dev);
    SQ_VEC(a, x, x, rows_of(x, a.lay.dv));
    SQ_VEC(a, dt, dt, rows_of(dt));
    SQ_VEC(a, B, B, rows_of(B, a.lay.dk));
    SQ_VEC(a, C, C, rows_of(C, a.lay.dk));
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    SQ_WANT(mamba2_model(a, v[8], v[9], v[10], v[11], v[12], dev));
    SQ_WANT(order_of(v[13], a.rows, dev, &a.order));
    return launch(lib.mamba2_step, a, dev, result);
}

// mamba2_lockstep(lay, fields, strides, rows, x, dt, B, C, out, A, D, dt_bias, dt_softplus, dt_limit)
bool mamba2_lockstep(PyObject* const* v, PyObject** result) {
    sq_mamba2_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    SQ_WANT(integer(v[3], &a.rows));
    SQ_WANT(a.rows > 0);
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], v[2], a.lay.hv, &a.st, &dev));
    const int64_t nk = int64_t(a.lay.hk) * a.lay.dk, nv = int64_t(a.lay.hv) * a.lay.dv;
    SQ_ROWS(a, x, v[4], dev, nv);
    SQ_ROWS(a, dt, v[5], dev, int64_t(a.lay.hv));
    SQ_ROWS(a, B, v[6], dev, nk);
    SQ_ROWS(a, C, v[7], dev, nk);
    SQ_TENSOR(out, v[8], dev);
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    SQ_WANT(mamba2_model(a, v[9], v[10], v[11], v[12], v[13], dev));
    return launch(lib.mamba2_step, a, dev, result);
}

// gga_step(slots, views, plan, idx, q, k, v, out, scale, g, beta, gate): `slots` an sq_gga_slots without its pointers,
// `plan` the layer's (offsets, widths, impact factors) on the device
bool gga_step(PyObject* const* v, PyObject** result) {
    sq_gga_args a = {};
    SQ_WANT(struct_of(v[0], &a.sl));
    SQ_WANT(PyDict_CheckExact(v[1]));
    PyObject* const blob_obj = PyDict_GetItemWithError(v[1], blob_name);
    SQ_WANT(blob_obj);
    const at::Tensor* const blob_p = plain(blob_obj);
    SQ_WANT(blob_p && blob_p->dim() == 2);
    const at::Tensor& blob = *blob_p;
    const c10::Device dev = blob.device();
    a.sl.blob = blob.data_ptr();
    a.sl.slot_stride = blob.stride(0);
    SQ_WANT(PyTuple_CheckExact(v[2]) && PyTuple_GET_SIZE(v[2]) == 3);
    SQ_TENSOR(offs, PyTuple_GET_ITEM(v[2], 0), dev);
    SQ_TENSOR(bits, PyTuple_GET_ITEM(v[2], 1), dev);
    SQ_TENSOR(w, PyTuple_GET_ITEM(v[2], 2), dev);
    a.sl.offs = static_cast<const int32_t*>(offs.data_ptr());
    a.sl.bits = static_cast<const int32_t*>(bits.data_ptr());
    a.sl.w = static_cast<const float*>(w.data_ptr());
    SQ_WANT(index_of(v[3], dev, &a.idx, &a.rows));
    SQ_TENSOR(q, v[4], dev);
    SQ_TENSOR(k, v[5], dev);
    SQ_TENSOR(vv, v[6], dev);
    SQ_TENSOR(out, v[7], dev);
    SQ_VEC(a, q, q, rows_of(q, a.sl.dk));
    SQ_VEC(a, k, k, rows_of(k, a.sl.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.sl.dv));
    SQ_WANT(out.is_contiguous() && out.dim() == 3 && out.size(0) >= a.rows && out.size(1) == a.sl.hv && out.size(2) == a.sl.dv);
    SQ_FLAT(a, out, out);
    SQ_WANT(number(v[8], &a.scale));
    SQ_WANT(gate_of(a, v[9], v[10], v[11], dev));
    return launch(lib.gga_step, a, dev, result);
}

// write(lay, views, idx, src): fp32 states [rows, hv, dv, dk], contiguous, into slots
bool write_slots(PyObject* const* v, PyObject** result) {
    sq_pack_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    c10::Device dev(c10::kCPU);
    sq_state st;
    SQ_WANT(state_of(v[1], Py_None, 0, &st, &dev));
    SQ_WANT(index_of(v[2], dev, &a.idx, &a.rows));
    const int64_t per_row = int64_t(a.lay.hv) * a.lay.dv * a.lay.dk;
    const at::Tensor* const src = flat(v[3], dev, a.rows * per_row);
    SQ_WANT(src && src->scalar_type() == at::kFloat);
    a.src = static_cast<const float*>(src->data_ptr());
    a.s_src = per_row;
    a.S = st.S;         a.sS = st.sS;
    const bool scaled = PyDict_GetItem(v[1], field_name[F_SC]) != nullptr;
    a.SC = scaled ? st.SC : nullptr;
    a.sSC = scaled ? st.sSC : 0;
    const at::Tensor& decay = THPVariable_Unpack(PyDict_GetItem(v[1], field_name[F_GCUR]));
    const at::Tensor& fill = THPVariable_Unpack(PyDict_GetItem(v[1], field_name[F_NPTR]));
    SQ_WANT(decay.size(0) > 0 && fill.size(0) > 0);
    a.GCUR = st.GCUR;   a.sGC = st.sGC;
    a.gcur_per_head = int32_t(decay.numel() / decay.size(0) / a.lay.hv);
    a.NPTR = st.NPTR;   a.sN = st.sN;
    a.nptr_copies = int32_t(fill.numel() / fill.size(0));
    return launch(lib.pack_vk, a, dev, result);
}

// read(lay, views, idx, kda) -> (status, fp32 states [rows, hv, dv, dk])
bool read_slots(PyObject* const* v, PyObject** result) {
    sq_read_args a = {};
    SQ_WANT(struct_of(v[0], &a.lay));
    c10::Device dev(c10::kCPU);
    SQ_WANT(state_of(v[1], Py_None, 0, &a.st, &dev));
    SQ_WANT(index_of(v[2], dev, &a.idx, &a.rows));
    SQ_WANT(PyBool_Check(v[3]));
    a.kda = v[3] == Py_True;
    at::Tensor out = at::empty({a.rows, a.lay.hv, a.lay.dv, a.lay.dk}, at::TensorOptions().dtype(at::kFloat).device(dev));
    SQ_WANT(!out.key_set().has(c10::DispatchKey::Python));
    a.out = static_cast<float*>(out.data_ptr());
    a.s_out = out.stride(0);
    PyObject* rc = nullptr;
    SQ_WANT(launch(lib.read, a, dev, &rc));
    PyObject* const t = rc ? THPVariable_Wrap(std::move(out)) : nullptr;
    *result = t ? PyTuple_Pack(2, rc, t) : nullptr;
    Py_XDECREF(rc);
    Py_XDECREF(t);
    return true;
}

// views(blob, fields, nbytes): the typed views {name: [slots, *shape]} of a blob, cut as the Python code cuts them (slice,
// dtype, shape) but without the interpreter between the 27 operations: 23 us of a decode step's 24 calls for one sequence
// went into the views that a program takes of its updated blob.
bool slot_views(PyObject* const* v, PyObject** result) {
    constexpr int64_t ALIGN = 16;
    const at::Tensor* const blob_p = plain(v[0]);
    int32_t nbytes;
    SQ_WANT(blob_p && !at::impl::torch_function_mode_enabled() && PyDict_CheckExact(v[1]) && integer(v[2], &nbytes));
    const at::Tensor& blob = *blob_p;
    SQ_WANT(blob.scalar_type() == at::kByte && blob.dim() == 2 && blob.size(1) >= nbytes && blob.stride(1) == 1 &&
            blob.stride(0) % ALIGN == 0 && reinterpret_cast<uintptr_t>(blob.data_ptr()) % ALIGN == 0);
    PyObject* const views = PyDict_New();
    if (!views) return true;                                   // (with a Python error set)
    PyObject *name, *field;
    Py_ssize_t at = 0;
    auto cut = [&]() {
        int32_t off, size, d;
        SQ_WANT(PyTuple_CheckExact(field) && PyTuple_GET_SIZE(field) == 4);
        PyObject* const dtype = PyTuple_GET_ITEM(field, 1);
        PyObject* const shape = PyTuple_GET_ITEM(field, 2);
        SQ_WANT(integer(PyTuple_GET_ITEM(field, 0), &off) && integer(PyTuple_GET_ITEM(field, 3), &size) && THPDtype_Check(dtype) &&
                PyTuple_CheckExact(shape));
        c10::SmallVector<int64_t, 4> sizes{blob.size(0)};
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); ++i) {
            SQ_WANT(integer(PyTuple_GET_ITEM(shape, i), &d));
            sizes.push_back(d);
        }
        PyObject* const t = THPVariable_Wrap(
            blob.slice(1, off, int64_t(off) + size).view(reinterpret_cast<THPDtype*>(dtype)->scalar_type).view(sizes));
        const bool kept = t && PyDict_SetItem(views, name, t) == 0;
        Py_XDECREF(t);
        return kept;
    };
    bool whole = true;
    try {
        while (whole && PyDict_Next(v[1], &at, &name, &field)) whole = cut();
    } catch (...) {                                            // (whatever torch refuses, the Python code refuses)
        whole = false;
    }
    if (!whole) {
        Py_DECREF(views);
        return false;
    }
    *result = views;
    return true;
}

// The functions above behind Python's calling convention: N arguments; None for whatever is not an ordinary call, a C++
// exception (out of memory in `read`, say: the Python path then meets it too) included.
template <bool (*FN)(PyObject* const*, PyObject**), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", N, n);
        return nullptr;
    }
    try {
        PyObject* result = nullptr;
        if (FN(args, &result)) return result;                 // (null: with a Python error set)
    } catch (...) {
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

// init(addresses of sq_gdn_step, sq_kda_step, sq_mamba2_step, sq_gga_step, sq_pack_vk, sq_read)
PyObject* init(PyObject*, PyObject* const* args, Py_ssize_t n) {
    void* p[6];
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "six function addresses expected");
        return nullptr;
    }
    for (int i = 0; i < 6; ++i) {
        p[i] = PyLong_AsVoidPtr(args[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    lib.gdn_step = reinterpret_cast<decltype(lib.gdn_step)>(p[0]);
    lib.kda_step = reinterpret_cast<decltype(lib.kda_step)>(p[1]);
    lib.mamba2_step = reinterpret_cast<decltype(lib.mamba2_step)>(p[2]);
    lib.gga_step = reinterpret_cast<decltype(lib.gga_step)>(p[3]);
    lib.pack_vk = reinterpret_cast<decltype(lib.pack_vk)>(p[4]);
    lib.read = reinterpret_cast<decltype(lib.read)>(p[5]);
    Py_RETURN_NONE;
}

#define SQ_ENTRY(name, fn, n) \
    {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<fn, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"init", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&init)), METH_FASTCALL, nullptr},
    SQ_ENTRY("gdn_step", gdn_step, 12),
    SQ_ENTRY("gdn_lockstep", gdn_lockstep, 11),
    SQ_ENTRY("kda_step", kda_step, 11),
    SQ_ENTRY("kda_lockstep", kda_lockstep, 11),
    SQ_ENTRY("mamba2_step", mamba2_step, 14),
    SQ_ENTRY("mamba2_lockstep", mamba2_lockstep, 14),
    SQ_ENTRY("gga_step", gga_step, 12),
    SQ_ENTRY("write", write_slots, 4),
    SQ_ENTRY("read", read_slots, 4),
    SQ_ENTRY("views", slot_views, 3),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sqhost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sqhost() {
    for (int f = 0; f < F_COUNT; ++f)
        if (!(field_name[f] = PyUnicode_InternFromString(FIELD_NAMES[f]))) return nullptr;
    if (!(blob_name = PyUnicode_InternFromString("blob"))) return nullptr;
    PyObject* const m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "TORCH", SQ_TORCH) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
