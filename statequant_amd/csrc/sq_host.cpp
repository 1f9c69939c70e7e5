// The Python side's calls into libsqhip.so, in native code: argument checks, the C ABI's structs and the launch of one
// decode step (or state hand-over) without an interpreted instruction in between.
//
// What it is for: a decode step calls the library once per layer, and reading some twenty tensors' pointers, strides and
// dtypes through Python took 17.5 us per call -- four times as long as the kernel itself runs for one sequence, so small
// batches waited for the host.  24 GDN layers, int8: 1 sequence 430 -> 155 us, 13 sequences (int4) 433 -> 198; six KDA
// layers in lockstep 103 -> 36 (5.4 to 6.5 us of each call is the kernel itself).
//
// Every function here takes exactly the calls that the Python code around it accepts in its ordinary form -- plain dense
// tensors on one GPU, the documented shapes -- and answers None to anything else (another tensor class, a tensor under a
// function transform, a CPU tensor, a wrong dtype or stride, a dict entry that is missing): the Python code then does the
// whole call itself, so what is refused, and with which message, is decided in one place.  Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
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

struct Other {};                                   // "not an ordinary call": ends as None
[[noreturn]] void other() { throw Other{}; }
inline void want(bool ok) { if (!ok) other(); }

// A dense GPU tensor that is nothing else: no subclass, no wrapper of a transform, no lazy conjugate or negative.
const at::Tensor& plain(PyObject* o) {
    const PyTypeObject* const t = Py_TYPE(o);
    want(reinterpret_cast<const PyObject*>(t) == THPVariableClass || reinterpret_cast<const PyObject*>(t) == ParameterClass);
    static const uint64_t ordinary =
        (c10::DispatchKeySet(c10::BackendComponent::CUDABit) | c10::DispatchKeySet(c10::DispatchKey::Dense) |
         c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutogradFunctionality) |
         c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA)).raw_repr();
    const at::Tensor& x = THPVariable_Unpack(o);
    want(x.defined() && (x.key_set().raw_repr() & ~ordinary) == 0 && x.is_cuda());
    return x;
}
// ... on the GPU `dev`.
const at::Tensor& on(PyObject* o, c10::Device dev) {
    const at::Tensor& x = plain(o);
    want(x.device() == dev);
    return x;
}
int dtype_code(const at::Tensor& x) {
    switch (x.scalar_type()) {
        case at::kFloat: return SQ_F32;
        case at::kBFloat16: return SQ_BF16;
        case at::kHalf: return SQ_F16;
        default: other();
    }
}
// [rows, heads, d] with contiguous rows of heads; returns the row stride.
int64_t rows_of(const at::Tensor& x, int64_t d) {
    want(x.dim() == 3 && x.stride(2) == 1 && x.stride(1) == d);
    return x.stride(0);
}
// [rows, heads]
int64_t rows_of(const at::Tensor& x) {
    want(x.dim() == 2 && x.stride(1) == 1);
    return x.stride(0);
}
double number(PyObject* o) {
    if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
    want(PyLong_CheckExact(o));
    const double v = PyLong_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); other(); }
    return v;
}
int32_t integer(PyObject* o) {
    want(PyLong_CheckExact(o));
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    want(!overflow && v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max());
    return int32_t(v);
}
// A ctypes struct's bytes.
template <class T>
T struct_of(PyObject* o) {
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) { PyErr_Clear(); other(); }
    T v;
    const bool fits = b.len == Py_ssize_t(sizeof(T));
    if (fits) memcpy(&v, b.buf, sizeof(T));
    PyBuffer_Release(&b);
    want(fits);
    return v;
}
int rows_of_index(const at::Tensor& idx) {
    want(idx.scalar_type() == at::kInt && idx.dim() == 1 && idx.is_contiguous() && idx.size(0) > 0 &&
         idx.size(0) <= std::numeric_limits<int32_t>::max());
    return int(idx.size(0));
}
const int32_t* order_of(PyObject* o, int rows, c10::Device dev) {
    if (o == Py_None) return nullptr;
    const at::Tensor& x = on(o, dev);
    want(x.scalar_type() == at::kInt && x.is_contiguous() && x.dim() >= 1 && x.size(0) >= rows);
    return static_cast<const int32_t*>(x.data_ptr());
}

// The nine tensors of a state, and their per-sequence strides: the tensors' own (`strides` None: slot views) or the
// given ones (lockstep states: eight of them, and `counters` for the fill counters).
sq_state state_of(PyObject* fields, PyObject* strides, int64_t counters, c10::Device* dev) {
    want(PyDict_CheckExact(fields));
    const at::Tensor* t[F_COUNT];
    for (int f = 0; f < F_COUNT; ++f) {
        PyObject* o = PyDict_GetItemWithError(fields, field_name[f]);
        if (!o) {
            if (PyErr_Occurred()) { PyErr_Clear(); other(); }
            want(f == F_SC || f == F_KBS || f == F_UBS);          // absent: no scales of that kind
            t[f] = nullptr;
        } else {
            t[f] = &plain(o);
            want(t[f]->dim() >= 1);
        }
    }
    *dev = t[F_S]->device();
    int64_t s[F_COUNT];
    if (strides == Py_None) {
        for (int f = 0; f < F_COUNT; ++f) s[f] = t[f] ? t[f]->stride(0) : 0;
    } else {
        want(PyTuple_CheckExact(strides) && PyTuple_GET_SIZE(strides) == F_COUNT - 1);
        for (int f = 0; f < F_NPTR; ++f) s[f] = integer(PyTuple_GET_ITEM(strides, f));
        s[F_NPTR] = counters;
    }
    auto ptr = [&](int f) { return (t[f] ? t[f] : t[F_GB])->data_ptr(); };
    sq_state st;
    st.S = ptr(F_S);                               st.sS = s[F_S];
    st.SC = ptr(F_SC);                             st.sSC = s[F_SC];
    st.KB = ptr(F_KB);                             st.sKB = s[F_KB];
    st.KBS = ptr(F_KBS);                           st.sKBS = s[F_KBS];
    st.UB = ptr(F_UB);                             st.sUB = s[F_UB];
    st.UBS = ptr(F_UBS);                           st.sUBS = s[F_UBS];
    st.GB = static_cast<float*>(ptr(F_GB));        st.sGB = s[F_GB];
    st.GCUR = static_cast<float*>(ptr(F_GCUR));    st.sGC = s[F_GCUR];
    st.NPTR = static_cast<int32_t*>(ptr(F_NPTR));  st.sN = s[F_NPTR];
    return st;
}

// The call itself, on the current stream; the interpreter is free meanwhile (a full queue makes a launch wait).
template <class Args>
PyObject* launch(int (*fn)(const Args*, void*), const Args& a, c10::Device dev) {
    want(fn != nullptr);
    void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(&a, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

#define SQ_VEC(a, name, x, stride)                              \
    do {                                                        \
        (a).name = (x).data_ptr();                              \
        (a).s_##name = (stride);                                \
        (a).name##_dtype = dtype_code(x);                       \
    } while (0)

// gate = (a, b, A_log, dt_bias), or g and beta
template <class Args>
void gate_of(Args& a, PyObject* g, PyObject* beta, PyObject* gate, c10::Device dev) {
    if (gate != Py_None) {
        want(g == Py_None && beta == Py_None && PyTuple_CheckExact(gate) && PyTuple_GET_SIZE(gate) == 4);
        const at::Tensor& ga = on(PyTuple_GET_ITEM(gate, 0), dev);
        const at::Tensor& gb = on(PyTuple_GET_ITEM(gate, 1), dev);
        const at::Tensor& A_log = on(PyTuple_GET_ITEM(gate, 2), dev);
        const at::Tensor& dt_bias = on(PyTuple_GET_ITEM(gate, 3), dev);
        want(A_log.is_contiguous() && dt_bias.is_contiguous());
        a.gate = 1;
        SQ_VEC(a, a, ga, rows_of(ga));
        SQ_VEC(a, b, gb, rows_of(gb));
        a.A_log = A_log.data_ptr();
        a.A_log_dtype = dtype_code(A_log);
        a.dt_bias = dt_bias.data_ptr();
        a.dt_bias_dtype = dtype_code(dt_bias);
    } else {
        const at::Tensor& tg = on(g, dev);
        const at::Tensor& tb = on(beta, dev);
        a.gate = 0;
        SQ_VEC(a, g, tg, rows_of(tg));
        SQ_VEC(a, beta, tb, rows_of(tb));
    }
}

// gdn_step(lay, views, idx, q, k, v, out, scale, g, beta, gate, order)
PyObject* gdn_step(PyObject* const* v) {
    sq_gdn_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], Py_None, 0, &dev);
    const at::Tensor& idx = on(v[2], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    const at::Tensor &q = on(v[3], dev), &k = on(v[4], dev), &vv = on(v[5], dev), &out = on(v[6], dev);
    SQ_VEC(a, q, q, rows_of(q, a.lay.dk));
    SQ_VEC(a, k, k, rows_of(k, a.lay.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.lay.dv));
    a.qk_per_key_head = 1;
    want(out.is_contiguous() && out.dim() >= 1 && out.size(0) >= a.rows);
    a.out = out.data_ptr();
    a.out_dtype = dtype_code(out);
    a.scale = float(number(v[7]));
    gate_of(a, v[8], v[9], v[10], dev);
    a.order = order_of(v[11], a.rows, dev);
    return launch(lib.gdn_step, a, dev);
}

// gdn_lockstep(lay, fields, strides, rows, q, k, v, g, beta, out, scale): contiguous tensors, q and k per key head or
// per value head
PyObject* gdn_lockstep(PyObject* const* v) {
    sq_gdn_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    a.rows = integer(v[3]);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], v[2], a.lay.hv, &dev);
    const at::Tensor &q = on(v[4], dev), &k = on(v[5], dev), &vv = on(v[6], dev), &g = on(v[7], dev), &beta = on(v[8], dev);
    const at::Tensor& out = on(v[9], dev);
    want(q.is_contiguous() && k.is_contiguous() && vv.is_contiguous() && g.is_contiguous() && beta.is_contiguous());
    want(q.dim() >= 1 && k.dim() >= 1);
    const int64_t heads = int64_t(a.rows) * a.lay.hv, keys = int64_t(a.rows) * a.lay.hk;
    a.qk_per_key_head = q.size(0) != heads;
    want(!a.qk_per_key_head || (q.size(0) == keys && k.size(0) == keys));
    const int64_t sqk = int64_t(a.qk_per_key_head ? a.lay.hk : a.lay.hv) * a.lay.dk;
    SQ_VEC(a, q, q, sqk);
    SQ_VEC(a, k, k, sqk);
    SQ_VEC(a, v, vv, int64_t(a.lay.hv) * a.lay.dv);
    SQ_VEC(a, g, g, a.lay.hv);
    SQ_VEC(a, beta, beta, a.lay.hv);
    a.out = out.data_ptr();
    a.out_dtype = dtype_code(out);
    a.scale = float(number(v[10]));
    return launch(lib.gdn_step, a, dev);
}

// kda_step(lay, views, idx, q, k, v, g, beta, out, scale, order)
PyObject* kda_step(PyObject* const* v) {
    sq_kda_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], Py_None, 0, &dev);
    const at::Tensor& idx = on(v[2], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    const at::Tensor &q = on(v[3], dev), &k = on(v[4], dev), &vv = on(v[5], dev), &g = on(v[6], dev), &beta = on(v[7], dev);
    const at::Tensor& out = on(v[8], dev);
    SQ_VEC(a, q, q, rows_of(q, a.lay.dk));
    SQ_VEC(a, k, k, rows_of(k, a.lay.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.lay.dv));
    SQ_VEC(a, g, g, rows_of(g, a.lay.dk));
    SQ_VEC(a, beta, beta, rows_of(beta));
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    a.scale = float(number(v[9]));
    a.order = order_of(v[10], a.rows, dev);
    return launch(lib.kda_step, a, dev);
}

// A tensor that flattens to rows x n as a view (what `reshape` of a contiguous tensor gives).
const at::Tensor& flat(PyObject* o, c10::Device dev, int64_t numel) {
    const at::Tensor& x = on(o, dev);
    want(x.is_contiguous() && x.numel() == numel);
    return x;
}

// kda_lockstep(lay, fields, strides, rows, q, k, v, g, beta, out, scale)
PyObject* kda_lockstep(PyObject* const* v) {
    sq_kda_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    a.rows = integer(v[3]);
    want(a.rows > 0);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], v[2], a.lay.hv, &dev);
    const int64_t nk = int64_t(a.lay.hv) * a.lay.dk, nv = int64_t(a.lay.hv) * a.lay.dv;
    SQ_VEC(a, q, flat(v[4], dev, a.rows * nk), nk);
    SQ_VEC(a, k, flat(v[5], dev, a.rows * nk), nk);
    SQ_VEC(a, v, flat(v[6], dev, a.rows * nv), nv);
    SQ_VEC(a, g, flat(v[7], dev, a.rows * nk), nk);
    SQ_VEC(a, beta, flat(v[8], dev, int64_t(a.rows) * a.lay.hv), a.lay.hv);
    const at::Tensor& out = on(v[9], dev);
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    a.scale = float(number(v[10]));
    return launch(lib.kda_step, a, dev);
}

void mamba2_model(sq_mamba2_args& a, PyObject* A, PyObject* D, PyObject* dt_bias, PyObject* softplus, PyObject* limit,
                  c10::Device dev) {
    const at::Tensor& tA = on(A, dev);
    want(tA.is_contiguous());
    a.A = tA.data_ptr();
    a.A_dtype = dtype_code(tA);
    if (D != Py_None) {
        const at::Tensor& t = on(D, dev);
        want(t.is_contiguous());
        a.D = t.data_ptr();
        a.D_dtype = dtype_code(t);
    }
    if (dt_bias != Py_None) {
        const at::Tensor& t = on(dt_bias, dev);
        want(t.is_contiguous());
        a.dt_bias = t.data_ptr();
        a.dt_bias_dtype = dtype_code(t);
    }
    want(PyBool_Check(softplus));
    a.dt_softplus = softplus == Py_True;
    if (limit != Py_None) {
        want(PyTuple_CheckExact(limit) && PyTuple_GET_SIZE(limit) == 2);
        const double lo = number(PyTuple_GET_ITEM(limit, 0)), hi = number(PyTuple_GET_ITEM(limit, 1));
        if (!(lo == 0.0 && hi == std::numeric_limits<double>::infinity())) {
            a.dt_clamp = 1;
            a.dt_min = float(lo);
            a.dt_max = float(hi);
        }
    }
}

// mamba2_step(lay, views, idx, x, dt, B, C, out, A, D, dt_bias, dt_softplus, dt_limit, order)
PyObject* mamba2_step(PyObject* const* v) {
    sq_mamba2_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], Py_None, 0, &dev);
    const at::Tensor& idx = on(v[2], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    const at::Tensor &x = on(v[3], dev), &dt = on(v[4], dev), &B = on(v[5], dev), &C = on(v[6], dev), &out = on(v[7], dev);
    SQ_VEC(a, x, x, rows_of(x, a.lay.dv));
    SQ_VEC(a, dt, dt, rows_of(dt));
    SQ_VEC(a, B, B, rows_of(B, a.lay.dk));
    SQ_VEC(a, C, C, rows_of(C, a.lay.dk));
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    mamba2_model(a, v[8], v[9], v[10], v[11], v[12], dev);
    a.order = order_of(v[13], a.rows, dev);
    return launch(lib.mamba2_step, a, dev);
}

// mamba2_lockstep(lay, fields, strides, rows, x, dt, B, C, out, A, D, dt_bias, dt_softplus, dt_limit)
PyObject* mamba2_lockstep(PyObject* const* v) {
    sq_mamba2_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    a.rows = integer(v[3]);
    want(a.rows > 0);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], v[2], a.lay.hv, &dev);
    const int64_t nk = int64_t(a.lay.hk) * a.lay.dk, nv = int64_t(a.lay.hv) * a.lay.dv;
    SQ_VEC(a, x, flat(v[4], dev, a.rows * nv), nv);
    SQ_VEC(a, dt, flat(v[5], dev, int64_t(a.rows) * a.lay.hv), a.lay.hv);
    SQ_VEC(a, B, flat(v[6], dev, a.rows * nk), nk);
    SQ_VEC(a, C, flat(v[7], dev, a.rows * nk), nk);
    const at::Tensor& out = on(v[8], dev);
    SQ_VEC(a, out, out, rows_of(out, a.lay.dv));
    mamba2_model(a, v[9], v[10], v[11], v[12], v[13], dev);
    return launch(lib.mamba2_step, a, dev);
}

// gga_step(slots, views, plan, idx, q, k, v, out, scale, g, beta, gate): `slots` an sq_gga_slots without its pointers,
// `plan` the layer's (offsets, widths, impact factors) on the device
PyObject* gga_step(PyObject* const* v) {
    sq_gga_args a = {};
    a.sl = struct_of<sq_gga_slots>(v[0]);
    want(PyDict_CheckExact(v[1]));
    PyObject* const blob_obj = PyDict_GetItemWithError(v[1], blob_name);
    if (!blob_obj) { PyErr_Clear(); other(); }
    const at::Tensor& blob = plain(blob_obj);
    const c10::Device dev = blob.device();
    want(blob.dim() == 2);
    a.sl.blob = blob.data_ptr();
    a.sl.slot_stride = blob.stride(0);
    want(PyTuple_CheckExact(v[2]) && PyTuple_GET_SIZE(v[2]) == 3);
    a.sl.offs = static_cast<const int32_t*>(on(PyTuple_GET_ITEM(v[2], 0), dev).data_ptr());
    a.sl.bits = static_cast<const int32_t*>(on(PyTuple_GET_ITEM(v[2], 1), dev).data_ptr());
    a.sl.w = static_cast<const float*>(on(PyTuple_GET_ITEM(v[2], 2), dev).data_ptr());
    const at::Tensor& idx = on(v[3], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    const at::Tensor &q = on(v[4], dev), &k = on(v[5], dev), &vv = on(v[6], dev), &out = on(v[7], dev);
    SQ_VEC(a, q, q, rows_of(q, a.sl.dk));
    SQ_VEC(a, k, k, rows_of(k, a.sl.dk));
    SQ_VEC(a, v, vv, rows_of(vv, a.sl.dv));
    want(out.is_contiguous() && out.dim() == 3 && out.size(0) >= a.rows && out.size(1) == a.sl.hv && out.size(2) == a.sl.dv);
    a.out = out.data_ptr();
    a.out_dtype = dtype_code(out);
    a.scale = float(number(v[8]));
    gate_of(a, v[9], v[10], v[11], dev);
    return launch(lib.gga_step, a, dev);
}

// write(lay, views, idx, src): fp32 states [rows, hv, dv, dk], contiguous, into slots
PyObject* write_slots(PyObject* const* v) {
    sq_pack_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    c10::Device dev(c10::kCPU);
    const sq_state st = state_of(v[1], Py_None, 0, &dev);
    const at::Tensor& idx = on(v[2], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    const int64_t per_row = int64_t(a.lay.hv) * a.lay.dv * a.lay.dk;
    const at::Tensor& src = flat(v[3], dev, a.rows * per_row);
    want(src.scalar_type() == at::kFloat);
    a.src = static_cast<const float*>(src.data_ptr());
    a.s_src = per_row;
    a.S = st.S;         a.sS = st.sS;
    const bool scaled = PyDict_GetItem(v[1], field_name[F_SC]) != nullptr;
    a.SC = scaled ? st.SC : nullptr;
    a.sSC = scaled ? st.sSC : 0;
    const at::Tensor& decay = THPVariable_Unpack(PyDict_GetItem(v[1], field_name[F_GCUR]));
    const at::Tensor& fill = THPVariable_Unpack(PyDict_GetItem(v[1], field_name[F_NPTR]));
    want(decay.size(0) > 0 && fill.size(0) > 0);
    a.GCUR = st.GCUR;   a.sGC = st.sGC;
    a.gcur_per_head = int32_t(decay.numel() / decay.size(0) / a.lay.hv);
    a.NPTR = st.NPTR;   a.sN = st.sN;
    a.nptr_copies = int32_t(fill.numel() / fill.size(0));
    return launch(lib.pack_vk, a, dev);
}

// read(lay, views, idx, kda) -> (status, fp32 states [rows, hv, dv, dk])
PyObject* read_slots(PyObject* const* v) {
    sq_read_args a = {};
    a.lay = struct_of<sq_layout>(v[0]);
    c10::Device dev(c10::kCPU);
    a.st = state_of(v[1], Py_None, 0, &dev);
    const at::Tensor& idx = on(v[2], dev);
    a.rows = rows_of_index(idx);
    a.idx = static_cast<const int32_t*>(idx.data_ptr());
    want(PyBool_Check(v[3]));
    a.kda = v[3] == Py_True;
    at::Tensor out = at::empty({a.rows, a.lay.hv, a.lay.dv, a.lay.dk}, at::TensorOptions().dtype(at::kFloat).device(dev));
    want(!out.key_set().has(c10::DispatchKey::Python));
    a.out = static_cast<float*>(out.data_ptr());
    a.s_out = out.stride(0);
    PyObject* const rc = launch(lib.read, a, dev);
    if (!rc) return nullptr;
    PyObject* const t = THPVariable_Wrap(std::move(out));
    if (!t) { Py_DECREF(rc); return nullptr; }
    PyObject* const pair = PyTuple_Pack(2, rc, t);
    Py_DECREF(rc);
    Py_DECREF(t);
    return pair;
}

// The functions above behind Python's calling convention: N arguments; None for whatever is not an ordinary call, C++
// exceptions included.
template <PyObject* (*FN)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", N, n);
        return nullptr;
    }
    try {
        return FN(args);
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
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
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sqhost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sqhost() {
    for (int f = 0; f < F_COUNT; ++f)
        if (!(field_name[f] = PyUnicode_InternFromString(FIELD_NAMES[f]))) return nullptr;
    if (!(blob_name = PyUnicode_InternFromString("blob"))) return nullptr;
    return PyModule_Create(&module);
}
