// Native host path of the Python operators: argument checks, output
// allocation and the library call of an operator's common form in one C call.
// A call costs the launch plus one to three microseconds, against ten to fifteen
// for the same work in Python and ctypes, which is what bounds the small
// launches (a decode layer is five of 5 to 13 us each).
//
// Every function here takes exactly the calls that the Python operator would
// pass through unchanged: plain strided GPU tensors on one device, of the
// expected types and shapes, rows of stride 1, nothing to convert or copy, no
// optional outputs. Anything else, errors included, returns None before any
// effect, and the operator goes on with its full path. A non-zero status of the
// library is returned as an int for the caller to raise.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>

#include "../../include/sparda.h"

namespace {

PyObject* g_raw_stream = nullptr;  // device index -> current stream handle (int)
struct Entries {
    decltype(&sparda_compress) compress;
    decltype(&sparda_route) route;
    decltype(&sparda_prefill) prefill;
    decltype(&sparda_prefill_routed) prefill_routed;
    decltype(&sparda_prefill_chunked) prefill_chunked;
    decltype(&sparda_decode) decode;
    decltype(&sparda_decode_workspace_bytes) decode_workspace_bytes;
    decltype(&sparda_decode_selected) decode_selected;
    decltype(&sparda_decode_dense_workspace_bytes) decode_dense_workspace_bytes;
    decltype(&sparda_decode_sums) decode_sums;
    decltype(&sparda_produce) produce;
    decltype(&sparda_produce_at) produce_at;
    decltype(&sparda_produce_cache_at) produce_cache_at;
    decltype(&sparda_ffn_decode) ffn_decode;
    decltype(&sparda_rows_residual) rows_residual;
    decltype(&sparda_norm_gemv) norm_gemv;
    decltype(&sparda_teacher_mass) teacher_mass;
} g;

// the call is not of the common form: the Python operator takes it
struct Decline {};
inline void need(bool ok) {
    if (!ok) throw Decline{};
}

int64_t as_int(PyObject* o) {
    need(PyLong_Check(o));  // bool included, as Python's int() of the slow path takes it
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        throw Decline{};
    }
    return v;
}
double as_float(PyObject* o) {
    need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        throw Decline{};
    }
    return v;
}
bool as_bool(PyObject* o) {
    need(o == Py_True || o == Py_False);
    return o == Py_True;
}
float scale_or(PyObject* o, int64_t dim) {
    return static_cast<float>(o == Py_None ? 1.0 / std::sqrt(static_cast<double>(dim)) : as_float(o));
}

// Tensors of one call: plain GPU tensors of one device
struct Args {
    int device = -1;
    const at::Tensor& tensor(PyObject* o, int64_t dim) {
        need(THPVariable_CheckExact(o));
        const at::Tensor& t = THPVariable_Unpack(o);
        need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.dim() == dim && !t.is_conj() && !t.is_neg());
        const int d = static_cast<int>(t.get_device());
        need(device < 0 || d == device);
        device = d;
        return t;
    }
    // an operand of the attention: no gradient recorded, rows of stride 1, fp32 or bf16
    const at::Tensor& operand(PyObject* o, int64_t dim) {
        const at::Tensor& t = tensor(o, dim);
        need(!(t.requires_grad() && c10::GradMode::is_enabled()));
        need(t.stride(dim - 1) == 1 && (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat));
        return t;
    }
    const at::Tensor& bf16(PyObject* o, int64_t dim) {
        const at::Tensor& t = operand(o, dim);
        need(t.scalar_type() == at::kBFloat16);
        return t;
    }
    const at::Tensor& weight(PyObject* o) {
        const at::Tensor& t = bf16(o, 2);
        need(t.is_contiguous());
        return t;
    }
    const at::Tensor& f32(PyObject* o, int64_t dim) {
        const at::Tensor& t = tensor(o, dim);
        need(t.scalar_type() == at::kFloat && t.is_contiguous());
        return t;
    }
    const int64_t* position(PyObject* o) {
        const at::Tensor& t = tensor(o, 1);
        need(t.scalar_type() == at::kLong && t.numel() == 1);
        return static_cast<const int64_t*>(t.data_ptr());
    }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dt) const {
        return at::empty(sizes, at::TensorOptions().dtype(dt).device(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device))));
    }
    void* stream() const {
        PyObject* i = PyLong_FromLong(device);
        if (i == nullptr) throw Decline{};
        PyObject* r = PyObject_CallOneArg(g_raw_stream, i);
        Py_DECREF(i);
        if (r == nullptr) {
            PyErr_Clear();
            throw Decline{};
        }
        void* s = PyLong_AsVoidPtr(r);
        Py_DECREF(r);
        return s;
    }
};

inline int code(const at::Tensor& t) { return t.scalar_type() == at::kFloat ? SPARDA_F32 : SPARDA_BF16; }
inline bool same_strides(const at::Tensor& a, const at::Tensor& b) { return a.strides() == b.strides(); }
inline bool aligned(const at::Tensor& t, uintptr_t n) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % n == 0; }
inline bool strides_of(const at::Tensor& t, int64_t n) {
    for (int64_t i = 0; i + 1 < t.dim(); ++i)
        if (t.stride(i) % n) return false;
    return true;
}

// the library call, without the interpreter lock (as ctypes makes it)
template <class F, class... A>
int run(F f, A... a) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(a...);
    Py_END_ALLOW_THREADS
    return rc;
}
PyObject* result(int rc, const at::Tensor& t) { return rc != 0 ? PyLong_FromLong(rc) : THPVariable_Wrap(t); }

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != N || g_raw_stream == nullptr) Py_RETURN_NONE;
    try {
        return F(a);
    } catch (const Decline&) {
    } catch (...) {  // a tensor without storage, an allocation that failed: the operator reports it
        PyErr_Clear();
    }
    Py_RETURN_NONE;
}

// compress(k, block_size)
PyObject* compress(PyObject* const* a) {
    Args x;
    const at::Tensor& k = x.operand(a[0], 4);
    const int64_t bs = as_int(a[1]);
    need(bs > 0);
    const at::Tensor out = x.empty({k.size(0), (k.size(1) + bs - 1) / bs, k.size(2), k.size(3)}, at::kFloat);
    return result(run(g.compress, k.data_ptr(), code(k), k.size(0), k.size(1), k.size(2), k.size(3), k.stride(0),
                      k.stride(1), k.stride(2), bs, static_cast<float*>(out.data_ptr()), x.stream()),
                  out);
}

// route(forecast, protos, block_size, top_k, causal, score_pos0, query_pos0, scale): the top-k picks alone
PyObject* route(PyObject* const* a) {
    Args x;
    const at::Tensor& f = x.operand(a[0], 4);
    const at::Tensor& p = x.f32(a[1], 4);
    const int64_t bs = as_int(a[2]), k = as_int(a[3]);
    const int causal = as_bool(a[4]);
    const int64_t NB = p.size(1), ke = k < NB ? k : NB;
    need(p.size(0) == f.size(0) && p.size(2) == f.size(2) && p.size(3) == f.size(3) && bs > 0 && ke > 0);
    const float scale = scale_or(a[7], f.size(3));
    const int64_t sp = as_int(a[5]), qp = as_int(a[6]);
    const at::Tensor out = x.empty({f.size(0), f.size(2), f.size(1), ke}, at::kInt);
    return result(run(g.route, f.data_ptr(), code(f), f.stride(0), f.stride(1), f.stride(2),
                      static_cast<const float*>(p.data_ptr()), f.size(0), f.size(1), f.size(2), f.size(3), NB, bs, k,
                      causal, sp, qp, scale, static_cast<int32_t*>(out.data_ptr()), static_cast<float*>(nullptr),
                      static_cast<int32_t*>(nullptr), static_cast<int32_t*>(nullptr), int64_t(0), x.stream()),
                  out);
}

struct Qkv {
    const at::Tensor &q, &k, &v;
    int64_t B, T, Hq, Hkv, D;
    Qkv(Args& x, PyObject* const* a)
        : q(x.operand(a[0], 4)), k(x.operand(a[1], 4)), v(x.operand(a[2], 4)), B(q.size(0)), T(q.size(1)),
          Hq(q.size(2)), Hkv(k.size(2)), D(q.size(3)) {
        need(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type() && same_strides(k, v));
        need(k.sizes() == v.sizes() && k.size(0) == B && k.size(1) == T && k.size(3) == D && Hkv > 0 && T > 0);
    }
};

// prefill(q, k, v, block_size, causal, scale): dense
PyObject* prefill(PyObject* const* a) {
    Args x;
    const Qkv t(x, a);
    const int64_t bs = as_int(a[3]);
    const int causal = as_bool(a[4]);
    const float scale = scale_or(a[5], t.D);
    const at::Tensor out = x.empty({t.B, t.T, t.Hq * t.D}, t.q.scalar_type());
    return result(run(g.prefill, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.q.stride(2), t.k.data_ptr(),
                      t.v.data_ptr(), t.k.stride(0), t.k.stride(1), t.k.stride(2), code(t.q),
                      static_cast<const int32_t*>(nullptr), static_cast<const int32_t*>(nullptr), int64_t(0), t.B, t.T,
                      t.Hq, t.Hkv, t.D, bs, causal, scale, out.data_ptr(), out.stride(0), out.stride(1), x.stream()),
                  out);
}

// prefill_routed(q, k, v, forecast, protos, block_size, top_k, causal, scale, route_scale): one launch
PyObject* prefill_routed(PyObject* const* a) {
    Args x;
    const Qkv t(x, a);
    const at::Tensor& f = x.operand(a[3], 4);
    const at::Tensor& p = x.f32(a[4], 4);
    const int64_t bs = as_int(a[5]), k = as_int(a[6]);
    const int causal = as_bool(a[7]);
    need(t.q.scalar_type() == at::kBFloat16 && t.D == 64 && f.size(3) == 64 && (bs == 32 || bs == 64));
    const int64_t NB = (t.T + bs - 1) / bs, R = t.Hq / t.Hkv, ke = k < NB ? k : NB;
    need(f.size(0) == t.B && f.size(1) == t.T && f.size(2) == t.Hkv);
    need(p.size(0) == t.B && p.size(1) == NB && p.size(2) == t.Hkv && p.size(3) == 64);
    need(ke >= 1 && ke <= 8 && t.Hq % t.Hkv == 0 && R >= 1 && R <= 4 && NB <= 1024);
    need(aligned(t.q, 16) && aligned(t.k, 16) && aligned(t.v, 16) && aligned(p, 16));
    need(strides_of(t.q, 8) && strides_of(t.k, 8));
    need(128 * t.q.stride(1) + R * t.q.stride(2) + 64 < (int64_t(1) << 30) && 64 * t.k.stride(1) + 64 < (int64_t(1) << 30));
    const float scale = scale_or(a[8], 64), rscale = scale_or(a[9], 64);
    const at::Tensor out = x.empty({t.B, t.T, t.Hq * 64}, at::kBFloat16);
    need(aligned(out, 16));
    return result(run(g.prefill_routed, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.q.stride(2), t.k.data_ptr(),
                      t.v.data_ptr(), t.k.stride(0), t.k.stride(1), t.k.stride(2), SPARDA_BF16, f.data_ptr(), code(f),
                      f.stride(0), f.stride(1), f.stride(2), static_cast<const float*>(p.data_ptr()), int64_t(64), k,
                      rscale, static_cast<int32_t*>(nullptr), static_cast<int32_t*>(nullptr), int64_t(0), t.B, t.T,
                      t.Hq, t.Hkv, t.D, bs, causal, scale, out.data_ptr(), out.stride(0), out.stride(1), x.stream()),
                  out);
}

// prefill_chunked(q, k, v, topk, block_size, top_k, scale): one launch
PyObject* prefill_chunked(PyObject* const* a) {
    Args x;
    const Qkv t(x, a);
    const int64_t bs = as_int(a[4]), k = as_int(a[5]);
    need(t.q.scalar_type() == at::kBFloat16 && t.D == 64 && bs == 64 && t.Hq % t.Hkv == 0 && t.Hq / t.Hkv <= 4);
    need(aligned(t.q, 16) && aligned(t.k, 16) && aligned(t.v, 16) && strides_of(t.q, 8) && strides_of(t.k, 8));
    const int32_t* picks = nullptr;
    int64_t ke = 0;
    if (a[3] != Py_None) {
        const at::Tensor& p = x.tensor(a[3], 4);
        need(p.scalar_type() == at::kInt && p.is_contiguous() && p.size(0) == t.B && p.size(1) == t.Hkv && p.size(2) == t.T);
        picks = static_cast<const int32_t*>(p.data_ptr());
        ke = p.size(3);
    }
    const float scale = scale_or(a[6], 64);
    const at::Tensor out = x.empty({t.B, t.T, t.Hq * 64}, at::kBFloat16);
    return result(run(g.prefill_chunked, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.q.stride(2), t.k.data_ptr(),
                      t.v.data_ptr(), t.k.stride(0), t.k.stride(1), t.k.stride(2), SPARDA_BF16, picks, ke, k,
                      static_cast<int32_t*>(nullptr), static_cast<int32_t*>(nullptr), int64_t(0), t.B, t.T, t.Hq, t.Hkv,
                      t.D, bs, scale, out.data_ptr(), out.stride(0), out.stride(1), x.stream()),
                  out);
}

struct DecodeQkv {
    const at::Tensor &q, &k, &v;
    int64_t B, Hq, D, Hkv, S;
    DecodeQkv(Args& x, PyObject* const* a)
        : q(x.operand(a[0], 3)), k(x.operand(a[1], 4)), v(x.operand(a[2], 4)), B(q.size(0)), Hq(q.size(1)),
          D(q.size(2)), Hkv(k.size(2)), S(as_int(a[3])) {
        need(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type() && same_strides(k, v));
        need(k.sizes() == v.sizes() && k.size(0) >= B && k.size(3) == D && S > 0 && S <= k.size(1) && Hkv > 0);
    }
};

// decode(q, k_cache, v_cache, S, forecast, block_size, top_k, absolute, scale, workspace)
PyObject* decode(PyObject* const* a) {
    Args x;
    const DecodeQkv t(x, a);
    const int64_t bs = as_int(a[5]), k = as_int(a[6]);
    need(bs > 0 && k > 0);
    const void* f = nullptr;
    int fdt = SPARDA_F32;
    int64_t fsb = 0, fsh = 0;
    if (a[4] != Py_None) {
        const at::Tensor& ft = x.tensor(a[4], 3);
        need(ft.stride(2) == 1 && (ft.scalar_type() == at::kBFloat16 || ft.scalar_type() == at::kFloat));
        need(ft.size(0) == t.B && ft.size(1) == t.Hkv && ft.size(2) == t.D);
        f = ft.data_ptr(), fdt = code(ft), fsb = ft.stride(0), fsh = ft.stride(1);
    }
    const int routing = as_bool(a[7]) ? SPARDA_ROUTE_ABSOLUTE : SPARDA_ROUTE_REFERENCE;
    const float scale = scale_or(a[8], t.D);
    const at::Tensor& ws = x.tensor(a[9], 1);
    const size_t bytes = g.decode_workspace_bytes(t.B, t.S, t.Hq, t.Hkv, t.D, bs, k);
    need(ws.scalar_type() == at::kByte && ws.is_contiguous() && static_cast<size_t>(ws.numel()) >= bytes);
    const at::Tensor out = x.empty({t.B, t.Hq * t.D}, t.q.scalar_type());
    return result(run(g.decode, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.k.data_ptr(), t.v.data_ptr(),
                      t.k.stride(0), t.k.stride(1), t.k.stride(2), code(t.q), f, fdt, fsb, fsh, t.B, t.S, t.Hq, t.Hkv,
                      t.D, bs, k, routing, scale, static_cast<const float*>(nullptr), static_cast<float*>(nullptr),
                      static_cast<int32_t*>(nullptr), static_cast<int32_t*>(nullptr), out.data_ptr(), out.stride(0),
                      ws.data_ptr(), static_cast<size_t>(ws.numel()), x.stream()),
                  out);
}

// decode_dense(q, k, v, S, block_size, scale)
PyObject* decode_dense(PyObject* const* a) {
    Args x;
    const DecodeQkv t(x, a);
    const int64_t bs = as_int(a[4]);
    const float scale = scale_or(a[5], t.D);
    void* ws = nullptr;
    size_t bytes = 0;
    at::Tensor part;  // split partials, held until the launch is enqueued
    if (t.q.scalar_type() == at::kBFloat16 && t.D == 64 && (bs == 32 || bs == 64)) {
        bytes = g.decode_dense_workspace_bytes(t.B, t.Hq, t.Hkv, t.D, t.S, bs);
        if (bytes > 0) {
            part = x.empty({static_cast<int64_t>(bytes / 4 + 4)}, at::kFloat);
            ws = part.data_ptr();
        }
    }
    const at::Tensor out = x.empty({t.B, t.Hq * t.D}, t.q.scalar_type());
    return result(run(g.decode_selected, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.k.data_ptr(), t.v.data_ptr(),
                      t.k.stride(0), t.k.stride(1), t.k.stride(2), code(t.q), 0, static_cast<const int32_t*>(nullptr),
                      static_cast<const int32_t*>(nullptr), int64_t(0), static_cast<const void*>(nullptr),
                      static_cast<const void*>(nullptr), int64_t(0), int64_t(0), t.B, t.S, t.Hq, t.Hkv, t.D, bs, scale,
                      out.data_ptr(), out.stride(0), ws, bytes, x.stream()),
                  out);
}

// decode_sums(q, k, v, S, forecast, block_sums, block_size, top_k, absolute, pos_dev, scale, update_current)
PyObject* decode_sums(PyObject* const* a) {
    Args x;
    const DecodeQkv t(x, a);
    const at::Tensor& f = x.tensor(a[4], 3);
    const at::Tensor& s = x.f32(a[5], 4);
    need(f.stride(2) == 1 && (f.scalar_type() == at::kBFloat16 || f.scalar_type() == at::kFloat));
    need(f.size(0) == t.B && f.size(1) == t.Hkv && f.size(2) == t.D);
    need(s.size(0) == t.B && s.size(2) == t.Hkv && s.size(3) == t.D);
    const int64_t bs = as_int(a[6]), k = as_int(a[7]);
    const int routing = as_bool(a[8]) ? SPARDA_ROUTE_ABSOLUTE : SPARDA_ROUTE_REFERENCE;
    const int64_t* pos = a[9] != Py_None ? x.position(a[9]) : nullptr;
    const float scale = scale_or(a[10], t.D), fscale = scale_or(Py_None, t.D);
    const int update = as_bool(a[11]);
    const at::Tensor out = x.empty({t.B, t.Hq * t.D}, t.q.scalar_type());
    return result(run(g.decode_sums, t.q.data_ptr(), t.q.stride(0), t.q.stride(1), t.k.data_ptr(), t.v.data_ptr(),
                      t.k.stride(0), t.k.stride(1), t.k.stride(2), code(t.q), f.data_ptr(), code(f), f.stride(0),
                      f.stride(1), static_cast<float*>(s.data_ptr()), s.size(1), update, t.B, t.S, pos, t.Hq, t.Hkv, t.D,
                      bs, k, routing, scale, fscale, static_cast<int32_t*>(nullptr), static_cast<int32_t*>(nullptr),
                      out.data_ptr(), out.stride(0), x.stream()),
                  out);
}

// x [B, T, C] as B * T rows without a copy
struct Rows {
    const at::Tensor& t;
    int64_t M, C, st;
    Rows(Args& x, PyObject* o) : t(x.bf16(o, 3)), M(t.size(0) * t.size(1)), C(t.size(2)), st(0) {
        need(M > 0);
        const int64_t B = t.size(0), T = t.size(1);
        if (T == 1) st = B == 1 ? C : t.stride(0);
        else st = t.stride(1);
        need(T == 1 || B == 1 || t.stride(0) == T * st);
        need(st >= C && st % 8 == 0);
    }
};

// produce(x, w, n_q, n_kv, n_f, eps, cos, sin, pos0, f_is_f32, pos_dev, k_cache, v_cache)
PyObject* produce(PyObject* const* a) {
    Args x;
    const Rows r(x, a[0]);
    const at::Tensor& w = x.weight(a[1]);
    const int64_t nq = as_int(a[2]), nkv = as_int(a[3]), nf = as_int(a[4]), pos0 = as_int(a[8]);
    const float eps = static_cast<float>(as_float(a[5]));
    const at::Tensor& cs = x.f32(a[6], 2);
    const at::Tensor& sn = x.f32(a[7], 2);
    const bool f32 = as_bool(a[9]);
    const int64_t B = r.t.size(0), T = r.t.size(1);
    need(nq > 0 && nkv > 0 && nf > 0 && nq % 64 == 0 && nkv % 64 == 0 && nf % 64 == 0);
    need(w.size(0) == nq + 2 * nkv + nf && w.size(1) == r.C && cs.size(1) == 32 && sn.sizes() == cs.sizes());
    const int64_t* pos = a[10] != Py_None ? x.position(a[10]) : nullptr;
    need(pos == nullptr || pos0 == 0);
    const bool cache = a[11] != Py_None;
    need(cache == (a[12] != Py_None) && (!cache || pos != nullptr));
    const at::Tensor q = x.empty({B, T, nq / 64, 64}, at::kBFloat16), k = x.empty({B, T, nkv / 64, 64}, at::kBFloat16),
                     v = x.empty({B, T, nkv / 64, 64}, at::kBFloat16),
                     f = x.empty({B, T, nf / 64, 64}, f32 ? at::kFloat : at::kBFloat16);
    const float* cp = static_cast<const float*>(cs.data_ptr());
    const float* sp = static_cast<const float*>(sn.data_ptr());
    const int fdt = f32 ? SPARDA_F32 : SPARDA_BF16;
    int rc;
    if (cache) {
        const at::Tensor& kc = x.tensor(a[11], 4);
        const at::Tensor& vc = x.tensor(a[12], 4);
        need(kc.scalar_type() == at::kBFloat16 && vc.scalar_type() == at::kBFloat16 && same_strides(kc, vc) &&
             kc.sizes() == vc.sizes() && kc.size(0) == B && kc.size(2) == nkv / 64 && kc.size(3) == 64 && kc.stride(3) == 1);
        rc = run(g.produce_cache_at, r.t.data_ptr(), r.st, w.data_ptr(), r.M, r.C, nq, nkv, nf, eps, cp, sp, cs.size(0),
                 T, pos, q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), fdt, kc.data_ptr(), vc.data_ptr(),
                 kc.stride(0), kc.stride(1), kc.stride(2), kc.size(1), x.stream());
    } else if (pos != nullptr) {
        rc = run(g.produce_at, r.t.data_ptr(), r.st, w.data_ptr(), r.M, r.C, nq, nkv, nf, eps, cp, sp, cs.size(0), T, pos,
                 q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), fdt, x.stream());
    } else {
        rc = run(g.produce, r.t.data_ptr(), r.st, w.data_ptr(), r.M, r.C, nq, nkv, nf, eps, cp, sp, cs.size(0), T, pos0,
                 q.data_ptr(), k.data_ptr(), v.data_ptr(), f.data_ptr(), fdt, x.stream());
    }
    if (rc != 0) return PyLong_FromLong(rc);
    PyObject* out = PyTuple_New(4);
    if (out == nullptr) return nullptr;
    const at::Tensor* ts[4] = {&q, &k, &v, &f};
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(*ts[i]));
    return out;
}

// ffn_decode(x, w_gate_up, w_down, eps)
PyObject* ffn_decode(PyObject* const* a) {
    Args x;
    const Rows r(x, a[0]);
    const at::Tensor& gu = x.weight(a[1]);
    const at::Tensor& dn = x.weight(a[2]);
    const int64_t F = gu.size(0) / 2;
    need(gu.size(0) == 2 * F && gu.size(1) == r.C && dn.size(0) == r.C && dn.size(1) == F);
    const float eps = static_cast<float>(as_float(a[3]));
    const at::Tensor act = x.empty({r.M, F}, at::kBFloat16);
    const at::Tensor out = x.empty(r.t.sizes(), at::kBFloat16);
    return result(run(g.ffn_decode, r.t.data_ptr(), r.st, gu.data_ptr(), dn.data_ptr(), r.M, r.C, F, eps, act.data_ptr(),
                      out.data_ptr(), r.C, x.stream()),
                  out);
}

// rows_residual(a, w, res)
PyObject* rows_residual(PyObject* const* a) {
    Args x;
    const Rows r(x, a[0]);
    const at::Tensor& w = x.weight(a[1]);
    const Rows res(x, a[2]);
    const int64_t N = w.size(0);
    need(w.size(1) == r.C && res.C == N && res.t.size(0) == r.t.size(0) && res.t.size(1) == r.t.size(1));
    const at::Tensor out = x.empty(res.t.sizes(), at::kBFloat16);
    return result(run(g.rows_residual, r.t.data_ptr(), r.st, w.data_ptr(), r.M, r.C, N, res.t.data_ptr(), res.st,
                      out.data_ptr(), N, x.stream()),
                  out);
}

// norm_gemv(x, w_folded, eps)
PyObject* norm_gemv(PyObject* const* a) {
    Args x;
    const Rows r(x, a[0]);
    const at::Tensor& w = x.weight(a[1]);
    need(w.size(1) == r.C);
    const float eps = static_cast<float>(as_float(a[2]));
    const at::Tensor out = x.empty({r.t.size(0), r.t.size(1), w.size(0)}, at::kBFloat16);
    return result(run(g.norm_gemv, r.t.data_ptr(), r.st, w.data_ptr(), r.M, r.C, w.size(0), eps, out.data_ptr(),
                      w.size(0), x.stream()),
                  out);
}

// teacher_mass(q, k, block_size, causal, scale)
PyObject* teacher_mass(PyObject* const* a) {
    Args x;
    const at::Tensor& q = x.operand(a[0], 4);
    const at::Tensor& k = x.operand(a[1], 4);
    const int64_t bs = as_int(a[2]);
    const int causal = as_bool(a[3]);
    need(k.size(0) == q.size(0) && k.size(1) == q.size(1) && k.size(3) == q.size(3) && bs > 0);
    const float scale = scale_or(a[4], q.size(3));
    const at::Tensor out = x.empty({q.size(0), k.size(2), q.size(1), (q.size(1) + bs - 1) / bs}, at::kFloat);
    return result(run(g.teacher_mass, q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), k.stride(0),
                      k.stride(1), k.stride(2), code(q), q.size(0), q.size(1), q.size(2), k.size(2), q.size(3), bs,
                      causal, scale, static_cast<float*>(out.data_ptr()), x.stream()),
                  out);
}

// bind(raw_stream, addresses): the current-stream query and the entry points' addresses, in Entries' order
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *raw, *list;
    if (!PyArg_ParseTuple(args, "OO!", &raw, &PyTuple_Type, &list)) return nullptr;
    constexpr Py_ssize_t kN = sizeof(Entries) / sizeof(void*);
    if (PyTuple_GET_SIZE(list) != kN) {
        PyErr_Format(PyExc_ValueError, "bind: %zd addresses", kN);
        return nullptr;
    }
    void* p[kN];
    for (Py_ssize_t i = 0; i < kN; ++i) {
        p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(list, i));
        if (p[i] == nullptr) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    }
    __builtin_memcpy(&g, p, sizeof(g));
    Py_INCREF(raw);
    Py_XSETREF(g_raw_stream, raw);
    Py_RETURN_NONE;
}

#define SPARDA_FAST(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    SPARDA_FAST(compress, 2),
    SPARDA_FAST(route, 8),
    SPARDA_FAST(prefill, 6),
    SPARDA_FAST(prefill_routed, 10),
    SPARDA_FAST(prefill_chunked, 7),
    SPARDA_FAST(decode, 10),
    SPARDA_FAST(decode_dense, 6),
    SPARDA_FAST(decode_sums, 12),
    SPARDA_FAST(produce, 13),
    SPARDA_FAST(ffn_decode, 4),
    SPARDA_FAST(rows_residual, 3),
    SPARDA_FAST(norm_gemv, 3),
    SPARDA_FAST(teacher_mass, 5),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__host() { return PyModule_Create(&kModule); }
