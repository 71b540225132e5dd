// torch_ops.cpp — the op calls of sapient_amd/ops.py on torch tensors: argument
// checks, the output tensor, the current stream and the C ABI call, natively.
//
// A decode step's kernels run 1.5-3 µs each; a call through Python checks, torch's
// Python stream and allocation calls and ctypes took the host 6.8-10.4 µs, so such
// callers waited on the host, not on the GPU. Here a call costs the launch
// (about 2.4 µs) and 0.3 µs around it, 1.2 with a fresh output. Nothing is kept
// between calls.
//
// Every function takes ops.py's arguments positionally, all of them, and raises what
// ops.py documents: ValueError / TypeError for arguments, SapientHipError (through
// _lib.check) for a status of the ABI. The GIL is released around the ABI call.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>

#include "sapient_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;

struct Raised {};  // a Python error is set

[[noreturn]] void raise(PyObject* type, const std::string& msg) {
    PyErr_SetString(type, msg.c_str());
    throw Raised{};
}
[[noreturn]] void bad(const std::string& msg) { raise(PyExc_ValueError, msg); }

// ───────────────────────────── arguments ─────────────────────────────
const Tensor& tensor(PyObject* o, const char* name) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, std::string(name) + " must be a torch.Tensor");
    return THPVariable_Unpack(o);
}

// A contiguous device tensor.
const Tensor& dev(PyObject* o, const char* name) {
    const Tensor& t = tensor(o, name);
    if (!t.is_cuda()) bad(std::string(name) + " must be a device tensor");
    if (!t.is_contiguous()) bad(std::string(name) + " must be contiguous");
    return t;
}

int64_t integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}

// int(o), float(o)
int64_t as_integer(PyObject* o) {
    if (PyLong_CheckExact(o)) return integer(o);
    PyObject* n = PyNumber_Long(o);
    if (!n) throw Raised{};
    const long long v = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}

float real(PyObject* o) {
    if (PyFloat_CheckExact(o)) return (float)PyFloat_AS_DOUBLE(o);
    PyObject* n = PyNumber_Float(o);
    if (!n) throw Raised{};
    const double v = PyFloat_AS_DOUBLE(n);
    Py_DECREF(n);
    return (float)v;
}

bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw Raised{};
    return v != 0;
}

std::string dtype_name(ScalarType t) {
    PyObject* o = reinterpret_cast<PyObject*>(torch::getTHPDtype(t));
    PyObject* s = PyObject_Str(o);
    if (!s) throw Raised{};
    const char* c = PyUnicode_AsUTF8(s);
    std::string r = c ? c : "?";
    Py_DECREF(s);
    return r;
}

int code(ScalarType t) {
    switch (t) {
    case ScalarType::Float: return SPH_F32;
    case ScalarType::Half: return SPH_F16;
    case ScalarType::BFloat16: return SPH_BF16;
    default: raise(PyExc_TypeError, "unsupported dtype " + dtype_name(t));
    }
}

void* ptr(const Tensor& t) { return t.data_ptr(); }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// A vector of n elements, or null for None.
const Tensor* vec(PyObject* o, int64_t n, const char* name) {
    if (o == Py_None) return nullptr;
    const Tensor& t = dev(o, name);
    if (t.numel() != n)
        bad(std::string(name) + " length " + std::to_string(t.numel()) + " does not match last dim " + std::to_string(n));
    return &t;
}
void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// An int32 device flag, or null for None.
int32_t* flag(PyObject* o, const char* name) {
    if (o == Py_None) return nullptr;
    const Tensor& t = dev(o, name);
    if (t.scalar_type() != ScalarType::Int || t.numel() < 1)
        bad(std::string(name) + " must be an int32 device tensor");
    return static_cast<int32_t*>(t.data_ptr());
}

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// The caller's output, after checking that it holds exactly what the kernel writes, or a fresh one.
struct Out {
    PyObject* given;
    Tensor t;
    Out(PyObject* o, at::IntArrayRef shape, ScalarType dtype, at::Device device, const char* name = "out")
        : given(o == Py_None ? nullptr : o) {
        if (!given) {
            // Without the GIL, as torch's own calls: the allocator may wait for its lock, or for the device. (It
            // costs a decode step's five calls 0.35 µs, 22.5 -> 22.85.)
            const NoGil release;
            t = at::empty(shape, at::TensorOptions().dtype(dtype).device(device));
            return;
        }
        t = dev(o, name);
        if (t.numel() != c10::multiply_integers(shape) || t.scalar_type() != dtype)
            bad(std::string(name) + " must hold " + std::to_string(c10::multiply_integers(shape)) + " elements of " +
                dtype_name(dtype));
    }
    PyObject* object() {  // a new reference
        if (!given) return THPVariable_Wrap(t);
        Py_INCREF(given);
        return given;
    }
};

PyObject* g_check = nullptr;  // _lib.check

// Run an ABI call without the GIL; a status other than SPH_OK raises through _lib.check.
template <typename F>
void call(const char* op, F&& f) {
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = f();
    Py_END_ALLOW_THREADS
    if (st == SPH_OK) return;
    PyObject* r = PyObject_CallFunction(g_check, "is", st, op);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s: status %d", op, st);
    throw Raised{};
}

PyObject* none() { Py_RETURN_NONE; }

void last_dim(const Tensor& x, int64_t& rows, int64_t& dim) {
    dim = x.dim() ? x.size(-1) : 1;
    rows = dim ? x.numel() / dim : 0;
}

// out_dtype, else out's type, else x's.
ScalarType out_type(PyObject* out_dtype, PyObject* out, const Tensor& x) {
    if (out_dtype != Py_None) {
        if (!THPDtype_Check(out_dtype)) raise(PyExc_TypeError, "out_dtype must be a torch.dtype");
        return reinterpret_cast<THPDtype*>(out_dtype)->scalar_type;
    }
    return out != Py_None ? tensor(out, "out").scalar_type() : x.scalar_type();
}

// ───────────────────────────── ops ─────────────────────────────
// (x, weight, eps, out, out_dtype)
PyObject* rms_norm(PyObject* const* a) {
    const Tensor& x = dev(a[0], "x");
    int64_t rows, dim;
    last_dim(x, rows, dim);
    Out out(a[3], x.sizes(), out_type(a[4], a[3], x), x.device());
    const Tensor* w = vec(a[1], dim, "weight");
    const int xd = code(x.scalar_type()), wd = w ? code(w->scalar_type()) : 0, od = code(out.t.scalar_type());
    const float eps = real(a[2]);
    void *xp = ptr(x), *wp = ptr(w), *op = ptr(out.t), *st = stream_of(x);
    call("rms_norm", [&] { return sph_rms_norm(xp, xd, wp, wd, op, od, rows, dim, eps, st); });
    return out.object();
}

// (x, weight, bias, eps, out, out_dtype)
PyObject* layer_norm(PyObject* const* a) {
    const Tensor& x = dev(a[0], "x");
    int64_t rows, dim;
    last_dim(x, rows, dim);
    Out out(a[4], x.sizes(), out_type(a[5], a[4], x), x.device());
    const Tensor *w = vec(a[1], dim, "weight"), *b = vec(a[2], dim, "bias");
    if (w && b && w->scalar_type() != b->scalar_type()) bad("weight and bias must share dtype");
    const Tensor* wb = w ? w : b;
    const int xd = code(x.scalar_type()), wd = wb ? code(wb->scalar_type()) : 0, od = code(out.t.scalar_type());
    const float eps = real(a[3]);
    void *xp = ptr(x), *wp = ptr(w), *bp = ptr(b), *op = ptr(out.t), *st = stream_of(x);
    call("layer_norm", [&] { return sph_layer_norm(xp, xd, wp, bp, wd, op, od, rows, dim, eps, st); });
    return out.object();
}

// (x, residual, weight, eps, out, out_dtype, sum_out)
PyObject* add_rms_norm(PyObject* const* a) {
    const Tensor &x = dev(a[0], "x"), &r = dev(a[1], "residual");
    if (r.sizes() != x.sizes() || r.scalar_type() != x.scalar_type()) bad("x and residual must share shape and dtype");
    PyObject* sum = a[6] == Py_None ? a[1] : a[6];
    if (a[6] != Py_None) {
        const Tensor& s = dev(sum, "sum_out");
        if (s.sizes() != x.sizes() || s.scalar_type() != x.scalar_type()) bad("sum_out must share x's shape and dtype");
    }
    if (x.dim() == 0) raise(PyExc_IndexError, "tuple index out of range");
    int64_t rows, dim;
    last_dim(x, rows, dim);
    Out out(a[4], x.sizes(), out_type(a[5], a[4], x), x.device());
    const Tensor* w = vec(a[2], dim, "weight");
    const int xd = code(x.scalar_type()), wd = w ? code(w->scalar_type()) : 0, od = code(out.t.scalar_type());
    const float eps = real(a[3]);
    void *xp = ptr(x), *rp = ptr(r), *wp = ptr(w), *op = ptr(out.t), *st = stream_of(x);
    if (a[6] == Py_None) {
        call("add_rms_norm", [&] { return sph_add_rms_norm(xp, rp, xd, wp, wd, op, od, rows, dim, eps, st); });
    } else {
        void* sp = ptr(THPVariable_Unpack(sum));
        call("add_rms_norm", [&] { return sph_add_rms_norm_to(xp, rp, sp, xd, wp, wd, op, od, rows, dim, eps, st); });
    }
    PyObject* y = out.object();
    if (!y) throw Raised{};
    PyObject* t = PyTuple_Pack(2, y, sum);
    Py_DECREF(y);
    return t;
}

using Binary = int (*)(const void*, int64_t, const void*, int64_t, void*, int, void*);
PyObject* binary(PyObject* const* a, const char* name, Binary fn) {
    const Tensor &x = dev(a[0], "a"), &y = dev(a[1], "b");
    if (x.scalar_type() != y.scalar_type()) bad("operands must share dtype");
    Out out(a[2], (x.numel() >= y.numel() ? x : y).sizes(), x.scalar_type(), x.device());
    const int d = code(x.scalar_type());
    const int64_t nx = x.numel(), ny = y.numel();
    void *xp = ptr(x), *yp = ptr(y), *op = ptr(out.t), *st = stream_of(x);
    call(name, [&] { return fn(xp, nx, yp, ny, op, d, st); });
    return out.object();
}
PyObject* add(PyObject* const* a) { return binary(a, "add", sph_add); }
PyObject* mul(PyObject* const* a) { return binary(a, "mul", sph_mul); }

using Unary = int (*)(const void*, void*, int, int64_t, void*);
PyObject* unary(PyObject* const* a, const char* name, Unary fn) {
    const Tensor& x = dev(a[0], "x");
    Out out(a[1], x.sizes(), x.scalar_type(), x.device());
    const int d = code(x.scalar_type());
    const int64_t n = x.numel();
    void *xp = ptr(x), *op = ptr(out.t), *st = stream_of(x);
    call(name, [&] { return fn(xp, op, d, n, st); });
    return out.object();
}
PyObject* silu(PyObject* const* a) { return unary(a, "silu", sph_silu); }
PyObject* gelu_tanh(PyObject* const* a) { return unary(a, "gelu", sph_gelu_tanh); }
PyObject* gelu_erf(PyObject* const* a) { return unary(a, "gelu_erf", sph_gelu_erf); }

// (gate, up, out)
PyObject* swiglu(PyObject* const* a) {
    const Tensor &g = dev(a[0], "gate"), &u = dev(a[1], "up");
    if (g.sizes() != u.sizes() || g.scalar_type() != u.scalar_type()) bad("gate and up must share shape and dtype");
    Out out(a[2], g.sizes(), g.scalar_type(), g.device());
    const int d = code(g.scalar_type());
    const int64_t n = g.numel();
    void *gp = ptr(g), *up = ptr(u), *op = ptr(out.t), *st = stream_of(g);
    call("swiglu", [&] { return sph_swiglu(gp, up, op, d, n, st); });
    return out.object();
}

// (y, bias, out)
PyObject* add_bias(PyObject* const* a) {
    const Tensor& y = dev(a[0], "y");
    if (y.dim() == 0) bad("empty tensor");
    const int64_t n = y.size(-1), total = y.numel();
    const Tensor* b = vec(a[1], n, "bias");
    if (!b) raise(PyExc_TypeError, "bias must be a torch.Tensor");
    Out out(a[2], y.sizes(), y.scalar_type(), y.device());
    const int bd = code(b->scalar_type()), d = code(y.scalar_type());
    void *yp = ptr(y), *bp = ptr(b), *op = ptr(out.t), *st = stream_of(y);
    call("add_bias", [&] { return sph_add_bias(yp, bp, bd, op, d, total, n, st); });
    return out.object();
}

// q [B, Hq, S, D] and k [B, Hk, S, D] or None.
struct QK {
    const Tensor* q;
    const Tensor* k = nullptr;
    int64_t B, Hq, S, D, Hk = 0;
    QK(PyObject* qo, PyObject* ko) : q(&dev(qo, "q")) {
        if (q->dim() != 4) bad("q must be [batch, heads, seq, head_dim]");
        B = q->size(0);
        Hq = q->size(1);
        S = q->size(2);
        D = q->size(3);
        if (ko == Py_None) return;
        k = &dev(ko, "k");
        if (k->dim() != 4 || k->size(0) != B || k->size(2) != S || k->size(3) != D || k->scalar_type() != q->scalar_type())
            bad("k must be [batch, kv_heads, seq, head_dim] like q");
        Hk = k->size(1);
    }
};

void check_positions(const Tensor& p, int64_t S, const char* what) {
    if (p.scalar_type() != ScalarType::Int || p.numel() != S) bad(what);
}

// (q, k, positions, base, rotary_dim, pos_scale, interleaved)
PyObject* rope_(PyObject* const* a) {
    const QK t(a[0], a[1]);
    const Tensor& pos = dev(a[2], "positions");
    check_positions(pos, t.S, "positions must be int32 with seq_len entries");
    const int64_t rd = a[4] == Py_None ? t.D : integer(a[4]);
    const int layout = truth(a[6]) ? SPH_ROPE_INTERLEAVED : SPH_ROPE_NEOX, d = code(t.q->scalar_type());
    const float base = real(a[3]), scale = real(a[5]);
    void *qp = ptr(t.q), *kp = ptr(t.k), *pp = ptr(pos), *st = stream_of(*t.q);
    call("rope", [&] {
        return sph_rope(qp, t.Hq, kp, t.Hk, d, layout, static_cast<const int32_t*>(pp), t.B, t.S, t.D, rd, base, scale, st);
    });
    return none();
}

// (q, k, cos_table, sin_table, positions, rotary_dim, interleaved, bad_pos_flag)
PyObject* rope_cached_(PyObject* const* a) {
    const QK t(a[0], a[1]);
    const int64_t rd = a[5] == Py_None ? t.D : integer(a[5]);
    const Tensor* tab[2];
    const char* names[2] = {"cos_table", "sin_table"};
    for (int i = 0; i < 2; ++i) {
        tab[i] = &dev(a[2 + i], names[i]);
        // rd / 2 as Python's floor division
        const int64_t half = rd >= 0 ? rd / 2 : -((1 - rd) / 2);
        if (tab[i]->scalar_type() != ScalarType::Float || tab[i]->dim() != 2 || tab[i]->size(1) != half)
            bad(std::string(names[i]) + " must be f32 [rows, rotary_dim / 2]");
    }
    if (tab[0]->sizes() != tab[1]->sizes()) bad("cos_table and sin_table must have the same shape");
    const Tensor* pos = nullptr;
    if (a[4] != Py_None) {
        pos = &dev(a[4], "positions");
        check_positions(*pos, t.S, "positions must be int32 with seq_len entries");
    }
    int32_t* fl = flag(a[7], "bad_pos_flag");
    const int layout = truth(a[6]) ? SPH_ROPE_INTERLEAVED : SPH_ROPE_NEOX, d = code(t.q->scalar_type());
    const int64_t rows = tab[0]->size(0);
    void *qp = ptr(t.q), *kp = ptr(t.k), *cp = ptr(tab[0]), *sp = ptr(tab[1]), *pp = ptr(pos), *st = stream_of(*t.q);
    call("rope_cached", [&] {
        return sph_rope_cached(qp, t.Hq, kp, t.Hk, d, layout, static_cast<const float*>(cp), static_cast<const float*>(sp),
                               rows, static_cast<const int32_t*>(pp), t.B, t.S, t.D, rd, fl, st);
    });
    return none();
}

// (table, table_dtype, vocab, hidden, ids, out, bad_id_flag)
PyObject* embed(PyObject* const* a) {
    const Tensor &table = dev(a[0], "table"), &ids = dev(a[4], "ids");
    if (ids.scalar_type() != ScalarType::Int && ids.scalar_type() != ScalarType::UInt32) bad("ids must be 32-bit");
    const int64_t dt = integer(a[1]), vocab = integer(a[2]), hidden = integer(a[3]), n = ids.numel();
    // Bytes per block and elements per block of each table type (crates/sapient-core/src/dtype.rs:136-145).
    int64_t num = 0, den = 1;
    switch (dt) {
    case SPH_F32: num = 4; break;
    case SPH_F16:
    case SPH_BF16: num = 2; break;
    case SPH_Q4_0: num = 18; den = 32; break;
    case SPH_Q8_0: num = 34; den = 32; break;
    case SPH_Q4_K: num = 144; den = 256; break;
    case SPH_Q5_K: num = 176; den = 256; break;
    case SPH_Q6_K: num = 210; den = 256; break;
    default: break;
    }
    if (num == 0 || hidden < 0 || vocab < 0) bad("unsupported table dtype or negative size");
    if (hidden % den == 0 &&
        (__int128)table.numel() * (int64_t)table.element_size() < (__int128)vocab * (hidden / den) * num)
        bad("table holds fewer than vocab rows");
    Out out(a[5], {n, hidden}, ScalarType::Float, ids.device());
    int32_t* fl = flag(a[6], "bad_id_flag");
    void *tp = ptr(table), *ip = ptr(ids), *op = ptr(out.t), *st = stream_of(ids);
    call("embed", [&] {
        return sph_embed(tp, (int)dt, vocab, hidden, static_cast<const uint32_t*>(ip), n, static_cast<float*>(op), fl, st);
    });
    return out.object();
}

// (x, out)
PyObject* transpose_heads(PyObject* const* a) {
    const Tensor& x = dev(a[0], "x");
    if (x.dim() != 3) bad("x must be [outer, inner, head_dim]");
    const int64_t outer = x.size(0), inner = x.size(1), hd = x.size(2);
    Out out(a[1], {inner, outer, hd}, x.scalar_type(), x.device());
    if (out.t.data_ptr() == x.data_ptr() && x.numel()) bad("out must not alias x");
    const int d = code(x.scalar_type());
    void *xp = ptr(x), *op = ptr(out.t), *st = stream_of(x);
    call("transpose_heads", [&] { return sph_transpose_heads(xp, op, d, outer, inner, hd, st); });
    return out.object();
}

// src [n_kv, seq, head_dim] and cache [n_kv, max_seq, row]; `next` is the second cache of the out-of-place update.
struct Cache {
    const Tensor &src, &cache;
    const Tensor* next = nullptr;
    bool q8;
    int64_t n_kv, seq, hd, max_seq;
    int sd, cd;
    Cache(PyObject* s, PyObject* c, PyObject* out = nullptr) : src(dev(s, "src")), cache(dev(c, "cache")) {
        if (out) next = &dev(out, "out");
        q8 = cache.scalar_type() == ScalarType::Byte;
        if (src.dim() != 3 || cache.dim() != 3 || src.size(0) != cache.size(0))
            bad("src must be [n_kv, seq, head_dim] and cache [n_kv, max_seq, row]");
        if (next && (next->sizes() != cache.sizes() || next->scalar_type() != cache.scalar_type()))
            bad("out must have the cache's shape and dtype");
        n_kv = src.size(0);
        seq = src.size(1);
        hd = src.size(2);
        if (cache.size(2) != (q8 ? hd / 32 * 34 : hd) || (q8 && hd % 32))
            bad("cache rows must hold head_dim elements (Q8_0: head_dim / 32 blocks of 34 bytes)");
        max_seq = cache.size(1);
        cd = q8 ? SPH_Q8_0 : code(cache.scalar_type());
        sd = code(src.scalar_type());
    }
};

// (src, cache, pos)
PyObject* kv_append(PyObject* const* a) {
    const Cache c(a[0], a[1]);
    const int64_t pos = as_integer(a[2]);
    void *sp = ptr(c.src), *cp = ptr(c.cache), *st = stream_of(c.src);
    call("kv_append", [&] { return sph_kv_append(sp, c.sd, cp, c.cd, c.n_kv, c.seq, c.hd, c.max_seq, pos, st); });
    return none();
}

// (src, cache, cur_len)
PyObject* kv_cache_update(PyObject* const* a) {
    const Cache c(a[0], a[1]);
    const int64_t cur = as_integer(a[2]);
    int64_t n = 0;
    void *sp = ptr(c.src), *cp = ptr(c.cache), *st = stream_of(c.src);
    call("kv_cache_update",
         [&] { return sph_kv_cache_update(sp, c.sd, cp, c.cd, c.n_kv, c.seq, c.hd, c.max_seq, cur, &n, st); });
    return PyLong_FromLongLong(n);
}

// (src, cache, out, cur_len)
PyObject* kv_cache_update_into(PyObject* const* a) {
    const Cache c(a[0], a[1], a[2]);
    const int64_t cur = as_integer(a[3]);
    int64_t n = 0;
    void *sp = ptr(c.src), *cp = ptr(c.cache), *op = ptr(c.next), *st = stream_of(c.src);
    call("kv_cache_update_into",
         [&] { return sph_kv_cache_update_into(sp, c.sd, cp, op, c.cd, c.n_kv, c.seq, c.hd, c.max_seq, cur, &n, st); });
    return PyLong_FromLongLong(n);
}

// Checks shared by the two fused steps.
struct Step {
    const Tensor *kc, *vc, *pos;
    const Tensor* b[3];
    int32_t* fl;
    int bd = 0;
    Step(PyObject* p, PyObject* kco, PyObject* vco, PyObject* f, PyObject* const* bias, int64_t Hq, int64_t Hkv, int64_t S,
         int64_t D)
        : kc(&dev(kco, "kcache")), vc(&dev(vco, "vcache")), pos(&dev(p, "positions")) {
        if (kc->sizes() != vc->sizes() || kc->dim() != 3 || kc->size(0) != Hkv || kc->size(2) != D ||
            kc->scalar_type() != vc->scalar_type())
            bad("caches must be [Hkv, max_seq, D] of one dtype");
        check_positions(*pos, S, "positions must be int32 with seq entries");
        fl = flag(f, "bad_pos_flag");
        b[0] = vec(bias[0], Hq * D, "bq");
        b[1] = vec(bias[1], Hkv * D, "bk");
        b[2] = vec(bias[2], Hkv * D, "bv");
        const Tensor* first = nullptr;
        for (const Tensor* t : b) {
            if (!t) continue;
            if (first && t->scalar_type() != first->scalar_type()) bad("biases must share dtype");
            first = t;
        }
        if (first) bd = code(first->scalar_type());
    }
};

// (q, k, v, positions, base, kcache, vcache, pos_scale, interleaved, bad_pos_flag, bq, bk, bv)
PyObject* rope_kv_append(PyObject* const* a) {
    const Tensor &q = dev(a[0], "q"), &k = dev(a[1], "k"), &v = dev(a[2], "v");
    if (q.dim() != 3 || k.dim() != 3 || k.sizes() != v.sizes() || q.size(1) != k.size(1) || q.size(2) != k.size(2))
        bad("q must be [Hq, S, D] and k, v [Hkv, S, D]");
    if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) bad("q, k and v must share dtype");
    const int64_t Hq = q.size(0), S = q.size(1), D = q.size(2), Hkv = k.size(0);
    const Step s(a[3], a[5], a[6], a[9], a + 10, Hq, Hkv, S, D);
    const int layout = truth(a[8]) ? SPH_ROPE_INTERLEAVED : SPH_ROPE_NEOX, d = code(q.scalar_type()),
              cd = code(s.kc->scalar_type());
    const float base = real(a[4]), scale = real(a[7]);
    const int64_t max_seq = s.kc->size(1);
    void *qp = ptr(q), *kp = ptr(k), *vp = ptr(v), *pp = ptr(s.pos), *kc = ptr(s.kc), *vc = ptr(s.vc), *bq = ptr(s.b[0]),
         *bk = ptr(s.b[1]), *bv = ptr(s.b[2]), *st = stream_of(q);
    call("rope_kv_append", [&] {
        return sph_rope_kv_append(qp, Hq, kp, vp, Hkv, d, layout, static_cast<const int32_t*>(pp), S, D, base, scale, kc,
                                  vc, cd, max_seq, bq, bk, bv, s.bd, s.fl, st);
    });
    return none();
}

// (q, k, v, positions, base, kcache, vcache, pos_scale, interleaved, bad_pos_flag, bq, bk, bv, out)
PyObject* rope_kv_append_tokens(PyObject* const* a) {
    const Tensor &q = dev(a[0], "q"), &k = dev(a[1], "k"), &v = dev(a[2], "v");
    if (q.dim() != 3 || k.dim() != 3 || k.sizes() != v.sizes() || q.size(0) != k.size(0) || q.size(2) != k.size(2))
        bad("q must be [S, Hq, D] and k, v [S, Hkv, D]");
    if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) bad("q, k and v must share dtype");
    const int64_t S = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
    const Step s(a[3], a[5], a[6], a[9], a + 10, Hq, Hkv, S, D);
    Out out(a[13], {Hq, S, D}, q.scalar_type(), q.device());
    const int layout = truth(a[8]) ? SPH_ROPE_INTERLEAVED : SPH_ROPE_NEOX, d = code(q.scalar_type()),
              cd = code(s.kc->scalar_type());
    const float base = real(a[4]), scale = real(a[7]);
    const int64_t max_seq = s.kc->size(1);
    void *qp = ptr(q), *op = ptr(out.t), *kp = ptr(k), *vp = ptr(v), *pp = ptr(s.pos), *kc = ptr(s.kc), *vc = ptr(s.vc),
         *bq = ptr(s.b[0]), *bk = ptr(s.b[1]), *bv = ptr(s.b[2]), *st = stream_of(q);
    call("rope_kv_append_tokens", [&] {
        return sph_rope_kv_append_tokens(qp, op, Hq, kp, vp, Hkv, d, layout, static_cast<const int32_t*>(pp), S, D, base,
                                         scale, kc, vc, cd, max_seq, bq, bk, bv, s.bd, s.fl, st);
    });
    return out.object();
}

// ───────────────────────────── module ─────────────────────────────
// No C++ exception leaves a function: torch's become Python errors.
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    try {
        return F(args);
    } catch (Raised&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

PyObject* set_check(PyObject*, PyObject* f) {
    Py_INCREF(f);
    Py_XSETREF(g_check, f);
    Py_RETURN_NONE;
}

#define SPH_OP(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {SPH_OP(rms_norm, 5),
                          SPH_OP(layer_norm, 6),
                          SPH_OP(add_rms_norm, 7),
                          SPH_OP(add, 3),
                          SPH_OP(mul, 3),
                          SPH_OP(silu, 2),
                          SPH_OP(gelu_tanh, 2),
                          SPH_OP(gelu_erf, 2),
                          SPH_OP(swiglu, 3),
                          SPH_OP(add_bias, 3),
                          SPH_OP(rope_, 7),
                          SPH_OP(rope_cached_, 8),
                          SPH_OP(embed, 7),
                          SPH_OP(transpose_heads, 2),
                          SPH_OP(kv_append, 3),
                          SPH_OP(kv_cache_update, 3),
                          SPH_OP(kv_cache_update_into, 4),
                          SPH_OP(rope_kv_append, 13),
                          SPH_OP(rope_kv_append_tokens, 14),
                          {"set_check", set_check, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() {
    PyObject* m = PyModule_Create(&kModule);
    // What it was built for: torch's C++ ABI changes with its version.
    if (m && (PyModule_AddStringConstant(m, "torch_version", SPH_TORCH_VERSION) < 0 ||
              PyModule_AddIntConstant(m, "abi_version", SPH_ABI_VERSION) < 0))
        Py_CLEAR(m);
    return m;
}
