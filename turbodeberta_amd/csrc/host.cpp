// Native front of the two attention operators: CPython functions that take the operators' arguments as they are,
// check the well-formed case, allocate the output and call the C ABI (include/tdb_attn.h).
//
// What bounds a small call is the host: packing ~60 fields through ctypes, torch.autograd.Function and the Python
// checks took 23 us per call where the kernel takes 8 (batch 1, 29 tokens).  Here the same call costs the output's
// allocation and the launch.  Anything out of the ordinary -- a wrong shape or type, a tensor that needs a copy, a
// gradient to record, another device than the current one, a tensor subclass, a tracer or dispatch mode -- returns None,
// and the caller takes the Python path (ops/*.py: prepare), which copies, switches the device, or raises the error.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/ExpandUtils.h>
#include <ATen/TracerMode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "host.h"
#include "tdb_attn.h"

namespace {

int (*g_fixed)(const tdb_fixed_args*, void*) = nullptr;
int (*g_varlen)(const tdb_varlen_args*, void*) = nullptr;

// Device copies of the relative-position tables, handed over by ops/_launch.py when it builds one (guarded by the GIL,
// as many as the Python cache holds).
struct Lut {
    int device;
    int64_t size, buckets, max_rel;
    at::Tensor table;
};
std::vector<Lut>& luts() {
    static std::vector<Lut>* v = new std::vector<Lut>;      // never destroyed: the allocator may be gone at exit
    return *v;
}

// One tensor argument: its implementation, or null for None.  `ok` is cleared for anything but a plain tensor.
const at::Tensor* tensor(PyObject* o, bool& ok) {
    if (o == Py_None) return nullptr;
    if (!THPVariable_CheckExact(o)) {
        ok = false;
        return nullptr;
    }
    return &THPVariable_Unpack(o);
}

bool as_int(PyObject* o, int64_t& out) {
    if (!PyLong_CheckExact(o)) return false;
    out = PyLong_AsLongLong(o);
    if (out == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return out >= INT32_MIN && out <= INT32_MAX;
}

bool as_flag(PyObject* o, bool& out) {
    out = o == Py_True;
    return o == Py_True || o == Py_False;
}

bool as_scale(PyObject* o, int64_t head_dim, float& out) {
    if (o == Py_None) {
        out = float(1.0 / std::sqrt(double(head_dim)));
        return true;
    }
    if (!PyFloat_CheckExact(o)) return false;
    out = float(PyFloat_AS_DOUBLE(o));
    return true;
}

// Rows the kernels can address: last dim contiguous, base and every outer stride 16-byte aligned.
bool strides_ok(at::IntArrayRef strides, int64_t elem) {
    const size_t n = strides.size();
    if (strides[n - 1] != 1) return false;
    for (size_t i = 0; i + 1 < n; ++i)
        if (strides[i] < 0 || (strides[i] * elem) % 16) return false;
    return true;
}
bool rows_ok(const at::Tensor& t) {
    return strides_ok(t.strides(), t.element_size()) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

int dtype_code(at::ScalarType t) {
    return t == at::kFloat ? TDB_F32 : t == at::kBFloat16 ? TDB_BF16 : t == at::kHalf ? TDB_F16 : -1;
}

// q's strides where q is dense, the dense strides of the same dimension order otherwise (torch.empty_like)
bool output_like(const at::Tensor& q, at::Tensor& o) {
    if (q.is_non_overlapping_and_dense()) {
        o = at::detail::empty_strided_cuda(q.sizes(), q.strides(), q.scalar_type(), q.device());
    } else {
        const auto strides = at::infer_dense_strides(q.sizes(), q.strides());
        o = at::detail::empty_strided_cuda(q.sizes(), strides, q.scalar_type(), q.device());
    }
    return rows_ok(o);
}

struct Common {
    const at::Tensor *q, *k, *v, *q_pos, *k_pos, *pk, *pq;
    int64_t buckets, max_rel;
    bool grad;
};

// q, k, v of one shape, type and device with addressable rows, on the current device
bool inputs_ok(const Common& c, int dims) {
    const at::Tensor &q = *c.q, &k = *c.k, &v = *c.v;
    if (q.dim() != dims || q.sizes() != k.sizes() || q.sizes() != v.sizes() || q.numel() == 0) return false;
    if (!q.is_cuda() || dtype_code(q.scalar_type()) < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
    if (q.device().index() != c10::hip::current_device()) return false;
    for (const at::Tensor* t : {c.q, c.k, c.v})
        if (!tdb_host_plain(*t, q, c.grad) || !rows_ok(*t)) return false;
    return true;
}

// span and delta table of sequences up to max_len; false where no such table has been handed over
bool fill_delta(tdb_pos_args& pos, int64_t buckets, int64_t max_rel, int64_t max_len, int device) {
    const int64_t span = buckets > 0 ? buckets : max_rel;
    if (span < 1) return false;
    int64_t size = 512;
    while (size < max_len) size *= 2;
    for (const Lut& l : luts())
        if (l.device == device && l.size == size && l.buckets == buckets && l.max_rel == max_rel) {
            pos.span = int32_t(span);
            pos.lut_half = int32_t(size - 1);
            pos.delta_lut = static_cast<const int32_t*>(l.table.data_ptr());
            return true;
        }
    return false;
}

bool fill_pos(tdb_pos_args& pos, const Common& c, int64_t heads, int64_t head_dim, int64_t max_len) {
    const at::Tensor& q = *c.q;
    if ((c.q_pos && c.pk) || (c.k_pos && c.pq)) return false;
    if (!c.q_pos && !c.k_pos && !c.pk && !c.pq) return true;
    if (!fill_delta(pos, c.buckets, c.max_rel, max_len, q.device().index())) return false;
    const int64_t span = pos.span;
    for (int n = 0; n < 2; ++n) {
        const at::Tensor* t = n ? c.pq : c.pk;
        if (!t) continue;
        const int64_t lead = t->dim() - 3;      // [H, rows, D], or with a leading 1
        if (lead < 0 || lead > 1 || (lead == 1 && t->size(0) != 1) || t->size(lead) != heads || t->size(lead + 1) < 2 * span ||
            t->size(lead + 2) != head_dim || t->scalar_type() != q.scalar_type() || !tdb_host_plain(*t, q, c.grad) || !rows_ok(*t))
            return false;
        if (n) {
            pos.pos_query = t->data_ptr();
            pos.pos_query_stride_h = t->stride(lead);
            pos.pos_query_stride_r = t->stride(lead + 1);
        } else {
            pos.pos_key = t->data_ptr();
            pos.pos_key_stride_h = t->stride(lead);
            pos.pos_key_stride_r = t->stride(lead + 1);
        }
    }
    const int64_t outer = q.dim() - 1;
    for (int n = 0; n < 2; ++n) {
        const at::Tensor* t = n ? c.k_pos : c.q_pos;
        if (!t) continue;
        if (t->dim() != outer + 1 || t->sizes().slice(0, outer) != q.sizes().slice(0, outer) || t->size(outer) != 2 * span ||
            t->stride(outer) != 1 || t->scalar_type() != q.scalar_type() || !tdb_host_plain(*t, q, c.grad))
            return false;
        const int64_t sb = outer == 3 ? t->stride(0) : 0;
        const int64_t sh = t->stride(1), sl = outer == 3 ? t->stride(2) : t->stride(0);
        if (n) {
            pos.p2c_strip = t->data_ptr();
            pos.p2c_stride_b = sb, pos.p2c_stride_h = sh, pos.p2c_stride_l = sl;
        } else {
            pos.c2p_strip = t->data_ptr();
            pos.c2p_stride_b = sb, pos.c2p_stride_h = sh, pos.c2p_stride_l = sl;
        }
    }
    return true;
}

bool int32_vector(const at::Tensor& t, const at::Tensor& q, bool grad) {
    return t.dim() == 1 && t.scalar_type() == at::kInt && t.is_contiguous() && tdb_host_plain(t, q, grad);
}

void* stream_of(const at::Tensor& q) { return c10::hip::getCurrentHIPStream(q.device().index()).stream(); }

// A launch that the C ABI refuses is repeated by the Python path, which raises its message.
PyObject* finish(int rc, at::Tensor&& o) {
    if (rc != TDB_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(o));
}

// fixed(q, k, v, q_pos, k_pos, causal, sm_scale, position_buckets, max_relative_distance, pos_key_layer,
//       pos_query_layer, seqlens_k, force_generic)
PyObject* py_fixed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 13 || !g_fixed || tdb_host_observed()) Py_RETURN_NONE;
    try {
        bool ok = true, causal, generic;
        Common c;
        c.q = tensor(args[0], ok), c.k = tensor(args[1], ok), c.v = tensor(args[2], ok);
        c.q_pos = tensor(args[3], ok), c.k_pos = tensor(args[4], ok);
        c.pk = tensor(args[9], ok), c.pq = tensor(args[10], ok);
        const at::Tensor* lens = tensor(args[11], ok);
        c.grad = c10::GradMode::is_enabled();
        tdb_fixed_args a;
        memset(&a, 0, sizeof(a));
        if (!ok || !c.q || !c.k || !c.v || !as_flag(args[5], causal) || causal || !as_flag(args[12], generic) ||
            !as_int(args[7], c.buckets) || !as_int(args[8], c.max_rel) || !inputs_ok(c, 4))
            Py_RETURN_NONE;
        const at::Tensor &q = *c.q, &k = *c.k, &v = *c.v;
        const int64_t B = q.size(0), H = q.size(1), L = q.size(2), D = q.size(3);
        if (B > INT32_MAX || H > INT32_MAX || L > INT32_MAX || D > INT32_MAX) Py_RETURN_NONE;
        if (!as_scale(args[6], D, a.sm_scale) || !fill_pos(a.pos, c, H, D, L)) Py_RETURN_NONE;
        if (lens) {
            if (!int32_vector(*lens, q, c.grad) || lens->size(0) != B) Py_RETURN_NONE;
            a.seqlens_k = static_cast<const int32_t*>(lens->data_ptr());
        }
        at::Tensor o;
        if (!output_like(q, o)) Py_RETURN_NONE;
        a.dtype = dtype_code(q.scalar_type());
        a.batch = int32_t(B), a.heads = int32_t(H), a.head_dim = int32_t(D), a.seqlen = int32_t(L);
        a.flags = generic ? TDB_FLAG_FORCE_GENERIC : 0;
        a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr(), a.o = o.data_ptr();
        a.q_stride_b = q.stride(0), a.q_stride_h = q.stride(1), a.q_stride_l = q.stride(2);
        a.k_stride_b = k.stride(0), a.k_stride_h = k.stride(1), a.k_stride_l = k.stride(2);
        a.v_stride_b = v.stride(0), a.v_stride_h = v.stride(1), a.v_stride_l = v.stride(2);
        a.o_stride_b = o.stride(0), a.o_stride_h = o.stride(1), a.o_stride_l = o.stride(2);
        return finish(g_fixed(&a, stream_of(q)), std::move(o));
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// varlen(q, k, v, q_pos, k_pos, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, causal, sm_scale,
//        position_buckets, max_relative_distance, pos_key_layer, pos_query_layer, force_generic, zero_output)
PyObject* py_varlen(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 17 || !g_varlen || tdb_host_observed()) Py_RETURN_NONE;
    try {
        bool ok = true, causal, generic, zero;
        Common c;
        int64_t mq, mk;
        c.q = tensor(args[0], ok), c.k = tensor(args[1], ok), c.v = tensor(args[2], ok);
        c.q_pos = tensor(args[3], ok), c.k_pos = tensor(args[4], ok);
        const at::Tensor *cu = tensor(args[5], ok), *cu_k = tensor(args[6], ok);
        c.pk = tensor(args[13], ok), c.pq = tensor(args[14], ok);
        c.grad = c10::GradMode::is_enabled();
        tdb_varlen_args a;
        memset(&a, 0, sizeof(a));
        if (!ok || !c.q || !c.k || !c.v || !cu || !cu_k || !as_int(args[7], mq) || !as_int(args[8], mk) || mq != mk ||
            !as_flag(args[9], causal) || causal || !as_flag(args[15], generic) || !as_flag(args[16], zero) ||
            !as_int(args[11], c.buckets) || !as_int(args[12], c.max_rel) || !inputs_ok(c, 3))
            Py_RETURN_NONE;
        const at::Tensor &q = *c.q, &k = *c.k, &v = *c.v;
        const int64_t T = q.size(0), H = q.size(1), D = q.size(2);
        if (T > INT32_MAX || H > INT32_MAX || D > INT32_MAX) Py_RETURN_NONE;
        if (!int32_vector(*cu, q, c.grad) || cu->size(0) < 1 || cu_k->sizes() != cu->sizes() || cu_k->device() != q.device()) Py_RETURN_NONE;
        a.max_seqlen = int32_t(mq < 1 ? 1 : mq);
        if (!as_scale(args[10], D, a.sm_scale) || !fill_pos(a.pos, c, H, D, a.max_seqlen)) Py_RETURN_NONE;
        at::Tensor o;
        if (!output_like(q, o)) Py_RETURN_NONE;
        if (zero && cu->size(0) == 1) o.zero_();       // (no sequence: nothing is launched)
        a.dtype = dtype_code(q.scalar_type());
        a.batch = int32_t(cu->size(0) - 1), a.heads = int32_t(H), a.head_dim = int32_t(D), a.total_tokens = int32_t(T);
        a.flags = (generic ? TDB_FLAG_FORCE_GENERIC : 0) | (zero ? TDB_FLAG_ZERO_UNCOVERED : 0);
        a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr(), a.o = o.data_ptr();
        a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1);
        a.k_stride_t = k.stride(0), a.k_stride_h = k.stride(1);
        a.v_stride_t = v.stride(0), a.v_stride_h = v.stride(1);
        a.o_stride_t = o.stride(0), a.o_stride_h = o.stride(1);
        a.cu_seqlens = static_cast<const int32_t*>(cu->data_ptr());
        return finish(g_varlen(&a, stream_of(q)), std::move(o));
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// bind(address of tdb_attn_fwd_fixed, address of tdb_attn_fwd_varlen)
PyObject* py_bind(PyObject*, PyObject* args) {
    unsigned long long f, v;
    if (!PyArg_ParseTuple(args, "KK", &f, &v)) return nullptr;
    g_fixed = reinterpret_cast<decltype(g_fixed)>(f);
    g_varlen = reinterpret_cast<decltype(g_varlen)>(v);
    Py_RETURN_NONE;
}

// add_lut(table, size, position_buckets, max_relative_distance): a device table to be found by later calls
PyObject* py_add_lut(PyObject*, PyObject* args) {
    PyObject* t;
    long long size, buckets, max_rel;
    if (!PyArg_ParseTuple(args, "OLLL", &t, &size, &buckets, &max_rel)) return nullptr;
    if (!THPVariable_Check(t)) {
        PyErr_SetString(PyExc_TypeError, "add_lut: a tensor is expected");
        return nullptr;
    }
    const at::Tensor& table = THPVariable_Unpack(t);
    luts().push_back(Lut{table.device().index(), size, buckets, max_rel, table});
    Py_RETURN_NONE;
}

// observed(): see tdb_host_observed
PyObject* py_observed(PyObject*, PyObject*) { return PyBool_FromLong(tdb_host_observed()); }

PyMethodDef kMethods[] = {
    {"observed", py_observed, METH_NOARGS, nullptr},
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"add_lut", py_add_lut, METH_VARARGS, nullptr},
    {"fixed", reinterpret_cast<PyCFunction>(py_fixed), METH_FASTCALL, nullptr},
    {"varlen", reinterpret_cast<PyCFunction>(py_varlen), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods};

}  // namespace

int (*tdb_host_fixed())(const tdb_fixed_args*, void*) { return g_fixed; }
int (*tdb_host_varlen())(const tdb_varlen_args*, void*) { return g_varlen; }

bool tdb_host_plain(const at::Tensor& t, const at::Tensor& q, bool grad) {
    static const c10::DispatchKeySet wrapped({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::Batched});
    if (t.key_set().has_any(wrapped)) return false;
    if (t.unsafeGetTensorImpl()->autograd_meta() && t._fw_grad(0).defined()) return false;
    return t.device() == q.device() && t.layout() == at::kStrided && !(grad && t.requires_grad()) && !t.is_neg() && !t.is_conj();
}

bool tdb_host_observed() { return c10::impl::dispatch_mode_enabled() || at::tracer::impl::is_dispatch_enabled(); }

bool tdb_host_fill_tables(tdb_pos_args& pos, const at::Tensor* pk, const at::Tensor* pq, int64_t buckets, int64_t max_rel, int64_t max_len, int device) {
    if (!pk && !pq) return true;
    if (!fill_delta(pos, buckets, max_rel, max_len, device)) return false;
    if (pk) pos.pos_key = pk->data_ptr(), pos.pos_key_stride_h = pk->stride(-3), pos.pos_key_stride_r = pk->stride(-2);
    if (pq) pos.pos_query = pq->data_ptr(), pos.pos_query_stride_h = pq->stride(-3), pos.pos_query_stride_r = pq->stride(-2);
    return true;
}

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&kModule);
    if (m && !tdb_host_add_encoder(m)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
