// Native encoder loop: a patched model's eval-mode forward from token ids to the last hidden state, as one call.
//
// What bounds a short request is the host: a 48-token text through 12 layers spent 2.4 ms in Python modules and the
// dispatch of 158 small kernels where the weights can be read in 38 us.  A *plan* holds what the loop needs of each layer
// (weights, the concatenated Q/K/V weight, the position tables) together with a snapshot of the module tree; every call
// first compares the tree with the snapshot -- types and their methods, children, parameters and their modification
// counters, attributes, training flags, hooks, replaced forwards -- and a difference makes the caller build a new plan or
// take the modules as they are.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include <chrono>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "host.h"
#include "tdb_attn.h"
#include "tdb_encoder.h"

namespace {

struct Enc {
    decltype(&tdb_enc_scan_mask) scan_mask;
    decltype(&tdb_enc_embed) embed;
    decltype(&tdb_enc_add_norm) add_norm;
    decltype(&tdb_enc_small_gemm) small_gemm;
    decltype(&tdb_enc_small_tiles) small_tiles;
    decltype(&tdb_enc_small_splits) small_splits;
    decltype(&tdb_enc_unpack) unpack;
    decltype(&tdb_enc_gemm) gemm;
    decltype(&tdb_enc_gemm_splits) gemm_splits;
    decltype(&tdb_enc_rows_fused) rows_fused;
    decltype(&tdb_enc_embed_rows) embed_rows;
    decltype(&tdb_enc_norm_gemm) norm_gemm;
    decltype(&tdb_enc_gemm_add) gemm_add;
    decltype(&tdb_enc_norm_rows) norm_rows;
} g_enc = {};

struct Decref {
    void operator()(PyObject* o) const { Py_XDECREF(o); }
};
using Owned = std::unique_ptr<PyObject, Decref>;

// Names looked up in module dictionaries (interned once, kept for the process).
PyObject* name(const char* s) { return PyUnicode_InternFromString(s); }
struct Names {
    PyObject *training = name("training"), *forward = name("forward"), *params = name("_parameters"), *modules = name("_modules"),
             *hooks = name("_forward_hooks"), *pre_hooks = name("_forward_pre_hooks");
    // methods of a module's type that the loop stands in for
    PyObject* methods[4] = {forward, name("__call__"), name("forward_packed"), name("get_rel_embedding")};
};
const Names& names() {
    static const Names* n = new Names;
    return *n;
}

// One module of the snapshot.  Module objects are compared by address and not owned (the plan must not keep its model
// alive): the root is alive during the call, and every other one is reached through its parent's verified dictionary.
struct ModuleRef {
    PyObject* object;
    PyTypeObject* type;
    struct Child {
        Owned key;
        PyObject* object;                   // a module, or None
        int index;                          // in the snapshot; -1 for None
    };
    struct Param {
        Owned key;
        at::Tensor tensor;                  // undefined for None
        uint32_t version;
        void* data;
    };
    struct Attr {                           // what else its dictionary holds: sizes, eps, an activation's function, ...
        Owned key, value;                   // (value: kept alive where it cannot be what keeps the model alive)
        PyObject* object;
    };
    std::vector<Child> children;
    std::vector<Param> params;
    std::vector<Attr> attrs;                // (not of the root, which callers may write to as they like)
    mutable uint64_t state;                 // of the dictionary when it last was as it should be
};

// A type of the tree and what its methods were (null: none of that name).
struct TypeRef {
    Owned type;
    Owned methods[4];
};

struct Layer {
    at::Tensor wqkv, bqkv, pk, pq, wo, bo, g1, b1, wi, bi, wf, bf, g2, b2;
    double eps1, eps2;
};

struct Plan {
    std::vector<ModuleRef> tree;
    std::vector<TypeRef> types;
    std::vector<Layer> layers;
    at::Tensor emb, emb_g, emb_b;
    double emb_eps;
    int64_t heads, head_dim, buckets, max_rel;
    float scale;
};
const char* const kPlan = "turbodeberta_amd.plan";

PyObject* dict_of(PyObject* module) {
    PyObject** d = _PyObject_GetDictPtr(module);
    return d ? *d : nullptr;
}

bool empty_dict(PyObject* dict, PyObject* key) {
    PyObject* v = PyDict_GetItem(dict, key);
    return v && PyDict_Check(v) && PyDict_GET_SIZE(v) == 0;
}

// What a module keeps for itself (its registries, which are looked at one by one, and caches).
bool is_private(PyObject* key) {
    return PyUnicode_Check(key) && PyUnicode_READY(key) == 0 && PyUnicode_GET_LENGTH(key) > 0 && PyUnicode_READ_CHAR(key, 0) == '_';
}

// The other attributes of an instance dictionary, in their order and by identity.
bool attrs_ok(const ModuleRef& m, PyObject* dict) {
    size_t n = 0;
    PyObject *k, *v;
    Py_ssize_t pos = 0;
    while (PyDict_Next(dict, &pos, &k, &v)) {
        if (n < m.attrs.size() && k == m.attrs[n].key.get() && v == m.attrs[n].object) ++n;
        else if (!is_private(k)) return false;
    }
    return n == m.attrs.size();
}

// A number that no other state of any dictionary has, or 0.
uint64_t state_of(PyObject* dict) {
#if PY_VERSION_HEX < 0x030c0000
    return reinterpret_cast<PyDictObject*>(dict)->ma_version_tag;
#else
    return 0;
#endif
}

bool module_ok(const ModuleRef& m, bool attrs) {
    const Names& n = names();
    if (Py_TYPE(m.object) != m.type) return false;
    PyObject* d = dict_of(m.object);
    if (!d) return false;
    if (!m.state || state_of(d) != m.state) {
        if (PyDict_GetItem(d, n.training) != Py_False || PyDict_GetItem(d, n.forward) || (attrs && !attrs_ok(m, d))) return false;
        m.state = state_of(d);
    }
    if (!empty_dict(d, n.hooks) || !empty_dict(d, n.pre_hooks)) return false;
    PyObject *params = PyDict_GetItem(d, n.params), *modules = PyDict_GetItem(d, n.modules);
    if (!params || !PyDict_Check(params) || PyDict_GET_SIZE(params) != Py_ssize_t(m.params.size())) return false;
    if (!modules || !PyDict_Check(modules) || PyDict_GET_SIZE(modules) != Py_ssize_t(m.children.size())) return false;
    for (const auto& p : m.params) {
        PyObject* o = PyDict_GetItem(params, p.key.get());
        if (!o) return false;
        if (!p.tensor.defined()) {
            if (o != Py_None) return false;
            continue;
        }
        if (!THPVariable_Check(o)) return false;
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.unsafeGetTensorImpl() != p.tensor.unsafeGetTensorImpl() || t._version() != p.version || t.data_ptr() != p.data) return false;
    }
    for (const auto& c : m.children)
        if (PyDict_GetItem(modules, c.key.get()) != c.object) return false;
    return true;
}

PyTypeObject* as_type(const Owned& o) { return reinterpret_cast<PyTypeObject*>(o.get()); }

bool tree_ok(const Plan& plan, PyObject* root) {
    if (plan.tree.empty() || plan.tree[0].object != root) return false;
    for (const auto& t : plan.types)
        for (int i = 0; i < 4; ++i)
            if (_PyType_Lookup(as_type(t.type), names().methods[i]) != t.methods[i].get()) return false;
    for (const auto& m : plan.tree)         // parents come before their children
        if (!module_ok(m, m.object != root)) return false;
    return true;
}

// Appends `module` and what is below it; false where something cannot be held to account later.
bool snapshot(Plan& plan, PyObject* module) {
    const Names& n = names();
    PyObject* d = dict_of(module);
    if (!d) return false;
    PyObject *params = PyDict_GetItem(d, n.params), *modules = PyDict_GetItem(d, n.modules);
    if (!params || !PyDict_Check(params) || !modules || !PyDict_Check(modules)) return false;
    const size_t at = plan.tree.size();
    plan.tree.emplace_back();
    plan.tree[at].object = module;
    plan.tree[at].type = Py_TYPE(module);
    plan.tree[at].state = 0;
    bool known = false;
    for (const auto& t : plan.types) known = known || as_type(t.type) == Py_TYPE(module);
    if (!known) {
        TypeRef t;
        auto own = [](Owned& to, PyObject* o) {
            Py_XINCREF(o);
            to.reset(o);
        };
        own(t.type, reinterpret_cast<PyObject*>(Py_TYPE(module)));
        for (int i = 0; i < 4; ++i) own(t.methods[i], _PyType_Lookup(Py_TYPE(module), n.methods[i]));
        plan.types.push_back(std::move(t));
    }
    PyObject *k, *v;
    Py_ssize_t pos = 0;
    while (PyDict_Next(d, &pos, &k, &v))
        if (PyType_HasFeature(Py_TYPE(v), Py_TPFLAGS_HEAPTYPE) && PyType_IsSubtype(Py_TYPE(v), reinterpret_cast<PyTypeObject*>(THPVariableClass)))
            return false;                   // a weight that is no parameter
    pos = 0;
    while (PyDict_Next(params, &pos, &k, &v)) {
        ModuleRef::Param p;
        Py_INCREF(k);
        p.key.reset(k);
        p.version = 0, p.data = nullptr;
        if (v != Py_None) {
            if (!THPVariable_CheckExact(v)) return false;
            p.tensor = THPVariable_Unpack(v);
            if (!tdb_host_plain(p.tensor, p.tensor, false) || p.tensor.is_inference()) return false;       // (inference: no modification counter)
            p.version = p.tensor._version();
            p.data = p.tensor.data_ptr();
        }
        plan.tree[at].params.push_back(std::move(p));
    }
    pos = 0;
    if (at > 0) plan.tree[at].attrs.reserve(8);
    while (at > 0 && PyDict_Next(d, &pos, &k, &v))
        if (!is_private(k)) {
            ModuleRef::Attr a;
            Py_INCREF(k);
            a.key.reset(k);
            a.object = v;
            if (!PyCallable_Check(v) || PyCFunction_Check(v)) {
                Py_INCREF(v);
                a.value.reset(v);
            }
            plan.tree[at].attrs.push_back(std::move(a));
        }
    pos = 0;
    std::vector<PyObject*> below;
    while (PyDict_Next(modules, &pos, &k, &v)) {
        ModuleRef::Child c;
        Py_INCREF(k);
        c.key.reset(k);
        c.object = v;
        plan.tree[at].children.push_back(std::move(c));
        if (v != Py_None) below.push_back(v);
    }
    for (PyObject* m : below)
        if (!snapshot(plan, m)) return false;
    return module_ok(plan.tree[at], at > 0);
}

Plan* plan_of(PyObject* o) { return static_cast<Plan*>(PyCapsule_GetPointer(o, kPlan)); }

bool get_tensor(PyObject* tuple, Py_ssize_t i, at::Tensor& t, bool optional = false) {
    PyObject* o = PyTuple_GetItem(tuple, i);
    if (!o) return false;
    if (optional && o == Py_None) return true;
    if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "plan: a tensor is expected");
        return false;
    }
    t = THPVariable_Unpack(o);
    return true;
}

hipStream_t current_stream(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void must(int hip_error) { TORCH_CHECK(hip_error == 0, "kernel launch failed: ", hipGetErrorString(hipError_t(hip_error))); }

int mask_type(at::ScalarType t) {
    switch (t) {
        case at::kLong: return TDB_MASK_I64;
        case at::kInt: return TDB_MASK_I32;
        case at::kBool: case at::kByte: return TDB_MASK_U8;
        case at::kFloat: return TDB_F32;
        case at::kBFloat16: return TDB_BF16;
        case at::kHalf: return TDB_F16;
        default: return -1;
    }
}

// Undefined where the attention is refused (a head size, a length): the modules raise its message.
at::Tensor encode(const Plan& p, const at::Tensor& ids, const at::Tensor* cu, int64_t T) {
    const int64_t B = ids.size(0), L = ids.size(1), H = p.heads, D = p.head_dim, hidden = p.emb.size(1);
    const auto type = p.emb.scalar_type();
    const auto device = p.emb.device();
    const int dt = type == at::kFloat ? TDB_F32 : type == at::kBFloat16 ? TDB_BF16 : TDB_F16;
    hipStream_t s = current_stream(p.emb);
    auto empty = [&](at::IntArrayRef size, at::ScalarType t) { return at::detail::empty_cuda(size, t, device, std::nullopt); };
    const int32_t* bounds = cu ? static_cast<const int32_t*>(cu->data_ptr()) : nullptr;

    const int64_t inner = p.layers[0].wi.size(0);
    const int tiles[] = {g_enc.small_tiles(int(T), int(3 * hidden), int(hidden), dt), g_enc.small_tiles(int(T), int(hidden), int(inner), dt),
                         g_enc.small_tiles(int(T), int(inner), int(hidden), dt)};
    const bool small = tiles[0] && tiles[1] && tiles[2];
    const int mt = small ? tiles[0] : 0;    // (the same for all three)
    const bool fused = small && g_enc.rows_fused(int(T), int(hidden), int(inner), dt);
    const int64_t rows = small ? 16 * mt : T;
    // Contractions with hidden-sized outputs are split where the output alone gives the CUs too little to do; the add + norm
    // behind them adds the parts up.
    const int few = g_enc.small_splits(int(hidden));
    const int splits_o = small ? few : g_enc.gemm_splits(int(T), int(hidden), int(hidden), dt);
    const int splits_f = small ? few : g_enc.gemm_splits(int(T), int(hidden), int(inner), dt);
    const bool own = !small && splits_o && splits_f && g_enc.gemm_splits(int(T), int(3 * hidden), int(hidden), dt) && g_enc.gemm_splits(int(T), int(inner), int(hidden), dt);
    at::Tensor attended = empty({T, hidden}, type);
    at::Tensor x, y, last, qkv, ff, part, proj;
    // Rows before their LayerNorm: those that a layer starts from, and those between its attention and its feed-forward products.
    at::Tensor wide[2];
    tdb_enc_rows from{}, between{};
    if (fused) {
        const int64_t sums = hidden / 8;    // (floats of a row)
        for (at::Tensor& w : wide) w = empty({rows, hidden + sums}, at::kFloat);
        auto rows_in = [&](const at::Tensor& w) {
            const float* const at = static_cast<const float*>(w.data_ptr());
            return tdb_enc_rows{at, at + rows * hidden, p.emb_g.data_ptr(), p.emb_b.data_ptr(), float(p.emb_eps)};
        };
        from = rows_in(wide[0]), between = rows_in(wide[1]);
    } else {
        x = empty({rows, hidden}, type), y = empty({rows, hidden}, type);
    }
    last = small ? empty({T, hidden}, type) : x;                        // the last layer's output, row after row
    if (small || own) qkv = empty({T, 3 * hidden}, type), ff = empty({rows, inner}, type);
    if ((small && !fused) || (own && std::max(splits_o, splits_f) > 1)) part = empty({std::max(splits_o, splits_f), T, hidden}, at::kFloat);
    if (own && std::min(splits_o, splits_f) == 1) proj = empty({T, hidden}, type);
    auto writable = [](const float* rows) { return const_cast<float*>(rows); };
    if (fused)
        must(g_enc.embed_rows(ids.data_ptr(), ids.scalar_type() == at::kLong, p.emb.data_ptr(), p.emb.size(0), bounds, int(B), int(L), int(T), int(hidden), dt, mt,
                              writable(from.x), writable(from.stats), s));
    else
        must(g_enc.embed(ids.data_ptr(), ids.scalar_type() == at::kLong, p.emb.data_ptr(), p.emb.size(0), p.emb_g.data_ptr(), p.emb_b.data_ptr(),
                     float(p.emb_eps), bounds, int(B), int(L), int(T), int(hidden), dt, mt, x.data_ptr(), s));
    auto ptr = [](const at::Tensor& t) { return t.data_ptr(); };
    auto norm = [&](const at::Tensor& d, int splits, const at::Tensor& bias, const at::Tensor& res, const at::Tensor& g, const at::Tensor& b, double eps, at::Tensor& out, int mt_out) {
        must(g_enc.add_norm(ptr(d), splits, ptr(bias), ptr(res), ptr(g), ptr(b), float(eps), int(T), int(hidden), dt, mt, mt_out, ptr(out), s));
    };
    for (const Layer& w : p.layers) {
        auto weight = [&](const at::Tensor& t, int norm) { return tdb_enc_next{t.data_ptr(), int(t.size(0)), int(t.size(1)), norm}; };
        const tdb_enc_next next[] = {weight(w.wo, 0), weight(w.wi, 1), weight(w.wf, 0), &w != &p.layers.back() ? weight((&w + 1)->wqkv, 1) : tdb_enc_next{}};
        if (fused) must(g_enc.norm_gemm(&from, ptr(w.wqkv), ptr(w.bqkv), 0, int(T), int(3 * hidden), int(hidden), dt, next, 1, ptr(qkv), s));
        else if (small) must(g_enc.small_gemm(ptr(x), ptr(w.wqkv), ptr(w.bqkv), TDB_ENC_IN, 0, int(T), int(3 * hidden), int(hidden), dt, ptr(qkv), s));
        else if (own) must(g_enc.gemm(ptr(x), ptr(w.wqkv), ptr(w.bqkv), 0, 1, int(T), int(3 * hidden), int(hidden), dt, ptr(qkv), s));
        else qkv = at::addmm(w.bqkv, x, w.wqkv.t());
        tdb_pos_args pos;
        memset(&pos, 0, sizeof(pos));
        TORCH_CHECK(tdb_host_fill_tables(pos, w.pk.defined() ? &w.pk : nullptr, w.pq.defined() ? &w.pq : nullptr, p.buckets, p.max_rel, L, device.index()),
                    "no position table for this length");
        const int64_t es = qkv.element_size();
        char* const base = static_cast<char*>(qkv.data_ptr());
        int rc;
        if (cu) {
            tdb_varlen_args a;
            memset(&a, 0, sizeof(a));
            a.dtype = dt, a.batch = int32_t(B), a.heads = int32_t(H), a.head_dim = int32_t(D);
            a.total_tokens = int32_t(T), a.max_seqlen = int32_t(L), a.sm_scale = p.scale;
            a.q = base, a.k = base + hidden * es, a.v = base + 2 * hidden * es, a.o = attended.data_ptr();
            a.q_stride_t = a.k_stride_t = a.v_stride_t = 3 * hidden, a.o_stride_t = hidden;
            a.q_stride_h = a.k_stride_h = a.v_stride_h = a.o_stride_h = D;
            a.cu_seqlens = bounds, a.pos = pos;
            rc = tdb_host_varlen()(&a, s);
        } else {
            tdb_fixed_args a;
            memset(&a, 0, sizeof(a));
            a.dtype = dt, a.batch = int32_t(B), a.heads = int32_t(H), a.head_dim = int32_t(D), a.seqlen = int32_t(L), a.sm_scale = p.scale;
            a.q = base, a.k = base + hidden * es, a.v = base + 2 * hidden * es, a.o = attended.data_ptr();
            a.q_stride_b = a.k_stride_b = a.v_stride_b = L * 3 * hidden, a.o_stride_b = L * hidden;
            a.q_stride_l = a.k_stride_l = a.v_stride_l = 3 * hidden, a.o_stride_l = hidden;
            a.q_stride_h = a.k_stride_h = a.v_stride_h = a.o_stride_h = D;
            a.pos = pos;
            rc = tdb_host_fixed()(&a, s);
        }
        if (rc != TDB_OK) return at::Tensor();
        at::Tensor& out = &w == &p.layers.back() ? last : x;
        const int mt_out = &w == &p.layers.back() ? 0 : mt;
        if (fused) {
            must(g_enc.gemm_add(ptr(attended), 0, ptr(w.wo), ptr(w.bo), &from, int(T), int(hidden), int(hidden), dt, next + 1, 2, writable(between.x), writable(between.stats), s));
            between.gamma = ptr(w.g1), between.beta = ptr(w.b1), between.eps = float(w.eps1);
            must(g_enc.norm_gemm(&between, ptr(w.wi), ptr(w.bi), 1, int(T), int(inner), int(hidden), dt, nullptr, 0, ptr(ff), s));
            must(g_enc.gemm_add(ptr(ff), 1, ptr(w.wf), ptr(w.bf), &between, int(T), int(hidden), int(inner), dt, next + 3, 1, writable(from.x), writable(from.stats), s));
            from.gamma = ptr(w.g2), from.beta = ptr(w.b2), from.eps = float(w.eps2);
        } else if (small) {
            must(g_enc.small_gemm(ptr(attended), ptr(w.wo), nullptr, 0, few, int(T), int(hidden), int(hidden), dt, ptr(part), s));
            norm(part, few, w.bo, x, w.g1, w.b1, w.eps1, y, mt);
            must(g_enc.small_gemm(ptr(y), ptr(w.wi), ptr(w.bi), TDB_ENC_IN | TDB_ENC_OUT | TDB_ENC_GELU, 0, int(T), int(inner), int(hidden), dt, ptr(ff), s));
            must(g_enc.small_gemm(ptr(ff), ptr(w.wf), nullptr, TDB_ENC_IN, few, int(T), int(hidden), int(inner), dt, ptr(part), s));
            norm(part, few, w.bf, y, w.g2, w.b2, w.eps2, out, mt_out);
        } else if (own) {
            auto product = [&](const at::Tensor& in, const at::Tensor& weight, const at::Tensor& bias, int splits, int64_t k) {
                at::Tensor& d = splits > 1 ? part : proj;
                must(g_enc.gemm(ptr(in), ptr(weight), ptr(bias), 0, splits, int(T), int(hidden), int(k), dt, ptr(d), s));
                return d;
            };
            norm(product(attended, w.wo, w.bo, splits_o, hidden), splits_o > 1 ? splits_o : 0, w.bo, x, w.g1, w.b1, w.eps1, y, 0);
            must(g_enc.gemm(ptr(y), ptr(w.wi), ptr(w.bi), TDB_ENC_GELU, 1, int(T), int(inner), int(hidden), dt, ptr(ff), s));
            norm(product(ff, w.wf, w.bf, splits_f, inner), splits_f > 1 ? splits_f : 0, w.bf, y, w.g2, w.b2, w.eps2, out, 0);
        } else {
            norm(at::addmm(w.bo, attended, w.wo.t()), 0, w.bo, x, w.g1, w.b1, w.eps1, y, 0);
            at::Tensor f = at::addmm(w.bi, y, w.wi.t());
            at::gelu_(f);
            norm(at::addmm(w.bf, f, w.wf.t()), 0, w.bf, y, w.g2, w.b2, w.eps2, out, 0);
        }
    }
    if (fused) must(g_enc.norm_rows(&from, int(T), int(hidden), dt, ptr(last), s));
    if (!cu) return last.view({B, L, hidden});
    at::Tensor out = empty({B, L, hidden}, type);
    must(g_enc.unpack(ptr(last), bounds, int(B), int(L), int(T), int(hidden), dt, ptr(out), s));
    return out;
}

#define TDB_TRY try {
#define TDB_CATCH                                                    \
    }                                                                \
    catch (const std::exception& e) {                                \
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what()); \
        return nullptr;                                              \
    }

// begin_plan(root): a plan that holds the snapshot only, or None where the tree below `root` cannot be held to account (a module
// in training mode, a hook, a forward of its own, parameters that are not plain or have no modification counter)
PyObject* py_begin_plan(PyObject*, PyObject* root) {
    TDB_TRY
    auto plan = std::make_unique<Plan>();
    if (!snapshot(*plan, root)) Py_RETURN_NONE;
    return PyCapsule_New(plan.release(), kPlan, [](PyObject* c) { delete plan_of(c); });
    TDB_CATCH
}

// complete_plan(plan, root, layers, embedding, heads, head_dim, scale, buckets, max_rel): whether the plan can be used; not where
// the tree has changed since it was begun.  layers: tuples of 14 tensors (tables may be None) and two epsilons.
PyObject* py_complete_plan(PyObject*, PyObject* args) {
    TDB_TRY
    PyObject *capsule, *root, *layers, *emb;
    long long heads, head_dim, buckets, max_rel;
    double scale;
    if (!PyArg_ParseTuple(args, "OOO!O!LLdLL", &capsule, &root, &PyList_Type, &layers, &PyTuple_Type, &emb, &heads, &head_dim, &scale, &buckets, &max_rel)) return nullptr;
    Plan* const plan = plan_of(capsule);
    if (!plan) return nullptr;
    plan->heads = heads, plan->head_dim = head_dim, plan->scale = float(scale), plan->buckets = buckets, plan->max_rel = max_rel;
    if (!get_tensor(emb, 0, plan->emb) || !get_tensor(emb, 1, plan->emb_g) || !get_tensor(emb, 2, plan->emb_b)) return nullptr;
    plan->emb_eps = PyFloat_AsDouble(PyTuple_GetItem(emb, 3));
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(layers); ++i) {
        PyObject* t = PyList_GET_ITEM(layers, i);
        Layer w;
        at::Tensor* const slots[] = {&w.wqkv, &w.bqkv, &w.pk, &w.pq, &w.wo, &w.bo, &w.g1, &w.b1, &w.wi, &w.bi, &w.wf, &w.bf, &w.g2, &w.b2};
        for (int k = 0; k < 14; ++k)
            if (!get_tensor(t, k, *slots[k], k == 2 || k == 3)) return nullptr;
        w.eps1 = PyFloat_AsDouble(PyTuple_GetItem(t, 14)), w.eps2 = PyFloat_AsDouble(PyTuple_GetItem(t, 15));
        plan->layers.push_back(std::move(w));
    }
    if (PyErr_Occurred()) return nullptr;
    return PyBool_FromLong(!plan->layers.empty() && tree_ok(*plan, root));
    TDB_CATCH
}

// plan_ok(plan, root)
PyObject* py_plan_ok(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TDB_TRY
    Plan* p = n == 2 ? plan_of(args[0]) : nullptr;
    if (!p) return nullptr;
    return PyBool_FromLong(tree_ok(*p, args[1]));
    TDB_CATCH
}

// Token ids that the kernels can read: [B, L] row after row, of x's device
bool ids_ok(const at::Tensor& ids, const at::Tensor& x) {
    return tdb_host_plain(ids, x, false) && ids.dim() == 2 && (ids.scalar_type() == at::kLong || ids.scalar_type() == at::kInt) && ids.is_contiguous();
}

// Pinned memory for the answers of mask scans: one page of slots for the process, handed out and given back with the GIL held,
// so that a call has a slot to itself whatever threads and streams there are.  (A slot whose kernel may still write to it,
// after an error, is not given back.)
struct Slot {
    int32_t flags[4], ticket;               // as tdb_enc_scan_mask writes them
    int32_t pad[11];                        // a cache line
};
constexpr int SLOTS = 64;
struct Slots {
    std::vector<Slot*> unused;
    bool ready = false;
} g_slots;

Slot* take_slot() {
    if (!g_slots.ready) {
        void* page = nullptr;
        if (hipHostMalloc(&page, SLOTS * sizeof(Slot), hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        memset(page, 0, SLOTS * sizeof(Slot));
        for (int i = 0; i < SLOTS; ++i) g_slots.unused.push_back(static_cast<Slot*>(page) + i);
        g_slots.ready = true;
    }
    if (g_slots.unused.empty()) return nullptr;
    Slot* s = g_slots.unused.back();
    g_slots.unused.pop_back();
    return s;
}

// scan_mask(mask [B, L]) -> (lengths, cu_seqlens, right_padded, total, ones), or None for a mask it does not take.
// scan_mask(mask, ids [B, L], vocab) -> the same and whether the ids of the valid tokens lie in [0, vocab) (ids that encode() does
// not take are not looked at).  Waits for the GPU.
PyObject* py_scan_mask(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TDB_TRY
    if ((n != 1 && n != 3) || tdb_host_observed() || !THPVariable_CheckExact(args[0])) Py_RETURN_NONE;
    const at::Tensor& m = THPVariable_Unpack(args[0]);
    if (!tdb_host_plain(m, m, false)) Py_RETURN_NONE;
    const int type = m.is_cuda() ? mask_type(m.scalar_type()) : -1;
    if (type < 0 || m.dim() != 2 || m.size(0) < 1 || m.size(0) > TDB_SCAN_MAX_BATCH || m.size(1) < 1 || m.size(1) > INT32_MAX ||
        m.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const void* ids = nullptr;
    int ids64 = 0;
    int64_t vocab = 0;
    if (n == 3 && THPVariable_CheckExact(args[1])) {
        const at::Tensor& t = THPVariable_Unpack(args[1]);
        vocab = PyLong_AsLongLong(args[2]);
        if (vocab == -1 && PyErr_Occurred()) return nullptr;
        if (ids_ok(t, m) && t.sizes() == m.sizes()) ids = t.data_ptr(), ids64 = t.scalar_type() == at::kLong;
    }
    const int64_t B = m.size(0);
    at::Tensor both = at::detail::empty_cuda({2 * B + 1}, at::kInt, m.device(), std::nullopt);
    int32_t* const lens = static_cast<int32_t*>(both.data_ptr());
    hipStream_t s = current_stream(m);
    // Watching the ticket that the kernel writes last is some 15 us quicker than waiting for the stream; what takes long (work
    // queued before it) waits for the stream.
    Slot* const slot = take_slot();
    if (!slot) Py_RETURN_NONE;
    const int32_t wanted = slot->ticket == INT32_MAX ? 1 : slot->ticket + 1;
    if (const int rc = g_enc.scan_mask(m.data_ptr(), type, m.stride(0), m.stride(1), int(B), int(m.size(1)), ids, ids64, vocab, lens, lens + B,
                                        reinterpret_cast<int32_t*>(slot), wanted, s)) {
        g_slots.unused.push_back(slot);     // (not launched)
        must(rc);
    }
    hipError_t e = hipSuccess;
    int32_t* const seen = &slot->ticket;
    Py_BEGIN_ALLOW_THREADS
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(20);
    while (__atomic_load_n(seen, __ATOMIC_ACQUIRE) != wanted)
        if (std::chrono::steady_clock::now() > until) {
            e = hipStreamSynchronize(s);
            break;
        }
    Py_END_ALLOW_THREADS
    TORCH_CHECK(e == hipSuccess, "attention mask: ", hipGetErrorString(e));
    const Slot got = *slot;
    g_slots.unused.push_back(slot);
    PyObject *lengths = THPVariable_Wrap(both.narrow(0, 0, B)), *cu = THPVariable_Wrap(both.narrow(0, B, B + 1));
    PyObject *right_padded = PyBool_FromLong(got.flags[0]), *ones = PyBool_FromLong(got.flags[2]);
    if (n == 1) return Py_BuildValue("(NNNiN)", lengths, cu, right_padded, int(got.flags[1]), ones);
    return Py_BuildValue("(NNNiNN)", lengths, cu, right_padded, int(got.flags[1]), ones, PyBool_FromLong(got.flags[3]));
    TDB_CATCH
}

// encode(plan, ids [B, L], cu_seqlens or None, tokens) -> last hidden state, or None for ids, boundaries or heads it does not take
PyObject* py_encode(PyObject*, PyObject* const* args, Py_ssize_t n) {
    TDB_TRY
    Plan* p = n == 4 ? plan_of(args[0]) : nullptr;
    if (!p) return nullptr;
    if (p->layers.empty() || tdb_host_observed() || !THPVariable_CheckExact(args[1]) || c10::GradMode::is_enabled()) Py_RETURN_NONE;
    const at::Tensor& ids = THPVariable_Unpack(args[1]);
    if (!ids_ok(ids, p->emb)) Py_RETURN_NONE;
    const at::Tensor* cu = nullptr;
    if (args[2] != Py_None) {
        if (!THPVariable_CheckExact(args[2])) Py_RETURN_NONE;
        cu = &THPVariable_Unpack(args[2]);
        if (!tdb_host_plain(*cu, ids, false) || cu->scalar_type() != at::kInt || cu->dim() != 1 || !cu->is_contiguous() || cu->size(0) != ids.size(0) + 1)
            Py_RETURN_NONE;
    }
    const int64_t T = PyLong_AsLongLong(args[3]);
    if (ids.device().index() != c10::hip::current_device() || T < 1 || ids.numel() > INT32_MAX || 3 * T * p->emb.size(1) > INT32_MAX)
        Py_RETURN_NONE;
    // (the boundaries may have been made on another stream and belong to the mask, whose owner does not know of them)
    if (cu) c10::hip::HIPCachingAllocator::recordStream(cu->storage().data_ptr(), c10::hip::getCurrentHIPStream(ids.device().index()));
    at::Tensor out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        out = encode(*p, ids, cu, T);
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    TDB_CATCH
}

// bind_encoder(addresses of the tdb_enc_* functions in the order of Enc)
PyObject* py_bind_encoder(PyObject*, PyObject* args) {
    unsigned long long f[14];
    if (!PyArg_ParseTuple(args, "KKKKKKKKKKKKKK", f, f + 1, f + 2, f + 3, f + 4, f + 5, f + 6, f + 7, f + 8, f + 9, f + 10, f + 11, f + 12, f + 13)) return nullptr;
    g_enc.scan_mask = reinterpret_cast<decltype(g_enc.scan_mask)>(f[0]);
    g_enc.embed = reinterpret_cast<decltype(g_enc.embed)>(f[1]);
    g_enc.add_norm = reinterpret_cast<decltype(g_enc.add_norm)>(f[2]);
    g_enc.small_gemm = reinterpret_cast<decltype(g_enc.small_gemm)>(f[3]);
    g_enc.small_tiles = reinterpret_cast<decltype(g_enc.small_tiles)>(f[4]);
    g_enc.small_splits = reinterpret_cast<decltype(g_enc.small_splits)>(f[5]);
    g_enc.unpack = reinterpret_cast<decltype(g_enc.unpack)>(f[6]);
    g_enc.gemm = reinterpret_cast<decltype(g_enc.gemm)>(f[7]);
    g_enc.gemm_splits = reinterpret_cast<decltype(g_enc.gemm_splits)>(f[8]);
    g_enc.rows_fused = reinterpret_cast<decltype(g_enc.rows_fused)>(f[9]);
    g_enc.embed_rows = reinterpret_cast<decltype(g_enc.embed_rows)>(f[10]);
    g_enc.norm_gemm = reinterpret_cast<decltype(g_enc.norm_gemm)>(f[11]);
    g_enc.gemm_add = reinterpret_cast<decltype(g_enc.gemm_add)>(f[12]);
    g_enc.norm_rows = reinterpret_cast<decltype(g_enc.norm_rows)>(f[13]);
    Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind_encoder", py_bind_encoder, METH_VARARGS, nullptr},
    {"begin_plan", py_begin_plan, METH_O, nullptr},
    {"complete_plan", py_complete_plan, METH_VARARGS, nullptr},
    {"plan_ok", reinterpret_cast<PyCFunction>(py_plan_ok), METH_FASTCALL, nullptr},
    {"scan_mask", reinterpret_cast<PyCFunction>(py_scan_mask), METH_FASTCALL, nullptr},
    {"encode", reinterpret_cast<PyCFunction>(py_encode), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

}  // namespace

bool tdb_host_add_encoder(PyObject* module) { return PyModule_AddFunctions(module, kMethods) == 0; }
