// Python extension module `_host`: the calls a model makes once per layer and step, without the interpreter's share.
//
// A forward pass of one quantized layer is two kernel launches of a few microseconds each.  Checking the arguments, looking
// at the parameters' version counters, allocating four tensors and filling two argument blocks took 19.6 us in Python (31.2
// for the fused MLP, 29.4 for the QKV projection, 11.4 for the AWQ layer), more than the GPU needs for a few hundred tokens;
// here it takes 8.8 (14.1, 8.4 and 5.1), most of it the launches themselves.  The operators called one by one keep their one
// way to the library (_native.launch); what is here is their checks, allocations and argument blocks.  They took 11.4 us
// (quantize), 14.8 (GEMM; 18.8 with linear attention, which adds up the shares of out_vk in a launch of its own) and 8.8
// (linearattn_vk_mul_q) of the caller's time, and take 7.3, 5.6 (8.4) and 3.5: linear attention over 256 tokens at K = 1024,
// four launches, went from 40.2 us to 19.4.
//
// Every function returns None when anything about the call is not the plain case it handles (another dtype, a parameter
// that has been replaced since the layer was converted, a tensor that is not contiguous, ...): the Python code behind it
// then takes the call, converts what has to be converted and raises what has to be raised.  Nothing is kept between
// calls but what the layer's own conversion keeps; the activations between the two launches live in one block of torch's
// caching allocator on the caller's stream.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "internal_api.h"

namespace {

constexpr int MAX_GROUPS = 64;  // 16-rank groups of the low-rank branch (rank 1024)

// What a layer keeps once its tensors are in the kernels' layouts (the counterpart of models/linear.py::_LayerCall).
struct Layer {
    struct Source {
        PyObject *name;  // owned
        bool present;
        const void *ptr;
        int64_t version;  // -1: the tensor keeps none
    };
    std::vector<Source> sources;  // the parameters the tensors were converted from
    std::vector<PyObject *> keep; // owned: the converted tensors
    svdq_quantize_args q;
    svdq_gemm_args g;
    int64_t act_bytes, scale_bytes, rank, N, K;  // bytes of codes and of scales per row
    int device;
};
const char *LAYER = "nunchaku_amd._host.Layer";

PyObject *s_parameters, *s_lora_scales, *s_qweight, *s_wscales, *s_wzeros, *s_bias, *s_in_features, *s_out_features, *s_group_size;
PyObject *s_native, *s_logical_shape, *s_colnorm, *s_nonzero, *s_lora_up, *s_lora_down, *s_vector, *s_smooth_rcp;

void free_layer(PyObject *capsule) {
    Layer *l = (Layer *)PyCapsule_GetPointer(capsule, LAYER);
    for (auto &s : l->sources) Py_DECREF(s.name);
    for (PyObject *t : l->keep) Py_DECREF(t);
    delete l;
}

bool as_tensor(PyObject *o, const at::Tensor **t) {
    if (!o || !THPVariable_Check(o)) return false;
    *t = &THPVariable_Unpack(o);
    return true;
}

// the instance's attribute dictionary (borrowed), or null
PyObject *dict_of(PyObject *module) {
    PyObject **p = _PyObject_GetDictPtr(module);
    return p ? *p : nullptr;
}
PyObject *parameters_of(PyObject *module) {
    PyObject *d = dict_of(module);
    PyObject *p = d ? PyDict_GetItem(d, s_parameters) : nullptr;
    return p && PyDict_Check(p) ? p : nullptr;
}

int64_t version_of(const at::Tensor &t) { return t.is_inference() ? -1 : (int64_t)t._version(); }

// no parameter has been replaced or written to since the conversion
bool unchanged(const Layer &l, PyObject *module) {
    PyObject *params = parameters_of(module);
    if (!params) return false;
    for (const auto &s : l.sources) {
        PyObject *o = PyDict_GetItem(params, s.name);
        const at::Tensor *t;
        if (!o || o == Py_None) {
            if (s.present) return false;
            continue;
        }
        if (!s.present || !as_tensor(o, &t) || t->data_ptr() != s.ptr || version_of(*t) != s.version) return false;
    }
    return true;
}

// The module's lora_scales (one factor per 16 ranks; None: all ones; missing entries count as zero) into `sc`.
bool read_lora_scales(PyObject *module, int groups, float *sc) {
    if (groups > MAX_GROUPS) return false;
    PyObject *d = dict_of(module);
    PyObject *ls = d ? PyDict_GetItem(d, s_lora_scales) : nullptr;
    if (!ls) return false;
    for (int i = 0; i < groups; i++) sc[i] = ls == Py_None ? 1.f : 0.f;
    if (ls == Py_None) return true;
    if (!PyList_Check(ls)) return false;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(ls) && i < groups; i++) {
        const double v = PyFloat_AsDouble(PyList_GET_ITEM(ls, i));
        if (v == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        sc[i] = (float)v;
    }
    return true;
}

bool plain_activations(const Layer &l, const at::Tensor &x) {
    return x.is_cuda() && x.dim() == 3 && x.scalar_type() == at::kBFloat16 && x.is_contiguous() && x.size(2) == l.K && x.numel() > 0 &&
           x.device().index() == l.device && c10::hip::current_device() == l.device;
}

struct Scratch {  // one block for all that lives between the launches of a call
    void *ptr;
    Scratch(size_t bytes, hipStream_t st) : ptr(c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, st)) {}
    ~Scratch() { c10::hip::HIPCachingAllocator::raw_delete(ptr); }
};

PyObject *raise(int rc) {
    PyErr_SetString(rc == SVDQ_EINVAL ? PyExc_ValueError : rc == SVDQ_EUNSUPPORTED ? PyExc_NotImplementedError : PyExc_RuntimeError, svdq_last_error());
    return nullptr;
}

// Where the quantized activations of M_pad rows of a layer lie in a block of memory.
struct Activations {
    uint8_t *codes, *scales;
    float *lora;
    size_t bytes;
    Activations(const Layer &l, int64_t M_pad, uint8_t *base) {
        const size_t nc = (size_t)(M_pad * l.act_bytes), ns = (size_t)(M_pad * l.scale_bytes), nl = (size_t)(M_pad * l.rank * 4);  // multiples of 256
        codes = base;
        scales = base + nc;
        lora = l.rank ? (float *)(base + nc + ns) : nullptr;
        bytes = nc + ns + nl;
    }
};

svdq_quantize_args quantize_args(const Layer &l, const void *x, int64_t M, int64_t M_pad, const Activations &a) {
    svdq_quantize_args q = l.q;
    q.input = x;
    q.output = a.codes;
    q.oscales = a.scales;
    q.lora_act_out = a.lora;
    q.M = M;
    q.M_pad = M_pad;
    return q;
}
svdq_gemm_args gemm_args(const Layer &l, int64_t M_pad, const Activations &a, const float *sc, int64_t k_split) {
    svdq_gemm_args g = l.g;
    g.act = a.codes;
    g.ascales = a.scales;
    g.lora_act_in = a.lora;
    g.lora_scales = sc;
    g.M_pad = M_pad;
    g.k_split = (int)k_split;
    return g;
}
int gemm(const svdq_gemm_args &g, bool no_alloc, hipStream_t st) { return no_alloc ? svdq_gemm_w4a4_noalloc(&g, st) : svdq_gemm_w4a4(&g, st); }

at::Tensor new_bf16(at::IntArrayRef sizes, int device) {
    return at::empty(sizes, at::TensorOptions().dtype(at::kBFloat16).device(at::Device(at::kCUDA, (c10::DeviceIndex)device)));
}

// a whole number among the arguments; false (and no exception left) where it is something else
bool as_int(PyObject *o, int64_t *v) {
    *v = PyLong_AsLongLong(o);
    if (*v != -1 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

// what `if o:` decides; false (and no exception left) where that raises
bool as_bool(PyObject *o, bool *v) {
    const int r = PyObject_IsTrue(o);
    *v = r > 0;
    if (r >= 0) return true;
    PyErr_Clear();
    return false;
}

Layer *layer_of(PyObject *capsule) { return (Layer *)PyCapsule_GetPointer(capsule, LAYER); }

#define SVDQ_NARGS(n)                                                              \
    if (nargs != n) {                                                              \
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", n, nargs); \
        return nullptr;                                                            \
    }

// make_layer(names, stamps, tensors, quantize block address, GEMM block address, sizes)
// names: the source parameters; stamps: (data_ptr, version or None) or None for each; tensors: what must stay alive; the
// addresses: ctypes blocks with everything filled in that does not change from call to call; sizes: (device index, bytes of
// codes per row, bytes of scales per row).
PyObject *make_layer(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    SVDQ_NARGS(6)
    PyObject *names = args[0], *stamps = args[1], *tensors = args[2], *sizes = args[5];
    if (!PyTuple_Check(names) || !PyTuple_Check(stamps) || PyTuple_GET_SIZE(names) != PyTuple_GET_SIZE(stamps) || !PyTuple_Check(tensors) ||
        !PyTuple_Check(sizes) || PyTuple_GET_SIZE(sizes) != 3) {
        PyErr_SetString(PyExc_TypeError, "make_layer: names, stamps, tensors and sizes are tuples");
        return nullptr;
    }
    const void *q = PyLong_AsVoidPtr(args[3]), *g = PyLong_AsVoidPtr(args[4]);
    if (!q || !g) return PyErr_Occurred() ? nullptr : (PyErr_SetString(PyExc_ValueError, "make_layer: null argument block"), nullptr);
    Layer *l = new Layer;
    l->q = *(const svdq_quantize_args *)q;
    l->g = *(const svdq_gemm_args *)g;
    l->device = (int)PyLong_AsLong(PyTuple_GET_ITEM(sizes, 0));
    l->act_bytes = PyLong_AsLongLong(PyTuple_GET_ITEM(sizes, 1));
    l->scale_bytes = PyLong_AsLongLong(PyTuple_GET_ITEM(sizes, 2));
    l->rank = l->g.R_up;
    l->N = l->g.N;
    l->K = l->g.K;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); i++) {
        PyObject *st = PyTuple_GET_ITEM(stamps, i);
        Layer::Source s{PyTuple_GET_ITEM(names, i), st != Py_None, nullptr, -1};
        if (s.present) {
            s.ptr = PyLong_AsVoidPtr(PyTuple_GetItem(st, 0));
            PyObject *v = PyTuple_GetItem(st, 1);
            s.version = v && v != Py_None ? PyLong_AsLongLong(v) : -1;
        }
        Py_INCREF(s.name);
        l->sources.push_back(s);
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tensors); i++) {
        l->keep.push_back(PyTuple_GET_ITEM(tensors, i));
        Py_INCREF(l->keep.back());
    }
    PyObject *capsule = PyErr_Occurred() ? nullptr : PyCapsule_New(l, LAYER, free_layer);
    if (!capsule) {
        for (auto &s : l->sources) Py_DECREF(s.name);
        for (PyObject *t : l->keep) Py_DECREF(t);
        delete l;
    }
    return capsule;
}

// linear(layer, module, x, output or None, k_split, no_alloc) -> bf16 [batch, rows, N]
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(6)
    Layer *l = layer_of(args[0]);
    if (!l) return nullptr;
    const at::Tensor *x, *given = nullptr;
    float sc[MAX_GROUPS];
    if (!as_tensor(args[2], &x) || !plain_activations(*l, *x) || !unchanged(*l, args[1]) || !read_lora_scales(args[1], (int)(l->rank + 15) / 16, sc)) Py_RETURN_NONE;
    const int64_t B = x->size(0), S = x->size(1), M = B * S, M_pad = (M + 255) / 256 * 256;
    if (args[3] != Py_None) {
        if (!as_tensor(args[3], &given) || !given->is_cuda() || given->device() != x->device() || given->scalar_type() != at::kBFloat16 ||
            !given->is_contiguous() || given->numel() != M * l->N || given->size(-1) != l->N) Py_RETURN_NONE;
    }
    int64_t k_split;
    bool no_alloc;
    if (!as_int(args[4], &k_split) || !as_bool(args[5], &no_alloc)) Py_RETURN_NONE;
    at::Tensor out = given ? given->view({B, S, l->N}) : new_bf16({B, S, l->N}, l->device);
    hipStream_t st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)l->device).stream();
    Scratch mem(Activations(*l, M_pad, nullptr).bytes, st);
    const Activations a(*l, M_pad, (uint8_t *)mem.ptr);
    const svdq_quantize_args q = quantize_args(*l, x->data_ptr(), M, M_pad, a);
    svdq_gemm_args g = gemm_args(*l, M_pad, a, sc, k_split);
    g.out = out.data_ptr();
    g.M_out = M;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = svdq_quantize_w4a4_act_fuse_lora(&q, st);
    if (rc == SVDQ_OK) rc = gemm(g, no_alloc, st);
    Py_END_ALLOW_THREADS
    if (rc != SVDQ_OK) return raise(rc);
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// gelu_mlp(layer 1, module 1, layer 2, module 2, x, pad_size, k_split, no_alloc) -> bf16 [batch, rows, N of layer 2]
PyObject *gelu_mlp(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(8)
    Layer *l1 = layer_of(args[0]), *l2 = layer_of(args[2]);
    if (!l1 || !l2) return nullptr;
    const at::Tensor *x;
    float sc1[MAX_GROUPS], sc2[MAX_GROUPS];
    int64_t pad, k_split;
    bool no_alloc;
    if (!as_int(args[5], &pad) || !as_int(args[6], &k_split) || !as_bool(args[7], &no_alloc) || !as_tensor(args[4], &x) || !plain_activations(*l1, *x) || l2->device != l1->device || l1->N != l2->K || l1->g.fp4 != l2->g.fp4 || pad <= 0 || pad % 256 ||
        !unchanged(*l1, args[1]) || !unchanged(*l2, args[3]) || !read_lora_scales(args[1], (int)(l1->rank + 15) / 16, sc1) ||
        !read_lora_scales(args[3], (int)(l2->rank + 15) / 16, sc2)) Py_RETURN_NONE;
    const int64_t B = x->size(0), S = x->size(1), M = B * S, M_pad = (M + pad - 1) / pad * pad;
    at::Tensor out = new_bf16({B, S, l2->N}, l1->device);
    hipStream_t st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)l1->device).stream();
    const size_t first = Activations(*l1, M_pad, nullptr).bytes;
    Scratch mem(first + Activations(*l2, M_pad, nullptr).bytes, st);
    const Activations a1(*l1, M_pad, (uint8_t *)mem.ptr), a2(*l2, M_pad, (uint8_t *)mem.ptr + first);
    const svdq_quantize_args q = quantize_args(*l1, x->data_ptr(), M, M_pad, a1);
    svdq_gemm_args g1 = gemm_args(*l1, M_pad, a1, sc1, k_split), g2 = gemm_args(*l2, M_pad, a2, sc2, k_split);
    g1.qout = a2.codes;
    g1.oscales = a2.scales;
    g1.next_smooth_rcp = l2->q.smooth_rcp;
    g1.next_lora_down = l2->q.lora_down;
    g1.next_lora_act_out = a2.lora;
    g1.R_down = l2->rank;
    g2.out = out.data_ptr();
    g2.M_out = M;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = svdq_quantize_w4a4_act_fuse_lora(&q, st);
    if (rc == SVDQ_OK) rc = svdq_gemm_w4a4_rows(&g1, M, no_alloc, st);  // (layer 2 reads nothing of the padding rows that reaches its output)
    if (rc == SVDQ_OK) rc = gemm(g2, no_alloc, st);
    Py_END_ALLOW_THREADS
    if (rc != SVDQ_OK) return raise(rc);
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// qkv_norm_rope(layer, module, x, norm_q weight, norm_k weight, converted rotary table, None or (q, k, v), attn_tokens,
// norm_eps, k_split, no_alloc) -> bf16 [batch, rows, N], or the tuple
PyObject *qkv_norm_rope(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(11)
    Layer *l = layer_of(args[0]);
    if (!l) return nullptr;
    const at::Tensor *x, *nq, *nk, *rot;
    float sc[MAX_GROUPS];
    if (!as_tensor(args[2], &x) || !plain_activations(*l, *x) || !as_tensor(args[3], &nq) || !as_tensor(args[4], &nk) || !as_tensor(args[5], &rot) ||
        !unchanged(*l, args[1]) || !read_lora_scales(args[1], (int)(l->rank + 15) / 16, sc) || l->N % 384) Py_RETURN_NONE;
    for (const at::Tensor *t : {nq, nk})
        if (t->device() != x->device() || t->scalar_type() != at::kBFloat16 || t->numel() != 128 || !t->is_contiguous()) Py_RETURN_NONE;
    if (rot->device() != x->device() || rot->scalar_type() != at::kFloat || rot->dim() != 2 || rot->size(1) != 128 || !rot->is_contiguous()) Py_RETURN_NONE;
    const int64_t B = x->size(0), S = x->size(1), M = B * S, M_pad = (M + 255) / 256 * 256;
    at::Tensor out;
    const at::Tensor *qkv[3] = {nullptr, nullptr, nullptr};
    int64_t attn_tokens, k_split;
    bool no_alloc;
    const double norm_eps = PyFloat_AsDouble(args[8]);
    if ((norm_eps == -1.0 && PyErr_Occurred()) || !as_int(args[7], &attn_tokens) || !as_int(args[9], &k_split) || !as_bool(args[10], &no_alloc)) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const bool split = args[6] != Py_None;
    if (split) {
        if (!PyTuple_Check(args[6]) || PyTuple_GET_SIZE(args[6]) != 3 || attn_tokens < 0 || attn_tokens > M_pad) Py_RETURN_NONE;
        for (int i = 0; i < 3; i++) {
            if (!as_tensor(PyTuple_GET_ITEM(args[6], i), &qkv[i])) Py_RETURN_NONE;
            const at::Tensor &t = *qkv[i];
            if (t.device() != x->device() || t.scalar_type() != at::kHalf || t.dim() != 4 || t.size(0) != 1 || t.size(1) != l->N / 384 || t.size(2) != M_pad ||
                t.size(3) != 128 || t.stride(3) != 1 || t.stride(2) != 128) Py_RETURN_NONE;
        }
    } else {
        out = new_bf16({M_pad, l->N}, l->device);
    }
    hipStream_t st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)l->device).stream();
    Scratch mem(Activations(*l, M_pad, nullptr).bytes, st);
    const Activations a(*l, M_pad, (uint8_t *)mem.ptr);
    const svdq_quantize_args q = quantize_args(*l, x->data_ptr(), M, M_pad, a);
    svdq_gemm_args g = gemm_args(*l, M_pad, a, sc, k_split);
    g.norm_q = nq->data_ptr();
    g.norm_k = nk->data_ptr();
    g.rotary_emb = (const float *)rot->data_ptr();
    g.rot_rows = rot->size(0);
    g.norm_eps = (float)norm_eps;
    if (split) {
        g.out_q = qkv[0]->data_ptr();
        g.out_k = qkv[1]->data_ptr();
        g.out_v = qkv[2]->data_ptr();
        for (int i = 0; i < 3; i++) g.qkv_head_stride[i] = qkv[i]->stride(1);
        g.attn_tokens = attn_tokens;
        g.qkv_rows = M_pad;
        g.N_out = 0;
    } else {
        g.out = out.data_ptr();
        g.M_out = M_pad;
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = svdq_quantize_w4a4_act_fuse_lora(&q, st);
    if (rc == SVDQ_OK) rc = gemm(g, no_alloc, st);
    Py_END_ALLOW_THREADS
    if (rc != SVDQ_OK) return raise(rc);
    if (split) {
        Py_INCREF(args[6]);
        return args[6];
    }
    return THPVariable_Wrap(out.narrow(0, 0, M).view({B, S, l->N}));
    END_HANDLE_TH_ERRORS
}

bool plain_on(const at::Tensor &t, const at::Tensor &x, at::ScalarType dt, int64_t numel) {
    return t.device() == x.device() && t.scalar_type() == dt && t.numel() == numel && t.is_contiguous();
}

PyObject *awq_call(const at::Tensor &x, const at::Tensor &w, const at::Tensor &s, const at::Tensor &z, const at::Tensor *bias, int64_t m, int64_t n, int64_t k,
                   int group_size) {
    if (!x.is_cuda() || x.device().index() != c10::hip::current_device() || x.dim() < 1 || x.scalar_type() != at::kBFloat16 || !x.is_contiguous() || k <= 0 ||
        x.size(-1) != k || x.numel() != m * k || w.device() != x.device() || !w.is_contiguous() || w.numel() * (int64_t)w.element_size() != n * k / 2 ||
        !plain_on(s, x, at::kBFloat16, k / 64 * n) || !plain_on(z, x, at::kBFloat16, k / 64 * n) || s.dim() != 2 || z.dim() != 2 || s.size(1) != n || z.size(1) != n ||
        (bias && !plain_on(*bias, x, at::kBFloat16, n))) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 4> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = n;
    at::Tensor out = new_bf16(sizes, x.device().index());
    svdq_awq_gemv_args a;
    a.x = x.data_ptr();
    a.qweight = w.data_ptr();
    a.scales = s.data_ptr();
    a.zeros = z.data_ptr();
    a.bias = bias ? bias->data_ptr() : nullptr;
    a.out = out.data_ptr();
    a.M = m;
    a.N = n;
    a.K = k;
    a.group_size = group_size;
    hipStream_t st = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = svdq_awq_gemv_w4a16(&a, st);
    Py_END_ALLOW_THREADS
    if (rc != SVDQ_OK) return raise(rc);
    return THPVariable_Wrap(out);
}

// awq_gemv(x, qweight, scales, zeros, m, n, k, group_size, bias or None)
PyObject *awq_gemv(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(9)
    const at::Tensor *t[4], *bias = nullptr;
    for (int i = 0; i < 4; i++)
        if (!as_tensor(args[i], &t[i])) Py_RETURN_NONE;
    if (args[8] != Py_None && !as_tensor(args[8], &bias)) Py_RETURN_NONE;
    int64_t v[4];
    for (int i = 0; i < 4; i++) {
        if (!PyLong_Check(args[4 + i]) || !as_int(args[4 + i], &v[i])) Py_RETURN_NONE;
    }
    return awq_call(*t[0], *t[1], *t[2], *t[3], bias, v[0], v[1], v[2], (int)v[3]);
    END_HANDLE_TH_ERRORS
}

// awq_linear(module, x): the same on an AWQW4A16Linear's own parameters
PyObject *awq_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(2)
    PyObject *d = dict_of(args[0]), *params = parameters_of(args[0]);
    const at::Tensor *x, *w, *s, *z, *bias = nullptr;
    if (!d || !params || !as_tensor(args[1], &x) || !as_tensor(PyDict_GetItem(params, s_qweight), &w) || !as_tensor(PyDict_GetItem(params, s_wscales), &s) ||
        !as_tensor(PyDict_GetItem(params, s_wzeros), &z)) Py_RETURN_NONE;
    // `module.bias` is what the instance's dictionary holds (None in a layer built without one), else the parameter; a bias
    // anywhere else (a buffer, a property, an attribute of the class) is not the plain case
    PyObject *own = PyDict_GetItem(d, s_bias), *b = own ? own : PyDict_GetItem(params, s_bias);
    if (!b || (b != Py_None && !as_tensor(b, &bias))) Py_RETURN_NONE;
    PyObject *in = PyDict_GetItem(d, s_in_features), *out = PyDict_GetItem(d, s_out_features), *gs = PyDict_GetItem(d, s_group_size);
    int64_t n, k, group_size;
    if (!in || !out || !gs || !as_int(in, &k) || !as_int(out, &n) || !as_int(gs, &group_size) || x->dim() < 1 || x->size(-1) <= 0) Py_RETURN_NONE;
    return awq_call(*x, *w, *s, *z, bias, x->numel() / x->size(-1), n, k, (int)group_size);
    END_HANDLE_TH_ERRORS
}

// ---- the operators: checks, allocations and argument blocks --------------------------------------------------------------
// an attribute of a tensor (new reference) or null without an exception
PyObject *attribute(PyObject *o, PyObject *name) {
    PyObject *a = PyObject_GetAttr(o, name);
    if (!a) PyErr_Clear();
    return a;
}
// `o` is a tensor in the layout `kind` of the kernels, contiguous, on x's device
bool native_tensor(PyObject *o, PyObject *kind, const at::Tensor &x, const at::Tensor **t) {
    if (!as_tensor(o, t) || (*t)->device() != x.device() || !(*t)->is_contiguous()) return false;
    PyObject *a = attribute(o, s_native);
    const bool ok = a && (a == kind || (PyUnicode_Check(a) && PyUnicode_Compare(a, kind) == 0));
    Py_XDECREF(a);
    return ok;
}
bool shape_is(const at::Tensor &t, at::IntArrayRef sizes) { return t.sizes() == sizes; }
bool checked(PyObject *o, const at::Tensor &x, at::ScalarType dt, at::IntArrayRef sizes, const at::Tensor **t) {
    return as_tensor(o, t) && (*t)->device() == x.device() && (*t)->scalar_type() == dt && (*t)->is_contiguous() && shape_is(**t, sizes);
}
at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dt, const at::Tensor &x) {
    return at::empty(sizes, at::TensorOptions().dtype(dt).device(x.device()));
}

// quantize_call(block address, input, lora_down, smooth or None, fp4, pad_size) -> (output, oscales, lora_act_out) with the block filled in, or None
PyObject *quantize_call(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(6)
    svdq_quantize_args *q = (svdq_quantize_args *)PyLong_AsVoidPtr(args[0]);
    if (!q) return PyErr_Occurred() ? nullptr : (PyErr_SetString(PyExc_ValueError, "quantize_call: null argument block"), nullptr);
    const at::Tensor *x, *down, *smooth = nullptr;
    bool fp4;
    int64_t pad;
    if (!as_tensor(args[1], &x) || !x->is_cuda() || x->dim() != 2 || x->scalar_type() != at::kBFloat16 || !x->is_contiguous() || x->size(0) <= 0 ||
        !as_bool(args[4], &fp4) || !as_int(args[5], &pad) || pad <= 0 || pad % 256) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1), M_pad = (M + pad - 1) / pad * pad, G = fp4 ? 16 : 64;
    if (K % 128 || !native_tensor(args[2], s_lora_down, *x, &down) || down->dim() != 2 || down->size(0) != K || down->scalar_type() != at::kBFloat16) Py_RETURN_NONE;
    if (args[3] != Py_None && (!native_tensor(args[3], s_smooth_rcp, *x, &smooth) || smooth->numel() != K || smooth->scalar_type() != at::kFloat)) Py_RETURN_NONE;
    const int64_t R = down->size(1);
    at::Tensor out = new_tensor({M_pad, fp4 ? K / 2 : K * 3 / 4}, at::kByte, *x), scales = new_tensor({K / G, M_pad}, fp4 ? at::kFloat8_e4m3fn : at::kBFloat16, *x),
               lora = new_tensor({M_pad, R}, at::kFloat, *x);
    *q = svdq_quantize_args{};
    q->input = x->data_ptr();
    q->output = out.data_ptr();
    q->oscales = scales.data_ptr();
    q->lora_down = R ? down->data_ptr() : nullptr;
    q->lora_act_out = R ? (float *)lora.data_ptr() : nullptr;
    q->smooth_rcp = smooth ? (const float *)smooth->data_ptr() : nullptr;
    q->M = M;
    q->M_pad = M_pad;
    q->K = K;
    q->R = R;
    q->fp4 = fp4;
    PyObject *r = PyTuple_New(3);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(out));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(scales));
    PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(lora));
    return r;
    END_HANDLE_TH_ERRORS
}

// gemm_call(block address, address of MAX_GROUPS floats, act, wgt, ascales, wscales, out or None, out_vk or None, out_linearattn or None, lora_act_in or None, lora_up or
// None, bias or None, wcscales or None, lora_scales or None, alpha, act_unsigned, fuse_silu, fp4, k_split) -> True with the block filled in, or None
PyObject *gemm_call(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(19)
    svdq_gemm_args *g = (svdq_gemm_args *)PyLong_AsVoidPtr(args[0]);
    float *sc = (float *)PyLong_AsVoidPtr(args[1]);
    if (!g || !sc) return PyErr_Occurred() ? nullptr : (PyErr_SetString(PyExc_ValueError, "gemm_call: null argument block"), nullptr);
    const at::Tensor *act, *wgt, *asc, *wsc, *out = nullptr, *vk = nullptr, *la = nullptr, *up = nullptr, *bias = nullptr, *wcs = nullptr, *colnorm = nullptr;
    bool unsigned_codes, silu, fp4;
    int64_t k_split, N, K;
    if (!as_bool(args[15], &unsigned_codes) || !as_bool(args[16], &silu) || !as_bool(args[17], &fp4) || !as_int(args[18], &k_split)) Py_RETURN_NONE;
    if (!as_tensor(args[2], &act) || !act->is_cuda() || act->dim() != 2 || act->scalar_type() != at::kByte || !act->is_contiguous() || !native_tensor(args[3], s_qweight, *act, &wgt) ||
        !native_tensor(args[5], s_wscales, *act, &wsc)) Py_RETURN_NONE;
    {
        PyObject *shape = attribute(args[3], s_logical_shape);
        const bool ok = shape && PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == 2 && as_int(PyTuple_GET_ITEM(shape, 0), &N) && as_int(PyTuple_GET_ITEM(shape, 1), &K);
        Py_XDECREF(shape);
        if (!ok) Py_RETURN_NONE;
    }
    const int64_t M_pad = act->size(0), G = fp4 ? 16 : 64;
    // (the native scales of the two precisions differ in type: those of the other one are not the plain case)
    if (M_pad <= 0 || M_pad % 256 || K <= 0 || K % 128 || N <= 0 || N % 128 || act->size(1) != (fp4 ? K / 2 : K * 3 / 4) ||
        !checked(args[4], *act, fp4 ? at::kFloat8_e4m3fn : at::kBFloat16, {K / G, M_pad}, &asc) || wsc->scalar_type() != (fp4 ? at::kHalf : at::kLong) ||
        wsc->numel() != (fp4 ? K / 16 * N : (N + 255) / 256 * (K / 64) * 256) || wgt->numel() != (fp4 ? N * (K / 2) : (N + 255) / 256 * 256 * (K * 3 / 4))) Py_RETURN_NONE;
    if (fp4) {
        // (the tensor is an attribute of the scales, which the caller holds)
        PyObject *c = attribute(args[5], s_colnorm);
        const bool ok = c && as_tensor(c, &colnorm) && colnorm->device() == act->device() && colnorm->numel() == N && colnorm->scalar_type() == at::kFloat;
        Py_XDECREF(c);
        if (!ok) Py_RETURN_NONE;
    }
    if (args[11] != Py_None && (!native_tensor(args[11], s_vector, *act, &bias) || bias->scalar_type() != at::kBFloat16 || !shape_is(*bias, {N}))) Py_RETURN_NONE;
    if (args[12] != Py_None && (!native_tensor(args[12], s_vector, *act, &wcs) || wcs->scalar_type() != at::kBFloat16 || !shape_is(*wcs, {N}))) Py_RETURN_NONE;
    int64_t R = 0;
    if ((args[9] == Py_None) != (args[10] == Py_None)) Py_RETURN_NONE;
    if (args[10] != Py_None) {
        if (!native_tensor(args[10], s_lora_up, *act, &up) || up->dim() != 2 || up->scalar_type() != at::kBFloat16 || up->size(0) != N || up->size(1) <= 0 ||
            up->size(1) > 16 * MAX_GROUPS) Py_RETURN_NONE;
        R = up->size(1);
        if (!checked(args[9], *act, at::kFloat, {M_pad, R}, &la)) Py_RETURN_NONE;
        if (fp4 && wcs) {  // (the wrapper's check for zeros, once per tensor, has been made)
            PyObject *z = attribute(args[12], s_nonzero);
            const bool ok = z == Py_True;
            Py_XDECREF(z);
            if (!ok) Py_RETURN_NONE;
        }
    }
    const int groups = (int)((R + 15) / 16);
    for (int i = 0; i < groups; i++) sc[i] = args[13] == Py_None ? 1.f : 0.f;
    if (args[13] != Py_None) {
        if (!PyList_Check(args[13])) Py_RETURN_NONE;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[13]) && i < groups; i++) {
            PyObject *v = PyList_GET_ITEM(args[13], i);
            if (!PyFloat_CheckExact(v)) Py_RETURN_NONE;
            sc[i] = (float)PyFloat_AS_DOUBLE(v);
        }
    }
    if (!PyFloat_CheckExact(args[14])) Py_RETURN_NONE;
    int64_t vk_rows = 0;
    if (args[7] != Py_None) {
        if (args[6] != Py_None || silu || N % 384 || !as_tensor(args[8], &out) || out->dim() != 3) Py_RETURN_NONE;
        const int64_t B = out->size(0);
        vk_rows = out->size(1);
        if (!checked(args[8], *act, at::kBFloat16, {B, vk_rows, N / 3}, &out) || !checked(args[7], *act, at::kFloat, {B, N / 96, 33, 32}, &vk) || vk_rows <= 0 || vk_rows % 256 ||
            B * vk_rows != M_pad) Py_RETURN_NONE;
    } else if (args[8] != Py_None || !as_tensor(args[6], &out) || out->device() != act->device() || out->scalar_type() != at::kBFloat16 || !out->is_contiguous() || out->dim() < 1 ||
               out->numel() == 0) {
        Py_RETURN_NONE;
    }
    *g = svdq_gemm_args{};
    g->act = act->data_ptr();
    g->ascales = asc->data_ptr();
    g->wgt = wgt->data_ptr();
    g->wscales = wsc->data_ptr();
    g->colnorm = colnorm ? (const float *)colnorm->data_ptr() : nullptr;
    g->bias = bias ? bias->data_ptr() : nullptr;
    g->wcscales = wcs ? wcs->data_ptr() : nullptr;
    g->lora_act_in = la ? (const float *)la->data_ptr() : nullptr;
    g->lora_up = up ? up->data_ptr() : nullptr;
    g->lora_scales = sc;
    g->out = out->data_ptr();
    g->M_pad = M_pad;
    g->N = N;
    g->K = K;
    g->N_out = out->size(-1);
    g->M_out = out->numel() / g->N_out;
    g->R_up = R;
    g->alpha = (float)PyFloat_AS_DOUBLE(args[14]);
    g->act_unsigned = unsigned_codes;
    g->fuse_silu = silu;
    g->fp4 = fp4;
    g->k_split = (int)k_split;
    g->out_vk = vk ? (float *)vk->data_ptr() : nullptr;
    g->vk_rows = vk_rows;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// vk_mul_q(q, vk, num_tokens, eps): linearattn_vk_mul_q on the current stream -> True, or None
PyObject *vk_mul_q(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    SVDQ_NARGS(4)
    const at::Tensor *q, *vk;
    int64_t tokens;
    if (!as_tensor(args[0], &q) || !q->is_cuda() || q->dim() != 3 || q->scalar_type() != at::kBFloat16 || !q->is_contiguous() || q->device().index() != c10::hip::current_device() ||
        !as_tensor(args[1], &vk) || vk->dim() != 4 || !PyFloat_CheckExact(args[3])) Py_RETURN_NONE;
    const int64_t B = q->size(0), tokens_pad = q->size(1), heads = vk->size(1);
    if (!checked(args[1], *q, at::kFloat, {B, heads, 33, 32}, &vk) || q->size(2) != heads * 32) Py_RETURN_NONE;
    if (args[2] == Py_None) tokens = tokens_pad;
    else if (!PyLong_CheckExact(args[2]) || !as_int(args[2], &tokens)) Py_RETURN_NONE;
    hipStream_t st = c10::hip::getCurrentHIPStream(q->device().index()).stream();
    int rc;
    const float eps = (float)PyFloat_AS_DOUBLE(args[3]);
    Py_BEGIN_ALLOW_THREADS
    rc = svdq_linearattn_vk_mul_q(q->data_ptr(), (const float *)vk->data_ptr(), B, tokens, tokens_pad, heads, eps, st);
    Py_END_ALLOW_THREADS
    if (rc != SVDQ_OK) return raise(rc);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

#define SVDQ_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SVDQ_METHOD(make_layer), SVDQ_METHOD(linear), SVDQ_METHOD(gelu_mlp), SVDQ_METHOD(qkv_norm_rope), SVDQ_METHOD(awq_gemv), SVDQ_METHOD(awq_linear),
                         SVDQ_METHOD(quantize_call), SVDQ_METHOD(gemm_call), SVDQ_METHOD(vk_mul_q),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Per-call host code of the quantized layers.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    s_parameters = PyUnicode_InternFromString("_parameters");
    s_lora_scales = PyUnicode_InternFromString("lora_scales");
    s_qweight = PyUnicode_InternFromString("qweight");
    s_wscales = PyUnicode_InternFromString("wscales");
    s_wzeros = PyUnicode_InternFromString("wzeros");
    s_bias = PyUnicode_InternFromString("bias");
    s_in_features = PyUnicode_InternFromString("in_features");
    s_out_features = PyUnicode_InternFromString("out_features");
    s_group_size = PyUnicode_InternFromString("group_size");
    s_native = PyUnicode_InternFromString("_svdq_native");
    s_logical_shape = PyUnicode_InternFromString("logical_shape");
    s_colnorm = PyUnicode_InternFromString("colnorm");
    s_nonzero = PyUnicode_InternFromString("_svdq_nonzero");
    s_lora_up = PyUnicode_InternFromString("lora_up");
    s_lora_down = PyUnicode_InternFromString("lora_down");
    s_vector = PyUnicode_InternFromString("vector");
    s_smooth_rcp = PyUnicode_InternFromString("smooth_rcp");
    return PyModule_Create(&module_def);
}
