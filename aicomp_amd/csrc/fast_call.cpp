// CPython entry for the drop-in operator's decode call at small batch: the leanest host route
// from CachedScaledDotProductAttention.forward (opt_prime/opt_prime/kv_cache.py:340-403) into
// aicomp_paged_decode_attn_append.  The reference's own engine decodes at batch 1
// (inference.py:1036-1044), where the GPU needs 5 to 8 us per call and every microsecond of host
// time is step time.  torch.ops.mi355_kv.decode_step (torch_ops.cpp) spends about three of its eight
// microseconds in the dispatcher and in re-checking tensors that never change between steps; here
// a layer's pools, table and context-length rows are checked once and kept in a capsule, and a
// step is one METH_FASTCALL function: three tensors unpacked, the output allocated, one C call.
//
//   layer = _aicomp_fast.layer(k_pool, v_pool, block_table, ctx_rows)
//   out   = _aicomp_fast.decode_step(layer, query, key, value, position, group, scale)
//   out   = _aicomp_fast.prompt_step(layer, slots, cu, query, key, value, position, group, scale)
//
// Same checks, same errors (RuntimeError), same results as the registered operator.
//
// Beside it, the plain calls of aicomp_amd.ops (kv_append, rope_kv_append, paged_decode_attn, rope_paged_decode_attn,
// paged_prefill_attn, append_prefill_attn, chunks_and_rows, sample_tokens): the same checks made here instead of in Python.  A call that
// passes them all is launched and returns true; any other returns false without having touched
// anything, and the Python function goes on to convert what may be converted or to name what is wrong.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <map>
#include <vector>
#include <mutex>
#include <utility>

#include "../../include/aicomp_kv.h"

namespace {

struct Layer {
    at::Tensor k_pool, v_pool, block_table, ctx_rows;     // kept alive; the pointers below are theirs
    void* kp;
    void* vp;
    const int32_t* table;
    const int32_t* ctx;
    int64_t table_stride, ctx_stride, ctx_count, nb;
    int B, hkv, bs, d, width, dt;
    at::ScalarType st;
    c10::Device dev{c10::DeviceType::CPU};
};

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return AICOMP_KV_F32;
        case at::kBFloat16: return AICOMP_KV_BF16;
        case at::kHalf: return AICOMP_KV_F16;
        default: return -1;
    }
}

void layer_free(PyObject* cap) { delete (Layer*)PyCapsule_GetPointer(cap, "aicomp_amd.layer"); }

// A call that uses the scratch below is two launches, and on one stream two of them must not interleave: the
// second call's partials would replace the first's before their merge reads them.  Two host threads on one
// stream can get there, one of them inside a plain call, which lets go of the interpreter lock.  Held over the
// launches alone and never across a wait for the interpreter lock.
std::mutex& scratch_launches() {
    static auto* mu = new std::mutex();
    return *mu;
}

// scratch of calls that need a merge: one growing buffer per (device, stream), never destroyed
// (tensors freed at interpreter exit, after the allocator, would fault)
at::Tensor cached_scratch(const c10::Device& dev, void* stream, size_t bytes) {
    static std::mutex mu;
    static auto* table = new std::map<std::pair<int, void*>, at::Tensor>();
    std::lock_guard<std::mutex> lock(mu);
    at::Tensor& t = (*table)[{(int)dev.index(), stream}];
    if (!t.defined() || (size_t)t.numel() < bytes)
        t = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(dev));
    return t;
}

#define FAIL(...)                                             \
    do {                                                      \
        PyErr_Format(PyExc_RuntimeError, __VA_ARGS__);        \
        return nullptr;                                       \
    } while (0)

PyObject* layer_new(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        if (nargs != 4) FAIL("layer(k_pool, v_pool, block_table, ctx_rows)");
        for (int i = 0; i < 4; ++i)
            if (!THPVariable_Check(args[i])) FAIL("layer: argument %d is not a tensor", i);
        auto L = std::make_unique<Layer>();
        L->k_pool = THPVariable_Unpack(args[0]);
        L->v_pool = THPVariable_Unpack(args[1]);
        L->block_table = THPVariable_Unpack(args[2]);
        L->ctx_rows = THPVariable_Unpack(args[3]);
        const at::Tensor &k = L->k_pool, &v = L->v_pool, &bt = L->block_table, &cr = L->ctx_rows;
        if (!k.is_cuda()) FAIL("tensors must live on a ROCm device (there is no CPU path)");
        if (k.dim() != 4 || v.sizes() != k.sizes() || k.scalar_type() != v.scalar_type() || !k.is_contiguous() ||
            !v.is_contiguous() || v.device() != k.device())
            FAIL("pools must both be contiguous [num_blocks, Hkv, BS, D] tensors of one dtype on one device");
        L->dt = dtype_code(k.scalar_type());
        if (L->dt < 0) FAIL("decode_step stores the rows as they are: float32, bfloat16 or float16 pools");
        L->B = (int)bt.size(0);
        if (bt.scalar_type() != at::kInt || bt.dim() != 2 || bt.stride(1) != 1 || bt.device() != k.device())
            FAIL("block_table must be int32 [B, max_blocks] on the pools' device, rows contiguous");
        if (cr.scalar_type() != at::kInt || cr.dim() != 2 || cr.size(1) != L->B || cr.stride(1) != 1 ||
            cr.device() != k.device())
            FAIL("ctx_rows must be int32 [positions + 1, B] on the pools' device");
        L->kp = k.data_ptr(); L->vp = v.data_ptr();
        L->table = bt.data_ptr<int32_t>(); L->table_stride = bt.stride(0); L->width = (int)bt.size(1);
        L->ctx = cr.data_ptr<int32_t>(); L->ctx_stride = cr.stride(0); L->ctx_count = cr.size(0);
        L->nb = k.size(0); L->hkv = (int)k.size(1); L->bs = (int)k.size(2); L->d = (int)k.size(3);
        L->st = k.scalar_type(); L->dev = k.device();
        return PyCapsule_New(L.release(), "aicomp_amd.layer", layer_free);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// Elements between the heads of new rows.  One head's stride is never taken, and is 0 in what is left of an expanded view
// (repeated heads, every group-th taken), which the library refuses.
int64_t head_stride(int hkv, int d, int64_t stride) { return hkv == 1 ? d : stride; }

PyObject* decode_step(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        if (nargs != 7) FAIL("decode_step(layer, query, key, value, position, group, scale)");
        const Layer* L = (const Layer*)PyCapsule_GetPointer(args[0], "aicomp_amd.layer");
        if (L == nullptr) return nullptr;
        if (!THPVariable_Check(args[1]) || !THPVariable_Check(args[2]) || !THPVariable_Check(args[3]))
            FAIL("decode_step: query, key and value must be tensors");
        const at::Tensor& q_in = THPVariable_Unpack(args[1]);
        const at::Tensor& key = THPVariable_Unpack(args[2]);
        const at::Tensor& value = THPVariable_Unpack(args[3]);
        const int64_t position = PyLong_AsLongLong(args[4]);
        const int64_t group = PyLong_AsLongLong(args[5]);
        const double scale = PyFloat_AsDouble(args[6]);
        if (PyErr_Occurred()) return nullptr;
        if (q_in.dim() != 4 || q_in.size(0) != L->B || q_in.size(2) != 1 || q_in.size(3) != L->d ||
            q_in.scalar_type() != L->st || q_in.device() != L->dev)
            FAIL("query must be a [%d, Hq, 1, %d] tensor of the pools' dtype on their device", L->B, L->d);
        const int hq = (int)q_in.size(1);
        if (hq % L->hkv) FAIL("%d query heads over %d KV heads", hq, L->hkv);
        const int64_t H = key.dim() == 4 ? key.size(1) : -1;
        const int64_t hstep = (group > 1 && H == (int64_t)L->hkv * group) ? group : 1;
        if (key.dim() != 4 || key.size(0) != L->B || H != L->hkv * hstep || key.size(2) != 1 || key.size(3) != L->d ||
            value.sizes() != key.sizes() || key.scalar_type() != L->st || value.scalar_type() != L->st ||
            key.device() != L->dev || value.device() != L->dev)
            FAIL("key/value must both be [%d, %d or %d*group, 1, %d] of the query dtype on its device", L->B, L->hkv,
                 L->hkv, L->d);
        if (position < 0 || position + 1 >= L->ctx_count) FAIL("ctx_rows does not hold row %lld", (long long)(position + 1));
        const c10::DeviceGuard guard(L->dev);              // launches go to the layer's device, whatever is current
        const at::Tensor query = q_in.is_contiguous() ? q_in : q_in.contiguous();
        at::Tensor k = key, v = value;
        if (k.stride(3) != 1 || k.strides() != v.strides()) { k = k.contiguous(); v = v.contiguous(); }
        // only the table columns that hold position + 1 tokens are in use: the library sizes the
        // split for the context as it is now (a short context: one launch, no scratch, no merge)
        const int width = (int)std::min<int64_t>(L->width, (position + L->bs) / L->bs);
        void* stream = (void*)c10::hip::getCurrentHIPStream(L->dev.index()).stream();
        size_t ws_bytes = aicomp_paged_decode_workspace_bytes(L->B, hq, L->hkv, L->d, L->bs, width, L->dt, L->dt, 0);
        void* ws = nullptr;
        at::Tensor scratch;
        if (ws_bytes) {
            scratch = cached_scratch(L->dev, stream, ws_bytes);
            ws = scratch.data_ptr();
            ws_bytes = (size_t)scratch.numel();
        }
        // (the allocator's own entry: at::empty goes through the dispatcher for the same result)
        at::Tensor out(at::detail::empty_cuda(query.sizes(), L->st, L->dev, c10::MemoryFormat::Contiguous));
        std::unique_lock<std::mutex> one_at_a_time(scratch_launches(), std::defer_lock);
        if (ws) one_at_a_time.lock();
        const int rc = aicomp_paged_decode_attn_append(
            out.data_ptr(), query.data_ptr(), k.data_ptr(), v.data_ptr(), k.stride(0),
            head_stride(L->hkv, L->d, k.stride(1) * hstep), L->kp, L->vp,
            L->table, L->table_stride, L->ctx + (position + 1) * L->ctx_stride, L->B, hq, L->hkv, L->d, L->bs, width,
            L->nb, (float)scale, L->dt, L->dt, nullptr, nullptr, 0, ws, ws_bytes, stream);
        if (ws) one_at_a_time.unlock();
        if (rc != AICOMP_KV_OK) FAIL("aicomp_kv error %d: %s", rc, aicomp_kv_last_error());
        return THPVariable_Wrap(std::move(out));
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// The tensor behind an argument, or null unless it is a plain strided tensor on a GPU with storage of
// its own (no subclass, no wrapper of a transform): those go the Python way.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

// runs a library call without the interpreter lock (a launch waits while the stream's queue is full)
template <typename F> int unlocked(F call) {
    PyThreadState* state = PyEval_SaveThread();
    const int rc = call();
    PyEval_RestoreThread(state);
    return rc;
}

// A prompt chunk of the operator: append of its rows and causal attention, [B, Hq, n, D] as decode_step returns its row.
// slots [B, positions]: where sequence b keeps its tokens; cu: int32 [B + 1], the multiples of n.  None, with nothing done,
// for what is not a plain call; the operator's own way through ops.py goes on from there.
PyObject* prompt_step(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        if (nargs != 9) FAIL("prompt_step(layer, slots, cu, query, key, value, position, group, scale)");
        const Layer* L = (const Layer*)PyCapsule_GetPointer(args[0], "aicomp_amd.layer");
        if (L == nullptr) return nullptr;
        const at::Tensor *slots = plain(args[1]), *cu = plain(args[2]), *q_in = plain(args[3]), *k_in = plain(args[4]),
                         *v_in = plain(args[5]);
        const int64_t position = PyLong_AsLongLong(args[6]), group = PyLong_AsLongLong(args[7]);
        const double scale = PyFloat_AsDouble(args[8]);
        if (PyErr_Occurred()) return nullptr;
        if (!slots || !cu || !q_in || !k_in || !v_in || q_in->dim() != 4 || k_in->dim() != 4) Py_RETURN_NONE;
        const int64_t B = L->B, hq = q_in->size(1), n = q_in->size(2), H = k_in->size(1), D = L->d;
        const int64_t hstep = (group > 1 && H == (int64_t)L->hkv * group) ? group : 1;
        if (n < 2 || hq <= 0 || hq > INT_MAX || hq % L->hkv || position < 0 || n > INT_MAX || position + n >= L->ctx_count ||
            q_in->size(0) != B || q_in->size(3) != D || H != L->hkv * hstep || k_in->size(0) != B || k_in->size(2) != n ||
            k_in->size(3) != D || v_in->sizes() != k_in->sizes() || q_in->scalar_type() != L->st ||
            k_in->scalar_type() != L->st || v_in->scalar_type() != L->st || q_in->device() != L->dev ||
            k_in->device() != L->dev || v_in->device() != L->dev || slots->device() != L->dev || cu->device() != L->dev ||
            slots->scalar_type() != at::kLong || slots->dim() != 2 || slots->size(0) != B || slots->stride(1) != 1 ||
            slots->size(1) < position + n || cu->scalar_type() != at::kInt || cu->dim() != 1 || cu->size(0) != B + 1 ||
            !cu->is_contiguous())
            Py_RETURN_NONE;
        const c10::DeviceGuard guard(L->dev);
        // token-major rows: a view where the tensors are projections seen head-major, as attention layers hand them over
        const at::Tensor q = q_in->permute({0, 2, 1, 3}).contiguous();
        at::Tensor k = k_in->permute({0, 2, 1, 3}), v = v_in->permute({0, 2, 1, 3});          // [B, n, H, D]
        if (hstep > 1) { k = k.slice(2, 0, H, hstep); v = v.slice(2, 0, H, hstep); }
        if (k.stride(3) != 1 || k.strides() != v.strides() || (B > 1 && k.stride(0) != n * k.stride(1))) {
            k = k.contiguous();
            v = v.contiguous();
        }
        const at::Tensor slot = B == 1 ? *slots : slots->narrow(1, position, n).contiguous();
        const int64_t* slot_ptr = (const int64_t*)slot.data_ptr() + (B == 1 ? position : 0);
        at::Tensor out(at::detail::empty_cuda({B, n, hq, D}, L->st, L->dev, c10::MemoryFormat::Contiguous));
        void* stream = (void*)c10::hip::getCurrentHIPStream(L->dev.index()).stream();
        const int rc = unlocked([&] {
            return aicomp_kv_append_prefill_attn_sized(
                out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), k.stride(1),
                head_stride(L->hkv, L->d, k.stride(2)), L->kp, L->vp, slot_ptr,
                L->table, L->table_stride, L->ctx + (position + n) * L->ctx_stride, (const int32_t*)cu->data_ptr(), (int)B,
                B * n, (int)n, (int)hq, L->hkv, (int)D, L->bs, L->width, L->nb, (float)scale, L->dt, L->dt, nullptr, nullptr,
                nullptr, 0, (int)(position + n), stream);
        });
        if (rc != AICOMP_KV_OK) FAIL("aicomp_kv error %d: %s", rc, aicomp_kv_last_error());
        return THPVariable_Wrap(out.permute({0, 2, 1, 3}));
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// ---------------------------------------------------------------- the plain calls of aicomp_amd.ops
// Host time was what bounded these calls: their checks alone, a few dozen attribute reads of Python
// tensors, cost 15 to 20 us a call, where the kernels of a decode or rotary call of ordinary size
// need 3 to 12 (measured per call: see the wrappers in ops.py).

int any_dtype_code(at::ScalarType t) { return t == at::kFloat8_e4m3fn ? AICOMP_KV_FP8_E4M3 : dtype_code(t); }

bool on(const at::Tensor& t, const at::Tensor& ref) { return t.device() == ref.device(); }

struct Pools {
    const at::Tensor *k, *v;
    int64_t nb;
    int hkv, bs, d, dt;
    const float *ks = nullptr, *vs = nullptr;

    bool get(PyObject* ko, PyObject* vo) {
        k = plain(ko); v = plain(vo);
        if (!k || !v || k->dim() != 4 || v->sizes() != k->sizes() || k->scalar_type() != v->scalar_type() ||
            !k->is_contiguous() || !v->is_contiguous() || !on(*v, *k))
            return false;
        dt = any_dtype_code(k->scalar_type());
        nb = k->size(0); hkv = (int)k->size(1); bs = (int)k->size(2); d = (int)k->size(3);
        return dt >= 0;
    }
    // the scales of an fp8 pool; other pools have none, whatever is passed
    bool scales(PyObject* kso, PyObject* vso) {
        if (dt != AICOMP_KV_FP8_E4M3) return true;
        const at::Tensor *a = plain(kso), *b = plain(vso);
        for (const at::Tensor* s : {a, b})
            if (!s || s->scalar_type() != at::kFloat || !s->is_contiguous() || s->numel() != hkv || !on(*s, *k)) return false;
        ks = (const float*)a->data_ptr(); vs = (const float*)b->data_ptr();
        return true;
    }
};

bool vector_of(const at::Tensor* t, at::ScalarType st, int64_t n, const at::Tensor& ref) {
    return t && t->scalar_type() == st && t->numel() == n && t->is_contiguous() && on(*t, ref);
}

bool as_double(PyObject* o, double& x) {
    if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
    x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

bool as_int(PyObject* o, int& x) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || v < INT_MIN || v > INT_MAX) return false;
    x = (int)v;
    return true;
}

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

#define DONE(rc)                                                                                     \
    do {                                                                                             \
        if ((rc) != AICOMP_KV_OK) FAIL("aicomp_kv error %d: %s", (rc), aicomp_kv_last_error());      \
        Py_RETURN_TRUE;                                                                              \
    } while (0)

PyObject* kv_append(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        if (nargs != 7) FAIL("kv_append(key, value, k_pool, v_pool, slot_mapping, k_scale, v_scale)");
        const at::Tensor *key = plain(args[0]), *value = plain(args[1]), *slots = plain(args[4]);
        if (!key || !value || !p.get(args[2], args[3]) || key->dim() != 3 || value->sizes() != key->sizes() ||
            value->scalar_type() != key->scalar_type() || key->size(1) != p.hkv || key->size(2) != p.d ||
            !slots || slots->dim() != 1 || !vector_of(slots, at::kLong, key->size(0), *key) || !on(*value, *key) ||
            !on(*p.k, *key) || key->stride(2) != 1 || key->strides() != value->strides())
            Py_RETURN_FALSE;
        const int dt = any_dtype_code(key->scalar_type());
        if (dt < 0 || (dt != p.dt && !p.scales(args[5], args[6]))) Py_RETURN_FALSE;
        const c10::DeviceGuard guard(key->device());
        void* stream = stream_of(*key);
        const int rc = unlocked([&] {
            return aicomp_kv_append(key->data_ptr(), value->data_ptr(), key->stride(0), key->stride(1), p.k->data_ptr(),
                                    p.v->data_ptr(), (const int64_t*)slots->data_ptr(), key->size(0), p.hkv, p.d, p.bs,
                                    p.nb, dt, p.dt, p.ks, p.vs, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

PyObject* rope_kv_append(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        if (nargs != 12)
            FAIL("rope_kv_append(query, key, value, cos, sin, positions, k_pool, v_pool, slot_mapping, k_scale, v_scale, out)");
        const at::Tensor *q = plain(args[0]), *key = plain(args[1]), *value = plain(args[2]), *cos = plain(args[3]),
                         *sin = plain(args[4]), *slots = plain(args[8]), *out = plain(args[11]);
        const bool by_row = args[5] == Py_None;
        const at::Tensor* pos = by_row ? nullptr : plain(args[5]);
        if (!q || !key || !value || !cos || !sin || !out || (!by_row && !pos) || !p.get(args[6], args[7]) ||
            q->dim() != 3 || key->dim() != 3 || value->sizes() != key->sizes() || out->sizes() != q->sizes())
            Py_RETURN_FALSE;
        const int64_t T = q->size(0);
        const at::ScalarType st = q->scalar_type();
        const int dt = dtype_code(st);
        if (T == 0 || dt < 0 || key->size(0) != T || key->size(1) != p.hkv || key->size(2) != p.d || q->size(2) != p.d ||
            key->scalar_type() != st || value->scalar_type() != st || out->scalar_type() != st || q->stride(2) != 1 ||
            out->stride(2) != 1 || key->stride(2) != 1 || key->strides() != value->strides() || cos->dim() != 2 ||
            cos->size(1) != p.d || sin->sizes() != cos->sizes() || cos->scalar_type() != st || sin->scalar_type() != st ||
            cos->stride(1) != 1 || cos->strides() != sin->strides())
            Py_RETURN_FALSE;
        if (by_row ? cos->size(0) < T : !vector_of(pos, at::kLong, T, *q)) Py_RETURN_FALSE;
        if (!vector_of(slots, at::kLong, T, *q) || !on(*key, *q) || !on(*value, *q) || !on(*out, *q) || !on(*cos, *q) ||
            !on(*sin, *q) || !on(*p.k, *q) || (p.dt != dt && p.dt != AICOMP_KV_FP8_E4M3) || !p.scales(args[9], args[10]))
            Py_RETURN_FALSE;
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        const int rc = unlocked([&] {
            return aicomp_rope_kv_append(
                q->data_ptr(), out->data_ptr(), q->stride(0), q->stride(1), out->stride(0), out->stride(1),
                key->data_ptr(), value->data_ptr(), key->stride(0), key->stride(1), cos->data_ptr(), sin->data_ptr(),
                cos->stride(0), cos->size(0), pos ? (const int64_t*)pos->data_ptr() : nullptr, p.k->data_ptr(),
                p.v->data_ptr(), (const int64_t*)slots->data_ptr(), T, (int)q->size(1), p.hkv, p.d, p.bs, p.nb, dt, p.dt,
                p.ks, p.vs, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// what a decode and a prefill call share
bool attention_args(PyObject* const* args, const at::Tensor*& out, const at::Tensor*& q, Pools& p, const at::Tensor*& table,
                    const at::Tensor*& ctx, int& dt, int64_t& rows) {
    out = plain(args[0]); q = plain(args[1]); table = plain(args[4]); ctx = plain(args[5]);
    if (!out || !q || !table || !ctx || !p.get(args[2], args[3]) || q->dim() != 3 || out->sizes() != q->sizes() ||
        out->scalar_type() != q->scalar_type() || q->size(2) != p.d || !q->is_contiguous() || !out->is_contiguous())
        return false;
    dt = any_dtype_code(q->scalar_type());
    rows = ctx->numel();
    return dt >= 0 && vector_of(ctx, at::kInt, rows, *q) && table->scalar_type() == at::kInt && table->dim() == 2 &&
           table->size(0) == rows && table->stride(1) == 1 && on(*table, *q) && on(*out, *q) && on(*p.k, *q);
}

PyObject* paged_decode_attn(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        const at::Tensor *out, *q, *table, *ctx;
        int dt, partition;
        int64_t B;
        double scale;
        if (nargs != 13)
            FAIL("paged_decode_attn(out, query, k_pool, v_pool, block_table, context_lens, scale, k_scale, v_scale, "
                 "partition_size, workspace, new_key, new_value)");
        if (!attention_args(args, out, q, p, table, ctx, dt, B) || B != q->size(0) || !as_double(args[6], scale) ||
            !p.scales(args[7], args[8]) || !as_int(args[9], partition))
            Py_RETURN_FALSE;
        const at::Tensor *nk = nullptr, *nv = nullptr;
        if (args[11] != Py_None) {
            nk = plain(args[11]); nv = plain(args[12]);
            if (!nk || !nv || nk->dim() != 3 || nk->size(0) != B || nk->size(1) != p.hkv || nk->size(2) != p.d ||
                nv->sizes() != nk->sizes() || nk->scalar_type() != q->scalar_type() ||
                nv->scalar_type() != q->scalar_type() || !on(*nk, *q) || !on(*nv, *q) || nk->stride(2) != 1 ||
                nk->strides() != nv->strides())
                Py_RETURN_FALSE;
        }
        const int hq = (int)q->size(1), width = (int)table->size(1);
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        at::Tensor scratch;
        bool shared = false;                           // the module's own scratch, not the caller's
        if (args[10] != Py_None) {
            const at::Tensor* w = plain(args[10]);
            if (!w) Py_RETURN_FALSE;
            scratch = *w;
        } else {
            const size_t need = aicomp_paged_decode_workspace_bytes((int)B, hq, p.hkv, p.d, p.bs, width, dt, p.dt, partition);
            shared = need != 0;
            if (shared) scratch = cached_scratch(q->device(), stream, need);
        }
        void* ws = scratch.defined() ? scratch.data_ptr() : nullptr;
        const size_t ws_bytes = scratch.defined() ? (size_t)(scratch.numel() * scratch.element_size()) : 0;
        const int rc = unlocked([&] {
            std::unique_lock<std::mutex> one_at_a_time(scratch_launches(), std::defer_lock);
            if (shared) one_at_a_time.lock();
            const int32_t *bt = (const int32_t*)table->data_ptr(), *cl = (const int32_t*)ctx->data_ptr();
            if (nk)
                return aicomp_paged_decode_attn_append(
                    out->data_ptr(), q->data_ptr(), nk->data_ptr(), nv->data_ptr(), nk->stride(0), nk->stride(1),
                    p.k->data_ptr(), p.v->data_ptr(), bt, table->stride(0), cl, (int)B, hq, p.hkv, p.d, p.bs, width, p.nb,
                    (float)scale, dt, p.dt, p.ks, p.vs, partition, ws, ws_bytes, stream);
            return aicomp_paged_decode_attn(out->data_ptr(), q->data_ptr(), p.k->data_ptr(), p.v->data_ptr(), bt,
                                            table->stride(0), cl, (int)B, hq, p.hkv, p.d, p.bs, width, p.nb, (float)scale,
                                            dt, p.dt, p.ks, p.vs, partition, ws, ws_bytes, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// The longest of `lens` (a contiguous int32 buffer of n lengths), which sizes a call and bounds nothing; 0, for the whole
// table, without such a buffer.
int longest_of(PyObject* lens, int64_t n) {
    if (lens == Py_None) return 0;
    Py_buffer b;
    if (PyObject_GetBuffer(lens, &b, PyBUF_FORMAT | PyBUF_ND) != 0) { PyErr_Clear(); return 0; }
    int longest = 0;
    if (b.itemsize == 4 && b.ndim == 1 && b.shape[0] == n && b.format && b.format[0] == 'i' && b.format[1] == 0) {
        longest = 1;
        for (int64_t i = 0; i < n; ++i) longest = std::max(longest, ((const int32_t*)b.buf)[i]);
    }
    PyBuffer_Release(&b);
    return longest;
}

// (a status that cannot be had counts as recording)
bool recording(void* stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

// Whether every row's slot is where its table has the row's last token, or none (a padding row): host copies of the
// lengths, slots and table (contiguous int32 [n], int64 [n], int32 [n, columns]).
bool slots_at_table(PyObject* lens, PyObject* slots, PyObject* table, int64_t n, int bs) {
    struct View {
        Py_buffer b{};
        bool held;
        View(PyObject* o, const char* kind, Py_ssize_t size) {
            held = PyObject_GetBuffer(o, &b, PyBUF_FORMAT | PyBUF_ND) == 0;
            if (!held) PyErr_Clear();
            ok = held && b.itemsize == size && b.format && strchr(kind, b.format[0]) && b.format[1] == 0;
        }
        ~View() { if (held) PyBuffer_Release(&b); }
        bool ok;
    };
    const View l(lens, "i", 4), s(slots, "lq", 8), t(table, "i", 4);
    if (!l.ok || !s.ok || !t.ok || l.b.ndim != 1 || s.b.ndim != 1 || t.b.ndim != 2 || l.b.shape[0] != n || s.b.shape[0] != n ||
        t.b.shape[0] != n)
        return false;
    const int64_t columns = t.b.shape[1];
    for (int64_t r = 0; r < n; ++r) {
        const int64_t slot = ((const int64_t*)s.b.buf)[r], last = (int64_t)((const int32_t*)l.b.buf)[r] - 1;
        if (slot < 0) continue;
        if (last < 0 || last / bs >= columns || slot != (int64_t)((const int32_t*)t.b.buf)[r * columns + last / bs] * bs + last % bs)
            return false;
    }
    return true;
}

// (the output comes back as a new tensor; None: not a plain call of the one launch, nothing done)
PyObject* rope_paged_decode_attn(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        double scale;
        if (nargs != 17)
            FAIL("rope_paged_decode_attn(query, key, value, cos, sin, positions, k_pool, v_pool, slot_mapping, block_table, "
                 "context_lens, host_lens, scale, k_scale, v_scale, host_slots, host_table)");
        const at::Tensor *q = plain(args[0]), *key = plain(args[1]), *value = plain(args[2]), *cos = plain(args[3]),
                         *sin = plain(args[4]), *pos = plain(args[5]), *slots = plain(args[8]), *table = plain(args[9]),
                         *ctx = plain(args[10]);
        if (!q || !key || !value || !cos || !sin || !pos || !slots || !table || !ctx || !p.get(args[6], args[7]) ||
            !as_double(args[12], scale) || q->dim() != 3 || key->dim() != 3 ||
            value->sizes() != key->sizes())
            Py_RETURN_NONE;
        const int64_t B = q->size(0);
        const at::ScalarType st = q->scalar_type();
        const int dt = dtype_code(st);
        if (B == 0 || B > INT_MAX || dt < 0 || key->size(0) != B || key->size(1) != p.hkv || key->size(2) != p.d ||
            q->size(2) != p.d || key->scalar_type() != st || value->scalar_type() != st || q->stride(2) != 1 ||
            key->stride(2) != 1 || key->strides() != value->strides() || cos->dim() != 2 || cos->size(1) != p.d ||
            sin->sizes() != cos->sizes() || cos->scalar_type() != st || sin->scalar_type() != st || cos->stride(1) != 1 ||
            cos->strides() != sin->strides() || table->scalar_type() != at::kInt || table->dim() != 2 ||
            p.bs <= 0 || table->size(0) != B || table->stride(1) != 1 || table->size(1) <= 0 || table->size(1) > INT_MAX ||
            !vector_of(pos, at::kLong, B, *q) || !vector_of(slots, at::kLong, B, *q) || !vector_of(ctx, at::kInt, B, *q) ||
            !on(*table, *q) || !on(*key, *q) || !on(*value, *q) || !on(*cos, *q) || !on(*sin, *q) || !on(*p.k, *q) ||
            (p.dt != dt && p.dt != AICOMP_KV_FP8_E4M3) || !p.scales(args[13], args[14]) ||
            (args[15] != Py_None && !slots_at_table(args[11], args[15], args[16], B, p.bs)))
            Py_RETURN_NONE;
        const int hq = (int)q->size(1);
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        // a recorded launch is sized for the whole table: the lengths of its replays may grow by any amount
        const int width = (int)table->size(1);
        int longest = longest_of(args[11], B);
        if (longest != 0 && ((int64_t)longest + p.bs - 1) / p.bs < width && recording(stream)) longest = 0;
        const int sized = longest == 0 ? width : (int)std::min<int64_t>(width, ((int64_t)longest + p.bs - 1) / p.bs);
        at::Tensor scratch;
        const size_t need = aicomp_paged_decode_workspace_bytes((int)B, hq, p.hkv, p.d, p.bs, sized, dt, p.dt, 0);
        if (need) scratch = cached_scratch(q->device(), stream, need);
        at::Tensor out(at::detail::empty_cuda(q->sizes(), st, q->device(), c10::MemoryFormat::Contiguous));
        const int rc = unlocked([&] {
            std::unique_lock<std::mutex> one_at_a_time(scratch_launches(), std::defer_lock);
            if (need) one_at_a_time.lock();
            return aicomp_rope_paged_decode_attn_sized(
                out.data_ptr(), q->data_ptr(), q->stride(0), q->stride(1), key->data_ptr(), value->data_ptr(), key->stride(0),
                key->stride(1), cos->data_ptr(), sin->data_ptr(), cos->stride(0), cos->size(0),
                (const int64_t*)pos->data_ptr(), (const int64_t*)slots->data_ptr(), p.k->data_ptr(), p.v->data_ptr(),
                (const int32_t*)table->data_ptr(), table->stride(0), (const int32_t*)ctx->data_ptr(), (int)B, hq, p.hkv, p.d,
                p.bs, width, p.nb, (float)scale, dt, p.dt, p.ks, p.vs, longest, need ? scratch.data_ptr() : nullptr,
                need ? (size_t)scratch.numel() : 0, stream);
        });
        if (rc == AICOMP_KV_EUNSUPPORTED) Py_RETURN_NONE;
        if (rc != AICOMP_KV_OK) FAIL("aicomp_kv error %d: %s", rc, aicomp_kv_last_error());
        return THPVariable_Wrap(std::move(out));
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

PyObject* paged_prefill_attn(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        const at::Tensor *out, *q, *table, *ctx;
        int dt, max_q_len;
        int64_t S;
        double scale;
        if (nargs != 12)
            FAIL("paged_prefill_attn(out, query, k_pool, v_pool, block_table, context_lens, cu_q_lens, scale, max_q_len, "
                 "k_scale, v_scale, items)");
        if (!attention_args(args, out, q, p, table, ctx, dt, S) || !as_double(args[7], scale) ||
            !as_int(args[8], max_q_len) || !p.scales(args[9], args[10]))
            Py_RETURN_FALSE;
        const at::Tensor* cu = plain(args[6]);
        if (!vector_of(cu, at::kInt, S + 1, *q)) Py_RETURN_FALSE;
        const at::Tensor* items = nullptr;
        if (args[11] != Py_None) {
            items = plain(args[11]);
            if (!items || items->numel() == 0 || items->scalar_type() != at::kInt || items->dim() != 2 ||
                items->size(1) != 2 || items->size(0) > INT_MAX || !items->is_contiguous() || !on(*items, *q))
                Py_RETURN_FALSE;
        }
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        const int rc = unlocked([&] {
            return aicomp_paged_prefill_attn_items(
                out->data_ptr(), q->data_ptr(), p.k->data_ptr(), p.v->data_ptr(), (const int32_t*)table->data_ptr(),
                table->stride(0), (const int32_t*)ctx->data_ptr(), (const int32_t*)cu->data_ptr(), (int)S, q->size(0),
                max_q_len, (int)q->size(1), p.hkv, p.d, p.bs, (int)table->size(1), p.nb, (float)scale, dt, p.dt, p.ks, p.vs,
                items ? (const int32_t*)items->data_ptr() : nullptr, items ? (int)items->size(0) : 0, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// key, value and slot_mapping None: the rows are in the pools already
PyObject* append_prefill_attn(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        const at::Tensor *out, *q, *table, *ctx;
        int dt, max_q_len;
        int64_t S;
        double scale;
        if (nargs != 16)
            FAIL("append_prefill_attn(out, query, k_pool, v_pool, block_table, context_lens, cu_q_lens, scale, max_q_len, "
                 "k_scale, v_scale, items, key, value, slot_mapping, host_lens)");
        if (!attention_args(args, out, q, p, table, ctx, dt, S) || !as_double(args[7], scale) ||
            !as_int(args[8], max_q_len) || !p.scales(args[9], args[10]))
            Py_RETURN_FALSE;
        const at::Tensor* cu = plain(args[6]);
        if (!vector_of(cu, at::kInt, S + 1, *q)) Py_RETURN_FALSE;
        const at::Tensor *items = nullptr, *key = nullptr, *value = nullptr, *slots = nullptr;
        if (args[11] != Py_None) {
            items = plain(args[11]);
            if (!items || items->numel() == 0 || items->scalar_type() != at::kInt || items->dim() != 2 ||
                items->size(1) != 2 || items->size(0) > INT_MAX || !items->is_contiguous() || !on(*items, *q))
                Py_RETURN_FALSE;
        }
        if (args[12] != Py_None) {
            key = plain(args[12]); value = plain(args[13]); slots = plain(args[14]);
            if (!key || !value || !slots || key->dim() != 3 || value->sizes() != key->sizes() ||
                key->scalar_type() != q->scalar_type() || value->scalar_type() != q->scalar_type() ||
                key->size(0) != q->size(0) || key->size(1) != p.hkv || key->size(2) != p.d || slots->dim() != 1 ||
                !vector_of(slots, at::kLong, key->size(0), *q) || !on(*key, *q) || !on(*value, *q) ||
                key->stride(2) != 1 || key->strides() != value->strides())
                Py_RETURN_FALSE;
        }
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        const int longest = dt == AICOMP_KV_F32 ? 0 : longest_of(args[15], S);       // (float32 has no line that looks at it)
        const int rc = unlocked([&] {
            return aicomp_kv_append_prefill_attn_sized(
                out->data_ptr(), q->data_ptr(), key ? key->data_ptr() : nullptr, key ? value->data_ptr() : nullptr,
                key ? key->stride(0) : 0, key ? key->stride(1) : 0, p.k->data_ptr(), p.v->data_ptr(),
                key ? (const int64_t*)slots->data_ptr() : nullptr, (const int32_t*)table->data_ptr(), table->stride(0),
                (const int32_t*)ctx->data_ptr(), (const int32_t*)cu->data_ptr(), (int)S, q->size(0), max_q_len,
                (int)q->size(1), p.hkv, p.d, p.bs, (int)table->size(1), p.nb, (float)scale, dt, p.dt, p.ks, p.vs,
                items ? (const int32_t*)items->data_ptr() : nullptr, items ? (int)items->size(0) : 0, longest, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// A layer's step of prompt chunks (the first `chunks` sequences, t_pre rows) and one-token rows after them, each through
// their own kernels: append and prefill of the chunks, append and decode of the rows; key, value and slot_mapping None where
// the new rows are in the pools already.  (Slices of a dozen tensors and three calls through Python were 36 us a step, this is 22.)
PyObject* chunks_and_rows(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        Pools p;
        const at::Tensor *out, *q, *table, *ctx;
        int dt, max_q_len, chunks, t_pre;
        int64_t S;
        double scale;
        if (nargs != 18)
            FAIL("chunks_and_rows(out, query, k_pool, v_pool, block_table, context_lens, cu_q_lens, scale, max_q_len, k_scale, "
                 "v_scale, items, key, value, slot_mapping, chunks, t_pre, chunk_lens)");
        if (!attention_args(args, out, q, p, table, ctx, dt, S) || !as_double(args[7], scale) ||
            !as_int(args[8], max_q_len) || !p.scales(args[9], args[10]) || !as_int(args[15], chunks) || !as_int(args[16], t_pre))
            Py_RETURN_FALSE;
        const int64_t T = q->size(0), rows = S - chunks;
        const at::Tensor* cu = plain(args[6]);
        if (!vector_of(cu, at::kInt, S + 1, *q) || chunks <= 0 || rows <= 0 || S > INT_MAX || t_pre <= 0 || t_pre + rows != T)
            Py_RETURN_FALSE;
        const at::Tensor *items = nullptr, *key = nullptr, *value = nullptr, *slots = nullptr;
        if (args[11] != Py_None) {
            items = plain(args[11]);
            if (!items || items->numel() == 0 || items->scalar_type() != at::kInt || items->dim() != 2 ||
                items->size(1) != 2 || items->size(0) > INT_MAX || !items->is_contiguous() || !on(*items, *q))
                Py_RETURN_FALSE;
        }
        if (args[12] != Py_None) {
            key = plain(args[12]); value = plain(args[13]); slots = plain(args[14]);
            if (!key || !value || !slots || key->dim() != 3 || value->sizes() != key->sizes() ||
                key->scalar_type() != q->scalar_type() || value->scalar_type() != q->scalar_type() ||
                key->size(0) != T || key->size(1) != p.hkv || key->size(2) != p.d || slots->dim() != 1 ||
                !vector_of(slots, at::kLong, T, *q) || !on(*key, *q) || !on(*value, *q) || key->stride(2) != 1 ||
                key->strides() != value->strides())
                Py_RETURN_FALSE;
        }
        const int hq = (int)q->size(1), width = (int)table->size(1);
        const c10::DeviceGuard guard(q->device());
        void* stream = stream_of(*q);
        at::Tensor scratch;
        const size_t need = aicomp_paged_decode_workspace_bytes((int)rows, hq, p.hkv, p.d, p.bs, width, dt, p.dt, 0);
        if (need) scratch = cached_scratch(q->device(), stream, need);
        // (with the chunks' lengths they may take the kernel for few chunks)
        const bool few = args[17] != Py_None && dt != AICOMP_KV_F32;
        const int longest = few ? longest_of(args[17], chunks) : 0;
        const int rc = unlocked([&] {
            const int32_t *bt = (const int32_t*)table->data_ptr(), *cl = (const int32_t*)ctx->data_ptr();
            const int64_t done = (int64_t)t_pre * hq * p.d * q->element_size();            // query and output of the chunks
            void *kp = p.k->data_ptr(), *vp = p.v->data_ptr();
            const int64_t* slot = key ? (const int64_t*)slots->data_ptr() : nullptr;
            const int32_t *off = (const int32_t*)cu->data_ptr(), *list = items ? (const int32_t*)items->data_ptr() : nullptr;
            const int pairs = items ? (int)items->size(0) : 0;
            int rc = AICOMP_KV_OK;
            if (few) {
                rc = aicomp_kv_append_prefill_attn_sized(
                    out->data_ptr(), q->data_ptr(), key ? key->data_ptr() : nullptr, key ? value->data_ptr() : nullptr,
                    key ? key->stride(0) : 0, key ? key->stride(1) : 0, kp, vp, slot, bt, table->stride(0), cl, off, chunks, t_pre,
                    max_q_len, hq, p.hkv, p.d, p.bs, width, p.nb, (float)scale, dt, p.dt, p.ks, p.vs, list, pairs, longest, stream);
            } else {
                if (key)
                    rc = aicomp_kv_append(key->data_ptr(), value->data_ptr(), key->stride(0), key->stride(1), kp, vp, slot, t_pre,
                                          p.hkv, p.d, p.bs, p.nb, dt, p.dt, p.ks, p.vs, stream);
                if (rc == AICOMP_KV_OK)
                    rc = aicomp_paged_prefill_attn_items(out->data_ptr(), q->data_ptr(), kp, vp, bt, table->stride(0), cl, off, chunks,
                                                         t_pre, max_q_len, hq, p.hkv, p.d, p.bs, width, p.nb, (float)scale, dt,
                                                         p.dt, p.ks, p.vs, list, pairs, stream);
            }
            if (rc != AICOMP_KV_OK) return rc;
            std::unique_lock<std::mutex> one_at_a_time(scratch_launches(), std::defer_lock);
            if (need) one_at_a_time.lock();
            char *o = (char*)out->data_ptr() + done;
            const char* qr = (const char*)q->data_ptr() + done;
            bt += chunks * table->stride(0); cl += chunks;
            void* ws = need ? scratch.data_ptr() : nullptr;
            const size_t ws_bytes = need ? (size_t)scratch.numel() : 0;
            if (key) {
                const int64_t later = t_pre * key->stride(0) * (int64_t)key->element_size();
                return aicomp_paged_decode_attn_append(
                    o, qr, (const char*)key->data_ptr() + later, (const char*)value->data_ptr() + later, key->stride(0),
                    key->stride(1), kp, vp, bt, table->stride(0), cl, (int)rows, hq, p.hkv, p.d, p.bs, width, p.nb,
                    (float)scale, dt, p.dt, p.ks, p.vs, 0, ws, ws_bytes, stream);
            }
            return aicomp_paged_decode_attn(o, qr, kp, vp, bt, table->stride(0), cl, (int)rows, hq, p.hkv, p.d, p.bs, width, p.nb,
                                            (float)scale, dt, p.dt, p.ks, p.vs, 0, ws, ws_bytes, stream);
        });
        DONE(rc);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// (tokens come back as a new tensor; None: take the Python way)
PyObject* sample_tokens(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        if (nargs != 6) FAIL("sample_tokens(logits, temperature, top_k, top_p, do_sample, uniforms)");
        const at::Tensor *x = plain(args[0]), *u = nullptr;
        double temperature, top_p;
        int top_k;
        if (!x || x->dim() != 2 || x->size(0) == 0 || x->size(0) > INT_MAX || x->size(1) > INT_MAX || x->stride(1) != 1 ||
            dtype_code(x->scalar_type()) < 0 || !as_double(args[1], temperature) || !as_int(args[2], top_k) ||
            !as_double(args[3], top_p) || !PyBool_Check(args[4]))
            Py_RETURN_NONE;
        const bool sample = args[4] == Py_True;
        if (sample && !vector_of(u = plain(args[5]), at::kFloat, x->size(0), *x)) Py_RETURN_NONE;
        const c10::DeviceGuard guard(x->device());
        void* stream = stream_of(*x);
        at::Tensor out(at::detail::empty_cuda({x->size(0)}, at::kLong, x->device(), c10::MemoryFormat::Contiguous));
        const size_t need = aicomp_sample_workspace_bytes((int)x->size(0), (int)x->size(1), x->stride(0), (float)temperature, top_k,
                                                          sample ? 0 : 1, dtype_code(x->scalar_type()));
        at::Tensor scratch;                 // the allocator orders its next user behind this call
        if (need) scratch = at::detail::empty_cuda({(int64_t)need}, at::kByte, x->device(), c10::MemoryFormat::Contiguous);
        const int rc = unlocked([&] {
            return aicomp_sample_tokens_split((int64_t*)out.data_ptr(), x->data_ptr(), x->stride(0), nullptr,
                                              sample ? (const float*)u->data_ptr() : nullptr, (int)x->size(0),
                                              (int)x->size(1), (float)temperature, top_k, (float)top_p, sample ? 0 : 1,
                                              dtype_code(x->scalar_type()), need ? scratch.data_ptr() : nullptr, need,
                                              stream);
        });
        if (rc != AICOMP_KV_OK) FAIL("aicomp_kv error %d: %s", rc, aicomp_kv_last_error());
        return THPVariable_Wrap(std::move(out));
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// ---------------------------------------------------------------- the step planner's decode step
// What StepPlanner.schedule and _pack do with about forty numpy operations of a microsecond each, for a step that is one
// token per running sequence and nothing else: 52 us of host time at 8 sequences, of which these functions leave 20
// (most of that the copy's own call, its event and the plan's tensors).

// A contiguous buffer of at least n elements of `size` bytes, released with the object; null data where it is not one.
struct Buf {
    Py_buffer b{};
    bool held = false;
    void* data(PyObject* o, Py_ssize_t size, int64_t n, bool writable = false) {
        held = PyObject_GetBuffer(o, &b, PyBUF_ND | (writable ? PyBUF_WRITABLE : 0)) == 0;
        if (!held) { PyErr_Clear(); return nullptr; }
        return b.itemsize == size && b.len >= size * n ? b.buf : nullptr;
    }
    int64_t items() const { return held && b.itemsize ? (int64_t)(b.len / b.itemsize) : 0; }
    ~Buf() { if (held) PyBuffer_Release(&b); }
};

// per row of the planner: live (bool), len, prompt, orig, nblk (int32), maxnew, arrival (int64)
struct Rows {
    Buf b[7];
    int64_t n = 0;
    const uint8_t* live;
    int32_t *len, *nblk;
    const int32_t *prompt, *orig;
    const int64_t *maxnew, *arrival;
    bool get(PyObject* const* a, bool writable) {
        live = (const uint8_t*)b[0].data(a[0], 1, 0);
        n = b[0].items();
        len = (int32_t*)b[1].data(a[1], 4, n, writable);
        prompt = (const int32_t*)b[2].data(a[2], 4, n);
        orig = (const int32_t*)b[3].data(a[3], 4, n);
        nblk = (int32_t*)b[4].data(a[4], 4, n, writable);
        maxnew = (const int64_t*)b[5].data(a[5], 8, n);
        arrival = (const int64_t*)b[6].data(a[6], 8, n);
        return live && len && prompt && orig && nblk && maxnew && arrival;
    }
    int64_t generated(int64_t r) const { return (int64_t)len[r] - orig[r] + 1; }
};

PyObject* rows_done(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    Rows R;
    if (nargs != 7) FAIL("rows_done(live, len, prompt, orig, nblk, maxnew, arrival)");
    if (!R.get(args, false)) Py_RETURN_NONE;
    PyObject* out = PyList_New(0);
    for (int64_t r = 0; out && r < R.n; ++r) {
        if (!R.live[r] || R.maxnew[r] < 0 || R.len[r] < R.prompt[r] || R.generated(r) < R.maxnew[r]) continue;
        PyObject* i = PyLong_FromLongLong(r);
        if (!i || PyList_Append(out, i) != 0) Py_CLEAR(out);
        Py_XDECREF(i);
    }
    return out;
}

// -> (rows in plan order, blocks taken), the plan packed into `raw` and the rows' state moved on; None with nothing
// changed where the step is another one (a prompt to ingest, no free block, a sequence too long, nothing to do).
PyObject* plan_decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 15)
        FAIL("plan_decode(live, len, prompt, orig, nblk, maxnew, arrival, table, free, owned, top, block_size, max_seq_len, "
             "budget, raw)");
    Rows R;
    int top, bs, longest, budget;
    if (!R.get(args, true) || !as_int(args[10], top) || !as_int(args[11], bs) || !as_int(args[12], longest) ||
        !as_int(args[13], budget) || bs <= 0 || R.n == 0)
        Py_RETURN_NONE;
    Buf bt, bf, bo, br;
    int32_t* table = (int32_t*)bt.data(args[7], 4, R.n, true);
    const int32_t* free_ids = (const int32_t*)bf.data(args[8], 4, 0);
    uint8_t* owned = (uint8_t*)bo.data(args[9], 1, 0, true);
    uint8_t* raw = (uint8_t*)br.data(args[14], 1, 0, true);
    if (!table || !free_ids || !owned || !raw || top < 0 || top > bf.items() || (uintptr_t)raw % 8) Py_RETURN_NONE;
    const int64_t MB = bt.items() / R.n;
    try {
        std::vector<int> rows;
        for (int64_t r = 0; r < R.n; ++r) {
            if (!R.live[r]) continue;
            if (R.len[r] < R.prompt[r]) Py_RETURN_NONE;
            if (R.maxnew[r] < 0 || R.generated(r) < R.maxnew[r]) rows.push_back((int)r);
        }
        std::stable_sort(rows.begin(), rows.end(), [&](int a, int b) { return R.arrival[a] < R.arrival[b]; });
        if ((int64_t)rows.size() > budget) rows.resize(std::max(budget, 0));
        const int64_t S = (int64_t)rows.size(), end = 16 * S + 4 * (S * MB + 2 * S + 1);
        int taken = 0;
        for (int r : rows) {
            if (R.len[r] + 1 > longest || R.len[r] < 0 || R.len[r] / bs >= MB || R.nblk[r] < 0 || R.nblk[r] > MB) Py_RETURN_NONE;
            const bool opens = (int64_t)R.nblk[r] * bs == R.len[r];
            if (!opens && R.len[r] / bs >= R.nblk[r]) Py_RETURN_NONE;
            taken += opens;
        }
        if (S == 0 || taken > top || end > br.items()) Py_RETURN_NONE;
        for (int i = 0; i < taken; ++i)
            if (free_ids[top - 1 - i] < 0 || free_ids[top - 1 - i] >= bo.items()) Py_RETURN_NONE;
        PyObject* ids = PyList_New(S);
        if (!ids) return nullptr;
        int64_t* slot = (int64_t*)raw;
        int64_t* pos = slot + S;
        int32_t* tab = (int32_t*)(pos + S);
        int32_t *ctx = tab + S * MB, *cu = ctx + S;
        cu[0] = 0;
        int next = top;
        for (int64_t i = 0; i < S; ++i) {
            const int r = rows[i];
            int32_t* mine = table + (int64_t)r * MB;
            const int32_t p = R.len[r];
            if ((int64_t)R.nblk[r] * bs == p) {
                const int32_t blk = free_ids[--next];
                owned[blk] = 1;
                mine[R.nblk[r]++] = blk;
            }
            std::copy(mine, mine + MB, tab + i * MB);
            slot[i] = (int64_t)mine[p / bs] * bs + p % bs;
            pos[i] = p;
            ctx[i] = R.len[r] = p + 1;
            cu[i + 1] = (int32_t)(i + 1);
            PyList_SET_ITEM(ids, i, PyLong_FromLong(r));
        }
        return Py_BuildValue("(Ni)", ids, taken);
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

// The packed plan's copy to the device, and its five tensors there: block_table, context_lens, cu_q_lens, slot_mapping,
// positions of a step of one token per sequence.
PyObject* plan_upload(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    try {
        int S, MB;
        if (nargs != 6) FAIL("plan_upload(host, device, device as int32, device as int64, sequences, table width)");
        for (int i = 0; i < 4; ++i)
            if (!THPVariable_Check(args[i])) FAIL("plan_upload: argument %d is not a tensor", i);
        if (!as_int(args[4], S) || !as_int(args[5], MB) || S <= 0 || MB < 0) FAIL("plan_upload: bad sizes");
        const at::Tensor &host = THPVariable_Unpack(args[0]), &dev = THPVariable_Unpack(args[1]);
        const at::Tensor &d32 = THPVariable_Unpack(args[2]), &d64 = THPVariable_Unpack(args[3]);
        const int64_t t = 4 * (int64_t)S, c = t + (int64_t)S * MB, end = 4 * (c + 2 * (int64_t)S + 1);
        if (!dev.is_same(host)) dev.narrow(0, 0, end).copy_(host.narrow(0, 0, end), /*non_blocking=*/true);
        return Py_BuildValue("(NNNNN)", THPVariable_Wrap(d32.narrow(0, t, c - t).view({S, MB})),
                             THPVariable_Wrap(d32.narrow(0, c, S)), THPVariable_Wrap(d32.narrow(0, c + S, S + 1)),
                             THPVariable_Wrap(d64.narrow(0, 0, S)), THPVariable_Wrap(d64.narrow(0, S, S)));
    } catch (const std::exception& e) {
        FAIL("%s", e.what());
    }
}

#define FAST(f) (PyCFunction)(void (*)(void))f, METH_FASTCALL

PyMethodDef methods[] = {
    {"layer", (PyCFunction)(void (*)(void))layer_new, METH_FASTCALL,
     "layer(k_pool, v_pool, block_table, ctx_rows) -> handle: a layer's static tensors, checked once"},
    {"decode_step", (PyCFunction)(void (*)(void))decode_step, METH_FASTCALL,
     "decode_step(layer, query, key, value, position, group, scale) -> out [B, Hq, 1, D]"},
    {"prompt_step", FAST(prompt_step),
     "prompt_step(layer, slots, cu, query, key, value, position, group, scale) -> out [B, Hq, n, D], or None"},
    {"kv_append", FAST(kv_append), "ops.kv_append of a plain call: True once launched, False if it is not one"},
    {"rope_kv_append", FAST(rope_kv_append), "ops.rope_kv_append of a plain call, out given"},
    {"paged_decode_attn", FAST(paged_decode_attn), "ops.paged_decode_attn of a plain call"},
    {"rope_paged_decode_attn", FAST(rope_paged_decode_attn), "a layer's decode step in one launch: the output, or None if it is not one"},
    {"rows_done", FAST(rows_done), "planner rows that have produced their tokens"},
    {"plan_decode", FAST(plan_decode), "a step of one token per running sequence, packed: (rows, blocks taken), or None"},
    {"plan_upload", FAST(plan_upload), "the packed plan on its way to the device: its five tensors there"},
    {"paged_prefill_attn", FAST(paged_prefill_attn), "ops.paged_prefill_attn of a plain call, max_q_len given"},
    {"append_prefill_attn", FAST(append_prefill_attn), "ops.append_prefill_attn of a plain call"},
    {"chunks_and_rows", FAST(chunks_and_rows), "prompt chunks and one-token rows of a step, each through their own kernels"},
    {"sample_tokens", FAST(sample_tokens), "ops.sample_tokens of a plain call: the tokens, or None if it is not one"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_aicomp_fast", "lean host routes into the paged KV-cache library",
                      -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__aicomp_fast(void) { return PyModule_Create(&module); }
