// Host path of the Python operators in native code: what flash_sparse_attn_func, flash_sparse_attn_varlen_func,
// dynamic_mask_bias and create_mask do between their arguments and the C ABI of libfdma_hip.so for ordinary calls --
// checks, output and scratch allocation, argument blocks, autograd nodes.
//
// What bounds it: a small attention call takes 10 to 40 us on the device, and the same steps in Python (shape checks,
// a ctypes block, a Python autograd node and its backward) took 19 us without and 150 us with a backward; a forward
// call through this file takes 5 to 8 us, a forward and backward about 40, most of them the autograd engine's own.
//
// Every function returns NotImplemented for a call it was not made for -- tensor subclasses, dispatch or function
// modes, functorch wrappers, forward-mode duals, shapes that need padding or raise an error -- and the Python operator
// then takes its general path, so the semantics (and all messages) are stated in one place, there.
//
// The library's functions arrive as addresses (bind()): the library that Python has loaded is the one that is called.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/Exception.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/version.h>

#include <cstdio>
#include <list>
#include <utility>

#include "../../include/fdma.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

struct Api {
    decltype(&::fdma_fwd) fwd;
    decltype(&::fdma_bwd) bwd;
    decltype(&::fdma_fwd_workspace_bytes) fwd_workspace_bytes;
    decltype(&::fdma_fwd_takes_lists) fwd_takes_lists;
    decltype(&::fdma_fwd_optional_bytes) fwd_optional_bytes;
    decltype(&::fdma_bwd_workspace_bytes) bwd_workspace_bytes;
    decltype(&::fdma_bwd_optional_bytes) bwd_optional_bytes;
    decltype(&::fdma_fwd_counter_bytes) fwd_counter_bytes;
    decltype(&::fdma_set_stream_min_items) stream_min_items;
    decltype(&::fdma_varlen_fwd) varlen_fwd;
    decltype(&::fdma_varlen_bwd_ws) varlen_bwd_ws;
    decltype(&::fdma_varlen_bwd_optional_bytes) varlen_bwd_optional_bytes;
    decltype(&::fdma_create_mask) create_mask;
    decltype(&::fdma_dyn_bias_fwd) dyn_bias_fwd;
    decltype(&::fdma_dyn_bias_bwd) dyn_bias_bwd;
    decltype(&::fdma_dyn_bias_bwd_workspace_bytes) dyn_bias_bwd_workspace_bytes;
    decltype(&::fdma_last_error) last_error;
} api;

PyObject *s_kept = nullptr, *s_bits = nullptr;  // names of the attributes that the mask builder leaves on a mask

void check(int rc) { TORCH_CHECK(rc == FDMA_OK, api.last_error()); }

inline size_t up256(size_t x) { return (x + 255) / 256 * 256; }
inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Scratch of `need` bytes and, where the device has that much left, of `room` more, which the call can do without (then 0).
Tensor scratch_with_room(size_t need, size_t &room, const at::TensorOptions &opt) {
    if (room) {
        try {
            return at::empty({(int64_t)(need + room)}, opt.dtype(at::kByte));
        } catch (const c10::OutOfMemoryError &) {
            room = 0;
        }
    }
    return need ? at::empty({(int64_t)need}, opt.dtype(at::kByte)) : Tensor();
}

// ---- arguments -----------------------------------------------------------------------------------------------------

// Nothing but the device would see a call on plain tensors right now (torch.jit.trace would: it records operators).
bool plain_state() {
    return !at::tracer::impl::is_dispatch_enabled() && c10::impl::TorchDispatchModeTLS::stack_len() == 0 && at::impl::PythonTorchFunctionTLS::stack_len() == 0;
}

// An ordinary torch.Tensor on `dev` (any GPU while dev is negative): not a subclass, not wrapped by functorch or
// functionalisation, no forward-mode tangent.
bool plain_tensor(PyObject *o, int &dev) {
    if (Py_TYPE(o) != (PyTypeObject *)THPVariableClass) return false;
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda()) return false;
    const c10::DispatchKeySet ks = t.key_set();
    if (ks.has(c10::DispatchKey::FuncTorchBatched) || ks.has(c10::DispatchKey::FuncTorchGradWrapper) ||
        ks.has(c10::DispatchKey::Functionalize) || ks.has(c10::DispatchKey::Python))
        return false;
    if (dev < 0) dev = t.get_device();
    return t.get_device() == dev && !t._fw_grad(/*level=*/0).defined();
}

bool half_type(const Tensor &t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int dtype_code(const Tensor &t) { return t.scalar_type() == at::kBFloat16 ? FDMA_DTYPE_BF16 : FDMA_DTYPE_FP16; }

// The kernels' vector accesses: last dim contiguous, 16-byte aligned base, other strides multiples of `elems`.
bool vec_ok(const Tensor &t, int64_t elems) {
    const int64_t n = t.dim();
    if (t.stride(n - 1) != 1 || ((uintptr_t)t.data_ptr() & 15)) return false;
    for (int64_t i = 0; i + 1 < n; i++)
        if (t.size(i) != 1 && t.stride(i) % elems != 0) return false;
    return true;
}

void strides3(const Tensor &t, int64_t *s) { s[0] = t.stride(0); s[1] = t.stride(1); s[2] = t.stride(2); }
void bcast3(const Tensor &t, int64_t *s) {
    for (int i = 0; i < 3; i++) s[i] = t.size(i) == 1 ? 0 : t.stride(i);
}

void *stream_of(int dev) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// None: 0; otherwise whether the object is true, -1 (and no exception) where it has no truth value.
int truth(PyObject *o) {
    const int t = o == Py_None ? 0 : PyObject_IsTrue(o);
    if (t < 0) PyErr_Clear();
    return t;
}

bool same_shape(const Tensor &t, PyObject *tup) {
    if (!PyTuple_Check(tup) || PyTuple_GET_SIZE(tup) != t.dim()) return false;
    for (int64_t i = 0; i < t.dim(); i++)
        if (PyLong_AsLongLong(PyTuple_GET_ITEM(tup, i)) != t.size(i)) return false;
    return true;
}

// Attribute `name` of a plain tensor object's own dictionary, or nullptr (borrowed; no exception is raised for a missing one).
PyObject *instance_attr(PyObject *o, PyObject *name) {
    PyObject *dict = PyObject_GenericGetDict(o, nullptr);
    if (!dict) {
        PyErr_Clear();
        return nullptr;
    }
    PyObject *attr = PyDict_GetItem(dict, name);
    Py_DECREF(dict);  // (the object keeps it)
    return attr;
}

// (version, data pointer, shape) left at the end of a record by the mask builder still describe the tensor
bool record_valid(const Tensor &t, PyObject *rec, Py_ssize_t at) {
    return !t.is_inference() && PyLong_AsLongLong(PyTuple_GET_ITEM(rec, at)) == (long long)t._version() &&
           (uintptr_t)PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(rec, at + 1)) == (uintptr_t)t.data_ptr() &&
           same_shape(t, PyTuple_GET_ITEM(rec, at + 2));
}

struct SideInputs {  // the mask builder's second outputs (see utils/mask.py: kept_keys_of, mask_bits_of)
    Tensor idx, cnt, count, bits;
    int32_t ld = 0;
};

void side_inputs(PyObject *mask_obj, const Tensor &mask, int64_t seqlen_k, SideInputs &s) {
    if (PyObject *rec = instance_attr(mask_obj, s_kept))
        if (mask.size(3) == seqlen_k && PyTuple_Check(rec) && PyTuple_GET_SIZE(rec) == 7 && record_valid(mask, rec, 4)) {
            s.idx = THPVariable_Unpack(PyTuple_GET_ITEM(rec, 0));
            s.cnt = THPVariable_Unpack(PyTuple_GET_ITEM(rec, 1));
            s.count = THPVariable_Unpack(PyTuple_GET_ITEM(rec, 2));
            s.ld = (int32_t)PyLong_AsLong(PyTuple_GET_ITEM(rec, 3));
        }
    if (PyObject *rec = instance_attr(mask_obj, s_bits))
        if (PyTuple_Check(rec) && PyTuple_GET_SIZE(rec) == 4 && record_valid(mask, rec, 1))
            s.bits = THPVariable_Unpack(PyTuple_GET_ITEM(rec, 0));
}

// ---- attention -----------------------------------------------------------------------------------------------------

// Arrival counters of the one-launch decode: zero before and after every call, so calls on one stream share a buffer
// and calls on different streams, which may overlap, have one each.  At most kCounterStreams are kept; the one that has
// not been used for longest is given back to the allocator, which hands memory on in the order of the stream it served.
// Only touched with the interpreter lock held.
constexpr size_t kCounterStreams = 32;
struct Counters {
    int dev;
    void *stream;
    Tensor buf;
};
std::list<Counters> &counter_pool() {
    static auto *pool = new std::list<Counters>;  // (not destroyed at exit: the device may be gone by then)
    return *pool;
}
Tensor &counters_for(int dev, void *stream, size_t bytes, const at::TensorOptions &opt) {
    auto &pool = counter_pool();
    for (auto it = pool.begin(); it != pool.end(); ++it)
        if (it->dev == dev && it->stream == stream) {
            if (it->buf.nbytes() < bytes) it->buf = at::zeros({(int64_t)bytes}, opt);
            if (it != pool.begin()) pool.splice(pool.begin(), pool, it);
            return pool.front().buf;
        }
    if (pool.size() >= kCounterStreams) pool.pop_back();
    pool.push_front({dev, stream, at::zeros({(int64_t)(bytes > 4096 ? bytes : 4096)}, opt)});
    return pool.front().buf;
}

void fill_fwd(fdma_fwd_args &a, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &mask, const Tensor &bias,
              const Tensor &out, float *lse, double scale, bool causal, int compact_mode, const SideInputs &side) {
    a = fdma_fwd_args{};
    a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr();
    a.out = out.data_ptr();
    a.lse = lse;
    strides3(q, a.q_strides); strides3(k, a.k_strides); strides3(v, a.v_strides); strides3(out, a.o_strides);
    a.batch = (int32_t)q.size(0); a.seqlen_q = (int32_t)q.size(1); a.seqlen_k = (int32_t)k.size(1);
    a.num_heads = (int32_t)q.size(2); a.num_heads_k = (int32_t)k.size(2);
    a.num_heads_mask = a.num_heads_bias = 1;
    a.head_dim = (int32_t)q.size(3);
    a.dtype = dtype_code(q);
    a.is_causal = causal;
    a.softmax_scale = (float)scale;
    a.compact_mode = compact_mode;
    if (mask.defined()) {
        a.mask = mask.data_ptr();
        bcast3(mask, a.mask_strides);
        a.num_heads_mask = (int32_t)mask.size(1);
    }
    if (bias.defined()) {
        a.bias = bias.data_ptr();
        bcast3(bias, a.bias_strides);
        a.num_heads_bias = (int32_t)bias.size(1);
    }
    if (side.idx.defined()) {
        a.kept.idx = (const int32_t *)side.idx.data_ptr();
        a.kept.cnt = (const int32_t *)side.cnt.data_ptr();
        a.kept.count = (const int32_t *)side.count.data_ptr();
        a.kept.ld = side.ld;
    }
    if (side.bits.defined()) {
        a.mask_bits.bits = (const uint8_t *)side.bits.data_ptr();
        bcast3(side.bits, a.mask_bits.strides);
    }
}

Tensor aligned_grad(const Tensor &g) {  // what the caller's graph hands back may be an expanded or oddly sliced tensor
    return vec_ok(g, 8) ? g : g.clone(at::MemoryFormat::Contiguous);
}

struct AttentionBackward : public Node {
    SavedVariable q_, k_, v_, mask_, bias_, out_, lse_;
    Tensor ws;  // the forward's workspace (lists and compacted copies), which the backward reuses
    SideInputs side;
    size_t ws_off = 0, ws_bytes = 0;  // (ws_off: of the workspace in `ws` -- the LSE in front of it, unless it is saved as lse_)
    double scale = 1;
    bool causal = false, deterministic = false, has_mask = false, has_bias = false;
    int compact_mode = 0, stream_min = 0;

    std::string name() const override { return "FlashDMAttnFuncBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable *s : {&q_, &k_, &v_, &mask_, &bias_, &out_, &lse_}) s->reset_data();
        ws.reset();
        side = SideInputs{};
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor q = q_.unpack(), k = k_.unpack(), v = v_.unpack(), out = out_.unpack(shared_from_this()), lse = ws_off ? ws : lse_.unpack();
        const Tensor mask = has_mask ? mask_.unpack() : Tensor(), bias = has_bias ? bias_.unpack() : Tensor();
        if (!grads[0].defined()) return variable_list(has_bias ? 4 : 3);
        at::NoGradGuard no_grad;
        const Tensor dout = aligned_grad(grads[0]);
        const auto opt = q.options().requires_grad(false);
        // every element of the gradients is written by the kernels: no zero fill
        Tensor dq = at::empty(q.sizes(), opt), dk = at::empty(k.sizes(), opt), dv = at::empty(v.sizes(), opt), dbias;
        fdma_bwd_args a{};
        fill_fwd(a.f, q, k, v, mask, bias, out, (float *)lse.data_ptr(), scale, causal, compact_mode, side);
        a.dout = dout.data_ptr();
        a.dq = dq.data_ptr(); a.dk = dk.data_ptr(); a.dv = dv.data_ptr();
        strides3(dout, a.do_strides); strides3(dq, a.dq_strides); strides3(dk, a.dk_strides); strides3(dv, a.dv_strides);
        if (has_bias) {
            const int64_t n = bias.size(3), np = round_up(n, 8);  // rows of whole 16-byte vectors
            dbias = at::empty({bias.size(0), bias.size(1), bias.size(2), np}, opt);
            a.dbias = dbias.data_ptr();
            bcast3(dbias, a.dbias_strides);
            if (np != n) dbias = dbias.narrow(3, 0, n);
        }
        a.deterministic = deterministic;
        if (ws_bytes && stream_min == api.stream_min_items(0)) {
            a.fwd_workspace = (const char *)ws.data_ptr() + ws_off;
            a.fwd_workspace_bytes = ws_bytes;
        }
        const size_t d_bytes = up256((size_t)q.size(0) * q.size(2) * round_up(q.size(1), 128) * 4);
        const size_t need = api.bwd_workspace_bytes(&a);
        size_t room = api.bwd_optional_bytes(&a);
        Tensor scratch = scratch_with_room(d_bytes + need, room, opt);
        a.softmax_d = (float *)scratch.data_ptr();
        if (need + room) {
            a.workspace = (char *)scratch.data_ptr() + d_bytes;
            a.workspace_bytes = need + room;
        }
        check(api.bwd(&a, stream_of(q.get_device())));
        if (has_bias) return {std::move(dq), std::move(dk), std::move(dv), std::move(dbias)};
        return {std::move(dq), std::move(dk), std::move(dv)};
    }
};

// attention(q, k, v, mask, bias, softmax_scale, is_causal, softcap, deterministic, return_attn_probs, compact_mode)
PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 11, "attention() takes 11 arguments");
    int dev = -1;
    if (!plain_state()) Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 5; i++)
        if (!(i >= 3 && args[i] == Py_None) && !plain_tensor(args[i], dev)) Py_RETURN_NOTIMPLEMENTED;
    if (truth(args[7]) != 0 || truth(args[9]) != 0 || truth(args[6]) < 0 || truth(args[8]) < 0) Py_RETURN_NOTIMPLEMENTED;  // softcap, LSE wanted
    const Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
    const Tensor mask = args[3] == Py_None ? Tensor() : THPVariable_Unpack(args[3]);
    const Tensor bias = args[4] == Py_None ? Tensor() : THPVariable_Unpack(args[4]);
    // (what _inputs_plainly_ok checks; anything else is for the general path to accept or to name)
    if (!half_type(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || q.dim() != 4 || k.dim() != 4 ||
        v.sizes() != k.sizes())
        Py_RETURN_NOTIMPLEMENTED;
    const int64_t B = q.size(0), Lq = q.size(1), H = q.size(2), d = q.size(3), Lk = k.size(1), Hk = k.size(2);
    if (B < 1 || Lq < 1 || Lk < 1 || H < 1 || Hk < 1 || H % Hk != 0 || d < 8 || d > 256 || d % 8 != 0 || k.size(0) != B || k.size(3) != d)
        Py_RETURN_NOTIMPLEMENTED;
    if (!vec_ok(q, 8) || !vec_ok(k, 8) || !vec_ok(v, 8)) Py_RETURN_NOTIMPLEMENTED;
    const int compact_mode = (int)PyLong_AsLong(args[10]);
    for (const Tensor *t : {&mask, &bias}) {
        if (!t->defined()) continue;
        if (t->scalar_type() != (t == &mask ? at::kBool : q.scalar_type()) || t->dim() != 4 || (t->size(0) != B && t->size(0) != 1) ||
            (t->size(1) != 1 && t->size(1) != Hk && t->size(1) != H) || (t->size(2) != 1 && t->size(2) != Lq) ||
            (t == &mask ? t->size(3) < Lk : t->size(3) != Lk) || t->stride(3) != 1)
            Py_RETURN_NOTIMPLEMENTED;
    }
    // (rows are taken as they lie, unless they differ per query and are shorter than a chunk: fdma.h.  Such rows need strides
    // that a backward may not find again: a saved-tensor hook can hand the tensor back without them)
    const bool rows = Lq > 1 && Lk < 8 && ((mask.defined() && mask.size(2) != 1) || (bias.defined() && bias.size(2) != 1));
    if (rows && (at::GradMode::is_enabled() || (mask.defined() && !vec_ok(mask, 16)) || (bias.defined() && !vec_ok(bias, 8)))) Py_RETURN_NOTIMPLEMENTED;
    if (mask.defined()) {
        // a row per query head over grouped kv heads (its backward is taken apart), or rows that may turn out to be a
        // column mask under the policy "always": general path
        if (mask.size(1) == H && H != Hk) Py_RETURN_NOTIMPLEMENTED;
        if (mask.size(2) != 1 && compact_mode == FDMA_COMPACT_ALWAYS) Py_RETURN_NOTIMPLEMENTED;
    }
    const bool deterministic = truth(args[8]) > 0;
    if (deterministic && bias.defined() && ((bias.size(0) == 1 && B > 1) || (bias.size(1) == 1 && Hk > 1))) Py_RETURN_NOTIMPLEMENTED;
    const bool record = at::GradMode::is_enabled();
    const bool is_grad = record && (q.requires_grad() || k.requires_grad() || v.requires_grad());
    if (record && !is_grad && bias.defined() && bias.requires_grad()) Py_RETURN_NOTIMPLEMENTED;
    if (c10::hip::current_device() != dev) Py_RETURN_NOTIMPLEMENTED;
    double scale = 1.0 / std::sqrt((double)d);
    if (args[5] != Py_None) {
        scale = PyFloat_AsDouble(args[5]);
        if (scale == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            Py_RETURN_NOTIMPLEMENTED;
        }
    }
    const bool causal = truth(args[6]) > 0;
    SideInputs side;
    if (mask.defined()) side_inputs(args[3], mask, Lk, side);

    std::shared_ptr<AttentionBackward> node;
    if (is_grad) {
        node = std::shared_ptr<AttentionBackward>(new AttentionBackward(), torch::autograd::deleteNode);
        node->set_next_edges(bias.defined() ? torch::autograd::collect_next_edges(q, k, v, bias) : torch::autograd::collect_next_edges(q, k, v));
    }
    const auto opt = q.options().requires_grad(false), bytes = opt.dtype(at::kByte);
    Tensor out = at::empty(q.sizes(), opt);
    fdma_fwd_args a;
    fill_fwd(a, q, k, v, mask, bias, out, nullptr, scale, causal, compact_mode, side);
    // LSE and workspace in one piece -- except where a backward will want the LSE and there is no workspace to go with it, or
    // saved-tensor hooks are waiting (they may move it off the device until then): it is a tensor of its own there, which the
    // node saves as autograd does
    // (without a backward nobody else wants the compacted copies)
    const size_t need = !is_grad && side.idx.defined() && api.fwd_takes_lists(&a) ? 0 : api.fwd_workspace_bytes(&a);
    const bool apart = is_grad && (need == 0 || Lq == 1 || !at::SavedTensorDefaultHooks::get_tls_state().stack.empty());
    const size_t lse_bytes = apart ? 0 : up256((size_t)B * H * Lq * 4);
    Tensor lse, buf;
    if (apart) lse = at::empty({B, H, Lq}, opt.dtype(at::kFloat));
    if (lse_bytes + need) buf = at::empty({(int64_t)(lse_bytes + need)}, bytes);
    a.lse = (float *)(apart ? lse : buf).data_ptr();
    void *stream = stream_of(dev);
    if (need) {
        a.workspace = (char *)buf.data_ptr() + lse_bytes;
        a.workspace_bytes = need;
    }
    Tensor shares;  // (of the call alone: the node does not keep it)
    if (!need && ((mask.defined() && mask.size(2) > 1) || (bias.defined() && bias.size(2) > 1)))
        if (size_t room = api.fwd_optional_bytes(&a)) {
            shares = scratch_with_room(0, room, opt);
            if (room) { a.workspace = shares.data_ptr(); a.workspace_bytes = room; }
        }
    if (a.workspace)
        if (const size_t cbytes = api.fwd_counter_bytes(&a)) {
            Tensor &c = counters_for(dev, stream, cbytes, bytes);
            a.counters = (int32_t *)c.data_ptr();
            a.counters_bytes = c.nbytes();
        }
    check(api.fwd(&a, stream));
    if (is_grad) {
        torch::autograd::set_history(out, node);
        node->q_ = SavedVariable(q, false);
        node->k_ = SavedVariable(k, false);
        node->v_ = SavedVariable(v, false);
        if ((node->has_mask = mask.defined())) node->mask_ = SavedVariable(mask, false);
        if ((node->has_bias = bias.defined())) node->bias_ = SavedVariable(bias, false);
        node->out_ = SavedVariable(out, true);
        if (apart) node->lse_ = SavedVariable(lse, false);
        node->side = side;
        if (need && Lq > 1) { node->ws = buf; node->ws_off = lse_bytes; node->ws_bytes = need; }
        node->scale = scale; node->causal = causal; node->deterministic = deterministic;
        node->compact_mode = compact_mode;
        node->stream_min = api.stream_min_items(0);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- ragged batches ------------------------------------------------------------------------------------------------

void fill_varlen(fdma_varlen_fwd_args &a, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_q, const Tensor &cu_k,
                 const Tensor &out, float *lse, int64_t max_q, int64_t max_k, double scale, bool causal) {
    a = fdma_varlen_fwd_args{};
    a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr();
    a.out = out.data_ptr();
    a.lse = lse;
    a.cu_seqlens_q = (const int32_t *)cu_q.data_ptr(); a.cu_seqlens_k = (const int32_t *)cu_k.data_ptr();
    const Tensor *src[4] = {&q, &k, &v, &out};
    int64_t *dst[4] = {a.q_strides, a.k_strides, a.v_strides, a.o_strides};
    for (int i = 0; i < 4; i++) { dst[i][0] = src[i]->stride(0); dst[i][1] = src[i]->stride(1); }
    a.batch = (int32_t)cu_q.numel() - 1;
    a.total_q = (int32_t)q.size(0); a.total_k = (int32_t)k.size(0);
    a.max_seqlen_q = (int32_t)max_q; a.max_seqlen_k = (int32_t)max_k;
    a.num_heads = (int32_t)q.size(1); a.num_heads_k = (int32_t)k.size(1); a.head_dim = (int32_t)q.size(2);
    a.dtype = dtype_code(q);
    a.is_causal = causal;
    a.softmax_scale = (float)scale;
}

struct VarlenBackward : public Node {
    SavedVariable q_, k_, v_, out_, cu_q_, cu_k_, lse_;
    int64_t max_q = 0, max_k = 0;
    double scale = 1;
    bool causal = false, deterministic = false;

    std::string name() const override { return "FlashAttnVarlenFuncBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable *s : {&q_, &k_, &v_, &out_, &cu_q_, &cu_k_, &lse_}) s->reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor q = q_.unpack(), k = k_.unpack(), v = v_.unpack(), out = out_.unpack(shared_from_this());
        const Tensor cu_q = cu_q_.unpack(), cu_k = cu_k_.unpack(), lse = lse_.unpack();
        if (!grads[0].defined()) return variable_list(3);
        at::NoGradGuard no_grad;
        const Tensor dout = aligned_grad(grads[0]);
        const auto opt = q.options().requires_grad(false);
        Tensor dq = at::empty(q.sizes(), opt), dk = at::empty(k.sizes(), opt), dv = at::empty(v.sizes(), opt);
        Tensor softmax_d = at::empty({q.size(1), q.size(0)}, opt.dtype(at::kFloat));
        fdma_varlen_bwd_args a{};
        fill_varlen(a.f, q, k, v, cu_q, cu_k, out, (float *)lse.data_ptr(), max_q, max_k, scale, causal);
        a.dout = dout.data_ptr();
        a.dq = dq.data_ptr(); a.dk = dk.data_ptr(); a.dv = dv.data_ptr();
        const Tensor *src[4] = {&dout, &dq, &dk, &dv};
        int64_t *dst[4] = {a.do_strides, a.dq_strides, a.dk_strides, a.dv_strides};
        for (int i = 0; i < 4; i++) { dst[i][0] = src[i]->stride(0); dst[i][1] = src[i]->stride(1); }
        a.softmax_d = (float *)softmax_d.data_ptr();
        a.deterministic = deterministic;
        size_t room = api.varlen_bwd_optional_bytes(&a);
        const Tensor scratch = scratch_with_room(0, room, opt);
        check(api.varlen_bwd_ws(&a, room ? scratch.data_ptr() : nullptr, room, stream_of(q.get_device())));
        return {std::move(dq), std::move(dk), std::move(dv)};
    }
};

// varlen_attention(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, softmax_scale, is_causal, softcap,
//                  deterministic, return_attn_probs, block_table)
PyObject *varlen_attention(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 13, "varlen_attention() takes 13 arguments");
    int dev = -1;
    if (!plain_state()) Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 5; i++)
        if (!plain_tensor(args[i], dev)) Py_RETURN_NOTIMPLEMENTED;
    if (truth(args[9]) != 0 || truth(args[11]) != 0 || args[12] != Py_None || truth(args[8]) < 0 || truth(args[10]) < 0) Py_RETURN_NOTIMPLEMENTED;
    const Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
    const Tensor &cu_q = THPVariable_Unpack(args[3]), &cu_k = THPVariable_Unpack(args[4]);
    if (!half_type(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || q.dim() != 3 || k.dim() != 3 ||
        v.sizes() != k.sizes() || cu_q.scalar_type() != at::kInt || cu_k.scalar_type() != at::kInt || !cu_q.is_contiguous() ||
        !cu_k.is_contiguous() || cu_q.numel() < 2 || cu_k.numel() != cu_q.numel())
        Py_RETURN_NOTIMPLEMENTED;
    const int64_t H = q.size(1), Hk = k.size(1), d = q.size(2);
    if (q.size(0) < 1 || k.size(0) < 1 || H < 1 || Hk < 1 || H % Hk != 0 || d < 8 || d > 256 || d % 8 != 0 || k.size(2) != d ||
        !vec_ok(q, 8) || !vec_ok(k, 8) || !vec_ok(v, 8) || !PyLong_Check(args[5]) || !PyLong_Check(args[6]))
        Py_RETURN_NOTIMPLEMENTED;
    const int64_t max_q = PyLong_AsLongLong(args[5]), max_k = PyLong_AsLongLong(args[6]);
    if (max_q < 1 || max_k < 1 || max_q > INT32_MAX || max_k > INT32_MAX || c10::hip::current_device() != dev) Py_RETURN_NOTIMPLEMENTED;
    double scale = 1.0 / std::sqrt((double)d);
    if (args[7] != Py_None) {
        scale = PyFloat_AsDouble(args[7]);
        if (scale == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            Py_RETURN_NOTIMPLEMENTED;
        }
    }
    const bool causal = truth(args[8]) > 0;
    const bool is_grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
    std::shared_ptr<VarlenBackward> node;
    if (is_grad) {
        node = std::shared_ptr<VarlenBackward>(new VarlenBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
    }
    const auto opt = q.options().requires_grad(false);
    Tensor out = at::empty(q.sizes(), opt);
    Tensor lse = at::empty({H, q.size(0)}, opt.dtype(at::kFloat));
    fdma_varlen_fwd_args a;
    fill_varlen(a, q, k, v, cu_q, cu_k, out, (float *)lse.data_ptr(), max_q, max_k, scale, causal);
    check(api.varlen_fwd(&a, stream_of(dev)));
    if (is_grad) {
        torch::autograd::set_history(out, node);
        node->q_ = SavedVariable(q, false);
        node->k_ = SavedVariable(k, false);
        node->v_ = SavedVariable(v, false);
        node->cu_q_ = SavedVariable(cu_q, false);
        node->cu_k_ = SavedVariable(cu_k, false);
        node->out_ = SavedVariable(out, true);
        node->lse_ = SavedVariable(lse, false);
        node->max_q = max_q; node->max_k = max_k;
        node->scale = scale; node->causal = causal; node->deterministic = truth(args[10]) > 0;
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- bias producer -------------------------------------------------------------------------------------------------

struct DynBiasBackward : public Node {
    SavedVariable v_, w_, a_, pb_, dt_;
    bool has_pb = false;

    std::string name() const override { return "DynamicMaskBiasBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable *s : {&v_, &w_, &a_, &pb_, &dt_}) s->reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor v = v_.unpack(), w = w_.unpack(), av = a_.unpack(), pb = has_pb ? pb_.unpack() : Tensor(), dt = dt_.unpack();
        const size_t n_in = has_pb ? 4 : 3;
        if (!grads[0].defined()) return variable_list(n_in);
        at::NoGradGuard no_grad;
        const Tensor g = grads[0].stride(3) == 1 ? grads[0] : grads[0].contiguous();
        const auto opt = v.options().requires_grad(false);
        Tensor dv = at::empty(v.sizes(), opt), dw = at::empty(w.sizes(), opt), da = at::empty(av.sizes(), opt), dpb;
        if (has_pb) dpb = at::empty(pb.sizes(), opt);
        fdma_dyn_bias_args a{};
        a.value = v.data_ptr(); a.weight = w.data_ptr(); a.a = av.data_ptr();
        a.proj_bias = has_pb ? pb.data_ptr() : nullptr;
        a.dt = (float *)dt.data_ptr();
        a.bias = dt.data_ptr();  // (not used by the backward; any device pointer)
        strides3(v, a.value_strides);
        a.batch = (int32_t)v.size(0); a.seqlen_k = (int32_t)v.size(1); a.num_heads_k = (int32_t)v.size(2); a.head_dim = (int32_t)v.size(3);
        a.dtype = dtype_code(v);
        a.dbias = g.data_ptr();
        a.dbias_strides[0] = g.stride(0); a.dbias_strides[1] = g.stride(1);
        a.dvalue = dv.data_ptr();
        strides3(dv, a.dvalue_strides);
        a.dweight = dw.data_ptr(); a.da = da.data_ptr();
        a.dproj_bias = has_pb ? dpb.data_ptr() : nullptr;
        const size_t need = api.dyn_bias_bwd_workspace_bytes(&a);
        Tensor ws = at::empty({(int64_t)(need ? need : 1)}, opt.dtype(at::kByte));
        a.workspace = ws.data_ptr();
        a.workspace_bytes = need;
        check(api.dyn_bias_bwd(&a, stream_of(v.get_device())));
        if (has_pb) return {std::move(dv), std::move(dw), std::move(da), std::move(dpb)};
        return {std::move(dv), std::move(dw), std::move(da)};
    }
};

// dyn_bias(value_states, weight, a, proj_bias)
PyObject *dyn_bias(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 4, "dyn_bias() takes 4 arguments");
    int dev = -1;
    if (!plain_state()) Py_RETURN_NOTIMPLEMENTED;
    const bool has_pb = args[3] != Py_None;
    for (int i = 0; i < (has_pb ? 4 : 3); i++) {
        // (parameters of a module are what this function is called with)
        if (Py_TYPE(args[i]) != (PyTypeObject *)THPVariableClass && Py_TYPE(args[i]) != (PyTypeObject *)ParameterClass) Py_RETURN_NOTIMPLEMENTED;
        if (Py_TYPE(args[i]) == (PyTypeObject *)THPVariableClass && !plain_tensor(args[i], dev)) Py_RETURN_NOTIMPLEMENTED;
    }
    const Tensor &v = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &av = THPVariable_Unpack(args[2]);
    const Tensor pb = has_pb ? THPVariable_Unpack(args[3]) : Tensor();
    if (!v.is_cuda() || !half_type(v) || v.dim() != 4 || v.get_device() != c10::hip::current_device()) Py_RETURN_NOTIMPLEMENTED;
    const int64_t b = v.size(0), l = v.size(1), hk = v.size(2), d = v.size(3);
    if (b < 1 || l < 1 || hk < 1 || hk > 32 || d % 8 != 0 || (hk * d) % 16 != 0 || !vec_ok(v, 8)) Py_RETURN_NOTIMPLEMENTED;
    for (const Tensor *t : {&w, &av, &pb})
        if (t->defined() && (t->scalar_type() != v.scalar_type() || t->device() != v.device() || !t->is_contiguous() || t->is_meta() ||
                             t->_fw_grad(0).defined() || ((uintptr_t)t->data_ptr() & (t == &w ? 15 : 1))))
            Py_RETURN_NOTIMPLEMENTED;
    if (w.dim() != 2 || w.size(0) != hk || w.size(1) != hk * d || av.numel() != hk || (has_pb && pb.numel() != hk)) Py_RETURN_NOTIMPLEMENTED;
    const bool is_grad = at::GradMode::is_enabled() && (v.requires_grad() || w.requires_grad() || av.requires_grad() || (has_pb && pb.requires_grad()));
    std::shared_ptr<DynBiasBackward> node;
    if (is_grad) {
        node = std::shared_ptr<DynBiasBackward>(new DynBiasBackward(), torch::autograd::deleteNode);
        node->set_next_edges(has_pb ? torch::autograd::collect_next_edges(v, w, av, pb) : torch::autograd::collect_next_edges(v, w, av));
    }
    const auto opt = v.options().requires_grad(false);
    // rows of the bias are handed to the attention kernels' 16-byte loads: a row pitch of whole vectors
    const int64_t lp = round_up(l, 8);
    Tensor bias = at::empty_strided({b, hk, 1, l}, {hk * lp, lp, lp, 1}, opt);
    Tensor dt;  // (read by the backward only)
    if (is_grad) dt = at::empty({b * l, hk}, opt.dtype(at::kFloat));
    fdma_dyn_bias_args a{};
    a.value = v.data_ptr(); a.weight = w.data_ptr(); a.a = av.data_ptr();
    a.proj_bias = has_pb ? pb.data_ptr() : nullptr;
    a.bias = bias.data_ptr();
    a.dt = is_grad ? (float *)dt.data_ptr() : nullptr;
    strides3(v, a.value_strides);
    a.bias_strides[0] = hk * lp; a.bias_strides[1] = lp;
    a.batch = (int32_t)b; a.seqlen_k = (int32_t)l; a.num_heads_k = (int32_t)hk; a.head_dim = (int32_t)d;
    a.dtype = dtype_code(v);
    check(api.dyn_bias_fwd(&a, stream_of(v.get_device())));
    if (is_grad) {
        torch::autograd::set_history(bias, node);
        node->v_ = SavedVariable(v, false);
        node->w_ = SavedVariable(w, false);
        node->a_ = SavedVariable(av, false);
        if ((node->has_pb = has_pb)) node->pb_ = SavedVariable(pb, false);
        node->dt_ = SavedVariable(dt, false);
    }
    return THPVariable_Wrap(std::move(bias));
    END_HANDLE_TH_ERRORS
}

// ---- keep-mask builder ---------------------------------------------------------------------------------------------

// create_mask(bias, mask_in, window, min_value, block_size, type)
PyObject *create_mask(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(nargs == 6, "create_mask() takes 6 arguments");
    int dev = -1;
    if (!plain_state() || !plain_tensor(args[0], dev) || (args[1] != Py_None && !plain_tensor(args[1], dev))) Py_RETURN_NOTIMPLEMENTED;
    const Tensor &bias = THPVariable_Unpack(args[0]);
    const Tensor in = args[1] == Py_None ? Tensor() : THPVariable_Unpack(args[1]);
    if (bias.dim() != 4 || !half_type(bias) || bias.numel() == 0 || (bias.size(3) > 1 && bias.stride(3) != 1) || c10::hip::current_device() != dev)
        Py_RETURN_NOTIMPLEMENTED;
    const int64_t L = bias.size(3);
    fdma_mask_args a{};
    if (in.defined()) {
        if (in.dim() != 4 || in.scalar_type() != at::kBool || in.size(3) != L || (L > 1 && in.stride(3) != 1)) Py_RETURN_NOTIMPLEMENTED;
        for (int i = 0; i < 3; i++)
            if (in.size(i) != 1 && in.size(i) != bias.size(i)) Py_RETURN_NOTIMPLEMENTED;
        a.mask_in = in.data_ptr();
        bcast3(in, a.mask_in_strides);
    }
    const long type = PyLong_AsLong(args[5]);
    const long long window = type == FDMA_MASK_TOPK ? PyLong_AsLongLong(args[2]) : 0;
    const long long block = args[4] == Py_None ? 0 : PyLong_AsLongLong(args[4]);
    const double min_value = PyFloat_AsDouble(args[3]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NOTIMPLEMENTED;
    }
    if (window < 0 || window > L || block > INT32_MAX) Py_RETURN_NOTIMPLEMENTED;
    const auto opt = bias.options().requires_grad(false);
    Tensor out = at::empty(bias.sizes(), opt.dtype(at::kBool));
    a.bias = bias.data_ptr();
    a.mask_out = out.data_ptr();
    strides3(bias, a.bias_strides);
    strides3(out, a.mask_out_strides);
    a.batch = (int32_t)bias.size(0); a.heads = (int32_t)bias.size(1); a.rows = (int32_t)bias.size(2); a.seqlen_k = (int32_t)L;
    a.window = (int32_t)window;
    a.block_size = block > 1 ? (int32_t)block : 0;
    a.type = (int32_t)type;
    a.dtype = dtype_code(bias);
    a.min_value = (float)min_value;
    // the second outputs (see utils/mask.py): lists of the kept columns for a mask that is broadcast over the queries,
    // bit rows for one that is not
    Tensor idx, cnt, count, bits;
    if (bias.size(2) == 1) {
        const int64_t ld = round_up(L, 16), rows = bias.size(0) * bias.size(1);
        idx = at::empty({rows, ld}, opt.dtype(at::kInt));
        cnt = at::empty({rows, ld}, opt.dtype(at::kInt));
        count = at::empty({rows}, opt.dtype(at::kInt));
        a.kept_idx = (int32_t *)idx.data_ptr(); a.kept_cnt = (int32_t *)cnt.data_ptr(); a.kept_count = (int32_t *)count.data_ptr();
        a.kept_ld = (int32_t)ld;
    } else {
        a.bits_row_bytes = round_up((L + 7) / 8, 16);
        bits = at::empty({bias.size(0), bias.size(1), bias.size(2), a.bits_row_bytes}, opt.dtype(at::kByte));
        a.bits = (uint8_t *)bits.data_ptr();
    }
    check(api.create_mask(&a, stream_of(dev)));
    const bool inference = out.is_inference();
    const long long version = inference ? 0 : (long long)out._version();
    const auto ptr = (unsigned long long)(uintptr_t)out.data_ptr();
    const int64_t s0 = out.size(0), s1 = out.size(1), s2 = out.size(2);
    PyObject *res = THPVariable_Wrap(std::move(out));
    if (!res || inference) return res;  // (tensors without a version counter carry no record)
    PyObject *rec = idx.defined()
        ? Py_BuildValue("(NNNiLK(LLLL))", THPVariable_Wrap(idx), THPVariable_Wrap(cnt), THPVariable_Wrap(count), (int)a.kept_ld, version, ptr,
                        (long long)s0, (long long)s1, (long long)s2, (long long)L)
        : Py_BuildValue("(NLK(LLLL))", THPVariable_Wrap(bits), version, ptr, (long long)s0, (long long)s1, (long long)s2, (long long)L);
    if (!rec || PyObject_SetAttr(res, idx.defined() ? s_kept : s_bits, rec) < 0) {
        Py_XDECREF(rec);
        Py_DECREF(res);
        return nullptr;
    }
    Py_DECREF(rec);
    return res;
    END_HANDLE_TH_ERRORS
}

// ---- module --------------------------------------------------------------------------------------------------------

// bind({name: address, ...}): the functions of the library that Python has loaded
PyObject *bind(PyObject *, PyObject *dict) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(PyDict_Check(dict), "bind() takes a dict");
    auto get = [&](const char *name) -> void * {
        PyObject *o = PyDict_GetItemString(dict, name);
        TORCH_CHECK(o, "bind(): no ", name);
        return PyLong_AsVoidPtr(o);
    };
#define FDMA_BIND(f) api.f = (decltype(api.f))get("fdma_" #f)
    FDMA_BIND(fwd);
    FDMA_BIND(bwd);
    FDMA_BIND(fwd_workspace_bytes);
    FDMA_BIND(fwd_takes_lists);
    FDMA_BIND(fwd_optional_bytes);
    FDMA_BIND(bwd_workspace_bytes);
    FDMA_BIND(bwd_optional_bytes);
    FDMA_BIND(fwd_counter_bytes);
    FDMA_BIND(varlen_fwd);
    FDMA_BIND(varlen_bwd_ws);
    FDMA_BIND(varlen_bwd_optional_bytes);
    FDMA_BIND(create_mask);
    FDMA_BIND(dyn_bias_fwd);
    FDMA_BIND(dyn_bias_bwd);
    FDMA_BIND(dyn_bias_bwd_workspace_bytes);
    FDMA_BIND(last_error);
#undef FDMA_BIND
    api.stream_min_items = (decltype(api.stream_min_items))get("fdma_set_stream_min_items");
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"attention", (PyCFunction)(void (*)(void))attention, METH_FASTCALL, nullptr},
    {"varlen_attention", (PyCFunction)(void (*)(void))varlen_attention, METH_FASTCALL, nullptr},
    {"dyn_bias", (PyCFunction)(void (*)(void))dyn_bias, METH_FASTCALL, nullptr},
    {"create_mask", (PyCFunction)(void (*)(void))create_mask, METH_FASTCALL, nullptr},
    {"bind", bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fdma_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fdma_torch(void) {
    s_kept = PyUnicode_InternFromString("_fdma_kept");
    s_bits = PyUnicode_InternFromString("_fdma_bits");
    PyObject *mod = PyModule_Create(&module_def);
    // what this file is tied to (major and minor version of Python); whoever loads it compares
    char python[16];
    snprintf(python, sizeof(python), "%d.%d", PY_MAJOR_VERSION, PY_MINOR_VERSION);
    PyObject *built_for = mod ? Py_BuildValue("(ss)", TORCH_VERSION, python) : nullptr;
    if (!built_for || PyModule_AddObject(mod, "built_for", built_for) < 0) {
        Py_XDECREF(built_for);
        Py_XDECREF(mod);
        return nullptr;
    }
    return mod;
}
