// Host path of the attention functions in native code: flash_attn._host.
//
// Short calls wait for the host.  The Python layer (flash_attn/_native.py and the autograd functions of
// flash_attn/flash_attn_interface.py) takes 14 us for a forward, 20 us for a decoding step and 86-190 us (by the machine) for a
// training step, of which the GPU works 7-11, 11-14 and 30-90 us at the smallest sizes; the same calls from here take half of it
// (figures in flash_attn_interface._apply).  Each function takes the arguments of its Python counterpart, and either does the whole
// call or returns None before it has done anything, in which case the Python layer does it: whatever is not an ordinary call --
// tensor subclasses, functorch, modes, tracing, hooks on saved tensors, padded head dims, other strides, empty tensors, anything
// that an argument check would refuse -- is left to it, and so are its error messages.  What is done here is done as there: the
// same library calls with the same parameters, the same tensors allocated, the words of _native._counters; only the node of autograd
// is another one, of C++, whose saved tensors Python does not see.
#include <Python.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/anomaly_mode.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "fa_mi355x.h"

namespace {

using at::Tensor;

// libfa_mi355x.so, as _native.py has loaded it
struct Library {
    int (*fwd_rng)(const fa_fwd_params*, uint64_t, uint64_t, void*) = nullptr;
    int (*varlen_fwd_rng)(const fa_fwd_params*, uint64_t, uint64_t, void*) = nullptr;
    int (*fwd_kvcache)(const fa_fwd_params*, void*) = nullptr;
    int (*plan_splits)(const fa_fwd_params*, int32_t, int32_t*) = nullptr;
    int64_t (*work_list_words)(const fa_fwd_params*) = nullptr;
    const char* (*last_error)() = nullptr;
    int64_t (*bwd_lend_bytes)(const fa_bwd_params*, int64_t, int64_t) = nullptr;
    int (*bwd_lent)(const fa_bwd_params*, int64_t, int64_t, void*, int64_t, void*) = nullptr;
    int (*rotary)(const fa_rotary_params*, void*) = nullptr;
};
Library lib;
PyObject* native_dict = nullptr;                     // _native.__dict__
PyObject *name_counters, *name_words, *name_list, *name_reset;    // interned keys of it

// The functions of the Python layer that are not called from here: where a program has put its own in their place, it is asked.
struct StoodIn { PyObject *dict, *name, *function; };
std::vector<StoodIn> stood_in;
bool as_bound() {
    for (const auto& f : stood_in)
        if (PyDict_GetItem(f.dict, f.name) != f.function) return false;
    return true;
}

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// Nothing that takes part in tensor operations is active on this thread.
bool plain_thread() {
    using c10::DispatchKey;
    static const c10::DispatchKeySet special({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::PythonDispatcher, DispatchKey::PreDispatch,
                                              DispatchKey::Functionalize, DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                              DispatchKey::FuncTorchVmapMode, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::VmapMode,
                                              DispatchKey::Batched, DispatchKey::Tracer});
    if (c10::impl::tls_local_dispatch_key_set().included_.has_any(special)) return false;
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0;
}
// An autograd node may be one of C++: nobody packs what it saves or asks where it was made.
bool plain_autograd() { return !at::SavedTensorDefaultHooks::get_hooks().has_value() && !torch::autograd::AnomalyMode::is_enabled(); }

// An ordinary tensor on the GPU: torch.Tensor or Parameter itself, strided, no wrapper of a transform.
const Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet allowed({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || (t.key_set().raw_repr() & ~allowed.raw_repr()) != 0) return nullptr;
    return &t;
}
// The same for q, k, v: 16 bits, rows of whole 16-byte pieces.
const Tensor* plain16(PyObject* o, int64_t dim) {
    const Tensor* t = plain(o);
    if (!t || t->dim() != dim || (t->scalar_type() != at::kHalf && t->scalar_type() != at::kBFloat16)) return nullptr;
    const int64_t d = t->size(dim - 1);
    return t->numel() > 0 && t->stride(dim - 1) == 1 && d % 8 == 0 && d <= 256 ? t : nullptr;
}
bool like(const Tensor& a, const Tensor& b) { return a.scalar_type() == b.scalar_type() && a.device() == b.device(); }
// int32 words on q's device, one after the other
const Tensor* words32(PyObject* o, const Tensor& q, int64_t n) {
    const Tensor* t = plain(o);
    return t && t->scalar_type() == at::kInt && t->device() == q.device() && t->dim() == 1 && t->is_contiguous() && (n < 0 || t->size(0) == n) ? t : nullptr;
}
bool number(PyObject* o, double& x) {
    if (PyFloat_CheckExact(o)) { x = PyFloat_AS_DOUBLE(o); return true; }
    if (!PyLong_CheckExact(o)) return false;
    x = PyLong_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}
bool integer(PyObject* o, int32_t& x) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || v < INT32_MIN || v > INT32_MAX) return false;
    x = (int32_t)v;
    return true;
}
bool boolean(PyObject* o, bool& x) {
    if (o != Py_True && o != Py_False) return false;
    x = o == Py_True;
    return true;
}
bool pair(PyObject* o, int32_t& a, int32_t& b) {
    return PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == 2 && integer(PyTuple_GET_ITEM(o, 0), a) && integer(PyTuple_GET_ITEM(o, 1), b);
}

// What a call says beside its tensors.
struct Options {
    double dropout = 0, scale = 0;
    bool causal = false;
    int32_t left = -1, right = -1;
    int32_t max_q = 0, max_k = 0;        // packed calls
    Tensor cu_q, cu_k;
    // filled in before the launch
    int32_t* counter = nullptr;
    int32_t counter_len = 0;
};
bool parse(PyObject* const* a, int64_t d, Options& o) {      // dropout_p, softmax_scale, causal, window_size, return_softmax
    if (!number(a[0], o.dropout) || !(o.dropout >= 0.0 && o.dropout < 1.0)) return false;
    if (a[1] == Py_None) o.scale = std::pow((double)d, -0.5);
    else if (!number(a[1], o.scale)) return false;
    bool ret;
    return boolean(a[2], o.causal) && pair(a[3], o.left, o.right) && boolean(a[4], ret) && !ret;
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
// the tensor's own device: another one may be the current one
bool capturing(const Tensor& t) {
    const c10::DeviceGuard guard(t.device());
    return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

// _native._counters(device, words): its dictionary where that has the words, else the function.  Holds the GIL.
// The words live in that dictionary; `keep` holds those that it does not.
int32_t* counters(PyObject* q_obj, const Tensor& q, int64_t words, at::Tensor& keep) {
    PyObject* dict = PyDict_GetItem(native_dict, name_counters);
    if (dict && PyDict_CheckExact(dict) && (words <= FA_WORK_COUNTER_WORDS || !capturing(q))) {
        PyObject* key = Py_BuildValue("(iL)", (int)q.device().index(), (long long)(intptr_t)stream_of(q));
        if (!key) { PyErr_Clear(); return nullptr; }
        PyObject* t = PyDict_GetItem(dict, key);
        Py_DECREF(key);
        if (t && THPVariable_Check(t) && THPVariable_Unpack(t).numel() >= words) {
            keep = THPVariable_Unpack(t);
            return keep.data_ptr<int32_t>();
        }
    }
    const c10::DeviceGuard guard(q.device());
    PyObject* fn = PyDict_GetItem(native_dict, name_words);
    PyObject* device = PyObject_GetAttrString(q_obj, "device");
    PyObject* t = fn && device ? PyObject_CallFunction(fn, "OL", device, (long long)words) : nullptr;
    Py_XDECREF(device);
    if (!t) throw python_error();
    keep = THPVariable_Unpack(t);
    Py_DECREF(t);
    return keep.data_ptr<int32_t>();
}
bool use_list() { return PyDict_GetItem(native_dict, name_list) == Py_True; }

// (batch, row, head) strides of a (b, s, h, d) tensor, (0, row, head) of a packed (total, h, d) one
void strides(const Tensor& t, int64_t& b, int64_t& r, int64_t& h) {
    const auto st = t.strides();
    const size_t n = st.size();
    b = n == 4 ? st[0] : 0; r = st[n - 3]; h = st[n - 2];
}
int32_t dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? FA_DTYPE_BF16 : FA_DTYPE_FP16; }

// q, k, v and the sizes that they and the options give; out and softmax_lse are not there yet.
fa_fwd_params forward_params(const Tensor& q, const Tensor& k, const Tensor& v, const Options& o) {
    fa_fwd_params p;
    std::memset(&p, 0, sizeof p);
    p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr();
    // (checked before they are set: any place that an output could be)
    p.o = const_cast<void*>(p.q);
    p.softmax_lse = reinterpret_cast<float*>(p.o);
    strides(q, p.q_batch_stride, p.q_row_stride, p.q_head_stride);
    strides(k, p.k_batch_stride, p.k_row_stride, p.k_head_stride);
    strides(v, p.v_batch_stride, p.v_row_stride, p.v_head_stride);
    const int64_t n = q.dim();
    p.h = (int32_t)q.size(n - 2); p.h_k = (int32_t)k.size(n - 2); p.d = (int32_t)q.size(n - 1);
    const bool packed = o.cu_q.defined();
    if (packed) {
        p.cu_seqlens_q = o.cu_q.data_ptr<int32_t>(); p.cu_seqlens_k = o.cu_k.data_ptr<int32_t>();
        p.b = (int32_t)o.cu_q.size(0) - 1; p.seqlen_q = o.max_q; p.seqlen_k = o.max_k;
        p.num_splits = 1;
    } else {
        p.b = (int32_t)q.size(0); p.seqlen_q = (int32_t)q.size(1); p.seqlen_k = (int32_t)k.size(1);
    }
    p.is_causal = o.causal && (packed || p.seqlen_q != 1);
    p.window_left = o.left;
    p.window_right = p.is_causal ? 0 : o.right;
    p.is_seqlens_k_cumulative = 1;
    p.dtype = dtype_code(q);
    p.softmax_scale = (float)o.scale;
    return p;
}

Tensor new_like(const Tensor& q) { return at::empty_like(q.requires_grad() ? q.detach() : q); }
Tensor new_floats(const Tensor& q, at::IntArrayRef sizes) { return at::empty(sizes, q.options().dtype(at::kFloat).requires_grad(false)); }

// A call of the library that returned an error, without the GIL: raises its message, for a forward launch after _native._reset_counters.
[[noreturn]] void library_error(int rc, const Tensor* launched) {
    std::string message = lib.last_error();
    if (message.empty()) message = "libfa_mi355x: error " + std::to_string(rc);
    if (launched) {
        const PyGILState_STATE state = PyGILState_Ensure();
        PyObject* const fn = PyDict_GetItem(native_dict, name_reset);
        PyObject* const device = THPDevice_New(launched->device());
        PyObject* const done = fn && device ? PyObject_CallFunctionObjArgs(fn, device, nullptr) : nullptr;
        if (!done) PyErr_Clear();
        Py_XDECREF(done);
        Py_XDECREF(device);
        PyGILState_Release(state);
    }
    throw std::runtime_error(message);
}

struct Result { Tensor out, lse, rng; };

// Allocates and launches; without the GIL.
Result run_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Options& o) {
    const c10::DeviceGuard guard(q.device());
    fa_fwd_params p = forward_params(q, k, v, o);
    p.work_counter = o.counter;
    p.work_counter_len = o.counter_len;
    Result r;
    r.out = new_like(q);
    r.lse = new_floats(q, {p.b, p.h, p.seqlen_q});
    p.o = r.out.data_ptr();
    p.softmax_lse = r.lse.data_ptr<float>();
    strides(r.out, p.o_batch_stride, p.o_row_stride, p.o_head_stride);
    void* const stream = stream_of(q);
    uint64_t seed = 0, offset = 0;
    if (o.dropout > 0.0) {
        r.rng = at::empty({2}, q.options().dtype(at::kLong).requires_grad(false));
        at::Generator gen = at::globalContext().defaultGenerator(q.device());
        {
            std::lock_guard<std::mutex> lock(gen.mutex());
            seed = gen.current_seed();
            offset = gen.get_offset();
            gen.set_offset(offset + (uint64_t)p.b * p.h * 32);
        }
        p.p_dropout = (float)o.dropout;
        p.rng_state = reinterpret_cast<uint64_t*>(r.rng.data_ptr<int64_t>());
    }
    Tensor accum;
    const bool packed = o.cu_q.defined();
    if (!packed) {
        int32_t n = 0;
        if (const int rc = lib.plan_splits(&p, 0, &n)) library_error(rc, nullptr);
        if (n > 1) {
            const int64_t rows = (int64_t)n * p.b * p.h * p.seqlen_q, width = (p.d + 31) / 32 * 32;
            accum = new_floats(q, {rows * (width + 1)});
            p.o_accum = accum.data_ptr<float>();
            p.lse_accum = p.o_accum + rows * width;
        }
    }
    const int rc = packed ? lib.varlen_fwd_rng(&p, seed, offset, stream) : lib.fwd_rng(&p, seed, offset, stream);
    if (rc != 0) library_error(rc, &q);
    return r;
}

// The counter words of a forward call; holds the GIL.
void lend_words(PyObject* q_obj, const Tensor& q, const Tensor& k, const Tensor& v, Options& o, Tensor& keep) {
    int64_t words = FA_WORK_COUNTER_WORDS;
    if (o.cu_q.defined() && use_list()) {
        fa_fwd_params p = forward_params(q, k, v, o);
        words = lib.work_list_words(&p);
    }
    o.counter = counters(q_obj, q, words, keep);
    o.counter_len = (int32_t)words;
}

// Gradients into dq, dk, dv (views of one tensor where the inputs were).
void run_backward(Tensor dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse, const Tensor& rng, const Tensor& dq,
                  const Tensor& dk, const Tensor& dv, const Options& o) {
    const int64_t n = q.dim();
    if (dout.stride(n - 1) != 1) dout = dout.contiguous();
    TORCH_CHECK(dout.scalar_type() == q.scalar_type(), "query and dout must have the same dtype");
    TORCH_CHECK(dout.is_cuda(), "Input tensor must be on CUDA device");
    TORCH_CHECK(dout.sizes() == q.sizes(), "dout must have the shape of out");
    fa_bwd_params p;
    std::memset(&p, 0, sizeof p);
    p.dout = dout.data_ptr(); p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.out = out.data_ptr();
    p.softmax_lse = lse.data_ptr<float>();
    p.dq = dq.data_ptr(); p.dk = dk.data_ptr(); p.dv = dv.data_ptr();
    strides(q, p.q_batch_stride, p.q_row_stride, p.q_head_stride);
    strides(k, p.k_batch_stride, p.k_row_stride, p.k_head_stride);
    strides(v, p.v_batch_stride, p.v_row_stride, p.v_head_stride);
    strides(out, p.o_batch_stride, p.o_row_stride, p.o_head_stride);
    strides(dout, p.do_batch_stride, p.do_row_stride, p.do_head_stride);
    strides(dq, p.dq_batch_stride, p.dq_row_stride, p.dq_head_stride);
    strides(dk, p.dk_batch_stride, p.dk_row_stride, p.dk_head_stride);
    strides(dv, p.dv_batch_stride, p.dv_row_stride, p.dv_head_stride);
    p.h = (int32_t)q.size(n - 2); p.h_k = (int32_t)k.size(n - 2); p.d = (int32_t)q.size(n - 1);
    int64_t total_q = 0, total_k = 0;
    if (o.cu_q.defined()) {
        p.cu_seqlens_q = o.cu_q.data_ptr<int32_t>(); p.cu_seqlens_k = o.cu_k.data_ptr<int32_t>();
        p.b = (int32_t)o.cu_q.size(0) - 1; p.seqlen_q = o.max_q; p.seqlen_k = o.max_k;
        total_q = q.size(0); total_k = k.size(0);
    } else {
        p.b = (int32_t)q.size(0); p.seqlen_q = (int32_t)q.size(1); p.seqlen_k = (int32_t)k.size(1);
    }
    p.seqlen_q_rounded = (p.seqlen_q + 127) / 128 * 128;
    const Tensor softmax_d = new_floats(q, {p.b, p.h, p.seqlen_q_rounded});
    p.softmax_d = softmax_d.data_ptr<float>();
    p.softmax_scale = (float)o.scale;
    p.is_causal = o.causal; p.window_left = o.left; p.window_right = o.causal ? 0 : o.right;
    p.dtype = dtype_code(q);
    if (o.dropout > 0.0) {
        p.p_dropout = (float)o.dropout;
        p.rng_state = reinterpret_cast<const uint64_t*>(rng.data_ptr<int64_t>());
    }
    // work space as in _native._lend_scratch: without room for it another form runs
    Tensor scratch;
    const int64_t bytes = lib.bwd_lend_bytes(&p, total_q, total_k);
    if (bytes > 0) {
        try {
            scratch = at::empty({bytes}, q.options().dtype(at::kByte).requires_grad(false));
        } catch (const c10::OutOfMemoryError&) {
        }
    }
    if (const int rc = lib.bwd_lent(&p, total_q, total_k, scratch.defined() ? scratch.data_ptr() : nullptr, scratch.defined() ? bytes : 0, stream_of(q)))
        library_error(rc, nullptr);
}

// ------------------------------------------------------------------------------------------------
// Autograd: q, k and v as KIND separate tensors (3), as one packed tensor (1), or as q and a packed tensor of k and v (2).  What is
// saved are the inputs themselves (not views of them), out, the log-sum-exp, and what a packed or dropout call needs.
// ------------------------------------------------------------------------------------------------
struct Views { Tensor q, k, v; };
template <int KIND> Views views(const Tensor& a, const Tensor& b, const Tensor& c) {
    if constexpr (KIND == 3) return {a, b, c};
    const int64_t dim = (KIND == 1 ? a : b).dim() - 3;
    if constexpr (KIND == 1) return {a.select(dim, 0), a.select(dim, 1), a.select(dim, 2)};
    else return {a, b.select(dim, 0), b.select(dim, 1)};
}

template <class... X>      // one Tensor for each input
struct Attention : torch::autograd::Function<Attention<X...>> {
    static constexpr int KIND = sizeof...(X);
    static Tensor forward(torch::autograd::AutogradContext* ctx, const X&... x, const Options& o) {
        torch::autograd::variable_list saved = {x...};
        const Views w = views<KIND>(saved[0], KIND >= 2 ? saved[KIND >= 2] : Tensor(), KIND == 3 ? saved[2] : Tensor());
        Result r = run_forward(w.q, w.k, w.v, o);
        saved.push_back(r.out);
        saved.push_back(r.lse);
        if (o.cu_q.defined()) { saved.push_back(o.cu_q); saved.push_back(o.cu_k); }
        if (r.rng.defined()) saved.push_back(r.rng);
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["o"] = c10::List<double>({o.dropout, o.scale, o.causal ? 1.0 : 0.0, (double)o.left, (double)o.right, (double)o.max_q, (double)o.max_k, o.cu_q.defined() ? 1.0 : 0.0});
        return r.out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const auto w = ctx->saved_data["o"].toDoubleVector();
        Options o;
        o.dropout = w[0]; o.scale = w[1]; o.causal = w[2] != 0; o.left = (int32_t)w[3]; o.right = (int32_t)w[4]; o.max_q = (int32_t)w[5]; o.max_k = (int32_t)w[6];
        // (gradients are not differentiated: what is formed here has no history, as where Python's functions form it)
        const at::NoGradGuard no_grad;
        const Tensor a = saved[0], b = KIND >= 2 ? saved[1] : Tensor(), c = KIND == 3 ? saved[2] : Tensor();
        size_t next = KIND + 2;
        if (w[7] != 0) { o.cu_q = saved[next++]; o.cu_k = saved[next++]; }
        Tensor rng;
        if (o.dropout > 0.0) rng = saved[next];
        const c10::DeviceGuard guard(a.device());
        const Views x = views<KIND>(a, b, c);
        Tensor da, db, dc;
        if constexpr (KIND == 1) {
            da = at::empty(a.sizes(), a.options().requires_grad(false));
        } else {
            da = new_like(a);
            if constexpr (KIND == 2) db = at::empty(b.sizes(), b.options().requires_grad(false));
            else { db = new_like(b); dc = new_like(c); }
        }
        const Views d = views<KIND>(da, db, dc);
        run_backward(grads[0], x.q, x.k, x.v, saved[KIND], saved[KIND + 1], rng, d.q, d.k, d.v, o);
        torch::autograd::variable_list out = {da};
        if constexpr (KIND >= 2) out.push_back(db);
        if constexpr (KIND == 3) out.push_back(dc);
        out.push_back(Tensor());        // the options
        return out;
    }
};

// a, b, c: the KIND input tensors; args: what follows them (cu_seqlens and maxima of a packed call, then the options)
template <int KIND, bool PACKED>
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    constexpr int kCu = !PACKED ? 0 : KIND == 1 ? 2 : 4;
    if (!lib.fwd_rng || nargs != KIND + kCu + 5 || !as_bound() || !plain_thread()) Py_RETURN_NONE;
    constexpr int64_t rows = PACKED ? 3 : 4;                   // dimensions of q
    const Tensor* a = plain16(args[0], KIND == 1 ? rows + 1 : rows);
    const Tensor* b = KIND >= 2 ? plain16(args[1], KIND == 2 ? rows + 1 : rows) : a;
    const Tensor* c = KIND == 3 ? plain16(args[2], rows) : b;
    if (!a || !b || !c || !like(*a, *b) || !like(*a, *c)) Py_RETURN_NONE;
    if (KIND == 1 && a->size(rows - 2) != 3) Py_RETURN_NONE;
    if (KIND == 2 && b->size(rows - 2) != 2) Py_RETURN_NONE;
    if (KIND == 3 && b->sizes() != c->sizes()) Py_RETURN_NONE;
    const Tensor &q = *a, &k = *b;
    const int64_t d = q.size(q.dim() - 1), h = q.size(q.dim() - 2), hk = k.size(k.dim() - 2);
    if (k.size(k.dim() - 1) != d || h % hk != 0 || (!PACKED && k.size(0) != q.size(0))) Py_RETURN_NONE;
    // (sizes and strides of the batch within what the library counts in 32 bits)
    for (const Tensor* t : {a, b, c})
        for (int64_t n : t->sizes())
            if (n > INT32_MAX) Py_RETURN_NONE;
    Options o;
    if (!parse(args + KIND + kCu, d, o)) Py_RETURN_NONE;
    if constexpr (PACKED) {
        const Tensor* x = words32(args[KIND], q, -1);
        if (!x || x->size(0) < 2) Py_RETURN_NONE;
        const Tensor* y = KIND == 1 ? x : words32(args[KIND + 1], q, x->size(0));
        if (!y) Py_RETURN_NONE;
        if (!integer(args[KIND == 1 ? 2 : KIND + 2], o.max_q) || !integer(args[KIND == 1 ? 2 : KIND + 3], o.max_k)) Py_RETURN_NONE;
        if (o.max_q <= 0 || o.max_k <= 0) Py_RETURN_NONE;
        o.cu_q = *x;
        o.cu_k = *y;
    }
    const bool grad = at::GradMode::is_enabled() && (a->requires_grad() || b->requires_grad() || c->requires_grad());
    if (grad && !plain_autograd()) Py_RETURN_NONE;
    if (o.dropout > 0.0 && capturing(*a)) Py_RETURN_NONE;
    Tensor keep, out;
    {
        const at::NoGradGuard no_grad;
        const Views x = views<KIND>(*a, *b, *c);
        lend_words(args[0], x.q, x.k, x.v, o, keep);
    }
    const Tensor ta = *a, tb = KIND >= 2 ? *b : Tensor(), tc = KIND == 3 ? *c : Tensor();
    {
        NoGil no_gil;
        if (grad) {
            if constexpr (KIND == 1) out = Attention<Tensor>::apply(ta, o);
            else if constexpr (KIND == 2) out = Attention<Tensor, Tensor>::apply(ta, tb, o);
            else out = Attention<Tensor, Tensor, Tensor>::apply(ta, tb, tc, o);
        } else {
            const at::NoGradGuard no_grad;
            const Views x = views<KIND>(ta, tb, tc);
            out = run_forward(x.q, x.k, x.v, o).out;
        }
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// flash_attn_with_kvcache: q, k_cache, v_cache, k, v, rotary_cos, rotary_sin, cache_seqlens, cache_batch_idx, softmax_scale, causal,
// window_size, rotary_interleaved, num_splits
PyObject* kvcache(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!lib.fwd_kvcache || nargs != 14 || !as_bound() || !plain_thread()) Py_RETURN_NONE;
    const Tensor *q = plain16(args[0], 4), *kc = plain16(args[1], 4), *vc = plain16(args[2], 4);
    if (!q || !kc || !vc || !like(*q, *kc) || !like(*q, *vc)) Py_RETURN_NONE;
    const int64_t b = q->size(0), sq = q->size(1), h = q->size(2), d = q->size(3), sk = kc->size(1), hk = kc->size(2);
    if (kc->size(3) != d || kc->sizes() != vc->sizes() || h % hk != 0 || b > INT32_MAX || sq > INT32_MAX || sk > INT32_MAX) Py_RETURN_NONE;
    if (args[8] == Py_None && kc->size(0) < b) Py_RETURN_NONE;
    Options o;
    bool interleaved;
    int32_t splits;
    if (args[9] == Py_None) o.scale = std::pow((double)d, -0.5);
    else if (!number(args[9], o.scale)) Py_RETURN_NONE;
    if (!boolean(args[10], o.causal) || !pair(args[11], o.left, o.right) || !boolean(args[12], interleaved) || !integer(args[13], splits) || splits > 128) Py_RETURN_NONE;
    fa_fwd_params p = forward_params(*q, *kc, *vc, o);
    p.num_splits = splits > 0 ? splits : 0;
    Tensor seqlens, index;
    if (args[7] != Py_None) {
        const Tensor* t = words32(args[7], *q, b);
        if (!t) Py_RETURN_NONE;
        seqlens = *t;
        p.cu_seqlens_k = t->data_ptr<int32_t>();
        p.is_seqlens_k_cumulative = 0;
    }
    Tensor k_new, v_new, cos, sin;
    if (args[3] != Py_None) {
        const Tensor *kn = plain16(args[3], 4), *vn = plain16(args[4], 4);
        if (!kn || !vn || !seqlens.defined() || sq > sk || !like(*q, *kn) || !like(*q, *vn) || kn->sizes() != vn->sizes()) Py_RETURN_NONE;
        if (kn->size(0) != b || kn->size(2) != hk || kn->size(3) != d || kn->size(1) > INT32_MAX) Py_RETURN_NONE;
        p.seqlen_knew = (int32_t)kn->size(1);
        p.k_new = kn->data_ptr();
        p.v_new = vn->data_ptr();
        strides(*kn, p.knew_batch_stride, p.knew_row_stride, p.knew_head_stride);
        strides(*vn, p.vnew_batch_stride, p.vnew_row_stride, p.vnew_head_stride);
        k_new = *kn;
        v_new = *vn;
        if (args[5] != Py_None) {
            const Tensor *c = plain(args[5]), *s = plain(args[6]);
            if (!c || !s || c->dim() != 2 || s->dim() != 2 || !like(*q, *c) || !like(*q, *s) || c->sizes() != s->sizes() || !c->is_contiguous() || !s->is_contiguous()) Py_RETURN_NONE;
            const int64_t rot = 2 * c->size(1);
            if (rot <= 0 || rot > d || rot % 16 != 0 || c->size(0) < sk) Py_RETURN_NONE;
            p.rotary_cos = c->data_ptr();
            p.rotary_sin = s->data_ptr();
            p.rotary_dim = (int32_t)rot;
            p.is_rotary_interleaved = interleaved;
            cos = *c;
            sin = *s;
        } else if (args[6] != Py_None) {
            Py_RETURN_NONE;
        }
    } else if (args[4] != Py_None || args[5] != Py_None || args[6] != Py_None) {
        Py_RETURN_NONE;
    }
    if (args[8] != Py_None) {
        const Tensor* t = words32(args[8], *q, b);
        if (!t) Py_RETURN_NONE;
        index = *t;
        p.cache_batch_idx = t->data_ptr<int32_t>();
    }
    // plan, then the words: the plan does not depend on where they are
    const Tensor tq = *q, tk = *kc, tv = *vc;
    Tensor keep, more;
    p.work_counter = counters(args[0], tq, FA_WORK_COUNTER_WORDS, keep);
    p.work_counter_len = FA_WORK_COUNTER_WORDS;
    int32_t n = 0;
    if (lib.plan_splits(&p, 2, &n) != 0) Py_RETURN_NONE;
    if (n == 1 && sq >= 32 && use_list()) {
        const int64_t words = lib.work_list_words(&p);
        if (words > FA_WORK_COUNTER_WORDS) {
            p.work_counter = counters(args[0], tq, words, more);
            p.work_counter_len = (int32_t)words;
        }
    }
    Tensor out;
    {
        NoGil no_gil;
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(tq.device());
        out = new_like(tq);
        const int64_t rows = (int64_t)n * p.b * p.h * p.seqlen_q, width = (p.d + 31) / 32 * 32;
        const Tensor lse = new_floats(tq, {p.b, p.h, p.seqlen_q});
        Tensor accum;
        p.o = out.data_ptr();
        p.softmax_lse = lse.data_ptr<float>();
        strides(out, p.o_batch_stride, p.o_row_stride, p.o_head_stride);
        if (n > 1) {
            accum = new_floats(tq, {rows * (width + 1)});
            p.o_accum = accum.data_ptr<float>();
            p.lse_accum = p.o_accum + rows * width;
        }
        if (const int rc = lib.fwd_kvcache(&p, stream_of(tq))) library_error(rc, &tq);
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// apply_rotary_emb_qkv_ where no gradient is asked for: qkv, cos, sin, interleaved, seqlen_offsets.  q and k of a dense projection are
// one run of heads; the result is a view of qkv, as an autograd function returns an input.
PyObject* rotary_qkv(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!lib.rotary || nargs != 5 || !as_bound() || !plain_thread()) Py_RETURN_NONE;
    const Tensor *x = plain16(args[0], 5), *cos = plain(args[1]), *sin = plain(args[2]);
    bool interleaved;
    int32_t offset;
    if (!x || !cos || !sin || !boolean(args[3], interleaved) || !integer(args[4], offset) || offset < 0) Py_RETURN_NONE;
    if (at::GradMode::is_enabled() && (x->requires_grad() || cos->requires_grad() || sin->requires_grad())) Py_RETURN_NONE;
    const auto cs = cos->scalar_type();
    if ((cs != at::kHalf && cs != at::kBFloat16 && cs != at::kFloat) || sin->scalar_type() != cs || cos->device() != x->device() || sin->device() != x->device()) Py_RETURN_NONE;
    if (cos->dim() != 2 || cos->sizes() != sin->sizes() || !cos->is_contiguous() || !sin->is_contiguous() || !x->is_contiguous() || x->size(2) != 3) Py_RETURN_NONE;
    const int64_t b = x->size(0), s = x->size(1), h = x->size(3), d = x->size(4), rot = 2 * cos->size(1);
    if (rot <= 0 || rot > d || offset + s > cos->size(0) || b > INT32_MAX || cos->size(0) > INT32_MAX || h > INT32_MAX / 2) Py_RETURN_NONE;
    fa_rotary_params p;
    std::memset(&p, 0, sizeof p);
    p.x = x->data_ptr(); p.out = x->data_ptr(); p.cos = cos->data_ptr(); p.sin = sin->data_ptr();
    p.x_batch_stride = p.o_batch_stride = s * 3 * h * d;
    p.x_row_stride = p.o_row_stride = 3 * h * d;
    p.x_head_stride = p.o_head_stride = d;
    p.cs_row_stride = rot / 2;
    p.b = (int32_t)b; p.seqlen = (int32_t)s; p.h = (int32_t)(2 * h); p.d = (int32_t)d;
    p.rotary_dim = (int32_t)rot; p.seqlen_ro = (int32_t)cos->size(0); p.seqlen_offset = offset;
    p.interleaved = interleaved;
    p.dtype = dtype_code(*x);
    p.cs_dtype = cs == at::kFloat ? FA_DTYPE_FP32 : dtype_code(*cos);
    const Tensor tx = *x;
    Tensor out;
    {
        NoGil no_gil;
        const at::NoGradGuard no_grad;
        const c10::DeviceGuard guard(tx.device());
        if (const int rc = lib.rotary(&p, stream_of(tx))) library_error(rc, nullptr);
        out = at::alias(tx);
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// bind(_native.__dict__, sizes of the parameter blocks, addresses in the order of Library)
PyObject* bind(PyObject*, PyObject* args) {
    PyObject* dict;
    int fwd_size, bwd_size, rotary_size;
    unsigned long long f[9];
    if (!PyArg_ParseTuple(args, "O!iiiKKKKKKKKK", &PyDict_Type, &dict, &fwd_size, &bwd_size, &rotary_size, f, f + 1, f + 2, f + 3, f + 4, f + 5, f + 6, f + 7, f + 8)) return nullptr;
    if (fwd_size != (int)sizeof(fa_fwd_params) || bwd_size != (int)sizeof(fa_bwd_params) || rotary_size != (int)sizeof(fa_rotary_params)) {
        PyErr_SetString(PyExc_ImportError, "flash_attn: parameter layout mismatch between libfa_mi355x.so and flash_attn._host; rebuild both");
        return nullptr;
    }
    Py_INCREF(dict);
    Py_XDECREF(native_dict);
    native_dict = dict;
    name_counters = PyUnicode_InternFromString("_COUNTERS");
    name_words = PyUnicode_InternFromString("_counters");
    name_list = PyUnicode_InternFromString("WORK_LIST");
    name_reset = PyUnicode_InternFromString("_reset_counters");
    Library l;
    l.fwd_rng = reinterpret_cast<decltype(l.fwd_rng)>(f[0]);
    l.varlen_fwd_rng = reinterpret_cast<decltype(l.varlen_fwd_rng)>(f[1]);
    l.fwd_kvcache = reinterpret_cast<decltype(l.fwd_kvcache)>(f[2]);
    l.plan_splits = reinterpret_cast<decltype(l.plan_splits)>(f[3]);
    l.work_list_words = reinterpret_cast<decltype(l.work_list_words)>(f[4]);
    l.last_error = reinterpret_cast<decltype(l.last_error)>(f[5]);
    l.bwd_lend_bytes = reinterpret_cast<decltype(l.bwd_lend_bytes)>(f[6]);
    l.bwd_lent = reinterpret_cast<decltype(l.bwd_lent)>(f[7]);
    l.rotary = reinterpret_cast<decltype(l.rotary)>(f[8]);
    lib = l;
    Py_RETURN_NONE;
}

// watch(module.__dict__, names): functions of the module that the Python layer calls where this one does not
PyObject* watch(PyObject*, PyObject* args) {
    PyObject *dict, *names;
    if (!PyArg_ParseTuple(args, "O!O!", &PyDict_Type, &dict, &PyTuple_Type, &names)) return nullptr;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); i++) {
        PyObject* const name = PyTuple_GET_ITEM(names, i);
        PyObject* const function = PyDict_GetItemWithError(dict, name);
        if (!function) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_KeyError, "%S", name);
        Py_INCREF(dict);
        Py_INCREF(name);
        Py_INCREF(function);
        stood_in.push_back({dict, name, function});
    }
    Py_RETURN_NONE;
}

#define FA_FAST(name, ...) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&__VA_ARGS__)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"watch", watch, METH_VARARGS, nullptr},
    FA_FAST("func", attention<3, false>),
    FA_FAST("qkvpacked_func", attention<1, false>),
    FA_FAST("kvpacked_func", attention<2, false>),
    FA_FAST("varlen_func", attention<3, true>),
    FA_FAST("varlen_qkvpacked_func", attention<1, true>),
    FA_FAST("varlen_kvpacked_func", attention<2, true>),
    FA_FAST("with_kvcache", kvcache),
    FA_FAST("rotary_emb_qkv_", rotary_qkv),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native host path of the attention functions", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
