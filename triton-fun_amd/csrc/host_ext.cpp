// The host path of the operators that a program calls in a loop, in native code: argument checks, strides, allocations and the
// C-ABI call of one operator, and the differentiable attention as an autograd node.
//
// Bound: the host.  A call of the fused forward through ctypes costs the interpreter 14 us, of which the launch itself is 3;
// sizes whose kernels take less than that (a few hundred row blocks) run at the interpreter's speed, and a training step, whose
// backward an autograd thread runs under the interpreter's lock, at 90 us.  Here a call reads the tensors' fields directly.
//
// Every entry point (of the three operators together as well) handles the ordinary case (tensors on the current device, rows in whole 16-byte pieces) and returns False
// (attend: None) for anything else, before it has done anything: the Python launchers then take the call, with their copies and
// their messages.  The kernels are reached through the addresses that `bind` receives, so that both layers use one library.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/custom_class.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/splat_hip.h"

namespace {

// ---- the library's entry points -------------------------------------------------------------------------------------
struct Api {
    decltype(&splat_last_error) last_error;
    decltype(&splat_attention_fwd_hinted) fwd_hinted;
    decltype(&splat_attention_fwd_keys) fwd_keys;
    decltype(&splat_transpose_keys) transpose_keys;
    decltype(&splat_attention_bwd) bwd;
    decltype(&splat_attention_bwd_keys) bwd_keys;
    decltype(&splat_attention_bwd_f32) bwd_f32;
    decltype(&splat_attention_bwd_keys_f32) bwd_keys_f32;
    decltype(&splat_sddmm) sddmm;
    decltype(&splat_sddmm_probs) sddmm_probs;
    decltype(&splat_sddmm_planned) sddmm_planned;
    decltype(&splat_softmax) softmax;
    decltype(&splat_sddmm_softmax) sddmm_softmax;
    decltype(&splat_operators) operators;
    decltype(&splat_spmm) spmm;
    decltype(&splat_spmm_planned) spmm_planned;
    decltype(&splat_acsr_build_record) build_record;
    decltype(&splat_attention_plan_report) plan_report;
} api;
PyObject* g_error = nullptr;  // SplatError

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return SPLAT_F32;
        case at::kHalf: return SPLAT_F16;
        case at::kBFloat16: return SPLAT_BF16;
        default: return -1;
    }
}

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// rows of the last dimension contiguous, in whole 16-byte pieces
bool rows_in_pieces(const at::Tensor& t, int64_t epc) {
    return t.stride(3) == 1 && t.stride(0) % epc == 0 && t.stride(1) % epc == 0 && t.stride(2) % epc == 0 && aligned16(t);
}

bool is_shape(const at::Tensor& t, int64_t a, int64_t b, int64_t c, int64_t d) {
    return t.size(0) == a && t.size(1) == b && t.size(2) == c && t.size(3) == d;
}

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Uninitialised memory on the current device, contiguous: at::empty without the dispatcher (0.6 us instead of 1.5).
at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType type) {
    return at::Tensor(at::detail::empty_cuda(sizes, type, at::Device(at::kCUDA, c10::hip::current_device()), c10::nullopt));
}

std::string failure(const char* what, int rc) {
    return std::string(what) + " failed (code " + std::to_string(rc) + "): " + api.last_error();
}

// ---- a mask: its segments as the C ABI takes them, the plan table, and the tensors that own the memory -----------------
struct Mask : torch::CustomClassHolder {
    splat_acsr_seg segs[SPLAT_MAX_SEGMENTS];
    int n_seg = 0;
    int64_t rows = 0;
    int max_step = 1;
    bool one_step = false;         // the plan's blocks walk slots (splat_operators)
    at::Tensor plan;               // may be undefined
    int live_percent = 0;          // of the positions that the plan walks, 0: unknown
    std::vector<at::Tensor> keep;  // the arrays that `segs` points into
    int device = 0;
    const void* plan_ptr() const { return plan.data_ptr(); }
    int64_t plan_bytes() const { return plan.nbytes(); }
};

// What the differentiable attention needs besides q, k and v.
struct GradState : torch::CustomClassHolder {
    c10::intrusive_ptr<Mask> fwd;   // the mask, with its plan
    c10::intrusive_ptr<Mask> keys;  // the transposed mask's segments that are walked by blocks of keys, with their plan
    c10::intrusive_ptr<Mask> rows;  // its row-sparse segments, listed row by row (may be null)
    at::Tensor key_of_row;
    int64_t per_stretch = 0;
    int64_t B = 0, H = 0, L = 0, d = 0;
    at::ScalarType dtype = at::kFloat;
};

const char* const kMaskName = "splat.mask";
const char* const kGradName = "splat.grad";

template <typename H>
void drop(PyObject* cap) {
    auto* p = static_cast<H*>(PyCapsule_GetPointer(cap, PyCapsule_GetName(cap)));
    if (p) c10::raw::intrusive_ptr::decref(p);
}
template <typename H>
PyObject* capsule(c10::intrusive_ptr<H> h, const char* name) {
    return PyCapsule_New(h.release(), name, drop<H>);
}
template <typename H>
c10::intrusive_ptr<H> held(PyObject* cap, const char* name) {
    auto* p = static_cast<H*>(PyCapsule_GetPointer(cap, name));
    return p ? c10::intrusive_ptr<H>::reclaim_copy(p) : c10::intrusive_ptr<H>();
}
Mask* mask_of(PyObject* cap) { return static_cast<Mask*>(PyCapsule_GetPointer(cap, kMaskName)); }

// A call of the library that failed: SplatError in the program, as from the Python launchers.
struct Failure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
// The same from the autograd engine's thread: the engine carries a persisted Python error over to the thread that called backward.
[[noreturn]] void raise_on_engine_thread(const std::string& what) {
    pybind11::gil_scoped_acquire gil;
    PyErr_SetString(g_error, what.c_str());
    python_error e;
    e.persist();
    throw e;
}

// A 4-dimensional device tensor on the current device, or null.
const at::Tensor* tensor4(PyObject* o, int device) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.dim() != 4 || t.layout() != at::kStrided || t.get_device() != device) return nullptr;
    return &t;
}

PyObject* raise_rc(const char* what, int rc) {
    PyErr_SetString(g_error, failure(what, rc).c_str());
    return nullptr;
}
// The C++ exception being handled as the Python error that PyTorch's own functions raise for it (out of memory among them).
PyObject* raise_current() {
    if (!PyErr_Occurred()) torch::translate_exception_to_python(std::current_exception());
    return nullptr;
}

// K [B, H, L, d] with rows contiguous from K^T [B, H, d, L] with the keys contiguous: one streaming kernel.
at::Tensor transposed_keys(const at::Tensor& kT, int* rc) {
    at::Tensor k = fresh({kT.size(0), kT.size(1), kT.size(3), kT.size(2)}, kT.scalar_type());
    *rc = api.transpose_keys(kT.data_ptr(), kT.stride(0), kT.stride(1), kT.stride(2), k.data_ptr(), kT.size(0), kT.size(1),
                             kT.size(3), kT.size(2), dtype_code(kT.scalar_type()), stream_of(kT));
    return k;
}

// mask(arr_address, n_seg, rows, plan | None, live_percent, one_step, max_step, (tensors...)) -> capsule
PyObject* py_mask(PyObject*, PyObject* args) {
    unsigned long long addr;
    int n_seg, live, one_step, max_step;
    long long rows;
    PyObject *plan, *tensors;
    if (!PyArg_ParseTuple(args, "KiLOipiO!", &addr, &n_seg, &rows, &plan, &live, &one_step, &max_step, &PyTuple_Type, &tensors)) return nullptr;
    if (n_seg < 1 || n_seg > SPLAT_MAX_SEGMENTS) {
        PyErr_SetString(PyExc_ValueError, "number of segments");
        return nullptr;
    }
    auto m = c10::make_intrusive<Mask>();
    std::memcpy(m->segs, reinterpret_cast<const void*>(static_cast<uintptr_t>(addr)), n_seg * sizeof(splat_acsr_seg));
    m->n_seg = n_seg, m->rows = rows, m->live_percent = live, m->one_step = one_step != 0, m->max_step = max_step;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tensors); ++i) {
        PyObject* o = PyTuple_GET_ITEM(tensors, i);
        if (!THPVariable_Check(o)) continue;
        m->keep.push_back(THPVariable_Unpack(o));
        m->device = m->keep.back().get_device();
    }
    if (plan != Py_None && THPVariable_Check(plan)) m->plan = THPVariable_Unpack(plan);
    return capsule(std::move(m), kMaskName);
}

// ---- fused forward -------------------------------------------------------------------------------------------------------
// kNo: not an ordinary case, nothing was done; kYes: launched; kFailed: the library refused, its code is in `rc`
enum class Did { kNo, kYes, kFailed };

Did forward(const Mask& m, const at::Tensor& q, at::Tensor kT, const at::Tensor& v, const at::Tensor& out, double scale, float* lse,
            int* rc) {
    const auto dt = q.scalar_type();
    const int code = dtype_code(dt);
    if (code < 0 || kT.scalar_type() != dt || v.scalar_type() != dt || out.scalar_type() != dt || !m.plan.defined()) return Did::kNo;
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2), d = q.size(3);
    if ((d != 64 && d != 128) || L != m.rows || L <= 0 || !is_shape(kT, B, H, d, L) || !is_shape(v, B, H, L, d) || !is_shape(out, B, H, L, d))
        return Did::kNo;
    const int64_t epc = 16 / q.element_size();
    if (!rows_in_pieces(q, epc) || !rows_in_pieces(v, epc) || !rows_in_pieces(out, epc)) return Did::kNo;
    const bool k_rows = kT.stride(2) == 1 && kT.stride(3) >= d && kT.stride(0) % epc == 0 && kT.stride(1) % epc == 0 &&
                        kT.stride(3) % epc == 0 && aligned16(kT);
    if (!k_rows) {
        if (kT.stride(3) != 1 || kT.stride(2) < L) return Did::kNo;
        // keys contiguous: taken as they are where every row of keys is whole 16-byte pieces and no row of the mask steps over
        // columns (dense runs are all this layout can be read in), else turned around first
        const bool as_is = m.max_step < 2 && L % epc == 0 && kT.stride(0) % epc == 0 && kT.stride(1) % epc == 0 &&
                           kT.stride(2) % epc == 0 && aligned16(kT);
        if (!as_is && m.max_step < 2) {  // loaded from where it lies, if the launch can
            *rc = api.fwd_keys(q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), kT.data_ptr(), kT.stride(0), kT.stride(1), kT.stride(2),
                               v.data_ptr(), v.stride(0), v.stride(1), v.stride(2), out.data_ptr(), out.stride(0), out.stride(1),
                               out.stride(2), m.segs, m.n_seg, B, H, L, d, (float)scale, code, m.plan_ptr(), m.plan_bytes(), lse,
                               m.live_percent, stream_of(q));
            if (*rc == 0) return Did::kYes;
            if (*rc != SPLAT_E_UNSUPPORTED) return Did::kFailed;
            *rc = 0;
        }
        if (!as_is) {
            kT = transposed_keys(kT, rc).transpose(2, 3);
            if (*rc) return Did::kFailed;
        }
    }
    void* st = stream_of(q);
    *rc = api.fwd_hinted(q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), kT.data_ptr(), kT.stride(0), kT.stride(1), kT.stride(2),
                         kT.stride(3), v.data_ptr(), v.stride(0), v.stride(1), v.stride(2), out.data_ptr(), out.stride(0), out.stride(1),
                         out.stride(2), m.segs, m.n_seg, B, H, L, d, (float)scale, code, m.plan_ptr(), m.plan_bytes(), lse, m.live_percent,
                         st);
    return *rc ? Did::kFailed : Did::kYes;
}

// forward(mask, q, kT, v, out, scale) -> bool
PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "forward takes 6 arguments");
    Mask* m = mask_of(a[0]);
    if (!m) return nullptr;
    try {
        const int dev = c10::hip::current_device();
        const at::Tensor *q = tensor4(a[1], dev), *kT = tensor4(a[2], dev), *v = tensor4(a[3], dev), *out = tensor4(a[4], dev);
        if (!q || !kT || !v || !out || m->device != dev) Py_RETURN_FALSE;
        const double scale = PyFloat_AsDouble(a[5]);
        if (scale == -1.0 && PyErr_Occurred()) return nullptr;
        int rc = 0;
        const Did did = forward(*m, *q, *kT, *v, *out, scale, nullptr, &rc);
        if (did == Did::kFailed) return raise_rc("splat_attention_fwd_hinted", rc);
        return PyBool_FromLong(did == Did::kYes);
    } catch (...) {
        return raise_current();
    }
}

// ---- differentiable attention ----------------------------------------------------------------------------------------------
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// What the Python function handles or refuses, and a plain node would get silently or obscurely wrong: wrappers without memory of
// their own (functorch, fake tensors), and forward-mode tangents (an output without one would read as a derivative of zero).
bool is_wrapped(const at::Tensor& t) {
    return !t.has_storage() || t.unsafeGetTensorImpl()->is_python_dispatch() || t._fw_grad(/*level=*/0).defined();
}

// t itself where the kernels can read it (rows apart from each other: not the gradient of a sum over the rows, whose row stride is
// 0), else a copy
at::Tensor in_pieces(const at::Tensor& t) {
    return rows_in_pieces(t, 16 / t.element_size()) && t.stride(2) >= t.size(3) ? t : t.contiguous();
}

// The gradients of one call.  A node of its own rather than torch::autograd::Function: the engine runs it on its device thread,
// and what the generic one does there around two launches (a dictionary of saved values, an output saved with its history, a
// dispatch through the autograd keys for every workspace) took longer than the launches (B = 2, H = 4, L = 777, d = 64, float16:
// 74 us a step, here 62).
struct AttendBackward : public torch::autograd::Node {
    SavedVariable q_, k_, v_, lse_, out_;
    c10::intrusive_ptr<GradState> state;
    float scale = 1.f;

    std::string name() const override { return "AttendBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        q_.reset_data(), k_.reset_data(), v_.reset_data(), lse_.reset_data(), out_.reset_data();
    }
    // A saved tensor as the kernels read it.  Hooks of the program may have packed it and unpacked another one: what would be read
    // out of bounds is refused, rows that are not whole pieces are copied.
    at::Tensor checked(const char* name, const at::Tensor& t) const {
        const GradState& st = *state;
        if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.get_device() != st.fwd->device || t.scalar_type() != st.dtype ||
            t.dim() != 4 || !is_shape(t, st.B, st.H, st.L, st.d))
            raise_on_engine_thread(std::string("the saved tensor ") + name + " came back with another type, shape or device");
        return in_pieces(t);
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const at::Tensor q0 = q_.unpack(), k0 = k_.unpack(), v0 = v_.unpack(), lse0 = lse_.unpack(), out0 = out_.unpack(shared_from_this());
        const at::Tensor& grad = grads[0];
        at::AutoDispatchBelowADInplaceOrView below;
        const GradState& st = *state;
        const at::Tensor q = checked("q", q0), k = checked("k", k0), v = checked("v", v0), out = checked("out", out0);
        if (!lse0.defined() || !lse0.is_cuda() || lse0.get_device() != st.fwd->device || lse0.scalar_type() != at::kFloat ||
            lse0.sizes() != at::IntArrayRef({st.B, st.H, st.L}))
            raise_on_engine_thread("the saved row statistic came back with another type, shape or device");
        const at::Tensor lse = lse0.contiguous();
        const int64_t B = st.B, H = st.H, L = st.L, d = st.d;
        // (no gradient arrived: zeros, as the Python function gets them)
        const at::Tensor g = !grad.defined()                  ? at::zeros({B, H, L, d}, q.options())
                             : grad.scalar_type() == st.dtype ? in_pieces(grad)
                                                              : in_pieces(grad.to(st.dtype));
        const int code = dtype_code(st.dtype);
        at::Tensor dq = fresh({B, H, L, d}, st.dtype), dk = fresh({B, H, L, d}, st.dtype), dv = fresh({B, H, L, d}, st.dtype);
        at::Tensor delta = fresh({B, H, L}, at::kFloat);
        void* stream = stream_of(q);
        const Mask &m = *st.fwd, &mt = *st.keys;
#define SPLAT_ARGS                                                                                                                        \
    q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), v.data_ptr(), v.stride(0), \
        v.stride(1), v.stride(2), out.data_ptr(), out.stride(0), out.stride(1), out.stride(2), g.data_ptr(), g.stride(0), g.stride(1),   \
        g.stride(2), lse.data_ptr<float>(), delta.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), m.segs, m.n_seg,       \
        m.plan_ptr(), m.plan_bytes(), mt.segs, mt.n_seg, mt.plan_ptr(), mt.plan_bytes(), B, H, L, d, scale
        int rc = code == SPLAT_F32 ? api.bwd_f32(SPLAT_ARGS, stream) : api.bwd(SPLAT_ARGS, code, stream);
#undef SPLAT_ARGS
        if (rc) raise_on_engine_thread(failure("splat_attention_bwd", rc));
        if (st.rows) {  // the row-sparse segments of the transposed mask, row by row, onto what the others gave
            const Mask& r = *st.rows;
            at::Tensor part = fresh({2, B, H, r.rows, d}, st.dtype);
            char* half = static_cast<char*>(part.data_ptr()) + part.nbytes() / 2;
#define SPLAT_ARGS                                                                                                                        \
    q.data_ptr(), q.stride(0), q.stride(1), q.stride(2), k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), v.data_ptr(), v.stride(0), \
        v.stride(1), v.stride(2), g.data_ptr(), g.stride(0), g.stride(1), g.stride(2), lse.data_ptr<float>(), delta.data_ptr<float>(),   \
        st.key_of_row.data_ptr<int32_t>(), part.data_ptr(), half, r.segs, r.n_seg, r.plan_ptr(), r.plan_bytes(), B, H, L, r.rows, d, scale
            if (code == SPLAT_F32)
                rc = api.bwd_keys_f32(SPLAT_ARGS, dk.data_ptr(), dv.data_ptr(), st.per_stretch, stream);
            else
                rc = api.bwd_keys(SPLAT_ARGS, code, dk.data_ptr(), dv.data_ptr(), st.per_stretch, stream);
#undef SPLAT_ARGS
            if (rc) raise_on_engine_thread(failure("splat_attention_bwd_keys", rc));
        }
        return {dq, dk, dv};
    }
};

// The output, with the node that gives the gradients as its history; undefined when the forward leaves the case to the launcher.
at::Tensor attend(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const c10::intrusive_ptr<GradState>& st, double scale) {
    at::Tensor out, lse;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        out = fresh({st->B, st->H, st->L, st->d}, st->dtype);
        lse = fresh({st->B, st->H, st->L}, at::kFloat);
        int rc = 0;
        const Did did = forward(*st->fwd, q, k.transpose(2, 3), v, out, scale, lse.data_ptr<float>(), &rc);
        if (did == Did::kFailed) throw Failure(failure("splat_attention_fwd_hinted", rc));
        if (did == Did::kNo) return at::Tensor();
    }
    std::shared_ptr<AttendBackward> node(new AttendBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
    torch::autograd::set_history(out, node);
    // (the order of the Python function's save_for_backward, which saved-tensor hooks see)
    node->q_ = SavedVariable(q, false), node->k_ = SavedVariable(k, false), node->v_ = SavedVariable(v, false);
    node->lse_ = SavedVariable(lse, false), node->out_ = SavedVariable(out, true);
    node->state = st, node->scale = (float)scale;
    return out;
}

// grad_state(mask, keys_mask, rows_mask | None, key_of_row | None, per_stretch, B, H, L, d, like) -> capsule; `like` a tensor of the type
PyObject* py_grad_state(PyObject*, PyObject* args) {
    PyObject *m, *mt, *mr, *key, *like;
    long long per, B, H, L, d;
    if (!PyArg_ParseTuple(args, "OOOOLLLLLO", &m, &mt, &mr, &key, &per, &B, &H, &L, &d, &like)) return nullptr;
    auto st = c10::make_intrusive<GradState>();
    st->fwd = held<Mask>(m, kMaskName);
    st->keys = held<Mask>(mt, kMaskName);
    if (!st->fwd || !st->keys) return nullptr;
    if (mr != Py_None) {
        st->rows = held<Mask>(mr, kMaskName);
        if (!st->rows) return nullptr;
        st->key_of_row = THPVariable_Unpack(key);
    }
    st->per_stretch = per, st->B = B, st->H = H, st->L = L, st->d = d;
    st->dtype = THPVariable_Unpack(like).scalar_type();
    return capsule(std::move(st), kGradName);
}

// attend(state, q, k, v, scale) -> output, or None when the case is not an ordinary one
PyObject* py_attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) return PyErr_Format(PyExc_TypeError, "attend takes 5 arguments");
    try {
        auto st = held<GradState>(a[0], kGradName);
        if (!st) return nullptr;
        const int dev = c10::hip::current_device();
        const at::Tensor *q = tensor4(a[1], dev), *k = tensor4(a[2], dev), *v = tensor4(a[3], dev);
        // (under torch.jit.trace the Python function is recorded as an operation that runs again, a node would be a constant)
        if (!q || !k || !v || st->fwd->device != dev || at::tracer::impl::is_dispatch_enabled()) Py_RETURN_NONE;
        const int64_t epc = 16 / q->element_size();
        for (const at::Tensor* t : {q, k, v})
            if (is_wrapped(*t) || t->scalar_type() != st->dtype || !is_shape(*t, st->B, st->H, st->L, st->d) || !rows_in_pieces(*t, epc) ||
                t->stride(2) < st->d)
                Py_RETURN_NONE;
        const double scale = PyFloat_AsDouble(a[4]);
        if (scale == -1.0 && PyErr_Occurred()) return nullptr;
        const at::Tensor out = attend(*q, *k, *v, st, scale);
        if (!out.defined()) Py_RETURN_NONE;
        return THPVariable_Wrap(out);
    } catch (const Failure& e) {
        PyErr_SetString(g_error, e.what());
        return nullptr;
    } catch (...) {
        return raise_current();
    }
}

// ---- the three operators ------------------------------------------------------------------------------------------------------
// Each operator in two halves: whether its operands are ordinary ones, and the launch.  An operand that is none is found before anything runs.
struct Sampled {  // out = scale * x y on the mask's slots; `turn`: y is turned to rows first
    const at::Tensor *x, *y, *out;
    float* lse = nullptr;
    bool turn = false;
    bool find(const Mask& m, PyObject* x_, PyObject* y_, PyObject* out_, PyObject* lse_, int dev);
    int launch(const Mask& m, double scale, const at::Tensor* probs, const char** what) const;  // `probs`: the softmax of the output goes there
};

bool Sampled::find(const Mask& m, PyObject* x_, PyObject* y_, PyObject* out_, PyObject* lse_, int dev) {
    x = tensor4(x_, dev), y = tensor4(y_, dev), out = tensor4(out_, dev);
    if (!x || !y || !out || m.device != dev) return false;
    const int code = dtype_code(x->scalar_type()), out_code = dtype_code(out->scalar_type());
    const int64_t B = x->size(0), H = x->size(1), L = x->size(2), d = x->size(3), keys = y->size(3), T = out->size(3);
    if (code < 0 || out_code < 0 || y->scalar_type() != x->scalar_type() || L != m.rows || x->stride(3) != 1 || B * H * L * d * T == 0 ||
        !is_shape(*y, B, H, d, keys) || !is_shape(*out, B, H, L, T) || !out->is_contiguous() || (y->stride(2) != 1 && y->stride(3) != 1))
        return false;
    if (lse_ != Py_None) {
        if (!THPVariable_Check(lse_)) return false;
        const at::Tensor& t = THPVariable_Unpack(lse_);
        if (!t.is_cuda() || t.get_device() != dev || t.scalar_type() != at::kFloat || !t.is_contiguous() || t.dim() != 3 ||
            t.size(0) != B || t.size(1) != H || t.size(2) != L)
            return false;
        lse = t.data_ptr<float>();
    }
    // K^T with the keys contiguous is read in place by the general kernel and by the two named below.  Up to d = 64 a pass that turns it and a kernel on
    // the copy take less: the kernel of thin wavefronts where the launch has its shape (the three operators, bfloat16: 64 heads of
    // 4096 rows, 33 slots, d = 32: 114 -> 92 us; 512 slots, d = 64: 300 -> 263), in launches of fewer than 256 row blocks of more
    // than 256 slots the general kernel, which is faster on rows of K as well (4 heads of 4001 rows, 301 slots, d = 64: 49 -> 43).  Beyond d = 64 the copy costs as much as it gives (64 heads of 2048 rows, 255 slots: d = 80 122 -> 125,
    // d = 96 126 -> 129), and so does its launch below 64 row blocks (one head of 200 rows: 21 -> 25).
    const bool turned = code != SPLAT_F32 && out_code == code && d % 8 == 0 && d <= 64 && B * H * ((L + 127) / 128) >= 64;
    // Up to 128 inner values float32 (operators_f32.hip, but for the launches that its launcher leaves to the general kernel) and 16-bit launches of few row blocks (sddmm_rows16.hip, whose conditions are these;
    // a stride of n between a block's rows adds at most n - 1 blocks) turn K on its way into LDS, gathered or not: the three
    // operators, float32, 16 heads of 1605 rows, 176 slots with step 2, d = 128, 76.9 -> 72.3 us without the copy.
    const bool few = d % 8 == 0 && B * H * 2 * ((L + 127) / 128 + std::max(m.max_step - 1, 0)) <= 512 &&
                     (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15) == 0 && x->stride(0) % 8 == 0 && x->stride(1) % 8 == 0 &&
                     x->stride(2) % 8 == 0;
    const bool general_f32 = d <= 64 && T > (d > 32 && d <= 56 ? 450 : 600) && B * H * ((L + 63) / 64 + std::max(m.max_step - 1, 0)) >= 1024;
    const bool in_place = out_code == code && d <= 128 && (code == SPLAT_F32 ? !general_f32 : few);
    turn = (m.max_step >= 2 || turned) && !in_place && y->stride(3) == 1 && y->stride(2) != 1;
    return !turn || y->stride(2) >= keys;
}

int Sampled::launch(const Mask& m, double scale, const at::Tensor* probs, const char** what) const {
    int rc = 0;
    at::Tensor k = *y;
    if (turn) {
        k = transposed_keys(k, &rc).transpose(2, 3);
        *what = "splat_transpose_keys";
        if (rc) return rc;
    }
    *what = "splat_sddmm";
    void* st = stream_of(*x);
    const void* plan = m.plan.defined() ? m.plan_ptr() : nullptr;
    const int64_t plan_bytes = plan ? m.plan_bytes() : 0;
#define SPLAT_K x->data_ptr(), x->stride(0), x->stride(1), x->stride(2), k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), k.stride(3), out->data_ptr()
#define SPLAT_SIZES                                                                                                                   \
    m.segs, m.n_seg, x->size(0), x->size(1), x->size(2), k.size(3), x->size(3), out->size(3), (float)scale, dtype_code(x->scalar_type()), \
        dtype_code(out->scalar_type())
    if (probs) return api.sddmm_softmax(SPLAT_K, probs->data_ptr(), SPLAT_SIZES, plan, plan_bytes, st);
    if (plan) return api.sddmm_planned(SPLAT_K, SPLAT_SIZES, lse, plan, plan_bytes, st);
    if (lse) return api.sddmm_probs(SPLAT_K, SPLAT_SIZES, lse, st);
    return api.sddmm(SPLAT_K, SPLAT_SIZES, st);
#undef SPLAT_SIZES
#undef SPLAT_K
}

// y = softmax of x
struct Softmax {
    const at::Tensor *x, *out;
    bool find(const Mask& m, PyObject* x_, PyObject* out_, int dev) {
        x = tensor4(x_, dev), out = tensor4(out_, dev);
        return x && out && m.device == dev && x->sizes() == out->sizes() && x->is_contiguous() && out->is_contiguous() &&
               x->size(2) == m.rows && x->numel() != 0 && dtype_code(x->scalar_type()) >= 0 && dtype_code(out->scalar_type()) >= 0;
    }
    int launch(const Mask& m) const {
        return api.softmax(x->data_ptr(), out->data_ptr(), m.segs, m.n_seg, x->size(0) * x->size(1), x->size(2), x->size(3),
                           dtype_code(x->scalar_type()), dtype_code(out->scalar_type()), stream_of(*x));
    }
};

// out = x y, x on the mask's slots
struct Spmm {
    const at::Tensor *x, *y, *out;
    bool find(const Mask& m, PyObject* x_, PyObject* y_, PyObject* out_, int dev) {
        x = tensor4(x_, dev), y = tensor4(y_, dev), out = tensor4(out_, dev);
        if (!x || !y || !out || m.device != dev) return false;
        const int64_t B = x->size(0), H = x->size(1), L = x->size(2);
        return dtype_code(x->scalar_type()) >= 0 && dtype_code(out->scalar_type()) >= 0 && y->scalar_type() == x->scalar_type() &&
               L == m.rows && x->numel() != 0 && y->numel() != 0 && y->size(0) == B && y->size(1) == H &&
               is_shape(*out, B, H, L, y->size(3)) && x->is_contiguous() && out->is_contiguous() && y->stride(3) == 1;
    }
    int launch(const Mask& m) const {
#define SPLAT_ARGS                                                                                                                     \
    x->data_ptr(), y->data_ptr(), y->stride(0), y->stride(1), y->stride(2), out->data_ptr(), m.segs, m.n_seg, x->size(0), x->size(1), \
        x->size(2), y->size(2), y->size(3), x->size(3), dtype_code(x->scalar_type()), dtype_code(out->scalar_type())
        if (m.plan.defined()) return api.spmm_planned(SPLAT_ARGS, m.plan_ptr(), m.plan_bytes(), stream_of(*x));
        return api.spmm(SPLAT_ARGS, stream_of(*x));
#undef SPLAT_ARGS
    }
};

// sddmm(mask, x, y, output, scale, lse | None) -> bool; a plan in the mask is handed on
PyObject* py_sddmm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "sddmm takes 6 arguments");
    Mask* m = mask_of(a[0]);
    if (!m) return nullptr;
    try {
        Sampled s;
        if (!s.find(*m, a[1], a[2], a[3], a[5], c10::hip::current_device())) Py_RETURN_FALSE;
        const double scale = PyFloat_AsDouble(a[4]);
        if (scale == -1.0 && PyErr_Occurred()) return nullptr;
        const char* what;
        if (const int rc = s.launch(*m, scale, nullptr, &what)) return raise_rc(what, rc);
        Py_RETURN_TRUE;
    } catch (...) {
        return raise_current();
    }
}

// softmax(mask, x, output) -> bool
PyObject* py_softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 3) return PyErr_Format(PyExc_TypeError, "softmax takes 3 arguments");
    Mask* m = mask_of(a[0]);
    if (!m) return nullptr;
    try {
        Softmax s;
        if (!s.find(*m, a[1], a[2], c10::hip::current_device())) Py_RETURN_FALSE;
        if (const int rc = s.launch(*m)) return raise_rc("splat_softmax", rc);
        Py_RETURN_TRUE;
    } catch (...) {
        return raise_current();
    }
}

// spmm(mask, x, y, output) -> bool; a plan in the mask is handed on
PyObject* py_spmm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 4) return PyErr_Format(PyExc_TypeError, "spmm takes 4 arguments");
    Mask* m = mask_of(a[0]);
    if (!m) return nullptr;
    try {
        Spmm s;
        if (!s.find(*m, a[1], a[2], a[3], c10::hip::current_device())) Py_RETURN_FALSE;
        if (const int rc = s.launch(*m)) return raise_rc("splat_spmm", rc);
        Py_RETURN_TRUE;
    } catch (...) {
        return raise_current();
    }
}

// operators(mask | None, mask | None, mask, mask, q, kT, v, scores, probabilities, out, scale) -> bool: the three operators of one forward.  The
// masks are those of the sampled product, for rows of K and for K along the keys, of the softmax and of the last product.  What the
// interpreter does between three calls costs more than the launches (22 -> 12.6 us on the host), and than the kernels of a few row
// blocks (40 heads of 256 rows, 62 slots, bfloat16, d = 64: 20.1 -> 13.6 us a forward).
PyObject* py_operators(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 11) return PyErr_Format(PyExc_TypeError, "operators takes 11 arguments");
    try {
        const int dev = c10::hip::current_device();
        const at::Tensor *q = tensor4(a[4], dev), *kT = tensor4(a[5], dev), *out = tensor4(a[9], dev);
        // (the masks were chosen for the output's type and head dimension)
        if (!q || !kT || !out || q->scalar_type() != out->scalar_type() || q->size(3) != out->size(3)) Py_RETURN_FALSE;
        PyObject* const masks[] = {a[kT->stride(2) == 1 ? 0 : 1], a[2], a[3]};
        Mask* m[3];
        for (int i = 0; i < 3; ++i) {
            if (masks[i] == Py_None) Py_RETURN_FALSE;
            if (!(m[i] = mask_of(masks[i]))) return nullptr;
        }
        Sampled first;
        Softmax second;
        Spmm third;
        if (!first.find(*m[0], a[4], a[5], a[7], Py_None, dev) || !second.find(*m[1], a[7], a[8], dev) || !third.find(*m[2], a[8], a[6], a[9], dev))
            Py_RETURN_FALSE;
        const double scale = PyFloat_AsDouble(a[10]);
        if (scale == -1.0 && PyErr_Occurred()) return nullptr;
        const bool both = second.x->scalar_type() == second.out->scalar_type() && second.x->data_ptr() != second.out->data_ptr();
        const char* what;
        // One launch, where the kernel takes it.  K along the keys is turned on its way there, one key a lane; where the separate launches would turn it
        // and neighbouring lanes' keys lie further apart, it is turned before.  Shares of the separate launches' time, 640 to 4096 workgroups, inside and turned
        // before (mean; bfloat16, one segment, graphs of the forwards): no step 0.48 to 0.95 (0.70) and 0.55 to 0.91 (0.76); steps of 2 to 4, up to 256 slots
        // 0.61 to 0.91 (0.77) and 0.63 to 0.86 (0.78), longer rows d = 32 and 64 0.70 to 0.95 (0.83) and 0.67 to 0.89 (0.79), d = 80 and 128 0.78 to 1.05 (0.92)
        // and 0.72 to 0.92 (0.83); steps of 5 to 8 0.59 to 0.92 (0.77) and 0.58 to 0.87 (0.76).
        at::Tensor turned;
        const Mask& planned = m[0]->plan.defined() ? *m[0] : *m[2];
        if (both && planned.plan.defined() && planned.one_step && first.y->size(3) == third.y->size(2) && third.x->data_ptr() == second.out->data_ptr() &&
            third.out->scalar_type() == q->scalar_type()) {
            if (first.turn && (planned.max_step > 4 || (planned.max_step > 1 && first.out->size(3) > 256 && q->size(3) > 64))) {
                int rc = 0;
                turned = transposed_keys(*first.y, &rc).transpose(2, 3);
                if (rc) return raise_rc("splat_transpose_keys", rc);
                first.y = &turned, first.turn = false;
            }
            const at::Tensor &k = *first.y, &v = *third.y, &s = *first.out;
            const int rc = api.operators(q->data_ptr(), q->stride(0), q->stride(1), q->stride(2), k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), k.stride(3),
                                         v.data_ptr(), v.stride(0), v.stride(1), v.stride(2), s.data_ptr(), second.out->data_ptr(), out->data_ptr(),
                                         planned.segs, planned.n_seg, q->size(0), q->size(1), q->size(2), k.size(3), q->size(3), s.size(3), (float)scale,
                                         dtype_code(q->scalar_type()), planned.plan_ptr(), planned.plan_bytes(), planned.one_step, stream_of(*q));
            if (rc == 0) Py_RETURN_TRUE;
            if (rc != SPLAT_E_UNSUPPORTED) return raise_rc("splat_operators", rc);
        }
        if (const int rc = first.launch(*m[0], scale, both ? second.out : nullptr, &what)) return raise_rc(what, rc);
        if (!both)
            if (const int rc = second.launch(*m[1])) return raise_rc("splat_softmax", rc);
        if (const int rc = third.launch(*m[2])) return raise_rc("splat_spmm", rc);
        Py_RETURN_TRUE;
    } catch (...) {
        return raise_current();
    }
}

// ---- the ACSR and the plan of a mask ---------------------------------------------------------------------------------------------
constexpr int64_t kShareBlocks = 1024;  // row blocks of a build whose shares of the summary a kept buffer holds

// Pinned buffers for what builds and plans under way tell the host: one per call between its launch and its end (the call waits for
// the stream before it gives the buffer back), at most kKeep of them kept for the next ones, longer ones than usual not at all.
class ShareBuffers {
  public:
    at::Tensor take(int64_t n) {
        if (n <= kShareBlocks * 8) {
            std::lock_guard<std::mutex> hold(m_);
            if (!free_.empty()) {
                at::Tensor t = std::move(free_.back());
                free_.pop_back();
                return t;
            }
        }
        return at::empty({std::max(n, kShareBlocks * 8)}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    }
    void give(at::Tensor t) {
        std::lock_guard<std::mutex> hold(m_);
        if (t.numel() == kShareBlocks * 8 && free_.size() < kKeep) free_.push_back(std::move(t));
    }

  private:
    static constexpr size_t kKeep = 4;
    std::mutex m_;
    std::vector<at::Tensor> free_;
};
ShareBuffers* share_buffers() {
    static ShareBuffers* b = new ShareBuffers;  // (never destroyed: the allocator may be gone at the process's end)
    return b;
}

// A call that returned an error: its buffer is given back where the arguments were refused (negative codes), but not where an error of
// the runtime was found with the launch, which may have happened all the same and write to it later.
PyObject* refused(const char* what, int rc, at::Tensor& shares) {
    if (rc < 0)
        share_buffers()->give(std::move(shares));
    else
        new at::Tensor(std::move(shares));
    return raise_rc(what, rc);
}

// Waits for the stream without the interpreter's lock; false with a Python error set when that failed, and then the buffer is not
// given back either.
bool wait_for(const c10::hip::HIPStream& stream, at::Tensor& shares) {
    PyThreadState* const released = PyEval_SaveThread();
    std::exception_ptr failed;
    try {
        c10::hip::stream_synchronize(stream.stream());
    } catch (...) {
        failed = std::current_exception();
    }
    PyEval_RestoreThread(released);
    if (!failed) return true;
    new at::Tensor(std::move(shares));
    torch::translate_exception_to_python(failed);
    return false;
}

// plan(arr_address, n_seg, L, table) -> (whether every live row starts on a multiple of 8 positions of its block's walk, how much of what
// the blocks walk is live, in percent, whether all walk slots: no block's rows differ in step or phase).  Fills the plan table on the current device and waits for it, so that launches on any stream
// may use it.
PyObject* py_plan(PyObject*, PyObject* args) {
    unsigned long long addr;
    int n_seg, L;
    PyObject* o;
    if (!PyArg_ParseTuple(args, "KiiO", &addr, &n_seg, &L, &o)) return nullptr;
    if (!THPVariable_Check(o)) return PyErr_Format(PyExc_TypeError, "table must be a tensor");
    try {
        const at::Tensor& table = THPVariable_Unpack(o);
        const auto* segs = reinterpret_cast<const splat_acsr_seg*>(static_cast<uintptr_t>(addr));
        const int64_t bytes = table.nbytes(), blocks = n_seg > 0 ? bytes / (2 * (5 + 128) * 16 * (int64_t)n_seg) : 0;
        const auto stream = c10::hip::getCurrentHIPStream(table.get_device());
        at::Tensor shares = share_buffers()->take(4 * blocks);
        const int32_t* const sh = shares.data_ptr<int32_t>();
        const int rc = api.plan_report(segs, n_seg, L, table.data_ptr(), bytes, shares.data_ptr<int32_t>(), shares.nbytes(), stream.stream());
        if (rc) return refused("splat_attention_plan_report", rc, shares);
        if (!wait_for(stream, shares)) return nullptr;
        bool aligned = true, one_step = true;
        int64_t walked = 0, live = 0;
        for (int64_t b = 0; b < blocks; ++b) aligned = aligned && sh[4 * b] == 0, one_step = one_step && sh[4 * b + 3] == 0, walked += sh[4 * b + 1] * int64_t(64 * 128), live += sh[4 * b + 2];
        share_buffers()->give(std::move(shares));
        const long percent = walked > 0 ? (long)std::clamp<int64_t>((100 * live + walked - 1) / walked, 1, 100) : 1;
        return Py_BuildValue("NlN", PyBool_FromLong(aligned), percent, PyBool_FromLong(one_step));
    } catch (...) {
        return raise_current();
    }
}

// One array of a record, as a tensor of its own on the record's storage.
at::Tensor part_of(const at::Tensor& record, int64_t offset, int64_t n) {
    at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(record.storage()), record.key_set(), record.dtype());
    t.unsafeGetTensorImpl()->set_storage_offset(record.storage_offset() + offset);
    t.unsafeGetTensorImpl()->set_sizes_contiguous({n});
    return t;
}

// build(mask, block_height) -> ((9 tensors), (9 tensors), T, failed rows, smallest step, largest step, rows off phase): the arrays
// of a record and of its duplicate (without row_last), dTos_lin, dTos_trans, sTod_lin, sTod_trans, nnz, row_first, row_last, span_start, span_end.
// Waits for the stream (T comes back as a number).  None when the case is not an ordinary one.
PyObject* py_build(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2) return PyErr_Format(PyExc_TypeError, "build takes 2 arguments");
    try {
        if (!THPVariable_Check(a[0])) Py_RETURN_NONE;
        const at::Tensor& mask = THPVariable_Unpack(a[0]);
        const long long bh = PyLong_AsLongLong(a[1]);
        if (bh == -1 && PyErr_Occurred()) return nullptr;
        if (!mask.is_cuda() || mask.scalar_type() != at::kByte || mask.dim() != 2 || mask.get_device() != c10::hip::current_device() ||
            mask.numel() == 0 || mask.stride(1) != 1 || mask.stride(0) < mask.size(1) || bh < 1 || bh > (1 << 23))
            Py_RETURN_NONE;
        const int64_t rows = mask.size(0), cols = mask.size(1), blocks = (rows + bh - 1) / bh;
        // the one-kernel build gives a row block to a workgroup: short blocks and very tall ones leave wavefronts or CUs idle
        if (blocks > kShareBlocks || bh < 4 || bh > 64) Py_RETURN_NONE;
        if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) Py_RETURN_NONE;  // (it waits)
        const auto stream = c10::hip::getCurrentHIPStream(mask.get_device());
        const int64_t row_step = (rows + 63) / 64 * 64, span_step = (blocks + 63) / 64 * 64, twin = 5 * row_step + 2 * span_step;
        // (a storage per type: torch.save takes no tensors of two types on one)
        const at::Tensor record = fresh({2 * twin}, at::kFloat), extents = fresh({4 * row_step}, at::kInt);
        at::Tensor shares = share_buffers()->take(8 * blocks);
        const int32_t* const sh = shares.data_ptr<int32_t>();
        const int rc = api.build_record(mask.data_ptr<uint8_t>(), rows, cols, mask.stride(0), (int32_t)bh, record.data_ptr<float>(),
                                        extents.data_ptr<int32_t>(), 1, shares.data_ptr<int32_t>(), stream.stream());
        if (rc) return refused("splat_acsr_build_record", rc, shares);
        // while the kernel runs: the arrays as tensors of their own (a call over 8192 x 8192: 37.6 -> 36.6 us)
        struct Written {  // (the kernel writes the shares: a way out before the wait does not give them back)
            at::Tensor& shares;
            bool waited = false;
            ~Written() {
                if (!waited) new at::Tensor(std::move(shares));
            }
        } written{shares};
        THPObjectPtr sets[2];
        for (int k = 0; k < 2; ++k) {
            sets[k] = PyTuple_New(9);
            if (!sets[k]) return nullptr;
            for (int i = 0; i < 9; ++i) {
                if (k == 1 && i == 6) {  // (the caller's set: nobody reads its row_last)
                    Py_INCREF(Py_None);
                    PyTuple_SET_ITEM(sets[k].get(), i, Py_None);
                    continue;
                }
                at::Tensor t;
                if (i == 5 || i == 6)
                    t = part_of(extents, (2 * k + i - 5) * row_step, rows);
                else if (i < 5)
                    t = part_of(record, k * twin + i * row_step, rows);
                else
                    t = part_of(record, k * twin + 5 * row_step + (i - 7) * span_step, blocks);
                PyObject* const wrapped = THPVariable_Wrap(std::move(t));
                if (!wrapped) return nullptr;
                PyTuple_SET_ITEM(sets[k].get(), i, wrapped);
            }
        }
        written.waited = true;
        if (!wait_for(stream, shares)) return nullptr;
        int32_t t_max = 0, bad = 0, step_min = 0x7fffffff, step_max = 0, res_min = 0x7fffffff, res_max = 0;
        for (int64_t b = 0; b < blocks; ++b) {
            const int32_t* s = sh + 8 * b;
            t_max = std::max(t_max, s[0]), bad += s[1], step_min = std::min(step_min, s[2]), step_max = std::max(step_max, s[3]);
            res_min = std::min(res_min, s[5]), res_max = std::max(res_max, s[6]);
        }
        share_buffers()->give(std::move(shares));
        return Py_BuildValue("NNiiiiii", sets[0].release(), sets[1].release(), t_max, bad, step_min, step_max, res_min, res_max);
    } catch (...) {
        return raise_current();
    }
}

// bind({entry point: address}, SplatError)
PyObject* py_bind(PyObject*, PyObject* args) {
    PyObject *table, *err;
    if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &table, &err)) return nullptr;
    auto take = [&](const char* name, auto& fn) {
        PyObject* o = PyDict_GetItemString(table, name);
        if (!o) {
            PyErr_Format(PyExc_KeyError, "%s", name);
            return false;
        }
        fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(o)));
        return !PyErr_Occurred();
    };
    if (!take("splat_last_error", api.last_error) || !take("splat_attention_fwd_hinted", api.fwd_hinted) || !take("splat_attention_fwd_keys", api.fwd_keys) ||
        !take("splat_transpose_keys", api.transpose_keys) ||
        !take("splat_attention_bwd", api.bwd) || !take("splat_attention_bwd_keys", api.bwd_keys) ||
        !take("splat_attention_bwd_f32", api.bwd_f32) || !take("splat_attention_bwd_keys_f32", api.bwd_keys_f32) || !take("splat_sddmm", api.sddmm) ||
        !take("splat_sddmm_probs", api.sddmm_probs) || !take("splat_sddmm_planned", api.sddmm_planned) ||
        !take("splat_softmax", api.softmax) || !take("splat_sddmm_softmax", api.sddmm_softmax) || !take("splat_operators", api.operators) || !take("splat_spmm", api.spmm) || !take("splat_spmm_planned", api.spmm_planned) ||
        !take("splat_acsr_build_record", api.build_record) || !take("splat_attention_plan_report", api.plan_report))
        return nullptr;
    Py_INCREF(err);
    Py_XSETREF(g_error, err);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, "bind({entry point: address}, error class)"},
    {"mask", py_mask, METH_VARARGS, "the segments of a mask, with its plan"},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_forward)), METH_FASTCALL, "fused forward"},
    {"grad_state", py_grad_state, METH_VARARGS, "what the differentiable attention keeps"},
    {"attend", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_attend)), METH_FASTCALL, "differentiable attention"},
    {"plan", py_plan, METH_VARARGS, "the plan table of a mask"},
    {"build", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_build)), METH_FASTCALL, "the ACSR of a mask tensor"},
    {"sddmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_sddmm)), METH_FASTCALL, "sampled product"},
    {"softmax", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_softmax)), METH_FASTCALL, "softmax of compressed rows"},
    {"spmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_spmm)), METH_FASTCALL, "compressed rows times dense"},
    {"operators", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_operators)), METH_FASTCALL, "the three of them"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_splat_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__splat_host(void) { return PyModule_Create(&module); }
