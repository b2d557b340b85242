// The host side of the Python ops in native code: operand checks, allocation and launch in one call for the plain case.
//
// A call that is anything but plain -- another type than torch.Tensor, another device or dtype, a view that is not contiguous,
// gradients to be recorded, a tangent, a mode or trace that watches calls, shapes that do not fit, a status that is not SWC_OK -- gets
// None back, and the Python code around it, which has the whole rules and the messages, goes its own way.
//
// What it saves, times of a pass that the host bounds: the layer pair 1x16x16x64 23.4 -> 13.7 us, a training step 3x6x6x32 183 -> 98,
// the model with one image 712 -> 398 (ctypes calls, one Python check after the other, and keys of Python tuples before).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/record_stream.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cstring>
#include <memory>

#include "../../include/winograd2x2.h"

namespace {

struct NoGil {   // launches and allocations run without the interpreter's lock, as ctypes and torch's own calls do
    PyThreadState *state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// A mode that watches calls, or a trace that records them.
bool watched()
{
    return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}

const c10::DispatchKeySet kWrappers({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                     c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                     c10::DispatchKey::Negative, c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor});

// The tensor behind `o`, or nullptr where it is not a plain one of that dtype and rank.
const at::Tensor *plain(PyObject *o, at::ScalarType dtype, int64_t rank)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != dtype || t.dim() != rank) return nullptr;
    if (t.key_set().has_any(kWrappers) || !t.has_storage() || !t.is_contiguous()) return nullptr;
    if (t._fw_grad(0).defined()) return nullptr;   // carries a tangent of forward-mode differentiation
    return &t;
}

// An optional operand: *ok is cleared where it is given and not plain, on another device or of another size.
const float *optional(PyObject *o, const at::Tensor &like, at::IntArrayRef sizes, bool *ok)
{
    if (o == Py_None) return nullptr;
    const at::Tensor *t = plain(o, at::kFloat, static_cast<int64_t>(sizes.size()));
    if (t == nullptr || t->device() != like.device() || t->sizes() != sizes) {
        *ok = false;
        return nullptr;
    }
    return static_cast<const float *>(t->const_data_ptr());
}

// A flag; *ok is cleared where its truth value raises, which the general path then does again in its own place.
bool truth(PyObject *o, bool *ok)
{
    const int value = PyObject_IsTrue(o);
    if (value < 0) {
        PyErr_Clear();
        *ok = false;
    }
    return value > 0;
}

bool records(const at::Tensor &t) { return at::GradMode::is_enabled() && t.requires_grad(); }
const float *floats(const at::Tensor &t) { return static_cast<const float *>(t.const_data_ptr()); }
float *floats_of(at::Tensor &t) { return static_cast<float *>(t.mutable_data_ptr()); }
const uint16_t *shorts(const at::Tensor &t) { return static_cast<const uint16_t *>(t.const_data_ptr()); }
at::Tensor make(const at::Tensor &like, at::IntArrayRef sizes, at::ScalarType dtype = at::kFloat)
{
    return at::empty(sizes, at::TensorOptions().device(like.device()).dtype(dtype));
}
swc_stream_t stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool fits(at::IntArrayRef sizes)
{
    for (const int64_t n : sizes)
        if (n <= 0 || n > 0x7fffffff) return false;
    return true;
}
int as_int(int64_t n) { return static_cast<int>(n); }
PyObject *none()
{
    Py_INCREF(Py_None);
    return Py_None;
}
#define SWC_ARGS(n)                                                        \
    HANDLE_TH_ERRORS                                                       \
    if (count != (n)) {                                                    \
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");     \
        return nullptr;                                                    \
    }

// Version counter, address and device of each tensor (None: zeros), to tell whether any was written to, replaced or moved since.
struct Key {
    struct Entry {
        int64_t version, device;
        const void *data;
    } entries[8];
    Py_ssize_t bytes = -1;   // -1: the arguments are wrong and an error is set

    Key(PyObject *const *args, Py_ssize_t count)
    {
        if (count > 8) {
            PyErr_SetString(PyExc_TypeError, "at most eight tensors");
            return;
        }
        for (Py_ssize_t i = 0; i < count; ++i) {
            entries[i] = {0, 0, nullptr};
            if (args[i] == Py_None) continue;
            if (!THPVariable_Check(args[i])) {
                PyErr_SetString(PyExc_TypeError, "tensors or None");
                return;
            }
            const at::Tensor &t = THPVariable_Unpack(args[i]);
            entries[i] = {t._version() + 1, 256 * static_cast<int64_t>(t.device().type()) + t.device().index(), t.const_data_ptr()};
        }
        bytes = count * static_cast<Py_ssize_t>(sizeof(Entry));
    }
};

// key(*tensors): the above as bytes.
PyObject *key(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    const Key k(args, count);
    return k.bytes < 0 ? nullptr : PyBytes_FromStringAndSize(reinterpret_cast<const char *>(k.entries), k.bytes);
    END_HANDLE_TH_ERRORS
}

// Behind which work a tensor has been written: the stream, and an event in it once another stream has asked.  An event at once would
// cost every write 2 us of the host and 3 of the GPU; one that is recorded later is behind more of that stream's work than needed.
struct Mark {
    hipStream_t stream = nullptr;
    hipEvent_t event = nullptr;   // made and read under the interpreter's lock
    bool gpu = false;
    std::atomic<bool> reached{false};
    ~Mark()
    {
        if (event != nullptr) (void)hipEventDestroy(event);
    }
    hipError_t record()
    {
        hipEvent_t e;
        hipError_t st = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        if (st != hipSuccess) return st;
        st = hipEventRecord(e, stream);
        if (st == hipSuccess)
            event = e;
        else
            (void)hipEventDestroy(e);
        return st;
    }
};
constexpr const char *kMark = "swc.mark";

// What is asked about streams here is allowed while a stream is captured, by this thread or another, only in the relaxed mode.
struct Relaxed {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool changed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    ~Relaxed()
    {
        if (changed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

bool capturing(hipStream_t stream)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) (void)hipGetLastError();
    return status != hipStreamCaptureStatusNone;
}

PyObject *hip_error(hipError_t st)
{
    (void)hipGetLastError();
    PyErr_SetString(PyExc_RuntimeError, hipGetErrorString(st));
    return nullptr;
}

// mark(tensor): behind what the current stream has been given on the tensor's device, or None while that stream records a graph.
PyObject *mark(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(1)
    if (!THPVariable_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "a tensor");
        return nullptr;
    }
    const at::Tensor &t = THPVariable_Unpack(args[0]);
    auto m = std::make_unique<Mark>();
    if (t.is_cuda()) {
        const c10::DeviceGuard guard(t.device());
        const Relaxed relaxed;
        const c10::hip::HIPStream current = c10::hip::getCurrentHIPStream(t.device().index());
        m->gpu = true;
        m->stream = current.stream();
        if (capturing(m->stream)) return none();
        // torch's own streams live as long as the process; one from elsewhere may be gone when it would be asked
        const bool own = m->stream == nullptr || c10::hip::getStreamFromExternal(m->stream, t.device().index()).id() != current.id();
        const hipError_t st = own ? hipSuccess : m->record();
        if (st != hipSuccess) return hip_error(st);
    }
    PyObject *capsule = PyCapsule_New(m.get(), kMark, [](PyObject *o) { delete static_cast<Mark *>(PyCapsule_GetPointer(o, kMark)); });
    if (capsule != nullptr) m.release();
    return capsule;
    END_HANDLE_TH_ERRORS
}

// kept(entry, *tensors): what `entry`, a tuple (key, tensor, mark, ...), holds, for use on the current stream, or None where there is no entry
// or its key is not that of the tensors by now.  The current stream waits for the mark where it is another than the mark's; a stream that
// records a graph cannot wait for what was recorded outside of it, then this thread waits.  None also where there is no telling, since
// the mark's stream records a graph by now.  One call, since a layer makes it on every pass: 0.25 us less than a key, its comparison and the wait.
PyObject *kept(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    if (count < 1) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    if (args[0] == Py_None) return none();
    if (!PyTuple_CheckExact(args[0]) || PyTuple_GET_SIZE(args[0]) < 3 || !PyBytes_CheckExact(PyTuple_GET_ITEM(args[0], 0)) ||
        !THPVariable_Check(PyTuple_GET_ITEM(args[0], 1))) {
        PyErr_SetString(PyExc_TypeError, "(key, tensor, mark, ...)");
        return nullptr;
    }
    PyObject *const bytes = PyTuple_GET_ITEM(args[0], 0), *const tensor = PyTuple_GET_ITEM(args[0], 1);
    Mark *m = static_cast<Mark *>(PyCapsule_GetPointer(PyTuple_GET_ITEM(args[0], 2), kMark));
    if (m == nullptr) return nullptr;
    const Key k(args + 1, count - 1);
    if (k.bytes < 0) return nullptr;
    if (PyBytes_GET_SIZE(bytes) != k.bytes || std::memcmp(PyBytes_AS_STRING(bytes), k.entries, static_cast<size_t>(k.bytes)) != 0) return none();
    const at::Tensor &t = THPVariable_Unpack(tensor);
    if (m->gpu) {
        const c10::hip::HIPStream current = c10::hip::getCurrentHIPStream(t.device().index());
        if (current.stream() != m->stream) {
            const c10::DeviceGuard guard(t.device());
            if (!m->reached) {
                const Relaxed relaxed;
                hipError_t st = hipSuccess;
                if (m->event == nullptr) {
                    if (capturing(m->stream)) return none();
                    st = m->record();
                }
                if (st == hipSuccess) {
                    const bool wait = capturing(current.stream());
                    NoGil nogil;
                    st = wait ? hipEventSynchronize(m->event) : hipEventQuery(m->event);
                }
                if (st == hipSuccess) {
                    m->reached = true;
                } else if (st == hipErrorNotReady) {
                    (void)hipGetLastError();
                    st = hipStreamWaitEvent(current.stream(), m->event, 0);
                }
                if (st != hipSuccess) return hip_error(st);
            }
            t.record_stream(c10::Stream(c10::Stream::UNSAFE, t.device(), current.id()));   // of torch's own device type
        }
    }
    Py_INCREF(tensor);
    return tensor;
    END_HANDLE_TH_ERRORS
}

// imtrans(I, relu, scale, shift, bf16)
PyObject *imtrans(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(5)
    const at::Tensor *I = plain(args[0], at::kFloat, 4);
    if (I == nullptr || watched() || records(*I) || !fits(I->sizes())) return none();
    const int64_t B = I->size(0), H = I->size(1), W = I->size(2), C = I->size(3);
    bool ok = (args[2] == Py_None) == (args[3] == Py_None);
    const bool relu = truth(args[1], &ok), bf16 = truth(args[4], &ok);
    const float *scale = optional(args[2], *I, {C}, &ok), *shift = optional(args[3], *I, {C}, &ok);
    if (!ok) return none();
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(I->device());
        out = make(*I, {16, B, (H + 1) / 2, (W + 1) / 2, C}, bf16 ? at::kBFloat16 : at::kFloat);
        if (bf16)
            st = swc_winograd2x2_imtrans_bf16out(floats(*I), scale, shift, static_cast<uint16_t *>(out.mutable_data_ptr()), as_int(C), as_int(B),
                                                 as_int(H), as_int(W), 1, 1, relu, stream_of(*I));
        else if (scale != nullptr)
            st = swc_winograd2x2_imtrans_affine(floats(*I), scale, shift, floats_of(out), as_int(C), as_int(B), as_int(H), as_int(W), 1, 1, relu,
                                                stream_of(*I));
        else
            st = swc_winograd2x2_imtrans(floats(*I), floats_of(out), as_int(C), as_int(B), as_int(H), as_int(W), 1, 1, relu, stream_of(*I));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// weight_pieces(W, bf16 operands)
PyObject *weight_pieces(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(2)
    const at::Tensor *W = plain(args[0], at::kFloat, 3);
    const int bf16 = PyObject_IsTrue(args[1]);
    if (bf16 < 0) return nullptr;
    if (W == nullptr || watched() || W->size(0) != 16 || !fits(W->sizes())) return none();
    const int C = as_int(W->size(1)), K = as_int(W->size(2));
    const size_t bytes = (bf16 ? swc_winograd2x2_weight_pieces_bf16_bytes : swc_winograd2x2_weight_pieces_bytes)(C, K);
    if (bytes == 0) return none();
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(W->device());
        out = make(*W, {static_cast<int64_t>(bytes)}, at::kByte);
        st = (bf16 ? swc_winograd2x2_weight_pieces_bf16 : swc_winograd2x2_weight_pieces)(floats(*W), out.mutable_data_ptr(), C, K, stream_of(*W));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// conv(I, W, bf16 operands, scale, shift, residual, residual_relu, pieces)
PyObject *conv(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(8)
    const at::Tensor *I = plain(args[0], at::kFloat, 5), *W = plain(args[1], at::kFloat, 3);
    if (I == nullptr || W == nullptr || watched() || records(*I) || records(*W) || I->device() != W->device()) return none();
    const int64_t B = I->size(1), nH = I->size(2), nW = I->size(3), C = I->size(4), K = W->size(2);
    if (I->size(0) != 16 || W->size(0) != 16 || W->size(1) != C || !fits(I->sizes()) || !fits(W->sizes())) return none();
    bool ok = (args[3] == Py_None) == (args[4] == Py_None);
    const bool bf16 = truth(args[2], &ok), residual_relu = truth(args[6], &ok);
    if (residual_relu && args[5] == Py_None) ok = false;
    const float *scale = optional(args[3], *I, {K}, &ok), *shift = optional(args[4], *I, {K}, &ok),
                *residual = optional(args[5], *I, {B, 2 * nH, 2 * nW, K}, &ok);
    const bool for_this_call = args[7] == Py_True;
    at::Tensor pieces;
    if (ok && args[7] != Py_None && !for_this_call) {
        const at::Tensor *p = plain(args[7], at::kByte, 1);
        if (p == nullptr || p->device() != I->device() ||
            static_cast<size_t>(p->size(0)) !=
                (bf16 ? swc_winograd2x2_weight_pieces_bf16_bytes : swc_winograd2x2_weight_pieces_bytes)(as_int(C), as_int(K)))
            return none();
        pieces = *p;
    }
    if (!ok) return none();
    at::Tensor out;
    int st = SWC_OK;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(I->device());
        const swc_stream_t stream = stream_of(*I);
        out = make(*I, {B, 2 * nH, 2 * nW, K});
        if (for_this_call && !bf16 && swc_winograd2x2_conv_pieces_gain(as_int(C), as_int(B), as_int(nH), as_int(nW), as_int(K)) == 2) {
            pieces = make(*I, {static_cast<int64_t>(swc_winograd2x2_weight_pieces_bytes(as_int(C), as_int(K)))}, at::kByte);
            st = swc_winograd2x2_weight_pieces(floats(*W), pieces.mutable_data_ptr(), as_int(C), as_int(K), stream);
        }
        if (st == SWC_OK && pieces.defined())
            st = (bf16 ? swc_winograd2x2_conv_prepared_bf16 : swc_winograd2x2_conv_prepared)(
                floats(*I), floats(*W), pieces.const_data_ptr(), floats_of(out), scale, shift, residual, residual_relu, as_int(C), as_int(B),
                as_int(nH), as_int(nW), as_int(K), 1, 1, stream);
        else if (st == SWC_OK)
            st = swc_winograd2x2_conv_epilogue(floats(*I), floats(*W), floats_of(out), scale, shift, residual, residual_relu, as_int(C), as_int(B),
                                               as_int(nH), as_int(nW), as_int(K), 1, 1, bf16, stream);
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// pieces_gain(I, K, bf16 operands): swc_winograd2x2_conv_pieces_gain or its bf16 sibling for I [16,B,nH,nW,C], 0 where that is not I's shape
PyObject *pieces_gain(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(3)
    const long K = PyLong_AsLong(args[1]);
    if (K == -1 && PyErr_Occurred()) return nullptr;
    const at::Tensor *I = plain(args[0], at::kFloat, 5);
    const int bf16 = PyObject_IsTrue(args[2]);
    if (bf16 < 0) return nullptr;
    if (I == nullptr || I->size(0) != 16 || !fits(I->sizes()) || !fits({K})) return PyLong_FromLong(0);
    const c10::DeviceGuard guard(I->device());
    return PyLong_FromLong((bf16 ? swc_winograd2x2_conv_pieces_bf16_gain : swc_winograd2x2_conv_pieces_gain)(
        as_int(I->size(4)), as_int(I->size(1)), as_int(I->size(2)), as_int(I->size(3)), as_int(K)));
    END_HANDLE_TH_ERRORS
}

// conv_stored(I bf16, W16 [16,K,C] bf16, scale, shift, residual, residual_relu, workspace)
PyObject *conv_stored(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(7)
    const at::Tensor *I = plain(args[0], at::kBFloat16, 5), *W = plain(args[1], at::kBFloat16, 3);
    if (I == nullptr || W == nullptr || watched() || records(*I) || records(*W) || I->device() != W->device()) return none();
    const int64_t B = I->size(1), nH = I->size(2), nW = I->size(3), C = I->size(4), K = W->size(1);
    if (I->size(0) != 16 || W->size(0) != 16 || W->size(2) != C || !fits(I->sizes()) || !fits(W->sizes())) return none();
    bool ok = (args[2] == Py_None) == (args[3] == Py_None);
    const bool residual_relu = truth(args[5], &ok), workspace = truth(args[6], &ok);
    const float *scale = optional(args[2], *I, {K}, &ok), *shift = optional(args[3], *I, {K}, &ok),
                *residual = optional(args[4], *I, {B, 2 * nH, 2 * nW, K}, &ok);
    if (!ok) return none();
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(I->device());
        out = make(*I, {B, 2 * nH, 2 * nW, K});
        const size_t floats_needed =
            workspace ? swc_winograd2x2_conv_bf16in_workspace_floats(as_int(C), as_int(B), as_int(nH), as_int(nW), as_int(K)) : 0;
        at::Tensor tmp;
        if (floats_needed > 0) tmp = make(*I, {static_cast<int64_t>(floats_needed)});
        st = swc_winograd2x2_conv_bf16in_ws(shorts(*I), shorts(*W), floats_of(out), scale, shift, residual, residual_relu,
                                            tmp.defined() ? floats_of(tmp) : nullptr, floats_needed, as_int(C), as_int(B), as_int(nH), as_int(nW),
                                            as_int(K), 1, 1, stream_of(*I));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// conv_grad(I, W, grad) -> (dI, dW)
PyObject *conv_grad(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(3)
    const at::Tensor *I = plain(args[0], at::kFloat, 5), *W = plain(args[1], at::kFloat, 3), *G = plain(args[2], at::kFloat, 4);
    if (I == nullptr || W == nullptr || G == nullptr || watched() || I->device() != W->device() || I->device() != G->device()) return none();
    const int64_t B = I->size(1), C = I->size(4), K = W->size(2);
    if (!fits(I->sizes()) || !fits(W->sizes()) || !fits(G->sizes())) return none();
    int64_t tmp_floats = 0, i_grad[5], w_grad[3];
    if (swc_winograd2x2_conv_grad_op_shape(5, I->sizes().data(), 3, W->sizes().data(), 4, G->sizes().data(), i_grad, w_grad, &tmp_floats) != SWC_OK)
        return none();
    at::Tensor dI, dW;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(I->device());
        dI = make(*I, I->sizes());
        dW = make(*I, W->sizes());
        at::Tensor tmp = make(*I, {tmp_floats});
        st = swc_winograd2x2_conv_grad(floats(*I), floats(*W), floats(*G), floats_of(dI), floats_of(dW), floats_of(tmp), nullptr, as_int(C), as_int(B),
                                       as_int(G->size(1)), as_int(G->size(2)), as_int(K), 1, 1, stream_of(*I));
    }
    if (st != SWC_OK) return none();
    PyObject *a = THPVariable_Wrap(std::move(dI)), *b = THPVariable_Wrap(std::move(dW));
    PyObject *pair = a != nullptr && b != nullptr ? PyTuple_Pack(2, a, b) : nullptr;
    Py_XDECREF(a);
    Py_XDECREF(b);
    return pair;
    END_HANDLE_TH_ERRORS
}

// imtrans_grad(grad, H, W, relu_input or None)
PyObject *imtrans_grad(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(4)
    const at::Tensor *G = plain(args[0], at::kFloat, 5);
    const long H = PyLong_AsLong(args[1]), W = PyLong_AsLong(args[2]);
    if ((H == -1 || W == -1) && PyErr_Occurred()) {   // beyond 64 bits
        PyErr_Clear();
        return none();
    }
    if (G == nullptr || watched() || G->size(0) != 16 || !fits(G->sizes()) || !fits({H, W})) return none();
    const int64_t B = G->size(1), C = G->size(4);
    bool ok = (H + 1) / 2 == G->size(2) && (W + 1) / 2 == G->size(3);
    const float *relu_input = optional(args[3], *G, {B, H, W, C}, &ok);
    if (!ok) return none();
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(G->device());
        out = make(*G, {B, H, W, C});
        if (relu_input != nullptr)
            st = swc_winograd2x2_imtrans_grad_relu_input(floats(*G), relu_input, floats_of(out), as_int(C), as_int(B), as_int(H), as_int(W), 1, 1,
                                                         stream_of(*G));
        else
            st = swc_winograd2x2_imtrans_grad(floats(*G), nullptr, floats_of(out), as_int(C), as_int(B), as_int(H), as_int(W), 1, 1, stream_of(*G));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// pointwise(x [B,H,W,C], w [K,C], relu, scale, shift)
PyObject *pointwise(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(5)
    const at::Tensor *x = plain(args[0], at::kFloat, 4), *w = plain(args[1], at::kFloat, 2);
    if (x == nullptr || w == nullptr || watched() || records(*x) || records(*w) || x->device() != w->device() || w->size(1) != x->size(3) ||
        !fits(x->sizes()) || !fits(w->sizes()))
        return none();
    bool ok = (args[3] == Py_None) == (args[4] == Py_None);
    const bool relu = truth(args[2], &ok);
    if (!relu && args[3] != Py_None) ok = false;
    const float *scale = optional(args[3], *x, {x->size(3)}, &ok), *shift = optional(args[4], *x, {x->size(3)}, &ok);
    if (!ok) return none();
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(x->device());
        out = make(*x, {x->size(0), x->size(1), x->size(2), w->size(0)});
        const int64_t rows = x->size(0) * x->size(1) * x->size(2);
        if (relu)
            st = swc_winograd2x2_relu_pointwise_conv(floats(*x), scale, shift, floats(*w), floats_of(out), as_int(x->size(3)), rows,
                                                     as_int(w->size(0)), stream_of(*x));
        else
            st = swc_winograd2x2_pointwise_conv(floats(*x), floats(*w), floats_of(out), as_int(x->size(3)), rows, as_int(w->size(0)), stream_of(*x));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

// max_pool(x [B,H,W,C]) and relu_mean(x [B,H,W,C])
template <bool POOL>
PyObject *pixels(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    SWC_ARGS(1)
    const at::Tensor *x = plain(args[0], at::kFloat, 4);
    if (x == nullptr || watched() || records(*x) || !fits(x->sizes())) return none();
    const int64_t B = x->size(0), H = x->size(1), W = x->size(2), C = x->size(3);
    at::Tensor out;
    int st;
    {
        NoGil nogil;
        const c10::DeviceGuard guard(x->device());
        out = POOL ? make(*x, {B, (H + 1) / 2, (W + 1) / 2, C}) : make(*x, {B, C});
        st = (POOL ? swc_max_pool_same : swc_relu_mean)(floats(*x), floats_of(out), as_int(C), as_int(B), as_int(H), as_int(W), stream_of(*x));
    }
    return st == SWC_OK ? THPVariable_Wrap(std::move(out)) : none();
    END_HANDLE_TH_ERRORS
}

using Fast = PyObject *(*)(PyObject *, PyObject *const *, Py_ssize_t);
PyMethodDef method(const char *name, Fast f)
{
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {method("key", key),
                         method("mark", mark),
                         method("kept", kept),
                         method("imtrans", imtrans),
                         method("conv", conv),
                         method("weight_pieces", weight_pieces),
                         method("pieces_gain", pieces_gain),
                         method("conv_stored", conv_stored),
                         method("conv_grad", conv_grad),
                         method("imtrans_grad", imtrans_grad),
                         method("pointwise", pointwise),
                         method("max_pool", pixels<true>),
                         method("relu_mean", pixels<false>),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_swc_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__swc_torch(void) { return PyModule_Create(&module_def); }
