// Python's way into the operator library for torch tensors: one builtin function per operator, generated from the
// operator's own prototype.
//
// What bounds a small call is the host.  Through ctypes a call of seven tensors took 45-65 us: a heap handle, two shape arrays
// and a foreign call for each tensor, and two event hops between torch's stream and a context's own, which also left the
// device idle between calls.  Here a tensor becomes a handle on the C++ stack that borrows torch's own shape and stride
// arrays, the operator is called directly, and without an explicit context it runs on torch's current stream, where
// everything before and after it is already in order.  Four calls of a decode step over one sequence of 700 tokens, 32 heads
// of 128: 259 -> 18.9 us (17 of them kernels); over 64 sequences of 512..2048 tokens 308 -> 226 us; RMSNorm forward and
// backward in bf16 [1237, 5120]: 144 -> 24 us.
//
// A function takes the context first: None for torch's current stream, with scratch from torch's caching allocator (which
// keeps a block in that stream's order, bounds what it holds and is safe with any number of threads), or the address of a
// context made by diopirtContextCreate.  Tensors may be None (a null handle).  The answer is the operator's return code; an
// operator with an int64_t* in its prototype answers (code, value after the call).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/core/Allocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <atomic>
#include <tuple>
#include <utility>

#include <diopi/functions_ext.h>
#include <diopi/functions_lmdeploy.h>

#include "handles.hpp"

namespace {

bool dtypeOf(c10::ScalarType s, diopiDtype_t* dtype) {
    switch (s) {
        case c10::ScalarType::Char: *dtype = diopi_dtype_int8; return true;
        case c10::ScalarType::Byte: *dtype = diopi_dtype_uint8; return true;
        case c10::ScalarType::Short: *dtype = diopi_dtype_int16; return true;
        case c10::ScalarType::Int: *dtype = diopi_dtype_int32; return true;
        case c10::ScalarType::Long: *dtype = diopi_dtype_int64; return true;
        case c10::ScalarType::Half: *dtype = diopi_dtype_float16; return true;
        case c10::ScalarType::Float: *dtype = diopi_dtype_float32; return true;
        case c10::ScalarType::Double: *dtype = diopi_dtype_float64; return true;
        case c10::ScalarType::Bool: *dtype = diopi_dtype_bool; return true;
        case c10::ScalarType::BFloat16: *dtype = diopi_dtype_bfloat16; return true;
        default: return false;
    }
}

// Scratch of the calls on torch's current stream, all threads together, in blocks as a context's pool counts them.
std::atomic<int64_t> scratchInUse{0}, scratchPeak{0};

// The context of one call on torch's current stream.  Its scratch goes back to torch's allocator when the call has
// queued its work; a later owner on this stream is ordered behind it.
struct CurrentStreamContext final : diopiContext {
    struct Scratch {
        diopiTensor* tensor;
        c10::DataPtr memory;
    };
    std::vector<Scratch> scratch;
    int64_t held = 0;

    hipStream_t getStream() override { return c10::hip::getCurrentHIPStream().stream(); }

    diopiTensor* keepScratch(diopiTensor* t, int64_t bytes) override {
        try {
            const auto where = t->device == diopi_device ? c10::DeviceType::CUDA : c10::DeviceType::CPU;
            c10::DataPtr memory = c10::GetAllocator(where)->allocate(bytes > 0 ? static_cast<size_t>(bytes) : 1);
            t->data = memory.get();
            if (t->data == nullptr) return nullptr;
            scratch.push_back({t, std::move(memory)});
            const int64_t block = (bytes > 0 ? bytes + 1023 : 1024) / 1024 * 1024;
            held += block;
            const int64_t now = scratchInUse.fetch_add(block) + block;
            for (int64_t peak = scratchPeak.load(); peak < now && !scratchPeak.compare_exchange_weak(peak, now);) {
            }
            return t;
        } catch (const std::exception&) {
            return nullptr;  // out of memory: the operator reports that its scratch was refused
        }
    }

    ~CurrentStreamContext() override {
        for (auto& s : scratch) delete s.tensor;
        scratchInUse.fetch_sub(held);
    }
};

// ---- one argument of an operator: take() from Python, get() for the call ----
template <typename P>
struct Arg;

struct TensorArg {
    diopiTensor tensor;
    diopiTensor* handle = nullptr;
    bool take(PyObject* o) {
        if (o == Py_None) return true;
        if (!THPVariable_Check(o)) {
            PyErr_Format(PyExc_TypeError, "expected a torch.Tensor or None, got %s", Py_TYPE(o)->tp_name);
            return false;
        }
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!dtypeOf(t.scalar_type(), &tensor.dtype)) {
            PyErr_Format(PyExc_TypeError, "unsupported dtype %s", c10::toString(t.scalar_type()));
            return false;
        }
        const auto sizes = t.sizes();
        tensor.shape = sizes.data();
        tensor.stride = t.strides().data();
        tensor.ndim = static_cast<int64_t>(sizes.size());
        tensor.numel = t.numel();
        tensor.device = t.is_cuda() ? diopi_device : diopi_host;
        tensor.data = tensor.numel > 0 ? t.data_ptr() : nullptr;
        handle = &tensor;
        return true;
    }
};
template <>
struct Arg<diopiTensorHandle_t> : TensorArg {
    diopiTensorHandle_t get() { return handle; }
};
template <>
struct Arg<diopiConstTensorHandle_t> : TensorArg {
    diopiConstTensorHandle_t get() { return handle; }
};
template <>
struct Arg<diopiGeneratorHandle_t> {
    bool take(PyObject* o) {
        if (o != Py_None) PyErr_SetString(PyExc_TypeError, "no operator here takes a generator: pass None");
        return o == Py_None;
    }
    diopiGeneratorHandle_t get() { return nullptr; }
};
template <>
struct Arg<bool> {
    bool value = false;
    bool take(PyObject* o) {
        const int truth = PyObject_IsTrue(o);
        value = truth == 1;
        return truth >= 0;
    }
    bool get() { return value; }
};
template <typename I>
struct IntArg {
    I value = 0;
    bool take(PyObject* o) {
        const long long v = PyLong_AsLongLong(o);
        value = static_cast<I>(v);
        return !(v == -1 && PyErr_Occurred());
    }
    I get() { return value; }
};
template <>
struct Arg<int32_t> : IntArg<int32_t> {};
template <>
struct Arg<int64_t> : IntArg<int64_t> {};
template <>
struct Arg<int64_t*> : IntArg<int64_t> {
    int64_t* get() { return &value; }
};
template <typename F>
struct FloatArg {
    F value = 0;
    bool take(PyObject* o) {
        const double v = PyFloat_AsDouble(o);
        value = static_cast<F>(v);
        return !(v == -1.0 && PyErr_Occurred());
    }
    F get() { return value; }
};
template <>
struct Arg<float> : FloatArg<float> {};
template <>
struct Arg<double> : FloatArg<double> {};
template <>
struct Arg<diopiSize_t> {
    std::vector<int64_t> values;
    bool take(PyObject* o) {
        PyObject* seq = PySequence_Fast(o, "expected a sequence of integers");
        if (seq == nullptr) return false;
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
        values.resize(n > 0 ? n : 1);
        bool ok = true;
        for (Py_ssize_t i = 0; ok && i < n; ++i) {
            PyObject* index = PyNumber_Long(PySequence_Fast_GET_ITEM(seq, i));
            ok = index != nullptr;
            if (ok) values[i] = PyLong_AsLongLong(index);
            Py_XDECREF(index);
            ok = ok && !(values[i] == -1 && PyErr_Occurred());
        }
        len = n;
        Py_DECREF(seq);
        return ok;
    }
    int64_t len = 0;
    diopiSize_t get() { return diopiSize_t{values.data(), len}; }
};

template <typename P>
PyObject* pointedTo(Arg<P>&) {
    return nullptr;
}
PyObject* pointedTo(Arg<int64_t*>& a) { return PyLong_FromLongLong(a.value); }

// ---- one operator ----
template <auto Fn>
struct Operator;

template <typename... P, diopiError_t (*Fn)(diopiContextHandle_t, P...)>
struct Operator<Fn> {
    template <size_t... I>
    static PyObject* call(PyObject* const* args, std::index_sequence<I...>) {
        std::tuple<Arg<P>...> a;
        if (!(std::get<I>(a).take(args[I + 1]) && ...)) return nullptr;
        diopiError_t code = diopiErrorOccurred;
        if (args[0] == Py_None) {
            CurrentStreamContext ctx;
            Py_BEGIN_ALLOW_THREADS
            code = Fn(&ctx, std::get<I>(a).get()...);
            Py_END_ALLOW_THREADS
        } else {
            auto* ctx = static_cast<diopiContextHandle_t>(PyLong_AsVoidPtr(args[0]));
            if (ctx == nullptr && PyErr_Occurred()) return nullptr;
            Py_BEGIN_ALLOW_THREADS
            code = Fn(ctx, std::get<I>(a).get()...);
            Py_END_ALLOW_THREADS
        }
        if constexpr ((std::is_same<P, int64_t*>::value || ...)) {
            PyObject* value = nullptr;
            ((value = value != nullptr ? value : pointedTo(std::get<I>(a))), ...);
            return Py_BuildValue("iN", static_cast<int>(code), value);
        } else {
            return PyLong_FromLong(code);
        }
    }

    static PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
        if (n != static_cast<Py_ssize_t>(sizeof...(P)) + 1) {
            PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", static_cast<Py_ssize_t>(sizeof...(P)) + 1, n);
            return nullptr;
        }
        try {
            return call(args, std::index_sequence_for<P...>{});
        } catch (const std::exception& e) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
            return nullptr;
        }
    }
};

PyObject* scratchPeakOf(PyObject*, PyObject*) { return PyLong_FromLongLong(scratchPeak.load()); }

#define DIOPI_BOUND(name) \
    { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Operator<&name>::entry)), METH_FASTCALL, nullptr }
PyMethodDef kMethods[] = {
    DIOPI_BOUND(diopiRotaryEmbedding),
    DIOPI_BOUND(diopiRotaryEmbeddingV2),
    DIOPI_BOUND(diopiApplyPenalty),
    DIOPI_BOUND(diopiApplyPenaltyV2),
    DIOPI_BOUND(diopiRMSNorm),
    DIOPI_BOUND(diopiRMSNormBackward),
    DIOPI_BOUND(diopiDestIndexCopyKV),
    DIOPI_BOUND(diopiTokenAttentionInference),
    DIOPI_BOUND(diopiTokenSoftmaxReduceVInference),
    DIOPI_BOUND(diopiContextAttentionInference),
    DIOPI_BOUND(diopiContextAttentionInferenceNoAlloc),
    DIOPI_BOUND(diopiFlashAttentionVarLen),
    DIOPI_BOUND(diopiFlashAttention),
    DIOPI_BOUND(diopiMultiHeadAttention),
    DIOPI_BOUND(diopiMultiHeadAttentionVarLen),
    DIOPI_BOUND(diopiPagedAttention),
    DIOPI_BOUND(diopiPromptFlashAttention),
    DIOPI_BOUND(diopiRootMeanSquareNormInp),
    DIOPI_BOUND(diopiFusedAddRootMeanSquareNormInp),
    DIOPI_BOUND(diopiFusedDecoderAttentionInp),
    {"scratch_peak", scratchPeakOf, METH_NOARGS, "Most bytes of scratch that calls on torch's current stream have held at a time."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "diopi_torch", "The DIOPI operators on torch tensors.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_diopi_torch(void) { return PyModule_Create(&kModule); }
