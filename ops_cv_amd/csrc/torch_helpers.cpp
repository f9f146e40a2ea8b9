// Native side of the torch helpers in aclnn.py: both phases of an operator on torch tensors in one call from Python.
//
// The helpers used to build every aclTensor handle, array and output from Python through ctypes: 18 us of host time for
// a forward call, 31 to 39 us for a backward one, where the kernels of a small call run for 3 us (fp32 1x3x64x64 sampled
// at 32x32 points) and the library's own two phases take 3.  Here the operands' sizes and strides are read from the
// tensors directly, handles live for the call only, and nothing is kept from one call to the next.
//
// The functions are positional and internal to the package: aclnn.py holds the public signatures and their defaults.
#include <Python.h>

#include <optional>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "aclnn_grid_sampler2d.h"
#include "aclnn_grid_sampler2d_backward.h"
#include "aclnn_grid_sampler3d.h"
#include "aclnn_grid_sampler3d_backward.h"
#include "aclnn_resize.h"
#include "aclnn_upsample_bilinear_2d.h"
#include "aclnn_upsample_bilinear_2d_backward.h"

namespace {

PyObject* g_error_class = nullptr;  // aclnn.AclnnError, handed over when the module is first used

// A Python exception has been set.
struct Raised {};

[[noreturn]] void raise_status(const char* api, aclnnStatus st)
{
    PyObject* e = PyObject_CallFunction(g_error_class, "si", api, (int)st);
    if (e != nullptr) {
        PyErr_SetObject(g_error_class, e);
        Py_DECREF(e);
    }
    throw Raised();
}

const at::Tensor& tensor_arg(PyObject* o)
{
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a torch.Tensor, got %s", Py_TYPE(o)->tp_name);
        throw Raised();
    }
    return THPVariable_Unpack(o);
}

int64_t int_arg(PyObject* o)
{
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred() != nullptr) {
        throw Raised();
    }
    return v;
}

// int(o): what the extents of an array are made from where no tensor is allocated by them
int64_t whole_arg(PyObject* o)
{
    PyObject* whole = PyNumber_Long(o);
    if (whole == nullptr) {
        throw Raised();
    }
    const int64_t v = PyLong_AsLongLong(whole);
    Py_DECREF(whole);
    if (v == -1 && PyErr_Occurred() != nullptr) {
        throw Raised();
    }
    return v;
}

// float(o)
double float_arg(PyObject* o)
{
    PyObject* number = PyNumber_Float(o);
    if (number == nullptr) {
        throw Raised();
    }
    const double v = PyFloat_AS_DOUBLE(number);
    Py_DECREF(number);
    return v;
}

// int(v); not a number or infinite: ValueError, OverflowError
int64_t truncated(double v)
{
    PyObject* whole = PyLong_FromDouble(v);
    if (whole == nullptr) {
        throw Raised();
    }
    const int64_t t = PyLong_AsLongLong(whole);
    Py_DECREF(whole);
    if (t == -1 && PyErr_Occurred() != nullptr) {
        throw Raised();
    }
    return t;
}

bool bool_arg(PyObject* o)
{
    const int v = PyObject_IsTrue(o);
    if (v < 0) {
        throw Raised();
    }
    return v != 0;
}

// the elements of a Python sequence
template <typename T, typename F>
c10::SmallVector<T, 8> sequence_arg(PyObject* o, F&& one)
{
    PyObject* s = PySequence_Fast(o, "expected a sequence of numbers");
    if (s == nullptr) {
        throw Raised();
    }
    c10::SmallVector<T, 8> v;
    try {
        for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(s); i++) {
            v.push_back((T)one(PySequence_Fast_GET_ITEM(s, i)));
        }
    } catch (...) {
        Py_DECREF(s);
        throw;
    }
    Py_DECREF(s);
    return v;
}

// the extents of a tensor; `allocates`: those of an output that the call allocates, which have to be integers, while
// those of one that the caller brings may be any numbers
c10::SmallVector<int64_t, 8> extents_arg(PyObject* o, bool allocates)
{
    return sequence_arg<int64_t>(o, allocates ? int_arg : whole_arg);
}

aclDataType dtype_of(const at::Tensor& t)
{
    switch (t.scalar_type()) {
        case at::kFloat: return ACL_FLOAT;
        case at::kHalf: return ACL_FLOAT16;
        case at::kBFloat16: return ACL_BF16;
        case at::kDouble: return ACL_DOUBLE;
        case at::kInt: return ACL_INT32;
        case at::kLong: return ACL_INT64;
        case at::kByte: return ACL_UINT8;
        case at::kChar: return ACL_INT8;
        case at::kShort: return ACL_INT16;
        case at::kBool: return ACL_BOOL;
        default: break;
    }
    PyErr_SetString(PyExc_KeyError, c10::toString(t.scalar_type()));
    throw Raised();
}

// The stream of a call on the device `like`: the caller's, or PyTorch's current one where the caller named none.
//
// The caching allocator orders the reuse of a block by the stream that the block was allocated for.  A stream that is not
// the current one is therefore made current for the call, so that the workspace and the outputs come from its own pool:
// nothing on another stream still uses them, and they go back to work that runs behind the call's kernels.  The caller's
// tensors are noted as in use on that stream, the outputs that the call made as in use on the caller's current one.
class Queue {
public:
    Queue(PyObject* stream, const at::Tensor& like)
    {
        if (!like.is_cuda()) {
            return;  // refused by Call::handle
        }
        if (stream == Py_None) {
            raw_ = c10::hip::getCurrentHIPStream().stream();
            return;
        }
        raw_ = (hipStream_t)int_arg(stream);
        current_ = c10::hip::getCurrentHIPStream(like.device().index());
        if (raw_ != current_->stream()) {
            own_ = c10::hip::getStreamFromExternal(raw_, like.device().index());
            c10::hip::setCurrentHIPStream(*own_);
        }
    }
    ~Queue()
    {
        if (own_) {
            c10::hip::setCurrentHIPStream(*current_);
        }
    }
    Queue(const Queue&) = delete;
    Queue& operator=(const Queue&) = delete;
    void* raw() const { return (void*)raw_; }
    // a tensor that the kernels of the call use; `made`: by the call, else the caller's
    void uses(const at::Tensor& t, bool made) const
    {
        if (own_ && t.is_cuda()) {
            c10::hip::HIPCachingAllocator::recordStream(t.storage().data_ptr(), made ? *current_ : *own_);
        }
    }

private:
    std::optional<c10::hip::HIPStream> current_, own_;
    hipStream_t raw_ = nullptr;
};

// The handles of one call, destroyed at its end.
class Call {
public:
    explicit Call(const Queue& queue) : queue_(queue) {}
    ~Call()
    {
        for (int i = 0; i < count_; i++) {
            aclDestroyTensor(handles_[i]);
        }
    }
    // aclTensor over the tensor's memory; strides and storage offset of the view are honoured.  `made`: an output that
    // the call allocated
    aclTensor* handle(const at::Tensor& t, aclFormat fmt = ACL_FORMAT_ND, bool made = false)
    {
        if (!t.is_cuda()) {
            PyErr_SetString(PyExc_RuntimeError, "ops_cv_amd needs device tensors: there is no CPU path");
            throw Raised();
        }
        // a copy-on-write tensor gets memory of its own first: an output must not be written through into the tensor it
        // was cloned from, and memory shared that way is not the allocator's to note as in use
        void* const base = t.storage().mutable_data();
        queue_.uses(t, made);
        const int64_t storage = (int64_t)(t.storage().nbytes() / t.element_size());
        aclTensor* h = aclCreateTensor(t.sizes().data(), (uint64_t)t.dim(), dtype_of(t), t.strides().data(),
                                       t.storage_offset(), fmt, &storage, 1, base);
        if (h != nullptr) {
            handles_[count_++] = h;
        }
        return h;
    }

private:
    const Queue& queue_;
    aclTensor* handles_[5];
    int count_ = 0;
};

// Second phase: the workspace (the caller's where it is large enough) and the launch on the stream.
void launch(const char* api, aclnnStatus (*phase2)(void*, uint64_t, aclOpExecutor*, aclrtStream), uint64_t bytes,
            aclOpExecutor* ex, const at::Tensor& like, PyObject* workspace, const Queue& queue)
{
    at::Tensor ws;
    void* at = nullptr;
    try {
        if (bytes > 0) {
            if (workspace != Py_None) {
                ws = tensor_arg(workspace);
            }
            if (!ws.defined() || (uint64_t)ws.nbytes() < bytes) {
                ws = at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
                at = ws.mutable_data_ptr();
            } else {
                at = ws.mutable_data_ptr();  // before it is noted, as in Call::handle
                queue.uses(ws, false);
            }
        }
    } catch (...) {
        aclDestroyAclOpExecutor(ex);
        throw;
    }
    const uint64_t size = bytes > 0 ? (uint64_t)ws.nbytes() : 0u;
    aclnnStatus st;
    // a launch may wait for room in the stream's queue: other Python threads go on meanwhile
    Py_BEGIN_ALLOW_THREADS
    st = phase2(at, size, ex, queue.raw());
    Py_END_ALLOW_THREADS
    if (st != ACLNN_SUCCESS) {
        raise_status(api, st);
    }
}

int64_t size_of(const at::Tensor& t, int64_t dim)
{
    if (dim >= t.dim()) {
        PyErr_SetString(PyExc_IndexError, "tuple index out of range");
        throw Raised();
    }
    return t.sizes()[dim];
}

typedef c10::SmallVector<int64_t, 8> Sizes;

// The caller's output, or one of the sizes that `sizes` gives.  They are asked for only then: operands of too few
// dimensions beside a given output are the library's to refuse.
template <typename F>
at::Tensor out_arg(PyObject* out, const at::Tensor& like, F&& sizes, PyObject* dtype = Py_None)
{
    if (out != Py_None) {
        return tensor_arg(out);
    }
    at::TensorOptions options = like.options().memory_format(at::MemoryFormat::Contiguous);
    if (dtype != Py_None) {
        if (!THPDtype_Check(dtype)) {
            PyErr_Format(PyExc_TypeError, "expected a torch.dtype, got %s", Py_TYPE(dtype)->tp_name);
            throw Raised();
        }
        options = options.dtype(reinterpret_cast<THPDtype*>(dtype)->scalar_type);
    }
    return at::empty(sizes(), options);
}

template <typename F>
PyObject* guarded(Py_ssize_t nargs, Py_ssize_t want, F&& body)
{
    HANDLE_TH_ERRORS
    if (nargs != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, nargs);
        return nullptr;
    }
    try {
        return body();
    } catch (const Raised&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// (inp, grid, interpolation, padding, align, out, workspace, stream)
PyObject* grid_sampler2d(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 8, [&]() -> PyObject* {
        const at::Tensor& x = tensor_arg(a[0]);
        const at::Tensor& g = tensor_arg(a[1]);
        const Queue queue(a[7], x);
        const at::Tensor y = out_arg(a[5], x, [&] {
            return Sizes{size_of(x, 0), size_of(x, 1), size_of(g, 1), size_of(g, 2)};
        });
        Call c(queue);
        aclTensor *hx = c.handle(x), *hg = c.handle(g), *hy = c.handle(y, ACL_FORMAT_ND, a[5] == Py_None);
        uint64_t ws = 0;
        aclOpExecutor* ex = nullptr;
        const aclnnStatus st = aclnnGridSampler2DGetWorkspaceSize(hx, hg, int_arg(a[2]), int_arg(a[3]), bool_arg(a[4]), hy,
                                                                  &ws, &ex);
        if (st != ACLNN_SUCCESS) {
            raise_status("aclnnGridSampler2DGetWorkspaceSize", st);
        }
        launch("aclnnGridSampler2D", aclnnGridSampler2D, ws, ex, x, a[6], queue);
        return THPVariable_Wrap(y);
    });
}

// (inp, grid, interpolation, padding, align, out, workspace, stream, channels_last)
PyObject* grid_sampler3d(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 9, [&]() -> PyObject* {
        const at::Tensor& x = tensor_arg(a[0]);
        const at::Tensor& g = tensor_arg(a[1]);
        const bool last = bool_arg(a[8]);
        const aclFormat fmt = last ? ACL_FORMAT_NDHWC : ACL_FORMAT_NCDHW;
        const Queue queue(a[7], x);
        const at::Tensor y = out_arg(a[5], x, [&] {
            const int64_t n = size_of(x, 0), d = size_of(g, 1), h = size_of(g, 2), w = size_of(g, 3);
            return last ? Sizes{n, d, h, w, size_of(x, 4)} : Sizes{n, size_of(x, 1), d, h, w};
        });
        Call c(queue);
        aclTensor *hx = c.handle(x, fmt), *hg = c.handle(g), *hy = c.handle(y, fmt, a[5] == Py_None);
        uint64_t ws = 0;
        aclOpExecutor* ex = nullptr;
        const aclnnStatus st = aclnnGridSampler3DGetWorkspaceSize(hx, hg, int_arg(a[2]), int_arg(a[3]), bool_arg(a[4]), hy,
                                                                  &ws, &ex);
        if (st != ACLNN_SUCCESS) {
            raise_status("aclnnGridSampler3DGetWorkspaceSize", st);
        }
        launch("aclnnGridSampler3D", aclnnGridSampler3D, ws, ex, x, a[6], queue);
        return THPVariable_Wrap(y);
    });
}

// (grad_out, inp, grid, interpolation, padding, align, output_mask, input_grad, grid_grad, workspace, stream,
// channels_last) of either backward
typedef aclnnStatus (*backward_phase1)(const aclTensor*, const aclTensor*, const aclTensor*, int64_t, int64_t, bool,
                                       const aclBoolArray*, aclTensor*, aclTensor*, uint64_t*, aclOpExecutor**);
typedef aclnnStatus (*backward_phase2)(void*, uint64_t, aclOpExecutor*, aclrtStream);

PyObject* sampler_backward(PyObject* const* a, bool volume, const char* api1, backward_phase1 phase1, const char* api2,
                           backward_phase2 phase2)
{
    const at::Tensor& go = tensor_arg(a[0]);
    const at::Tensor& x = tensor_arg(a[1]);
    const at::Tensor& g = tensor_arg(a[2]);
    const Queue queue(a[10], x);
    const at::Tensor dx = (a[7] == Py_None) ? at::empty_like(x) : tensor_arg(a[7]);
    const at::Tensor dg = (a[8] == Py_None) ? at::empty_like(g) : tensor_arg(a[8]);
    const aclFormat fmt = !volume ? ACL_FORMAT_ND : (bool_arg(a[11]) ? ACL_FORMAT_NDHWC : ACL_FORMAT_NCDHW);
    const auto flags = sequence_arg<bool>(a[6], bool_arg);
    Call c(queue);
    aclTensor *hgo = c.handle(go, fmt), *hx = c.handle(x, fmt), *hg = c.handle(g),
              *hdx = c.handle(dx, fmt, a[7] == Py_None), *hdg = c.handle(dg, ACL_FORMAT_ND, a[8] == Py_None);
    const int64_t interp = int_arg(a[3]), pad = int_arg(a[4]);
    const bool align = bool_arg(a[5]);
    aclBoolArray* mask = aclCreateBoolArray(flags.data(), flags.size());
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    const aclnnStatus st = phase1(hgo, hx, hg, interp, pad, align, mask, hdx, hdg, &ws, &ex);
    aclDestroyBoolArray(mask);
    if (st != ACLNN_SUCCESS) {
        raise_status(api1, st);
    }
    launch(api2, phase2, ws, ex, x, a[9], queue);
    PyObject* pair = PyTuple_New(2);
    if (pair == nullptr) {
        throw Raised();
    }
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(dx));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(dg));
    return pair;
}

PyObject* grid_sampler2d_backward(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 12, [&]() -> PyObject* {
        return sampler_backward(a, false, "aclnnGridSampler2DBackwardGetWorkspaceSize",
                                aclnnGridSampler2DBackwardGetWorkspaceSize, "aclnnGridSampler2DBackward",
                                aclnnGridSampler2DBackward);
    });
}

PyObject* grid_sampler3d_backward(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 12, [&]() -> PyObject* {
        return sampler_backward(a, true, "aclnnGridSampler3DBackwardGetWorkspaceSize",
                                aclnnGridSampler3DBackwardGetWorkspaceSize, "aclnnGridSampler3DBackward",
                                aclnnGridSampler3DBackward);
    });
}

// (self, output_size, align, scales_h, scales_w, out, workspace, stream, channels_last)
PyObject* upsample_bilinear2d(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 9, [&]() -> PyObject* {
        const at::Tensor& x = tensor_arg(a[0]);
        const auto size = extents_arg(a[1], a[5] == Py_None);
        const bool last = bool_arg(a[8]);
        const aclFormat fmt = last ? ACL_FORMAT_NHWC : ACL_FORMAT_NCHW;
        const Queue queue(a[7], x);
        const at::Tensor y = out_arg(a[5], x, [&] {
            if (size.size() < 2) {
                PyErr_SetString(PyExc_IndexError, "output_size holds two extents");
                throw Raised();
            }
            return last ? Sizes{size_of(x, 0), size[0], size[1], size_of(x, 3)}
                        : Sizes{size_of(x, 0), size_of(x, 1), size[0], size[1]};
        });
        Call c(queue);
        aclTensor *hx = c.handle(x, fmt), *hy = c.handle(y, fmt, a[5] == Py_None);
        const bool align = bool_arg(a[2]);
        const double sh = float_arg(a[3]), sw = float_arg(a[4]);
        aclIntArray* hs = aclCreateIntArray(size.data(), size.size());
        uint64_t ws = 0;
        aclOpExecutor* ex = nullptr;
        const aclnnStatus st = aclnnUpsampleBilinear2dGetWorkspaceSize(hx, hs, align, sh, sw, hy, &ws, &ex);
        aclDestroyIntArray(hs);
        if (st != ACLNN_SUCCESS) {
            raise_status("aclnnUpsampleBilinear2dGetWorkspaceSize", st);
        }
        launch("aclnnUpsampleBilinear2d", aclnnUpsampleBilinear2d, ws, ex, x, a[6], queue);
        return THPVariable_Wrap(y);
    });
}

// (self, scales, mode, out, workspace, stream, channels_last)
PyObject* resize(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 7, [&]() -> PyObject* {
        const at::Tensor& x = tensor_arg(a[0]);
        const auto scales64 = sequence_arg<double>(a[1], float_arg);
        const char* mode = PyUnicode_AsUTF8(a[2]);
        if (mode == nullptr) {
            throw Raised();
        }
        const bool last = bool_arg(a[6]);
        const aclFormat fmt = last ? ACL_FORMAT_NHWC : ACL_FORMAT_NCHW;
        const Queue queue(a[5], x);
        const at::Tensor y = out_arg(a[3], x, [&] {
            Sizes sizes(x.sizes().begin(), x.sizes().end());
            for (const int64_t d : {last ? 1 : 2, last ? 2 : 3}) {
                if (d >= x.dim() || d >= (int64_t)scales64.size()) {
                    PyErr_SetString(PyExc_IndexError, "list index out of range");
                    throw Raised();
                }
                sizes[d] = truncated((double)sizes[d] * scales64[d]);
            }
            return sizes;
        });
        Call c(queue);
        aclTensor *hx = c.handle(x, fmt), *hy = c.handle(y, fmt, a[3] == Py_None);
        c10::SmallVector<float, 8> scales(scales64.begin(), scales64.end());
        aclFloatArray* hs = aclCreateFloatArray(scales.data(), scales.size());
        uint64_t ws = 0;
        aclOpExecutor* ex = nullptr;
        const aclnnStatus st = aclnnResizeGetWorkspaceSize(hx, hs, mode, hy, &ws, &ex);
        aclDestroyFloatArray(hs);
        if (st != ACLNN_SUCCESS) {
            raise_status("aclnnResizeGetWorkspaceSize", st);
        }
        launch("aclnnResize", aclnnResize, ws, ex, x, a[4], queue);
        return THPVariable_Wrap(y);
    });
}

// (grad_out, input_size, align, scales_h, scales_w, out, workspace, stream, channels_last, out_dtype)
PyObject* upsample_bilinear2d_backward(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return guarded(n, 10, [&]() -> PyObject* {
        const at::Tensor& go = tensor_arg(a[0]);
        const auto isize = extents_arg(a[1], a[5] == Py_None);
        const bool last = bool_arg(a[8]);
        const aclFormat fmt = last ? ACL_FORMAT_NHWC : ACL_FORMAT_NCHW;
        const Queue queue(a[7], go);
        const at::Tensor y = out_arg(a[5], go, [&] { return isize; }, a[9]);
        const int64_t osize[2] = {size_of(go, last ? 1 : 2), size_of(go, last ? 2 : 3)};
        Call c(queue);
        aclTensor *hgo = c.handle(go, fmt), *hy = c.handle(y, fmt, a[5] == Py_None);
        const bool align = bool_arg(a[2]);
        const double sh = float_arg(a[3]), sw = float_arg(a[4]);
        aclIntArray* ho = aclCreateIntArray(osize, 2);
        aclIntArray* hi = aclCreateIntArray(isize.data(), isize.size());
        uint64_t ws = 0;
        aclOpExecutor* ex = nullptr;
        const aclnnStatus st =
            aclnnUpsampleBilinear2dBackwardGetWorkspaceSize(hgo, ho, hi, align, sh, sw, hy, &ws, &ex);
        aclDestroyIntArray(ho);
        aclDestroyIntArray(hi);
        if (st != ACLNN_SUCCESS) {
            raise_status("aclnnUpsampleBilinear2dBackwardGetWorkspaceSize", st);
        }
        launch("aclnnUpsampleBilinear2dBackward", aclnnUpsampleBilinear2dBackward, ws, ex, go, a[6], queue);
        return THPVariable_Wrap(y);
    });
}

// (AclnnError): the class of the errors raised for a status other than success
PyObject* set_error_class(PyObject*, PyObject* cls)
{
    Py_INCREF(cls);
    Py_XSETREF(g_error_class, cls);
    Py_RETURN_NONE;
}

#define OPSCV_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {OPSCV_FAST(grid_sampler2d),
                          OPSCV_FAST(grid_sampler3d),
                          OPSCV_FAST(grid_sampler2d_backward),
                          OPSCV_FAST(grid_sampler3d_backward),
                          OPSCV_FAST(upsample_bilinear2d),
                          OPSCV_FAST(upsample_bilinear2d_backward),
                          OPSCV_FAST(resize),
                          {"set_error_class", set_error_class, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_helpers", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_helpers() { return PyModule_Create(&kModule); }
