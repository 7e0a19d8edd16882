// The operators on PyTorch tensors: what lies between a Python call and the C ABI (include/mxd_msda.h) -- reading the
// tensors, allocating results and workspace, the launch on the current stream and the autograd node -- in C++.
//
// Bound by the host: a decoder call of 300 queries keeps the GPU busy for 6 us, and the same steps in Python (an autograd
// Function, a ctypes call with 15 arguments) took 22 us per call (now 6.3, what the kernel takes), 900 queries of two images 171 us
// with the backward (now 63).
//
// Three functions per operator, all of which return None for anything but plain inputs (GPU tensors of one device and
// of the dtypes, shapes and contiguous layout that the kernels read): drivingsdk_amd/_C.py then checks, names what is
// wrong or brings the tensors into that form.
//   <op>(...)           with autograd; also None where Python's own autograd Function has to see the call (autocast,
//                       functorch transforms, dispatch modes, tensor subclasses, tracing)
//   <op>_forward(...)   the forward alone, into a tensor given behind the inputs or a new one
//   <op>_backward(...)  the gradients alone
// (PyTorch-ROCm presents its devices as "cuda": the guard and stream types that go with that are these)
#include <Python.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <array>

#include "../../include/mxd_msda.h"

namespace {

using at::Tensor;

// ---- what every operator needs -------------------------------------------------------------------------------------

int dtype_code(const Tensor& t)
{
    switch (t.scalar_type()) {
        case at::kFloat: return MXD_DTYPE_F32;
        case at::kHalf: return MXD_DTYPE_F16;
        case at::kBFloat16: return MXD_DTYPE_BF16;
        default: return -1;
    }
}

// An ordinary dense GPU tensor whose data can be handed to a kernel as it is.
bool plain(const Tensor& t)
{
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped);
}
bool plain(const Tensor& t, const Tensor& like)
{
    return plain(t) && t.is_contiguous() && t.device() == like.device();
}
bool plain(const Tensor& t, const Tensor& like, at::ScalarType type) { return plain(t, like) && t.scalar_type() == type; }

// Level metadata: [nl, 2] and [nl], both int32 or both int64 (returns the C ABI's flag for it), -1 otherwise.
int meta_flag(const Tensor& shapes, const Tensor& starts, int64_t levels, const Tensor& like)
{
    const at::ScalarType t = shapes.scalar_type();
    if ((t != at::kInt && t != at::kLong) || !plain(shapes, like) || !plain(starts, like, t)) return -1;
    if (shapes.dim() != 2 || shapes.size(0) != levels || shapes.size(1) != 2 || starts.numel() != levels) return -1;
    return t == at::kLong ? MXD_META_I64 : 0;
}

Tensor new_tensor(at::IntArrayRef size, const Tensor& like)
{
    return Tensor(at::detail::empty_cuda(size, like.scalar_type(), like.device(), std::nullopt));
}
Tensor new_like(const Tensor& t) { return new_tensor(t.sizes(), t); }

// The current stream of a tensor's device, and scratch memory from PyTorch's allocator: given back when the object goes,
// which the allocator orders behind the work enqueued on that stream.
struct Launch {
    explicit Launch(const Tensor& t) : guard(t.device()) {}
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
    c10::DataPtr memory;
    void* stream() const { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }
    void* scratch(size_t bytes)
    {
        memory = c10::hip::HIPCachingAllocator::get()->allocate(bytes < 16 ? 16 : bytes);
        return memory.get();
    }
};

void check(int rc) { TORCH_CHECK(rc == MXD_OK, mxd_msda_last_error()); }

const int32_t* meta(const Tensor& t) { return static_cast<const int32_t*>(t.data_ptr()); }

// The arguments of a call: tensors and numbers in the order of the Python call.
struct Args {
    std::array<Tensor, 6> t;
    std::array<int64_t, 3> i{};
    Tensor out;  // backward of an operator that keeps its result
};

// ---- the operators ---------------------------------------------------------------------------------------------------
// kGradOf: which tensors have gradients.  kFloat32: the tensor that is float32 whatever the others are (-1: none).  kKeepsOutput:
// the backward reads the result.  kOnce: gradients of gradients raise an error.  kFloat32InAutocast: autocast has the inputs cast to
// float32 (left to Python).  takes(): whether a call is in the form the kernels read, grad_output aside.

struct Msda {
    static constexpr const char* kNode = "MultiScaleDeformableAttnFunctionBackward";
    static constexpr int kTensors = 5, kInts = 0, kFloat32 = -1;
    static constexpr std::array<int, 3> kGradOf{0, 3, 4};
    static constexpr bool kKeepsOutput = false, kOnce = true, kFloat32InAutocast = true;
    static bool takes(const Args& a)
    {
        const Tensor &v = a.t[0], &loc = a.t[3], &attn = a.t[4];
        const at::ScalarType t = v.scalar_type();
        if (dtype_code(v) < 0 || !plain(v, v) || !plain(loc, v, t) || !plain(attn, v, t)) return false;
        if (v.dim() != 4 || loc.dim() != 6 || attn.dim() != 5 || a.t[1].dim() != 2) return false;
        const int64_t nl = a.t[1].size(0);
        return meta_flag(a.t[1], a.t[2], nl, v) >= 0 && v.size(3) <= 256 && loc.size(5) == 2 && loc.size(0) == v.size(0) &&
               loc.size(2) == v.size(2) && loc.size(3) >= nl && attn.sizes() == loc.sizes().slice(0, 5);
    }
    static Tensor new_output(const Args& a) { return new_tensor({a.t[3].size(0), a.t[3].size(1), a.t[0].size(2) * a.t[0].size(3)}, a.t[0]); }
    static void forward(const Args& a, Tensor& out)
    {
        const Tensor &v = a.t[0], &loc = a.t[3];
        Launch l(v);
        check(mxd_msda_forward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), loc.data_ptr(), a.t[4].data_ptr(), out.data_ptr(),
                               dtype_code(v) | meta_flag(a.t[1], a.t[2], a.t[1].size(0), v), v.size(0), v.size(1), v.size(2), v.size(3),
                               a.t[1].size(0), loc.size(3), loc.size(1), loc.size(4), l.stream()));
    }
    static void backward(const Args& a, const Tensor& grad, std::array<Tensor, 3>& g, unsigned)
    {
        const Tensor &v = a.t[0], &loc = a.t[3];
        const int code = dtype_code(v) | meta_flag(a.t[1], a.t[2], a.t[1].size(0), v);
        const int64_t bs = v.size(0), nk = v.size(1), nh = v.size(2), hd = v.size(3), nl = a.t[1].size(0), na = loc.size(3),
                      nq = loc.size(1), np = loc.size(4);
        Launch l(v);
        const size_t bytes = mxd_msda_backward_workspace_bytes(code, bs, nk, nh, hd, nl, na, nq, np);
        check(mxd_msda_backward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), loc.data_ptr(), a.t[4].data_ptr(), grad.data_ptr(),
                                g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr(), l.scratch(bytes), bytes, code, bs, nk, nh, hd, nl, na,
                                nq, np, 0, l.stream()));
    }
};

struct Fused {
    static constexpr const char* kNode = "MultiScaleDeformableAttnFusedFunctionBackward";
    static constexpr int kTensors = 6, kInts = 0, kFloat32 = -1;
    static constexpr std::array<int, 4> kGradOf{0, 3, 4, 5};
    static constexpr bool kKeepsOutput = true, kOnce = true, kFloat32InAutocast = true;
    static bool takes(const Args& a)
    {
        const Tensor &v = a.t[0], &ref = a.t[3], &off = a.t[4], &logits = a.t[5];
        const at::ScalarType t = v.scalar_type();
        if (dtype_code(v) < 0 || !plain(v, v) || !plain(ref, v, t) || !plain(off, v, t) || !plain(logits, v, t)) return false;
        if (v.dim() != 4 || off.dim() != 6 || ref.dim() != 4 || logits.dim() < 1) return false;
        const int64_t bs = v.size(0), nq = off.size(1), nl = off.size(3);
        return meta_flag(a.t[1], a.t[2], nl, v) >= 0 && v.size(3) <= 256 && off.size(5) == 2 && off.size(0) == bs &&
               off.size(2) == v.size(2) && ref.size(0) == bs && ref.size(1) == nq && ref.size(2) == nl &&
               (ref.size(3) == 2 || ref.size(3) == 4) && 2 * logits.numel() == off.numel() && logits.size(0) == bs;
    }
    static Tensor new_output(const Args& a) { return new_tensor({a.t[4].size(0), a.t[4].size(1), a.t[0].size(2) * a.t[0].size(3)}, a.t[0]); }
    static void forward(const Args& a, Tensor& out)
    {
        const Tensor &v = a.t[0], &ref = a.t[3], &off = a.t[4];
        Launch l(v);
        check(mxd_msda_fused_forward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), ref.data_ptr(), (int)ref.size(3), off.data_ptr(),
                                     a.t[5].data_ptr(), out.data_ptr(), dtype_code(v) | meta_flag(a.t[1], a.t[2], off.size(3), v), v.size(0),
                                     v.size(1), v.size(2), v.size(3), off.size(3), off.size(1), off.size(4), l.stream()));
    }
    static void backward(const Args& a, const Tensor& grad, std::array<Tensor, 4>& g, unsigned need)
    {
        const Tensor &v = a.t[0], &ref = a.t[3], &off = a.t[4];
        const int code = dtype_code(v) | meta_flag(a.t[1], a.t[2], off.size(3), v), want = (need >> 1) & 1, rd = (int)ref.size(3);
        const int64_t bs = v.size(0), nk = v.size(1), nh = v.size(2), hd = v.size(3), nl = off.size(3), nq = off.size(1), np = off.size(4);
        Launch l(v);
        const size_t bytes = mxd_msda_fused_backward_workspace_bytes(code, bs, nk, nh, hd, nl, nq, np, rd, want);
        check(mxd_msda_fused_backward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), ref.data_ptr(), rd, off.data_ptr(), a.t[5].data_ptr(),
                                      a.out.data_ptr(), grad.data_ptr(), g[0].data_ptr(), want ? g[1].data_ptr() : nullptr, g[2].data_ptr(),
                                      g[3].data_ptr(), l.scratch(bytes), bytes, code, bs, nk, nh, hd, nl, nq, np, 0, l.stream()));
    }
};

struct Dagg {
    static constexpr const char* kNode = "AdsDeformableAggregationBackward";
    static constexpr int kTensors = 5, kInts = 0, kFloat32 = -1;
    static constexpr std::array<int, 3> kGradOf{0, 3, 4};
    static constexpr bool kKeepsOutput = false, kOnce = false, kFloat32InAutocast = false;
    static bool takes(const Args& a)
    {
        const Tensor &f = a.t[0], &ss = a.t[1], &si = a.t[2], &loc = a.t[3], &w = a.t[4];
        const at::ScalarType t = f.scalar_type();
        if (dtype_code(f) < 0 || !plain(f, f) || !plain(loc, f, t) || !plain(w, f, t) || !plain(ss, f, at::kInt) || !plain(si, f, at::kInt))
            return false;
        if (f.dim() != 3 || ss.dim() != 3 || si.dim() != 2 || loc.dim() != 5 || w.dim() != 6) return false;
        const int64_t bs = f.size(0), A = w.size(1), P = w.size(2), cams = w.size(3), scales = w.size(4), G = w.size(5);
        return w.size(0) == bs && ss.sizes() == at::IntArrayRef({cams, scales, 2}) && si.sizes() == at::IntArrayRef({cams, scales}) &&
               loc.sizes() == at::IntArrayRef({bs, A, P, cams, 2}) && G > 0 && f.size(2) % G == 0;
    }
    static Tensor new_output(const Args& a) { return new_tensor({a.t[0].size(0), a.t[4].size(1), a.t[0].size(2)}, a.t[0]); }
    static void forward(const Args& a, Tensor& out)
    {
        const Tensor &f = a.t[0], &w = a.t[4];
        Launch l(f);
        check(mxd_dagg_forward(f.data_ptr(), meta(a.t[1]), meta(a.t[2]), a.t[3].data_ptr(), w.data_ptr(), out.data_ptr(), dtype_code(f),
                               f.size(0), f.size(1), f.size(2), w.size(3), w.size(4), w.size(1), w.size(2), w.size(5), l.stream()));
    }
    static void backward(const Args& a, const Tensor& grad, std::array<Tensor, 3>& g, unsigned)
    {
        const Tensor &f = a.t[0], &w = a.t[4];
        const int code = dtype_code(f);
        Launch l(f);
        const size_t bytes = mxd_dagg_backward_workspace_bytes(code, f.size(0), f.size(1), f.size(2), w.size(3), w.size(4), w.size(1),
                                                               w.size(2), w.size(5));
        check(mxd_dagg_backward(f.data_ptr(), meta(a.t[1]), meta(a.t[2]), a.t[3].data_ptr(), w.data_ptr(), grad.data_ptr(), g[0].data_ptr(),
                                g[1].data_ptr(), g[2].data_ptr(), l.scratch(bytes), bytes, code, f.size(0), f.size(1), f.size(2), w.size(3),
                                w.size(4), w.size(1), w.size(2), w.size(5), l.stream()));
    }
};

struct Gka {
    static constexpr const char* kNode = "GeometricKernelAttentionFuncBackward";
    static constexpr int kTensors = 5, kInts = 0, kFloat32 = 3;
    static constexpr std::array<int, 2> kGradOf{0, 4};
    static constexpr bool kKeepsOutput = false, kOnce = false, kFloat32InAutocast = false;
    static bool takes(const Args& a)
    {
        const Tensor &v = a.t[0], &loc = a.t[3], &attn = a.t[4];
        // (pixel indices travel as float32 whatever value's dtype is: exact below 2^24, where a 16-bit float is not)
        if (dtype_code(v) < 0 || !plain(v, v) || !plain(loc, v, at::kFloat) || !plain(attn, v, v.scalar_type())) return false;
        if (v.dim() != 4 || loc.dim() != 6 || attn.dim() != 5) return false;
        return meta_flag(a.t[1], a.t[2], loc.size(3), v) >= 0 && loc.size(5) == 2 && loc.size(0) == v.size(0) &&
               loc.size(2) == v.size(2) && attn.sizes() == loc.sizes().slice(0, 5);
    }
    static Tensor new_output(const Args& a) { return new_tensor({a.t[3].size(0), a.t[3].size(1), a.t[0].size(2) * a.t[0].size(3)}, a.t[0]); }
    static void forward(const Args& a, Tensor& out)
    {
        const Tensor &v = a.t[0], &loc = a.t[3];
        Launch l(v);
        check(mxd_gka_forward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), loc.data_ptr(), a.t[4].data_ptr(), out.data_ptr(),
                              dtype_code(v) | meta_flag(a.t[1], a.t[2], loc.size(3), v), v.size(0), v.size(1), v.size(2), v.size(3), loc.size(3), loc.size(1), loc.size(4), l.stream()));
    }
    static void backward(const Args& a, const Tensor& grad, std::array<Tensor, 2>& g, unsigned)
    {
        const Tensor &v = a.t[0], &loc = a.t[3];
        const int code = dtype_code(v) | meta_flag(a.t[1], a.t[2], loc.size(3), v);
        Launch l(v);
        const size_t bytes =
            mxd_gka_backward_workspace_bytes(code, v.size(0), v.size(1), v.size(2), v.size(3), loc.size(3), loc.size(1), loc.size(4));
        check(mxd_gka_backward(v.data_ptr(), meta(a.t[1]), meta(a.t[2]), loc.data_ptr(), a.t[4].data_ptr(), grad.data_ptr(), g[0].data_ptr(),
                               g[1].data_ptr(), l.scratch(bytes), bytes, code, v.size(0), v.size(1), v.size(2), v.size(3), loc.size(3),
                               loc.size(1), loc.size(4), l.stream()));
    }
};

struct Grid {
    static constexpr const char* kNode = "GridSampler2dV2FunctionBackward";
    static constexpr int kTensors = 2, kInts = 3, kFloat32 = -1;  // interpolation and padding mode, align_corners: see mxd_grid_sampler2d_forward
    static constexpr std::array<int, 2> kGradOf{0, 1};
    static constexpr bool kKeepsOutput = false, kOnce = true, kFloat32InAutocast = false;
    static bool takes(const Args& a)
    {
        const Tensor &x = a.t[0], &grid = a.t[1];
        if (dtype_code(x) < 0 || !plain(x, x) || !plain(grid, x, x.scalar_type()) || x.dim() != 4 || grid.dim() != 4) return false;
        return a.i[0] == 0 && (a.i[1] == 0 || a.i[1] == 1) && (a.i[2] == 0 || a.i[2] == 1) && grid.size(0) == x.size(0) && grid.size(3) == 2 &&
               mxd_grid_sampler2d_planes_fit(x.size(0), x.size(1), x.size(2), x.size(3), grid.size(1), grid.size(2));
    }
    static Tensor new_output(const Args& a) { return new_tensor({a.t[0].size(0), a.t[0].size(1), a.t[1].size(1), a.t[1].size(2)}, a.t[0]); }
    static void forward(const Args& a, Tensor& out)
    {
        const Tensor &x = a.t[0], &grid = a.t[1];
        Launch l(x);
        check(mxd_grid_sampler2d_planes_forward(x.data_ptr(), grid.data_ptr(), out.data_ptr(), dtype_code(x), x.size(0), x.size(1), x.size(2),
                                                x.size(3), grid.size(1), grid.size(2), (int)a.i[0], (int)a.i[1], (int)a.i[2], l.stream()));
    }
    static void backward(const Args& a, const Tensor& grad, std::array<Tensor, 2>& g, unsigned need)
    {
        const Tensor &x = a.t[0], &grid = a.t[1];
        const int code = dtype_code(x);
        if ((need & 3) == 0) return;
        Launch l(x);
        const size_t bytes = (need & 2) ? mxd_grid_sampler2d_planes_backward_workspace_bytes(code, x.size(0), x.size(1), x.size(2), x.size(3),
                                                                                              grid.size(1), grid.size(2))
                                        : 0;
        check(mxd_grid_sampler2d_planes_backward(grad.data_ptr(), x.data_ptr(), grid.data_ptr(), (need & 1) ? g[0].data_ptr() : nullptr,
                                                 (need & 2) ? g[1].data_ptr() : nullptr, l.scratch(bytes), bytes, code, x.size(0), x.size(1),
                                                 x.size(2), x.size(3), grid.size(1), grid.size(2), (int)a.i[0], (int)a.i[1], (int)a.i[2],
                                                 l.stream()));
    }
};

// ---- autograd ----------------------------------------------------------------------------------------------------------

bool usable_grad(const Tensor& grad, const Tensor& like, int64_t numel)
{
    return like.defined() && plain(grad, like, like.scalar_type()) && grad.numel() == numel;
}

template <class Op>
constexpr size_t kGrads = Op::kGradOf.size();

template <class Op>
int64_t output_numel(const Args& a);
template <>
int64_t output_numel<Msda>(const Args& a) { return a.t[3].size(0) * a.t[3].size(1) * a.t[0].size(2) * a.t[0].size(3); }
template <>
int64_t output_numel<Fused>(const Args& a) { return a.t[4].size(0) * a.t[4].size(1) * a.t[0].size(2) * a.t[0].size(3); }
template <>
int64_t output_numel<Dagg>(const Args& a) { return a.t[0].size(0) * a.t[4].size(1) * a.t[0].size(2); }
template <>
int64_t output_numel<Grid>(const Args& a) { return a.t[0].size(0) * a.t[0].size(1) * a.t[1].size(1) * a.t[1].size(2); }
template <>
int64_t output_numel<Gka>(const Args& a) { return output_numel<Msda>(a); }

template <class Op>
bool kept_as_taken(const Args& a)
{
    for (int k = 0; k < Op::kTensors; ++k)
        if (!a.t[k].defined()) return false;
    return Op::takes(a) && (!Op::kKeepsOutput || usable_grad(a.out, a.t[0], output_numel<Op>(a)));
}

// What is unpacked in the backward need not be what the forward checked: hooks for saved tensors (torch.autograd.graph) hand
// back whatever they like -- a view with other strides, another dtype, a tensor of another device.  Strides and dtypes are brought
// into the form that the kernels read, value's dtype deciding as in the forward; everything else is an error.
template <class Op>
void bring_into_form(Args& a)
{
    auto bring = [&](Tensor& t, at::ScalarType type) {
        TORCH_CHECK(t.defined() && t.is_cuda() && t.device() == a.t[0].device(), Op::kNode,
                    ": a tensor saved for the backward was handed back on another device (this build has no CPU implementation)");
        t = (t.is_floating_point() ? t.to(type) : t).contiguous();
    };
    TORCH_CHECK(a.t[0].defined(), Op::kNode, ": a tensor saved for the backward was not handed back");
    const at::ScalarType type = a.t[0].scalar_type();
    for (int k = 0; k < Op::kTensors; ++k) bring(a.t[k], k == Op::kFloat32 ? at::kFloat : type);
    if (Op::kKeepsOutput) bring(a.out, type);
    TORCH_CHECK(kept_as_taken<Op>(a), Op::kNode, ": the tensors saved for the backward were handed back in a form that the kernels do not take");
}

template <class Op>
struct Backward : torch::autograd::Node {
    std::array<torch::autograd::SavedVariable, Op::kTensors> saved;
    torch::autograd::SavedVariable saved_out;
    std::array<int64_t, 3> ints{};

    std::string name() const override { return Op::kNode; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto& s : saved) s.reset_data();
        saved_out.reset_data();
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override
    {
        Args a;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (int k = 0; k < Op::kTensors; ++k) a.t[k] = saved[k].unpack();
            if (Op::kKeepsOutput) a.out = saved_out.unpack(shared_from_this());
            a.i = ints;
        }
        std::array<Tensor, kGrads<Op>> g;
        const bool again = at::GradMode::is_enabled();  // (a graph of the backward is wanted)
        {
            at::AutoDispatchBelowAutograd below;
            if (!kept_as_taken<Op>(a)) bring_into_form<Op>(a);
            Tensor grad = grads[0];
            if (!grad.defined()) {
                grad = Op::new_output(a);
                grad.zero_();
            } else if (!usable_grad(grad, a.t[0], output_numel<Op>(a))) {
                grad = grad.to(a.t[0].options()).contiguous();
                TORCH_CHECK(grad.numel() == output_numel<Op>(a), Op::kNode, ": grad_output has another size than the output");
                TORCH_CHECK(usable_grad(grad, a.t[0], output_numel<Op>(a)), Op::kNode, ": grad_output is no tensor that the kernels can read");
            }
            unsigned need = 0;
            for (size_t k = 0; k < kGrads<Op>; ++k) {
                need |= task_should_compute_output(k) ? 1u << k : 0u;
                g[k] = new_like(a.t[Op::kGradOf[k]]);
            }
            Op::backward(a, grad, g, need);
            for (size_t k = 0; k < kGrads<Op>; ++k)
                if (!((need >> k) & 1)) g[k].reset();
        }
        torch::autograd::variable_list out(g.begin(), g.end());
        if (Op::kOnce && again && grads[0].defined()) {
            // what torch.autograd.function.once_differentiable does: gradients of these gradients raise an error
            bool any = grads[0].requires_grad();
            for (const Tensor& t : a.t) any = any || (t.defined() && t.requires_grad());
            if (any) {
                for (Tensor& t : out)
                    if (t.defined()) t = t.detach().requires_grad_(true);
                auto error = std::make_shared<torch::autograd::DelayedError>(
                    "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)out.size());
                out = (*error)(std::move(out));
            }
        }
        return out;
    }
};

// Nothing but PyTorch's eager reverse-mode autograd is to see the call.
template <class Op>
bool eager(const Args& a)
{
    for (int k = 0; k < Op::kTensors; ++k)
        if (a.t[k].numel() == 0 || a.t[k]._fw_grad(0).defined()) return false;
    return !(Op::kFloat32InAutocast && at::autocast::is_autocast_enabled(at::kCUDA)) && !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !torch::jit::tracer::isTracing();
}

template <class Op>
Tensor call(const Args& a)
{
    bool wanted = false;
    if (at::GradMode::is_enabled())
        for (int k : Op::kGradOf) wanted = wanted || a.t[k].requires_grad();
    Tensor out;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        out = Op::new_output(a);
        Op::forward(a, out);
    }
    if (!wanted) return out;
    auto node = std::shared_ptr<Backward<Op>>(new Backward<Op>(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges;
    edges.reserve(kGrads<Op>);
    for (int k : Op::kGradOf)
        edges.push_back(a.t[k].requires_grad() ? torch::autograd::impl::gradient_edge(a.t[k]) : torch::autograd::Edge());
    node->set_next_edges(std::move(edges));
    for (int k = 0; k < Op::kTensors; ++k) node->saved[k] = torch::autograd::SavedVariable(a.t[k], false);
    node->ints = a.i;
    torch::autograd::set_history(out, node);
    if (Op::kKeepsOutput) node->saved_out = torch::autograd::SavedVariable(out, true);
    return out;
}

// ---- Python --------------------------------------------------------------------------------------------------------------

bool unpack(PyObject* o, Tensor* t)
{
    if (!THPVariable_CheckExact(o)) return false;
    *t = THPVariable_Unpack(o);
    return true;
}

template <class Op>
bool unpack(PyObject* const* args, Py_ssize_t n, Args* a)
{
    if (n < Op::kTensors + Op::kInts) return false;
    for (int k = 0; k < Op::kTensors; ++k)
        if (!unpack(args[k], &a->t[k])) return false;
    for (int k = 0; k < Op::kInts; ++k) {
        a->i[k] = PyLong_AsLongLong(args[Op::kTensors + k]);
        if (a->i[k] == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    }
    return true;
}

struct NoGil {
    PyThreadState* s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

template <class Op>
PyObject* py_call(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    Args a;
    if (n != Op::kTensors + Op::kInts || !unpack<Op>(args, n, &a) || !Op::takes(a) || !eager<Op>(a)) Py_RETURN_NONE;
    Tensor out;
    {
        NoGil free;
        out = call<Op>(a);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

template <class Op>
PyObject* py_forward(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    constexpr int kIn = Op::kTensors + Op::kInts;
    Args a;
    Tensor out;
    if (n > kIn + 1 || !unpack<Op>(args, n, &a) || !Op::takes(a)) Py_RETURN_NONE;
    if (n > kIn && (!unpack(args[kIn], &out) || !usable_grad(out, a.t[0], output_numel<Op>(a)))) Py_RETURN_NONE;
    {
        NoGil free;
        at::AutoDispatchBelowADInplaceOrView below;
        if (!out.defined()) out = Op::new_output(a);
        Op::forward(a, out);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// inputs, [forward result,] grad_output[, a tensor or None for every gradient]
template <class Op>
PyObject* py_backward(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    constexpr int kIn = Op::kTensors + Op::kInts, kG = (int)kGrads<Op>, kAt = kIn + (Op::kKeepsOutput ? 1 : 0);
    Args a;
    Tensor grad;
    std::array<Tensor, kGrads<Op>> g;
    if ((n != kAt + 1 && n != kAt + 1 + kG) || !unpack<Op>(args, n, &a) || !Op::takes(a)) Py_RETURN_NONE;
    if (!unpack(args[kAt], &grad) || !usable_grad(grad, a.t[0], output_numel<Op>(a))) Py_RETURN_NONE;
    if (Op::kKeepsOutput && (!unpack(args[kIn], &a.out) || !usable_grad(a.out, a.t[0], output_numel<Op>(a)))) Py_RETURN_NONE;
    unsigned need = (1u << kG) - 1;
    if (n > kAt + 1) {
        for (int k = 0; k < kG; ++k) {
            PyObject* o = args[kAt + 1 + k];
            if (o == Py_False) need &= ~(1u << k);
            else if (o != Py_None && (!unpack(o, &g[k]) || !usable_grad(g[k], a.t[Op::kGradOf[k]], a.t[Op::kGradOf[k]].numel()))) Py_RETURN_NONE;
        }
    }
    {
        NoGil free;
        at::AutoDispatchBelowADInplaceOrView below;
        for (int k = 0; k < kG; ++k)
            if (!g[k].defined()) g[k] = new_like(a.t[Op::kGradOf[k]]);
        Op::backward(a, grad, g, need);
    }
    PyObject* tuple = PyTuple_New(kG);
    if (!tuple) return nullptr;
    for (int k = 0; k < kG; ++k) {
        PyObject* o = (need >> k) & 1 ? THPVariable_Wrap(std::move(g[k])) : Py_NewRef(Py_None);
        if (!o) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, k, o);
    }
    return tuple;
    END_HANDLE_TH_ERRORS
}

#define MXD_OP(name, op)                                                                             \
    {name, (PyCFunction)(void (*)(void)) & py_call<op>, METH_FASTCALL, nullptr},                     \
    {name "_forward", (PyCFunction)(void (*)(void)) & py_forward<op>, METH_FASTCALL, nullptr},       \
    {name "_backward", (PyCFunction)(void (*)(void)) & py_backward<op>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {MXD_OP("msda", Msda), MXD_OP("fused", Fused), MXD_OP("dagg", Dagg), MXD_OP("gka", Gka), MXD_OP("grid", Grid),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "The operators on PyTorch tensors (csrc/torch_ops.cpp).", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
