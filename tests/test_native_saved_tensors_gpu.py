"""The autograd node of the extension module where something stands between the forward and the backward: hooks for saved tensors
that hand back other strides, another dtype or another device, checkpointing, tensors kept on the CPU in between, another stream,
several threads -- and the transforms that are left to the Python Functions (functorch, forward mode, batched gradients, tracing)."""
import threading

import pytest
import torch
from torch.utils.checkpoint import checkpoint

from drivingsdk_amd import _C
from drivingsdk_amd.ops.deformable_aggregation import AdsDeformableAggregation
from drivingsdk_amd.ops.geometric_kernel_attention import GeometricKernelAttentionFunc
from drivingsdk_amd.ops.grid_sampler2d_v2 import GridSampler2dV2Function
from drivingsdk_amd.ops.msda_fused import MultiScaleDeformableAttnFusedFunction
from drivingsdk_amd.ops.multi_scale_deformable_attn import MultiScaleDeformableAttnFunction

pytestmark = pytest.mark.gpu

OPS = ("msda", "fused", "dagg", "gka", "grid")


class Case:
    """An operator on small inputs: `x` are the tensors with gradients, `call` the public entry point, `python` its autograd Function
    without the extension module's node, `grads` the gradients of inputs as they are given, in their dtypes."""

    def __init__(self, op, device):
        g = torch.Generator(device=device).manual_seed(7)
        rand = lambda *s: torch.rand(*s, generator=g, device=device)
        shapes = torch.tensor([[9, 13], [5, 7]], device=device, dtype=torch.int32)
        starts = torch.tensor([0, 117], device=device, dtype=torch.int32)
        bs, nk, nh, hd, nq, nl, npts = 2, 152, 2, 16, 21, 2, 3
        if op == "msda":
            self.x = [rand(bs, nk, nh, hd), rand(bs, nq, nh, nl, npts, 2), rand(bs, nq, nh, nl, npts)]
            fn, self.args = MultiScaleDeformableAttnFunction, lambda x: (x[0], shapes, starts, x[1], x[2])
            self.grads = lambda x, go, out: _C.multi_scale_deformable_attn_backward(*self.args(x), go)
        elif op == "fused":
            self.x = [rand(bs, nk, nh, hd), rand(bs, nq, nl, 2), rand(bs, nq, nh, nl, npts, 2), rand(bs, nq, nh, nl * npts)]
            fn, self.args = MultiScaleDeformableAttnFusedFunction, lambda x: (x[0], shapes, starts, *x[1:])
            self.grads = lambda x, go, out: _C.msda_fused_backward(*self.args(x), out, go)
        elif op == "dagg":
            self.x = [rand(bs, 2 * nk, 32), rand(bs, nq, npts, 2, 2), rand(bs, nq, npts, 2, nl, 4)]
            ss, si = shapes.expand(2, 2, 2).contiguous(), torch.stack((starts, starts + nk)).contiguous()
            fn, self.args = AdsDeformableAggregation, lambda x: (x[0], ss, si, x[1], x[2])
            self.grads = lambda x, go, out: _C.deformable_aggregation_backward(*self.args(x), go)
        elif op == "gka":
            self.x = [rand(bs, nk, nh, hd), rand(bs, nq, nh, nl, npts)]
            loc = (rand(bs, nq, nh, nl, npts, 2) * 12 - 2).trunc()
            fn, self.args = GeometricKernelAttentionFunc, lambda x: (x[0], shapes, starts, loc, x[1])
            self.grads = lambda x, go, out: _C.geometric_kernel_attention_backward(x[0], shapes, starts, loc, x[1], go)
        else:
            self.x = [rand(bs, 5, 9, 13), rand(bs, 7, 11, 2) * 2 - 1]
            fn, self.args = GridSampler2dV2Function, lambda x: (x[0], x[1], "bilinear", "zeros", False)

            def grads(x, go, out):
                gx, gg = _C.grid_sampler2d_v2_backward(go.permute(0, 2, 3, 1), x[0].permute(0, 2, 3, 1), x[1], 0, 0, False)
                return gx, gg
            self.grads = grads
        self.call = lambda x: fn.apply(*self.args(x))
        self.python = lambda x: type("PythonPath", (fn,), {}).apply(*self.args(x))
        self.x = [t.requires_grad_() for t in self.x]
        self.out = self.call(self.x)
        assert self.out.grad_fn.name() == fn.__name__ + "Backward"
        self.go = torch.randn(self.out.shape, generator=g, device=device)
        self.want = torch.autograd.grad(self.out, self.x, self.go, retain_graph=True)

    def check(self, got, want=None, rel=1e-5):
        """(float32 sums that atomics may put in another order; `rel` of the largest value)"""
        for g, w, x in zip(got, want or self.want, self.x):
            assert g.shape == x.shape and g.dtype == x.dtype
            assert float((g - w).abs().max()) <= rel * float(w.abs().max())

    def backward_with(self, unpack, picks=None):
        """Gradients when the saved tensors (numbered in the order in which they are saved) come back as unpack(number, tensor)."""
        count = [0]

        def pack(t):
            count[0] += 1
            return count[0] - 1, t
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda p: unpack(*p)):
            out = self.call(self.x)
        assert count[0] > 0
        return torch.autograd.grad(out, self.x, self.go)


@pytest.fixture(params=OPS)
def case(request, gpu_device):
    return Case(request.param, gpu_device)


def strided(t):
    return torch.stack((t, torch.full_like(t, 3)), -1)[..., 0]


def test_other_strides_come_back(case):
    assert not strided(case.x[0]).is_contiguous()
    case.check(case.backward_with(lambda k, t: strided(t)))
    for pick in range(7):
        case.check(case.backward_with(lambda k, t: strided(t) if k == pick else t))


def test_transposed_memory_comes_back(case):
    swap = lambda t: t.transpose(0, 1).contiguous().transpose(0, 1) if t.dim() > 1 else t
    case.check(case.backward_with(lambda k, t: swap(t)))


def test_another_dtype_comes_back(case):
    """All 16-bit tensors: gradients as the kernels form them for such inputs, in the input's dtype; single tensors: value's dtype
    decides, as where the Python functions are given mixed dtypes."""
    half = lambda t: t.half() if t.is_floating_point() and t.dtype == torch.float32 else t
    want = case.grads([half(t).detach() for t in case.x], half(case.go), half(case.out.detach()))
    case.check(case.backward_with(lambda k, t: half(t)), [w.float() for w in want], rel=2e-3)
    case.check(case.backward_with(lambda k, t: half(t) if k == 0 else t), [w.float() for w in want], rel=2e-3)
    # (float64 holds what was saved: the same gradients)
    double = lambda k, t: t.double() if k > 0 and t.is_floating_point() else t
    case.check(case.backward_with(double))


def test_another_device_or_shape_is_an_error(case):
    for pick in (0, 1):
        with pytest.raises(RuntimeError, match="another device"):
            case.backward_with(lambda k, t: t.cpu() if k == pick else t)
        with pytest.raises(RuntimeError):
            case.backward_with(lambda k, t: t[..., :1, :].contiguous() if k == pick else t)


def test_saved_on_cpu_and_checkpointed(case):
    with torch.autograd.graph.save_on_cpu():
        out = case.call(case.x)
    case.check(torch.autograd.grad(out, case.x, case.go))
    out = checkpoint(lambda *x: case.call(x), *case.x, use_reentrant=False)
    case.check(torch.autograd.grad(out, case.x, case.go))


def test_forward_on_another_stream(case):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        out = case.call(case.x)
        inside = torch.autograd.grad(out, case.x, case.go, retain_graph=True)
    torch.cuda.current_stream().wait_stream(s)
    case.check(torch.autograd.grad(out, case.x, case.go))
    case.check(inside)
    assert torch.equal(out, case.out) or float((out - case.out).abs().max()) <= 1e-5 * float(case.out.abs().max())


def test_threads_with_streams_of_their_own(case):
    torch.cuda.synchronize()
    failures = []

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(4):
                    case.check(torch.autograd.grad(case.call(case.x), case.x, case.go))
        except BaseException as e:  # noqa: B902 (reported by the test)
            failures.append(e)
    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures


def outcome(fn):
    try:
        r = fn()
    except Exception as e:
        return type(e), None
    return None, r


@pytest.mark.parametrize("what", ["func.grad", "vmap", "forward mode", "batched gradients", "trace"])
def test_what_is_left_to_python_has_its_outcome(case, what):
    """The public entry point does what the Python Function does: the same error, or the same result."""
    def run(f):
        x = [t.detach().clone().requires_grad_() for t in case.x]
        if what == "func.grad":
            return torch.func.grad(lambda v: (f([v] + x[1:]) * case.go).sum())(x[0].detach())
        if what == "vmap":
            return torch.func.vmap(lambda v: f([v] + x[1:]))(torch.stack((x[0].detach(), x[0].detach())))
        if what == "forward mode":
            import torch.autograd.forward_ad as fwad
            with fwad.dual_level():
                return fwad.unpack_dual(f([fwad.make_dual(x[0].detach(), torch.ones_like(x[0]))] + x[1:])).tangent
        if what == "batched gradients":
            return torch.autograd.grad(f(x), x, torch.stack((case.go, case.go)), is_grads_batched=True)[-1]
        return torch.jit.trace(lambda *t: f(list(t)), tuple(t.detach() for t in x), check_trace=False)(*[t.detach() for t in x])
    (e1, r1), (e2, r2) = (outcome(lambda: run(f)) for f in (case.call, case.python))
    print(what, e1, e2)
    assert e1 == e2
    if r1 is not None and r2 is not None:
        assert float((r1 - r2).abs().max()) <= 1e-5 * float(r2.abs().max())
    else:
        assert r1 is None and r2 is None
