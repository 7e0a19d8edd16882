"""The autograd node of the extension module against the operators' Python autograd Functions (which take over under autocast and
for subclasses): same gradients, and the same answers where a second backward, a changed input or a graph of the backward is
asked for."""
import pytest
import torch

import drivingsdk_amd
import mx_driving
from drivingsdk_amd import workloads
from util import to_device

pytestmark = pytest.mark.gpu


class _PythonPath(mx_driving.MultiScaleDeformableAttnFunction):
    pass


def _inputs(device):
    d = to_device(workloads.make_inputs("tiny", with_grad_output=True), device)
    return d, [t.clone().requires_grad_() for t in (d.value, d.sampling_locations, d.attention_weights)]


def _call(fn, d, x):
    return fn(x[0], d.spatial_shapes, d.level_start_index, x[1], x[2])


def test_same_results_as_the_python_function(gpu_device):
    d, x = _inputs(gpu_device)
    a, b = (_call(f, d, x) for f in (mx_driving.multi_scale_deformable_attn, _PythonPath.apply))
    assert torch.equal(a, b) and a.grad_fn.name() == "MultiScaleDeformableAttnFunctionBackward"
    for n in (3, 1):   # all gradients, value's alone
        ga, gb = (torch.autograd.grad(o, x[:n], d.grad_output, retain_graph=True) for o in (a, b))
        for k, (p, q) in enumerate(zip(ga, gb)):
            assert torch.allclose(p, q, rtol=1e-5, atol=1e-5 * float(q.abs().max())) if k == 0 else torch.equal(p, q)
    # an expanded grad_output, and none of the gradients asked for
    assert torch.equal(torch.autograd.grad(a.sum(), x[2])[0], torch.autograd.grad(b.sum(), x[2])[0])
    with torch.no_grad():
        assert not _call(mx_driving.multi_scale_deformable_attn, d, x).requires_grad


def test_autocast_computes_in_float32(gpu_device):
    d, x = _inputs(gpu_device)
    with torch.autocast("cuda", dtype=torch.float16):
        out = _call(mx_driving.multi_scale_deformable_attn, d, [t.half() for t in x])
    assert out.dtype == torch.float32


def test_errors_of_a_second_use(gpu_device):
    d, x = _inputs(gpu_device)
    out = _call(mx_driving.multi_scale_deformable_attn, d, x)
    out.backward(d.grad_output)
    with pytest.raises(RuntimeError, match="backward through the graph a second time"):
        out.backward(d.grad_output)
    out = _call(mx_driving.multi_scale_deformable_attn, d, x)
    with torch.no_grad():
        x[2].mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(d.grad_output)
    out = _call(mx_driving.multi_scale_deformable_attn, d, x)
    g = torch.autograd.grad(out, x[0], d.grad_output, create_graph=True)[0]
    with pytest.raises(RuntimeError, match="once_differentiable"):
        g.sum().backward()


def test_fused_form_keeps_its_result_for_the_backward(gpu_device):
    d, x = _inputs(gpu_device)
    g = torch.Generator(device=gpu_device).manual_seed(3)
    bs, nq, nh, nl, npts, _ = x[1].shape
    ref = torch.rand(bs, nq, nl, 2, generator=g, device=gpu_device, requires_grad=True)
    off = torch.randn(x[1].shape, generator=g, device=gpu_device, requires_grad=True)
    logits = torch.randn(bs, nq, nh, nl * npts, generator=g, device=gpu_device, requires_grad=True)
    args = (x[0], d.spatial_shapes, d.level_start_index, ref, off, logits)

    class PythonPath(drivingsdk_amd.MultiScaleDeformableAttnFusedFunction):
        pass

    for want in ([ref, off, logits], [off, logits]):
        got = [torch.autograd.grad(f(*args), want, d.grad_output)
               for f in (drivingsdk_amd.multi_scale_deformable_attn_fused, PythonPath.apply)]
        for p, q in zip(*got):
            assert torch.equal(p, q)
