"""Grid sampler on planes at the sizes where its kernels change course, against torch on the CPU in float64: planes of odd size
(no 16-byte boundaries), one and many planes per workgroup, one and several output pixels per thread, ranges and splits of
the output pixels, chunks of the channels, planes that take a CU's LDS whole, and planes too large for it (channel-last form)."""
import pytest
import torch
import torch.nn.functional as F

import mx_driving
from drivingsdk_amd.ops.grid_sampler2d_v2 import GridSampler2dV2Function
from test_grid_sampler_gpu import check, make_inputs
from util import BF16, BWD_FP32, FWD_FP32, HALF, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [([1, 1, 1, 1], [1, 1, 1, 2]), ([2, 3, 5, 7], [2, 3, 5, 2]), ([3, 5, 37, 41], [3, 23, 29, 2]), ([1, 19, 20, 31], [1, 70, 90, 2]),
          ([2, 33, 16, 20], [2, 13, 200, 2]), ([24, 40, 17, 21], [24, 9, 11, 2]), ([1, 2, 101, 181], [1, 100, 181, 2]),
          ([1, 4, 160, 256], [1, 40, 50, 2]), ([1, 3, 161, 256], [1, 10, 10, 2]), ([2, 256, 9, 33], [2, 31, 17, 2])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("input_shape,grid_shape", SHAPES)
def test_planes(gpu_device, input_shape, grid_shape, dtype):
    x, grid, go = make_inputs(input_shape, grid_shape, seed=input_shape[1], span=1.2)
    if dtype == torch.float32:
        # (a float32 pixel coordinate of up to 180 is off by up to 1e-5)
        print(check(x, grid, go, "zeros", False, gpu_device, fwd_tol=2 * FWD_FP32, bwd_tol=BWD_FP32))
        return
    x, grid, go = x.to(dtype), grid.to(dtype), go.to(dtype)
    xr, gr = x.double().requires_grad_(), grid.double().requires_grad_()
    want = F.grid_sample(xr, gr, "bilinear", "border", True)
    want.backward(go.double())
    xd, gd = x.to(gpu_device).requires_grad_(), grid.to(gpu_device).requires_grad_()
    out = mx_driving.grid_sampler2d_v2(xd, gd, "bilinear", "border", True)
    out.backward(go.to(gpu_device))
    tol = HALF if dtype == torch.float16 else BF16
    for got, ref in ((out.detach(), want.detach()), (xd.grad, xr.grad)):
        assert got.dtype == dtype and rel_err(got.double().cpu().numpy(), ref.numpy()) <= tol


# (planes of more than 10240 pixels, 256 and more of them: both gradients by the same workgroups.  One and many chunks of the channels, the
#  last of them short; one, two, three, six and nine output pixels per thread, full and partly so; the largest plane in float32 and in 16 bits)
LARGE = [([257, 1, 97, 107], [257, 3, 5, 2]), ([131, 22, 97, 107], [131, 5, 7, 2]), ([2, 129, 103, 101], [2, 32, 32, 2]), ([1, 256, 64, 161], [1, 25, 41, 2]),
         ([5, 70, 80, 168], [5, 37, 83, 2]), ([3, 100, 75, 140], [3, 48, 128, 2]), ([3, 100, 75, 140], [3, 96, 96, 2]),
         ([3, 100, 75, 140], [3, 97, 96, 2]), ([2, 130, 120, 135], [2, 9, 7, 2])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("input_shape,grid_shape", LARGE)
def test_large_planes(gpu_device, input_shape, grid_shape, dtype):
    test_planes(gpu_device, input_shape, grid_shape, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("input_shape,grid_shape", [([8, 130, 79, 157], [8, 3, 5, 2]), ([8, 131, 79, 157], [8, 41, 50, 2]),
                                                    ([6, 176, 79, 157], [6, 48, 128, 2]), ([4, 131, 79, 157], [4, 97, 95, 2]),
                                                    ([513, 3, 67, 97], [513, 9, 7, 2]), ([5, 128, 160, 255], [5, 9, 7, 2]),
                                                    ([8, 190, 79, 157], [8, 3, 5, 2]), ([3, 255, 160, 252], [3, 9, 7, 2])])
def test_runs_of_planes(gpu_device, input_shape, grid_shape, dtype):
    """Many planes per workgroup, one after the other (the last run short; one, three, six and nine output pixels per thread; planes of
    odd size; a plane that takes a CU's LDS whole), and sizes just outside of that form: the same bits as few planes, which get a workgroup each."""
    g = torch.Generator().manual_seed(7)
    grid = ((2 * torch.rand(grid_shape, generator=g) - 1) * 1.2).to(gpu_device, dtype)
    x = torch.rand(input_shape[1:], generator=g).to(gpu_device, dtype) + torch.arange(input_shape[0], device=gpu_device, dtype=dtype).view(-1, 1, 1, 1)
    for padding, align in (("zeros", False), ("border", True)):
        out = mx_driving.grid_sampler2d_v2(x, grid, "bilinear", padding, align)
        for i in (0, input_shape[0] - 1):
            few = mx_driving.grid_sampler2d_v2(x[i:i + 1, -3:].contiguous(), grid[i:i + 1], "bilinear", padding, align)
            assert torch.equal(out[i:i + 1, -3:], few)
            assert torch.equal(out[i:i + 1, :2], mx_driving.grid_sampler2d_v2(x[i:i + 1, :2].contiguous(), grid[i:i + 1], "bilinear", padding, align))


def test_single_gradients_and_the_python_function(gpu_device):
    x, grid, go = [t.to(gpu_device) for t in make_inputs([2, 20, 30, 40], [2, 25, 35, 2], seed=2)]

    class PythonPath(GridSampler2dV2Function):
        pass

    x.requires_grad_()
    grid.requires_grad_()
    a, b = (f(x, grid, "bilinear", "zeros", False) for f in (mx_driving.grid_sampler2d_v2, PythonPath.apply))
    assert torch.equal(a, b) and a.grad_fn.name() == b.grad_fn.name().replace("PythonPath", "GridSampler2dV2Function")
    both = torch.autograd.grad(a, [x, grid], go, retain_graph=True)
    for k, t in enumerate((x, grid)):
        for o in (a, b):
            assert torch.allclose(torch.autograd.grad(o, t, go, retain_graph=True)[0], both[k], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("input_shape", [[1, 4, 8, 8], [2, 128, 80, 130]])
def test_infinite_pixels_outside_the_samples(gpu_device, input_shape):
    """A pixel that no sample reaches must not enter a result, whatever it holds (corners outside the image read some pixel)."""
    x, grid, go = make_inputs(input_shape, [input_shape[0], 6, 6, 2], seed=6)
    grid = grid * 0.05 + torch.tensor([1.0, 1.0])   # around the lower right corner, part of it outside
    x[:, :, 0, 0] = float("inf")
    xd, gd = x.to(gpu_device).requires_grad_(), grid.to(gpu_device).requires_grad_()
    out = mx_driving.grid_sampler2d_v2(xd, gd, "bilinear", "zeros", False)
    out.backward(go.to(gpu_device))
    assert all(torch.isfinite(t).all() for t in (out, xd.grad, gd.grad))
