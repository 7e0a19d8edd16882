"""Rows that no whole number of 16-byte pieces covers: the last piece of a row overlaps the one before it.  Head sizes around
the edges of the pieces and of the tile pass's channel blocks, against the oracle, and the neighbouring head filled with NaN (what
a piece reads beyond its row must not reach the row's results)."""
import pytest
import torch

from drivingsdk_amd import workloads
from test_msda_gpu import _check_all
from util import BWD_FP32, FWD_FP32, half_tol, run_gpu

pytestmark = pytest.mark.gpu


def _inputs(hd, nh, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    shapes, lsi = workloads.level_tensors(((31, 33), (9, 7)))
    bs, nk, nq, npts = 2, int(shapes.prod(1).sum()), 157, 3
    value = torch.randn(bs, nk, nh, hd, generator=g)
    loc = torch.rand(bs, nq, nh, 2, npts, 2, generator=g) * 1.2 - 0.1
    attn = torch.rand(bs, nq, nh, 2, npts, generator=g)
    gout = torch.randn(bs, nq, nh * hd, generator=g)
    return workloads.MsdaInputs(*[t.to(dtype) if t.is_floating_point() else t for t in (value, shapes, lsi, loc, attn, gout)])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [3, 5, 7, 9, 31, 33, 37, 63, 65, 67, 129, 131, 255])
def test_head_sizes_around_the_pieces(gpu_device, hd, dtype):
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(_inputs(hd, 3, dtype, hd), gpu_device, fwd, bwd)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [5, 37, 67])
def test_the_next_head_does_not_leak(gpu_device, hd, dtype):
    inp = _inputs(hd, 2, dtype, hd + 1)
    nan = inp.value.clone()
    nan[:, :, 1] = float("nan")
    gout = inp.grad_output.clone().reshape(*inp.grad_output.shape[:2], 2, hd)
    gout[:, :, 1] = float("nan")
    clean, dirty = (run_gpu(x, gpu_device) for x in (inp, inp._replace(value=nan, grad_output=gout.flatten(2))))
    for k, (a, b) in enumerate(zip(clean, dirty)):
        a, b = (x.reshape(*x.shape[:2], 2, -1)[:, :, 0] for x in (a, b))
        if k == 1:   # (order of the sums over samples)
            assert abs(a - b).max() <= (BWD_FP32 if dtype == torch.float32 else half_tol(dtype)) * abs(a).max()
        else:
            assert (a == b).all()
