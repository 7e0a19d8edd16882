"""Units of few samples, whose samples are packed over the lanes of a pass, and rows of up to 32 bytes, which more lanes share than
their 16-byte pieces ask for: sample counts around the edges of a pass and of a chunk of 16, against the oracle."""
import pytest
import torch

from drivingsdk_amd import workloads
from test_first_pass_gpu import _takes_4_lanes
from test_msda_gpu import _check_all
from util import BWD_FP32, FWD_FP32, half_tol, set_tuning

pytestmark = pytest.mark.gpu


def _inputs(maps, npts, nq, nh, hd, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    shapes, lsi = workloads.level_tensors(maps)
    bs, nl, nk = 2, len(maps), int(shapes.prod(1).sum())
    value = torch.randn(bs, nk, nh, hd, generator=g)
    loc = torch.rand(bs, nq, nh, nl, npts, 2, generator=g) * 1.2 - 0.1
    attn = torch.rand(bs, nq, nh, nl, npts, generator=g)
    gout = torch.randn(bs, nq, nh * hd, generator=g)
    return workloads.MsdaInputs(*[t.to(dtype) if t.is_floating_point() else t for t in (value, shapes, lsi, loc, attn, gout)])


_MAPS = ((17, 23), (9, 12), (5, 6))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nl,npts", [(1, 1), (1, 2), (1, 3), (1, 5), (1, 7), (2, 4), (3, 3), (3, 5), (1, 17), (2, 9), (3, 7)])
def test_sample_counts_around_a_pass(gpu_device, nl, npts, dtype):
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    for nq in (1, 67):
        _check_all(_inputs(_MAPS[:nl], npts, nq, 3, 32, dtype, 10 * nl + npts), gpu_device, fwd, bwd)


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 4), (torch.float32, 8), (torch.float16, 8), (torch.float16, 12), (torch.float16, 16),
                                      (torch.bfloat16, 16)])
@pytest.mark.parametrize("nl,npts", [(1, 3), (3, 4), (1, 13), (3, 6)])
def test_short_rows(gpu_device, nl, npts, dtype, hd):
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(_inputs(_MAPS[:nl], npts, 131, 4, hd, dtype, hd + npts), gpu_device, fwd, bwd)


@pytest.mark.parametrize("hd", [1, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_narrow_16_bit_rows_with_a_forced_tile_size(gpu_device, monkeypatch, dtype, hd):
    set_tuning(monkeypatch, MXD_MSDA_TILE_PX_LOG2=7)
    _check_all(_inputs(_MAPS, 4, 131, 4, hd, dtype, hd), gpu_device, half_tol(dtype), half_tol(dtype))


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 32), (torch.float32, 13), (torch.float16, 32), (torch.bfloat16, 24), (torch.float16, 64), (torch.bfloat16, 33)])
@pytest.mark.parametrize("nl,npts", [(1, 8), (2, 8), (3, 8), (1, 16), (1, 10), (3, 10), (1, 24), (1, 30)])
def test_eight_points_side_by_side(gpu_device, nl, npts, dtype, hd):
    """Levels of eight points and more, with one unit per query and with two, whole and cut off at their last queries; rows of 8 lanes, and
    of 4 where a launch has workgroups enough for them."""
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    nqs = (1, 67)
    if 32 < hd * (torch.finfo(dtype).bits // 8) <= 64:
        nqs += (10003,)
        assert _takes_4_lanes(2, sum(h * w for h, w in _MAPS[:nl]), 3, hd, nl, nqs[-1], npts, dtype)
    for nq in nqs:
        _check_all(_inputs(_MAPS[:nl], npts, nq, 3, hd, dtype, 10 * nl + npts), gpu_device, fwd, bwd)
