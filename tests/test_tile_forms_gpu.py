"""The grad_value pass in its forms -- 4, 8 and 16 lanes per row, loads of 8 and 16 bytes -- at the edges of their tiles: maps of a few
pixels more and fewer than a tile and than a tile without a lane group, pairs that straddle groups and tiles, tiles held in copies
and tiles split by query range; against the oracle."""
import pytest
import torch

from drivingsdk_amd import workloads
from test_msda_gpu import _check_all
from util import BWD_FP32, FWD_FP32, half_tol, set_tuning

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,hd", [(torch.float16, 8), (torch.bfloat16, 32), (torch.float16, 36), (torch.float16, 40), (torch.bfloat16, 64),
                                      (torch.float16, 72), (torch.float16, 100), (torch.bfloat16, 128), (torch.float16, 136),
                                      (torch.float32, 32), (torch.float32, 50), (torch.float32, 70), (torch.float32, 128),
                                      (torch.float32, 130)])
@pytest.mark.parametrize("maps,nq", [(((1, 505), (3, 2)), 40), (((21, 24), (8, 16)), 300), (((500, 1), (127, 1)), 300), (((27, 19), (5, 25)), 60),
                                     (((16, 16), (1, 129)), 2500)], ids=["505+6", "504+128", "500+127", "513+125", "256+129"])
def test_edges_of_tiles(gpu_device, maps, nq, dtype, hd):
    g = torch.Generator().manual_seed(hd + nq)
    shapes, lsi = workloads.level_tensors(maps)
    bs, nh, nl, npts, nk = 1, 2, len(maps), 3, int(shapes.prod(1).sum())
    tensors = (torch.randn(bs, nk, nh, hd, generator=g), torch.rand(bs, nq, nh, nl, npts, 2, generator=g) * 1.2 - 0.1,
               torch.rand(bs, nq, nh, nl, npts, generator=g), torch.randn(bs, nq, nh * hd, generator=g))
    value, loc, attn, gout = (t.to(dtype) for t in tensors)
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(workloads.MsdaInputs(value, shapes, lsi, loc, attn, gout), gpu_device, fwd, bwd)


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 32), (torch.float32, 37), (torch.float32, 70), (torch.bfloat16, 32), (torch.float16, 130)])
@pytest.mark.parametrize("target", [128, 100000], ids=["shared", "owned"])
@pytest.mark.parametrize("maps", [((15, 25),), ((10, 10), (1, 3)), ((7, 18), (21, 24))], ids=["375", "100+3", "126+504"])
def test_copies_and_extra_lists_are_added_up(gpu_device, monkeypatch, maps, target, dtype, hd):
    """More records than a round holds, three quarters of them on a few pixels: tiles in copies with extra lists for the hot pixels, of
    one workgroup that stores them and of several that add to them."""
    set_tuning(monkeypatch, MXD_MSDA_TILE_TARGET=target)
    g = torch.Generator().manual_seed(hd + len(maps))
    shapes, lsi = workloads.level_tensors(maps)
    bs, nh, nl, npts, nq, nk = 1, 2, len(maps), 4, 2500, int(shapes.prod(1).sum())
    loc = torch.rand(bs, nq, nh, nl, npts, 2, generator=g)
    loc[:, :, :, :, 1:] = 0.4 + 0.05 * loc[:, :, :, :, 1:]
    tensors = (torch.randn(bs, nk, nh, hd, generator=g), loc, torch.rand(bs, nq, nh, nl, npts, generator=g),
               torch.randn(bs, nq, nh * hd, generator=g))
    value, loc, attn, gout = (t.to(dtype) for t in tensors)
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(workloads.MsdaInputs(value, shapes, lsi, loc, attn, gout), gpu_device, fwd, bwd)


@pytest.mark.parametrize("nq", [31, 33, 700, 17000])
@pytest.mark.parametrize("order", ["sorted", "random"])
@pytest.mark.parametrize("dtype,hd", [(torch.float32, 8), (torch.float16, 32)])
def test_runs_of_records(gpu_device, dtype, hd, order, nq):
    """Runs of no, few and many records of a tile: queries in the order of the map, which leave most tiles no record of most slabs, and in
    no order; fewer runs than a wavefront looks through at a time and more, batches and windows of records that end within and between runs."""
    g = torch.Generator().manual_seed(nq)
    maps = ((40, 41), (9, 7))
    shapes, lsi = workloads.level_tensors(maps)
    bs, nh, nl, npts, nk = 1, 1, 2, 2, int(shapes.prod(1).sum())
    loc = torch.rand(bs, nq, 1, 1, 1, 2, generator=g).expand(bs, nq, nh, nl, npts, 2) + 0.01 * torch.randn(bs, nq, nh, nl, npts, 2, generator=g)
    if order == "sorted":
        loc = loc[:, loc[0, :, 0, 0, 0, 1].argsort()]
    tensors = (torch.randn(bs, nk, nh, hd, generator=g), loc.contiguous(), torch.rand(bs, nq, nh, nl, npts, generator=g),
               torch.randn(bs, nq, nh * hd, generator=g))
    value, loc, attn, gout = (t.to(dtype) for t in tensors)
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(workloads.MsdaInputs(value, shapes, lsi, loc, attn, gout), gpu_device, fwd, bwd)
