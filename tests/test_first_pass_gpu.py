"""The backward's first kernel for rows of up to 128 bytes whose workgroups make one pass: rows that 4 lanes share and that no piece
divides, odd sample counts with one unit per query and with two, more tiles than a wavefront has lanes, workgroups that are partly
or wholly without queries -- against the oracle, plain and fused."""
import pytest
import torch

from drivingsdk_amd import workloads
from oracle import msda_oracle as orc
from test_msda_fused_gpu import _compare, _run
from test_msda_gpu import _check_all
from util import BWD_FP32, FWD_FP32, half_tol

pytestmark = pytest.mark.gpu

_MANY_TILES = ((200, 171), (3, 5))  # 34 215 keys: 68 tiles of 512 pixels
_FEW_TILES = ((11, 7), (6, 4))


def _inputs(maps, npts, bs, nq, nh, hd, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    shapes, lsi = workloads.level_tensors(maps)
    nl, nk = len(maps), int(shapes.prod(1).sum())
    tensors = (torch.randn(bs, nk, nh, hd, generator=g), torch.rand(bs, nq, nh, nl, npts, 2, generator=g) * 1.2 - 0.1,
               torch.rand(bs, nq, nh, nl, npts, generator=g), torch.randn(bs, nq, nh * hd, generator=g))
    value, loc, attn, gout = (t.to(dtype) for t in tensors)
    return workloads.MsdaInputs(value, shapes, lsi, loc, attn, gout)


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 9), (torch.float32, 16), (torch.float32, 31), (torch.float16, 17), (torch.float16, 20),
                                      (torch.bfloat16, 31), (torch.float16, 63)])
@pytest.mark.parametrize("npts,nq", [(1, 1), (3, 33), (8, 257), (13, 70), (16, 129)])
@pytest.mark.parametrize("maps", [_MANY_TILES, _FEW_TILES], ids=["68-tiles", "2-tiles"])
def test_plain(gpu_device, maps, npts, nq, dtype, hd):
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(_inputs(maps, npts, 2, nq, 3, hd, dtype, 100 * npts + hd), gpu_device, fwd, bwd)


@pytest.mark.parametrize("hd", [9, 16, 32])
@pytest.mark.parametrize("npts,nq,ref_dim", [(1, 5, 2), (3, 65, 4), (8, 131, 2), (4, 31, 4)])
def test_fused(gpu_device, npts, nq, ref_dim, hd):
    g = torch.Generator().manual_seed(1000 + 10 * npts + hd)
    shapes, _ = workloads.level_tensors(_FEW_TILES)
    bs, nh, nl, nk = 2, 4, len(_FEW_TILES), int(shapes.prod(1).sum())
    ref = torch.rand(bs, nq, nl, ref_dim, generator=g)
    inp = (torch.randn(bs, nk, nh, hd, generator=g), shapes, ref, torch.randn(bs, nq, nh, nl, npts, 2, generator=g),
           torch.randn(bs, nq, nh, nl * npts, generator=g), torch.randn(bs, nq, nh * hd, generator=g))
    want = orc.fused_fwd_bwd(*inp, loc_dtype=torch.float32)
    value, _, ref, off, logits, gout = inp
    got = _run(value, *workloads.level_tensors(_FEW_TILES), ref, off, logits, gout, gpu_device)
    _compare(got, want, shapes, ref, off, logits, (FWD_FP32,) + (BWD_FP32,) * 4)
