"""The backward's first kernel for rows of up to 128 bytes whose workgroups make one pass: rows that no piece divides, odd sample counts
with one unit per query and with two, more tiles than a wavefront has lanes, workgroups that are partly or wholly without queries
-- against the oracle, plain and fused.  Rows of 33 to 64 bytes are shared by 4 lanes in launches of more than 1792 workgroups, by 8
in smaller ones: the first two tests have the smaller ones, the last two the larger ones."""
import numpy as np
import pytest
import torch

from drivingsdk_amd import _lib, workloads
from oracle import msda_oracle as orc
from test_msda_fused_gpu import _compare, _edge_masks, _run
from test_msda_gpu import _check_all
from util import BWD_FP32, FWD_FP32, half_tol, rel_err, run_gpu, set_tuning

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


_CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def _takes_4_lanes(bs, nk, nh, hd, nl, nq, npts, dtype):
    """(The library's plan is of rows read in whole pieces, the launch's of rows read in pieces that overlap: those of 64 bytes agree.)"""
    size = torch.finfo(dtype).bits // 8
    plan = _lib.make_plan(1, _CODE[dtype], bs, nk, nh, 64 // size, nl, nl, nq, npts)
    return 32 < hd * size <= 64 and plan.lanes_per_row * plan.vec * size == 64 and plan.iters == plan.npass == 1 and plan.grid > 1792


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 9), (torch.float32, 15), (torch.float32, 16), (torch.float16, 17), (torch.float16, 20),
                                      (torch.float16, 32), (torch.bfloat16, 31), (torch.bfloat16, 32)])
@pytest.mark.parametrize("nl,npts", [(1, 1), (2, 3), (1, 13), (2, 8), (2, 13), (2, 16)])
def test_plain_by_4_lanes(gpu_device, monkeypatch, nl, npts, dtype, hd):
    """Units of 1, 6, 13 and 16 samples, two units of 16 per query; the last workgroup of a (batch, head) has a query or a few.  The gradients
    of the locations and weights are the general kernel's bit for bit where 16-byte pieces divide the row (otherwise the last piece
    of 16 bytes shares more channels with the one before it than one of 8 does, and the sums are formed in another order)."""
    bs, nh, maps = 2, 8, _FEW_TILES[:nl] if npts != 8 else _MANY_TILES
    nq = 1793 if nl * npts > 16 else 3585 + npts
    nk = sum(h * w for h, w in maps)
    assert _takes_4_lanes(bs, nk, nh, hd, nl, nq, npts, dtype)
    inp = _inputs(maps, npts, bs, nq, nh, hd, dtype, 10 * npts + hd)
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    _check_all(inp, gpu_device, fwd, bwd)
    if hd * inp.value.element_size() % 16 != 0:
        return
    got = run_gpu(inp, gpu_device)
    set_tuning(monkeypatch, MXD_MSDA_BWD_FIXED=0)
    general = run_gpu(inp, gpu_device)
    assert np.array_equal(got[2], general[2]) and np.array_equal(got[3], general[3])


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 9), (torch.float32, 16), (torch.float16, 32), (torch.bfloat16, 31), (torch.bfloat16, 32)])
@pytest.mark.parametrize("npts,ref_dim", [(1, 2), (3, 4), (4, 2), (8, 4), (7, 2)])
def test_fused_by_4_lanes(gpu_device, npts, ref_dim, dtype, hd):
    g = torch.Generator().manual_seed(100 * npts + hd)
    shapes, lsi = workloads.level_tensors(_FEW_TILES)
    bs, nh, nl, nk, nq = 2, 8, len(_FEW_TILES), int(shapes.prod(1).sum()), 3585 + npts
    assert _takes_4_lanes(bs, nk, nh, hd, nl, nq, npts, dtype)
    value, ref, off, logits, gout = (t.to(dtype) for t in (
        torch.randn(bs, nk, nh, hd, generator=g), torch.rand(bs, nq, nl, ref_dim, generator=g), torch.randn(bs, nq, nh, nl, npts, 2, generator=g),
        torch.randn(bs, nq, nh, nl * npts, generator=g), torch.randn(bs, nq, nh * hd, generator=g)))
    want = orc.fused_fwd_bwd(value.double(), shapes, ref.double(), off.double(), logits.double(), gout.double(), loc_dtype=torch.float32)
    got = _run(value, shapes, lsi, ref, off, logits, gout, gpu_device)
    # 16-bit results are rounded once (bfloat16: by up to 2^-9 of themselves); the logits' gradient takes a sum from the rounded
    # forward result and is rounded itself
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else half_tol(dtype)
    near, ref_near = _edge_masks(shapes, ref, off, logits)
    assert near.mean() < 1e-2
    keep = {2: ~ref_near[..., None], 3: ~near[..., None]}
    for k, (g_, w_) in enumerate(zip(got, want)):
        lim = (FWD_FP32 if k == 0 else BWD_FP32) if dtype == torch.float32 else 2 * tol if k == 4 else tol
        assert rel_err(g_ * keep.get(k, 1), w_.numpy() * keep.get(k, 1)) <= lim, k
