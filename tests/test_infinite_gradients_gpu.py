"""An infinite row of grad_output reaches the rows of the maps' gradient that its samples touch, and no other: the pixel to the right of
a map's last column, the next slot of a tile or of a strip and the pixels behind a lane group's last one stay what they are."""
import numpy as np
import pytest
import torch

from drivingsdk_amd import workloads
from util import BWD_FP32, half_tol, oracle_all, rel_err, run_gpu

pytestmark = pytest.mark.gpu


def _touched(maps, starts, nk, loc):
    """Pixels that samples at loc [n, level, point, 2] have as a corner."""
    hit = np.zeros(nk, dtype=bool)
    for l, (h, w) in enumerate(maps):
        x, y = (np.floor(loc[:, l, :, k].astype(np.float64) * n - 0.5).astype(int) for k, n in enumerate((w, h)))
        for dy, dx in ((0, 0), (0, 1), (1, 0), (1, 1)):
            ok = (x + dx >= 0) & (x + dx < w) & (y + dy >= 0) & (y + dy < h)
            hit[starts[l] + ((y + dy) * w + x + dx)[ok]] = True
    return hit


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 9), (torch.float32, 32), (torch.float32, 50), (torch.float32, 128), (torch.float16, 2),
                                      (torch.float16, 32), (torch.float16, 36), (torch.float16, 64), (torch.bfloat16, 100), (torch.bfloat16, 128),
                                      (torch.float32, 130), (torch.float16, 136)])
@pytest.mark.parametrize("maps,nq", [(((1, 505), (3, 2)), 40), (((21, 24), (8, 16), (1, 1)), 300), (((60, 1), (27, 19)), 40), (((5, 6), (1, 9)), 2500)])
def test_gradient_of_the_maps(gpu_device, maps, nq, dtype, hd):
    g = torch.Generator().manual_seed(hd + nq)
    shapes, lsi = workloads.level_tensors(maps)
    bs, nh, nl, npts, nk, at = 2, 2, len(maps), 3, int(shapes.prod(1).sum()), nq // 2
    loc = (torch.rand(bs, nq, nh, nl, npts, 2, generator=g) * 1.2 - 0.1).to(dtype)
    loc[0, at, 0, :, 0, 0] = 1.0 - 0.25 / shapes[:, 1]  # (beyond the centre of the last column: nothing to the right)
    loc[0, at, 0, :, 0, 1] = 1.0 - 0.25 / shapes[:, 0]
    loc[0, at, 0, :, 1, 0] = 0.25 / shapes[:, 1]        # (before the centre of the first one: nothing to the left)
    gout = torch.randn(bs, nq, nh, hd, generator=g).to(dtype)
    gout[0, at, 0] = 0.0
    inp = workloads.MsdaInputs(torch.randn(bs, nk, nh, hd, generator=g).to(dtype), shapes, lsi, loc,
                               (torch.rand(bs, nq, nh, nl, npts, generator=g) + 0.1).to(dtype), gout.flatten(2))
    want = np.asarray(oracle_all(inp)[1]).reshape(bs, nk, nh, hd)
    gout[0, at, 0] = float("inf")
    got = run_gpu(inp._replace(grad_output=gout.flatten(2)), gpu_device)[1].reshape(bs, nk, nh, hd)
    hit = np.zeros((bs, nk, nh), dtype=bool)
    hit[0, :, 0] = _touched(maps, [int(s) for s in lsi], nk, loc[0, at, 0].float().numpy()[None])
    assert 0 < hit.sum() < nk
    assert np.array_equal(~np.isfinite(got).all(-1), hit) and not np.isfinite(got[hit]).any()
    assert rel_err(got[~hit], want[~hit]) <= (BWD_FP32 if dtype == torch.float32 else half_tol(dtype))
