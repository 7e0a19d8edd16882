"""Geometric kernel attention with value in LDS at the sizes where its kernels change course, against the CPU oracle: rows of two
to 32 lanes, one to 16 pixels per lane group, more samples than one pass stages, one query and many tiles of them, all samples
on one pixel, channels in two parts, maps just inside and outside of what fits, levels that overlap."""
import pytest
import torch

import mx_driving

from oracle import gka_oracle as gka
from test_gka_gpu import make_inputs, run_gpu
from util import BWD_FP32, FWD_FP32, HALF, rel_err, set_tuning

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _wherever_it_fits(monkeypatch):
    set_tuning(monkeypatch, MXD_MSDA_GKA_SLAB=1)


def compare(inp, device, dtype=torch.float32):
    value, sh, lsi, loc, attn, go = inp
    v, a, g = (t.to(dtype).double() for t in (value, attn, go))
    want = (gka.forward(v, sh, lsi, loc, a),) + gka.backward(v, sh, lsi, loc, a, g)
    got = run_gpu(value, sh, lsi, loc, attn, go, device, dtype=dtype, loc_dtype=torch.float32)
    tol = {torch.float32: (FWD_FP32, BWD_FP32, BWD_FP32), torch.float16: (HALF,) * 3, torch.bfloat16: (2.0 ** -8,) * 3}[dtype]
    for name, g_, w_, t in zip(("output", "grad_value", "grad_attn_weights"), got, want, tol):
        assert rel_err(g_, w_) <= t, (name, rel_err(g_, w_))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,hw", [
    # bs, nq, hd, nh, nl, np; map
    ([2, 700, 8, 2, 1, 7], (9, 13)), ([1, 1, 16, 2, 1, 4], (8, 12)), ([2, 333, 16, 3, 1, 20], (40, 60)), ([1, 911, 32, 2, 2, 9], (17, 19)),
    ([3, 257, 64, 4, 1, 16], (24, 25)), ([1, 130, 128, 2, 1, 5], (10, 20)), ([1, 5000, 32, 1, 1, 1], (3, 5)), ([2, 90, 64, 1, 3, 17], (7, 11)),
    ([1, 300, 16, 2, 1, 17], (60, 68)), ([1, 300, 64, 2, 1, 6], (25, 26)), ([1, 300, 64, 2, 1, 6], (31, 33)), ([2, 257, 64, 2, 1, 18], (24, 48)),
    ([1, 40, 16, 2, 1, 6], (64, 74)),
    # maps whose slab does not fit the LDS but whose scatter does, up to the most pixels it takes
    ([1, 2100, 16, 2, 1, 17], (60, 43)), ([1, 1900, 64, 1, 1, 6], (32, 32)), ([1, 700, 32, 2, 1, 9], (32, 64)), ([1, 300, 16, 1, 2, 9], (32, 64))])
def test_sizes(gpu_device, shape, hw, dtype):
    compare(make_inputs(shape, hw, seed=shape[1]), gpu_device, dtype)


def test_all_samples_on_one_pixel_and_nan_locations(gpu_device):
    inp = list(make_inputs([1, 600, 32, 2, 1, 15], (6, 10), seed=3))
    inp[3] = torch.full_like(inp[3], 2.0)
    compare(inp, gpu_device)
    want = run_gpu(*inp, gpu_device)
    inp[3][:, ::3, :, :, 4] = float("nan")              # no pixel: as with a weight of zero
    got = run_gpu(*inp, gpu_device)
    inp[3][:, ::3, :, :, 4] = 2.0
    inp[4][:, ::3, :, :, 4] = 0.0
    want = run_gpu(*inp, gpu_device)
    assert rel_err(got[0], want[0]) <= FWD_FP32 and rel_err(got[1], want[1]) <= BWD_FP32
    assert (got[2][:, ::3, :, :, 4] == 0).all()


def test_levels_that_overlap(gpu_device):
    value, sh, lsi, loc, attn, go = make_inputs([2, 200, 16, 2, 2, 5], (9, 13), seed=4)
    compare((value, sh, torch.tensor([0, 40]), loc, attn, go), gpu_device)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd", [8, 16, 32, 64])
@pytest.mark.parametrize("offset", [0, 1])
def test_many_tiles_with_border_pixels_of_many_samples(gpu_device, hd, dtype, offset):
    """Workgroups of several tiles, which deal the pixels by their samples in the first one, an infinite row of grad_out and rows of it that
    start on any element: 2500 queries sampling far beyond the border, then none of them inside it."""
    value, sh, lsi, loc, attn, go = make_inputs([1, 2500, hd, 2, 1, 5], (13, 22), seed=hd)
    loc[:, 1700:] = loc[:, 1700:] * 0 - 5.0                     # all on the first pixel
    v, a, g = (t.to(dtype).double() for t in (value, attn, go))
    want = gka.backward(v, sh, lsi, loc, a, g)
    dev = gpu_device
    dv, da = value.to(dev, dtype).requires_grad_(), attn.to(dev, dtype).requires_grad_()
    buf = torch.empty(go.numel() + offset, device=dev, dtype=dtype)[offset:].view(go.shape)
    buf.copy_(go.to(dev, dtype))
    out = mx_driving.geometric_kernel_attention(dv, sh.to(dev), lsi.to(dev), loc.to(dev), da)
    got = torch.autograd.grad(out, (dv, da), buf, retain_graph=True)
    tol = {torch.float32: BWD_FP32, torch.float16: HALF, torch.bfloat16: 2.0 ** -8}[dtype]
    for name, g_, w_ in zip(("grad_value", "grad_attn_weights"), got, want):
        assert rel_err(g_.double().cpu().numpy(), w_) <= tol, name
    buf[0, 7] = float("inf")                                    # pixels that query 7 does not sample stay finite
    gv, ga = torch.autograd.grad(out, (dv, da), buf)
    px = (loc[0, 7, :, 0, :, 1].clamp(0, 12) * 22 + loc[0, 7, :, 0, :, 0].clamp(0, 21)).long()
    for h in range(2):
        hit = torch.zeros(13 * 22, dtype=torch.bool)
        hit[px[h]] = True
        assert torch.isfinite(gv[0, ~hit.to(dev), h]).all() and not torch.isfinite(gv[0, hit.to(dev), h]).any()
    assert torch.isfinite(ga[0, torch.arange(2500, device=dev) != 7]).all()
