"""Deformable aggregation at the sizes where its kernels change course, against the oracle: groups narrower and wider than a cache
line and than a lane's piece, more locations than a wavefront looks through at once, scale counts that do not divide 64, levels
with so few pixels that their records are split, levels larger than one sort workgroup counts, and level starts that do not
tile the features (rows shared by two levels, rows of none)."""
import numpy as np
import pytest
import torch

from drivingsdk_amd import _lib
from oracle import dagg_oracle as dagg
from test_dagg_gpu import _edge_mask, check, make_inputs, run_gpu
from util import BWD_FP32, FWD_FP32, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,G", [(16, 4), (40, 8), (32, 8), (64, 16), (80, 4), (256, 8), (36, 2), (37, 1), (6, 3), (512, 8), (520, 4), (128, 128)])
def test_group_widths(gpu_device, C, G):
    print(check(make_inputs(2, C, G, 21, 5, [[(9, 13), (5, 7)]] * 2, seed=C, pad=True), gpu_device))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C,G", [(256, 8), (32, 8), (40, 8), (36, 2), (12, 2)])
def test_group_widths_16_bit(gpu_device, C, G, dtype):
    inp = [np.asarray(torch.from_numpy(t).to(dtype).float()) if t.dtype == np.float32 else t
           for t in make_inputs(2, C, G, 21, 5, [[(9, 13), (2, 3)]] * 2, seed=C, pad=True)]
    want = (dagg.direct_forward(*inp[:5]),) + dagg.direct_backward(*inp)
    tol = {torch.float16: 2e-3, torch.bfloat16: 2.0 ** -7}[dtype]
    for k, (g, r) in enumerate(zip(run_gpu(*inp, gpu_device, dtype=dtype), want)):
        assert rel_err(g, r) <= tol, k


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C,G", [(128, 128), (64, 64), (70, 70), (130, 65), (48, 48)])
def test_many_narrow_groups_in_16_bits(gpu_device, C, G, dtype):
    """128 bytes of a row hold 64 groups of one channel: the weights of a wavefront's samples have to fit its share of LDS."""
    inp = [np.asarray(torch.from_numpy(t).to(dtype).float()) if t.dtype == np.float32 else t
           for t in make_inputs(1, C, G, 9, 5, [[(9, 13), (5, 7)]] * 2, seed=C, pad=True)]
    want = (dagg.direct_forward(*inp[:5]),) + dagg.direct_backward(*inp)
    tol = {torch.float16: 2e-3, torch.bfloat16: 2.0 ** -7}[dtype]
    for k, (g, r) in enumerate(zip(run_gpu(*inp, gpu_device, dtype=dtype), want)):
        assert rel_err(g, r) <= tol, k


@pytest.mark.parametrize("P,cams,scales", [(1, 1, 1), (65, 1, 1), (43, 3, 3), (130, 2, 1), (7, 5, 7), (2, 1, 40)])
def test_location_and_scale_counts(gpu_device, P, cams, scales):
    print(check(make_inputs(1, 32, 4, 9, P, [[(6 + s % 3, 7) for s in range(scales)]] * cams, seed=P, pad=True), gpu_device))


def test_few_pixels_many_records(gpu_device):
    print(check(make_inputs(2, 64, 8, 700, 13, [[(11, 12), (2, 3), (1, 1)]], seed=8, pad=True), gpu_device))


def test_a_level_of_several_sort_ranges(gpu_device):
    print(check(make_inputs(1, 16, 2, 150, 9, [[(130, 197), (33, 50)]], seed=9), gpu_device))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_levels_that_do_not_tile_the_features(gpu_device, dtype):
    feat, ss, ssi, loc, w, go = make_inputs(2, 32, 4, 33, 5, [[(9, 13), (5, 7)]], seed=10, pad=True)
    feat = np.concatenate([feat, feat[:, :20]], 1)          # rows that no level covers
    ssi = np.array([[3, 3 + 60]], dtype=np.int32)           # the second level starts inside the first
    inp = (feat, ss, ssi, loc, w, go)
    want = (dagg.direct_forward(*inp[:5]),) + dagg.direct_backward(*inp)
    for k, (g, r) in enumerate(zip(run_gpu(*inp, gpu_device, dtype=dtype), want)):
        assert rel_err(g, r) <= ((FWD_FP32 if k == 0 else BWD_FP32) if dtype == torch.float32 else 4e-3), k


def _shared_map(cams, maps, starts, nf, C, G, A, P, dtype, seed):
    """Inputs (float32 arrays that `dtype` holds exactly) for `cams` cameras whose levels start at `starts` in nf rows."""
    inp = list(make_inputs(2, C, G, A, P, [maps] * cams, seed=seed, pad=True))
    inp[0] = np.random.default_rng(seed).random((2, nf, C), dtype=np.float32)
    inp[2] = np.array(starts, dtype=np.int32).reshape(cams, len(maps))
    return [np.asarray(torch.from_numpy(t).to(dtype).float()) if t.dtype == np.float32 else t for t in inp]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cams,maps,starts,nf,C,G,A,P", [
    # two cameras that name one map: more pixels between them than the tensor has rows
    (2, [(9, 13)], [0, 0], 117, 32, 4, 33, 5),
    (2, [(9, 13)], [0, 0], 117, 256, 8, 33, 5),
    # eight levels of 36 x 41 pixels in 2000 rows: the table of record starts (2000 + 8 * 513 entries) holds four of them
    (8, [(36, 41)], [0, 10, 100, 37, 500, 524, 3, 0], 2000, 64, 8, 41, 3),
    (8, [(36, 41)], [0, 10, 100, 37, 500, 524, 3, 0], 2000, 256, 8, 9, 3),
    # groups that lanes straddle; two scales, the first of which finds room in the first six cameras only, the second everywhere
    (8, [(36, 41), (2, 3)], [0, 1994] * 6 + [524, 5, 3, 1990], 2000, 40, 8, 23, 4)])
def test_levels_that_share_rows(gpu_device, cams, maps, starts, nf, C, G, A, P, dtype):
    """Every level counts in the gradient of the maps, however far the levels overlap."""
    inp = _shared_map(cams, maps, starts, nf, C, G, A, P, dtype, cams + C)
    want = (dagg.direct_forward(*inp[:5]),) + dagg.direct_backward(*inp)
    tol = {torch.float32: BWD_FP32, torch.float16: 2e-3, torch.bfloat16: 2.0 ** -7}[dtype]
    for k, (g, r) in enumerate(zip(run_gpu(*inp, gpu_device, dtype=dtype), want)):
        assert rel_err(g, r) <= tol, k


def _dots_with_rows(inp):
    """Whether the backward forms the dots in the order of the pixels: its workspace has room for them, 16 bytes per sample and group beside
    32 bytes of records per sample."""
    feat, ss, _, loc, w, _ = inp
    (bs, nf, C), (cams, scales), (_, A, P), G = feat.shape, ss.shape[:2], loc.shape[:3], w.shape[-1]
    samples = w.size // G
    need = _lib.load().mxd_dagg_backward_workspace_bytes(0, bs, nf, C, cams, scales, A, P, G)
    return need >= 32 * samples + 16 * G * samples


@pytest.mark.parametrize("C,G,shared", [(256, 8, False), (256, 1, False), (256, 64, False), (512, 16, False), (256, 8, True), (256, 4, "lost")])
def test_dots_with_the_rows(gpu_device, C, G, shared):
    """As many samples as have their dot products formed in the order of the pixels; most lie outside the images.  (Every strip is split
    here, or its level overlaps others: its rows are added to zeros.)"""
    maps = [[(9, 13), (5, 7), (1, 17), (1, 1)]] * 6
    if shared == "lost":
        maps = [[(40, 61), (40, 61), (40, 61), (40, 60)]] * 6
    A = 1440 * 256 // C
    feat, ss, ssi, loc, w, go = make_inputs(2, C, G, A, 31, maps, seed=C + G, pad=True)
    loc[np.random.default_rng(1).random(loc.shape[:3] + (6,)) < 0.97] += 2.0
    if shared:  # every camera names the same rows; "lost": more of them than the table of record starts has room for
        ssi = np.broadcast_to(np.array([0, 17, 5, 60], dtype=np.int32), (6, 4)).copy()
        feat = np.ascontiguousarray(feat[:, :2460 if shared == "lost" else 150])
    assert _dots_with_rows((feat, ss, ssi, loc, w, go))
    print(check((feat, ss, ssi, loc, w, go), gpu_device))


def _around(inp, device, before, after, dtype=torch.float32):
    """Results on the GPU and the oracle's, which reads rows of zeros where a level reaches out of the tensor."""
    feat, ss, ssi, loc, w, go = inp
    rows = np.zeros((feat.shape[0], before + feat.shape[1] + after, feat.shape[2]), dtype=np.float32)
    rows[:, before:before + feat.shape[1]] = feat
    args = rows, ss, (ssi + before).astype(np.int32), loc, w
    want = [dagg.direct_forward(*args), *dagg.direct_backward(*args, go)]
    want[1] = want[1][:, before:before + feat.shape[1]]
    del rows
    torch.full((1 << 27,), float("nan"), device=device)  # (what a workspace finds in its memory)
    return run_gpu(*inp, device, dtype=dtype), want


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("C,G", [(256, 8), (64, 8), (40, 8)])
def test_a_level_that_starts_before_the_tensor(gpu_device, C, G, dtype):
    feat, ss, _, loc, w, go = make_inputs(2, C, G, 33, 5, [[(9, 13), (5, 7)]] * 2, seed=C, pad=True)
    ssi = np.array([[-20, 97], [-117, 290]], dtype=np.int32)  # (the third lies wholly before it, the last one reaches behind it)
    inp = [np.asarray(torch.from_numpy(t).to(dtype).float()) if t.dtype == np.float32 else t for t in (feat, ss, ssi, loc, w, go)]
    tol = {torch.float32: BWD_FP32, torch.float16: 2e-3, torch.bfloat16: 2.0 ** -7}[dtype]
    for k, (g, r) in enumerate(zip(*_around(inp, gpu_device, 117, 40, dtype))):
        assert rel_err(g, r) <= tol, k


def test_a_level_that_starts_before_the_tensor_with_the_rows_dots(gpu_device):
    """The same where the dot products are formed in the order of the pixels: a level without records has its own from elsewhere."""
    feat, ss, _, loc, w, go = make_inputs(2, 256, 8, 1440, 31, [[(9, 13), (5, 7), (1, 17), (1, 1)]] * 6, seed=7, pad=True)
    loc[np.random.default_rng(1).random(loc.shape[:3] + (6,)) < 0.97] += 2.0
    ssi = np.cumsum(np.concatenate([[-50], ss.reshape(-1, 2).prod(1)[:-1]])).reshape(6, 4).astype(np.int32)
    ssi[3, 1] = -30
    inp = feat, ss, ssi, loc, w, go
    assert _dots_with_rows(inp)
    keep = ~_edge_mask(ss, loc)[..., None]
    for k, (g, r) in enumerate(zip(*_around(inp, gpu_device, 50, 10))):
        assert rel_err(*((g * keep, r * keep) if k == 2 else (g, r))) <= (FWD_FP32 if k == 0 else BWD_FP32), k


def _whole_strips(C, G, seed):
    """Samples enough for the dots in the order of the pixels, spread so evenly that most strips of 8 pixels have one wavefront (4 200 of
    them, of up to 884 records if every location were inside), the last ones of a level partly filled; the levels of 17
    pixels are split."""
    inp = make_inputs(2, C, G, 1440 * 256 // C, 31, [[(37, 25), (23, 40), (9, 101), (1, 17)]] * 6, seed=seed, pad=True)
    loc = inp[3]
    keep = np.array([0.3, 0.03, 0.03, 0.03, 0.01, 0.0])
    loc[np.random.default_rng(1).random(loc.shape[:4]) >= keep] += 2.0
    assert _dots_with_rows(inp)
    return inp


@pytest.mark.parametrize("C,G", [(256, 8), (256, 1), (256, 64), (512, 16)])
def test_dots_with_rows_that_are_stored_whole(gpu_device, C, G):
    print(check(_whole_strips(C, G, C + G), gpu_device))


@pytest.mark.parametrize("C,G,dtype", [(256, 8, torch.float32), (64, 8, torch.float32), (40, 8, torch.float32), (6, 2, torch.float32),
                                       (512, 8, torch.float16), (256, 8, torch.bfloat16), (36, 2, torch.float16), ("dots", 8, torch.float32)])
def test_an_infinite_gradient_stays_with_the_rows_it_reaches(gpu_device, C, G, dtype):
    """Rows of the maps' gradient that samples of the anchor have as a corner, in the channels of the group; the pixel to the right of a
    map's last column and the second pixel of the strip to the right of a sample do not."""
    if C == "dots":
        C, inp = 256, _whole_strips(256, G, 3)
        feat, ss, ssi, loc, w, go = inp
        loc[1, 5, :, :2] = np.random.default_rng(2).random(loc[1, 5, :, :2].shape)
    else:
        feat, ss, ssi, loc, w, go = make_inputs(2, C, G, 33, 9, [[(9, 13), (21, 24), (1, 1)]] * 2, seed=C, pad=True)
    loc[1, 5, 0, 0], loc[1, 5, 1, 0] = 0.99, 0.01
    feat, loc, w, go = (np.asarray(torch.from_numpy(t).to(dtype).float()) for t in (feat, loc, w, go))
    hd = C // G
    go[1, 5, :hd] = 0
    want = dagg.direct_backward(feat, ss, ssi, loc, w, go)[0].reshape(2, -1, G, hd)
    go[1, 5, :hd] = np.inf
    hit = np.zeros(want.shape[:3], dtype=bool)
    for cam in range(ss.shape[0]):
        x, y = loc[1, 5, :, cam].astype(np.float64).T
        ok = (x > 0) & (x < 1) & (y > 0) & (y < 1)
        for sc in range(ss.shape[1]):
            h, wd = ss[cam, sc]
            x0, y0 = np.floor(x[ok] * wd - 0.5).astype(int), np.floor(y[ok] * h - 0.5).astype(int)
            for yy, xx in ((y0, x0), (y0, x0 + 1), (y0 + 1, x0), (y0 + 1, x0 + 1)):
                m = (yy >= 0) & (yy < h) & (xx >= 0) & (xx < wd)
                hit[1, ssi[cam, sc] + (yy * wd + xx)[m], 0] = True
    got = run_gpu(feat, ss, ssi, loc, w, go, gpu_device, dtype=dtype)[1].reshape(want.shape)
    assert 0 < hit.sum() < hit[1, :, 0].size
    assert np.array_equal(~np.isfinite(got).all(-1), hit) and not np.isfinite(got[hit]).any()
    assert rel_err(got[~hit], want[~hit]) <= {torch.float32: BWD_FP32, torch.float16: 2e-3, torch.bfloat16: 2.0 ** -7}[dtype]
