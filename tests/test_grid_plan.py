"""How the planes of the grid sampler are dealt to the workgroups, forward one after the other or each to its own, gradients both by one
kind of workgroups or by two: the library's own plan functions, compiled into a small host program."""
import os
import shutil
import subprocess

import pytest

from drivingsdk_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256

PROGRAM = r"""
#include "msda_capi.hip"
int main()
{
    long long v[7];
    while (scanf("%lld %lld %lld %lld %lld %lld %lld", v, v + 1, v + 2, v + 3, v + 4, v + 5, v + 6) == 7) {
        mxd::GridArgs a;
        if (grid_planes_args((int)v[0], v[1], v[2], v[3], v[4], v[5], v[6], 1, &a) != MXD_OK) return 1;
        if (grid_planes_backward_plan(elem_size((int)v[0]), true, true, &a) != MXD_OK) return 2;
        printf("%d %d %d %d %d ", a.gb_wgs, a.gb_chunks, a.gb_channels, a.gg_chunks, a.sum_chunks);
        if (grid_planes_args((int)v[0], v[1], v[2], v[3], v[4], v[5], v[6], 1, &a) != MXD_OK) return 3;
        if (grid_planes_forward_plan(elem_size((int)v[0]), &a) != MXD_OK) return 4;
        printf("%d %d\n", a.run_px, a.planes);
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.hip").write_text("#include <stdio.h>\n" + PROGRAM)
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-I", os.path.join(ROOT, "drivingsdk_amd", "csrc"),
                    str(d / "plan.hip"), "-o", str(d / "plan"), "-L", libdir, "-lmxd_msda", f"-Wl,-rpath,{libdir}"], check=True,
                   capture_output=True, text=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "plan")], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
        return [tuple(map(int, line.split())) for line in out if line]
    return run


def test_chunks_cover_the_channels_and_keep_the_chip_busy(plans):
    """Every image count from one to several per CU: whole channels, no more chunks than the workspace holds, and no workgroup that walks
    more than a half beyond its share of the planes (128 images and more used to get one chunk each, whatever their number)."""
    cases = [(code, n, c, h, w, ho, wo) for code, h, w, ho, wo in ((0, 64, 176, 24, 176), (1, 80, 160, 20, 60))
             for n in (1, 2, 24, 64, 85, 86, 100, 127, 128, 129, 130, 160, 200, 255, 256, 257, 300, 384, 400, 511) for c in (32, 64, 128, 256)
             if n * c >= CUS]
    for (code, n, c, *_), (wgs, chunks, channels, most, summed, *_) in zip(cases, plans(cases)):
        assert wgs == n * chunks and chunks * channels >= c > (chunks - 1) * channels and 1 <= chunks <= most and summed == chunks
        walked, share = -(-wgs // CUS) * channels, n * c / CUS
        assert walked <= 1.5 * share + 1, (n, c, chunks)


@pytest.mark.parametrize("n,c,out,both", [(257, 1, (24, 176), False), (300, 1, (24, 176), False), (400, 1, (24, 176), True),
                                          (513, 3, (24, 176), False), (520, 16, (24, 176), True), (257, 1, (12, 20), True),
                                          (257, 2, (24, 176), True), (255, 1, (24, 176), False)])
def test_two_kinds_where_the_last_round_would_be_nearly_empty(plans, n, c, out, both):
    """(255 planes of one channel are fewer than the CUs, which the first condition of the plan leaves to the two kinds.)"""
    (wgs, chunks, channels, *_), = plans([(0, n, c, 64, 176) + out])
    assert (wgs > 0) == both and (not both or (wgs, chunks, channels) == (n, 1, c))


@pytest.mark.parametrize("code,n,c,maps,out,runs", [
    (0, 24, 128, (64, 176), (24, 176), True), (1, 24, 128, (64, 176), (24, 176), True), (0, 8, 128, (100, 180), (12, 20), True),
    (0, 130, 16, (100, 180), (64, 96), True), (0, 260, 5, (80, 90), (64, 96), True),
    # few output pixels in long runs, runs that fill half of their rounds, small planes that do not fill theirs
    (0, 170, 256, (58, 114), (17, 23), False), (0, 26, 256, (127, 72), (50, 29), False), (1, 94, 80, (141, 81), (11, 106), False),
    (1, 260, 5, (160, 255), (12, 20), False), (0, 260, 5, (120, 200), (48, 64), False), (0, 130, 16, (75, 75), (96, 96), False),
    (1, 260, 5, (80, 160), (64, 96), False)])
def test_forward_takes_the_form_that_measured_faster(plans, code, n, c, maps, out, runs):
    (*_, run_px, planes), = plans([(code, n, c) + maps + out])
    assert (run_px > 0) == runs and (not runs or planes >= 2)
