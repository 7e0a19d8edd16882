"""Host-side checks that need no GPU: the C-ABI library loads and exports what the header
declares, argument checking, launch geometry, and the error behaviour of the Python layer."""
import ctypes
import os
import re

import pytest
import torch

import drivingsdk_amd
import mx_driving
from conftest import ROOT
from drivingsdk_amd import _C, _lib, workloads


def test_library_exports_every_declared_symbol():
    with open(os.path.join(ROOT, "include", "mxd_msda.h")) as f:
        header = f.read()
    declared = set(re.findall(r"\b(mxd_(?:msda|dagg|gka|grid_sampler2d)_[a-z_]+)\s*\(", header))
    declared.discard("mxd_msda_plan")
    assert declared == set(_lib.EXPORTS)
    lib = _lib.load()
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.mxd_msda_version() == 103


def test_public_names_match_the_reference_module():
    for mod in (mx_driving, drivingsdk_amd):
        assert mod.multi_scale_deformable_attn == mod.MultiScaleDeformableAttnFunction.apply
        assert callable(mod.npu_multi_scale_deformable_attn_function)
    assert mx_driving._C.multi_scale_deformable_attn is _C.multi_scale_deformable_attn
    assert mx_driving._C.multi_scale_deformable_attn_backward is _C.multi_scale_deformable_attn_backward


@pytest.mark.parametrize("backward", [0, 1])
@pytest.mark.parametrize("dims", [
    # bs, nk, nh, hd, nl, nl_attn, nq, np
    (2, 19947, 8, 32, 4, 4, 19947, 4),
    (6, 30825, 8, 32, 4, 4, 9675, 8),
    (1, 19947, 8, 128, 4, 4, 19947, 4),
    (1, 2400, 5, 16, 3, 3, 27216, 1),
    (3, 2400, 4, 37, 5, 5, 301, 3),
    (1, 2400, 7, 147, 3, 3, 1450, 21),
    (2, 100, 16, 8, 1, 2, 33, 2),
    (1, 100, 1, 256, 1, 1, 1, 1),
    (2, 100, 2, 64, 2, 2, 1000, 4),
])
def test_plan_covers_every_unit_exactly_once(backward, dims):
    bs, nk, nh, hd, nl, nl_attn, nq, npts = dims
    lib = _lib.load()
    for dtype in (0, 1, 2):
        plan = _lib.make_plan(backward, dtype, *dims)
        assert plan.lanes_per_row * plan.units_per_wave == 64
        assert plan.vec * plan.lanes_per_row * plan.npass >= hd
        assert hd % plan.vec == 0
        assert plan.block == 64 * plan.waves_per_block
        if plan.block == 1024:
            # the forward's one-workgroup-per-CU form: a workgroup takes a whole CU's LDS and any multiple of
            # units_per_wave queries, its wavefronts taking groups of units_per_wave in turn
            assert not backward and plan.lds_bytes == 160 * 1024
            assert plan.tile_q % plan.units_per_wave == 0
            assert plan.tile_q <= plan.units_per_wave * plan.waves_per_block * plan.iters
        else:
            # the backward's first kernel gives queries of 25 to 32 samples two units each (16 samples per unit)
            # when its workgroups make one pass
            split = 2 if backward and 24 < nl * npts <= 32 and plan.iters == 1 and plan.units_per_wave >= 2 else 1
            assert plan.tile_q * split == plan.units_per_wave * plan.waves_per_block * plan.iters
            # two workgroups per CU (forward), the default dynamic LDS limit (backward)
            assert plan.lds_bytes <= (64 if backward else 80) * 1024
        seen = {}
        work = (ctypes.c_int32 * 4)()
        for bid in range(plan.grid):
            if not lib.mxd_msda_decode_block(ctypes.byref(plan), bid, bs, nh, nq, ctypes.byref(work)):
                continue
            b, h, q0, q1 = work
            assert 0 <= b < bs and 0 <= h < nh and 0 <= q0 < q1 <= nq and q1 - q0 <= plan.tile_q
            if plan.xcd_mode == 1:
                assert h // plan.heads_per_xcd == bid % 8   # a head never leaves its XCD
            elif plan.xcd_mode == 2:
                assert h == (bid % 8) % nh
            assert (b, h, q0) not in seen
            seen[(b, h, q0)] = q1
        covered = sum(q1 - q0 for (_, _, q0), q1 in seen.items())
        assert covered == bs * nh * nq
        assert len(seen) == bs * nh * plan.ntiles


@pytest.mark.parametrize("backward", [0, 1])
@pytest.mark.parametrize("dtype,hd,share", [(1, 32, 2), (2, 16, 4), (0, 16, 2), (1, 24, 2), (1, 33, 1), (0, 32, 1)])
@pytest.mark.parametrize("bs,nh,nq", [(1, 8, 1), (1, 8, 2300), (3, 4, 130), (6, 8, 77), (5, 2, 33), (2, 16, 65), (2, 12, 65)])
def test_heads_that_share_lines_share_xcds(backward, dtype, hd, share, bs, nh, nq):
    """Rows of up to 64 bytes of neighbouring heads lie in one line of 128 bytes: such heads run on the same XCDs, every (batch element,
    head, tile) once, and every XCD has as many workgroups as any other (but for the last of a part)."""
    lib = _lib.load()
    plan = _lib.make_plan(backward, dtype, bs, 500, nh, hd, 2, 2, nq, 4, 16)
    while nh % share:
        share //= 2
    groups = nh // share
    assert (plan.xcd_mode == 3) == (share > 1 and groups < 8 and 8 % groups == 0)
    if plan.xcd_mode != 3:
        return
    seen, xcds, work = set(), {}, (ctypes.c_int32 * 4)()
    for bid in range(plan.grid):
        if lib.mxd_msda_decode_block(ctypes.byref(plan), bid, bs, nh, nq, ctypes.byref(work)):
            b, h, q0, _ = work
            assert (b, h, q0) not in seen
            seen.add((b, h, q0))
            xcds.setdefault(bid % 8, set()).add(h // share)
    assert len(seen) == bs * nh * plan.ntiles and all(len(g) == 1 for g in xcds.values())
    assert plan.grid == 8 * -(-bs * plan.ntiles * share * groups // 8)


def test_plan_vector_width_follows_alignment_and_head_dim():
    assert _lib.make_plan(0, 0, 1, 10, 1, 32, 1, 1, 1, 1, 16).vec == 4
    assert _lib.make_plan(0, 0, 1, 10, 1, 32, 1, 1, 1, 1, 8).vec == 2
    assert _lib.make_plan(0, 0, 1, 10, 1, 32, 1, 1, 1, 1, 4).vec == 1
    assert _lib.make_plan(0, 1, 1, 10, 1, 32, 1, 1, 1, 1, 16).vec == 8
    assert _lib.make_plan(0, 0, 1, 10, 1, 37, 1, 1, 1, 1, 16).vec == 1
    assert _lib.make_plan(0, 0, 1, 10, 1, 147, 1, 1, 1, 1, 16).npass == 4
    assert _lib.make_plan(0, 1, 1, 10, 1, 250, 1, 1, 1, 1, 16).vec == 2


@pytest.mark.parametrize("dims,fragment", [
    ((1, 10, 1, 257, 1, 1, 1, 1), "less than or equal to 256"),
    ((1, 10, 1, 32, 65, 65, 1, 1), "levels"),
    ((1, 10, 1, 32, 2, 1, 1, 1), "levels"),
    ((0, 10, 1, 32, 1, 1, 1, 1), "empty"),
    ((1, 1 << 22, 8, 32, 1, 1, 1, 1), "2 GiB"),
])
def test_c_abi_rejects_bad_sizes(dims, fragment):
    with pytest.raises(RuntimeError) as e:
        _lib.make_plan(0, 0, *dims)
    assert fragment in str(e.value)
    plan = _lib.Plan()
    assert _lib.load().mxd_msda_make_plan(0, 7, 1, 10, 1, 32, 1, 1, 1, 1, 16, ctypes.byref(plan)) == -1
    assert _lib.load().mxd_msda_make_plan(0, 0, 1, 10, 1, 32, 1, 1, 1, 1, 16, None) == -3


def test_workspace_size():
    lib = _lib.load()
    # bs 2, nk 100, nh 8, hd 32, nl 4, nq 50, np 3.  The first backward kernel runs 32-query workgroups for rows
    # of more than 32 bytes (eight units per wavefront: two workgroups per (batch, head) here) and 64-query ones
    # for shorter rows (sixteen units: one); a workgroup's slab holds two pair records (12 B) per sample (the
    # record area is padded to 256 bytes); the run
    # table has one column per possible tile (nk // 512 + nl) plus one per workgroup, padded to 256 bytes
    def expect(tile_q):
        nwg = -(-50 // tile_q)
        table = -(-(2 * 8 * nwg * (100 // 512 + 4 + 1) * 4) // 256) * 256
        return table + -(-(2 * 8 * nwg * (2 * tile_q * 4 * 3) * 12) // 256) * 256
    image = 2 * 100 * 8 * 32 * 4
    assert lib.mxd_msda_backward_workspace_bytes(0, 2, 100, 8, 32, 4, 4, 50, 3) == expect(32)
    assert lib.mxd_msda_backward_workspace_bytes(1, 2, 100, 8, 32, 4, 4, 50, 3) == expect(32) + image
    assert lib.mxd_msda_backward_workspace_bytes(2, 2, 100, 8, 32, 4, 4, 50, 3) == expect(32) + image
    image16 = 2 * 100 * 8 * 16 * 4
    assert lib.mxd_msda_backward_workspace_bytes(1, 2, 100, 8, 16, 4, 4, 50, 3) == expect(64) + image16
    assert lib.mxd_msda_backward_workspace_bytes(0, 2, 100, 8, 300, 4, 4, 50, 3) == 0  # invalid sizes


def _cpu_inputs(dtype=torch.float32):
    return workloads.reference_test_inputs([1, 7, 8, 2, 2, 3], dtype=dtype)


def test_binding_dtype_checks_raise_before_any_launch():
    inp = _cpu_inputs()
    sh, ls = inp.spatial_shapes.int(), inp.level_start_index.int()
    with pytest.raises(RuntimeError, match="value: float16, bfloat16 or float32"):
        _C.multi_scale_deformable_attn(inp.value.double(), sh, ls, inp.sampling_locations, inp.attention_weights)
    with pytest.raises(RuntimeError, match="value_spatial_shapes: int32 or int64"):
        _C.multi_scale_deformable_attn(inp.value, inp.spatial_shapes.float(), ls, inp.sampling_locations,
                                       inp.attention_weights)
    # int32 and int64 metadata are both taken, but not one of each
    with pytest.raises(RuntimeError, match="value_level_start_index: torch.int64 tensor"):
        _C.multi_scale_deformable_attn(inp.value, inp.spatial_shapes, ls, inp.sampling_locations,
                                       inp.attention_weights)
    with pytest.raises(RuntimeError, match="value_level_start_index: torch.int32 tensor"):
        _C.multi_scale_deformable_attn(inp.value, sh, inp.level_start_index, inp.sampling_locations,
                                       inp.attention_weights)
    with pytest.raises(RuntimeError, match="sampling_locations: float16"):
        _C.multi_scale_deformable_attn(inp.value, sh, ls, inp.sampling_locations.double(), inp.attention_weights)
    with pytest.raises(RuntimeError, match="attention_weights: float16"):
        _C.multi_scale_deformable_attn(inp.value, sh, ls, inp.sampling_locations, inp.attention_weights.long())
    big = torch.zeros(1, 4, 1, 257)
    with pytest.raises(RuntimeError, match="less than or equal to 256"):
        _C.multi_scale_deformable_attn(big, sh, ls, inp.sampling_locations, inp.attention_weights)
    with pytest.raises(RuntimeError, match="grad_output: float16"):
        _C.multi_scale_deformable_attn_backward(inp.value, sh, ls, inp.sampling_locations, inp.attention_weights,
                                                inp.grad_output.double())


def test_cpu_tensors_are_refused_not_silently_computed():
    inp = _cpu_inputs()
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        mx_driving.multi_scale_deformable_attn(inp.value, inp.spatial_shapes, inp.level_start_index,
                                               inp.sampling_locations, inp.attention_weights)


def test_empty_tensors_raise_plain_exception_like_the_reference():
    inp = _cpu_inputs()
    with pytest.raises(Exception, match="can not be a empty Tensor"):
        mx_driving.multi_scale_deformable_attn(inp.value[:0], inp.spatial_shapes, inp.level_start_index,
                                               inp.sampling_locations, inp.attention_weights)


def test_deprecated_alias_warns():
    inp = _cpu_inputs()
    with pytest.warns(DeprecationWarning):
        with pytest.raises(RuntimeError):
            mx_driving.npu_multi_scale_deformable_attn_function(
                inp.value, inp.spatial_shapes, inp.level_start_index, inp.sampling_locations, inp.attention_weights)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libmxd_msda.so"))
    with pytest.raises(ImportError, match="no CPU or eager fallback"):
        _lib.load()


def test_algorithmic_bytes_match_the_published_table():
    """Compulsory HBM bytes per call of the five workloads (decimal MB)."""
    mb = lambda name, dt=torch.float32, bwd=False: workloads.algorithmic_bytes(
        workloads.make_inputs(name, dtype=dt, scale_queries=1.0), backward=bwd) / 1e6
    assert abs(mb("tiny") - 4.87) < 0.01
    assert abs(mb("detr_encoder") - 142.98) < 0.01
    assert abs(mb("detr_encoder_bwd", bwd=True) - 245.11) < 0.01
    assert abs(mb("head_dim_128", torch.float16) - 97.02) < 0.01
    assert abs(mb("bevformer_sca") - 427.16) < 0.01
    assert abs(mb("bevformer_sca", torch.float16) - 213.58) < 0.01


def test_bench_refuses_more_than_one_gpu():
    """This build runs on one GPU: bench.py --gpus N (N > 1) says so and exits before touching a device."""
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 2 and "one GPU" in r.stderr and r.stdout.strip() == ""


def test_fused_backward_workspace_adds_the_reference_point_partials():
    lib = _lib.load()
    args = (0, 2, 19947, 8, 32, 4, 19947, 4)
    plain = lib.mxd_msda_backward_workspace_bytes(0, 2, 19947, 8, 32, 4, 4, 19947, 4)
    assert lib.mxd_msda_fused_backward_workspace_bytes(*args, 2, 0) == plain
    assert lib.mxd_msda_fused_backward_workspace_bytes(*args, 2, 1) == plain + 8 * 2 * 19947 * 4 * 2 * 4
    assert lib.mxd_msda_fused_backward_workspace_bytes(*args, 4, 1) == plain + 8 * 2 * 19947 * 4 * 4 * 4
    assert lib.mxd_msda_fused_backward_workspace_bytes(*args, 3, 1) == 0


def test_reference_module_paths_below_the_package_root():
    """The reference's operator files do ``import mx_driving._C`` (mx_driving/ops/multi_scale_deformable_attn.py:15,38)
    and its package re-exports from ``.ops.<operator>`` (mx_driving/__init__.py:106-113): both paths resolve, to the
    same objects, and ``_C`` carries the names the reference binds (mx_driving/csrc/pybind.cpp:110-111,121-122,131-132,
    205-208)."""
    import importlib
    c = importlib.import_module("mx_driving._C")
    for name in ("multi_scale_deformable_attn", "multi_scale_deformable_attn_backward", "npu_deformable_aggregation",
                 "npu_deformable_aggregation_backward", "geometric_kernel_attention_forward",
                 "geometric_kernel_attention_backward", "grid_sampler2d_v2", "grid_sampler2d_v2_backward"):
        assert callable(getattr(c, name)), name
    assert c.multi_scale_deformable_attn is _C.multi_scale_deformable_attn
    assert c.npu_deformable_aggregation is _C.deformable_aggregation
    m = importlib.import_module("mx_driving.ops.multi_scale_deformable_attn")
    assert m.MultiScaleDeformableAttnFunction is mx_driving.MultiScaleDeformableAttnFunction
    assert m.multi_scale_deformable_attn is mx_driving.multi_scale_deformable_attn
    assert importlib.import_module("mx_driving.ops.npu_deformable_aggregation").npu_deformable_aggregation \
        is mx_driving.npu_deformable_aggregation
    assert importlib.import_module("mx_driving.ops.geometric_kernel_attention").geometric_kernel_attention \
        is mx_driving.geometric_kernel_attention
    assert importlib.import_module("mx_driving.ops.grid_sampler2d_v2").grid_sampler2d_v2 is mx_driving.grid_sampler2d_v2


C_PROGRAM = r"""
/* A C99 host: the header compiles as C, the library links, and the entry points that need no GPU behave. */
#include <stdio.h>
#include <string.h>
#include "mxd_msda.h"

int main(void)
{
    mxd_msda_plan plan;
    int32_t work[4];
    int rc;
    if (mxd_msda_version() != MXD_MSDA_VERSION) return 1;
    if (strcmp(mxd_msda_last_error(), "") != 0) return 2;
    rc = mxd_msda_make_plan(0, MXD_DTYPE_F32, 2, 19947, 8, 32, 4, 4, 19947, 4, 16, &plan);
    if (rc != MXD_OK || plan.vec != 4 || plan.lanes_per_row != 8 || plan.grid == 0) return 3;
    if (!mxd_msda_decode_block(&plan, 0, 2, 8, 19947, work) || work[0] != 0 || work[2] != 0) return 4;
    if (mxd_msda_make_plan(0, 7, 1, 10, 1, 32, 1, 1, 1, 1, 16, &plan) != MXD_E_DTYPE) return 5;
    if (mxd_msda_make_plan(0, MXD_DTYPE_F16, 1, 10, 1, 257, 1, 1, 1, 1, 16, &plan) != MXD_E_SHAPE) return 6;
    if (strstr(mxd_msda_last_error(), "256") == NULL) return 7;
    if (mxd_msda_make_plan(0, MXD_DTYPE_F32, 1, 10, 1, 32, 1, 1, 1, 1, 16, NULL) != MXD_E_NULL) return 8;
    if (mxd_msda_forward(NULL, NULL, NULL, NULL, NULL, NULL, MXD_DTYPE_F32, 1, 10, 1, 32, 1, 1, 1, 1, NULL) != MXD_E_NULL)
        return 9;
    if (mxd_msda_backward_workspace_bytes(MXD_DTYPE_F32 | MXD_META_I64, 2, 100, 8, 32, 4, 4, 50, 3) == 0) return 10;
    if (mxd_msda_backward_workspace_bytes(MXD_DTYPE_F32, 2, 100, 8, 300, 4, 4, 50, 3) != 0) return 11;
    if (mxd_msda_backward_static_limit() != MXD_MSDA_STATIC_SCRATCH_BYTES) return 12;
    printf("ok %d\n", mxd_msda_version());
    return 0;
}
"""


def test_header_compiles_as_c99_and_the_library_links(tmp_path):
    """include/mxd_msda.h through a C compiler (not C++), linked against the built library, run."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    src = tmp_path / "host.c"
    src.write_text(C_PROGRAM)
    exe = tmp_path / "host"
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["gcc", "-std=c99", "-pedantic", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe), "-L", libdir, "-lmxd_msda", f"-Wl,-rpath,{libdir}",
                    "-Wl,-rpath,/opt/rocm/lib"], check=True, capture_output=True, text=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
    assert res.stdout.startswith("ok 103")


def test_backward_runs_every_fallible_step_before_its_first_launch(monkeypatch):
    """A problem that passes the size checks and the workspace check but whose grad_value pass would need more
    workgroups than a launch can have: the call must fail with MXD_E_SHAPE having enqueued nothing.  Without a GPU a
    launch attempted first would have surfaced as MXD_E_LAUNCH instead.  (No pointer is dereferenced on the host.)"""
    if torch.cuda.is_available():
        pytest.skip("meant for a box without a GPU: the sizes describe terabytes of (never touched) memory")
    from util import set_tuning
    set_tuning(monkeypatch, MXD_MSDA_TILE_TARGET=128)   # (small work items: 259 per (batch, head) here)
    lib = _lib.load()
    dims = (1 << 20, 64, 8, 32, 1, 1, 32, 512)   # bs, nk, nh, hd, nl, nl_attn, nq, np
    need = lib.mxd_msda_backward_workspace_bytes(0, *dims)
    assert need > 0
    fake = 4096   # a non-NULL, 16-byte aligned value standing for device pointers that are never used
    rc = lib.mxd_msda_backward(fake, fake, fake, fake, fake, fake, fake, fake, fake, fake, need, 0, *dims, 0, None)
    assert rc == -2, (rc, _lib.last_error())
    assert "workgroups" in _lib.last_error()


def test_backward_plans_stay_inside_the_default_lds_limit():
    """The first backward kernel does not opt in to more than 64 KiB of LDS: for every row size and up to the largest
    key count a call accepts its plan must fit, the launcher falling back to the one-kernel form (no tile counters in
    LDS) where the tile bookkeeping would not."""
    for dtype in (0, 1, 2):
        for hd in (1, 4, 8, 16, 32, 64, 128, 256):
            es = 4 if dtype == 0 else 2
            for nh in (1, 8):
                limit = ((1 << 31) - 1) // (nh * hd * 4)
                for nk in (1000, 500_000, 1_800_000, 2_090_000, 16_000_000, limit):
                    if nk > limit:
                        continue
                    for nl in (1, 4):
                        plan = _lib.make_plan(1, dtype, 1, nk, nh, hd, nl, nl, 1000, 4)
                        assert plan.lds_bytes <= 64 * 1024, (dtype, hd, nh, nk, nl, plan.lds_bytes, es)


@pytest.mark.parametrize("forced", [None, 1])
def test_forward_cu_form_is_refused_beyond_its_index_arithmetic(monkeypatch, forced):
    """The forward's one-workgroup-per-CU form multiplies pixel indices and pixel strides as 24-bit integers and
    addresses the locations, weights and results of a batch element with 32-bit byte offsets: problems beyond that must
    get the general kernel's plan (block != 1024), also when the environment forces the form on
    (reference: the same class of overflow is flagged in kernels/multi_scale_deformable_attn/op_kernel/msda.h:428)."""
    from util import set_tuning
    if forced is not None:
        set_tuning(monkeypatch, MXD_MSDA_FWD_CU=forced)
    # bs, nk, nh, hd, nl, nl_attn, nq, np -- each just beyond one of the limits, all inside what a call accepts
    beyond = [
        (1, (1 << 23) + 1, 8, 4, 4, 4, 300_000, 4),          # key count: 24-bit pixel index
        (2, 19947, 8, 32, 4, 4, 1 << 21, 4),                  # locations of a batch element: 2^21*8*16*8 B = 2 GiB
        (2, 19947, 8, 32, 4, 4, (1 << 21) + 1, 1),            # results of a batch element: > 2 GiB
    ]
    for dtype in (0, 1, 2):
        es = 4 if dtype == 0 else 2
        for dims in beyond:
            bs, nk, nh, hd, nl, nla, nq, npts = dims
            if nk * nh * hd * 4 >= 1 << 31:
                continue
            plan = _lib.make_plan(0, dtype, *dims)
            over_loc = nq * nh * nla * npts * 2 * es >= 1 << 31
            over_out = nq * nh * hd * es >= 1 << 31
            if nk >= 1 << 23 or over_loc or over_out:
                assert plan.block != 1024, (dtype, dims, plan.as_dict())
    # the form is still what the benchmark shape gets (forced or by default)
    assert _lib.make_plan(0, 0, 2, 19947, 8, 32, 4, 4, 19947, 4).block == 1024
    # distance between neighbouring pixels of 2^23 bytes and more (fp32, forced form): general kernel
    if forced:
        plan = _lib.make_plan(0, 0, 1, 60, 32768, 64, 1, 1, 1 << 16, 16)
        assert plan.block != 1024, plan.as_dict()


@pytest.mark.parametrize("code", [0, 1, 2])
@pytest.mark.parametrize("nk,nq,nl,one_tile", [(257, 2185, 1, True), (375, 7156, 1, True), (384, 2185, 1, True), (256, 2185, 1, False),
                                               (385, 2185, 1, False), (375, 2184, 1, False), (375, 2185, 2, False)])
def test_geometric_kernel_attention_keeps_a_small_map_in_one_tile(monkeypatch, code, nk, nq, nl, one_tile):
    """From 3 * 2^20 samples on maps of 257 to 384 pixels go through the grad_value pass as one tile (the size of the workspace
    tells the tile size), for geometric kernel attention alone."""
    lib = _lib.load()
    for hd in (48, 96, 160):
        dims, rest = (24, nk, 4, hd), (nq, 15)

        def sizes():
            return (lib.mxd_gka_backward_workspace_bytes(code, *dims, nl, *rest),
                    lib.mxd_msda_backward_workspace_bytes(code, *dims, nl, nl, *rest))
        by_rule = sizes()
        monkeypatch.setenv("MXD_MSDA_TILE_PX_LOG2", "9")
        _lib.reload_tuning()
        forced = sizes()
        assert (by_rule[0] == forced[0]) == one_tile and by_rule[1] != forced[1]
        monkeypatch.delenv("MXD_MSDA_TILE_PX_LOG2")
        _lib.reload_tuning()


@pytest.mark.parametrize("nk,hd,bs,nq,nh,npts,parts", [
    (375, 64, 1, 400, 8, 6, 1), (2580, 16, 1, 400, 8, 6, 1), (2580, 16, 24, 7156, 4, 15, 1), (900, 64, 24, 7156, 4, 15, 1), (900, 64, 2, 2500, 8, 8, 2),
    (2048, 32, 12, 7156, 4, 15, 1), (2048, 32, 6, 900, 4, 4, 2), (1152, 64, 24, 7156, 4, 15, 2)])
def test_geometric_kernel_attention_takes_channels_whole_where_that_measured_faster(nk, hd, bs, nq, nh, npts, parts):
    """float32, backward: maps whose slab of value exceeds the LDS (the workspace holds the dots of the parts where there are several)."""
    size = _lib.load().mxd_gka_backward_workspace_bytes(0, bs, nk, nh, hd, 1, nq, npts)
    image, dots = bs * nk * nh * hd * 4, parts * bs * nq * nh * npts * 4 if parts > 1 else 0
    assert any(size == (splits * image + 255) // 256 * 256 + dots for splits in range(1, 65))


@pytest.mark.parametrize("code,hd,honoured", [(1, 3, False), (2, 1, False), (1, 4, True), (0, 3, True)])
def test_tile_sizes_that_no_kernel_is_built_for_are_not_taken(monkeypatch, code, hd, honoured):
    """16-bit rows of fewer than 4 channels have the grad_value pass for tiles of 512 pixels alone: there MXD_MSDA_TILE_PX_LOG2
    changes nothing (the size of the workspace tells which tiles a backward call lays its run table out for)."""
    lib = _lib.load()
    dims = (2, 20000, 8, hd, 1, 1, 3000, 4)
    default = lib.mxd_msda_backward_workspace_bytes(code, *dims)
    for v in (7, 8):
        monkeypatch.setenv("MXD_MSDA_TILE_PX_LOG2", str(v))
        _lib.reload_tuning()
        assert (lib.mxd_msda_backward_workspace_bytes(code, *dims) != default) == honoured


@pytest.mark.parametrize("code,dims,takes", [
    # bs, nk, nh, hd, nl, nq, np: measured, this form / the general kernel in us
    (0, (1, 6180, 8, 16, 4, 30000, 8), True),         # 52 / 97: half of the rows from LDS, chunks full
    (1, (1, 19947, 8, 16, 4, 30000, 4), True),        # 40 / 58
    (0, (4, 20017, 8, 16, 5, 14000, 6), True),        # 161 / 218: two chunks, the second nearly full
    (2, (2, 6180, 8, 32, 4, 19947, 4), True),         # 53 / 69
    (1, (1, 30825, 8, 16, 4, 30000, 4), True),        # 51 / 65
    (1, (6, 19700, 8, 64, 3, 9675, 2), False),        # 147 / 83: chunks of 6 samples of 16
    (1, (4, 30825, 8, 96, 4, 14000, 3), False),       # 411 / 244: rows of 16 lanes, most of them from memory
    (0, (3, 30825, 16, 32, 4, 7001, 1), False),       # 107 / 54
    (0, (4, 19947, 16, 32, 4, 14000, 2), False),      # 292 / 193
    (2, (6, 20017, 8, 128, 5, 9675, 4), False),       # 529 / 396: 20 samples in two chunks, conversions
    (0, (2, 30825, 8, 64, 4, 5355, 6), False),        # 138 / 96: slices of 8 MB
    (0, (2, 19947, 8, 32, 4, 900, 4), False),         # too few samples
    (0, (2, 40000, 8, 32, 1, 19947, 16), False),      # no level fits the LDS
])
def test_forward_takes_the_form_that_measured_faster(code, dims, takes):
    bs, nk, nh, hd, nl, nq, npts = dims
    assert (_lib.make_plan(0, code, bs, nk, nh, hd, nl, nl, nq, npts).block == 1024) == takes


@pytest.mark.parametrize("code,nk,nh,hd,nq,npts,split", [
    (1, 19947, 8, 32, 20000, 5, True),      # from 16 384 keys on
    (1, 12000, 8, 32, 20000, 5, False),
    (0, 6000, 8, 32, 20000, 5, True),       # rows of 128 bytes in float32
    (0, 6000, 8, 16, 20000, 5, False),
    (1, 6000, 8, 32, 4096, 5, True),        # 2 x 8 x 4096 units
    (1, 6000, 8, 32, 4097, 5, False),
    (1, 6000, 8, 32, 20000, 7, True),       # from 25 samples on
    (0, 19947, 8, 32, 20000, 4, False)])    # a unit of 16
def test_queries_of_17_to_24_samples_get_two_units_where_it_pays(code, nk, nh, hd, nq, npts, split):
    """The queries per workgroup of the first backward kernel tell: a workgroup that makes one pass holds half as many."""
    plan = _lib.make_plan(1, code, 2, nk, nh, hd, 4, 4, nq, npts)
    assert (plan.tile_q * 2 == plan.units_per_wave * plan.waves_per_block) == split
    # the fused form's workspace is that of whole queries, or of queries from 25 samples on
    lib = _lib.load()
    fused = lib.mxd_msda_fused_backward_workspace_bytes(code, 2, nk, nh, hd, 4, nq, npts, 2, 0)
    assert (fused == lib.mxd_msda_backward_workspace_bytes(code, 2, nk, nh, hd, 4, 4, nq, npts)) == (not split or 4 * npts >= 25)


def test_two_units_for_17_samples_never_cost_a_problem_its_form_or_the_static_array():
    """Sizes just below the limits of the hand-over with whole queries: they keep it (and the static array) although two units per
    query, with twice as many workgroups, would not."""
    lib = _lib.load()
    limit = lib.mxd_msda_backward_static_limit()
    fits = [nq for nq in range(4000, 7000, 16) if lib.mxd_msda_backward_workspace_bytes(0, 1, 19947, 8, 32, 4, 4, nq, 5) <= limit]
    records = 2 * 8 * 20 * 12                                # bytes per query, 2 records of 12 bytes per sample
    whole = lambda nq: -(-nq // 32) * 32 * records + -(-8 * -(-nq // 32) * 43 * 4 // 256) * 256   # (43 = 19947 // 512 + 4 + 1 columns)
    assert max(fits) == max(nq for nq in range(4000, 7000, 16) if -(-whole(nq) // 256) * 256 <= limit)
    # a run table of 256 MiB: 48 (batch, head) pairs, 129 columns
    nk, nl = 64000, 4
    for nq in (320_000, 338_000):
        rows = 48 * -(-nq // 32)
        assert rows * (nk // 512 + nl + 1) * 4 <= 1 << 28 < 2 * rows * (nk // 512 + nl + 1) * 4
        total = lib.mxd_msda_backward_workspace_bytes(1, 6, nk, 8, 32, nl, nl, nq, 5)
        assert total > 48 * nq * 20 * 2 * 12                 # the hand-over is there: not the form with global atomics


def test_the_gather_of_dots_is_built_for_lane_pairs_alone():
    """Rows of four lanes and more have their dots formed by the scatter: of the kernels that gather them one can be launched."""
    import shutil
    import subprocess
    nm = shutil.which("nm")
    if nm is None:
        pytest.skip("no nm")
    names = subprocess.run([nm, "-C", _lib.LIB_PATH], check=True, capture_output=True, text=True).stdout
    gathers = {n for n in names.split("\n") if "__device_stub__gka_slab_kernel" in n and "true>" in n}
    assert len(gathers) == 1 and "float, 1, true" in gathers.pop()


@pytest.mark.parametrize("kernel,report,builds", [
    ("grid_planes_both_kernel", "VGPRs Spill: 0", True), ("grid_planes_both_kernel", "VGPRs Spill: 6", False),
    ("grid_planes_fwd_run_kernel", "VGPRs Spill: 10", False), ("grid_planes_fwd_run_kernel", "", False), ("grid_planes_bwd_kernel", "VGPRs Spill: 2", False)])
def test_the_build_refuses_spilled_registers_where_they_were_lost(tmp_path, kernel, report, builds):
    """The Makefile's rule, with a compiler that reports what it is told to (and with nothing said of the kernels in question)."""
    import shutil
    import subprocess
    if shutil.which("make") is None or shutil.which("awk") is None:
        pytest.skip("no make or awk")
    src = os.path.join(ROOT, "drivingsdk_amd", "csrc")
    for name in os.listdir(src):
        if name == "Makefile" or name.endswith((".hip", ".h")):
            os.makedirs(tmp_path / "a" / "csrc", exist_ok=True)
            shutil.copy(os.path.join(src, name), tmp_path / "a" / "csrc")
    os.makedirs(tmp_path / "include")
    shutil.copy(os.path.join(ROOT, "include", "mxd_msda.h"), tmp_path / "include")
    cc = tmp_path / "cc"
    cc.write_text("#!/bin/sh\nfor a; do last=$a; done\ntouch $last\n"
                  f"echo 'x.hip:1:0: remark: Function Name: _ZN3mxd23{kernel}IfLi9EEEv [-Rpass-analysis=kernel-resource-usage]' >&2\n"
                  f"echo 'x.hip:1:0: remark:     SGPRs Spill: 5 [-Rpass]' >&2\necho 'x.hip:1:0: remark:     {report} [-Rpass]' >&2\n")
    cc.chmod(0o755)
    res = subprocess.run(["make", "-C", str(tmp_path / "a" / "csrc"), "PYTHON=true", f"HIPCC={cc}", "grid_planes.o"], capture_output=True, text=True)
    assert (res.returncode == 0) == builds and (tmp_path / "a" / "csrc" / "grid_planes.o").exists() == builds, res.stderr
