"""Levels whose start index is negative: samples on them reach the rows that lie inside the tensor, and only those.  The reference
values come from the oracle on a tensor with rows of zeros in front of the first."""
import numpy as np
import pytest
import torch

from drivingsdk_amd import workloads
from oracle import gka_oracle as gka
from test_gka_gpu import run_gpu as run_gka
from test_msda_gpu import _cell_edge_mask
from util import BWD_FP32, FWD_FP32, half_tol, oracle_all, rel_err, run_gpu, set_tuning

pytestmark = pytest.mark.gpu

_LEVELS, _BEFORE, _NK = ((40, 30), (20, 15), (33, 31), (5, 4)), 1200, 1400
# (the second level ends behind the tensor, the third has three tiles' worth of pixels before it; in the second layout the first
#  level lies before it altogether and the last one, whose tiles come behind all others, reaches into it)
_STARTS = {"some": (0, 1290, -1000, 1200), "all": (-1200, -20, -300, -7)}


@pytest.mark.parametrize("dtype,hd", [(torch.float32, 32), (torch.float32, 9), (torch.float16, 32), (torch.bfloat16, 128)])
@pytest.mark.parametrize("npts", [3, 5])
@pytest.mark.parametrize("starts", sorted(_STARTS))
def test_plain(gpu_device, monkeypatch, starts, npts, dtype, hd):
    set_tuning(monkeypatch, MXD_MSDA_FWD_CU=npts & 1)
    bs, nq, nh, nl = 2, 700, 3, len(_LEVELS)
    g = torch.Generator().manual_seed(hd + npts)
    inp = workloads.MsdaInputs(torch.randn(bs, _NK, nh, hd, generator=g).to(dtype), torch.tensor(_LEVELS), torch.tensor(_STARTS[starts]),
                               (torch.rand(bs, nq, nh, nl, npts, 2, generator=g) * 1.1 - 0.05).to(dtype),
                               torch.rand(bs, nq, nh, nl, npts, generator=g).to(dtype), torch.randn(bs, nq, nh * hd, generator=g).to(dtype))
    rows = torch.zeros(bs, _BEFORE + _NK + 200, nh, hd, dtype=dtype)
    rows[:, _BEFORE:_BEFORE + _NK] = inp.value
    want = [np.asarray(t) for t in oracle_all(inp._replace(value=rows, level_start_index=inp.level_start_index + _BEFORE))]
    want[1] = want[1][:, _BEFORE:_BEFORE + _NK]
    keep = ~_cell_edge_mask(inp)[..., None]
    fwd, bwd = (FWD_FP32, BWD_FP32) if dtype == torch.float32 else (half_tol(dtype),) * 2
    for k, (got, ref) in enumerate(zip(run_gpu(inp, gpu_device), want)):
        assert rel_err(*((got * keep, ref * keep) if k == 2 else (got, ref))) <= (fwd if k == 0 else bwd), k


def test_geometric_kernel_attention(gpu_device):
    """The shared kernels leave the level out of grad_value (and out of nothing else)."""
    bs, nq, nh, hd, npts, nl = 2, 400, 3, 20, 5, len(_LEVELS)
    g = torch.Generator().manual_seed(5)
    starts = torch.tensor(_STARTS["some"])
    loc = torch.stack((torch.randint(-2, 42, (bs, nq, nh, nl, npts), generator=g), torch.randint(-2, 42, (bs, nq, nh, nl, npts), generator=g)), -1).float()
    value, attn = torch.rand(bs, _NK, nh, hd, generator=g), torch.rand(bs, nq, nh, nl, npts, generator=g)
    go = torch.rand(bs, nq, nh * hd, generator=g)
    rows = torch.zeros(bs, _BEFORE + _NK + 200, nh, hd)
    rows[:, _BEFORE:_BEFORE + _NK] = value
    args = rows, torch.tensor(_LEVELS), starts + _BEFORE, loc
    kept = attn * (starts >= 0).reshape(-1, 1)
    want = gka.forward(*args, attn), gka.backward(*args, kept, go)[0][:, _BEFORE:_BEFORE + _NK], gka.backward(*args, attn, go)[1]
    got = run_gka(value, torch.tensor(_LEVELS), starts, loc, attn, go, gpu_device)
    for k, (g_, w_) in enumerate(zip(got, want)):
        assert rel_err(g_, w_) <= (FWD_FP32 if k == 0 else BWD_FP32), k
