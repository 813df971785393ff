"""The strip kernels' tuning: 4-row strips and the library's own choice can be
asked for and change no bit of the results; the autotuner reaches the 4-row
strips where the library would take them, and leaves a context's choice alone
when it fails.  The in-step budgets, whose partial sums follow the strips,
tell which choice a context holds."""
import numpy as np
import pytest
import torch

from code_amd import inputs
from code_amd import transport as gt
from tests.test_gpu_adjoint_f32 import VEL, problem, tracer_set

pytestmark = pytest.mark.gpu


def domain(ctx, f, vel):
    return dict(ctx=ctx, f_in=f, f_out=torch.empty_like(f), hires=torch.empty_like(vel[5]),
                budget=torch.zeros(f.shape[0] + 1, dtype=torch.float64, device=f.device),
                **dict(zip(VEL, vel)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_four_rows_and_the_default_again(device, dtype):
    dom, F, ctx, vel = problem(device, seed=5, size=(130, 47, 6))
    f = tracer_set(dom, 4, 11, device).to(dtype)
    d = domain(ctx, f, vel)
    res = []
    for tune in (None, (1, 1, 6), (1, 12, 6), (1, 12, 0), (1, -1, 3), (1, -1, 0)):
        if tune:
            ctx.set_tuning(*tune)
        gt.adv3d_batch([d], 4, F["dt"], gt.P2_PDM, gt.P2_PDM)
        res.append([d[n].clone() for n in ("f_out", "hires", "budget")])
    for r in res[1:]:
        assert torch.equal(r[0][:, 1:], res[0][0][:, 1:]) and torch.equal(r[1][1:], res[0][1][1:])
    assert not torch.equal(res[1][2], res[0][2])  # 32 rows: other partial sums
    assert torch.equal(res[-1][2], res[0][2])
    for bad in ((1, -2, 3), (1, 13, 3), (1, 0, 4), (1, 0, -1)):
        with pytest.raises(gt.GtError):
            ctx.set_tuning(*bad)
    assert gt.strip_rows(gt.tile_for_rows(4)) == (4, 4)
    with pytest.raises(ValueError):
        gt.tile_for_rows(4, 8)


def test_autotune_reaches_four_rows(device):
    """(100 x 100 x 20, one FP64 tracer: 31 us with 4 rows, 38 with 8)"""
    tr = inputs.blob_case(seed=5, imax=100, jmax=100, kmax=20)
    ctx = gt.Context.from_domain(tr.dom)
    vel = [torch.from_numpy(np.ascontiguousarray(a)).to(device)
           for a in (tr.uu, tr.vv, tr.ww, tr.hun, tr.hvn, tr.ho)]
    f = torch.from_numpy(tr.tracers["c"]).to(device)[None].contiguous()
    d = domain(ctx, f, vel)
    del d["budget"]
    bt, bg, ms, table = gt.autotune_batch([d], 1, tr.dt, gt.SUPERBEE, gt.SUPERBEE, reps=20)
    assert bt == 12 and ms < min(table.values()), (bt, ms, min(table.values()))


def test_a_failed_autotune_changes_no_choice(device):
    dom, F, ctx, vel = problem(device, seed=5, size=(130, 47, 6))
    f = tracer_set(dom, 4, 11, device)
    d = domain(ctx, f, vel)
    ctx.set_tuning(1, 1, 3)
    gt.adv3d_batch([d], 4, F["dt"], gt.P2_PDM, gt.P2_PDM)
    want = d["budget"].clone()
    with pytest.raises(gt.GtError):
        gt.autotune_batch([d], 4, F["dt"], gt.P2_PDM, gt.MUSCL)
    gt.adv3d_batch([d], 4, F["dt"], gt.P2_PDM, gt.P2_PDM)
    assert torch.equal(d["budget"], want)
