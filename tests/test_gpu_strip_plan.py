"""The strip kernels' own choice of strip heights and tracers per wavefront
(a context without gt_set_tuning) changes no bit: every result and hires
equals the one of a fixed choice (16 rows, 3 tracers per wavefront), for
tracer counts either side of each group size and grids from one strip to the
taller heights."""
import pytest
import torch

from code_amd import transport as gt
from tests.test_gpu_adjoint_f32 import VEL, problem, tracer_set

pytestmark = pytest.mark.gpu


def batch(ctx, f, vel, ntr, dt):
    out, hires = torch.empty_like(f), torch.empty_like(vel[5])
    gt.adv3d_batch([dict(ctx=ctx, f_in=f, f_out=out, hires=hires,
                         **dict(zip(VEL, vel)))], ntr, dt, gt.P2_PDM, gt.P2_PDM)
    return out, hires


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("size,ntrs", [((21, 17, 5), (1, 2, 3, 4, 6, 7, 9, 10, 13, 18)),
                                       ((130, 96, 12), (2, 5, 7, 11)),
                                       ((260, 250, 30), (1, 4)), ((300, 310, 40), (2, 9))])
def test_default_plan_changes_nothing(device, dtype, size, ntrs):
    dom, F, ctx, vel = problem(device, seed=5, kind="islands", size=size)
    fixed = gt.Context.from_domain(dom)
    fixed.set_tuning(fused=1, tile=0, group=3)
    for ntr in ntrs:
        f = tracer_set(dom, ntr, 11, device).to(dtype)
        got, want = batch(ctx, f, vel, ntr, F["dt"]), batch(fixed, f, vel, ntr, F["dt"])
        assert torch.equal(got[0][:, 1:], want[0][:, 1:]), ntr
        assert torch.equal(got[1][1:], want[1][1:]), ntr
