"""Work memory of the reverse mode: with keep_states 0 and 1 the caller's
checkpoint spacing bounds it, the default (which may take the whole window as
one segment) holds no more than that takes, and a change of the mode gives it
back.  Neither the spacing nor the mode changes a bit of the results."""
import gc

import pytest
import torch

from code_amd import inputs
from code_amd import transport as gt
from tests.test_gpu_adjoint_f32 import adjoint32, adjoint64, problem, tracer_set
from tests.util import to_dev

pytestmark = pytest.mark.gpu
SLACK = 48 << 20  # the allocator's granularity and kernels loaded on first use


@pytest.mark.parametrize("scheme", [gt.SUPERBEE, gt.P2_PDM])
def test_spacing_and_mode_change_nothing(device, scheme):
    tr = inputs.blob_case(seed=5, imax=40, jmax=27, kmax=5)
    vel = [to_dev(a, device) for a in (tr.uu, tr.vv, tr.ww, tr.hun, tr.hvn, tr.ho)]
    f0 = tracer_set(tr.dom, 3, 51, device)
    f0[0] = torch.from_numpy(tr.tracers["c"]).float().to(device)
    lam = tracer_set(tr.dom, 3, 53, device) - 0.5
    f64, l64 = f0[0].double().contiguous(), lam[0].double().contiguous()
    ref = None
    for mode in (0, 1, -1):
        for ck in (7, 3, 1, 2):
            ctx = gt.Context.from_domain(tr.dom)
            ctx.set_adjoint_mode(mode)
            got = (adjoint32(ctx, 3, 7, ck, tr.dt, f0, lam, vel, scheme, scheme)
                   + adjoint64(ctx, 7, ck, tr.dt, f64, l64, vel, scheme, scheme))
            ref = ref or got
            for a, b in zip(got, ref):
                assert torch.equal(a, b), (mode, ck)


def test_memory_is_bounded_and_given_back(device):
    dom, F, ctx, vel = problem(device, size=(196, 146, 19))
    n3 = 200 * 150 * 20 * 8
    n, ck = 40, 5
    f = tracer_set(dom, 1, 11, device)[0].double()
    lam = f - 0.5

    def used(mode):
        ctx.set_adjoint_mode(mode)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        res = adjoint64(ctx, n, ck, F["dt"], f, lam, vel, gt.MUSCL, gt.MUSCL)
        return free - torch.cuda.mem_get_info()[0], res

    adjoint64(ctx, 1, 1, F["dt"], f, lam, vel, gt.MUSCL, gt.MUSCL)  # (work fields of a step)
    ctx.set_adjoint_mode(0)  # (nothing held)
    gc.collect()
    torch.cuda.synchronize()
    start = torch.cuda.mem_get_info()[0]
    fields = {0: 5 + 2 + n // ck + ck - 1 + 4, 1: 5 + 2 + n // ck + ck - 1 + 4 * ck,
              -1: 5 + 2 + 1 + n - 1 + 4 * n}
    out = {}
    for mode in (-1, 0, 1, 0, -1):
        u, out[mode] = used(mode)
        assert u <= fields[mode] * n3 + SLACK, (mode, u)
    assert u >= fields[-1] * n3 - SLACK
    # held for the next call, given back with the mode
    adjoint64(ctx, n, ck, F["dt"], f, lam, vel, gt.MUSCL, gt.MUSCL)
    assert start - torch.cuda.mem_get_info()[0] >= fields[-1] * n3 - SLACK
    ctx.set_adjoint_mode(1)
    assert start - torch.cuda.mem_get_info()[0] <= SLACK
    for mode in (0, 1):
        for a, b in zip(out[mode], out[-1]):
            assert torch.equal(a, b)
