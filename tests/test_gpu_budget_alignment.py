"""Budgets formed in the batched step where the work fields before their
partials hold an odd number of values (odd NX, NY and level count, odd tracer
counts): the partials, read in pairs, start on 16 bytes, in a context grown on
demand and in one reserved for just this call.  The launch refuses any other
start.  Bound against the error-free pass: 1e-14 relative (a lane's sum of at
most 32 products of one sign and the six-level tree are within 38 roundings,
4.2e-15)."""
import numpy as np
import pytest
import torch

from code_amd import inputs
from code_amd import transport as gt
from tests.test_gpu_parity import random_domain, random_fields
from tests.util import to_dev

pytestmark = pytest.mark.gpu
VEL = ("uu", "vv", "ww", "hu", "hv", "ho")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ntr", [1, 2, 3, 7])
@pytest.mark.parametrize("reserve", [False, True])
def test_odd_work_fields(device, dtype, ntr, reserve):
    dom = random_domain(21, 15, 4, 5, "islands")  # 25 x 19 x 5 values a field
    F = random_fields(dom, 405, cmax=0.02)
    ctx = gt.Context.from_domain(dom)
    if reserve:
        ctx.reserve(**{"ntracers_f32" if dtype == torch.float32 else "ntracers_f64": ntr})
    f = to_dev(np.stack([inputs.uniform(dom.shape3, 7 + t, 1.0, 2.0) for t in range(ntr)]),
               device).to(dtype)
    out, hires = torch.empty_like(f), to_dev(F["ho"], device)
    bud = torch.full((ntr + 1,), float("nan"), dtype=torch.float64, device=device)
    gt.adv3d_batch([dict(ctx=ctx, f_in=f, f_out=out, hires=hires, budget=bud,
                         **{n: to_dev(F[n], device) for n in VEL})], ntr, F["dt"], gt.MUSCL,
                   gt.MUSCL)
    for t in range(ntr):
        m, v = ctx.budget(hires, out[t])
        assert abs(bud[t].item() - m) <= 1e-14 * abs(m)
        assert abs(bud[ntr].item() - v) <= 1e-14 * abs(v)
