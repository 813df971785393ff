"""uv_advect_3d through the strip kernels: every scheme at every strip height
equals the oracle bit for bit, on grids with the edges of strips of 60 columns
and of 4 to 32 rows near the last column and row (whose averages have no
neighbour); infinities, NaN and heights of zero or less give what the kernels
of one sub-step each give; and results written over an input equal those
written beside it (the kernels read the caller's fields directly, so such
calls go through copies)."""
import numpy as np
import pytest
import torch

from code_amd import inputs
from code_amd import transport as gt
from oracle import pyoracle as po
from tests.test_gpu_parity import random_domain, random_fields
from tests.util import to_dev, to_host

pytestmark = pytest.mark.gpu
SCHEMES = [gt.UPSTREAM, gt.P2, gt.SUPERBEE, gt.MUSCL, gt.P2_PDM]
NAMES = ("uu", "vv", "ww", "ho", "hn", "hu", "hv")


def run(ctx, dt, v, scheme, du, dv):
    ctx.uv_advect_3d(dt, *(v[n] for n in NAMES), gt.HALFSPLIT, scheme, scheme, du, dv)


@pytest.mark.parametrize("kind", ["walls", "open", "islands"])
@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("size", [(56, 11, 2), (57, 12, 3), (70, 45, 6), (117, 61, 4)])
def test_every_scheme_and_strip_height(device, scheme, size, kind):
    dom = random_domain(*size, 13, kind)
    F = random_fields(dom, 300, cmax=0.4)
    orc = po.Oracle.from_domain(dom)
    want = np.zeros(dom.shape3), np.zeros(dom.shape3)
    assert orc.uv_advect_3d(F["dt"], *(F[n] for n in NAMES), gt.HALFSPLIT, scheme, scheme,
                            *want) == 0
    v = {n: to_dev(F[n], device) for n in NAMES}
    for rows in (None, 8, 16, 32):
        ctx = gt.Context.from_domain(dom)
        if rows:
            ctx.set_tuning(fused=1, tile=gt.tile_for_rows(rows))
        got = [torch.full_like(v["uu"], 5.0) for _ in range(2)]
        run(ctx, F["dt"], v, scheme, *got)
        for g, w in zip(got, want):
            assert np.array_equal(to_host(g), w, equal_nan=True), rows


@pytest.mark.parametrize("value", [0.0, -1.0, 1e-310, np.nan, np.inf, 1e300])
@pytest.mark.parametrize("name", NAMES)
def test_degenerate_inputs_equal_the_sub_steps(device, name, value):
    dom = random_domain(130, 40, 6, 13, "islands")
    F = random_fields(dom, 300, cmax=0.4)
    m = inputs.uniform(dom.shape3, 61) < 0.003
    m[0] = False
    F[name] = np.where(m, value, F[name])
    v = {n: to_dev(F[n], device) for n in NAMES}
    ctx = gt.Context.from_domain(dom)
    for scheme in SCHEMES:
        res = []
        for fused in (1, 0):
            ctx.set_tuning(fused=fused)
            out = [torch.zeros_like(v["uu"]) for _ in range(2)]
            run(ctx, F["dt"], v, scheme, *out)
            res.append(out)
        for a, b in zip(*res):
            assert bool(((a == b) | (a.isnan() & b.isnan())).all()), scheme


@pytest.mark.parametrize("name", NAMES[:6])
def test_v_result_over_an_input(device, name):
    dom = random_domain(130, 70, 6, 13, "islands")
    ctx = gt.Context.from_domain(dom)
    F = random_fields(dom, 300, cmax=0.4)
    v = {n: to_dev(F[n], device) for n in NAMES}
    a, b, du = (torch.zeros_like(v["uu"]) for _ in range(3))
    run(ctx, F["dt"], v, gt.P2_PDM, a, b)
    run(ctx, F["dt"], v, gt.P2_PDM, du, v[name])
    assert torch.equal(du, a) and torch.equal(v[name], b)


@pytest.mark.parametrize("name", [n for n in NAMES if n != "hu"])
def test_u_result_over_an_input(device, name):
    """the V part then reads the result: as the kernels of one sub-step each do
    (tuning fused = 0, always through copies)"""
    dom = random_domain(130, 70, 6, 13, "islands")
    ctx = gt.Context.from_domain(dom)
    F = random_fields(dom, 300, cmax=0.4)
    v = {n: to_dev(F[n], device) for n in NAMES}
    a, b = torch.zeros_like(v["uu"]), torch.zeros_like(v["uu"])
    run(ctx, F["dt"], v, gt.P2_PDM, a, b)
    res = []
    for fused in (1, 0):
        ctx.set_tuning(fused=fused)
        w = {n: t.clone() for n, t in v.items()}
        dv = torch.zeros_like(a)
        run(ctx, F["dt"], w, gt.P2_PDM, w[name], dv)
        assert torch.equal(w[name], a)
        res.append(dv)
    assert torch.equal(res[0].isnan(), res[1].isnan())
    assert torch.equal(res[0].nan_to_num(), res[1].nan_to_num())
