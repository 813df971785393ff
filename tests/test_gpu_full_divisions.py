"""The second march with full divisions in every form of the strip kernels that
has one, at every strip height (4 rows are the default at this size): tracers
and velocities that run down into the denormals, through HALFSPLIT and
FULLSPLIT with hires and advres and without, a slice of either, the momentum
variants, and the states the reverse mode keeps.  Tolerance zero against the
oracle (or, for the reverse mode, against states recomputed by the kernels of
one sub-step each): both sides round every operation the same way."""
import numpy as np
import pytest
import torch

from code_amd import inputs
from code_amd import transport as gt
from oracle import pyoracle as po
from tests.test_gpu_parity import random_domain, random_fields
from tests.test_gpu_strip_ranges import tiny_tracer
from tests.util import to_dev, to_host

pytestmark = pytest.mark.gpu
SCHEMES = [gt.UPSTREAM, gt.P2, gt.SUPERBEE, gt.MUSCL, gt.P2_PDM]
VEL = ("uu", "vv", "ww", "hu", "hv", "ho")
RANGES = [(-270.0, -307.0), (-300.0, -322.0), (2.0, -320.0)]


@pytest.fixture(scope="module")
def case():
    dom = random_domain(70, 37, 6, 5, "islands")
    return dom, random_fields(dom, 411, plateaus=False), po.Oracle.from_domain(dom)


def context(dom, rows):
    ctx = gt.Context.from_domain(dom)
    if rows:
        ctx.set_tuning(fused=1, tile=gt.tile_for_rows(rows))
    return ctx


@pytest.mark.parametrize("rows", [None, 8, 16, 32])
@pytest.mark.parametrize("top,bottom", RANGES)
@pytest.mark.parametrize("split", [gt.HALFSPLIT, gt.FULLSPLIT])
def test_step(device, case, split, top, bottom, rows):
    dom, F, orc = case
    ctx = context(dom, rows)
    v = [to_dev(F[n], device) for n in VEL]
    f0 = tiny_tracer(dom.shape3, 31, top, bottom)
    for q, sch in enumerate(SCHEMES):
        for vs in (sch, gt.NOADV):
            for outs in (True, False):
                AH = 250.0 if (q + outs) % 2 else -1.0
                want = [f0.copy()] + [np.full(dom.shape3, 7.0) for _ in range(2 * outs)]
                f = to_dev(f0, device)
                got = [f] + [torch.full_like(f, 7.0) for _ in range(2 * outs)]
                kw = dict(zip(("hires", "advres"), want[1:]))
                orc.do_advection_3d(F["dt"], want[0], *(F[n] for n in VEL), F["ho"], split, sch,
                                    vs, AH, gt.H_TAG, **kw)
                kw = dict(zip(("hires", "advres"), got[1:]))
                ctx.do_advection_3d(F["dt"], f, *v, v[5], split, sch, vs, AH, gt.H_TAG, **kw)
                for a, b in zip(got, want):
                    assert np.array_equal(to_host(a), b, equal_nan=True), (sch, vs, outs)


@pytest.mark.parametrize("rows", [None, 8, 16, 32])
@pytest.mark.parametrize("top,bottom", RANGES)
@pytest.mark.parametrize("split", [gt.HALFSPLIT, gt.FULLSPLIT])
def test_slice(device, case, split, top, bottom, rows):
    dom, F, orc = case
    ctx = context(dom, rows)
    host = [np.ascontiguousarray(F[n][2]) for n in ("uu", "vv", "hu", "hv", "ho", "hn")]
    dev = [to_dev(a, device) for a in host]
    f0 = tiny_tracer(dom.shape3, 33, top, bottom)[2].copy()
    for q, sch in enumerate(SCHEMES):
        AH = 250.0 if q % 2 else -1.0
        want = [f0.copy(), np.full_like(f0, 7.0), np.full_like(f0, 7.0)]
        got = [to_dev(a, device) for a in want]
        orc.do_advection(F["dt"], want[0], *host, split, sch, AH, gt.H_TAG, *want[1:])
        ctx.do_advection(F["dt"], got[0], *dev, split, sch, AH, gt.H_TAG, Dires=got[1],
                         advres=got[2])
        for a, b in zip(got, want):
            assert np.array_equal(to_host(a), b, equal_nan=True), sch


@pytest.mark.parametrize("rows", [None, 8, 16, 32])
@pytest.mark.parametrize("top,bottom", RANGES)
def test_momentum(device, case, top, bottom, rows):
    dom, F, orc = case
    ctx = context(dom, rows)
    names = ("uu", "vv", "ww", "ho", "hn", "hu", "hv")
    H = dict(F, uu=tiny_tracer(dom.shape3, 35, top, bottom),
             vv=-tiny_tracer(dom.shape3, 37, top, bottom))
    for sch in SCHEMES:
        want = np.zeros(dom.shape3), np.zeros(dom.shape3)
        orc.uv_advect_3d(F["dt"], *(H[n] for n in names), gt.HALFSPLIT, sch, sch, *want)
        got = [torch.full(dom.shape3, 5.0, dtype=torch.float64, device=device) for _ in range(2)]
        ctx.uv_advect_3d(F["dt"], *(to_dev(H[n], device) for n in names), gt.HALFSPLIT, sch, sch,
                         *got)
        for a, b in zip(got, want):
            assert np.array_equal(to_host(a), b, equal_nan=True), sch


@pytest.mark.parametrize("rows", [None, 8, 16, 32])
@pytest.mark.parametrize("top,bottom", RANGES)
def test_kept_states(device, case, top, bottom, rows):
    dom, F, _ = case
    ctx = context(dom, rows)
    v = [to_dev(F[n], device) for n in VEL]
    f = to_dev(tiny_tracer(dom.shape3, 39, top, bottom), device)
    lam = to_dev(inputs.uniform(dom.shape3, 41, -1.0, 1.0), device)
    for sch in SCHEMES:
        res = []
        for mode in (0, 1):
            ctx.set_adjoint_mode(mode)
            lam0, ff = torch.empty_like(f), torch.empty_like(f)
            ctx.adv3d_adjoint(3, 3, F["dt"], f, lam, lam0, *v, sch, sch, f_final=ff)
            res.append((lam0, ff))
        for a, b in zip(*res):
            assert bool(((a == b) | (a.isnan() & b.isnan())).all()), sch
