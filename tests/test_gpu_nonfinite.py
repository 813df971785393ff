"""Infinities, NaN, huge tracers and layers of zero, negative or denormal
height in single cells: the FP64 strip kernels equal the oracle, the FP32 ones
and the other splits the kernels of one sub-step each (tuning fused = 0), bit
for bit with NaN in the same cells (tolerance zero: both sides round every
operation the same way).  A missing w face (below level 1, above kmax) carries
no flux and a cell that is not updated keeps its value whatever it is."""
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
VEL = ("uu", "vv", "ww", "hu", "hv", "ho")
KINDS = {"zero": 0.0, "negative": -1.0, "denormal": 1e-310, "nan": np.nan, "inf": np.inf,
         "-inf": -np.inf, "huge": 1e36}
BAD = [(k, w) for k in KINDS for w in ("hu", "hv", "ho", "uu", "ww", "f")]


def problem(kind, where, kmax=6):
    """random fields with the kind's value in 0.3% of the cells of one field,
    land and the top and bottom levels among them (not level 0)"""
    dom = random_domain(130, 40, kmax, 13, "islands")
    F = random_fields(dom, 300, cmax=0.4)
    m = inputs.uniform(dom.shape3, 61) < 0.003
    m[0] = False
    F[where] = np.where(m, KINDS[kind], F[where])
    if where == "ww":
        F["ww"][-1] = 0.0
    return dom, F


def same(a, b):
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


@pytest.mark.parametrize("kind,where", BAD)
def test_fp64_equals_the_oracle(device, kind, where):
    dom, F = problem(kind, where)
    ctx, orc = gt.Context.from_domain(dom), po.Oracle.from_domain(dom)
    v = {n: to_dev(F[n], device) for n in VEL}
    f = np.stack([F["f"], 2.0 * F["f"] - 1.0])
    for q, sch in enumerate(SCHEMES):
        AH = 250.0 if q % 2 else -1.0
        out = torch.empty(f.shape, dtype=torch.float64, device=device)
        gt.adv3d_batch([dict(ctx=ctx, f_in=to_dev(f, device), f_out=out, **v)], 2, F["dt"], sch,
                       sch, AH)
        got = to_host(out)
        for t in range(2):
            want = f[t].copy()
            orc.do_advection_3d(F["dt"], want, *(F[n] for n in VEL), F["ho"], gt.HALFSPLIT, sch,
                                sch, AH, gt.H_TAG)
            assert np.array_equal(got[t], want, equal_nan=True), (sch, t)


@pytest.mark.parametrize("kind,where", BAD)
def test_fp32_strips_equal_the_sub_steps(device, kind, where):
    dom, F = problem(kind, where)
    ctx = gt.Context.from_domain(dom)
    v = {n: to_dev(F[n], device) for n in VEL}
    f = to_dev(np.stack([F["f"] + t for t in range(4)]), device).float()
    for q, sch in enumerate(SCHEMES):
        res = []
        for fused in (1, 0):
            ctx.set_tuning(fused=fused)
            out = torch.empty_like(f)
            gt.adv3d_batch([dict(ctx=ctx, f_in=f, f_out=out, **v)], 4, F["dt"], sch, sch,
                           250.0 if q % 2 else -1.0)
            res.append(out)
        assert same(*res), sch


@pytest.mark.parametrize("split", [gt.FULLSPLIT, gt.HALFSPLIT])
@pytest.mark.parametrize("kind,where", BAD)
def test_other_splits_equal_the_sub_steps(device, split, kind, where):
    dom, F = problem(kind, where)
    ctx = gt.Context.from_domain(dom)
    v = [to_dev(F[n], device) for n in VEL]
    for q, sch in enumerate(SCHEMES):
        AH = 250.0 if q % 2 else -1.0
        # the whole step with all outputs, then its horizontal part alone
        for vs in (sch, gt.NOADV):
            res = []
            for fused in (1, 0):
                ctx.set_tuning(fused=fused)
                f, hr, ad = to_dev(F["f"], device), torch.empty_like(v[0]), torch.empty_like(v[0])
                ctx.do_advection_3d(F["dt"], f, *v, v[5], split, sch, vs, AH, gt.H_TAG, hires=hr,
                                    advres=ad)
                res.append((f, hr, ad))
            for n, a, b in zip(("f", "hires", "advres"), *res):
                assert same(a, b), (sch, vs, n)


@pytest.mark.parametrize("kind,where", BAD)
def test_reverse_mode_equals_the_sub_steps(device, kind, where):
    dom, F = problem(kind, where)
    ctx = gt.Context.from_domain(dom)
    v = [to_dev(F[n], device) for n in VEL]
    f = to_dev(F["f"], device)
    lam = torch.ones_like(f)
    for sch in (gt.P2, gt.SUPERBEE, gt.P2_PDM):
        res = []
        for fused in (1, 0):
            ctx.set_tuning(fused=fused)
            lam0, ff = torch.empty_like(f), torch.empty_like(f)
            ctx.adv3d_adjoint(2, 2, F["dt"], f, lam, lam0, *v, sch, sch, f_final=ff)
            res.append((lam0, ff))
        assert same(res[0][1], res[1][1]), sch
        assert same(res[0][0], res[1][0]), sch
