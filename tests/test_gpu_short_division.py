"""The FP64 strip kernels' short divisions where their remainders say nothing:
single cells whose numerators lie at the edge of the denormals over layers
thinner than 1 m (the remainder rounds to zero whether or not the quotient is
the nearest), and spikes whose ratio of differences is denormal over a large
denominator (the remainder is normal).  Such cells stand alone in their strip,
so no other lane's test answers for them; Courant number 1 as well, whose
P2-PDM bound is an infinity.  The tolerance is zero: both sides round every
operation the same way."""
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


def both(device, dom, F, f, scheme, AH=-1.0):
    """(GPU, oracle) after one HALFSPLIT step of the tracers f"""
    orc = po.Oracle.from_domain(dom)
    ctx = gt.Context.from_domain(dom)
    out = torch.empty(f.shape, dtype=torch.float64, device=device)
    gt.adv3d_batch([dict(ctx=ctx, f_in=to_dev(f, device), f_out=out,
                         **{n: to_dev(F[n], device) for n in VEL})],
                   len(f), F["dt"], scheme, scheme, AH)
    want = f.copy()
    for t in range(len(f)):
        orc.do_advection_3d(F["dt"], want[t], *(F[n] for n in VEL), F["ho"], gt.HALFSPLIT, scheme,
                            scheme, AH, gt.H_TAG)
    return to_host(out), want


def thin(dom, seed, cmax):
    """layers of 0.25 to 1 m, Courant numbers up to cmax"""
    F = random_fields(dom, seed, cmax=cmax, plateaus=False)
    for n in VEL:
        F[n] = 0.5 * F[n]
    return F


@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("cmax", [0.0, 0.05])
def test_lone_cells_at_the_edge_of_the_denormals(device, scheme, cmax):
    dom = random_domain(290, 90, 8, 5, "open")
    F = thin(dom, 411, cmax)
    sh = (2,) + dom.shape3
    f = np.zeros(sh)
    m = inputs.uniform(sh, 77, 1.0, 2.0)
    e = np.floor(inputs.uniform(sh, 78, -1030.0, -1019.0)).astype(np.int32)
    tiny = np.ldexp(np.where(inputs.uniform(sh, 79) < 0.5, m, -m), e)
    for t, (j, i) in enumerate(((11, 17), (3, 40))):  # one in a strip of either height
        f[t, 1:, j::16, i::60] = tiny[t, 1:, j::16, i::60]
    got, want = both(device, dom, F, f, scheme)
    assert np.count_nonzero(want) >= np.count_nonzero(f)
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("scheme", SCHEMES)
def test_denormal_ratio_over_a_large_difference(device, scheme):
    dom = random_domain(290, 90, 8, 5, "open")
    F = thin(dom, 413, 0.2)
    F["uu"] = np.abs(F["uu"])
    F["vv"], F["ww"] = np.zeros(dom.shape3), np.zeros(dom.shape3)
    f = np.zeros((2,) + dom.shape3)
    m = inputs.uniform(f.shape, 81, 1.0, 2.0)
    for t in range(2):  # 0, tiny, large, 0 along the flow
        f[t, ..., 1::4] = m[t, ..., 1::4] * 1e-289
        f[t, ..., 2::4] = m[t, ..., 2::4] * 10.0 ** (28 + 6 * t)
    got, want = both(device, dom, F, f, scheme)
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_courant_number_one(device, scheme, sign):
    dom = random_domain(130, 40, 5, 7, "islands")
    sh = dom.shape3
    h = np.full(sh, 2.0)
    F = dict(dt=25.0, hu=h, hv=h, ho=h, ww=np.zeros(sh))
    # u/2 and v/2 at Courant number 1: 500 m and 400 m in half of 25 s
    F["uu"], F["vv"] = sign * 40.0 * h, -sign * 32.0 * h
    f = inputs.uniform((2,) + sh, 91, -1.0, 3.0)
    got, want = both(device, dom, F, f, scheme)
    assert np.array_equal(got, want, equal_nan=True), int((got != want).sum())


@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("rows", [8, 16, 32])
def test_tails_through_part_of_the_strips(device, scheme, rows):
    """a tracer that falls off by 10**-3 per cell around two patches: strips
    before, in and past the tail, and tiny values on land"""
    dom = random_domain(190, 120, 4, 9, "islands")
    F = random_fields(dom, 419, cmax=0.3, plateaus=False)
    j, i = np.mgrid[:dom.NY, :dom.NX]
    f = np.zeros((2,) + dom.shape3)
    for t, (cj, ci) in enumerate(((9, 150), (61, 20))):
        d = np.abs(j - cj) + np.abs(i - ci)
        f[t, 1:] = inputs.uniform((dom.kmax,) + d.shape, 95 + t, 1.0, 9.0) * 10.0 ** (-3.0 * d)
    orc = po.Oracle.from_domain(dom)
    ctx = gt.Context.from_domain(dom)
    ctx.set_tuning(fused=1, tile=gt.tile_for_rows(rows), group=2)
    out = torch.empty(f.shape, dtype=torch.float64, device=device)
    gt.adv3d_batch([dict(ctx=ctx, f_in=to_dev(f, device), f_out=out,
                         **{n: to_dev(F[n], device) for n in VEL})], 2, F["dt"], scheme, scheme)
    got = to_host(out)
    for t in range(2):
        orc.do_advection_3d(F["dt"], f[t], *(F[n] for n in VEL), F["ho"], gt.HALFSPLIT, scheme,
                            scheme, -1.0, gt.H_TAG)
        assert np.array_equal(got[t], f[t]), (t, int((got[t] != f[t]).sum()))
