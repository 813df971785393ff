"""FULLSPLIT and the 2-D splits through the strip march equal the kernels of
one sub-step each (tuning fused = 0, held to the oracle elsewhere) bit for
bit: every tag and scheme, schemes that differ between the horizontal and the
vertical, diffusion on and off, level counts either side of the w sub-step's
chunks (at least 4 levels each), with and without the optional outputs, and
the result heights written over the heights given."""
import pytest
import torch

from code_amd import transport as gt
from tests.test_gpu_adjoint_f32 import VEL, problem, tracer_set

pytestmark = pytest.mark.gpu
SCHEMES = [gt.UPSTREAM, gt.P2, gt.SUPERBEE, gt.MUSCL, gt.P2_PDM]


def same(a, b):
    return torch.equal(a, b) or bool(((a == b) | (a.isnan() & b.isnan())).all())


@pytest.mark.parametrize("tag", [gt.H_TAG, gt.U_TAG, gt.V_TAG, gt.W_TAG])
@pytest.mark.parametrize("kmax", [2, 3, 8, 9, 13, 31])
def test_fullsplit(device, tag, kmax):
    dom, F, ctx, vel = problem(device, seed=7, kind="islands", size=(67, 19, kmax))
    v = dict(zip(VEL, vel))
    f0 = tracer_set(dom, 1, 11, device)[0].double()
    for q, hs in enumerate(SCHEMES):
        vs, AH = SCHEMES[(q + kmax) % 5], (250.0 if (q + kmax) % 2 else -1.0)
        for vsch, outs in ((vs, True), (vs, False), (gt.NOADV, True)):
            res = []
            for fused in (1, 0):
                ctx.set_tuning(fused=fused, tile=(q + kmax) % 3, group=1)
                f = f0.clone()
                hr, ad = (torch.full_like(f, 7.0) for _ in range(2))
                ctx.do_advection_3d(F["dt"], f, v["uu"], v["vv"], v["ww"], v["hu"], v["hv"],
                                    v["ho"], v["ho"], gt.FULLSPLIT, hs, vsch, AH, tag,
                                    hires=hr if outs else None, advres=ad if outs else None)
                res.append((f, hr, ad))
            for a, b in zip(*res):
                assert same(a, b), (hs, vsch, AH, outs)


@pytest.mark.parametrize("split", [gt.FULLSPLIT, gt.HALFSPLIT])
@pytest.mark.parametrize("tag", [gt.H_TAG, gt.U_TAG, gt.V_TAG])
@pytest.mark.parametrize("size", [(3, 3, 1), (59, 9, 1), (61, 33, 1), (130, 70, 1)])
def test_slice(device, split, tag, size):
    dom, F, ctx, vel = problem(device, seed=9, kind="islands", size=size)
    uu, vv, ww, hu, hv, ho = (t[1].contiguous() for t in vel)
    f0 = tracer_set(dom, 1, 11, device)[0, 1].double()
    for q, sch in enumerate(SCHEMES):
        AH = 250.0 if q % 2 else -1.0
        for outs in ("both", "none", "Do"):
            res = []
            for fused in (1, 0):
                ctx.set_tuning(fused=fused)
                f, Do, ad = f0.clone(), ho.clone(), torch.full_like(f0, 7.0)
                di = {"both": torch.full_like(f0, 7.0), "none": None, "Do": Do}[outs]
                ctx.do_advection(F["dt"], f, uu, vv, hu, hv, Do, ho, split, sch, AH, tag,
                                 Dires=di, advres=ad if outs != "none" else None)
                res.append([f, ad] + ([di] if di is not None else []))
            for a, b in zip(*res):
                assert same(a, b), (sch, AH, outs)
