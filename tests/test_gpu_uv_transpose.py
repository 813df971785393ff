"""The joint transposes of the horizontal sub-steps at the edges of their
strips (58 output columns) and marches (4 to 32 rows, by the size of the
grid): <M x, y> = <x, M^T y> over one step of the linear schemes, on random
island domains, with and without diffusion.  Bound, relative to the norms of
the two sums' factors: 1e-12 in FP64 and 1e-6 in FP32 (a few tens of
roundings per term of random sign; a term lost at an edge is O(1/edge))."""
import pytest
import torch

from code_amd import transport as gt
from tests.test_gpu_adjoint_f32 import adjoint32, adjoint64, dot, problem, tracer_set

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1, 2), (53, 3, 3), (54, 4, 3), (55, 5, 3), (112, 7, 2),
                                  (113, 12, 2), (20, 61, 3), (113, 557, 30)])
@pytest.mark.parametrize("scheme", [gt.UPSTREAM, gt.P2])
def test_dot_product_at_edges(device, scheme, size):
    dom, F, ctx, vel = problem(device, size=size)
    x = tracer_set(dom, 7, 41, device) - 0.5
    y = tracer_set(dom, 7, 43, device) - 0.5
    for AH in (-1.0, 300.0):
        lam, Mx = adjoint32(ctx, 7, 1, 1, F["dt"], x, y, vel, scheme, scheme, AH)
        scale = float(Mx.double().norm() * y.double().norm() +
                      x.double().norm() * lam.double().norm())
        assert abs(dot(Mx, y) - dot(x, lam)) <= 1e-6 * scale, (size, scheme, AH)
        x64, y64 = x[3].double().contiguous(), y[3].double().contiguous()
        lam, Mx = adjoint64(ctx, 1, 1, F["dt"], x64, y64, vel, scheme, scheme, AH)
        scale = float(Mx.norm() * y64.norm() + x64.norm() * lam.norm())
        assert abs(dot(Mx, y64) - dot(x64, lam)) <= 1e-12 * scale, (size, scheme, AH)
