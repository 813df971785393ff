"""do_advection of one slice takes work memory for slices, whatever the number
of levels of its context."""
import pytest
import torch

from code_amd import transport as gt
from tests.test_gpu_parity import random_domain, random_fields
from tests.util import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [gt.FULLSPLIT, gt.HALFSPLIT])
def test_a_slice_takes_slices(device, split):
    res = []
    for kmax in (1, 400):
        dom = random_domain(300, 200, 1, 7, "islands")
        F = random_fields(dom, 407, cmax=0.3)
        dom.kmax = kmax
        v = {n: to_dev(F[n][1], device) for n in ("f", "uu", "vv", "hu", "hv", "ho")}
        di, ad = torch.zeros_like(v["f"]), torch.zeros_like(v["f"])
        ctx = gt.Context.from_domain(dom)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        ctx.do_advection(F["dt"], v["f"], v["uu"], v["vv"], v["hu"], v["hv"], v["ho"], v["ho"],
                         split, gt.MUSCL, -1.0, gt.H_TAG, Dires=di, advres=ad)
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]
        # (a field of the context with 400 levels is 199 MB; the allocator
        # hands out 2 MB at a time, and a first launch may load its kernel)
        assert used <= 64 << 20, (kmax, used)
        res.append((v["f"], di, ad))
    for a, b in zip(*res):
        assert torch.equal(a, b)
