"""The reported tile shape is the kernel that runs: the default of a plan on the device, per stencil order, and the
FP32 plane kernel of 32 columns where it is pinned."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S

pytestmark = pytest.mark.gpu

E = complex(-0.3, 0.05)


def plan_of(order, k=(0.25, -1 / 3.0, 0.1)):
    fd = {8: (4, 4, 4), 16: (8, 8, 8), "mixed": (4, 8, 4)}[order]
    if order == 8:   # periodic images at a k-point
        plan = G.GreenPlan(S.make_system(0xA43C0800, (4, 4, 4), ngauss=4, natoms=2, numax=3), r_trunc=6.0, fd_range=fd)
        plan.set_inputs(E, k)
    else:
        sysm = S.make_system(0xA43C0801, (8, 8, 8), ngauss=4, natoms=2, numax=3, bc=(0, 0, 0))
        plan = G.GreenPlan(sysm, r_trunc=3.0, fd_range=fd)
        plan.set_inputs(E)
    return plan


def action(plan, x, fp):
    import torch
    y = torch.empty_like(x)
    plan.multiply(y, x, fp_bits=fp)
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("order,shape", [(8, (2, 32, 2)), (16, (0, 32, 2)), ("mixed", (0, 32, 2))])
def test_reported_default_is_what_runs(device, order, shape):
    import torch
    plan = plan_of(order)
    x = torch.from_numpy(np.random.default_rng(3).standard_normal((plan.nnzb, 2, 64, 64))).to(device)
    for fp, want in ((32, shape), (64, (2, 16, 2))):
        xf = x.float() if fp == 32 else x
        y = action(plan, xf, fp)
        assert plan.tile_shape(fp) == (*want, 0)
        plan.set_tile_shape(fp, *want)
        assert torch.equal(action(plan, xf, fp), y)
    plan.close()


def test_pinned_plane_kernel_is_not_the_line_kernel(device):
    """The two sum in other orders: a random block differs in its last bits, and by no more."""
    import torch
    plan = plan_of(8)
    x = torch.from_numpy(np.random.default_rng(4).standard_normal((plan.nnzb, 2, 64, 64))).to(device).float()
    plan.set_tile_shape(32, 1, 32, 0)
    assert plan.tile_shape(32) == (1, 32, 0, 1)
    plane = action(plan, x, 32)
    assert plan.tile_shape(32) == (1, 32, 0, 1)   # a shape pinned before the plan is on the device stays
    plan.set_tile_shape(32, 2, 32, 2)
    lines = action(plan, x, 32)
    assert not torch.equal(plane, lines)
    assert float((plane - lines).abs().max() / lines.abs().max()) < 2e-5
    plan.close()
