"""The atom-matrix multiply of the dyadic term at the edges of its tiles: one to 120 SHO coefficients (16-row tiles,
k-steps of 4, 64 columns of the matrix at a time), few and many chunks per (atom, column), one and several images per
atom with phases, and both widths of its right-hand-side slices.  The action equals the oracle's to 1e-12 (FP64) and
2e-5 (FP32), the bounds of the action's other tests."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

E = complex(-0.4, 0.1)


def relative_error(plan, k, fp, groups=1):
    import torch
    dt = torch.float64 if fp == 64 else torch.float32
    n = plan.nnzb
    x = np.random.default_rng(5).standard_normal((n // groups, 2, 64, 64))
    x = torch.from_numpy(x).to(dt)
    col = torch.from_numpy(plan.export("COLINDX").astype(np.int64))
    xd = torch.empty((n, 2, 64, 64), dtype=dt)
    for c in range(groups):
        xd[col == c] = x
    yd = torch.empty((n, 2, 64, 64), dtype=dt, device="cuda")
    plan.multiply(yd, xd.cuda(), fp_bits=fp)
    y = yd.cpu().double().numpy()
    one = plan
    if groups > 1:
        one = G.GreenPlan(plan.system, r_trunc=6.0, sources=[(0, 0, 0)])
        one.set_inputs(E, k)
    ref = O.Oracle(one, E, k).action(x.double().numpy())
    return max(np.abs(y[col.numpy() == c] - ref).max() for c in range(groups)) / np.abs(ref).max()


@pytest.mark.parametrize("fp", [64, 32])
@pytest.mark.parametrize("numax", range(8))
def test_every_numax_matches_oracle(device, numax, fp):
    sysm = S.make_system(0xA43C0100 + numax, (4, 3, 5), ngauss=4, natoms=3, numax=numax)
    k = (0.25, -1 / 3.0, 0.1)
    plan = G.GreenPlan(sysm, r_trunc=6.0)
    plan.set_inputs(E, k)
    assert relative_error(plan, k, fp) < (1e-12 if fp == 64 else 2e-5)


def test_many_pairs_take_the_wide_slices(device):
    """At least 512 (atom, column) pairs: 32 right-hand sides per work-group in FP32."""
    sysm = S.make_system(0xA43C0200, (3, 3, 3), ngauss=4, natoms=5, numax=4)
    plan = G.GreenPlan(sysm, r_trunc=6.0, sources=[(0, 0, 0)] * 110)
    plan.set_inputs(E, (0.0, 0.0, 0.0))
    assert plan.nAtoms * plan.nCols >= 512
    assert relative_error(plan, (0.0, 0.0, 0.0), 32, groups=110) < 2e-5
