"""The solver's reductions at the edges of their tiles: column groups whose segments hold 1, 2, 4 and 8 blocks, and on both
sides of the 1,024 blocks up to which the action's per-block products are folded in one pass.  Every column
group of a plan of one repeated source has the density of that source's own solve by the other method, to 1e-7 (two
solutions with residual 1e-10), and its residual, with the FP64 action, is at most the tolerance."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S

pytestmark = pytest.mark.gpu

E = complex(-0.4, 0.3)
TOL = 1e-10


def solve(sysm, groups, r_trunc, **kw):
    p = G.GreenPlan(sysm, r_trunc=r_trunc, sources=[(1, 1, 1)] * groups)
    p.set_inputs(E)
    rho, st = p.solve(tolerance=TOL, max_iterations=2000, **kw)
    assert st["max_residual"] <= TOL
    n = p.nnzb
    p.close()
    return rho, n


@pytest.mark.parametrize("nb,groups,kw", [
    ((8, 8, 8), 2, dict(method="cocg")),                    # segments of 1 block
    ((8, 8, 8), 9, dict(method="tfqmr")),
    ((10, 10, 10), 1, dict(method="cocg")),                 # 1,000 blocks in the group
    ((11, 10, 10), 1, dict(method="cocg")),                 # 1,100
    ((11, 10, 10), 2, dict(method="cocg", fp_bits=32, inner_tolerance=1e-30)),
    ((13, 13, 13), 1, dict(method="cocg")),                 # 2,197: segments of 2 blocks, the last one short
    ((13, 13, 13), 1, dict(method="tfqmr")),
    ((17, 16, 16), 1, dict(method="cocg", fp_bits=32, inner_tolerance=1e-30)),   # 4,352: 4 blocks
    ((21, 20, 20), 1, dict(method="cocg", fp_bits=32, inner_tolerance=1e-30)),   # 8,400: 8 blocks
])
def test_reductions_at_tile_edges(device, nb, groups, kw):
    sysm = S.make_system(0xA43C0300, nb, ngauss=6, natoms=3, numax=2)
    r = 0.5 * max(nb) + 1.0   # no direction is truncated
    rho, n = solve(sysm, groups, r, **kw)
    assert n == groups * nb[0] * nb[1] * nb[2]
    other = dict(method="cocg" if kw["method"] == "tfqmr" else "tfqmr")
    ref, _ = solve(sysm, 1, r, **other)
    err = np.abs(rho - ref).max() / np.abs(ref).max()
    assert err < 1e-7, f"{nb} x {groups} {kw}: {err:.2e}"
