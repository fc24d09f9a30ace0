"""The atom-matrix multiply with 32 right-hand sides per work-group (FP32, at least 128 (atom, column) pairs with
chunks), just below and at the fewest pairs that take it, and at many: where few coefficients split the chunk list into
parts, where they do not, and at the 120 coefficients of numax 7, the most LDS it takes.  The action equals the
oracle's to 2e-5, the bound of the action's other FP32 tests."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

E = complex(-0.4, 0.1)


@pytest.mark.parametrize("groups,pairs", [(25, 125), (26, 130), (110, 550)])
@pytest.mark.parametrize("numax", [0, 1, 2, 3, 5, 7])
def test_wide_slices_match_oracle(device, numax, groups, pairs):
    import torch
    sysm = S.make_system(0xA43C0210 + numax, (3, 3, 3), ngauss=4, natoms=5, numax=numax)
    plan = G.GreenPlan(sysm, r_trunc=6.0, sources=[(0, 0, 0)] * groups)
    plan.set_inputs(E)
    atoms = plan.export("IMAGE_ATOM")
    blocks = np.diff(plan.export("PRJ_START").astype(int), axis=1)   # per column group and image
    assert sum(len(set(atoms[row > 0])) for row in blocks) == pairs
    one = G.GreenPlan(sysm, r_trunc=6.0, sources=[(0, 0, 0)])
    one.set_inputs(E)
    x = np.random.default_rng(7).standard_normal((one.nnzb, 2, 64, 64)).astype(np.float32)
    ref = O.Oracle(one, E).action(x.astype(np.float64))
    col = torch.from_numpy(plan.export("COLINDX").astype(np.int64)).to(device)
    xd = torch.empty((plan.nnzb, 2, 64, 64), dtype=torch.float32, device=device)
    xs = torch.from_numpy(x).to(device)
    for c in range(groups):
        xd[col == c] = xs
    yd = torch.empty_like(xd)
    plan.multiply(yd, xd, fp_bits=32)
    first = yd[col == 0]
    assert np.abs(first.cpu().double().numpy() - ref).max() < 2e-5 * np.abs(ref).max()
    for c in range(1, groups):   # the same inputs in every group
        assert torch.equal(yd[col == c], first)
    plan.close()
    one.close()
