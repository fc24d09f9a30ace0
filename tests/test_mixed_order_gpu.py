"""The local kernels where their variants meet: 8th- and 16th-order directions in one plan, with periodic images at a
k-point in the 8th-order ones (the other plane's line of an image comes from another lane of the wave), for every kind
and width of the tile shapes.  The action equals the oracle's to 1e-12 (FP64) and 2e-5 (FP32), the bounds of the
action's other tests."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

E, K = complex(-0.3, 0.05), (0.2, -0.35, 0.15)


@pytest.mark.parametrize("kind,columns,lines", [(0, 16, 1), (0, 32, 4), (1, 32, 0), (1, 64, 0), (2, 16, 2), (2, 16, 3),
                                                (2, 32, 2), (2, 32, 3), (2, 64, 2)])
@pytest.mark.parametrize("bc,fd", [((1, 0, 0), (4, 8, 4)), ((0, 1, 0), (8, 4, 8)), ((1, 1, 0), (4, 4, 8)), ((1, 1, 1), (4, 4, 4))])
def test_orders_and_images_match_oracle(device, bc, fd, kind, columns, lines):
    import torch
    sysm = S.make_system(0xA43C0400, (4, 5, 3), ngauss=4, natoms=3, numax=2, bc=bc)
    plan = G.GreenPlan(sysm, r_trunc=3.0, nsources=(2, 1, 1), fd_range=fd)
    plan.set_inputs(E, K)
    x = np.random.default_rng(9).standard_normal((plan.nnzb, 2, 64, 64))
    ref = O.Oracle(plan, E, K).action(x)
    for fp, tol, dt in ((64, 1e-12, torch.float64), (32, 2e-5, torch.float32)):
        if columns == 64 and kind == 2 and fp == 64:
            continue   # no such FP64 shape
        plan.set_tile_shape(fp, kind, columns, lines)
        xd = torch.from_numpy(x).to(device=device, dtype=dt)
        yd = torch.empty_like(xd)
        plan.multiply(yd, xd, fp_bits=fp)
        err = np.abs(yd.double().cpu().numpy() - ref).max() / np.abs(ref).max()
        assert err < tol, f"{bc} {fd} fp{fp}: {err:.2e}"
