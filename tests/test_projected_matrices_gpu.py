"""The two contractions of collected atom coefficients on the GPU at the edges of their launches.

Atomic density matrices: 1 to 120 entries per row (a lane owns entry j and, past 64, entry j + 64), source blocks that do
not fill the four waves; equal to the closed form Im(P_left X P_right) with the projectors evaluated here from their
definition (the left ones over the blocks of the plan's projection lists, which leave out blocks that the sphere only
grazes), to 1e-11 of the largest entry (sums of at most 1e6 terms in FP64).

Adjoint gradient: cells of unequal edges (the grid order of dL/dV) and rows of 1 to 84 entries that do not fill the work-group
of four; with random X and lambda, sum (dL/dM dM) equals -Im sum_c w_c <lambda_c, (A(M + dM) - A(M)) X_c> from two actions
(exact: A is affine in the potential, h and s).  An action rounds at 1e-16 of |A| |X| (|A| of some 1e3), so the difference
of the two products of n random entries is off by about 1e-13 sqrt(n); 1e-9 sqrt(n) |w| is allowed, against values of the order
of sqrt(n)."""
import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S

pytestmark = pytest.mark.gpu


def projectors(pos, apos, L, h):
    """[block][point][entry] of the Hermite-Gauss functions about apos = (x, y, z, 1 / sqrt(sigma)), zero outside the
    sphere of radius 6 sigma (tested in float: z, then y, then x)."""
    i4 = np.arange(4)
    xi = apos[3] ** 2 * ((pos[:, :3, None].astype(float) * 4 + i4 + 0.5) * h - np.asarray(apos[:3])[None, :, None])
    xx = xi * xi
    f = xx.astype(np.float32)
    d2z = f[:, 2] - np.float32(36)
    d2yz = f[:, 1][:, None, :] + d2z[:, :, None]
    d2 = f[:, 0][:, None, None, :] + d2yz[:, :, :, None]
    mask = (d2z < 0)[:, :, None, None] & (d2yz < 0)[:, :, :, None] & (d2 < 0)   # [block][z][y][x]
    H = [np.where(xx < 36.0, np.exp(-0.5 * xx), 0.0)]
    for n in range(L):
        H.append(xi * H[n] - (0.5 * n * H[n - 1] if n else 0.0))
    out = []
    for iz in range(L + 1):
        for iy in range(L + 1 - iz):
            for ix in range(L + 1 - iz - iy):
                p = H[iz][:, 2, :, None, None] * H[iy][:, 1, None, :, None] * H[ix][:, 0, None, None, :]
                out.append((p * mask).reshape(len(pos), 64))
    return np.stack(out, axis=-1)


@pytest.mark.parametrize("numax,nsources", [(0, (1, 1, 1)), (3, (5, 1, 1)), (4, (2, 2, 1)), (5, (3, 1, 1)), (7, (3, 2, 1))])
def test_density_matrices_equal_the_closed_form(device, numax, nsources):
    import torch
    sysm = S.make_system(0xA43C0300 + numax, (6, 5, 7), ngauss=4, natoms=3, numax=numax, bc=(0, 0, 0))
    plan = G.GreenPlan(sysm, r_trunc=3.0, nsources=nsources)
    plan.set_inputs(complex(-0.3, 0.1))
    assert plan.nAtomImages == plan.nAtoms
    X = np.random.default_rng(numax).standard_normal((plan.nnzb, 2, 64, 64))
    D = plan.atom_density_matrices(torch.from_numpy(X).to(device), factor=1.5)
    ipos, lmax = plan.export("IMAGE_POS"), plan.export("IMAGE_LMAX").astype(int)
    col, row = plan.export("COLINDX").astype(int), plan.export("ROWINDX").astype(int)
    Xc = X[:, 0] + 1j * X[:, 1]
    assert len(D) == plan.nAtoms > 0
    start, index = plan.export("PRJ_START").reshape(plan.nCols, -1).astype(int), plan.export("PRJ_INDEX")
    first = np.concatenate([[0], np.cumsum(start[:, -1])])
    for a in range(plan.nAtoms):
        left = projectors(plan.export("ROW_POS")[row], ipos[a], lmax[a], sysm.h)
        listed = np.concatenate([index[first[c] + start[c, a]:first[c] + start[c, a + 1]] for c in range(plan.nCols)])
        left *= np.isin(np.arange(plan.nnzb), listed)[:, None, None]
        right = projectors(plan.export("COL_POS")[col], ipos[a], lmax[a], sysm.h)
        ref = 1.5 * np.einsum("bpi,bpj->ij", left, np.matmul(Xc, right)).imag
        assert np.abs(D[a] - ref).max() <= 1e-11 * np.abs(ref).max(), (numax, a)


@pytest.mark.parametrize("numax,nb,groups", [(0, (4, 3, 5), 1), (1, (3, 5, 4), 3), (3, (5, 4, 3), 5), (6, (4, 3, 3), 2)])
def test_gradient_equals_the_derivative_of_the_action(device, numax, nb, groups):
    import torch
    sysm = S.make_system(0xA43C0310 + numax, nb, ngauss=4, natoms=2, numax=numax)
    plan = G.GreenPlan(sysm, r_trunc=5.0, sources=[(1, 2, 1)] * groups)
    rng = np.random.default_rng(7)
    E = rng.standard_normal(groups) + 1j * rng.uniform(0.1, 1.0, groups)
    w = rng.standard_normal(groups) + 1j * rng.standard_normal(groups)
    plan.set_inputs(E)
    X, Lam = (torch.from_numpy(rng.standard_normal((plan.nnzb, 2, 64, 64))).to(device) for _ in range(2))
    gV, ghs = plan.gradient(X, Lam, E, w)

    def value(V, hs):
        plan.update_potential(V, hs)
        plan.update_energies(E)
        y = torch.empty_like(X)
        plan.multiply(y, X, fp_bits=64)
        z = (torch.complex(Lam[:, 0], -Lam[:, 1]) * torch.complex(y[:, 0], y[:, 1])).sum(dim=(1, 2)).cpu().numpy()
        return -np.imag((w[plan.export("COLINDX").astype(int)] * z).sum())

    base = value(sysm.V, sysm.hs)
    tol = 1e-9 * np.sqrt(2 * X.numel()) * np.abs(w).max()
    dV = rng.standard_normal(sysm.V.shape)
    assert abs((gV * dV).sum() - (value(sysm.V + dV, sysm.hs) - base)) <= tol
    for ia in range(sysm.natoms):
        for which in range(2):
            d = np.zeros_like(sysm.hs[ia])
            d[which] = rng.standard_normal(d[which].shape)
            hs = [m + d if k == ia else m for k, m in enumerate(sysm.hs)]
            assert abs((ghs[ia] * d).sum() - (value(sysm.V, hs) - base)) <= tol, (numax, ia, which)
