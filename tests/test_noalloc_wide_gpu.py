"""gfa_action_noalloc on plans of numax 7 atoms whose buffers just fit its 64 MiB: it asks for the projection partial
sums, the addition coefficients and the zero block, and for nothing that the action does not use."""
import ctypes as C

import numpy as np
import pytest

from angstromcube_amd import gfa as G
from angstromcube_amd import synthetic as S

pytestmark = pytest.mark.gpu

SCRATCH = 64 << 20


def buffers(plan, fp):
    """Bytes of the action's buffers: zero block, partial sums of every chunk, addition coefficients."""
    nsho = lambda name: np.array([S.nsho(int(n)) for n in plan.export(name)])
    blocks = np.diff(plan.export("PRJ_START").astype(int), axis=1)      # per column group and image
    K = min(16, max(2, int(blocks.sum()) // 4096))                      # blocks per chunk
    partial = int((-(-blocks // K) * nsho("IMAGE_LMAX")).sum())
    return (8192 + (partial + plan.sizes.natomcoeffs * plan.nCols) * 128) * fp // 8


@pytest.mark.parametrize("fp,r,fits", [(64, 0.3, True), (32, 0.5, True), (64, 0.5, False)])
def test_wide_atoms_up_to_the_scratch(device, fp, r, fits):
    import torch
    sysm = S.make_system(0xA43C0700, (2, 2, 2), ngauss=2, natoms=8, numax=7, bc=(0, 0, 0))
    plan = G.GreenPlan(sysm, r_trunc=r, sources=[(1, 1, 1)] * 20)
    plan.set_inputs(complex(-0.4, 0.1))
    assert (buffers(plan, fp) <= SCRATCH) == fits
    dt = torch.float64 if fp == 64 else torch.float32
    plan.prepare(fp)
    x = torch.from_numpy(np.random.default_rng(6).standard_normal((plan.nnzb, 2, 64, 64))).to(device=device, dtype=dt)
    y, ref = torch.full_like(x, float("nan")), torch.empty_like(x)
    st = G.lib().gfa_action_noalloc(plan.h, fp, C.c_void_p(y.data_ptr()), C.c_void_p(x.data_ptr()),
                                    C.c_void_p(torch.cuda.current_stream().cuda_stream), None)
    torch.cuda.synchronize()
    if fits:
        assert st == G.GFA_OK, G.lib().gfa_last_error()
        plan.multiply(ref, x, fp_bits=fp)
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
    else:
        assert st == G.GFA_ERR_ARGUMENT and b"allocation-free" in G.lib().gfa_last_error()
    plan.close()
