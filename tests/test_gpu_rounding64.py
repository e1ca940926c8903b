"""The plain FP64 form rounds a particle's gather, kick and push as the oracle does, bit for bit, on
the per-particle kernels and on the tile passes alike: only the sums over particles differ in order
and in fused multiply-adds.  From the same field u*, one kick (imex) or one advance (pc2) of both."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from oracle.pyoracle import Oracle
from oracle.pyoracle import lib as olib
from tests.test_gpu_zero_weights import put

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("deposit", [abi.DK_NGP, abi.DK_CIC, abi.DK_TSC])
@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("what", ["kick", "advance"])
@pytest.mark.parametrize("n", [60, 5000])        # (below and above the line of the tile passes)
def test_particles_are_the_oracles_bit_for_bit(n, what, shear, deposit):
    from athenak_amd.lib import DustContext
    L = 0.1 if shear else 0.5
    mesh, blocks = abi.uniform_mesh((12, 9, 8), (2, 2, 1), ((-L, L),) * 3, ng=2,
                                    bc_x1=abi.DK_X1_SHEAR if shear else abi.DK_X1_PERIODIC)
    pc2 = what == "advance"
    phys = workloads._phys(coupling=abi.DK_PC2 if pc2 else abi.DK_IMEX, sbox=shear, strat=shear,
                           solver=abi.DK_LOCAL if pc2 else abi.DK_DC1, deposit=deposit)
    rng = np.random.default_rng(n + deposit)
    f = rng.random((3, n))
    r = np.zeros((abi.DK_NRDATA, n))
    iv = np.zeros((abi.DK_NIDATA, n), dtype=np.int32)
    for d in range(3):
        r[2 * d] = r[abi.IPX1 + 2 * d] = L * (2.0 * f[d] - 1.0)
        r[2 * d + 1] = r[abi.IPVX1 + 2 * d] = 0.1 * rng.standard_normal(n)
    r[abi.IPTS], r[abi.IPM] = 10.0 ** rng.uniform(-2, 0, n), 1.0 / n
    iv[abi.PTAG] = np.arange(n)
    iv[abi.PGID] = (f[0] * 2).astype(np.int32) + 2 * (f[1] * 2).astype(np.int32)
    o = Oracle(mesh, blocks, phys, n)
    o.rdata()[:, :n], o.idata()[:, :n] = r, iv
    olib().or_set_npart(o.h, n)
    u = np.zeros(o.u0().shape)
    u[:, 0] = 1.0
    o.u0()[:], o.u1()[:] = u, u
    us = 0.1 * rng.standard_normal(o.field(1).shape)
    o.field(1)[:] = us
    g = DustContext(mesh, blocks, phys, n)
    g.load(r, iv, u, u)
    put(g, 1, us)
    st = abi.rk2_stages(0.0, 0.01)[1] if pc2 else abi.imex2p_stages(0.0, 0.01)[0]
    task = "explicit_push" if pc2 else "gather_kick_pmbr"
    g.prof(True)
    g.torch.cuda.synchronize()
    o.task(task, st)
    g.task(task, st)
    g.torch.cuda.synchronize()
    assert ("bins" in g.prof_read()) == (n == 5000)
    np.testing.assert_array_equal(g.rdata[:, :n].cpu().numpy(), o.rdata()[:, :n])
    dg, do = g.field(2), o.field(2)
    assert np.abs(dg - do).max() <= 1e-11 * np.abs(do).max()
    g.check_device_error()
    g.close()
