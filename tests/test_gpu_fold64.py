"""The ghost fold of the FP64 form at the block shapes where it can go wrong: blocks narrower than
two ghost widths (a cell near both faces of an axis), exactly two, odd ones, blocks that are their
own neighbours, sheared and walled faces.  Three steps against the oracle: velocities and gas
momenta within 1e-11 of the largest, block ids equal (the form's own bar, test_gpu_parity.py)."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("faces", ["periodic", "shear", "reflect"])
@pytest.mark.parametrize("nx,nb", [((2, 3, 4), (3, 2, 2)), ((3, 2, 2), (1, 3, 4)),
                                   ((4, 4, 4), (1, 2, 3)), ((5, 8, 4), (2, 2, 1)),
                                   ((9, 6, 7), (2, 1, 3)), ((32, 16, 12), (1, 1, 1))])
def test_fold_against_the_oracle(nx, nb, faces):
    import torch
    from athenak_amd.lib import DustContext
    shear = faces == "shear"
    mesh, blocks = abi.uniform_mesh(
        nx, nb, ((-0.5, 0.5),) * 3, ng=2,
        bc_x1=abi.DK_X1_SHEAR if shear else abi.DK_X1_PERIODIC,
        bc_x3=abi.DK_X3_REFLECT if faces == "reflect" else abi.DK_X3_PERIODIC)
    su = workloads._setup(seed=9, ppc=3, taus=(0.1,), eps=(0.5,), gas_noise=0.3, dust_noise=0.6)
    src = abi.dk_gas_src(shearing_box=1, stratified=0, omega0=1.0, qshear=1.5,
                         const_accel=0.1, const_accel_dir=1) if shear else None
    w = workloads.Workload("fold", mesh, blocks, workloads._phys(sbox=shear), su, src, 2e-3, 3)
    o = Oracle(w.mesh, w.blocks, w.phys, w.npart + 16, threads=1)
    o.setup(w.setup)
    g = DustContext(w.mesh, w.blocks, w.phys, w.npart + 16)
    g.load(o.rdata()[:, :o.npart].copy(), o.idata()[:, :o.npart].copy(), o.u0().copy())
    for _ in range(w.steps):
        o.step(w.dt, w.src)
        g.step(w.dt, w.src)
    g.check_device_error()
    torch.cuda.synchronize()
    n = o.npart
    ro, io = o.rdata()[:, :n], o.idata()[:, :n]
    rg, ig = g.rdata[:, :n].cpu().numpy(), g.idata[:, :n].cpu().numpy()
    oo, og = np.argsort(io[abi.PTAG], kind="stable"), np.argsort(ig[abi.PTAG], kind="stable")
    np.testing.assert_array_equal(io[abi.PGID][oo], ig[abi.PGID][og])
    v = [abi.IPVX, abi.IPVY, abi.IPVZ]
    assert np.abs(ro[v][:, oo] - rg[v][:, og]).max() <= 1e-11 * np.abs(ro[v]).max()
    a = mesh.ng
    uo, ug = o.u0(), g.u0.cpu().numpy()
    uo, ug = uo[:, 1:, a:-a, a:-a, a:-a], ug[:, 1:, a:-a, a:-a, a:-a]
    assert np.abs(uo - ug).max() <= 1e-11 * np.abs(uo).max()
    g.close()
