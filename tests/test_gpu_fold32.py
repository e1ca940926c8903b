"""The FP32 form's fused folds and its scans at the sizes where they can go wrong: tiles of one or
two cells along an axis (three tiles' regions on one cell, blocks that are their own neighbour),
sheared and walled faces, tiles of many parts, more than 1024 tiles, and more
cells than one workgroup of the key scan takes.  Against the oracle, with the form's own bar:
velocities and gas momenta within 1e-5 of the largest, block ids equal, positions within 1e-5 of
the distance travelled (as in test_gpu_fp32.py), and every export bit-identical when repeated."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def box(nx, nb, faces="periodic", **kw):
    shear = faces == "shear"
    x3 = {"outflow": abi.DK_X3_OUTFLOW, "reflect": abi.DK_X3_REFLECT}.get(
        faces, abi.DK_X3_PERIODIC)
    mesh, blocks = abi.uniform_mesh(nx, nb,
                                    ((-0.5, 0.5),) * 3, ng=2, bc_x3=x3,
                                    bc_x1=abi.DK_X1_SHEAR if shear else abi.DK_X1_PERIODIC)
    su = workloads._setup(seed=3, taus=(0.1,), eps=(0.5,), gas_noise=0.3, dust_noise=0.6, **kw)
    src = abi.dk_gas_src(shearing_box=1, stratified=0, omega0=1.0, qshear=1.5,
                         const_accel=0.1, const_accel_dir=1) if shear else None
    return workloads.Workload("box", mesh, blocks, workloads._phys(sbox=shear), su, src, 4e-3, 6)


CASES = {
    "one row tiles": lambda: box((8, 5, 4), (1, 3, 2), ppc=4),
    "one layer tiles": lambda: box((8, 4, 3), (1, 1, 1), ppc=4),
    "smallest tiles": lambda: box((12, 6, 10), (2, 1, 2), ppc=3),
    "two cell tiles": lambda: box((6, 4, 8), (2, 2, 1), ppc=3),
    "two row tiles, shear": lambda: box((8, 6, 4), (2, 3, 1), "shear", ppc=3),
    "one block, shear": lambda: box((8, 4, 6), (1, 1, 1), "shear", ppc=3),
    "whole tiles, shear": lambda: box((16, 8, 8), (1, 2, 2), "shear", ppc=3),
    "one row tiles, walls": lambda: box((8, 5, 4), (2, 2, 2), "reflect", ppc=3),
    "one layer tiles, walls": lambda: box((8, 4, 5), (1, 2, 1), "reflect", ppc=3),
    "whole tiles, walls": lambda: box((8, 8, 4), (2, 1, 1), "outflow", ppc=3),
    "many parts": lambda: box((8, 8, 8), (2, 2, 2), ppc=8, nclump=3, clump_frac=0.9,
                              clump_sigma=0.01),
    "many tiles": lambda: box((24, 18, 10), (3, 2, 3), ppc=1),
}


def exported(w, steps):
    import torch
    from athenak_amd.lib import DustContext
    g = DustContext(w.mesh, w.blocks, w.phys, w.npart + 16, form=abi.DK_FORM_FP32)
    g.setup(w.setup)
    for _ in range(steps):
        g.step(w.dt, w.src)
    g.check_device_error()
    g.export()
    torch.cuda.synchronize()
    n = g.npart
    r, i, u = g.rdata[:, :n].cpu().numpy(), g.idata[:, :n].cpu().numpy(), g.u0.cpu().numpy()
    g.close()
    order = np.argsort(i[abi.PTAG], kind="stable")
    return r[:, order], i[:, order], u


@pytest.mark.parametrize("name", sorted(CASES))
def test_folds_and_scans_against_the_oracle(name):
    w = CASES[name]()
    steps = 6
    o = Oracle(w.mesh, w.blocks, w.phys, w.npart + 16, threads=4)
    o.setup(w.setup)
    for _ in range(steps):
        o.step(w.dt, w.src)
    n = o.npart
    oo = np.argsort(o.idata()[abi.PTAG, :n], kind="stable")
    ro, io, uo = o.rdata()[:, :n][:, oo], o.idata()[:, :n][:, oo], o.u0()
    rg, ig, ug = exported(w, steps)
    np.testing.assert_array_equal(io[[abi.PTAG, abi.PGID]], ig[[abi.PTAG, abi.PGID]])
    v, x = [abi.IPVX, abi.IPVY, abi.IPVZ], [abi.IPX, abi.IPY, abi.IPZ]
    vmax = np.abs(ro[v]).max()
    a = w.mesh.ng
    ua, ub = uo[:, 1:, a:-a, a:-a, a:-a], ug[:, 1:, a:-a, a:-a, a:-a]
    errs = (np.abs(ro[v] - rg[v]).max() / vmax, np.abs(ua - ub).max() / np.abs(ua).max(),
            np.abs(ro[x] - rg[x]).max() / (vmax * w.dt * steps))
    print("[gpu-fold32] %s: velocity %.2e, gas %.2e, position %.2e" % ((name,) + errs), flush=True)
    assert max(errs) < 1e-5, errs
    again = exported(w, steps)
    for p, q in zip((rg, ig, ug), again):
        np.testing.assert_array_equal(p, q)
