"""Particles that cross a shear-periodic x1 face and a periodic x3 (or x2) face in one stage, in both
directions, in both forms: block ids and velocities against the oracle.  (The FP32 form's key pass
once gave such a particle the wrong block; a particle outside its block gathers with weights far
beyond 1, so the velocities show it at once.)  Tolerances: the forms' own, 1e-11 and 1e-5 relative
to the largest velocity, as in test_gpu_parity.py and test_gpu_fp32.py."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from oracle.pyoracle import Oracle
from oracle.pyoracle import lib as olib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,vtol", [(abi.DK_FORM_FP64, 1e-11), (abi.DK_FORM_FP32, 1e-5)])
def test_particles_crossing_a_shear_face_and_another_face_in_one_stage(form, vtol):
    import torch
    from athenak_amd.lib import DustContext
    w = workloads.c2(n=16, nbx=2, ppc=1)
    dt = 1.0e-3
    rng = np.random.default_rng(7)
    n = 4096
    sign = rng.choice([-1.0, 1.0], size=(3, n))
    sign[1, ::2] = 0.0      # every second particle crosses x1 and x3 only
    depth = rng.uniform(0.0, 1.0, (3, n))
    x = np.where(sign != 0.0, sign * (0.1 - 1.0e-3 * depth) * (1.0 - 1e-12),
                 rng.uniform(-0.1, 0.1, (3, n)))
    v = sign * rng.uniform(0.2, 2.0, (3, n))
    r = np.zeros((abi.DK_NRDATA, n))
    iv = np.zeros((abi.DK_NIDATA, n), dtype=np.int32)
    for d in range(3):
        r[2 * d], r[2 * d + 1] = x[d], v[d]
    r[abi.IPTS], r[abi.IPM] = 0.1, 1.0e-9
    iv[abi.PTAG] = np.arange(n)
    iv[abi.PGID] = (x[0] >= 0) + 2 * (x[1] >= 0) + 4 * (x[2] >= 0)
    m = w.mesh
    u = np.zeros((m.nmb, 4, m.nx3 + 4, m.nx2 + 4, m.nx1 + 4))
    u[:, 0] = 1.0
    o = Oracle(w.mesh, w.blocks, w.phys, n)
    o.rdata()[:, :n], o.idata()[:, :n] = r, iv
    olib().or_set_npart(o.h, n)
    o.u0()[:], o.u1()[:] = u, u
    g = DustContext(w.mesh, w.blocks, w.phys, n, form=form)
    g.load(r, iv, u)
    o.time = g.time = 0.3     # (the faces are sheared against each other)
    crossed = 0
    for _ in range(3):
        before = o.idata()[abi.PGID, :n].copy()
        o.step(dt, w.src)
        g.step(dt, w.src)
        a = before ^ o.idata()[abi.PGID, :n]
        crossed += int(((a & 5) == 5).sum())
    assert crossed > 500
    g.export()
    torch.cuda.synchronize()
    ig, rg = g.idata[:, :n].cpu().numpy(), g.rdata[:, :n].cpu().numpy()
    ro, io = o.rdata()[:, :n], o.idata()[:, :n]
    og, oo = np.argsort(ig[abi.PTAG], kind="stable"), np.argsort(io[abi.PTAG], kind="stable")
    np.testing.assert_array_equal(io[abi.PGID][oo], ig[abi.PGID][og])
    vc = [abi.IPVX, abi.IPVY, abi.IPVZ]
    assert np.abs(ro[vc][:, oo] - rg[vc][:, og]).max() <= vtol * np.abs(ro[vc]).max()
    g.close()
