"""The FP32 form's new time step over uneven stores: fewer particles than workgroups, blocks without
particles (the first, the last, several in a row), a fast particle in the last slot of a block, both
with and without a pending correction.  Against min dx/|v| of the exported particles in FP64; the
quotients are the same up to the rounding of the shear term and the cell size, 1e-12 relative."""

import numpy as np
import pytest

from athenak_amd import abi, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [0, 2])
@pytest.mark.parametrize("n,used", [(1, [5]), (7, [0, 7]), (1023, [2, 3]), (40000, [1, 4, 6]),
                                    (3 * 4096 + 5, list(range(8)))])
@pytest.mark.parametrize("shear", [False, True])
def test_new_time_step_over_uneven_blocks(n, used, steps, shear):
    import torch
    from athenak_amd.lib import DustContext
    w = workloads.c2(n=32, nbx=2, ppc=1) if shear else workloads.c1(n=32, nb=2)
    lo = np.array([w.mesh.x1min, w.mesh.x2min, w.mesh.x3min])
    size = np.array([w.mesh.x1max, w.mesh.x2max, w.mesh.x3max]) - lo
    rng = np.random.default_rng(n)
    b = np.sort(rng.choice(used, n))
    cell = size / 32
    off = np.stack([b & 1, (b >> 1) & 1, b >> 2]) * 0.5 * size[:, None]
    x = lo[:, None] + off + rng.uniform(0.1, 0.9, (3, n)) * 0.5 * size[:, None]
    r = np.zeros((abi.DK_NRDATA, n))
    iv = np.zeros((abi.DK_NIDATA, n), dtype=np.int32)
    dt = 1.0e-3
    v = rng.normal(0.0, 0.1, (3, n)) * cell[:, None] / dt
    v[:, -1] *= 3.0
    for d in range(3):
        r[2 * d], r[2 * d + 1] = x[d], v[d]
    r[abi.IPTS], r[abi.IPM] = 0.1, 1.0e-7
    iv[abi.PTAG], iv[abi.PGID] = np.arange(n), b
    u = np.zeros((8, 4, 20, 20, 20))
    u[:, 0] = 1.0
    g = DustContext(w.mesh, w.blocks, w.phys, n, form=abi.DK_FORM_FP32)
    g.load(r, iv, u)
    for _ in range(steps):
        g.step(dt, w.src)
    got = g.new_time_step(0.5)
    again = g.new_time_step(0.5)
    g.export()
    torch.cuda.synchronize()
    rg = g.rdata[:, :n].cpu().numpy()
    qo = w.phys.qshear * w.phys.omega0 if shear else 0.0
    vel = np.abs([rg[abi.IPVX], rg[abi.IPVY] - qo * rg[abi.IPX], rg[abi.IPVZ]])
    want = 0.5 * (cell[:, None] / np.maximum(vel, 1e-30)).min()
    if shear:     # (the frame limit of the FP32 form)
        xmax = max(abs(w.mesh.x1min), abs(w.mesh.x1max))
        want = min(want, 0.5 * cell[1] / (qo * 1.7071067811865475 * xmax) * (1.0 - 1e-9))
    assert again == got
    assert abs(got - want) <= 1e-12 * want, (got, want)
    g.close()
