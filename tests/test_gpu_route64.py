"""Which kernels the plain FP64 form's particle-mesh passes run on: tile by tile from one particle per
16 cells on, where that is at least 5 (imex) or 6 (pc2) a tile of 8 x 4 x 4 cells, whatever the
block's shape leaves of a tile.  The kernels' timers name them ("bins" belongs to the tile passes);
the results are the oracle's on either side of the line, compared as in test_gpu_tile64.py.  Without back-reaction nothing is deposited and the per-particle
kernels gather, whatever the count."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from tests.test_gpu_tile64 import UNIT, particles, run_pair

pytestmark = pytest.mark.gpu


def labels(mesh, blocks, phys, x, v, ts, mass, dt):
    """The kernels of one cycle."""
    from athenak_amd.lib import DustContext
    n = x.shape[1]
    r = np.zeros((abi.DK_NRDATA, n))
    iv = np.zeros((abi.DK_NIDATA, n), dtype=np.int32)
    for d in range(3):
        r[2 * d], r[2 * d + 1] = x[d], v[d]
    r[abi.IPTS], r[abi.IPM] = ts, mass
    for m in range(mesh.nmb):
        b = blocks[m]
        inside = np.ones(n, dtype=bool)
        for d, (lo, hi) in enumerate(((b.x1min, b.x1max), (b.x2min, b.x2max), (b.x3min, b.x3max))):
            inside &= (x[d] >= lo) & (x[d] < hi)
        iv[abi.PGID, inside] = m
    u = np.zeros((mesh.nmb, 4, mesh.nx3 + 4, mesh.nx2 + 4, mesh.nx1 + 4))
    u[:, 0] = 1.0
    g = DustContext(mesh, blocks, phys, n)
    g.load(r, iv, u)
    g.prof(True)
    g.step(dt)
    out = g.prof_read()
    g.close()
    return set(out)


# (blocks of whole tiles, where the line is 8 a tile; of a corner of one tile; of ragged tiles)
@pytest.mark.parametrize("nx,nb,imex,pc2", [((8, 4, 4), (1, 1, 1), 8, 8),
                                            ((8, 8, 8), (2, 1, 1), 64, 64),
                                            ((2, 2, 2), (2, 2, 2), 40, 48),
                                            ((5, 5, 5), (1, 2, 1), 40, 48),
                                            ((9, 4, 4), (1, 1, 3), 30, 36)])
@pytest.mark.parametrize("below", [1, 0])
@pytest.mark.parametrize("coupling", [abi.DK_IMEX, abi.DK_PC2])
def test_the_line_of_the_tile_passes(nx, nb, imex, pc2, below, coupling):
    mesh, blocks = abi.uniform_mesh(nx, nb, UNIT, ng=2)
    phys = workloads._phys(coupling=coupling,
                           solver=abi.DK_DC1 if coupling == abi.DK_IMEX else abi.DK_LOCAL)
    p = particles(mesh, (imex if coupling == abi.DK_IMEX else pc2) - below, 8, 0.2)
    assert ("bins" in labels(mesh, blocks, phys, *p, 1e-3)) == (not below)
    run_pair(mesh, blocks, phys, None, *p, 1e-3, 2)


@pytest.mark.parametrize("deposit", [abi.DK_CIC, abi.DK_TSC])
@pytest.mark.parametrize("what", ["imex", "pc2", "shear"])
@pytest.mark.parametrize("n,clump", [(100, 0), (6000, 3000)])
def test_without_back_reaction(what, n, clump, deposit):
    src = None
    if what == "shear":
        mesh, blocks = abi.uniform_mesh((6, 10, 5), (2, 2, 2), ((-0.1, 0.1),) * 3, ng=2,
                                        bc_x1=abi.DK_X1_SHEAR)
        phys = workloads._phys(sbox=True, deposit=deposit, back_reaction=0)
        src = abi.dk_gas_src(shearing_box=1, omega0=1.0, qshear=1.5, const_accel=0.1,
                             const_accel_dir=1)
    else:
        mesh, blocks = abi.uniform_mesh((8, 8, 6), (2, 1, 2), UNIT, ng=2)
        phys = workloads._phys(coupling=abi.DK_PC2 if what == "pc2" else abi.DK_IMEX,
                               solver=abi.DK_LOCAL if what == "pc2" else abi.DK_DC1,
                               deposit=deposit, back_reaction=0)
    p = particles(mesh, n, 9, 0.1, clump)
    if what != "shear":
        assert "bins" not in labels(mesh, blocks, phys, *p, 1e-3)
    run_pair(mesh, blocks, phys, src, *p, 2e-3, 3)
