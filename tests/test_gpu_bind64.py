"""Binding particles in the plain FP64 form: graphs that the caller captured of a stage are replayed
after other binds, with eager stages between the replays.  The same stages on a context of its own
give the values: both sides compute in FP64 and differ in the order of their atomic additions, 1e-13
of the largest for the one or two cycles."""

import ctypes as C

import numpy as np
import pytest

from athenak_amd import abi, workloads

pytestmark = pytest.mark.gpu


class Particles:
    """A particle set of its own, bound in turn with others."""

    def __init__(self, w, n, seed, cap=None):
        import torch
        rng = np.random.default_rng(seed)
        self.n, self.cap = n, cap or n
        r = np.zeros((abi.DK_NRDATA, self.cap))
        iv = np.zeros((abi.DK_NIDATA, self.cap), dtype=np.int32)
        m = w.mesh
        nb = (m.nmbx1, m.nmbx2, m.nmbx3)
        x = rng.random((3, n))
        for d in range(3):
            r[2 * d, :n], r[2 * d + 1, :n] = x[d], 0.2 * rng.standard_normal(n)
        r[abi.IPTS, :n], r[abi.IPM, :n] = 0.1, 1.0 / n
        b = [(x[d] * nb[d]).astype(np.int32) for d in range(3)]
        iv[abi.PGID, :n] = b[0] + nb[0] * (b[1] + nb[1] * b[2])
        iv[abi.PTAG, :n] = np.arange(n)
        self.r0, self.i0 = torch.from_numpy(r).cuda(), torch.from_numpy(iv).cuda()
        self.r, self.i = self.r0.clone(), self.i0.clone()

    def reset(self):
        self.r.copy_(self.r0)
        self.i.copy_(self.i0)


def bind(g, p, n=None):
    from athenak_amd.lib import lib
    g._check(lib().dk_bind_particles(g.h, C.c_void_p(p.r.data_ptr()), C.c_void_p(p.i.data_ptr()),
                                     p.cap, p.n if n is None else n), "dk_bind_particles")


def context(w, u, **kw):
    import torch
    from athenak_amd.lib import DustContext
    g = DustContext(w.mesh, w.blocks, w.phys, 1, stream=torch.cuda.Stream(), **kw)
    g.u0.copy_(u)
    g.u1.copy_(u)
    torch.cuda.synchronize()
    return g


def workload(coupling=abi.DK_IMEX):
    import torch
    w = workloads.c1(n=16, nb=2, coupling=coupling,
                     solver=abi.DK_DC1 if coupling == abi.DK_IMEX else abi.DK_LOCAL)
    gen = torch.Generator(device="cuda").manual_seed(3)
    u = torch.randn((8, 4, 12, 12, 12), dtype=torch.float64, device="cuda", generator=gen) * 0.1
    u[:, 0] = 1.0
    return w, u


def eager(w, u, p):
    """The cycle on a context of its own: the particles and the gas after it."""
    import torch
    p.reset()
    torch.cuda.synchronize()
    g = context(w, u)
    bind(g, p)
    g.step(w.dt, w.src)
    torch.cuda.synchronize()
    out = p.r.clone(), p.i.clone(), g.u0.clone()
    g.close()
    return out


def agree(got, want):
    assert bool((got[1] == want[1]).all())
    for a, b in ((got[0], want[0]), (got[2], want[2])):
        assert float((a - b).abs().max()) <= 1e-13 * float(b.abs().max())


@pytest.mark.parametrize("coupling", [abi.DK_IMEX, abi.DK_PC2])
def test_a_callers_graph_is_replayed_after_other_binds(coupling):
    import torch
    w, u = workload(coupling)
    sets = [Particles(w, n, seed) for n, seed in ((3000, 1), (5000, 2), (20000, 3))]
    want = [eager(w, u, p) for p in sets]
    g = context(w, u)
    graphs = []
    for p in sets:                      # every bind needs more than the last one reserved
        p.reset()
        torch.cuda.synchronize()
        bind(g, p)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=g.stream, capture_error_mode="thread_local"):
            g.step(w.dt, w.src, check=False)
        graphs.append(graph)
    # (memory that a bind gave back would be taken by these and written by a replay)
    guard = [torch.full((1 << 16,), 7, dtype=torch.int32, device="cuda") for _ in range(64)]
    for k in (0, 2, 1, 0, 1, 2):
        p = sets[k]
        p.reset()
        g.u0.copy_(u)
        g.u1.copy_(u)
        torch.cuda.synchronize()
        with torch.cuda.stream(g.stream):
            graphs[k].replay()
        torch.cuda.synchronize()
        agree((p.r, p.i, g.u0), want[k])
        other = sets[(k + 1) % 3]       # an eager cycle of other particles between the replays
        other.reset()
        torch.cuda.synchronize()
        bind(g, other)
        g.step(w.dt, w.src)
        torch.cuda.synchronize()
    assert all(bool((x == 7).all()) for x in guard)
    g.check_device_error()
    g.close()


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def big(coupling=abi.DK_IMEX, back_reaction=1):
    w = workloads.c1(n=64, nb=2, coupling=coupling,
                     solver=abi.DK_DC1 if coupling == abi.DK_IMEX else abi.DK_LOCAL)
    w.phys.back_reaction = back_reaction
    return w


@pytest.mark.parametrize("n,back_reaction", [(1000, 1), (1 << 20, 0)])
def test_a_bind_takes_no_memory_for_passes_that_do_not_run(n, back_reaction):
    import torch
    w = big(back_reaction=back_reaction)
    p = Particles(w, n, 1)
    g = context(w, torch.zeros((8, 4, 36, 36, 36), dtype=torch.float64, device="cuda"))
    before = free_bytes()
    bind(g, p)                  # (with the tile passes: 23 MB for the mesh, 12 MB a million)
    assert free_bytes() == before
    g.close()


def test_a_count_that_grows_within_the_arrays_allocates_once():
    import torch
    w = big()
    cap = 3 << 20
    p = Particles(w, cap, 2)
    u = torch.zeros((8, 4, 36, 36, 36), dtype=torch.float64, device="cuda")
    u[:, 0] = 1.0
    g = context(w, u)
    before = free_bytes()
    bind(g, p, 1 << 18)
    after = free_bytes()
    assert before - after >= 12 * cap
    for n in (1 << 19, 1000, 1 << 20, cap):
        bind(g, p, n)
        assert free_bytes() == after
        d0 = g.diag()
        g.step(1e-4, None)
        d1 = g.diag()           # (every count exchanges momentum without loss)
        assert np.abs((d1[0:3] + d1[3:6]) - (d0[0:3] + d0[3:6])).max() < 1e-13 * d0[8]
    g.check_device_error()
    g.close()


def test_the_sort_takes_the_workspaces_where_memory_is_short():
    # 128^3 cells and a million particles: the workspaces take 200 MB, the sort 180 MB and more;
    # half of that is left over when it is called
    import torch
    w = workloads.c1(n=128, nb=2)
    n = 1 << 20
    p = Particles(w, n, 5)
    u = torch.zeros((8, 4, 68, 68, 68), dtype=torch.float64, device="cuda")
    u[:, 0] = 1.0
    want = eager(w, u, p)
    p.reset()
    torch.cuda.empty_cache()
    g = context(w, u)
    bind(g, p)
    g.prof(True)
    filler = []
    for _ in range(6):                  # (torch gives its cached blocks back when it runs short)
        room = free_bytes() - 90 * n
        if room > 1 << 20:
            filler.append(torch.empty(room, dtype=torch.uint8, device="cuda"))
    assert free_bytes() < 180 * n
    g.sort()
    g.step(w.dt, w.src)
    torch.cuda.synchronize()
    del filler
    torch.cuda.empty_cache()
    assert "bins" not in g.prof_read()
    # every particle as the tile passes advance it, in the order of the start's blocks and cells
    i0, r0 = p.i0.cpu().numpy(), p.r0.cpu().numpy()
    c = [(r0[2 * d] * 128).astype(np.int64) % 64 for d in range(3)]
    order = np.argsort((i0[abi.PGID] * 64 + c[2]) * 4096 + c[1] * 64 + c[0], kind="stable")
    np.testing.assert_array_equal(p.i[abi.PTAG].cpu().numpy(), order)
    o = torch.from_numpy(order).cuda()
    agree((p.r, p.i, g.u0), (want[0][:, o], want[1][:, o], want[2]))
    bind(g, p)                          # (the next bind reserves them again)
    g.prof_reset()
    g.step(w.dt, w.src)
    assert "bins" in g.prof_read()
    g.close()


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("own_stream", [True, False])
def test_a_bind_while_another_stream_is_captured(mode, own_stream):
    # a bind does no work of the captured program's: the capture goes on, and the bound particles
    # have their tile passes
    import torch
    from athenak_amd.lib import DustContext
    w, u = workload()
    small, p = Particles(w, 2000, 6), Particles(w, 6000, 7)
    want = eager(w, u, p)
    p.reset()
    g = context(w, u) if own_stream else DustContext(w.mesh, w.blocks, w.phys, 1)
    g.u0.copy_(u)
    g.u1.copy_(u)
    torch.cuda.synchronize()
    bind(g, small)
    x = torch.zeros(1000, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(), capture_error_mode=mode):
        x.add_(1.0)
        bind(g, p)                      # (larger than the first: it needs other workspaces)
        x.add_(1.0)
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert bool((x == 6.0).all())
    g.prof(True)
    g.step(w.dt, w.src)
    torch.cuda.synchronize()
    assert "bins" in g.prof_read()
    agree((p.r, p.i, g.u0), want)
    g.close()
