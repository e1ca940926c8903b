"""The device error word: what a kernel has recorded stays until dk_error reads it, whatever calls
lie between.  A run that steps without a check and asks for its next time step (or for the stopping
times) sees a particle that a deposit left out, or a cell too full for the sort, at its next check;
an invalid stopping time is found also while the word holds an earlier error."""

import numpy as np
import pytest

from athenak_amd import abi, workloads
from tests.test_gpu_edges import base, pair
from tests.test_gpu_parity import make_pair

pytestmark = pytest.mark.gpu


def beyond_the_halo():
    """The FP64 form with a particle 2.5 cells beyond its block, recorded by the deposit."""
    w = workloads.c1(n=8, nb=2, ppc=1)
    _, g = make_pair(w)
    m = int(g.idata[abi.PGID, 5].item())
    g.rdata[abi.IPX, 5] = w.blocks[m].x1max + 2.5 / 8
    g.torch.cuda.synchronize()
    g.task("deposit_drag", abi.imex2p_stages(0.0, 1e-3)[0])
    return g, "halo"


def too_full_a_cell():
    """The FP32 form with more particles in one cell than its sort orders, recorded by the bind."""
    rng = np.random.default_rng(6)
    n = 17000
    xp = (np.array([3, 3, 3]) + rng.random((n, 3))) / 16.0
    _, g = pair(base(), xp, rng.normal(scale=0.1, size=(n, 3)), abi.DK_FORM_FP32,
                m=(1.0 / 16) ** 3 / n)
    return g, "fixed maximum"


@pytest.mark.parametrize("make", [beyond_the_halo, too_full_a_cell])
@pytest.mark.parametrize("call", ["new_time_step", "stopping_times"])
def test_a_recorded_error_outlives_the_reductions(make, call):
    from athenak_amd.lib import DustError
    g, match = make()
    for _ in range(2):
        if call == "new_time_step":
            assert g.new_time_step(0.5) > 0.0
        else:
            assert g.stopping_times() == (0.1 if g.form == abi.DK_FORM_FP64 else np.float32(0.1),) * 2
    with pytest.raises(DustError, match=match):
        g.check_device_error()
    g.check_device_error()   # cleared by the read
    g.close()


@pytest.mark.parametrize("ts", [0.0, -1.0, np.nan, np.inf])
@pytest.mark.parametrize("call", ["new_time_step", "stopping_times"])
def test_an_invalid_stopping_time_beside_an_earlier_error(call, ts):
    from athenak_amd.lib import DustError
    g, match = beyond_the_halo()
    g.rdata[abi.IPTS, 17] = ts
    g.torch.cuda.synchronize()
    with pytest.raises(DustError, match="stopping time"):
        getattr(g, call)(*((0.5,) if call == "new_time_step" else ()))
    with pytest.raises(DustError, match=match):
        g.check_device_error()
    g.close()
