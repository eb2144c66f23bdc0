"""Nuclei stamped by a wave, a lane per point, where that can go wrong: cells
across the 64-column tile edge, several nuclei in one wave, cells of 27 and of
125 points (fewer and more than a wave), a last wave with idle lanes.  A mark
that is missing would leave a nucleus out of the next steps.  Bar: the events
and ids of the oracle, phi within 1e-5 of it (device and host expf), and both
buffers equal to those of a context that processes every plane."""
import numpy as np
import pytest

from cupf_amd import capi, cases
from tests.helpers import compare_states, gpu_context, oracle_sim
from tests.test_gpu_activity import _dense_context, _same_state
from tests.test_gpu_nucleation import PHI_TOL, _macro_T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,pts_cell", [((72, 12, 12), 5, 1), ((131, 11, 11), 8, 2), ((66, 6, 9), 8, 1)])
def test_nuclei_are_marked(n, K, pts_cell):
    c = cases.make_line_case("marks", n=n, grains=3, K=K, seed=57, z0_cells=-20)
    c.params.update(pts_cell=pts_cell, nuc_Nmax=np.float32(30.0), z0=np.float32(3.0))
    T3d = _macro_T(c, b=0.0)
    ctx, sim = gpu_context(c, T3d=T3d), oracle_sim(c, T3d=T3d)
    dense = _dense_context(c, T3d=T3d)
    for x in (ctx, dense, sim):
        x.nucl_reset(0)
    seed = int(c.params["seed"])
    for s in range(1, 25, 8):
        for x in (ctx, dense):
            x.step(8, s, capi.PF_STEP_NUCLEATE)
        sim.step(8, s, nucleate=True, seed=seed)
        assert ctx.nucl_events() == dense.nucl_events() == sim.nucl_events, f"events after step {s + 7}"
        _same_state(ctx, dense)
    print(f"[marks {n} K={K} p={pts_cell}] events {sim.nucl_events}", flush=True)
    bad, dphi = compare_states(ctx, sim)
    assert bad == 0 and dphi <= PHI_TOL
    for x in (ctx, dense):
        x.close()
