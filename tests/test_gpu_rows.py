"""The step's rows against the oracle where they can go wrong: extents around
the 64-point row (a strip of 1 and 15 columns, the first partial tile, a grid
narrower than a strip), one wave's rows ending inside a tile, every slot bound
(grains from coarse, where rows hold one or two slots and take the narrow
path, to overflow), walls and wraps, both slot counts and gathers, and the
chunk depths that a mask's edge meets.  Bar: ids and phi bit-exact, equal
overflow counts, and both buffers equal to those of a context that processes
every plane with every slot."""
import numpy as np
import pytest

from cupf_amd import cases
from tests.helpers import compare_states, first_mismatch, gpu_context, oracle_sim
from tests.test_gpu_activity import _dense_context, _same_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,grains,K,bc,g27,depth", [
    ((64, 5, 12), 3, 8, (1, 1, 0), 0, 1),      # one column past a row, coarse
    ((78, 9, 10), 40, 8, (0, 0, 0), 0, 1),     # a strip of 15 columns, walls
    ((79, 6, 9), 12, 5, (1, 0, 1), 0, 3),      # the first partial tile, chunks of 3 planes
    ((12, 70, 9), 60, 8, (0, 1, 0), 0, 61),    # strip only, several waves of rows
    ((63, 3, 66), 5, 5, (0, 1, 1), 0, 61),     # full rows only, a chunk longer than the planes left
    ((66, 11, 8), 150, 8, (1, 1, 1), 1, 1),    # 27 points, two strip columns, overflow
    ((40, 7, 11), 4, 5, (0, 0, 0), 1, 2),      # 27 points, partial tile, coarse
])
def test_rows_against_oracle(n, grains, K, bc, g27, depth, monkeypatch):
    monkeypatch.setenv("CUPF_KCHUNK", str(depth))
    c = cases.make_line_case("rows", n=n, grains=grains, K=K, seed=71, z0_cells=n[2] / 2, bc=bc, gather27=g27)
    ctx, dense, sim = gpu_context(c), _dense_context(c), oracle_sim(c)
    s = 1
    for stop in (1, 2, 15):
        for x in (ctx, dense, sim):
            x.step(stop - s + 1, s)
        s = stop + 1
        _same_state(ctx, dense)
    print(f"[rows {n} K={K} g27={g27}] overflow {sim.overflow}", flush=True)
    assert ctx.overflow_count() == dense.overflow_count() == sim.overflow
    bad, dphi = compare_states(ctx, sim)
    p = c.params
    assert bad == 0 and dphi == 0.0, first_mismatch(ctx, sim, K, p["fnx"], p["fny"], p["fnz"])
    for x in (ctx, dense):
        x.close()


def test_row_bounds_follow_nucleation_upload_and_shift():
    """Rows whose bound changes other than by a step: balls nucleated into
    empty rows, a state uploaded with ids in its last slots only, and a frame
    shift, each followed by steps."""
    from cupf_amd import capi
    c = cases.make_line_case("bounds", n=(70, 46, 48), grains=40, K=8, seed=72, z0_cells=8, line_config=True,
                             nz_full=96)
    c.params.update(uc0=np.float32(8.0), nuc_Nmax0=np.float32(50.0))
    ctx, dense = gpu_context(c), _dense_context(c)
    for x in (ctx, dense):
        x.nucl_reset(0)
        x.step(6, 51, capi.PF_STEP_INITIAL_UC | capi.PF_STEP_NUCLEATE)  # undercooled by ~2 K, the mean
    assert ctx.nucl_events() == dense.nucl_events() and ctx.nucl_events() > 0
    _same_state(ctx, dense)
    ph, arg = ctx.download_state(0)
    ph, arg = ph.reshape(8, -1)[::-1].copy(), arg.reshape(8, -1)[::-1].copy()
    for x in (ctx, dense):
        x.upload_state(ph.ravel(), arg.ravel(), 0)
        x.step(5, 57)
        x.md_enable(100)
        x.md_shift(0)
        x.step(6, 62)
    _same_state(ctx, dense)
    for x in (ctx, dense):
        x.close()
