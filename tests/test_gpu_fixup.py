"""The fix-up's groups of lanes (8 per point for the 7-point gather, 16 for the
27-point) against the oracle: neighbourhoods over K ids on every wall and
corner of an odd grid, with lists that end inside a wave's last group and
lists of many waves per workgroup, for both slot counts and both gathers.
Bar: ids and phi bit-exact, equal overflow counts."""
import numpy as np
import pytest

from cupf_amd import capi, cases
from tests.helpers import compare_states, first_mismatch, gpu_context, oracle_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g27", [0, 1])
@pytest.mark.parametrize("K", [5, 8])
@pytest.mark.parametrize("n,bc,blocks", [
    ((5, 4, 6), (0, 0, 0), 0),       # a handful of points: one partly filled wave
    ((19, 13, 11), (0, 1, 0), 0),    # a wall next to every point's neighbourhood
    ((33, 21, 17), (1, 1, 1), 2),    # two workgroups take many points in turn
])
def test_fixup_groups_against_oracle(n, bc, blocks, K, g27, monkeypatch):
    if blocks:
        monkeypatch.setenv("CUPF_FIX_BLOCKS", str(blocks))
    grains = max(8, int(n[0] * n[1] / 3.0))
    c = cases.make_line_case("fixup", n=n, grains=grains, K=K, seed=61, z0_cells=n[2] / 2, bc=bc, gather27=g27)
    ctx = gpu_context(c)
    sim = oracle_sim(c)
    s = 1
    for stop in (1, 4, 12):
        ctx.step(stop - s + 1, s)
        sim.step(stop - s + 1, s)
        s = stop + 1
        print(f"[fixup {n} K={K} g27={g27}] step {stop}: overflow {sim.overflow}", flush=True)
        assert ctx.overflow_count() == sim.overflow
        bad, dphi = compare_states(ctx, sim)
        p = c.params
        assert bad == 0 and dphi == 0.0, first_mismatch(ctx, sim, K, p["fnx"], p["fny"], p["fnz"])
    assert sim.overflow > 0 or (K == 8 and n[0] < 10)
    ctx.close()
