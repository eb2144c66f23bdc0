"""The step's paths against each other on long runs that overflow: rows bounded
by their row words (narrow rows, classes of the general path, the keep test)
beside a context that takes every row through the general path with all K
slots (CUPF_NO_ACTIVITY=1), and a batch's graph and eager steps at two chunk
depths beside the members alone; a 65-point-wide grid has a full tile and a
one-column strip.  Bar: equal bits and overflow counts, through the start-up
(against the oracle too) and past it."""
import numpy as np
import pytest

from cupf_amd import capi, cases, ensemble
from tests.helpers import compare_states, first_mismatch, gpu_context, oracle_sim

pytestmark = pytest.mark.gpu


def _dense(name, n, seed, K):
    # grains ~3.6 cells wide: most points of the start-up overflow
    return cases.make_line_case(name, n=n, grains=int(round(n[0] * n[1] / 3.6 ** 2)), K=K, seed=seed)


@pytest.mark.parametrize("K", [5, 8])
def test_bounded_rows_and_the_general_path_end_with_the_same_bits(K, monkeypatch):
    c = _dense("paths", (64, 40, 24), 61, K)
    ctx, sim = gpu_context(c), oracle_sim(c)
    monkeypatch.setenv("CUPF_NO_ACTIVITY", "1")
    every = gpu_context(c)
    monkeypatch.delenv("CUPF_NO_ACTIVITY")
    p = c.params
    assert p["fnx"] - 2 == 65
    for s0, n in ((1, 150), (151, 250)):
        ctx.step(n, s0)
        every.step(n, s0)
        if s0 == 1:
            sim.step(n, s0)
            bad, dphi = compare_states(ctx, sim)
            assert bad == 0 and dphi == 0.0, first_mismatch(ctx, sim, K, p["fnx"], p["fny"], p["fnz"])
            assert ctx.overflow_count() == sim.overflow > 0
        print(f"[paths K={K}] step {s0 + n - 1}: overflow {ctx.overflow_count()}", flush=True)
        ctx.apply_bc(0)  # the states are compared whole, halo included
        every.apply_bc(0)
        assert ensemble.state_hash(every) == ensemble.state_hash(ctx)
        assert every.overflow_count() == ctx.overflow_count()
        (pa, aa), (pb, ab) = ctx.collect(0, capi.PF_COLLECT_CLEAR_ALPHA), every.collect(0, capi.PF_COLLECT_CLEAR_ALPHA)
        assert np.array_equal(pa.view(np.int32), pb.view(np.int32)) and np.array_equal(aa, ab)
    ctx.close()
    every.close()


@pytest.mark.parametrize("K", [5, 8])
def test_batch_graph_and_depths_end_with_the_bits_of_single_runs(K):
    members = [_dense("m0", (64, 40, 24), 67, K), _dense("m1", (40, 40, 20), 71, K)]
    alone = []
    for c in members:
        ctx = gpu_context(c)
        ctx.step(200, 1)
        assert ctx.overflow_count() > 0
        alone.append((ensemble.state_hash(ctx), ctx.overflow_count()))
        ctx.close()
    for flags, depth in ((capi.PF_BATCH_GRAPH, 2), (0, 8)):
        ctxs = [gpu_context(c) for c in members]
        b = capi.Batch(ctxs)
        b.kchunk = depth
        b.step(200, flags)
        print(f"[batch paths K={K}] flags {flags} depth {depth}", flush=True)
        b.close()
        for q, ctx in enumerate(ctxs):
            assert (ensemble.state_hash(ctx), ctx.overflow_count()) == alone[q], f"member {q}, depth {depth}"
            ctx.close()
