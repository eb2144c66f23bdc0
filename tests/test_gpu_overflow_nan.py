"""The overflow ranking where entries are not ordinary numbers: NaN of both
signs, infinities and -0 among the entries of neighbourhoods over K ids.  A NaN
is never larger than another entry and nothing is larger than it, so it is
taken only where it is the first entry left; the keep test in the row and the
fix-up have to agree on that.  Bar: ids equal to the oracle's, phi bit-exact
(NaN where the oracle has one), equal overflow counts."""
import numpy as np
import pytest

from cupf_amd import cases
from tests.helpers import gpu_context, interior, oracle_sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g27", [0, 1])
@pytest.mark.parametrize("K", [5, 8])
@pytest.mark.parametrize("over", [2, 50])  # ids beyond K around every point, at most
def test_nan_entries_rank_as_in_the_oracle(over, K, g27):
    n = (71, 13, 11)  # a full row and a strip
    c = cases.make_line_case("nan", n=n, grains=60, K=K, seed=83, z0_cells=n[2] / 2, gather27=g27)
    p = c.params
    pool = min(K + over, int(p["num_theta"]))
    rng = np.random.default_rng(100 * K + 10 * g27 + over)
    shape = (K, p["fnz"], p["fny"], p["fnx"])
    # every point holds distinct ids; the larger half of a small pool has the smaller phi
    arg = 1 + np.argsort(rng.random((pool,) + shape[1:]), axis=0)[:K].astype(np.int32)
    arg[rng.random(shape) < 0.4] = -1
    ph = rng.uniform(-1.0, 1.0, size=shape).astype(np.float32)
    if over == 2:
        ph = np.where(arg > K, np.float32(-0.9) - np.float32(0.05) * (1 + ph), np.float32(0.5) + ph / 4).astype(np.float32)
    odd = rng.random(shape)
    for lo, hi, v in ((0.0, 0.08, np.nan), (0.08, 0.16, -np.nan), (0.16, 0.18, np.inf), (0.18, 0.2, -np.inf),
                      (0.2, 0.22, -0.0), (0.22, 0.24, 0.0)):
        ph[(odd >= lo) & (odd < hi)] = np.float32(v)
    ph[arg == -1] = -1.0
    assert (np.isnan(ph) & np.signbit(ph)).any() and (np.isnan(ph) & ~np.signbit(ph)).any()
    ctx, sim = gpu_context(c), oracle_sim(c)
    ctx.upload_state(ph.ravel(), arg.ravel(), 0)
    sim.set_state(ph, arg)
    for s in (1, 2):
        ctx.step(1, s)
        sim.step(1, s)
        print(f"[nan K={K} g27={g27} over={over}] step {s}: overflow {sim.overflow}", flush=True)
        assert ctx.overflow_count() == sim.overflow > 0
        (pg, ag), (po, ao) = ((interior(v, K, p["fnx"], p["fny"], p["fnz"]) for v in x)
                              for x in (ctx.download_state(0), sim.state(0)))
        wrong = (int((ag != ao).sum()), int(((pg != po) & ~(np.isnan(pg) & np.isnan(po))).sum()))
        assert wrong == (0, 0)
    ctx.close()
