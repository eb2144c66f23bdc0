"""The collected fields and the grain counts where their kernels can go wrong:
field sizes that are and are not a multiple of the four points a thread takes,
rows with every bound from none to K (collect reads a row's filled slots only),
a halo just filled and one left as it was, more ids in one workgroup's run of
points than its table holds, and ids above the largest counted.  Bar: equal to
the same on the downloaded state."""
import numpy as np
import pytest

from cupf_amd import capi, cases
from tests.helpers import gpu_context

pytestmark = pytest.mark.gpu


def _collected(ph, arg, K, L):
    ph, arg = ph.reshape(K, L), arg.reshape(K, L)
    am = ph.argmax(axis=0)  # the first of equals, as a strict > from slot 0
    mv, id_ = ph[am, np.arange(L)], arg[am, np.arange(L)]
    solid = mv.astype(np.float64) > -0.995
    return mv, id_, solid


@pytest.mark.parametrize("n,K,bc,ids", [
    ((11, 5, 7), 8, (0, 1, 0), 60),        # odd field size, one partial row
    ((130, 9, 20), 5, (1, 0, 1), 4000),    # two tiles and a strip, a table half full
    ((130, 100, 90), 5, (1, 0, 1), 4000),  # longer runs, more ids than a table holds
    ((62, 30, 14), 8, (1, 1, 0), 900),     # field size a multiple of four
])
def test_collect_and_counts(n, K, bc, ids):
    c = cases.make_line_case("collect", n=n, grains=8, K=K, seed=91, z0_cells=n[2] / 2, bc=bc)
    ctx = gpu_context(c)
    rng = np.random.default_rng(7)
    fnx, fny, fnz = ctx.fnx, ctx.fny, ctx.fnz
    L = fnx * fny * fnz
    # rows bounded by 0 .. K slots, each point filled up to its row's bound at most
    bound = rng.integers(0, K + 1, size=(fnz, fny, 1))
    bound[: fnz // 3] = 0
    fill = (np.arange(K)[:, None, None, None] < bound) & (rng.random((K, fnz, fny, fnx)) < 0.7)
    arg = np.where(fill, rng.integers(1, ids + 1, size=fill.shape), -1).astype(np.int32)
    ph = np.where(fill, rng.uniform(-1.0, 1.0, size=fill.shape), -1.0).astype(np.float32)
    for flags in (capi.PF_COLLECT_NO_BC | capi.PF_COLLECT_CLEAR_ALPHA, capi.PF_COLLECT_CLEAR_ALPHA):
        ctx.upload_state(ph.ravel(), arg.ravel(), 0)
        phi, alpha = ctx.collect(0, flags)
        mv, id_, solid = _collected(*ctx.download_state(0), K, L)
        assert np.array_equal(alpha, np.where(solid, id_, 0))
        assert np.array_equal(phi[solid], mv[solid])
    a = alpha.reshape(fnz, fny, fnx)[1:-1, 1:-1, 1:-1].ravel()
    for top in (ids, max(1, ids // 2)):
        got_ids, got_counts, above = ctx.qoi_volume(top)
        u, first, counts = np.unique(a, return_index=True, return_counts=True)
        keep = (u > 0) & (u <= top)
        order = np.argsort(first[keep])
        assert got_ids == u[keep][order].tolist() and got_counts == counts[keep][order].tolist()
        assert above == int((a > top).sum())
    ctx.close()
