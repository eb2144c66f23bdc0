"""Performance cases of the APT phase-field step: what a user of cupf_amd runs.

Each case is one of a few kinds of program over the public API
(cupf_amd.capi, cupf_amd.cases, cupf_amd.ensemble):

run       a simulation from its initial fields: set them, step, take the
          result (the collected phi and grain ids, or the whole slot state)
nucleate  an all-liquid start: uniform cooling with nucleation, two steps per
          call, then growth under the melt-pool field, one step per call
window    the moving-domain loop of the phase_field command: single steps, the
          tip check, frame shifts and the tip scan every 20 steps, and a line
          QoI sample
ensemble  several simulations of uneven grids and thermal parameters stepped as
          one batch, from their initial fields to their collected fields
qoi       the quantities of interest of a developed state, computed on the device

Grids, grain densities and thermal parameters are those of the repository's
named workloads, tests and benchmark (cupf_amd/cases.py, cupf_amd/ensemble.py,
bench.py).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cupf_amd import capi, cases, ensemble

PHASE1 = capi.PF_STEP_INITIAL_UC | capi.PF_STEP_NUCLEATE


def listed():
    return [
        # the smallest simulation worth a call: latency of set-up, ten steps and the state's copy
        dict(name="run-16", kind="run", nx=16, ny=16, nz=16, K=8, grains=6, steps=10, out="slots"),
        # the reference's own slot count on the ensemble's smallest grid, two-angle orientations
        dict(name="run-32-k5", kind="run", nx=32, ny=32, nz=32, K=5, grains=25, steps=200, orient="angles",
             out="slots"),
        # the plain 64^3 simulation (100 grains) through start-up and steady growth
        dict(name="run-64", kind="run", nx=64, ny=64, nz=64, K=8, grains=100, steps=1000),
        # odd extents in every direction, no-flux walls, a cylindrical melt-pool field, and the
        # command's own loop of one step per call
        dict(name="run-ragged-cylinder", kind="run", nx=139, ny=74, nz=101, K=8, grains=250, steps=300, bc=0,
             thermal=2, per_call=1),
        # the 27-point id gather and line law of the one-GPU program, K of that program
        dict(name="run-gather27-k5", kind="run", nx=96, ny=96, nz=128, K=5, grains=225, steps=300, gather27=1,
             thermal=5),
        # nucleation from an all-liquid 256^3 cone melt pool
        dict(name="nucleate-256", kind="nucleate", nx=256, ny=256, nz=256, K=8, pre=80, steps=60),
        # the line configuration's start-up: a sharp substrate of ~5000 small grains whose
        # neighbourhoods overflow the slots
        dict(name="line-start", kind="run", nx=256, ny=256, nz=512, K=8, grains=5000, steps=100),
        # the same configuration on through competitive growth
        dict(name="line-run", kind="run", nx=256, ny=256, nz=512, K=8, grains=5000, steps=2000),
        # late in a line run: most of the window is solid, the grains have coarsened, the frame follows the front
        dict(name="window-late", kind="window", nx=256, ny=256, nz=256, K=8, grains=600, R=0.5, front=0.78,
             warm=240, steps=40),
        # a shallow window of the same kind with the reference's slot count
        dict(name="window-k5", kind="window", nx=160, ny=96, nz=80, K=5, grains=375, R=0.5, front=0.75, warm=300,
             steps=60),
        # a mixed ensemble (32^3 to 128x128x256) as one batch, replayed from a graph, tuned
        dict(name="ensemble-16", kind="ensemble", members=16, mix=0, K=8, steps=400),
        # QoIs of the 256x256x512 state during competitive growth
        dict(name="qoi-line", kind="qoi", nx=256, ny=256, nz=512, K=8, grains=5000, warm=300),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges (no larger than the largest listed one)."""
    kind = rng.choice(["run", "run", "run", "run", "nucleate", "window", "ensemble", "qoi"])
    K = rng.choice([5, 8, 8])
    if kind == "ensemble":
        return dict(kind="ensemble", members=rng.randint(3, 24), mix=rng.randint(0, 9999), K=K, steps=_log(rng, 100, 400))
    lo, hi = {"run": (14, 256), "nucleate": (40, 256), "window": (48, 224), "qoi": (64, 256)}[kind]
    size = _log(rng, lo, hi)

    def side(f0, f1):
        return max(12, min(512, int(round(size * math.exp(rng.uniform(math.log(f0), math.log(f1)))))))

    nx, ny, nz = size, side(0.6, 1.1), side(0.7, 1.9)
    grains = max(4, int(nx * ny / rng.uniform(13.0, 40.0)))
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, K=K)
    pts = nx * ny * nz
    if kind == "run":
        g27 = 1 if rng.random() < 0.2 else 0
        most = max(10, min(2000, int((1.0e10 if g27 else 2.5e10) / pts)))
        c.update(grains=grains, steps=_log(rng, 10, most), bc=rng.choice([110, 110, 0, 10, 111]), gather27=g27,
                 thermal=rng.choice([1, 1, 2, 5]), orient=rng.choice(["quat", "angles"]),
                 out="slots" if pts < 100000 else "fields")
        if rng.random() < 0.25 and c["steps"] <= 500:
            c["per_call"] = 1
    elif kind == "nucleate":
        c.update(nz=min(nz, 256), pre=_log(rng, 20, 100), steps=_log(rng, 10, 60))
    elif kind == "window":
        c.update(nz=min(nz, 256), grains=grains, R=rng.choice([0.1, 0.5]), front=round(rng.uniform(0.3, 0.79), 2),
                 warm=_log(rng, 100, 300), steps=20 * rng.randint(1, 4))
    else:
        c.update(grains=grains, warm=_log(rng, 50, 400))
    return c


# ------------------------------------------------------------------ inputs ---

def _case(c, seed):
    """The simulation's inputs (grid, parameters, substrate, orientations)."""
    n = (c["nx"], c["ny"], c["nz"])
    if c["kind"] == "nucleate":
        k = cases.make_cone_case("nucleate", n=n, K=c["K"], seed=seed % 100000)
        k.params.update(uc0=np.float32(8.0), nuc_Nmax0=np.float32(5.0))
        return k
    bc = c.get("bc", 110)
    thermal = c.get("thermal", 1)
    window = c["kind"] == "window"
    kw = dict(n=n, grains=c["grains"], K=c["K"], seed=seed % 100000, R=c.get("R", 0.1),
              bc=(bc // 100, bc // 10 % 10, bc % 10), gather27=c.get("gather27", 0), thermal_type=thermal,
              orient=c.get("orient", "quat"))
    if window:
        kw.update(z0_cells=c["front"] * c["nz"], line_config=True, nz_full=4 * c["nz"])
    elif c["nz"] < 64:
        kw.update(z0_cells=c["nz"] / 2)
    k = cases.make_line_case(c["kind"], **kw)
    if thermal == 2:  # a cylinder whose surface cuts the substrate
        k.params.update(r0=np.float32(0.6 * float(k.d["lyd"])))
    return k


def _context(k):
    ctx = capi.APTContext(k.params)
    ctx.set_coords(k.x, k.y, k.z)
    ctx.set_orientations(k.R9)
    return ctx


def prepare(case, seed):
    c = case
    if c["kind"] == "ensemble":
        # the mix of grids and thermal parameters is the case's, the substrates are the seed's
        specs = ensemble.ensemble_specs(c["members"], seed=c["mix"], nsteps=c["steps"])
        for q, s in enumerate(specs):
            s.seed = seed % 100000 + q
        ks = [ensemble.make_case(s, c["K"]) for s in specs]
        ctxs = [ensemble.new_context(k) for k in ks]
        return dict(c=c, ks=ks, ctxs=ctxs, batch=capi.Batch(ctxs))
    k = _case(c, seed)
    ctx = _context(k)
    st = dict(c=c, k=k, ctx=ctx)
    if c["kind"] in ("window", "qoi"):
        ctx.init_from_phi_alpha(k.phi0, k.alpha0)
        ctx.step(c["warm"], 1)
    if c["kind"] == "window":
        ctx.collect_on_device(0, capi.PF_COLLECT_CLEAR_ALPHA)
        ctx.md_enable(c["nz"] + 4000)  # the column's archive: room for every shift of a long run
        st.update(tip=0, moves=0, next=c["warm"] + 1)
    if c["kind"] == "qoi":
        st.update(max_id=int(k.params["num_theta"]), ids=np.zeros(c["grains"], np.int32),
                  counts=np.zeros(c["grains"], np.int32), rows=np.zeros((4 * c["nx"] * c["ny"], 8), np.int32))
        ctx.sync()
    if c["kind"] in ("window", "qoi"):  # a seed may leave a grain without a point: tables for all of them
        st.update(total=np.zeros(c["grains"], np.int32), extra=np.zeros(c["grains"], np.int32))
    return st


def _into(table, values):
    """`values` at the head of a table the caller keeps."""
    n = min(len(table), len(values))
    table[:n] = values[:n]
    return table


# ------------------------------------------------------------------- passes ---

def _run(st):
    c, k, ctx = st["c"], st["k"], st["ctx"]
    ctx.init_from_phi_alpha(k.phi0, k.alpha0)
    per = c.get("per_call", c["steps"])
    for s in range(1, c["steps"] + 1, per):
        ctx.step(min(per, c["steps"] + 1 - s), s)
    if c.get("out") == "slots":
        ctx.apply_bc(0)
        return list(ctx.download_state(0))
    return list(ctx.collect(0, capi.PF_COLLECT_CLEAR_ALPHA))


def _nucleate(st):
    c, k, ctx = st["c"], st["k"], st["ctx"]
    ctx.init_from_phi_alpha(k.phi0, k.alpha0)
    ctx.nucl_reset(0)
    for kt in range(c["pre"] // 2):
        ctx.step(2, 2 * kt + 1, PHASE1)
    for s in range(c["pre"] + 1, c["pre"] + c["steps"] + 1):
        ctx.step(1, s)
    return list(ctx.collect(0, capi.PF_COLLECT_CLEAR_ALPHA))


def _window(st):
    c, ctx = st["c"], st["ctx"]
    threshold = int(0.8 * ctx.fnz)
    low = 1
    for kt in range(c["steps"] // 2):
        s = st["next"]
        ctx.step(1, s)
        if (s + 1) % 20 == 0:
            st["tip"] = ctx.md_tip(st["tip"])
            while st["tip"] >= threshold:
                ctx.md_shift(st["moves"])
                st["moves"] += 1
                st["tip"] -= 1
            ctx.collect_on_device(0, 0)
            low = ctx.qoi_tip(1)
        ctx.step(1, s + 1)
        st["next"] = s + 2
    phi, alpha = ctx.collect(0, capi.PF_COLLECT_CLEAR_ALPHA)
    tip, total, extra = ctx.qoi_line(0)
    return [phi, alpha, st["tip"], st["moves"], low, tip, _into(st["total"], total), _into(st["extra"], extra)]


def _ensemble(st):
    c = st["c"]
    for k, ctx in zip(st["ks"], st["ctxs"]):
        ctx.init_from_phi_alpha(k.phi0, k.alpha0)
    b = st["batch"]
    b.next_step = [1] * len(st["ctxs"])
    b.step(c["steps"], capi.PF_BATCH_GRAPH | capi.PF_BATCH_AUTOTUNE)
    return [list(ctx.collect(0, capi.PF_COLLECT_CLEAR_ALPHA)) for ctx in st["ctxs"]]


def _qoi(st):
    ctx = st["ctx"]
    ctx.collect_on_device(0, capi.PF_COLLECT_CLEAR_ALPHA)
    ids, counts, above = ctx.qoi_volume(st["max_id"])
    rows = ctx.qoi_junction_rows()
    tip, total, extra = ctx.qoi_line(0)
    return [_into(st["ids"], ids), _into(st["counts"], counts), above, _into(st["rows"], rows), len(rows), tip,
            _into(st["total"], total), _into(st["extra"], extra)]


def run(state):
    kind = state["c"]["kind"]
    return {"run": _run, "nucleate": _nucleate, "window": _window, "ensemble": _ensemble, "qoi": _qoi}[kind](state)


# --------------------------------------------------------------------- work ---

def _solid_planes(c):
    """Planes that hold grains (the rest is liquid, whose slots are all empty and stay so)."""
    if c["kind"] == "window":
        return c["front"] * c["nz"] + 8
    if c["kind"] == "nucleate":
        return 0.05 * c["nz"]
    z0 = c["nz"] / 2 if c["nz"] < 64 else 25.0
    # a front that follows the isotherm at R, one plane in ~166 steps at 0.1 m/s
    return min(c["nz"], z0 + 8 + 0.5 * c.get("steps", 0) / 166.0)


def work(case):
    """Each step reads and writes the K (phi, id) slots of the points that hold or border a grain, and
    evaluates the right-hand side of about two filled slots of each; a call also reads its initial
    fields and writes its results once."""
    c = case
    if c["kind"] == "ensemble":
        cells = sum(n[0] * n[1] * n[2] for n in ensemble.GRIDS) / len(ensemble.GRIDS) * c["members"]
        act = sum(n[0] * n[1] * min(n[2], 35) for n in ensemble.GRIDS) / len(ensemble.GRIDS) * c["members"]
        steps = c["steps"]
    else:
        cells = c["nx"] * c["ny"] * c["nz"]
        act = c["nx"] * c["ny"] * _solid_planes(c)
        steps = c.get("steps", 0) + c.get("pre", 0)
    if c["kind"] == "qoi":
        return {"bytes": act * 8.0 * c["K"] + 8.0 * cells, "flops": 0}
    return {"bytes": steps * act * 16.0 * c["K"] + 16.0 * cells, "flops": steps * act * 160.0}


# ------------------------------------------------------------------ 64 bits ---

def _wrap(n, periodic):
    q = np.arange(n)
    q[0], q[-1] = (n - 2, 1) if periodic else (2, n - 3)
    return torch.from_numpy(q)


def _thermal(p, thermal, t, y, z):
    if thermal == 1:
        return p["G"] * (z - p["z0"]) - p["uc"] * 1e6 * t
    if thermal == 2:
        d = torch.sqrt((y - 0.5 * p["lyd"]) ** 2 + (z - p["z0"] - p["lzd"]) ** 2) - p["r0"]
        return -p["G"] * d - p["uc"] * 1e6 * t
    return p["G"] * (z - p["R"] * 1e6 * t - 2)


def exact(case, seed):
    """The run of a small case in float64: ids gathered in order of first appearance over the 7 points
    (down, back, left, centre, right, front, up), the K with the largest phi where there are more."""
    c = case
    cells = 0 if c["kind"] == "ensemble" else (c["nx"] + 1) * (c["ny"] + 1) * (c["nz"] + 1)
    if c["kind"] != "run" or c.get("gather27", 0) or cells * c["steps"] > 1.0e7:
        return None
    k = _case(c, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = {a: (float(b) if isinstance(b, (float, np.floating)) else b) for a, b in k.params.items()}
    K, nx, ny, nz = c["K"], p["fnx"], p["fny"], p["fnz"]
    f64 = dict(dtype=torch.float64, device=dev)
    x, y, z = (torch.from_numpy(v).to(**f64) for v in (k.x, k.y, k.z))
    R9 = torch.from_numpy(k.R9).to(**f64)
    unrotated = torch.eye(3, **f64).reshape(-1)
    phi0 = torch.from_numpy(k.phi0).to(**f64).reshape(nz, ny, nx)
    alpha0 = torch.from_numpy(k.alpha0).to(dev).reshape(nz, ny, nx).long()
    ph = torch.full((K, nz, ny, nx), -1.0, **f64)
    ar = torch.full((K, nz, ny, nx), -1, dtype=torch.int64, device=dev)
    on = phi0 > -0.995
    ph[0][on], ar[0][on] = phi0[on], alpha0[on]
    wx, wy, wz = (_wrap(n, b).to(dev) for n, b in ((nx, p["bcx"]), (ny, p["bcy"]), (nz, p["bcz"])))
    kk, jj, ii = torch.meshgrid(torch.arange(1, nz - 1, device=dev), torch.arange(1, ny - 1, device=dev),
                                torch.arange(1, nx - 1, device=dev), indexing="ij")
    kk, jj, ii = kk.reshape(-1), jj.reshape(-1), ii.reshape(-1)

    def at(dk, dj, di, k1, j1, i1):
        return (wz[k1 + dk] * ny + wy[j1 + dj]) * nx + wx[i1 + di]

    star = [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)]
    a_s = 1.0 + 3.0 * p["kin_delta"]
    epsv = -4.0 * p["kin_delta"] / a_s
    for s in range(1, c["steps"] + 1):
        fp, fa = ph.reshape(K, -1), ar.reshape(K, -1)
        nph, nar = torch.full_like(fp, -1.0), torch.full_like(fa, -1)
        seen = torch.zeros(kk.numel(), dtype=torch.bool, device=dev)
        for o in star:
            seen |= (fa[:, at(*o, kk, jj, ii)] != -1).any(0)
        k1, j1, i1 = kk[seen], jj[seen], ii[seen]
        b = [at(*o, k1, j1, i1) for o in star]
        ids = torch.cat([fa[:, q] for q in b])          # (7K, points), scan order
        val = torch.cat([fp[:, q] for q in b])
        E = 7 * K
        pos = torch.arange(E, device=dev)[:, None]
        rep = torch.zeros_like(ids, dtype=torch.bool)
        top = torch.full_like(val, -math.inf)
        topat = torch.zeros_like(ids)
        for e in range(E):
            m = ids == ids[e]
            rep[e] = (ids[e] != -1) & (torch.where(m, pos, E).amin(0) == e)
            v = torch.where(m, val, -math.inf)
            top[e] = v.amax(0)
            topat[e] = torch.where(v == top[e], pos, E).amin(0)
        keep = rep.clone()
        if int(rep.sum(0).max()) > K:
            for e in range(E):
                above = rep & ((top > top[e]) | ((top == top[e]) & (topat < topat[e])))
                keep[e] &= above.sum(0) < K
        slot = torch.where(keep, keep.cumsum(0) - 1, -1)
        n = keep.sum(0)
        la = torch.stack([torch.where(slot == q, ids, 0).sum(0) for q in range(K)])
        v = torch.full((7, K, k1.numel()), -1.0, **f64)
        for r in range(7):
            for u in range(K):
                m = (ids[r * K + u] == la) & (torch.arange(K, device=dev)[:, None] < n)
                v[r] = torch.where(m, val[r * K + u], v[r])
        pc = v[3]
        w = torch.where(torch.arange(K, device=dev)[:, None] < n, 0.25 * (pc + 1.0) ** 2, 0.0)
        t = s * p["dt"] * p["tau0"]
        Up = _thermal(p, p["thermal_type"], t, y[j1], z[k1]) / p["L_cp"]
        C = b[3]
        for q in range(K):
            g = la[q].clamp(min=0)
            g = torch.where(g <= p["num_theta"], g, g % p["num_theta"] + 1)
            m = torch.where((pc[q] > -0.995)[:, None], R9[g], unrotated).T
            gx, gy, gz = (v[4, q] - v[2, q]) * 0.5, (v[5, q] - v[1, q]) * 0.5, (v[6, q] - v[0, q]) * 0.5
            u2 = [(m[3 * h] * gx + m[3 * h + 1] * gy + m[3 * h + 2] * gz) ** 2 for h in range(3)]
            mag = u2[0] + u2[1] + u2[2]
            ani = a_s * (1.0 + epsv * (u2[0] ** 2 + u2[1] ** 2 + u2[2] ** 2) / torch.where(mag > p["eps"], mag ** 2, 1.0))
            ani = torch.where(mag > p["eps"], ani, 1.0)
            lap = v[4, q] + v[2, q] + v[5, q] + v[1, q] + v[6, q] + v[0, q] - 6.0 * pc[q]
            om = 1.0 - pc[q] ** 2
            rep_q = w.sum(0) - w[q]
            rhs = lap * p["hi"] ** 2 + om * pc[q] - p["lamd"] * Up * (om ** 2 - 6.0 * (pc[q] + 1.0) * rep_q)
            new = pc[q] + p["dt"] * rhs / ani
            live = n > q
            nph[q, C] = torch.where(live, new, -1.0)
            nar[q, C] = torch.where(live & (new >= -0.9999), la[q], -1)
        ph, ar = nph.reshape(K, nz, ny, nx), nar.reshape(K, nz, ny, nx)
    ph = ph[:, wz][:, :, wy][:, :, :, wx]
    if c.get("out") == "slots":
        return [ph.reshape(-1).cpu(), None]
    top = ph.amax(0)
    return [torch.where(top > -0.995, top, phi0).reshape(-1).cpu(), None]
