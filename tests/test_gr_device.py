"""GR effective monopole gravity on the device (gravity.c:142-375 with
GR_MONOPOLE) against the oracle's restatement, whose weak-field closed forms
test_gr_monopole.py pins: star columns (gamma law and table EOS, FP64 and
FP32-bulk, batched columns of several sizes) and 3D spherical stars on
uniform and dendritic grids.  The GR state the device keeps (TOV factor and
mass, lapses at the faces and zone centres, passes of the iteration) is
compared with the oracle's as well, and a guard checks that the GR field is
not the Newtonian one."""
import numpy as np
import pytest

from oracle import pyoracle as po
from medusa_amd import mds, problems
from parity_util import oracle_config

FP64_TOL = 1.0e-12
FP32_TOL = 1.0e-5


def _otab(T):
    t = T.t
    return po.eos_tab(dict(nr=t.nr, nt=t.nt, ny=t.ny, lr0=t.lr0, lr1=t.lr1, lt0=t.lt0, lt1=t.lt1, ye0=t.ye0,
                           ye1=t.ye1), T.data)


def _oracle(prob, T):
    kw = dict(nvars=6, monopole=2)
    if T is not None:
        kw["eos_tab"] = _otab(T)
    return po.Sim(oracle_config(prob, 0.5, **kw))


def _rel(a, b, w):
    return float(np.sum(np.abs(a - b) * w) / np.sum(np.abs(b) * w))


def _ctx(probs, precision, states, nsteps, graph=True):
    ctx = mds.Context(probs, precision=precision, rp=mds.run_params(cfl=0.5))
    for k, s in enumerate(states):
        ctx.upload(s, k)
    ctx.update_eos()
    ctx.run(nsteps, graph=graph)
    return ctx


def _v_over_cs_1d(dev, ref, g, cs):
    w = g.zone()[2:-2, mds.ZG_VOLUME]
    r = np.exp(g.moments(0)[1][2:-2] / g.moments(0)[2][2:-2])       # v_r = r v^x on a log-r column
    return float(np.sum(np.abs(dev[2].ravel() - ref[2].ravel()) * r * w) / np.sum(cs * w))


def _cs_1d(ref, T):
    if T is None:
        return np.sqrt(4.0 / 3.0 * (ref[1].ravel() / 3.0) / ref[0].ravel())
    ot = _otab(T)
    return np.array([po.eos_walk(ot, a, b, c)[0][1] for a, b, c in
                     zip(ref[0].ravel(), ref[1].ravel(), ref[5].ravel())])


def _gr_state_close(st, sim, tol):
    o = sim.gr_state()
    gtov, mr, lap, lape, it = o["gtov"], o["mr"], o["lapse"], o["lapse_edge"], o["iter"]
    for name, a, b in (("gtov", st["gtov"], gtov), ("mr", st["mr"][1:], mr[1:]),
                       ("lapse", st["lapse"], lap), ("lapse_edge", st["lapse_edge"], lape)):
        rel = float(np.max(np.abs(a - b) / np.abs(b)))
        print(f"[gr]   {name}: max rel {rel:.2e}", flush=True)
        assert rel <= tol, (name, rel)
    return it


@pytest.mark.gpu
@pytest.mark.parametrize("use_table", [False, True])
def test_gr_star_column_fp64_matches_oracle(use_table):
    T = mds.EosTable() if use_table else None
    g, prob, prims = problems.star1d(256, table=T, sigma=0.01)
    prob = dict(prob, monopole=mds.MONOPOLE_GR)
    print(f"[gr] FP64 GR star column n=256 table={use_table}, 60 steps", flush=True)
    ctx = _ctx([prob], mds.FP64, [prims], 60)
    sim = _oracle(prob, T)
    sim.set_prims(prims)
    sim.run(max_steps=60)
    dev, ref = ctx.download(), sim.get_prims()
    w = g.zone()[2:-2, mds.ZG_VOLUME]
    err = {"rho": _rel(dev[0].ravel(), ref[0].ravel(), w), "u": _rel(dev[1].ravel(), ref[1].ravel(), w),
           "v/cs": _v_over_cs_1d(dev, ref, g, _cs_1d(ref, T))}
    if use_table:
        err["ye"] = _rel(dev[5].ravel(), ref[5].ravel(), w)
    t, dt, ist = ctx.clock()
    print(f"[gr]   L1 {err}; t {t!r} vs {sim.t!r}", flush=True)
    assert ist == sim.istep and abs(t / sim.t - 1) < 1e-12
    for k, v in err.items():
        assert v <= FP64_TOL, (k, v)
    st = ctx.gr_state()
    it = _gr_state_close(st, sim, 1e-12)
    print(f"[gr]   passes {st['passes']} vs {it}; nonconverged {st['nonconverged']}", flush=True)
    assert st["passes"] == it and st["nonconverged"] == 0


@pytest.mark.gpu
def test_gr_field_differs_from_newtonian():
    g, prob, prims = problems.star1d(256, table=None, sigma=0.0)
    out = []
    for mono in (mds.MONOPOLE_NEWTON, mds.MONOPOLE_GR):
        ctx = _ctx([dict(prob, monopole=mono)], mds.FP64, [prims], 20)
        out.append(ctx.download())
    sim = _oracle(dict(prob, monopole=mds.MONOPOLE_GR), None)
    sim.set_prims(prims)
    ge_gr = sim.gr_edges()
    simn = po.Sim(oracle_config(prob, 0.5, nvars=6, monopole=True))
    simn.set_prims(prims)
    ge_n = simn.monopole_edges()
    corr = float(np.max(np.abs(ge_gr[1:] / ge_n[1:] - 1.0)))
    dv = float(np.max(np.abs(out[1][2] - out[0][2])))
    print(f"[gr] GR/Newtonian face gravity: max |ratio - 1| {corr:.3e}; device max |dv| {dv:.3e}", flush=True)
    assert corr > 1e-4 and dv > 0.0


@pytest.mark.gpu
def test_gr_star_column_fp32_within_tolerance():
    T = mds.EosTable()
    g, prob, prims = problems.star1d(256, table=T, sigma=0.01)
    prob = dict(prob, monopole=mds.MONOPOLE_GR)
    print("[gr] FP32-bulk GR star column n=256 table, 60 steps", flush=True)
    ctx = _ctx([prob], mds.FP32_BULK, [prims], 60)
    sim = _oracle(prob, T)
    sim.set_prims(prims)
    sim.run(max_steps=60)
    dev, ref = ctx.download(), sim.get_prims()
    w = g.zone()[2:-2, mds.ZG_VOLUME]
    err = {"rho": _rel(dev[0].ravel(), ref[0].ravel(), w), "u": _rel(dev[1].ravel(), ref[1].ravel(), w),
           "ye": _rel(dev[5].ravel(), ref[5].ravel(), w), "v/cs": _v_over_cs_1d(dev, ref, g, _cs_1d(ref, T))}
    print(f"[gr]   L1 {err}", flush=True)
    for k, v in err.items():
        assert v <= FP32_TOL, (k, v)
    _gr_state_close(ctx.gr_state(), sim, 1e-5)


@pytest.mark.gpu
def test_gr_batched_columns_fp64_match_oracle():
    """Columns of several sizes in one batch run to a common tmax (the median
    of their 20-step times), so some columns stop earlier than others and
    their field is no longer evaluated while the rest go on."""
    T = mds.EosTable()
    cols = [problems.star1d(n, table=T, sigma=0.01, seed=100 + n) for n in (128, 200, 333)]
    probs = [dict(c[1], monopole=mds.MONOPOLE_GR) for c in cols]
    ts = []
    for k, (g, prob, prims) in enumerate(cols):
        sim = _oracle(probs[k], T)
        sim.set_prims(prims)
        sim.run(max_steps=20)
        ts.append(sim.t)
    tmax = float(np.median(ts))
    print(f"[gr] 3 batched GR star columns FP64 to tmax={tmax:.4e}", flush=True)
    ctx = mds.Context(probs, precision=mds.FP64, rp=mds.run_params(cfl=0.5, tmax=tmax))
    for k, c in enumerate(cols):
        ctx.upload(c[2], k)
    ctx.update_eos()
    ctx.run_to(batch=8)
    for k, (g, prob, prims) in enumerate(cols):
        sim = _oracle(probs[k], T)
        sim.set_prims(prims)
        sim.run(tmax=tmax)
        dev, ref = ctx.download(k), sim.get_prims()
        t, dt, ist = ctx.clock(k)
        w = g.zone()[2:-2, mds.ZG_VOLUME]
        err = {"rho": _rel(dev[0].ravel(), ref[0].ravel(), w), "u": _rel(dev[1].ravel(), ref[1].ravel(), w),
               "ye": _rel(dev[5].ravel(), ref[5].ravel(), w)}
        print(f"[gr]   column {k} n={g.n[0]}: steps {ist} vs {sim.istep}, L1 {err}", flush=True)
        assert ist == sim.istep
        for kk, v in err.items():
            assert v <= FP64_TOL, (k, kk, v)
        _gr_state_close(ctx.gr_state(k), sim, 1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("dendritic,use_table,precision", [(False, False, 0), (True, True, 0), (True, True, 1)])
def test_gr_star3d_matches_oracle(dendritic, use_table, precision):
    from test_dendritic import star_sound_speed
    T = mds.EosTable() if use_table else None
    if dendritic:
        n = (32, 16, 32)
        g = problems.dend3d_grid(*n, dr0=2.0e6, rout=2.0e9)
        bc_lo = list(problems.SPH3D_BC_LO)
        bc_lo[0] = mds.BC_SPHERICAL_ORIGIN
        prob = dict(grid=g, bc_lo=bc_lo, bc_hi=list(problems.SPH3D_BC_HI), gam=4.0 / 3.0,
                    monopole=mds.MONOPOLE_GR, eos=T)
        prims = mds.init_polytrope(g, table=T, sigma=0.01) * g.valid_mask()[None]
        valid = g.valid_mask()
    else:
        n = (32, 8, 8)
        g, prob, prims = problems.star3d(*n, table=T, monopole=mds.MONOPOLE_GR)
        valid = np.ones(prims[0].shape, bool)
    nsteps = 10 if precision == 0 else 20
    print(f"[gr] 3D star {n} dendritic={dendritic} table={use_table} precision={precision}, {nsteps} steps",
          flush=True)
    ctx = _ctx([prob], precision, [prims], nsteps)
    sim = _oracle(prob, T)
    sim.set_prims(prims)
    sim.run(max_steps=nsteps)
    dev, ref = ctx.download(), sim.get_prims()
    w = np.broadcast_to(g.zone()[2:-2, 2:-2, mds.ZS_VOLUME][None], ref[0].shape) * valid
    err = {"rho": _rel(dev[0], ref[0], w), "u": _rel(dev[1], ref[1], w)}
    if use_table:
        err["ye"] = _rel(dev[5], ref[5], w)
    cs = star_sound_speed(ref, g, T, 4.0 / 3.0, valid)
    sc = g.zone()[2:-2, 2:-2, mds.ZS_SCALE0:mds.ZS_SCALE0 + 3]
    for d in range(3):
        err[f"v{d + 1}/cs"] = float(np.sum(np.abs(dev[2 + d] - ref[2 + d]) * sc[None, :, :, d] * w)
                                    / np.sum(cs * w))
    print(f"[gr]   L1 {err}", flush=True)
    tol = FP64_TOL if precision == 0 else FP32_TOL
    for k, v in err.items():
        assert v <= tol, (k, v)
    _gr_state_close(ctx.gr_state(), sim, 1e-12 if precision == 0 else 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("n, rho_c", [(12, 1.0e10), (256, 1.0e10), (257, 1.0e14), (1024, 1.0e14), (1025, 1.0e10)])
def test_gr_faces_at_the_edges_of_the_tiles_match_oracle(n, rho_c):
    """The face recurrence is solved a tile of 256 or 1024 faces at a time:
    columns of fewer faces than a tile, of exactly one and of one more, weak
    and (rho_c = 1e14, GM / R c^2 some 0.03) stronger fields.  The sums are
    trees of at most 1025 terms of one sign (errors below 20 eps) and the
    rounds stop within 2 eps, so five steps stay far within 1e-12."""
    g, prob, prims = problems.star1d(n, table=None, sigma=0.01, rho_c=rho_c)
    prob = dict(prob, monopole=mds.MONOPOLE_GR)
    print(f"[gr] GR star column n={n} rho_c={rho_c:g}, 5 steps", flush=True)
    ctx = _ctx([prob], mds.FP64, [prims], 5, graph=False)
    sim = _oracle(prob, None)
    sim.set_prims(prims)
    sim.run(max_steps=5)
    dev, ref = ctx.download(), sim.get_prims()
    w = g.zone()[2:-2, mds.ZG_VOLUME]
    assert _rel(dev[0].ravel(), ref[0].ravel(), w) <= FP64_TOL
    assert _rel(dev[1].ravel(), ref[1].ravel(), w) <= FP64_TOL
    assert ctx.gr_state()["passes"] == _gr_state_close(ctx.gr_state(), sim, 1e-12)
