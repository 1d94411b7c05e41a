"""Performance cases of the FIM dynamics library: forecasts, ocean intervals and
drop-in steps as a program that uses the library runs them.

A pass of a forecast case is the next stretch of a running forecast: some
device-resident steps, the conservation diagnostic (globsum), then the history
record copied into host arrays that the program keeps.  A forecast that has
reached its length begins again from its analysis (the seeded state), so the
synthetic atmosphere never leaves the range its time step is meant for.  A pass
of an ocean case is one transport interval of HYCOM's dynamics from the uploaded
ocean state.  The drop-in case is one dynamics step through the per-routine
entries on host arrays, as a Fortran model calls them.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from fimocn_subx_realtime_hera_apr2020_amd import fimhip, ocean, state as fimstate

NOISE, PERTURB, LOGNORMAL = fimhip.SYNTH_WIND_NOISE, fimhip.SYNTH_PERTURB, fimhip.SYNTH_LOGNORMAL
FORECAST_STEPS = 96               # length of a forecast before it begins again
CP, RD, P1000, QVMIN, GRAV = 1004.6855, 287.0586, 100000.0, 1.0e-10, 9.80665


def listed():
    return [
        # FP64, one member, the smallest grid in use (642 cells): launches and latency
        dict(name="fp64 G3 x 64", kind="fp64", level=3, nvl=64, ntra=4, steps=24),
        # FP64 on the accuracy grid
        dict(name="fp64 G5 x 64", kind="fp64", level=5, nvl=64, ntra=4, steps=24),
        # FP64 at the model's production resolution
        dict(name="fp64 G7 x 64", kind="fp64", level=7, nvl=64, ntra=4, steps=24),
        # the namelists' setting (mass_adv) with class-B tracers, a layer count that is not 64
        dict(name="fp64 G6 x 50 mass_adv class B", kind="fp64", level=6, nvl=50, ntra=5, steps=24, scheme=2, ntrb=3),
        # transport only, the time step of the reference's transport test
        dict(name="fp64 transport G5 x 64", kind="fp64", level=5, nvl=64, ntra=4, steps=10, mode=1),
        # an ensemble on the accuracy grid, mixed precision
        dict(name="ens 16 x G5 x 64", kind="ens", level=5, nvl=64, ntra=4, members=16, steps=24),
        # an ensemble at production resolution (the largest case)
        dict(name="ens 8 x G7 x 64", kind="ens", level=7, nvl=64, ntra=4, members=8, steps=12),
        # chemistry load: many log-normal tracers, transport only
        dict(name="ens transport G6 x 64 x 20 tr", kind="ens", level=6, nvl=64, ntra=20, members=1, steps=12, mode=1),
        # a small ragged ensemble with mass_adv and class-B tracers
        dict(name="ens 3 x G4 x 38 mass_adv class B", kind="ens", level=4, nvl=38, ntra=3, members=3, steps=24,
             scheme=2, ntrb=2),
        # a 30-step interval of HYCOM's dynamics
        dict(name="ocean G7 x 32", kind="ocean", level=7, kdm=32, numtr=1, steps=30),
        # more layers than half a wavefront, a small grid, the Janjic pressure force
        dict(name="ocean G4 x 48 janjic", kind="ocean", level=4, kdm=48, numtr=2, steps=10, janjic=True),
        # one step through the host-array drop-ins
        dict(name="drop-ins G5 x 64", kind="dropin", level=5, nvl=64, ntra=4),
    ]


def draw(rng):
    kind = rng.choice(["fp64", "fp64", "ens", "ens", "ens", "ocean"])
    if kind == "ocean":
        level = rng.choice([3, 4, 5, 6])
        return dict(kind=kind, level=level, kdm=rng.choice([32, 48, rng.randint(24, 64)]), numtr=rng.randint(0, 2),
                    steps=rng.choice([6, 10, 30]), janjic=rng.random() < 0.3)
    level = rng.choice([2, 3, 4, 5, 6])
    mode = 1 if rng.random() < 0.25 else 0
    c = dict(kind=kind, level=level, nvl=rng.choice([64, 64, rng.randint(30, 63)]), ntra=rng.randint(1, 8),
             steps=rng.choice([6, 12, 24]), mode=mode, scheme=rng.choice([1, 2]))
    if mode == 0 and rng.random() < 0.3:
        c["ntrb"] = rng.randint(1, 4)
    if kind == "ens":
        most = 96 // 4 ** max(0, level - 4)                # up to six G6 members
        c["members"] = max(1, round(math.exp(rng.uniform(0.0, math.log(most)))))
    return c


# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=8)
def _grid(level):
    return fimhip.icos_grid(level)


def _dt(case):
    """Two thirds of the reference's time step for the grid, at most 240 s; the
    transport test's 480 s (or the grid's own step) for transport alone."""
    own = 5760.0 / 2 ** (case["level"] - 1)
    return min(480.0, own) if case.get("mode") else min(240.0, own * 2.0 / 3.0)


def _host(shape):
    """A host array the program keeps, page-locked as one that talks to a GPU is."""
    return torch.zeros(shape, dtype=torch.float64, pin_memory=torch.cuda.is_available())


def _pd(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


def _ok(rc, what):
    if rc != 0:
        raise RuntimeError("%s: status %d" % (what, rc))


def _flags(case):
    return (NOISE | PERTURB) if case["kind"] == "ens" and not case.get("mode") else \
        (NOISE | LOGNORMAL) if case["ntra"] >= 8 else NOISE


def _fields(case):
    f = ["us", "vs", "dp", "pr", "tr"] if not case.get("mode") else ["dp", "pr", "ex", "tr", "trdp", "ws"]
    return f + (["trb"] if case.get("ntrb") else [])


def _trb(case, seed):
    """Class-B tracers of the forecast's start: smooth positive fields with noise."""
    g = _grid(case["level"])
    r = np.random.default_rng(seed + 77)
    base = 1.0 + 0.5 * np.sin(np.asarray(g.lat, np.float64))[None, :, None]
    return base * r.uniform(0.5, 1.5, (case["ntrb"], g.nip, case["nvl"]))


def _prepare_forecast(case, seed):
    g = _grid(case["level"])
    th, ds = fimstate.vertical_tables(case["nvl"])
    a = (g, case["nvl"], case["ntra"], _dt(case), th, ds)
    if case["kind"] == "ens":
        m = fimhip.Ensemble(a[0], case["members"], *a[1:])
    else:
        m = fimhip.Model(*a)
    s = dict(case=case, seed=int(seed), m=m, its=FORECAST_STEPS)
    if case.get("scheme", 1) != 1:
        m.set_flux_scheme(case["scheme"])
    if case.get("ntrb"):
        m.set_class_b(case["ntrb"], 6)
        s["trb"] = _trb(case, seed)
    s["out"] = {n: _host(m.shape(n)) for n in _fields(case)}
    _start_forecast(s)
    return s


def _start_forecast(s):
    """The forecast's analysis into the instance: the seeded state, then the start-up."""
    case, m = s["case"], s["m"]
    if case["kind"] == "ens":
        for i in range(case["members"]):
            m.synth(i, seed=s["seed"], flags=_flags(case))
            if case.get("ntrb"):
                m.load_class_b(i, s["trb"])
    else:
        m.synth(seed=s["seed"], member=0, flags=_flags(case))
        if case.get("ntrb"):
            m.upload("trb", s["trb"])
    m.init_state(not case.get("mode"))
    s["its"] = 0


def _run_forecast(s):
    case, m = s["case"], s["m"]
    if s["its"] + case["steps"] > FORECAST_STEPS:
        _start_forecast(s)
    mode = case.get("mode", 0)
    if case["kind"] == "ens":
        m.step(case["steps"], mode)
    else:
        for i in range(case["steps"]):
            m.step(s["its"] + i + 1, mode)
    s["its"] += case["steps"]
    sums = m.globsum()
    # the history record, the first member's for an ensemble
    for n, t in s["out"].items():
        if case["kind"] == "ens":
            _ok(m.lib.fimhip_ens_download(m.h, 0, fimhip.FIELD_ID[n], _pd(t)), "download " + n)
        else:
            _ok(m.lib.fimhip_download(m.h, fimhip.FIELD_ID[n], _pd(t)), "download " + n)
    out = dict(s["out"])
    out["mass"], out["totals"] = sums[0], sums[1]
    return out


# ---------------------------------------------------------------------------
OCN_STATE = ["dp", "pres", "uclin", "vclin", "temp", "saln", "dens"]


def _prepare_ocean(case, seed):
    g = _grid(case["level"])
    c = ocean.hycom_ocean_case(g, kdm=case["kdm"], seed=int(seed) % 100000 + 1, numtr=max(1, case["numtr"]))
    o = fimhip.Ocean(g, case["kdm"], c["wet"], c["dtleap"])
    o.set_momtum(c["batrop"], c["veldff"], c["smagcf"])
    o.set_transport(case["numtr"], c["temdff"])
    o.set_hybgen(c["targt"], c["salmin"], c["dpmin"], c["latij"])
    if case.get("janjic"):
        o.set_janjic(True)
    for n in fimhip.OCN_MOMTUM_FIELDS + ["cumuflx", "dpinit"]:
        o.upload(n, c[n])
    names = OCN_STATE + (["passv"] if case["numtr"] else [])
    init = {n: _host(c[n].shape) for n in names if n != "passv"}
    if case["numtr"]:
        init["passv"] = _host((case["numtr"],) + c["temp"].shape)
    for n, t in init.items():
        t.numpy()[...] = c[n][:case["numtr"]] if n == "passv" else c[n]
    return dict(case=case, o=o, init=init, out={n: _host(t.shape) for n, t in init.items()})


def _run_ocean(s):
    case, o = s["case"], s["o"]
    for n, t in s["init"].items():                       # the ocean state the interval starts from
        _ok(o.lib.fimhip_ocn_upload(o.h, fimhip.OCN_FIELDS.index(n), _pd(t)), "upload " + n)
    o.mass = (0.0, 0.0, 0.0)
    o.step_transp0(1)
    leapn = 2
    for st in range(1, case["steps"] + 1):               # hycom_run's order
        leapm = 1 + st % 2
        leapn = 3 - leapm
        o.step_edgvar(leapm, leapn)
        o.step(st, leapm, leapn)
        o.step_momtum(leapm, leapn)
        if st % 2 == 0:
            o.step_transp1()
    o.step_transp2(leapn)
    o.step_hybgn1(leapn)
    o.step_transp0(leapn)
    for n, t in s["out"].items():
        _ok(o.lib.fimhip_ocn_download(o.h, fimhip.OCN_FIELDS.index(n), _pd(t)), "download " + n)
    out = dict(s["out"])
    out["mass"] = np.array(o.mass)
    return out


# ---------------------------------------------------------------------------
def _prepare_dropin(case, seed):
    g = _grid(case["level"])
    nip, nvl, ntra = g.nip, case["nvl"], case["ntra"]
    th, ds = fimstate.vertical_tables(nvl)
    inst = fimhip.Instance(g, nvl, ntra, _dt(case), th, ds)
    st = fimhip.synth_state(g.lat, g.lon, nvl, ntra, seed=int(seed), flags=NOISE)
    c, l, e = (nip, nvl), (nip, nvl + 1), (nip, 6, nvl)
    a = {n: st[n] for n in ("us", "vs", "dp", "pr", "ex", "ph", "tr")}
    for n, sh in dict(mp=c, trdp=(ntra,) + c, ws=c, relvor=c, sdot=l, psrf=(nip,), ptdcy=(2, nip), u_tdcy=(3,) + c,
                      v_tdcy=(3,) + c, dp_tdcy=(3,) + c, dpl_tdcy=(3,) + c, trc_tdcy=(ntra, 3) + c,
                      trl_tdcy=(ntra, 3) + c, massfx=(3,) + e, u_edg=e, v_edg=e, dp_edg=e, lp_edg=e, geop_edg=e,
                      mont_edg=e, uvsq_edg=e, trc_edg=(ntra,) + e).items():
        a[n] = np.zeros(sh)
    inst.hystat(0, a["ph"], a["ex"], a["mp"], a["dp"], a["tr"], a["trdp"], a["psrf"], a["ptdcy"])
    keep = {n: v.copy() for n, v in a.items() if n in ("us", "vs", "dp", "pr", "ex", "ph", "mp", "tr", "trdp", "psrf")}
    return dict(case=case, inst=inst, a=a, start=keep, targt=th)


def _run_dropin(s):
    inst, a = s["inst"], s["a"]
    for n, v in s["start"].items():                      # the model's arrays at the start of the step
        a[n][...] = v
    inst.nf, inst.of, inst.vof = 0, 2, 1
    inst.abstart(1)
    edge = [a[n] for n in ("us", "vs", "dp", "pr", "ex", "ph", "mp", "tr", "u_edg", "v_edg", "dp_edg", "lp_edg",
                           "geop_edg", "mont_edg", "uvsq_edg", "trc_edg")]
    inst.edgvar1(1, *edge)
    inst.edgvar3(1, *edge)
    inst.cnuity(1, *[a[n] for n in ("us", "vs", "u_edg", "v_edg", "dp_edg", "lp_edg", "dp", "pr", "ex", "dp_tdcy",
                                    "dpl_tdcy", "massfx", "ws")])
    inst.trcadv(1, *[a[n] for n in ("trc_edg", "tr", "trdp", "trc_tdcy", "trl_tdcy", "massfx", "dp")])
    inst.momtum(1, *[a[n] for n in ("us", "vs", "ex", "relvor", "u_edg", "v_edg", "trc_edg", "geop_edg", "mont_edg",
                                    "uvsq_edg", "u_tdcy", "v_tdcy", "dp")])
    inst.hybgen(1, s["targt"], *[a[n] for n in ("us", "vs", "tr", "sdot", "ex", "dp", "pr")])
    inst.hystat(1, *[a[n] for n in ("ph", "ex", "mp", "dp", "tr", "trdp", "psrf", "ptdcy")])
    return {n: a[n] for n in ("us", "vs", "dp", "pr", "ex", "ph", "mp", "tr", "trdp", "ws", "relvor", "psrf",
                              "u_edg", "v_edg", "dp_edg", "lp_edg", "mont_edg", "uvsq_edg", "trc_edg")}


# ---------------------------------------------------------------------------
def prepare(case, seed):
    return {"ocean": _prepare_ocean, "dropin": _prepare_dropin}.get(case["kind"], _prepare_forecast)(case, seed)


def run(state):
    return {"ocean": _run_ocean, "dropin": _run_dropin}.get(state["case"]["kind"], _run_forecast)(state)


def work(case):
    """Bytes: the state a step (or interval) reads and writes once (the values a
    cell-level keeps between steps), and the record copied out.  Flops: the
    arithmetic of the stencils, roughly."""
    g = 10 * 4 ** case["level"] + 2
    if case["kind"] == "ocean":
        # 8 edge arrays and the thickness, pressure and velocities per step; the tracers per interval; 70 % ocean
        cl = g * case["kdm"]
        return dict(bytes=cl * (case["steps"] * 0.7 * 432.0 + 880.0 + 16.0 * (11 + case["numtr"])),
                    flops=cl * case["steps"] * 0.7 * 1500.0)
    cl, t = g * case["nvl"], case["ntra"]
    if case["kind"] == "dropin":
        # every array of the routines' argument lists that is intent(in) up, and that is written down
        return dict(bytes=8.0 * cl * (2 * (9 + 3 * t) + 2 * 6 * (6 + t) + 6 * 2), flops=cl * 3000.0)
    size = 4 if case["kind"] == "ens" else 8
    values = (10 if case.get("mode") else 18) + 8 * t
    out = 8.0 * cl * (4 + (2 * t if case.get("mode") else t) + case.get("ntrb", 0))
    moved = size * values + (76 if size == 4 and not case.get("mode") else 0)   # the FP64 fields of the mixed form
    n = case.get("members", 1)
    return dict(bytes=cl * case["steps"] * n * float(moved) + out, flops=cl * case["steps"] * n * (400.0 + 350.0 * t))


def tolerance(case):
    # the FP64 forms give the same bits whatever the launch: every sum has the reference's order
    if case["kind"] != "ens":
        return "exact"
    # FP32 winds and tracers: a change of rounding in one stage grows through the
    # steps that follow.  Measured against the FP64 form on the same state after one
    # and two passes (about four times the largest is stated): whole steps 1.8e-4
    # (thickness) and 2.3e-2 at one value, transport 4.9e-5 and 2.9e-3 (omega).
    return {"rel": 2e-4, "max": 1.2e-2} if case.get("mode") else {"rel": 7e-4, "max": 0.1}


# ---------------------------------------------------------------------------
def exact(case, seed):
    """Transport alone (abstart, edgvar1's winds, edgvar3, cnuity or mass_adv's
    FCT form, trcadv), in 64 bits from the same seeded state; the whole step ends
    in hybgen's column algorithm, which has no short form."""
    if case["kind"] not in ("fp64", "ens") or not case.get("mode") or case.get("scheme", 1) != 1:
        return None
    g = _grid(case["level"])
    if g.nip * case["nvl"] * case["ntra"] * case["steps"] > 8e8:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    members = case.get("members", 1)
    mass, totals, first = [], [], None
    for mem in range(members):
        st = fimhip.synth_state(g.lat, g.lon, case["nvl"], case["ntra"], seed=int(seed), member=mem,
                                flags=_flags(case))
        r = _transport(g, {n: torch.from_numpy(v).to(dev) for n, v in st.items()}, _dt(case), case["steps"])
        area = torch.from_numpy(np.asarray(g.area, np.float64)).to(dev)[:, None]
        mass.append(float((area * r["dp"]).sum()) / GRAV)
        totals.append([float((area * r["dp"] * t).sum()) for t in r["tr"]])
        first = first or {n: v.cpu().numpy() for n, v in r.items()}
    first["mass"] = np.array(mass) if case["kind"] == "ens" else mass[0]
    first["totals"] = np.array(totals) if case["kind"] == "ens" else np.array(totals[0])
    return first


def _transport(g, st, dt, steps):
    dev = st["dp"].device
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float64)).to(dev)   # noqa: E731
    nip, nvl = st["dp"].shape
    npx = torch.from_numpy(np.asarray(g.nprox, np.int64)).to(dev)
    slot = torch.arange(6, device=dev)[None, :].expand(nip, 6)
    live = slot < npx[:, None]
    at = torch.minimum(slot, npx[:, None] - 1)            # a pentagon's sixth slot is its fifth
    prox = torch.gather(torch.from_numpy(np.asarray(g.prox, np.int64)).to(dev) - 1, 1, at)
    proxs = torch.gather(torch.from_numpy(np.asarray(g.proxs, np.int64)).to(dev) - 1, 1, at)
    prev = torch.gather(prox, 1, (at - 1) % npx[:, None])
    nxt = torch.gather(prox, 1, (at + 1) % npx[:, None])
    L = live[:, :, None].double()
    cs, sn = f(g.cs)[:, :, :, None], f(g.sn)[:, :, :, None]
    svc, sve = f(g.sidevec_c)[:, :, :, None], f(g.sidevec_e)[:, :, :, None]
    hf = f(g.hfcoef) * live[:, :, None] * live[:, None, :]
    area = f(g.area)[:, None]
    ra = 1.0 / area
    pos, neg = (lambda x: x.clamp(min=0.0)), (lambda x: x.clamp(max=0.0))
    us, vs, dp, pr, ex = (st[n].clone() for n in ("us", "vs", "dp", "pr", "ex"))
    tr = st["tr"].clone()
    for t in (1, 2):
        if t < tr.shape[0]:
            tr[t] = tr[t].clamp(min=QVMIN)
    trdp = tr * dp
    ws = torch.zeros_like(dp)
    zero = torch.zeros_like(dp)
    h = dict(dl=[zero, zero], dd=[zero, zero], tl=[[zero, zero] for _ in tr], tt=[[zero, zero] for _ in tr])

    def own(x):                                           # least-squares edge values of a cell
        d = x[prox] - x[:, None, :]
        return x[:, None, :] + torch.einsum("nij,njk->nik", hf, d)

    def across(e):                                        # the edge's value in the cell on its other side
        return e[prox, proxs]

    def eq(x):
        return (2.0 * (x[:, None, :] + x[prox]) + x[prev] + x[nxt]) / 6.0

    for its in range(1, steps + 1):
        a1, a2, a3 = [(dt, 0.0, 0.0), (1.5 * dt, -0.5 * dt, 0.0), (dt * 23 / 12, -dt * 16 / 12, dt * 5 / 12)][min(its, 3) - 1]
        w = []
        for j, (u, v) in enumerate(((us[:, None, :], vs[:, None, :]), (us[prox], vs[prox]), (us[prev], vs[prev]),
                                    (us[nxt], vs[nxt]))):
            w.append((cs[:, :, j] * u + sn[:, :, j] * v, cs[:, :, j] * v - sn[:, :, j] * u))
        ue = (2 * (w[0][0] + w[1][0]) + w[2][0] + w[3][0]) / 6
        ve = (2 * (w[0][1] + w[1][1]) + w[2][1] + w[3][1]) / 6
        mg = [torch.sqrt(a * a + b * b) for a, b in w]
        sc = (2 * (mg[0] + mg[1]) + mg[2] + mg[3]) / 6 / torch.sqrt(ue * ue + ve * ve).clamp(min=0.001)
        vn = (sve[:, :, 1] * ue - sve[:, :, 0] * ve) * sc
        vx = across(vn)
        pm = pr[:, :-1] + pr[:, 1:]
        lp = (pm[:, None, :] + pm[prox] + 0.5 * (pm[prev] + pm[nxt])) / 6
        px, py = (lp * svc[:, :, 1] * L).sum(1), -(lp * svc[:, :, 0] * L).sum(1)
        del w, mg, sc, lp
        o = own(dp)
        m = 0.5 * ((vn + vn.abs()) * dp[:, None, :] - (vx + vx.abs()) * dp[prox]) * L
        a = (vn * 0.5 * (o + across(o)) - m) * L
        dplo = -m.sum(1) * ra
        lo = dp + a1 * dplo + a2 * h["dl"][0] + a3 * h["dl"][1]
        mx = pos(torch.maximum(torch.maximum(lo, dp), torch.maximum(lo[prox], dp[prox]).amax(1)))
        mn = pos(torch.minimum(torch.minimum(lo, dp), torch.minimum(lo[prox], dp[prox]).amin(1)))
        to, tv = h["dd"]
        rp = ((mx - lo - (a2 * neg(to) + a3 * pos(tv))) / a1 * area / (-neg(a)).sum(1).clamp(min=1e-11)).clamp(0, 1)
        rm = ((lo - mn + (a2 * pos(to) + a3 * neg(tv))) / a1 * area / pos(a).sum(1).clamp(min=1e-11)).clamp(0, 1)
        a = a * torch.where(a >= 0, torch.minimum(rm[:, None, :], rp[prox]), torch.minimum(rp[:, None, :], rm[prox]))
        m = m + a
        dtn = dplo - a.sum(1) * ra
        inc = a1 * dtn + a2 * to + a3 * tv
        h["dl"], h["dd"] = [dplo, h["dl"][0]], [dtn, to]
        dp = dp + inc
        lt = inc / dt
        below = lambda x: torch.flip(torch.cumsum(torch.flip(x, (1,)), 1), (1,))   # noqa: E731
        pr = torch.cat([pr[:, -1:] + below(dp), pr[:, -1:]], 1)
        ex = torch.cat([CP * (pr[:, :-1] / P1000) ** (RD / CP), ex[:, -1:]], 1)
        ws = below(lt) - 0.5 * lt + (us * px + vs * py) * ra
        mxs = across(m)
        new = []
        for t in range(tr.shape[0]):
            q = tr[t]
            if t == 0:
                te = eq(q)
            else:
                te = own(q)
                te = 0.5 * (te + across(te))
            fl = 0.5 * ((m + m.abs()) * q[:, None, :] - (mxs + mxs.abs()) * q[prox]) * L
            a = (m * te - fl) * L
            tlo = -fl.sum(1) * ra
            mx = pos(torch.maximum(q, q[prox].amax(1)))
            mn = pos(torch.minimum(q, q[prox].amin(1)))
            lo = trdp[t] + a1 * tlo + a2 * h["tl"][t][0] + a3 * h["tl"][t][1]
            lo = torch.maximum(mn, torch.minimum(mx, lo / dp.clamp(min=1e-11)))
            mx = pos(torch.maximum(torch.maximum(mx, lo), lo[prox].amax(1)))
            mn = pos(torch.minimum(torch.minimum(mn, lo), lo[prox].amin(1)))
            to, tv = h["tt"][t]
            rp = (((mx - lo) * dp - (a2 * neg(to) + a3 * pos(tv))) / a1 * area / (-neg(a)).sum(1).clamp(min=1e-11)).clamp(0, 1)
            rm = (((lo - mn) * dp + (a2 * pos(to) + a3 * neg(tv))) / a1 * area / pos(a).sum(1).clamp(min=1e-11)).clamp(0, 1)
            a = a * torch.where(a >= 0, torch.minimum(rm[:, None, :], rp[prox]), torch.minimum(rp[:, None, :], rm[prox]))
            tt = tlo - a.sum(1) * ra
            h["tl"][t], h["tt"][t] = [tlo, h["tl"][t][0]], [tt, to]
            trdp[t] = trdp[t] + a1 * tt + a2 * to + a3 * tv
            new.append(torch.maximum(mn, torch.minimum(mx, trdp[t] / dp.clamp(min=1e-11))))
        tr = torch.stack(new)
    return dict(dp=dp, pr=pr, ex=ex, tr=tr, trdp=trdp, ws=ws)
