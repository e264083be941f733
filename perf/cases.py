"""Timing cases of the engine: what a host program has it do, through its
public entry points, over the sizes it meets.

A case is a dict of plain values; "kind" selects the path:

  block   drop-in regular block of the Fortran host: gpunb_send_ of all
          predicted bodies, then gpunb_regf_ of the active ones in calls of
          1024 (host arrays in and out, gpunb_regfnn_ with "nearest").
  step    device-resident regular step with every body due: gpunb_jpset_ of
          the corrected bodies, gpunb_predict_, gpunb_regf_dev of all bodies
          against all bodies, gpunb_regcor_dev.
  ens     one regular step of every cluster of an ensemble: gpunb_ens_send,
          gpunb_ens_regf_dev.
  irr     one irregular block: predictor records and neighbour lists staged,
          irr_simd_firr_vec_ (host arrays in and out).
  pot     gpupot_ of the energy check (host arrays in and out).
  energy  energy check with KS pairs on device arrays: gpunb_energy_dev with
          the O(N^2) potential, the c.m. corrections and both sums.
  train   one epoch of the learned neighbour radius (rsnet.train).
  rs      learned neighbour radii of one regular block (rsnet.predict).

The engine is process-wide, as it is in a host program: a pass uploads the
bodies it works on, so passes of several states can follow each other.
"""
import ctypes
import math
import os

import numpy as np
import torch

os.environ.setdefault("GPUNB_QUIET", "1")   # no per-call log lines

from nbody6ppgpu_amd import energy, gpunb, ics, regcor, rsnet  # noqa: E402

CHUNK = 1024          # active bodies per gpunb_regf_ call (util_gpu.F)
NNBMAX = 500          # list capacity of the drop-in calls (LMAX = 501)
DEV_NNBMAX, DEV_LMAX = 550, 600
TIME = 1.0
DEV = "cuda"


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # The N = 1000 sample deck late in a block: a handful of active
        # bodies, where a call is all latency.
        dict(name="block_1k", kind="block", n=1000, ni=20, model="plummer",
             imf="equal", binaries=0.0, m_flag=0, nearest=False),
        # 16k Kroupa stars with a tenth of them in binaries (c.m. bodies),
        # mass-weighted lists, nearest neighbours: one full call.
        dict(name="block_16k_mflag", kind="block", n=16384, ni=1024,
             model="plummer", imf="kroupa", binaries=0.1, m_flag=1,
             nearest=True),
        # A regular block of the N = 131072 King cluster through the drop-in
        # ABI: three calls, the last one ragged.
        dict(name="block_131k", kind="block", n=131072, ni=3001, model="king",
             imf="kroupa", binaries=0.0, m_flag=0, nearest=False),
        # Every body due at once, device-resident: a medium cluster of an odd
        # size, and the benchmark cluster.
        dict(name="step_16k", kind="step", n=16411, model="plummer",
             imf="equal"),
        dict(name="step_131k", kind="step", n=131072, model="king",
             imf="kroupa"),
        # An ensemble of small and medium clusters.
        dict(name="ens_24", kind="ens", ncl=24, nmin=1024, nmax=16384,
             layout=5),
        # Irregular blocks: part of a small cluster, all of a large one.
        dict(name="irr_2k", kind="irr", n=2048, ni=300),
        dict(name="irr_131k", kind="irr", n=131072, ni=131072),
        # Energy checks: the drop-in potential, and the device sum with KS
        # pairs.
        dict(name="pot_131k", kind="pot", n=131072, ni=131072),
        dict(name="energy_31k", kind="energy", nsingle=30011, npairs=600),
        # Learned radius: an epoch over logged pairs, and a block's radii.
        dict(name="train_60k", kind="train", n=60000, batch=1024),
        dict(name="rs_20k", kind="rs", n=20011),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "step", "step", "ens", "irr",
                       "irr", "pot", "energy", "train", "rs"])
    if kind == "block":
        n = _logint(rng, 1000, 131072)
        return dict(kind=kind, n=n, ni=min(n, _logint(rng, 16, 4096)),
                    model=rng.choice(["plummer", "king"]),
                    imf=rng.choice(["equal", "kroupa"]),
                    binaries=rng.choice([0.0, 0.1]), m_flag=rng.choice([0, 1]),
                    nearest=rng.choice([False, True]))
    if kind == "step":
        return dict(kind=kind, n=_logint(rng, 2000, 131072),
                    model=rng.choice(["plummer", "king"]),
                    imf=rng.choice(["equal", "kroupa"]))
    if kind == "ens":
        nmin = _logint(rng, 500, 2000)
        return dict(kind=kind, ncl=rng.randint(4, 40), nmin=nmin,
                    nmax=nmin * rng.randint(2, 8), layout=rng.randint(1, 9999))
    if kind == "irr":
        n = _logint(rng, 1000, 131072)
        return dict(kind=kind, n=n, ni=min(n, _logint(rng, 32, n)))
    if kind == "pot":
        n = _logint(rng, 1000, 131072)
        return dict(kind=kind, n=n, ni=rng.choice([n, (n + 1) // 2]))
    if kind == "energy":
        return dict(kind=kind, nsingle=_logint(rng, 1000, 32000),
                    npairs=_logint(rng, 8, 700))
    if kind == "train":
        return dict(kind=kind, n=_logint(rng, 4000, 65536),
                    batch=rng.choice([256, 1024, 1024, 4096]))
    return dict(kind="rs", n=_logint(rng, 64, 131072))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _cluster(n, model, imf, seed, binaries=0.0):
    m = ics.kroupa(n, seed=seed + 1) if imf == "kroupa" else None
    c = ics.king(n, 6.0, seed=seed, m=m) if model == "king" else \
        ics.plummer(n, seed=seed, m=m)
    return ics.with_binaries(c, binaries, seed=seed + 2) if binaries else c


def _predictor_state(c, stepr, rng):
    """X0, X0DOT, F = a/2, FDOT = jerk/6, T0 of bodies last corrected within
    STEPR before TIME (a and jerk of the smooth cluster)."""
    r2 = np.sum(c.x * c.x, axis=1)
    a = -c.x / (r2 + 0.35)[:, None] ** 1.5
    j = -c.v / (r2 + 0.35)[:, None] ** 1.5
    step = stepr / 2.0 ** rng.integers(0, 5, c.n)
    return dict(x0=c.x, v0=c.v, f=0.5 * a, fdot=j / 6.0, t0=TIME - step, step=step)


def _predicted(p, t):
    """xbpredall.f:18-26 in the association of the engine."""
    s = (t - p["t0"])[:, None]
    x = ((p["fdot"] * s + p["f"]) * s + p["v0"]) * s + p["x0"]
    v = (p["fdot"] * (1.5 * s) + p["f"]) * (2.0 * s) + p["v0"]
    return x, v


_held = {}     # what the process-wide engine is open for


def _engine(n):
    if _held.get("reg") != n:
        if "reg" in _held:
            gpunb.gpunb_close()
        gpunb.gpunb_open(n + 10)
        _held["reg"] = n


def _irr_engine(n, lmax):
    if _held.get("irr") != (n, lmax):
        if "irr" in _held:
            gpunb.irr_close()
        gpunb.irr_open(n, lmax)
        _held["irr"] = (n, lmax)


def _rc(rc):
    if rc != 0:
        gpunb._check()


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _empty(shape, dtype=torch.float64):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _regf_dev(h2, dtr, x, v, o, nnbmax, lib):
    return lib.gpunb_regf_dev(
        h2.shape[0], h2.data_ptr(), dtr.data_ptr(), x.data_ptr(), v.data_ptr(),
        o["acc"].data_ptr(), o["jrk"].data_ptr(), o["pot"].data_ptr(), nnbmax,
        0, o["nnb"].data_ptr(), None, o["lst"].data_ptr(), o["off"].data_ptr(),
        o["total"].data_ptr(), o["lst"].shape[0])


def _regf_out(n, nnbmax):
    i = torch.int32
    return dict(acc=_empty((n, 3)), jrk=_empty((n, 3)), pot=_empty(n),
                nnb=_empty(n, i), off=_empty(n, i), total=_empty(1, i),
                lst=_empty(n * nnbmax, i))


def _rows(o, lmax):
    """Compact lists (0-based, body included) as LIST rows: count, 1-based
    members without the body."""
    nnb, off = o["nnb"].long(), o["off"].long()
    n = nnb.shape[0]
    if int(nnb.min()) < 1 or int(nnb.max()) + 1 > lmax:
        raise RuntimeError("a neighbour list of the case is out of range")
    row = torch.repeat_interleave(torch.arange(n, device=DEV), nnb)
    k = torch.arange(row.shape[0], device=DEV) - (torch.cumsum(nnb, 0) - nnb)[row]
    mem = o["lst"][off[row] + k].long()
    own = mem == row
    at = _empty(n, torch.int64)
    at[row[own]] = k[own]
    before = (k > at[row]).long()
    rows = _empty((n, lmax), torch.int32)
    rows[:, 0] = (nnb - 1).int()
    keep = ~own
    rows[row[keep], (1 + k - before)[keep]] = (mem[keep] + 1).int()
    return rows


def _ens_sizes(case):
    rng = np.random.default_rng(case["layout"])
    return np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]),
                              case["ncl"])).astype(int)


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _host_block(case, seed):
    c = _cluster(case["n"], case["model"], case["imf"], seed, case["binaries"])
    rs, dtr = ics.neighbour_radii(c)
    h2 = rs * rs
    if case["m_flag"]:
        h2 = h2 / c.m.mean()
    act = np.sort(np.random.default_rng(seed + 5).permutation(c.n)[:case["ni"]])
    return c, h2[act], dtr[act], act


def _prepare_block(case, seed):
    c, h2, dtr, act = _host_block(case, seed)
    ni, lmax = len(act), NNBMAX + 1
    _engine(c.n)
    return dict(kind="block", lib=gpunb.load(), m=c.m, x=c.x, v=c.v, h2=h2, dtr=dtr,
                xi=c.x[act].copy(), vi=c.v[act].copy(), acc=np.zeros((ni, 3)),
                jrk=np.zeros((ni, 3)), pot=np.zeros(ni),
                lst=np.zeros((ni, lmax), np.int32),
                nnid=np.zeros(ni, np.int32), lmax=lmax,
                m_flag=case["m_flag"], nearest=case["nearest"])


def _step_inputs(case, seed):
    c = _cluster(case["n"], case["model"], case["imf"], seed)
    rs, stepr = ics.neighbour_radii(c)
    p = _predictor_state(c, stepr, np.random.default_rng(seed + 7))
    return c, rs, stepr, p


def _prepare_step(case, seed):
    c, rs, stepr, p = _step_inputs(case, seed)
    n, lib = c.n, gpunb.load()
    _engine(n)
    pd = {k: _dev(a) for k, a in p.items()}
    xi, vi = _predicted(pd, TIME)
    xi, vi = xi.contiguous(), vi.contiguous()
    s = dict(kind="step", lib=lib, n=n, p=p, m=c.m,
             addr=np.arange(1, n + 1, dtype=np.int32), xi=xi, vi=vi,
             h2=_dev(rs * rs), dtr=_dev(stepr), out=_regf_out(n, DEV_NNBMAX),
             idx=torch.arange(1, n + 1, dtype=torch.int32, device=DEV),
             cnt=_empty(4, torch.int32))
    s["stream"] = torch.cuda.ExternalStream(gpunb.gpunb_stream())
    # The old lists (radius 0.9 RS) that the corrector compares with; the new
    # ones have to fit too.
    gpunb.gpunb_jpset(s["addr"], p["x0"], p["v0"], p["f"], p["fdot"], c.m, p["t0"])
    gpunb.gpunb_predict(TIME)
    for fac in (1.0, 0.81):
        h2 = s["h2"] * fac
        torch.cuda.synchronize()
        _rc(_regf_dev(h2, s["dtr"], xi, vi, s["out"], DEV_NNBMAX, lib))
        gpunb.gpunb_sync()
        if int(s["out"]["nnb"].min()) < 1:
            raise RuntimeError("a neighbour list of the case overflows")
    old = {k: a.clone() for k, a in s["out"].items() if k != "lst"}
    rows = _rows(s["out"], DEV_LMAX)
    g = torch.Generator(device=DEV).manual_seed(seed)
    wob = lambda a: a * (1.0 + 0.01 * torch.randn(  # noqa: E731
        a.shape, dtype=a.dtype, device=DEV, generator=g))
    step = pd["step"]
    pristine = dict(x0=xi, x0dot=vi, fi=0.3 * wob(old["acc"]),
                    fidot=0.3 * wob(old["jrk"]), fr=wob(old["acc"]),
                    frdot=wob(old["jrk"]), t0r=TIME - s["dtr"],
                    stepr=s["dtr"].clone(), step=step, t0=torch.full_like(step, TIME),
                    timenw=TIME + step, rs=_dev(0.9 * rs), body=_dev(c.m), list=rows)
    for k in ("xn", "xndot", "d0", "d0r", "d1r", "d2r", "d3r"):
        pristine[k] = _empty((n, 3))
    # What a block changes, as it was before the block: restored by each
    # pass, so that a pass corrects the same block every time.
    changed = ("fi", "fidot", "fr", "frdot", "t0r", "stepr", "step", "timenw",
               "rs", "list")
    s["state"] = {k: a.clone() for k, a in pristine.items()}
    s["from"] = [pristine[k] for k in changed]
    s["to"] = [s["state"][k] for k in changed]
    st = gpunb.RegcorState()
    for k in gpunb.REGCOR_VEC + gpunb.REGCOR_SCAL + ("list",):
        setattr(st, k, s["state"][k].data_ptr())
    st.h = None
    s["st"] = st
    s["par"] = regcor.make_par(
        time=TIME, rscale=1.0, rdens=(0.0, 0.0, 0.0), rc2=0.0025, rsfac=2.0,
        znbmin=10.0, smax=0.125, dtmin=1e-9, etar=0.02, smin=0.0,
        bodym=float(c.m.mean()), tidal4=0.0, nnbopt=50, nnbmax=DEV_NNBMAX, n=n,
        ntot=n, ifirst=1, lmax=DEV_LMAX, nb_flag=1, m_flag=0)
    return s


def _ens_inputs(case, seed):
    out = []
    for c, n in enumerate(_ens_sizes(case)):
        cl = _cluster(int(n), "plummer", "kroupa" if c % 2 else "equal",
                      seed + 17 * c)
        rs, dtr = ics.neighbour_radii(cl)
        out.append((cl, rs * rs, dtr))
    return out


def _prepare_ens(case, seed):
    cl = _ens_inputs(case, seed)
    key = tuple(c[0].n for c in cl)
    if _held.get("ens") != key:
        if "ens" in _held:
            gpunb.gpunb_ens_close()
        gpunb.gpunb_ens_open(key)
        _held["ens"] = key
    cat = lambda f: np.ascontiguousarray(np.concatenate([f(c) for c in cl]))  # noqa: E731
    n = sum(key)
    x, v = cat(lambda c: c[0].x), cat(lambda c: c[0].v)
    s = dict(kind="ens", lib=gpunb.load(), m=cat(lambda c: c[0].m), x=x, v=v,
             nj=np.array(key, np.int32), xi=_dev(x), vi=_dev(v),
             h2=_dev(cat(lambda c: c[1])), dtr=_dev(cat(lambda c: c[2])),
             out=_regf_out(n, DEV_NNBMAX))
    s["out"]["nnid"] = _empty(n, torch.int32)
    return s


def _prepare_irr(case, seed):
    n, ni = case["n"], case["ni"]
    rng = np.random.default_rng(seed + 9)
    c = _cluster(n, "plummer", "kroupa", seed)
    rs, stepr = ics.neighbour_radii(c)
    p = _predictor_state(c, stepr, rng)
    act = np.sort(rng.permutation(n)[:ni])
    # Neighbour lists of the active bodies, as the regular force left them.
    _engine(n)
    gpunb.gpunb_send(c.m, c.x, c.v)
    o = _regf_out(n, DEV_NNBMAX)
    h2, dtr, x, v = (_dev(a) for a in (rs * rs, 0.0 * stepr, c.x, c.v))
    torch.cuda.synchronize()
    _rc(_regf_dev(h2, dtr, x, v, o, DEV_NNBMAX, gpunb.load()))
    gpunb.gpunb_sync()
    rows = _rows(o, DEV_LMAX)[torch.from_numpy(act).to(DEV)]
    nnb = rows[:, 0].long()
    keep = torch.arange(DEV_LMAX - 1, device=DEV)[None, :] < nnb[:, None]
    mem = rows[:, 1:][keep].cpu().numpy()
    _irr_engine(n, DEV_LMAX)
    return dict(kind="irr", lib=gpunb.load(), n=n, ni=ni, p=p, m=c.m,
                addr=np.arange(1, n + 1, dtype=np.int32),
                act=(act + 1).astype(np.int32), nnb=nnb.int().cpu().numpy(),
                mem=np.ascontiguousarray(mem), acc=np.zeros((ni, 3)),
                jrk=np.zeros((ni, 3)), nnid=np.zeros(ni, np.int32))


def _prepare_pot(case, seed):
    c = _cluster(case["n"], "plummer", "kroupa", seed)
    return dict(kind="pot", lib=gpunb.load(), n=c.n, ni=case["ni"], m=c.m, x=c.x,
                pot=np.zeros(case["ni"]))


CMSEP2 = 0.03 ** 2


def _ks(case, seed):
    return ics.ks_system(nsingle=case["nsingle"], npairs=case["npairs"],
                         seed=seed, rnb=0.08, rpert=0.1)


def _prepare_energy(case, seed):
    k = _ks(case, seed)
    return dict(kind="energy", par=energy.make_par(k["n"], k["ntot"], k["lmax"], CMSEP2),
                body=_dev(k["body"]), x=_dev(k["x"]), xdot=_dev(k["xdot"]),
                list=_dev(k["list"]), phi=_empty(k["ntot"]), out=_empty(2))


def _pairs(n, seed):
    """Feature / target pairs of the driver's training log, in distribution."""
    rng = np.random.default_rng(seed)
    mean = np.array([1.0, 0.8, 0.2, 0.4, -0.1, -0.2, 5.0, -0.8])
    std = np.array([0.9, 0.3, 0.4, 0.7, 0.3, 0.4, 1.0, 0.35])
    z = rng.normal(0.0, 1.0, (n, rsnet.NI))
    t = (-0.8 + 0.3 * z[:, 7] - 0.12 * z[:, 0] + 0.05 * np.sin(2.0 * z[:, 2]) -
         0.06 * z[:, 1] + rng.normal(0.0, 0.02, n))
    return ((mean + std * z).astype(np.float32), t.astype(np.float32),
            mean.astype(np.float32), std.astype(np.float32))


def _prepare_train(case, seed):
    X, t, mean, std = _pairs(case["n"], seed)
    rsnet.init(seed % 1000 + 1)
    return dict(kind="train", X=X, t=t, norm=(mean, std, -0.8, 0.35),
                p0=rsnet.get_params(), batch=case["batch"])


def _prepare_rs(case, seed):
    X, _, mean, std = _pairs(case["n"], seed)
    rsnet.init(1)                       # the weights the program keeps
    rsnet.set_norm(mean, std, -0.8, 0.35)
    return dict(kind="rs", X=X)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_block(s):
    gpunb.gpunb_send(s["m"], s["x"], s["v"])
    P, I, lib = gpunb._p, gpunb._i, s["lib"]
    for k in range(0, len(s["h2"]), CHUNK):
        q = slice(k, k + CHUNK)
        args = (I(len(s["h2"][q])), P(s["h2"][q]), P(s["dtr"][q]), P(s["xi"][q]),
                P(s["vi"][q]), P(s["acc"][q]), P(s["jrk"][q]), P(s["pot"][q]),
                I(s["lmax"]), I(NNBMAX), P(s["lst"][q]), I(s["m_flag"]))
        if s["nearest"]:
            lib.gpunb_regfnn_(*args, P(s["nnid"][q]))
        else:
            lib.gpunb_regf_(*args)
        gpunb._check()
    return {k: s[k] for k in ("acc", "jrk", "pot", "lst", "nnid")}


def _run_step(s):
    p, lib, o = s["p"], s["lib"], s["out"]
    gpunb.gpunb_jpset(s["addr"], p["x0"], p["v0"], p["f"], p["fdot"], s["m"], p["t0"])
    gpunb.gpunb_predict(TIME)
    with torch.cuda.stream(s["stream"]):
        torch._foreach_copy_(s["to"], s["from"])
        s["cnt"].zero_()
    _rc(_regf_dev(s["h2"], s["dtr"], s["xi"], s["vi"], o, DEV_NNBMAX, lib))
    _rc(lib.gpunb_regcor_dev(
        ctypes.byref(s["par"]), ctypes.byref(s["st"]), s["n"], s["idx"].data_ptr(),
        s["xi"].data_ptr(), s["vi"].data_ptr(), o["acc"].data_ptr(),
        o["jrk"].data_ptr(), o["nnb"].data_ptr(), o["off"].data_ptr(),
        o["lst"].data_ptr(), o["lst"].shape[0], s["cnt"].data_ptr()))
    # The compact lists come in no fixed order of bodies: LIST holds them.
    return dict(acc=o["acc"], jrk=o["jrk"], pot=o["pot"], nnb=o["nnb"],
                total=o["total"], counters=s["cnt"],
                state={k: s["state"][k] for k in
                       ("xn", "xndot", "fi", "fidot", "fr", "frdot", "d0", "d0r",
                        "d1r", "d2r", "d3r", "t0r", "stepr", "step", "timenw",
                        "rs", "list")})


def _run_ens(s):
    o, P, lib = s["out"], gpunb._p, s["lib"]
    ncl = len(s["nj"])
    _rc(lib.gpunb_ens_send(ncl, P(s["nj"]), P(s["m"]), P(s["x"]), P(s["v"])))
    _rc(lib.gpunb_ens_regf_dev(
        ncl, P(s["nj"]), s["h2"].data_ptr(), s["dtr"].data_ptr(),
        s["xi"].data_ptr(), s["vi"].data_ptr(), o["acc"].data_ptr(),
        o["jrk"].data_ptr(), o["pot"].data_ptr(), DEV_NNBMAX, 0,
        o["nnb"].data_ptr(), o["nnid"].data_ptr(), o["lst"].data_ptr(),
        o["off"].data_ptr(), o["total"].data_ptr(), o["lst"].shape[0]))
    # The compact lists come in no fixed order of bodies.
    return {k: o[k] for k in ("acc", "jrk", "pot", "nnb", "nnid", "total")}


def _run_irr(s):
    P, p, lib = gpunb._p, s["p"], s["lib"]
    gpunb.irr_set_jp(s["addr"], p["x0"], p["v0"], p["f"], p["fdot"], s["m"], p["t0"])
    _rc(lib.gpunb_irr_set_lists(s["ni"], P(s["act"]), P(s["nnb"]), P(s["mem"])))
    lib.irr_simd_firr_vec_(ctypes.byref(ctypes.c_double(TIME)), gpunb._i(s["ni"]),
                           P(s["act"]), P(s["acc"]), P(s["jrk"]), P(s["nnid"]))
    gpunb._check()
    return {k: s[k] for k in ("acc", "jrk", "nnid")}


def _run_pot(s):
    P, I = gpunb._p, gpunb._i
    s["lib"].gpupot_(I(0), I(1), I(s["ni"]), I(s["n"]), P(s["m"]), P(s["x"]), P(s["pot"]))
    gpunb._check()
    return s["pot"]


def _run_energy(s):
    energy.energy_dev(s["par"], s["body"].data_ptr(), s["x"].data_ptr(),
                      s["xdot"].data_ptr(), s["list"].data_ptr(), True,
                      s["phi"].data_ptr(), s["out"].data_ptr())
    return dict(phi=s["phi"], pot_zkin=s["out"])


def _run_train(s):
    rsnet.set_params(s["p0"])
    rsnet.set_norm(*s["norm"])
    loss = rsnet.train(s["X"], s["t"], 1, s["batch"], 2e-3, 3)
    return dict(loss=loss, params=rsnet.get_params())


def _run_rs(s):
    return rsnet.predict(s["X"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

PAIR_FLOPS = 60       # of the force and jerk of one pair, as the host reports
POT_FLOPS = 10


def work(case):
    k = case["kind"]
    if k == "block":
        n, ni = case["n"], case["ni"]
        return dict(bytes=56 * n + (64 + 56 + 4 * 57) * ni, flops=PAIR_FLOPS * n * ni)
    if k == "step":
        n = case["n"]
        return dict(bytes=n * (112 + 64 + 56 + 660 + 4 * 3 * 52), flops=PAIR_FLOPS * n * n)
    if k == "ens":
        z = [int(n) for n in _ens_sizes(case)]
        return dict(bytes=sum(z) * (56 + 64 + 56 + 4 * 55),
                    flops=PAIR_FLOPS * sum(n * n for n in z))
    if k == "irr":
        n, ni = case["n"], case["ni"]
        return dict(bytes=112 * n + ni * (4 + 4 * 50 + 52), flops=PAIR_FLOPS * ni * 48)
    if k == "pot":
        return dict(bytes=32 * case["n"] + 8 * case["ni"],
                    flops=POT_FLOPS * case["n"] * case["ni"])
    if k == "energy":
        n = case["nsingle"] + case["npairs"]
        return dict(bytes=n * (8 + 24 + 24 + 8), flops=POT_FLOPS * n * n)
    fwd = 2 * (rsnet.NI * rsnet.NH + rsnet.NH * rsnet.NH + rsnet.NH)
    if k == "train":
        return dict(bytes=case["n"] * 36 + 8 * rsnet.NP, flops=3 * fwd * case["n"])
    return dict(bytes=case["n"] * 36, flops=fwd * case["n"])


# ---------------------------------------------------------------------------
# The same outputs in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _rows_at_a_time(n):
    return max(1, (1 << 26) // max(n, 1))


def _exact_regf(m, x, v, h2, dtr, xi, vi, m_flag):
    """acc, jrk, pot over the bodies that are not neighbours (gpunb.h)."""
    n, ni = m.shape[0], h2.shape[0]
    acc, jrk, pot = _empty((ni, 3)), _empty((ni, 3)), _empty(ni)
    b = _rows_at_a_time(n)
    for k in range(0, ni, b):
        q = slice(k, k + b)
        d = [x[None, :, c] - xi[q, None, c] for c in range(3)]
        u = [v[None, :, c] - vi[q, None, c] for c in range(3)]
        r2 = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]
        e = [d[c] + dtr[q, None] * u[c] for c in range(3)]
        near = torch.minimum(r2, (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2])
        del e
        near = near < ((m[None, :] * h2[q, None]) if m_flag else h2[q, None])
        near |= r2 == 0.0
        rinv = torch.where(near, torch.zeros_like(r2), 1.0 / torch.sqrt(r2))
        del near, r2
        mr = m[None, :] * rinv
        pot[q] = mr.sum(1)
        rinv *= rinv
        mr *= rinv
        al = (d[0] * u[0] + d[1] * u[1] + d[2] * u[2]) * rinv * -3.0
        for c in range(3):
            acc[q, c] = (mr * d[c]).sum(1)
            jrk[q, c] = (mr * (u[c] + al * d[c])).sum(1)
    return acc, jrk, pot


def _exact_pot(m, x, ni):
    pot = _empty(ni)
    b = _rows_at_a_time(m.shape[0])
    for k in range(0, ni, b):
        r2 = 0.0
        for c in range(3):
            d = x[None, :, c] - x[k:min(k + b, ni), None, c]
            r2 = r2 + d * d
        pot[k:k + b] = torch.where(r2 > 0.0, m[None, :] / torch.sqrt(r2), 0.0).sum(1)
    return pot


def exact(case, seed):
    f = globals().get("_exact_case_" + case["kind"])
    return f(case, seed) if f else None


def _exact_case_block(case, seed):
    c, h2, dtr, act = _host_block(case, seed)
    m, x, v = _dev(c.m), _dev(c.x), _dev(c.v)
    a = torch.from_numpy(act).to(DEV)
    acc, jrk, pot = _exact_regf(m, x, v, _dev(h2), _dev(dtr), x[a], v[a], case["m_flag"])
    return dict(acc=acc, jrk=jrk, pot=pot, lst=None, nnid=None)


def _exact_case_step(case, seed):
    c, rs, stepr, p = _step_inputs(case, seed)
    x, v = _predicted({k: _dev(a) for k, a in p.items()}, TIME)
    acc, jrk, pot = _exact_regf(_dev(c.m), x, v, _dev(rs * rs), _dev(stepr), x, v, 0)
    return dict(acc=acc, jrk=jrk, pot=pot, nnb=None, total=None, counters=None,
                state=None)


def _exact_case_ens(case, seed):
    out = []
    for c, h2, dtr in _ens_inputs(case, seed):
        x, v = _dev(c.x), _dev(c.v)
        out.append(_exact_regf(_dev(c.m), x, v, _dev(h2), _dev(dtr), x, v, 0))
    acc, jrk, pot = (torch.cat(a) for a in zip(*out))
    return dict(acc=acc, jrk=jrk, pot=pot, nnb=None, nnid=None, total=None)


def _exact_case_irr(case, seed):
    s = _prepare_irr(case, seed)
    x, v = _predicted({k: _dev(a) for k, a in s["p"].items()}, TIME)
    nnb = _dev(s["nnb"]).long()
    row = torch.repeat_interleave(torch.arange(case["ni"], device=DEV), nnb)
    i, j = _dev(s["act"]).long()[row] - 1, _dev(s["mem"]).long() - 1
    d, u = x[j] - x[i], v[j] - v[i]
    r2 = (d * d).sum(1)
    mr3 = _dev(s["m"])[j] / (r2 * torch.sqrt(r2))
    al = -3.0 * (d * u).sum(1) / r2
    zero = _empty((case["ni"], 3))
    return dict(acc=zero.index_add(0, row, mr3[:, None] * d),
                jrk=zero.index_add(0, row, mr3[:, None] * (u + al[:, None] * d)),
                nnid=None)


def _exact_case_pot(case, seed):
    c = _cluster(case["n"], "plummer", "kroupa", seed)
    return _exact_pot(_dev(c.m), _dev(c.x), case["ni"])


def _exact_case_energy(case, seed):
    k = _ks(case, seed)
    n, ntot, first = k["n"], k["ntot"], k["ifirst"] - 1
    b, x, lst = k["body"], k["x"], k["list"]
    phi = np.zeros(ntot)
    phi[first:] = _exact_pot(_dev(b[first:]), _dev(x[first:]), ntot - first).cpu().numpy()
    term = lambda i, j: b[j] / np.sqrt(np.sum((x[j] - x[i]) ** 2, axis=-1))  # noqa: E731
    # Singles: c.m. neighbours inside the resolution radius by components.
    at = np.arange(1, k["lmax"])[None, :] <= lst[:, :1]
    i, col = np.nonzero(at & (lst[:, 1:] > n))
    j = lst[i, col + 1] - 1
    use = (i >= first) & (np.sum((x[i] - x[j]) ** 2, axis=1) < CMSEP2)
    i, j = i[use], j[use]
    j1 = 2 * (j - n)
    np.add.at(phi, i, term(i, j1) + term(i, j1 + 1) - term(i, j))
    # Components: the c.m. value, its perturbers resolved against each.
    for p in range(k["npairs"]):
        cm, mem = n + p, lst[2 * p, 1:1 + lst[2 * p, 0]] - 1
        s, g = mem[mem < n], mem[mem >= n]
        for i in (2 * p, 2 * p + 1):
            phi[i] = (phi[cm] - term(cm, mem).sum() + term(i, s).sum() +
                      term(i, 2 * (g - n)).sum() + term(i, 2 * (g - n) + 1).sum())
    pot = 0.5 * np.sum(b[:n] * phi[:n])
    kin = 0.5 * np.sum(b[first:] * np.sum(k["xdot"][first:] ** 2, axis=1))
    return dict(phi=phi, pot_zkin=np.array([pot, kin]))


def _exact_case_rs(case, seed):
    X, _, mean, std = _pairs(case["n"], seed)
    rsnet.init(1)
    w = rsnet.get_params().astype(np.float64)
    ni, nh = rsnet.NI, rsnet.NH
    cut = np.cumsum([nh * ni, nh, nh * nh, nh, nh])
    w1, b1, w2, b2, w3, b3 = np.split(w, cut)
    h = (X.astype(np.float64) - mean) / std
    for a, c in ((w1.reshape(nh, ni), b1), (w2.reshape(nh, nh), b2)):
        z = h @ a.T + c
        h = z / (1.0 + np.exp(-z))
    return (h @ w3 + b3) * 0.35 - 0.8
