"""Timing cases of the spectral-synthesis path, through its public entry points.

A case is a dict of plain values; ``kind`` names the entry point:

* ``spectrum``  one request on a resident line list, ``SpectrumBatch.run``
  (``option``: simple or min-RMS weights, two-temperature strengths, or the
  derived quantities written beside abscoeff);
* ``iterate``   ``gpuApp.iterate``: one condition in, one host array out;
* ``noalloc``   ``run_noalloc``: one request in the fixed scratch array;
* ``batch``     many windows of one list replayed as one hipGraph;
* ``serve``     a burst of requests through ``SpectrumServer``;
* ``slit``      ``slit.convolve_device``: an instrumental slit on a spectrum.

Line lists are synthetic with the repository's benchmark distributions
(wavenumbers and broadening uniform, intensities log-uniform, lower-state
energies exponential).  ``columns`` is ``plain`` (one isotopologue, no shift,
n_self = n_air, as the benchmark lists) or ``hitran`` (three isotopologues,
pressure shifts and n_self, as a HITRAN list has them).
"""
import math

import numpy as np
import torch

from radis_amd import engine, gpu_app, serve, slit, workloads

H, KB, C = 6.62607015e-34, 1.3806490e-23, 2.99792458e8
NA, KB_CGS, C_CGS = 6.02214076e23, 1.380648813e-16, 2.99792458e10
C2 = H * C / KB * 100
ATM = 1.01325
TREF = 296.0
DXL = math.log((0.01 / 0.20) ** 0.5 + 1)
DXG = math.log((0.01 / 0.46) ** 0.5 + 1)
FOLD = 1e-6
MOLAR_MASS = (0.0, 44.0, 45.0, 46.0)
PATH = 10.0  # cm, derived quantities


def listed():
    s = dict(kind="spectrum", columns="plain", option="simple", dx=0.0)
    return [
        # an interactive caller: a HITRAN-sized list on RADIS's default step, one
        # new spectrum on the host per call
        dict(name="iterate_40k", kind="iterate", columns="hitran", n=5_000, lo=1900.0, hi=2300.0, wmin=1900.0,
             wmax=2300.0, wstep=0.01, T=700.0, p=1.0, x=0.1, dx=0.0),
        # the smallest call: a narrow window without any allocation
        dict(name="noalloc_20k", kind="noalloc", columns="hitran", n=20_000, lo=2000.0, hi=2100.0, wmin=2020.0,
             wmax=2060.0, wstep=0.002, T=1200.0, p=0.5, x=0.2, dx=0.0),
        # few lines on a long grid: the transforms are everything (co_5k)
        dict(s, name="co_5k", n=5_000, lo=1900.0, hi=2300.0, wmin=1900.0, wmax=2300.0, wstep=0.002, T=700.0,
             p=ATM, x=0.1, dx=0.2),
        # the CO2 benchmark workload (co2_5m)
        dict(s, name="co2_5m", n=5_000_000, lo=2000.0, hi=2500.0, wmin=2000.0, wmax=2500.0, wstep=0.001, T=1500.0,
             p=ATM, x=0.1),
        # a dense hot list at high pressure, twelve nodes on both width axes
        # (the h2o_100m grid and conditions on a 20 M-line list)
        dict(s, name="h2o_20m", n=20_000_000, lo=1000.0, hi=4000.0, wmin=1000.0, wmax=4000.0, wstep=0.005, T=2500.0,
             p=5 * ATM, x=0.1),
        # a ragged window inside a list with every HITRAN column
        dict(s, name="window_hitran_1m", columns="hitran", n=1_000_000, lo=2000.0, hi=2500.0, wmin=2113.37,
             wmax=2269.91, wstep=0.0013, T=960.0, p=0.3, x=0.25),
        # two-temperature absorption
        dict(s, name="noneq_500k", columns="hitran", n=500_000, lo=2000.0, hi=2400.0, wmin=2000.0, wmax=2400.0,
             wstep=0.003, T=1100.0, p=0.7, x=0.4, option="noneq"),
        # min-RMS weights
        dict(s, name="min_rms_300k", n=300_000, lo=3000.0, hi=3200.0, wmin=3000.0, wmax=3200.0, wstep=0.004,
             T=450.0, p=2.5, x=0.05, option="min-RMS"),
        # the factory's quantities: absorbance, emissivity, transmittance, radiance
        dict(s, name="derived_200k", columns="hitran", n=200_000, lo=2100.0, hi=2400.0, wmin=2100.0, wmax=2400.0,
             wstep=0.002, T=1800.0, p=1.0, x=0.1, option="derived"),
        # many windows and conditions in one captured graph (batch_256's form)
        dict(name="batch_32", kind="batch", columns="plain", n=2_000_000, lo=2000.0, hi=2500.0, count=32,
             wstep=0.001, width=50.0, dx=0.0),
        # served requests: planning, launch, copies to the host and completion
        dict(name="serve_16", kind="serve", columns="plain", n=1_000_000, lo=2000.0, hi=2500.0, count=16,
             wstep=0.002, width=50.0, dx=0.0),
        # a 0.5 cm-1 slit on the 500,002-point grid
        dict(name="slit_500k", kind="slit", points=500_002, wstep=0.001, shape="gaussian", fwhm=0.5, mode="valid"),
    ]


def _logu(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choice(["spectrum"] * 6 + ["iterate", "noalloc", "batch", "serve", "slit", "slit"])
    if kind == "slit":
        ws = rng.choice([0.001, 0.002, 0.005, 0.01])
        pts = int(_logu(rng, 5_000, 500_000))
        taps = _logu(rng, 20, min(1700, pts / 3))
        # points of each shape per grid step of FWHM: 2 (triangular), 3.4 (gaussian)
        shape = rng.choice(["triangular", "gaussian"])
        return dict(kind="slit", points=pts, wstep=ws, shape=shape,
                    fwhm=round(max(6.3, taps / (2 if shape == "triangular" else 3.4)) * ws, 6),
                    mode=rng.choice(["valid", "same"]))
    columns = rng.choice(["plain", "hitran"])
    if kind in ("batch", "serve"):
        return dict(kind=kind, columns=columns, n=int(_logu(rng, 50_000, 2_000_000)), lo=2000.0, hi=2500.0,
                    count=rng.randint(2, 32 if kind == "batch" else 16), wstep=rng.choice([0.001, 0.002, 0.005]),
                    width=round(rng.uniform(15.0, 50.0), 3), dx=0.0)
    lo = round(rng.uniform(800.0, 4000.0), 3)
    points = int(_logu(rng, 2_000, 100_000 if kind != "spectrum" else 600_000))
    wstep = rng.choice([0.001, 0.002, 0.005, 0.01])
    hi = round(lo + points * wstep, 6)
    n = int(min(60 * points, _logu(rng, 1_000, 200_000 if kind != "spectrum" else 5_000_000)))
    wmin, wmax = lo, hi
    if kind != "iterate" and rng.random() < 0.5:  # a window strictly inside the list
        wmin, wmax = round(lo + 0.07 * (hi - lo), 5), round(hi - 0.05 * (hi - lo), 5)
    case = dict(kind=kind, columns=columns, n=n, lo=lo, hi=hi, wmin=wmin, wmax=wmax, wstep=wstep,
                T=round(rng.uniform(300.0, 3000.0), 2), p=round(_logu(rng, 0.1, 10.0), 4),
                x=round(rng.uniform(0.01, 1.0), 3), dx=rng.choice([0.0, 0.0, 0.2]))
    if kind == "spectrum":
        case["option"] = rng.choice(["simple", "simple", "simple", "noneq", "min-RMS", "derived"])
    return case


# ---- inputs -----------------------------------------------------------------
def _q(iso, T):
    return (100.0 + 20.0 * iso) * (T / TREF) ** 1.3


def _qneq(iso, Tvib, Trot):
    return (100.0 + 20.0 * iso) * (Tvib / TREF) ** 0.3 * (Trot / TREF)


def _lines(case, seed):
    """The list's columns, sorted by nu0, in the types the device keeps."""
    rng = np.random.default_rng([seed, case["n"], 20])
    n, lo, hi = case["n"], case["lo"], case["hi"]
    f32 = np.float32
    gaps = rng.standard_exponential(n + 1)
    nu0 = np.cumsum(gaps)
    nu0 = lo + (hi - lo) * (nu0[:-1] / nu0[-1])

    def uni(a, b):
        return rng.random(n, dtype=f32) * f32(b - a) + f32(a)

    El = np.minimum(rng.standard_exponential(n, dtype=f32) * f32(1500.0), f32(4000.0))
    # intensity without the Boltzmann factor: log-uniform over six decades
    S = np.exp(uni(math.log(1e-27), math.log(1e-21)) - f32(C2 / TREF) * El)
    d = dict(nu0=nu0, S_ref=S, El=El, g_air=uni(0.03, 0.10), g_self=uni(0.05, 0.10), n_air=uni(0.5, 0.8))
    if case["columns"] == "hitran":
        if case["kind"] != "iterate":  # gpuApp's arguments hold one temperature exponent
            d["n_self"] = uni(0.4, 0.9)
        d["delta"] = uni(-0.01, 0.01)
        d["iso"] = rng.choice(np.array([1, 1, 1, 1, 1, 1, 2, 2, 2, 3], dtype=np.uint8), n)
    if case.get("option") == "noneq":
        d["Evib_l"] = El * uni(0.2, 0.9)
        d["Evib_u"] = d["Evib_l"] + (nu0 * 0.9).astype(f32)
    return d


def _with_functions(case, cols):
    mm = np.array(MOLAR_MASS if case["columns"] == "hitran" else MOLAR_MASS[:2])
    return dict(cols, molar_mass=mm, Q=_q, Qneq=_qneq)


def _steps(case):
    return (case["dx"], case["dx"]) if case["dx"] else (DXG, DXL)


def _conditions(case, seed):
    """The windows of a batch or a burst (the case's own) and their conditions (the seed's)."""
    rng, cnd = np.random.default_rng([case["count"], case["n"], 21]), np.random.default_rng([seed, 23])
    lo, hi = case["lo"], case["hi"]
    out = []
    for _ in range(case["count"]):
        W = float(np.clip(case["width"] * math.exp(0.8 * rng.standard_normal()), 10.0, 0.6 * (hi - lo)))
        a = rng.uniform(lo, hi - W)
        out.append(dict(wmin=round(a, 6), wmax=round(a + W, 6), T=cnd.uniform(300.0, 3000.0),
                        p=math.exp(cnd.uniform(math.log(0.1), math.log(20.0))), x=cnd.uniform(0.01, 1.0)))
    return out


def _request(db, case, c):
    dxG, dxL = _steps(case)
    kw = {}
    if case.get("option") == "noneq":
        kw = dict(Tvib=c["T"] * 1.8, Trot=c["T"])
    elif case.get("option") == "min-RMS":
        kw = dict(optimization="min-RMS")
    return engine.make_request(db, c["wmin"], c["wmax"], case["wstep"], c["T"], c["p"], c["x"], dxG=dxG, dxL=dxL,
                               Tref=TREF, **kw)


def _gpu_app_args(case, cols):
    iso = cols["iso"].astype(np.uint32) if "iso" in cols else np.ones(case["n"], dtype=np.uint32)
    El64, nu0 = cols["El"].astype(np.float64), cols["nu0"]
    q = np.array([1.0] + [_q(i, TREF) for i in (1, 2, 3)])[iso]
    S0 = cols["S_ref"].astype(np.float64) * q / (np.exp(-C2 * El64 / TREF) * (1 - np.exp(-C2 * nu0 / TREF)))
    gamma = np.stack([cols["g_self"], cols["g_air"]])
    da = cols.get("delta", np.zeros(case["n"], dtype=np.float32))
    nv = np.arange(case["wmin"], case["wmax"] + case["wstep"], case["wstep"]).size
    dxG, dxL = _steps(case)
    qs = [lambda T: 1.0] + [lambda T, i=i: _q(i, T) for i in (1, 2, 3)]
    return (case["wmin"], nv, case["wstep"], dxG, dxL, nu0, da, cols["n_air"], S0, cols["El"], gamma, iso,
            np.array(MOLAR_MASS), qs)


def _spectrum_and_slit(case, seed):
    """A transmittance-like spectrum (a continuum with lines) and the slit on its grid."""
    rng = np.random.default_rng([seed, case["points"], 22])
    n = case["points"]
    w = np.arange(n) * case["wstep"]
    depth = np.zeros(n)
    depth[rng.integers(0, n, max(4, n // 40))] = rng.exponential(3.0, max(4, n // 40))
    d = np.arange(-60, 61)
    I = np.exp(-np.convolve(depth, 1.0 / (1.0 + (d / rng.uniform(3.0, 12.0)) ** 2), mode="same"))
    ws, Is = slit.get_slit_function(case["fwhm"], shape=case["shape"], center_wavespace=w[n // 2], wstep=case["wstep"])
    return I.astype(np.float32), np.asarray(slit.slit_on_grid(ws, Is, case["wstep"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "slit":
        I, k = _spectrum_and_slit(case, seed)
        return dict(kind=kind, x=torch.as_tensor(I, device="cuda"), slit=k, wstep=case["wstep"], mode=case["mode"])
    cols = _lines(case, seed)
    if kind == "iterate":
        return dict(kind=kind, app=gpu_app.gpuApp(*_gpu_app_args(case, cols)), cond=(case["p"], case["T"], case["x"]))
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, _with_functions(case, cols))
    st = dict(kind=kind, dev=dev, db=db)
    if kind == "serve":
        dxG, dxL = _steps(case)
        st["server"] = serve.SpectrumServer(dev, {"list": db}, max_batch=8)
        st["conds"] = [workloads.Conditions(c["wmin"], c["wmax"], case["wstep"], c["T"], c["p"], c["x"], dxG=dxG,
                                            dxL=dxL, Tref=TREF) for c in _conditions(case, seed)]
        return st
    conds = _conditions(case, seed) if kind == "batch" else [case]
    reqs = [_request(db, case, c) for c in conds]
    if kind == "noalloc":
        _, inf = db.request_bytes(reqs[0])
        st["req"] = reqs[0]
        st["out"] = torch.empty(int(inf.n_v), dtype=torch.float32, device="cuda")
        return st
    b = engine.SpectrumBatch(db, reqs)
    st["batch"] = b
    st["outs"] = b.alloc_outputs()
    if case.get("option") == "derived":
        st["derived"] = b.set_derived(0, PATH)
    if kind == "batch":
        b.run(st["outs"])
        torch.cuda.synchronize()
        b.capture(st["outs"])
    return st


def run(state):
    kind = state["kind"]
    if kind == "spectrum":
        outs = state["batch"].run(state["outs"])
        return {"abscoeff": outs[0], **state["derived"]} if "derived" in state else outs
    if kind == "iterate":
        return state["app"].iterate(*state["cond"])[0]
    if kind == "noalloc":
        engine.run_noalloc(state["db"], state["req"], state["out"])
        return state["out"]
    if kind == "batch":
        return state["batch"].replay()
    if kind == "serve":
        recs = [state["server"].submit("list", c) for c in state["conds"]]
        state["server"].drain()
        state["server"].done.clear()
        return [r.result for r in recs]
    return slit.convolve_device(state["x"], state["slit"], state["wstep"], mode=state["mode"])


# ---- what a pass cannot do without ---------------------------------------------
def work(case):
    if case["kind"] == "slit":
        k = case["fwhm"] / case["wstep"] * (2.0 if case["shape"] == "triangular" else 3.4)
        return {"bytes": 8.0 * case["points"] + 4.0 * k, "flops": 2.0 * case["points"] * k}
    per = 28.0 + (9.0 if case["columns"] == "hitran" else 0.0) + (8.0 if case.get("option") == "noneq" else 0.0)
    if case["kind"] in ("batch", "serve"):
        width = 1.37 * case["width"] * case["count"]  # the mean of the log-normal widths
        lines, points = case["n"] * width / (case["hi"] - case["lo"]), width / case["wstep"]
    else:
        lines = case["n"] * (case["wmax"] - case["wmin"]) / (case["hi"] - case["lo"])
        points = (case["wmax"] - case["wmin"]) / case["wstep"]
    return {"bytes": per * lines + 4.0 * points * (5.0 if case.get("option") == "derived" else 1.0),
            "flops": 60.0 * lines + 10.0 * points * math.log2(max(2.0, points))}


# ---- the same in 64 bits ---------------------------------------------------------
def _axis(w, dx):
    n = math.ceil((math.log(float(w.max()) + 1e-4) - math.log(float(w.min()))) / dx) + 1
    return float(w.min()) * np.exp(dx * np.arange(n))


def _split(pos, n):
    pos = pos.clamp(0.0, float(n - 1))
    i = pos.floor().clamp(max=n - 2 if n > 1 else 0)
    return i.to(torch.int64), pos - i


def _exact_abscoeff(case, c, cols, dev):
    """RADIS's DIT spectrum (FFT length twice the grid) of one window, float64."""
    wmin, wmax, ws, T, p, x = c["wmin"], c["wmax"], case["wstep"], c["T"], c["p"], c["x"]
    nv = np.arange(wmin, wmax + ws, ws).size
    delta = (wmin + ws) - wmin
    i0, i1 = np.searchsorted(cols["nu0"], wmin, "left"), np.searchsorted(cols["nu0"], wmax, "right")
    t = {k: torch.as_tensor(v[i0:i1], device=dev) for k, v in cols.items()}
    nu0, El, S = t["nu0"], t["El"].double(), t["S_ref"].double()
    iso = t["iso"].long() if "iso" in t else None
    per_iso = (lambda f: torch.tensor([1.0] + [f(i) for i in (1, 2, 3)], device=dev, dtype=torch.float64)[iso]) \
        if iso is not None else (lambda f: f(1))
    patm = p / ATM
    lr = math.log(TREF / T)
    na = t["n_air"].double()
    ns = t["n_self"].double() if "n_self" in t else na
    wL = 2 * patm * (torch.exp(na * lr) * t["g_air"].double() * (1 - x) + torch.exp(ns * lr) * t["g_self"].double() * x)
    wG = 2 * nu0 / C_CGS * per_iso(lambda i: math.sqrt(2 * NA * KB_CGS * T * math.log(2.0) / MOLAR_MASS[i]))
    if case.get("option") == "noneq":
        Tv, Tr = 1.8 * T, T
        evl, dev_ = t["Evib_l"].double(), t["Evib_u"].double() - t["Evib_l"].double()
        S = S * per_iso(lambda i: _q(i, TREF) / _qneq(i, Tv, Tr)) \
            * torch.exp(-C2 * (evl / Tv + (El - evl) / Tr - El / TREF)) \
            * torch.expm1(-C2 * (dev_ / Tv + (nu0 - dev_) / Tr)) / torch.expm1(-C2 * nu0 / TREF)
    else:
        S = S * per_iso(lambda i: _q(i, TREF) / _q(i, T)) * torch.exp(-C2 * El * (1 / T - 1 / TREF)) \
            * torch.expm1(-C2 * nu0 / T) / torch.expm1(-C2 * nu0 / TREF)
    S = S * (x * (p * 1e5) / (KB * T) * 1e-6)
    nu = nu0 + t["delta"].double() * patm if "delta" in t else nu0
    dxG, dxL = _steps(case)
    aG, aL = _axis(wG, dxG), _axis(wL, dxL)
    k0, tv = _split((nu - wmin) / delta, nv + 1)
    clamp = nu >= wmin + (nv - 1) * delta
    k0, tv = torch.where(clamp, nv - 1, k0), torch.where(clamp, 0.0, tv)
    l0, tg = _split((wG.log() - math.log(aG[0])) / dxG, len(aG))
    m0, tl = _split((wL.log() - math.log(aL[0])) / dxL, len(aL))
    if case.get("option") == "min-RMS":
        a, pi, ln2 = wL / wG, math.pi, math.log(2.0)
        gg = 2 - 1 / (((6 * pi - 16) / (15 * pi - 32)) ** (1 / 1.5) + (2 * ln2 / 15) ** (1 / 1.5) * a ** (2 / 1.5)) ** 1.5
        lg = 1 / (((6 * pi - 16) / 3 * (ln2 / (2 * pi)) ** 0.5) ** (1 / 2.25) * a ** (1 / 2.25)
                  + (4 * ln2 * ln2 / 15) ** (1 / 2.25) * a ** (4 / 2.25)) ** 2.25
        qv, qg, ql = tv * (tv - 1), tg * (tg - 1), tl * (tl - 1)
        tg = tg + (8 * ln2 * qv * (ws / wG) ** 2 + gg * qg * dxG**2 - 2 * ln2 * a**2 * ql * dxL**2) / (2 * dxG)
        tl = tl + (lg * qg * dxG**2 + ql * dxL**2) / (2 * dxL)
    V, nl = nv + 1, len(aL)
    ldm = torch.zeros(len(aG) * nl * V, device=dev, dtype=torch.float64)
    for dl in (0, 1):
        for dm in (0, 1):
            w = S * (tg if dl else 1 - tg) * (tl if dm else 1 - tl)
            at = ((l0 + dl) * nl + m0 + dm) * V + k0
            ldm.scatter_add_(0, at, w * (1 - tv))
            ldm.scatter_add_(0, at + 1, w * tv)
    ldm = ldm.view(len(aG) * nl, V)
    L = 2 * nv
    f = torch.arange(L // 2 + 1, device=dev, dtype=torch.float64) / (L * ws)
    rev = f.flip(0)

    def ft(y, g, l):
        return torch.exp(-((math.pi * y * g) ** 2) / (4 * math.log(2.0)) - math.pi * y * l)

    acc = torch.zeros(L // 2 + 1, device=dev, dtype=torch.complex128)
    for a in range(len(aG)):
        for b in range(nl):
            v = ft(f, aG[a], aL[b])
            k = 1
            while math.exp(-((math.pi * k / (2 * ws) * aG[a]) ** 2) / (4 * math.log(2.0))
                           - math.pi * k / (2 * ws) * aL[b]) >= FOLD:
                v = v + ft(k / (2 * ws) + (rev if k & 1 else f), aG[a], aL[b])
                k += 1
            acc += torch.fft.rfft(ldm[a * nl + b], n=L) * (v / v[0])
    return torch.fft.irfft(acc, n=L)[:nv] / ws


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "slit":
        I, k = _spectrum_and_slit(case, seed)
        n, K = I.size, k.size
        m = n + K
        full = np.fft.irfft(np.fft.rfft(I.astype(np.float64), 2 * m) * np.fft.rfft(k.astype(np.float32), 2 * m), 2 * m)
        out = full[(K - 1) // 2:(K - 1) // 2 + n] * case["wstep"]
        if case["mode"] == "valid":
            la = min(n, K)
            a, b = (la - 1) // 2, la // 2
            out[:a] = np.nan
            out[n - b:] = np.nan
        return out
    cols = _lines(case, seed)
    if case["kind"] in ("batch", "serve"):
        return [_exact_abscoeff(case, c, cols, dev).cpu() for c in _conditions(case, seed)]
    A = _exact_abscoeff(case, case, cols, dev)
    if case["kind"] != "spectrum":
        return A.cpu()
    if case["option"] != "derived":
        return [A.cpu()]
    nv = A.numel()
    grid = case["wmin"] + torch.arange(nv, device=dev, dtype=torch.float64) * ((case["wmin"] + case["wstep"]) - case["wmin"])
    lam = 1.0 / grid * 1e7 * 1e-9
    planck = 2 * H * C**2 / lam**5 / torch.expm1(H * C / (lam * KB * case["T"])) * 1e-10
    em = -torch.expm1(-A * PATH)
    return {k: v.cpu() for k, v in dict(abscoeff=A, absorbance=A * PATH, emissivity=em, transmittance=1 - em,
                                       radiance=em * planck).items()}
