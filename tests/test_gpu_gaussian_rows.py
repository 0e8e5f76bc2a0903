"""LDM rows of G-axis nodes that a fill tile's lines cannot reach are neither
written nor read: wide ranges of wavenumbers (up to a dozen nodes), several
isotopologues far apart in mass, lines clamped onto both ends of the grid,
row-grouped and run-time-sized transforms, against the FP64 oracle."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import engine, workloads

pytestmark = pytest.mark.gpu

# FP32 transforms of up to 2^19 points: 2 * 19 stages of 6e-8 on each of the
# two passes' sides
TOL = 5e-6


def _lines(lo, hi, n, seed, masses):
    rng = np.random.default_rng(seed)
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    iso = None if len(masses) == 2 else rng.integers(1, len(masses), n).astype(np.uint8)
    return workloads.LineList(nu0=np.sort(rng.uniform(lo, hi, n)), S_ref=f32(10.0 ** rng.uniform(-23.0, -20.0, n)),
                              El=f32(rng.uniform(0.0, 3000.0, n)), g_air=f32(rng.uniform(0.03, 0.08, n)),
                              g_self=f32(rng.uniform(0.05, 0.10, n)), n_air=f32(rng.uniform(0.5, 0.8, n)),
                              delta=f32(rng.uniform(-0.02, 0.02, n)) if iso is not None else None, iso=iso,
                              molar_mass=np.array(masses), q_coef=(0.94, 1.1))


# (lo, hi, wstep, p, T, dxG, dxL, masses, generic passes)
CASES = [
    (1000.0, 4000.0, 0.02, 2.0, 1500.0, 0.14, 0.2, [0.0, 18.0], False),
    (800.0, 7000.0, 0.05, 5.0, 2500.0, 0.14, 0.3, [0.0, 18.0], True),
    (1000.0, 3000.0, 0.02, 1.0, 900.0, 0.1, 0.2, [0.0, 2.0, 18.0, 44.0], False),
    (700.0, 5000.0, 0.1, 3.0, 700.0, 0.03, 0.08, [0.0, 18.0], False),  # 70 nodes: more than a wave's lanes, row groups
    (2000.0, 2600.0, 0.0015, 0.5, 1100.0, 0.137, 0.2, [0.0, 44.0], False),  # three nodes
]


def _oracle(d, wmin, wmax, ws, p, T, x, dxG, dxL):
    """abscoeff in FP64 from every line of the list (those outside the grid
    clamped onto its ends, as np.interp does)."""
    w = oracle.wavenumber_grid(wmin, wmax, ws)
    S, nu, wG, wL = oracle.line_parameters(d, T, p, x)
    aG, aL = oracle.init_w_axis(wG, dxG), oracle.init_w_axis(wL, dxL)
    ki0, ki1, tv = oracle.get_indices(nu, w)
    li0, li1, tG = oracle.get_indices(np.log(wG), np.log(aG))
    mi0, mi1, tL = oracle.get_indices(np.log(wL), np.log(aL))
    L = 2 * w.size
    ldm = oracle.ldm_scatter(L, aG.size, aL.size, ki0, ki1, tv, li0, li1, tG, mi0, mi1, tL, S)
    F = oracle.lineshape_templates(L, ws, aG, aL)
    return oracle.ldm_apply_fft(ldm, F, w.size, ws) * oracle.number_density(x, p, T)


@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_rows_of_distant_nodes(k, outside):
    lo, hi, ws, p, T, dxG, dxL, masses, generic = CASES[k]
    lines = _lines(lo, hi, 6000, 90 + k, masses)
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, lines)
    wmin, wmax, kw = lo, hi, {}
    if outside:  # lines on both sides of the grid
        wmin, wmax = lo + 0.2 * (hi - lo), hi - 0.3 * (hi - lo)
        kw = dict(line_window=(-np.inf, np.inf))
    b = engine.SpectrumBatch(db, [engine.make_request(db, wmin, wmax, ws, T, p, 0.3, dxG=dxG, dxL=dxL,
                                                      generic_fft=generic, **kw)])
    got = b.results(b.run())[0]
    inf, t = b.info(0), b.line_terms(0)
    assert inf.status == 0 and inf.n_g >= 3, (inf.status, inf.n_g)
    # the LDM that the passes see holds every corner of every line
    want = np.zeros((inf.n_g * inf.n_l, inf.n_v + 1))
    for dl in (0, 1):
        for dm in (0, 1):
            wt = t["I"].astype(np.float64) * (t["tg"] if dl else 1 - t["tg"]) * (t["tl"] if dm else 1 - t["tl"])
            r = (t["l0"] + dl) * inf.n_l + t["m0"] + dm
            np.add.at(want, (r, t["k0"]), wt * (1 - t["tv"]))
            np.add.at(want, (r, t["k0"] + 1), wt * t["tv"])
    # (FP32 products of three weights and one rounding per cell)
    assert np.max(np.abs(b.ldm(0) - want)) <= 1e-6 * want.max()
    ref = _oracle(lines.as_dict(), wmin, wmax, ws, p, T, 0.3, dxG, dxL)
    err = oracle.rel_peak_error(got, ref)
    print(f"case {k}: N_v={inf.n_v} M={inf.n_g}x{inf.n_l} W={inf.tile_w}: {err:.2e}", flush=True)
    assert err <= TOL
    b.close()
    db.close()
    dev.close()
