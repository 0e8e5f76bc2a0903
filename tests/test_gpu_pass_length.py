"""The length the FFT passes run at is the one planned for the request (half
of fft_len, or all of it), and the spectrum is RADIS's at L = 2 N_v either way:
strong lines at both ends of the grid, whose nearest images are the largest,
gaps from 2.7 % of the grid up."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import engine, workloads

pytestmark = pytest.mark.gpu

# Up to 36 butterfly stages there and back, rounding 3e-8 rms each: 1.8e-7 of the
# spectrum's rms in quadrature, five times that at the worst of 10^5 outputs; the
# image correction's own terms are below 1e-7 of an image
TOL = 1e-6


def _lines(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    S = 10.0 ** rng.uniform(-23.0, -20.0, n)
    S[:3] = S[-3:] = 1e-18
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    return workloads.LineList(nu0=np.sort(rng.uniform(lo, hi, n)), S_ref=f32(S), El=f32(rng.uniform(0.0, 3000.0, n)),
                              g_air=f32(rng.uniform(0.03, 0.08, n)), g_self=f32(rng.uniform(0.05, 0.10, n)),
                              n_air=f32(rng.uniform(0.5, 0.8, n)), molar_mass=np.array([0.0, 44.0]), q_coef=(0.94, 1.1))


# grid points, wstep, p, T, LDM steps, requests in the batch, half the length
CASES = [
    (40_001, 0.01, 1.0, 700.0, 0.2, 1, True),
    (40_001, 0.01, 1.0, 700.0, 0.45, 1, False),  # few points: the whole length is as fast
    (64_100, 0.002, 3.0, 1000.0, 0.45, 1, True),
    (64_100, 0.002, 3.0, 1000.0, 0.03, 5, True),
    (103_003, 0.001, 0.1, 3000.0, 0.06, 5, True),
    (63_800, 0.0005, 20.0, 400.0, 0.2, 5, False),  # a short gap
    (127_500, 0.001, 3.0, 1000.0, 0.2, 1, True),  # the same, but one request leaves the chip idle
    (127_500, 0.001, 3.0, 1000.0, 0.2, 5, False),
    (127_500, 0.001, 3.0, 1000.0, 0.06, 5, True),
    (159_600, 0.0002, 5.0, 2000.0, 0.2, 1, True),
    (191_009, 0.003, 1.0, 1100.0, 0.2, 5, True),
    (255_000, 0.001, 2.0, 1200.0, 0.06, 1, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_passes_run_at_the_planned_length(case):
    nv, ws, p, T, dx, count, half = case
    wmin = 2000.0
    wmax = wmin + (nv - 1.5) * ws
    lines = _lines(4000, wmin, wmax, nv)
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, lines)
    mk = lambda **k: engine.make_request(db, wmin, wmax, ws, T, p, 0.3, dxG=dx, dxL=dx, **k)  # noqa: E731
    b = engine.SpectrumBatch(db, [mk()] * count)
    res = b.results(b.run())
    inf = b.info(0)
    length, shares = b.pass_length(0)
    assert length == (inf.fft_len // 2 if half else inf.fft_len) and 1 <= shares <= 4
    err = oracle.rel_peak_error(res[0], oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, 0.3, dx, dx))
    print(f"N_v={nv} L={inf.fft_len} runs {length}, {shares} shares, W={inf.tile_w}: {err:.2e}", flush=True)
    assert err <= TOL
    for other in res[1:]:
        np.testing.assert_array_equal(res[0], other)
    # never for min-RMS weights or a period of the caller's
    for kw in (dict(optimization="min-RMS"), dict(period_fft_len=True), dict(generic_fft=True)):
        c = engine.SpectrumBatch(db, [mk(**kw)] * count)
        assert c.pass_length(0)[0] == c.info(0).fft_len
        c.close()
    b.close()
    db.close()
    dev.close()


@pytest.mark.parametrize("nv", [4_000, 9_000, 20_001, 50_001, 150_001])
def test_a_budget_of_request_bytes_is_enough(nv):
    """A lone request with several pass B shares is laid out, and computed,
    within the bytes that admission counts for it."""
    ws, wmin, T, p, dx = 0.002, 2000.0, 900.0, 1.3, 0.1
    wmax = wmin + (nv - 1.5) * ws
    lines = _lines(3000, wmin, wmax, nv)
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, lines)
    for kw in ({}, dict(period_fft_len=True)):
        req = engine.make_request(db, wmin, wmax, ws, T, p, 0.3, dxG=dx, dxL=dx, **kw)
        dev.set_budget(dev.bytes_in_use() + db.request_bytes(req)[0])
        b = engine.SpectrumBatch(db, [req])
        got = b.results(b.run())[0]
        length, shares = b.pass_length(0)
        # (run-time-sized passes walk every pair in one workgroup)
        assert (shares > 2 if b.info(0).compiled_fft else shares == 1) and (length == b.info(0).fft_len or not kw)
        L = int(b.info(0).fft_len) if kw else None
        assert oracle.rel_peak_error(got, oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, 0.3, dx, dx, L=L)) <= TOL
        b.close()
        dev.set_budget(0)
    db.close()
    dev.close()
