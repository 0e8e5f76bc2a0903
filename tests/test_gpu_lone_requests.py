"""Lone requests, whose launches leave most of the chip idle: narrow pass A and C
tiles, several pass B shares at the whole length (dropped where a budget leaves
no room for them), narrow fill tiles, with and without derived quantities,
against the FP64 oracle."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import engine, workloads

pytestmark = pytest.mark.gpu

# FP32 transforms of up to 2^18 points: 2 * 18 stages of 6e-8 on each of the
# two passes' sides
TOL = 5e-6

# grid points: whole length 256 x 64, 320 x 64, 384 x 128, 512 x 256; half length
# 320 x 512, 384 x 128, 512 x 512
POINTS = [4_000, 9_000, 20_001, 50_001, 150_001, 23_000, 240_000]


def _lines(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    return workloads.LineList(nu0=np.sort(rng.uniform(lo, hi, n)), S_ref=f32(10.0 ** rng.uniform(-23.0, -20.0, n)),
                              El=f32(rng.uniform(0.0, 3000.0, n)), g_air=f32(rng.uniform(0.03, 0.08, n)),
                              g_self=f32(rng.uniform(0.05, 0.10, n)), n_air=f32(rng.uniform(0.5, 0.8, n)),
                              molar_mass=np.array([0.0, 44.0]), q_coef=(0.94, 1.1))


@pytest.mark.parametrize("nv", POINTS)
def test_lone_request_and_derived(nv):
    ws, wmin, T, p, x, path = 0.002, 2000.0, 900.0, 1.3, 0.3, 5.0
    wmax = wmin + (nv - 1.5) * ws
    lines = _lines(3000, wmin, wmax, nv)
    ref = oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, x, 0.2, 0.2)
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, lines)
    req = engine.make_request(db, wmin, wmax, ws, T, p, x, dxG=0.2, dxL=0.2)
    b = engine.SpectrumBatch(db, [req])
    plain = b.results(b.run())[0]
    err = oracle.rel_peak_error(plain, ref)
    inf, full = b.info(0), b.workspace_bytes()
    print(f"N_v={nv} L={inf.fft_len} {inf.n1}x{inf.n2} M={inf.n_g}x{inf.n_l} W={inf.tile_w}: {err:.2e}", flush=True)
    assert err <= TOL
    out = b.set_derived(0, path)
    again = b.results(b.run())[0]
    np.testing.assert_array_equal(again, plain)
    w = oracle.wavenumber_grid(wmin, wmax, ws)
    want = oracle.derived_quantities(w, plain, path, T)
    for name in ("emissivity", "transmittance", "radiance"):
        got = out[name].double().cpu().numpy()
        # the device derives them in FP64 from the abscoeff it stores: FP32 rounding only
        assert np.max(np.abs(got - want[name])) <= 2e-7 * np.max(np.abs(want[name])), name
    b.close()
    # a budget that the further shares (a third to the fourth spectrum) do not fit
    used = dev.bytes_in_use() if hasattr(dev, "bytes_in_use") else None
    if used is not None:
        dev.set_budget(used + full - int(inf.fft_len) * 8)
        try:
            b = engine.SpectrumBatch(db, [req])
        except Exception:  # refused with two shares as well: no room before either
            b = None
        if b is not None:
            assert b.workspace_bytes() < full
            assert oracle.rel_peak_error(b.results(b.run())[0], ref) <= TOL
            b.close()
    db.close()
    dev.close()
