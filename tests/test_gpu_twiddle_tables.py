"""A batch whose requests share a transform length but not the kind of its W_L
table: compiled passes (FP64 table) beside run-time-sized ones (FP32)."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import engine, workloads

pytestmark = pytest.mark.gpu

# up to 34 butterfly stages there and back, 3e-8 rms each, five times that at the
# worst of 10^5 outputs
TOL = 1e-6


@pytest.mark.parametrize("nv", [30_000, 60_001])
def test_one_length_both_kinds_of_passes(nv):
    rng = np.random.default_rng(nv)
    ws, wmin, T, p, dx, n = 0.002, 2000.0, 900.0, 1.3, 0.1, 3000
    wmax = wmin + (nv - 1.5) * ws
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    lines = workloads.LineList(nu0=np.sort(rng.uniform(wmin, wmax, n)), S_ref=f32(10.0 ** rng.uniform(-23.0, -20.0, n)),
                               El=f32(rng.uniform(0.0, 3000.0, n)), g_air=f32(rng.uniform(0.03, 0.08, n)),
                               g_self=f32(rng.uniform(0.05, 0.10, n)), n_air=f32(rng.uniform(0.5, 0.8, n)),
                               molar_mass=np.array([0.0, 44.0]), q_coef=(0.94, 1.1))
    dev = engine.Device(0)
    db = engine.LineDatabase(dev, lines)
    mk = lambda **k: engine.make_request(db, wmin, wmax, ws, T, p, 0.3, dxG=dx, dxL=dx, **k)  # noqa: E731
    L = int(db.request_bytes(mk(period_fft_len=True))[1].fft_len)
    b = engine.SpectrumBatch(db, [mk(fft_len=L, period_fft_len=True), mk(fft_len=L, period_fft_len=True, generic_fft=True),
                                  mk()])
    got = b.results(b.run())
    assert [int(b.info(i).compiled_fft) for i in range(3)] == [1, 0, 1]
    assert b.pass_length(0)[0] == b.pass_length(1)[0] == L
    ref = oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, 0.3, dx, dx, L=L)
    assert oracle.rel_peak_error(got[0], ref) <= TOL and oracle.rel_peak_error(got[1], ref) <= TOL
    assert oracle.rel_peak_error(got[2], oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, 0.3, dx, dx)) <= TOL
    b.close()
    db.close()
    dev.close()
