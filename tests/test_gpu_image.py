"""Half-length transforms (compiled passes at a period just above N_v, the
circular images corrected from tile moments) against the FP64 oracle at
RADIS's L = 2 N_v."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import engine, workloads

pytestmark = pytest.mark.gpu

# FP32 transforms of up to 2^19 points: 2 * 19 stages of 6e-8 on each of the
# two passes' sides add to about 2.5e-6 of peak at worst; the correction's own
# terms (ldm_job.h) are below 5e-7 of an image, itself below the peak
TOL = 5e-6


def _lines(n, lo, hi, seed, ends=False):
    rng = np.random.default_rng(seed)
    nu = np.sort(rng.uniform(lo, hi, n))
    S = 10.0 ** rng.uniform(-23.0, -20.0, n)
    if ends:  # the strongest lines at both ends: the nearest images are theirs
        S[:3] = S[-3:] = 1e-18
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    return workloads.LineList(nu0=nu, S_ref=f32(S), El=f32(rng.uniform(0.0, 3000.0, n)),
                              g_air=f32(rng.uniform(0.03, 0.08, n)), g_self=f32(rng.uniform(0.05, 0.10, n)),
                              n_air=f32(rng.uniform(0.5, 0.8, n)), molar_mass=np.array([0.0, 44.0]),
                              q_coef=(0.94, 1.1))


@pytest.fixture(scope="module")
def dev():
    d = engine.Device(0)
    yield d
    d.close()


# (grid points, wstep, p, T): the shortest and longest grids of a planned
# length (gaps from 2.6 % to 40 % of the grid), the smallest half-length
# split (256 x 64), halves of n2 (384 x 64 of 384 x 128), three- and
# five-fold n1, widths from a few to thousands of grid steps (wider than the
# gap), and a Gaussian of tens of steps
CASES = [
    (13_000, 0.001, 15.0, 900.0),
    (15_900, 0.001, 0.3, 2900.0),
    (20_001, 0.002, 10.0, 300.0),
    (23_100, 0.001, 1.0, 1500.0),
    (40_001, 0.01, 1.0, 700.0),
    (63_800, 0.0005, 20.0, 400.0),
    (64_100, 0.002, 3.0, 1000.0),
    (103_003, 0.001, 0.1, 3000.0),
    (159_600, 0.0002, 5.0, 2000.0),
    (191_009, 0.003, 1.0, 1100.0),
]


@pytest.mark.parametrize("ends", [False, True])
def test_half_length_transforms_match_radis_length(dev, ends):
    for k, (nv, ws, p, T) in enumerate(CASES):
        wmin = 2000.0
        wmax = wmin + (nv - 1.5) * ws
        lines = _lines(4000, wmin, wmax, 50 + k, ends)
        db = engine.LineDatabase(dev, lines)
        for dx in (0.2, 0.45):  # taller and shorter LDMs: odd and even numbers of rows and nodes
            # several at once: a lone small request keeps the whole length
            req = engine.make_request(db, wmin, wmax, ws, T, p, 0.3, dxG=dx, dxL=dx)
            b = engine.SpectrumBatch(db, [req] * (9 if nv < 30_000 else 5))
            res = b.results(b.run())
            got, inf = res[0], b.info(0)
            for other in res[1:]:
                np.testing.assert_array_equal(got, other)
            ref = oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, 0.3, dx, dx)
            err = oracle.rel_peak_error(got, ref)
            print(f"N_v={inf.n_v} L={inf.fft_len} {inf.n1}x{inf.n2} M={inf.n_g}x{inf.n_l} p={p} T={T} "
                  f"W={inf.tile_w}: {err:.2e}", flush=True)
            assert inf.compiled_fft == 1 and err <= TOL, (nv, ws, p, T, dx, err)
            b.close()
        db.close()


def test_conditions_change_on_one_layout(dev):
    """set_request over conditions from cold to hotter than the half-length
    rule's temperature (whole-length transforms from there on), and an empty
    window beside an ordinary one: each equal to the oracle."""
    lines = _lines(3000, 2000.0, 2040.0, 7)
    db = engine.LineDatabase(dev, lines)
    mk = lambda T, p, a=2000.0: engine.make_request(db, a, a + 40.0, 0.001, T, p, 0.3, dxG=0.3, dxL=0.3)  # noqa: E731
    b = engine.SpectrumBatch(db, [mk(300.0, 1.0), mk(300.0, 1.0, 2100.0)] + [mk(300.0, 1.0)] * 2)
    for T, p in [(300.0, 1.0), (3000.0, 18.0), (4.0e6, 2.0), (900.0, 0.2)]:
        b.set_request(0, mk(T, p))
        got = b.results(b.run())
        ref = oracle.eq_abscoeff(lines.as_dict(), 2000.0, 2040.0, 0.001, T, p, 0.3, 0.3, 0.3)
        assert oracle.rel_peak_error(got[0], ref) <= TOL, (T, p)
        assert not np.any(got[1])
    b.close()
    db.close()
