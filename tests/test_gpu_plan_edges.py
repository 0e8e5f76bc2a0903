"""Edges of request planning through the library's entry points."""
import numpy as np
import pytest

from oracle import ldm_oracle as oracle
from radis_amd import _native, engine, workloads

pytestmark = pytest.mark.gpu

# FP32 transforms of up to 2^19 points: 2 * 19 stages of 6e-8 on each of the
# two passes' sides
TOL = 5e-6


def _lines(n, lo, hi, seed):
    rng = np.random.default_rng(seed)
    f32 = lambda a: np.ascontiguousarray(a, dtype=np.float32)  # noqa: E731
    return workloads.LineList(nu0=np.sort(rng.uniform(lo, hi, n)), S_ref=f32(10.0 ** rng.uniform(-23.0, -20.0, n)),
                              El=f32(rng.uniform(0.0, 3000.0, n)), g_air=f32(rng.uniform(0.03, 0.08, n)),
                              g_self=f32(rng.uniform(0.05, 0.10, n)), n_air=f32(rng.uniform(0.5, 0.8, n)),
                              molar_mass=np.array([0.0, 44.0]), q_coef=(0.94, 1.1))


@pytest.fixture(scope="module")
def dev():
    d = engine.Device(0)
    yield d
    d.close()


def test_tile_too_wide_for_two_rows_is_an_error(dev):
    """Refused with ERANGE by every entry point that plans, alone and beside a
    request that plans."""
    import torch

    db = engine.LineDatabase(dev, _lines(2000, 2000.0, 2040.0, 3))
    mk = lambda w: engine.make_request(db, 2000.0, 2040.0, 0.002, 900.0, 1.3, 0.3, dxG=0.2, dxL=0.2, tile_w=w)  # noqa: E731
    out = torch.empty(20001, dtype=torch.float32, device="cuda")
    for call in (lambda: db.request_bytes(mk(4096)), lambda: engine.SpectrumBatch(db, [mk(4096)]),
                 lambda: engine.SpectrumBatch(db, [mk(0), mk(4096)]), lambda: engine.run_noalloc(db, mk(4096), out)):
        with pytest.raises(_native.LdmError, match="does not fit two LDM rows"):
            call()
    b = engine.SpectrumBatch(db, [mk(2048)])
    ref = oracle.eq_abscoeff(_lines(2000, 2000.0, 2040.0, 3).as_dict(), 2000.0, 2040.0, 0.002, 900.0, 1.3, 0.3, 0.2, 0.2)
    assert oracle.rel_peak_error(b.results(b.run())[0], ref) <= TOL
    b.close()
    db.close()


def test_ldm_copy_after_the_workspace_grew(dev):
    """The LDM of the last run goes with its workspace: an error until the
    next run, which fills it again."""
    db = engine.LineDatabase(dev, _lines(2000, 2000.0, 2040.0, 5))
    mk = lambda dx: engine.make_request(db, 2000.0, 2040.0, 0.002, 900.0, 1.3, 0.3, dxG=dx, dxL=dx)  # noqa: E731
    b = engine.SpectrumBatch(db, [mk(0.45)])
    b.run()
    assert b.ldm(0).max() > 0
    rows = int(b.info(0).m_cap)
    b.set_request(0, mk(0.05))
    assert b.info(0).m_cap > rows
    with pytest.raises(_native.LdmError, match="run it first"):
        b.ldm(0)
    b.run()
    ldm = b.ldm(0)
    assert ldm.shape[0] > rows and np.all(np.isfinite(ldm)) and ldm.max() > 0
    b.close()
    db.close()
