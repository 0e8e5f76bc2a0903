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


def test_conditions_that_end_the_half_length_keep_graph_and_ldm(dev):
    """set_request to min-RMS weights and to a temperature that the
    half-length passes do not take: the LDM of the last run stays readable,
    and the C entry's replays of the captured graph go on (no capture by the
    caller), with eager runs between them."""
    lines = _lines(3000, 2000.0, 2040.0, 7)
    db = engine.LineDatabase(dev, lines)
    mk = lambda T, p, opt="simple": engine.make_request(db, 2000.0, 2040.0, 0.001, T, p, 0.3, dxG=0.3, dxL=0.3,  # noqa: E731
                                                        optimization=opt)
    ref = {}
    for T, p, opt in [(900.0, 1.0, "simple"), (900.0, 1.0, "min-RMS"), (4.0e6, 2.0, "simple"), (300.0, 1.5, "simple")]:
        ref[T, p, opt] = oracle.eq_abscoeff(lines.as_dict(), 2000.0, 2040.0, 0.001, T, p, 0.3, 0.3, 0.3,
                                            optimization=opt)
    for first in ("min-RMS", "hot"):
        change = (900.0, 1.0, "min-RMS") if first == "min-RMS" else (4.0e6, 2.0, "simple")
        # (neighbouring rows hold tens of times a line with opposite signs: the parity bound)
        tol = 1e-4 if first == "min-RMS" else TOL
        rows = [mk(4.0e6, 2.0)] * 4  # row capacity for every condition
        b = engine.SpectrumBatch(db, [mk(900.0, 1.0)] * 4)
        for i, r in enumerate(rows):
            b.set_request(i, r)  # (grows the workspace before the capture)
            b.set_request(i, mk(900.0, 1.0))
        outs = b.capture()
        replay = lambda: b._lib.radis_ldm_batch_graph_replay(b._h, engine._stream_handle(None))  # noqa: E731
        assert replay() == 0
        assert oracle.rel_peak_error(b.results(outs)[1], ref[900.0, 1.0, "simple"]) <= TOL
        ldm = b.ldm(1)
        b.set_request(1, mk(*change))
        np.testing.assert_array_equal(b.ldm(1), ldm)
        for k in range(3):
            assert replay() == 0
            got = b.results(outs)
            assert oracle.rel_peak_error(got[1], ref[change]) <= tol, (first, k)
            assert oracle.rel_peak_error(got[0], ref[900.0, 1.0, "simple"]) <= TOL, (first, k)
            eager = b.results(b.run())
            assert oracle.rel_peak_error(eager[1], ref[change]) <= tol, (first, k)
        b.set_request(1, mk(300.0, 1.5))
        for k in range(2):
            assert replay() == 0
            assert oracle.rel_peak_error(b.results(outs)[1], ref[300.0, 1.5, "simple"]) <= TOL, (first, k)
        b.close()
    db.close()


def test_batch_after_a_layout_that_did_not_fit(dev):
    """A growth refused by the budget leaves no buffers: runs report the error
    (nothing is launched) until the budget allows the layout."""
    lines = _lines(2000, 2000.0, 2040.0, 9)
    db = engine.LineDatabase(dev, lines)
    mk = lambda dx: engine.make_request(db, 2000.0, 2040.0, 0.002, 900.0, 1.3, 0.3, dxG=dx, dxL=dx)  # noqa: E731
    b = engine.SpectrumBatch(db, [mk(0.45)])
    b.run()
    dev.set_budget(dev.bytes_in_use())
    try:
        with pytest.raises(_native.BudgetExceeded):
            b.set_request(0, mk(0.05))
        for _ in range(2):
            with pytest.raises(_native.BudgetExceeded):
                b.run()
    finally:
        dev.set_budget(0)
    ref = oracle.eq_abscoeff(lines.as_dict(), 2000.0, 2040.0, 0.002, 900.0, 1.3, 0.3, 0.05, 0.05)
    assert oracle.rel_peak_error(b.results(b.run())[0], ref) <= TOL
    b.close()
    db.close()


@pytest.mark.parametrize("nv", [4_000, 9_000, 20_001, 50_001, 150_001])
def test_noalloc_with_several_pass_b_shares(dev, nv):
    """The scratch array's lone requests split a whole-length transform's pairs
    over up to four pass B workgroups per row block."""
    import torch

    ws, wmin, T, p, x = 0.002, 2000.0, 900.0, 1.3, 0.3
    wmax = wmin + (nv - 1.5) * ws
    lines = _lines(3000, wmin, wmax, nv)
    db = engine.LineDatabase(dev, lines)
    for dx in (0.1, 0.2):
        for opt, tol in (("simple", TOL), ("min-RMS", 1e-4)):
            out = torch.full((nv,), float("nan"), dtype=torch.float32, device="cuda")
            res = torch.zeros(48, dtype=torch.uint8, device="cuda")
            req = engine.make_request(db, wmin, wmax, ws, T, p, x, dxG=dx, dxL=dx, optimization=opt)
            inf = engine.run_noalloc(db, req, out, res)
            assert engine.read_result(res).status == 0
            ref = oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, x, dx, dx, optimization=opt)
            err = oracle.rel_peak_error(np.ldexp(out.double().cpu().numpy(), inf.scale_log2), ref)
            print(f"N_v={nv} L={inf.fft_len} {inf.n1}x{inf.n2} rows={inf.m_cap} {opt}: {err:.2e}", flush=True)
            assert err <= tol
    db.close()


@pytest.mark.parametrize("nv", [4_000, 9_000, 20_001, 50_001, 150_001])
def test_partial_spectra_in_y(dev, nv):
    """A batch's lone whole-length request keeps pass B's partial spectra in Y:
    as many pairs as planned, and so few (after set_request) that shares have
    none."""
    ws, wmin, T, p, x = 0.002, 2000.0, 900.0, 1.3, 0.3
    wmax = wmin + (nv - 1.5) * ws
    lines = _lines(3000, wmin, wmax, nv)
    db = engine.LineDatabase(dev, lines)
    mk = lambda dx: engine.make_request(db, wmin, wmax, ws, T, p, x, dxG=dx, dxL=dx, period_fft_len=True)  # noqa: E731
    b = engine.SpectrumBatch(db, [mk(0.1)])
    assert b.workspace_bytes() <= db.request_bytes(mk(0.1))[0]
    for dx in (0.1, 3.0, 1.0, 0.5, 0.3, 0.2, 0.1):
        b.set_request(0, mk(dx))
        for k in range(2):
            got = b.results(b.run())[0]
            inf = b.info(0)
            ref = oracle.eq_abscoeff(lines.as_dict(), wmin, wmax, ws, T, p, x, dx, dx, L=int(inf.fft_len))
            err = oracle.rel_peak_error(got, ref)
            print(f"N_v={nv} dx={dx} M={inf.n_g}x{inf.n_l} of {inf.m_cap}: {err:.2e}", flush=True)
            assert err <= TOL
    b.close()
    db.close()
