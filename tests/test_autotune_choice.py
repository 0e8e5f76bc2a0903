"""The autotuner's choice, on made-up stage times (CPU): the schedule with the
least time in all, whatever stage it falls in, and keys that separate what runs
differently."""
import types

import pytest

from radis_amd import _native, autotune, engine


class _Db:
    """Plans every request at 40,001 points, 16 rows."""

    def request_bytes(self, req):
        return 1 << 20, types.SimpleNamespace(n_v=40_001, fft_len=98_304, n1=384, m_cap=16, tile_w=128, compiled_fft=1)


def _batch(stage_ms):
    class Batch:
        def __init__(self, db, reqs):
            self.req = reqs[0]

        def alloc_outputs(self):
            return []

        def run(self, outs):
            pass

        def enable_timing(self, on):
            pass

        def stage_ms(self):
            return stage_ms(self.req)

        def info(self, i):
            return types.SimpleNamespace(compiled_fft=0 if self.req.flags & _native.GENERIC_FFT else 1)

        def close(self):
            pass

    return Batch


@pytest.fixture
def cache(tmp_path, monkeypatch):
    monkeypatch.setenv("RADIS_AMD_TUNE_CACHE", str(tmp_path / "tune.json"))


def test_tile_width_by_the_whole_step(cache, monkeypatch):
    """A wide tile fills fastest, but the passes then run at the whole length."""

    def stage_ms(req):
        wide = req.tile_w > 128
        st = dict.fromkeys(_native.STAGE_NAMES, 0.0)
        st.update(axis=0.010, finalize=0.006, fill=0.012 if wide else 0.015, fft_a=0.020 if wide else 0.010,
                  fft_b=0.020 if wide else 0.012, fft_c=0.006)
        if req.tile_w < 128:
            st["fill"] += 0.003
        return st

    monkeypatch.setattr(engine, "SpectrumBatch", _batch(stage_ms))
    e = autotune.tune(_Db(), _native.Request(), reps=3)
    assert e["tile_w"] == 128
    assert e["fill_ms"] == pytest.approx(0.015) and e["fft_ms"] == pytest.approx(0.028)


def test_fft_schedule_by_the_whole_step(cache, monkeypatch):
    """The split with the fastest passes, but a fill and an axis launch (the
    tile bounds are in it) that cost more than it saves."""

    def stage_ms(req):
        st = dict.fromkeys(_native.STAGE_NAMES, 0.0)
        quick = req.fft_n1 == 512
        st.update(axis=0.012 if quick else 0.010, finalize=0.006, fill=0.030 if quick else 0.015,
                  fft_a=0.008 if quick else 0.010, fft_b=0.008 if quick else 0.010, fft_c=0.006)
        if req.flags & _native.GENERIC_FFT:
            st["fft_b"] = 1.0
        return st

    monkeypatch.setattr(engine, "SpectrumBatch", _batch(stage_ms))
    e = autotune.tune(_Db(), _native.Request(), reps=3)
    assert e["fft_n1"] != 512 and not e["generic"]


def test_planner_schedule_unless_another_is_clearly_faster(cache, monkeypatch):
    """Within the spread between runs the planner's tile and split stay."""

    def stage_ms(req):
        st = dict.fromkeys(_native.STAGE_NAMES, 0.0)
        st.update(axis=0.010, finalize=0.006, fill=0.0495 if req.tile_w == 64 else 0.050,
                  fft_a=0.0195 if req.fft_n1 == 1024 else 0.020, fft_b=0.020, fft_c=0.006)
        return st

    monkeypatch.setattr(engine, "SpectrumBatch", _batch(stage_ms))
    e = autotune.tune(_Db(), _native.Request(), reps=3)
    assert (e["tile_w"], e["fft_len"], e["fft_n1"], e["generic"]) == (128, 98_304, 384, False)


def test_keys_separate_the_weights_and_the_schedules_of_other_builds(cache):
    """min-RMS requests run other passes than simple ones of the same size;
    entries timed on other kernels (keys without a schedule number) are not
    applied."""
    db, a, b = _Db(), _native.Request(), _native.Request()
    b.flags = _native.MIN_RMS
    assert autotune.key_of(db, a) != autotune.key_of(db, b)
    old = f"L=98304/mcap=16/dxG={a.dxG:.6g}/dxL={a.dxL:.6g}"
    autotune._load()[old] = {"fft_len": 98304, "fft_n1": 384, "generic": False, "tile_w": 512}
    assert autotune.lookup(db, a) is None and not autotune.apply(db, a)
    assert a.tile_w == 0
