"""The autotuner times the dispatch it installs, and tunes again when the
kernels behind a stored choice have changed (no GPU: a recorded operator)."""

import json

import pytest
import torch

from mrrt.nufft_amd import autotune


class _Lib(object):
    def __init__(self, op):
        self.op = op

    def mi355nufft_abi_version(self):
        return 2

    def mi355nufft_interp(self, *a):
        self.op.timed.append(("interp", self.op.mode))
        return 0

    def mi355nufft_spread(self, *a):
        self.op.timed.append(("spread", self.op.mode))
        return 0


class _Op(object):
    """Records the binning mode of every launch; two frames, so that no FFT is tuned."""
    ndim, Nd, Kd, Jd, Ld = 2, (8, 8), (16, 16), (6, 6), 64
    precision, phasing, nframes, M = "single", "real", 2, 10
    _tcdt, device = torch.complex64, torch.device("cpu")
    _plan = None

    def __init__(self):
        self._lib = _Lib(self)
        self.timed, self.mode = [], None

    def plan_info(self):
        return {"fixed_point_scatter": True}

    def set_binning(self, b, p, mode, th):
        if b == (99, 99) and mode != "auto":  # a tile beyond the LDS: "auto" would run other kernels
            raise ValueError("tile exceeds the LDS budget")
        self.mode = mode

    def set_fft(self, m):
        pass

    def _sync_stream(self):
        pass


@pytest.fixture
def op(tmp_path, monkeypatch):
    monkeypatch.setenv("MI355NUFFT_TUNE_CACHE", str(tmp_path / "tune.json"))
    op = _Op()
    monkeypatch.setattr(autotune._lib, "get_lib", lambda: op._lib)
    monkeypatch.setattr(autotune._lib, "check", lambda rc: None)

    def run(fn, reps):
        fn()
        return 1.0
    monkeypatch.setattr(autotune, "_time", run)
    return op


CANDS = [((16, 16), 256, 256), ((99, 99), 256, 256), ((32, 32), 256, 256)]


def test_candidates_are_timed_under_the_installed_dispatch(op):
    b, p, timings = autotune.tune(op, nreps=1, cands=CANDS)
    # "tiled" and "auto" choose the same kernels for a tile that fits; "tiled" refuses the others
    assert op.timed and {m for _, m in op.timed} == {"tiled"}
    assert op.mode == "auto" and len(timings) == 2 and (b, p) == ((16, 16), 256)


def test_choices_of_other_kernels_are_tuned_again(op):
    autotune.tune(op, nreps=1, cands=CANDS)
    path = autotune.cache_path()
    (key, entry), = json.load(open(path)).items()
    first = len(op.timed)
    autotune.tune(op, nreps=1, cands=CANDS)
    assert len(op.timed) == first  # from the cache
    # an entry of the same library interface, stored before the kernels had a revision
    old = "|".join(str(v) for v in (2, op.ndim, op.Nd, op.Kd, op.Jd, op.Ld, op.precision, op.phasing, 8, 1, 2, 1))
    assert key != old
    json.dump({old: entry}, open(path, "w"))
    autotune.tune(op, nreps=1, cands=CANDS)
    assert len(op.timed) == 2 * first


@pytest.mark.parametrize("bins,P", [((16, 16), 384), ((32, 16), 384), ((32, 32), 384), ((32, 16), 256), ((32, 32), 256)])
def test_candidates_hold_the_2d_defaults(bins, P):
    """A tuned plan is no slower than an untuned one."""
    assert (bins, P, 256) in autotune.candidates(2)
