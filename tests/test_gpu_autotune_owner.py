"""The autotuner times the owner scatter where the tuned operator will run it."""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase, autotune

pytestmark = pytest.mark.gpu


def test_tune_times_the_owner_scatter():
    Kd, m = (256, 256), 2000
    om = np.random.default_rng(0).uniform(-np.pi, np.pi, (m, 2))
    A = NufftBase((128, 128), om, Jd=6, Kd=Kd, Ld=256, order="C", device=torch.device("cuda", 0))
    reps = (320 << 20) // (8 * 256 * 256) + 1  # grids beyond the size from which the path is taken
    A.set_kernel_timing(True, count_atomics=True)
    b, p, timings = autotune.tune(A, nreps=reps, cands=[((32, 32), 384, 256)], use_cache=False, reps=1)
    assert b == (32, 32) and len(timings) == 1
    assert A.read_flush_atomics() == 0  # no grid atomics: no bin is dense here
    # another workgroup size turns the path off, and is timed as it will run
    autotune.tune(A, nreps=reps, cands=[((32, 32), 384, 128)], use_cache=False, reps=1)
    assert A.read_flush_atomics() > 0
