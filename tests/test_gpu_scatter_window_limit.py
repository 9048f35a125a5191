"""The 2-D fixed-point scatter with large bins and thousands of points per
subproblem, all of them on a few cells, against the float64 tile.

A tap is rounded to half a step of 2^-30 1.001 A cmax, A = n |y| at most, so
the n taps that a cell collects err by about sqrt(n / 3) 2^-31 n |y| cmax
against a sum of n |y| c: 2.5e-8 cmax / c for n = 8192, below 1e-6 for the
cells (c > cmax / 40) that carry the norm; the float products and the FFT add
a few 1e-7.
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phasing", ["real", "complex"])
@pytest.mark.parametrize("reps", [1, 2])
@pytest.mark.parametrize("bins", [(32, 16), (32, 32), (64, 64)])
@pytest.mark.parametrize("P", [4095, 4096, 8192, 20000])
def test_dense_cells_vs_float64(P, bins, reps, phasing):
    m = 8190 if P == 4095 else 8192 if P <= 8192 else 20000  # whole subproblems of P points
    Nd, Kd = (128, 128), (256, 256)
    lo, width = 2 * np.pi * 34.0 / 256, 2 * np.pi * 4.0 / 256
    om = lo + np.random.default_rng(P).uniform(0, 1, (m, 2)) * width
    A = NufftBase(Nd, om, Jd=6, Kd=Kd, Ld=256, phasing=phasing, n_shift=(64, 64), order="C",
                  device=torch.device("cuda", 0))
    A.set_binning(bins, P)
    assert A.plan_info()["fixed_point_scatter"]
    # the largest samples below a power of two
    y = torch.full((reps, m), 1 - 2.0 ** -24, dtype=torch.complex64, device="cuda")
    y = y[0] if reps == 1 else y
    got = A.adj(y).cpu().numpy()
    A.set_scatter("float64")
    assert rel_l2(got, A.adj(y).cpu().numpy()) <= 2e-6
