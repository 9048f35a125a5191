"""Several repetitions, whose passes run in separate rows of workgroups, equal
the repetitions transformed one at a time.

The gather's sums are the same operations; the scatter's differ by the order
of its float adds on the grid, a few units of rounding (eps 6e-8, 1.1e-16)
of cell sums that a few tiles share: 1e-6 and 1e-14 leave a factor of ten.
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("single", 1e-6), ("double", 1e-14)])
@pytest.mark.parametrize("Nd,Kd,bins,P,reps", [
    ((300,), (600,), None, 0, 9),                  # more than one pass of eight
    ((40, 36), (80, 72), None, 0, 2),
    ((40, 36), (80, 72), (32, 32), 1024, 7),       # pairs and a last single repetition
    ((40, 36), (80, 72), None, 128, 5),            # the coefficient cache: one row
    ((20, 18, 16), (40, 36, 32), None, 0, 3),      # one repetition per pass
])
def test_passes_equal_single_repetitions(precision, tol, Nd, Kd, bins, P, reps):
    m = 3001
    om = np.random.default_rng(0).uniform(-np.pi, np.pi, (m, len(Nd)))
    A = NufftBase(Nd, om, Jd=5, Kd=Kd, Ld=256, precision=precision, order="C", device=torch.device("cuda", 0))
    if bins or P:
        A.set_binning(bins, P)
    x = torch.from_numpy(trj.complex_gaussian((reps,) + Nd, seed=1)).cuda().to(A._tcdt)
    y = torch.from_numpy(trj.complex_gaussian((reps, m), seed=2)).cuda().to(A._tcdt)
    yf, xa = A.fft(x).cpu().numpy(), A.adj(y).cpu().numpy()
    for r in range(reps):
        assert rel_l2(yf[r], A.fft(x[r].contiguous()).cpu().numpy()) <= tol
        assert rel_l2(xa[r], A.adj(y[r].contiguous()).cpu().numpy()) <= tol
