"""3-D scatter of subproblems around multiples of the workgroup's 256 threads
and of the six samples each thread keeps in flight, against the oracle.

All points lie in one bin, so the counts are those of its subproblems (at most
3,072 points each).  Held to the parity bar of complex64 (1e-5).
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from oracle import nufft_oracle as O
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J,phasing,reps", [(5, "real", 1), (6, "complex", 1), (7, "real", 1), (6, "real", 2)])
@pytest.mark.parametrize("M", [1, 2, 255, 256, 257, 512, 513, 1535, 1536, 1537, 3072, 3073, 3585])
def test_adjoint_vs_oracle(M, J, phasing, reps):
    Nd, Kd = (20, 18, 16), (40, 36, 32)
    lo = 2 * np.pi * np.array([17.0 / 40, 17.0 / 36, 17.0 / 32])
    om = lo + np.random.default_rng(M).uniform(0, 1, (M, 3)) * 2 * np.pi * np.array([9.0 / 40, 9.0 / 36, 9.0 / 32])
    kw = dict(Jd=J, Kd=Kd, Ld=256, precision="single", phasing=phasing, n_shift=np.asarray(Nd) / 2)
    A, B = NufftBase(Nd, om, device=torch.device("cuda", 0), **kw), O.NufftOracle(Nd, om, **kw)
    y = trj.complex_gaussian((M, reps), seed=3)
    assert rel_l2(A.adj(y), B.adj(y)) <= 1e-5
