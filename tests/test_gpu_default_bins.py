"""Default 2-D bins: larger on large sparse grids, and the same transforms as
with 16x16 bins there (the sums differ by the order of float adds and by the
fixed-point steps, a few 1e-7; 1e-14 in double)."""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from mrrt.nufft_amd.batched import NufftFrames
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Kd,m,bins", [
    ((504, 512), 20000, (16, 16)),      # 1,008 bins' worth of cells
    ((512, 512), 16384, (16, 16)),      # few points
    ((512, 512), 16385, (32, 16)),
    ((512, 512), 100000, (16, 16)),     # 0.38 points per cell
    ((736, 720), 40000, (32, 32)),
    ((736, 720), 200000, (16, 16)),     # 0.38 points per cell
])
@pytest.mark.parametrize("precision,tol", [("single", 2e-6), ("double", 1e-13)])
def test_default_bins(Kd, m, bins, precision, tol):
    Nd = tuple(k // 2 for k in Kd)
    om = np.random.default_rng(0).uniform(-np.pi, np.pi, (m, 2))
    A = NufftBase(Nd, om, Jd=6, Kd=Kd, Ld=256, precision=precision, order="C", device=torch.device("cuda", 0))
    assert A.plan_info()["bin_size"][:2] == bins
    x = torch.from_numpy(trj.complex_gaussian(Nd, seed=1)).cuda().to(A._tcdt)
    y = torch.from_numpy(trj.complex_gaussian((m,), seed=2)).cuda().to(A._tcdt)
    yf, xa = A.fft(x).cpu().numpy(), A.adj(y).cpu().numpy()
    A.set_binning((16, 16), 384)
    assert rel_l2(yf, A.fft(x).cpu().numpy()) <= tol
    assert rel_l2(xa, A.adj(y).cpu().numpy()) <= tol


def test_default_bins_count_all_frames():
    om = [np.random.default_rng(f).uniform(-np.pi, np.pi, (3000, 2)) for f in range(8)]
    F = NufftFrames((128, 128), om, 2, Jd=6, Kd=(256, 256), Ld=256, device=torch.device("cuda", 0))
    assert F.op.plan_info()["bin_size"][:2] == (32, 32)
