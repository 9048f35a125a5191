"""Default 2-D bins of sparse k-space by mode, and transforms that equal those
with 16x16 bins (float sums in another order and other fixed-point steps: a
few 1e-7, 1e-14 in double)."""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from mrrt.nufft_amd.autograd import nufft
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


def _op(Kd, m, precision="single", **kw):
    om = np.random.default_rng(0).uniform(-np.pi, np.pi, (m, 2))
    return NufftBase(tuple(k // 2 for k in Kd), om, Jd=6, Kd=Kd, Ld=256, precision=precision, order="C",
                     device=torch.device("cuda", 0), **kw)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("Kd", [(512, 512), (736, 720)])
def test_sparse_matrix_rows_keep_16x16(Kd, precision):
    A = _op(Kd, 40000, precision, mode="sparse")
    assert A.plan_info()["bin_size"][:2] == (16, 16)


@pytest.mark.parametrize("J", [4, 5, 6, 7])  # two 32x32 tiles at a time for J = 4 to 6 and four coils or more
@pytest.mark.parametrize("reps", [3, 4, 5])
def test_double_gather_and_gradient_of_several_coils(J, reps):
    om = torch.from_numpy(np.random.default_rng(0).uniform(-np.pi, np.pi, (60000, 2))).cuda()
    A = NufftBase((368, 360), om, Jd=J, Kd=(736, 720), Ld=256, precision="double", order="C", device=om.device)
    x = torch.from_numpy(trj.complex_gaussian((reps, 368, 360), seed=1)).cuda()
    w = torch.from_numpy(trj.complex_gaussian((reps, 60000), seed=2)).cuda()
    got = []
    for bins in ((32, 32), (16, 16)):
        if bins == (16, 16):
            A.set_binning(bins, 384)
        o = om.clone().requires_grad_(True)
        y = nufft(A, x, o)
        assert A.plan_info()["bin_size"][:2] == bins
        got.append((y.detach().cpu().numpy(), torch.autograd.grad(y, (o,), w)[0].cpu().numpy()))
    for u, v in zip(*got):
        assert rel_l2(u, v) <= 1e-13


@pytest.mark.parametrize("m,P", [(16385, 256), (32768, 256), (32769, 384)])
@pytest.mark.parametrize("precision,tol", [("single", 2e-6), ("double", 1e-13)])
@pytest.mark.parametrize("J", [5, 7])
def test_few_points_have_one_per_thread(m, P, precision, tol, J):
    """Radial spokes, whose centre bins hold several subproblems, with one
    image and a pair and a half, against 16x16 bins."""
    om = trj.golden_angle_2d(-(-m // 256), 256)[:m]
    A = NufftBase((256, 256), om, Jd=J, Kd=(512, 512), Ld=256, precision=precision, order="C",
                  device=torch.device("cuda", 0))
    info = A.plan_info()
    assert info["bin_size"][:2] == (32, 16) and info["max_points"] == P
    for reps in (1, 3):
        x = torch.from_numpy(trj.complex_gaussian((reps, 256, 256), seed=1)).cuda().to(A._tcdt)
        y = torch.from_numpy(trj.complex_gaussian((reps, m), seed=2)).cuda().to(A._tcdt)
        A.set_binning()
        yf, xa = A.fft(x).cpu().numpy(), A.adj(y).cpu().numpy()
        A.set_binning((16, 16), 384)
        assert rel_l2(yf, A.fft(x).cpu().numpy()) <= tol
        assert rel_l2(xa, A.adj(y).cpu().numpy()) <= tol


@pytest.mark.parametrize("reps,two_phase", [(850, True), (1000, False)])
def test_two_phase_budget_counts_16x16_slots(reps, two_phase):
    """180,000 points on Kd 736 x 720: the slots of one repetition take 8.96 MB
    with 16x16 bins (850 repetitions 7.1 GiB, 1,000 8.3) and 10.9 MB with the
    default 32x32 (8.7 and 10.2).  Beyond 8 GiB the scatter adds atomically, not
    reproducibly."""
    A = _op((736, 720), 180000)
    A.set_binning(method="tiled_two_phase")
    info = A.plan_info()
    assert info["bin_size"][:2] == (32, 32)
    assert info["subproblem_slots"] * info["tile"] * 8 * 850 > 8 << 30
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    y = torch.randn((reps, 180000), generator=g, device="cuda", dtype=torch.complex64)
    A.set_kernel_timing(True, count_atomics=True)
    a = A.adj(y)
    assert (A.read_flush_atomics() == 0) == two_phase
    if two_phase:
        assert torch.equal(a, A.adj(y))
