"""Fused FFT passes of lengths with the prime factors 2, 3, 5 and 7, against
numpy's float64 FFT and against the rocFFT path of the same plan.

Tolerances are those of the power-of-two passes: rounding grows like
log2(K) eps, about 11 x 6e-8 (1.1e-16) at K = 2048 before the factor of three
that the tests leave for the constants of the odd radices.
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from tests.cases import rel_l2
from tests.test_gpu_fft import TOL, _adjoint_image, _forward_grid, _image, _op, dev

pytestmark = pytest.mark.gpu

# every radix in every position of the list, one to five passes, the smallest
# and largest lengths, lines that do not fill a wave, line counts that do not
# divide by the lines of a workgroup, and mixtures with powers of two
GEOMS = [
    ((40, 100), (70, 140)), ((81, 100), (81, 128)), ((50, 60), (98, 100)), ((100, 80), (125, 81)),
    ((121, 30), (243, 48)), ((343, 40), (343, 45)), ((512, 15), (1029, 18)), ((7, 100), (75, 135)),
    ((1001, 10), (2000, 16)), ((9, 1500), (21, 2025)), ((3, 320), (16, 640)), ((240, 200), (360, 300)),
    ((24, 25, 26), (48, 50, 84)), ((30, 16, 9), (45, 32, 18)), ((12, 90, 20), (16, 135, 40)), ((9, 10, 11), (18, 21, 27)),
]


def _need(A):
    assert A.plan_info()["fused_fft"]


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("Nd,Kd", GEOMS)
def test_mixed_passes_vs_numpy(precision, Nd, Kd):
    A = _op(Nd, Kd, precision, adjoint_scalefactor=0.75)
    _need(A)
    sn = A.sn.cpu().numpy().astype(np.float64)
    xn, xt = _image(Nd, 3, A._tcdt, seed=5)
    g = _forward_grid(A, xt, 3).cpu().numpy()
    for r in range(3):
        assert rel_l2(g[r].reshape(tuple(reversed(Kd))).T, np.fft.fftn(xn[r].T * sn, s=Kd)) <= TOL[precision]
    gn = trj.complex_gaussian((2, int(np.prod(Kd))), seed=6)
    x = _adjoint_image(A, torch.from_numpy(gn).to(dev()).to(A._tcdt), 2).cpu().numpy()
    sl = tuple(slice(0, n) for n in Nd)
    for r in range(2):
        ref = np.fft.ifftn(gn[r].reshape(tuple(reversed(Kd))).T)[sl] * np.prod(Kd) * 0.75 * sn
        assert rel_l2(x[r].T, ref) <= TOL[precision]


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("phasing,ortho", [("real", False), ("real", True), ("complex", True)])
@pytest.mark.parametrize("order", ["F", "C"])
@pytest.mark.parametrize("Nd,Kd", [((33, 80), (64, 150)), ((45, 81), (90, 105)),
                                   ((20, 24, 16), (30, 48, 70)), ((21, 10, 35), (42, 20, 72))])
def test_operator_mixed_vs_rocfft(precision, phasing, ortho, order, Nd, Kd):
    """Whole transforms in both orders, plain and strided images, one and
    three repetitions, twice through the plan's own grid."""
    om = np.random.default_rng(1).uniform(-np.pi, np.pi, (500, len(Nd)))
    A = NufftBase(Nd, om, Jd=5, Kd=Kd, Ld=256, precision=precision, ortho=ortho, phasing=phasing, order=order,
                  n_shift=tuple(n / 2 for n in Nd), device=dev())
    for reps in (1, 3):
        shape = ((reps,) + Nd if order == "C" else Nd + (reps,)) if reps > 1 else Nd
        x = torch.from_numpy(trj.complex_gaussian(shape, seed=7)).to(dev()).to(A._tcdt)
        strided = torch.stack([x, x], dim=-1)[..., 0]
        y = torch.from_numpy(trj.complex_gaussian((reps, 500), seed=8)).to(dev()).to(A._tcdt)
        y = y[0] if reps == 1 else (y if order == "C" else y.t().contiguous())
        got = []
        for method in ("auto", "rocfft", "auto"):
            A.set_fft(method)
            assert A.plan_info()["fused_fft"] == (method == "auto")
            got.append((A.fft(x).cpu().numpy(), A.fft(strided).cpu().numpy(), A.adj(y).cpu().numpy()))
        for a in (got[0], got[2]):
            for u, v in zip(a, got[1]):
                assert u.shape == v.shape
                assert rel_l2(u, v) <= 3 * TOL[precision]


@pytest.mark.parametrize("Kd", [(66, 640), (2187, 16), (1000,), (15, 900), (1701, 16), (96, 96), (60, 48)])
def test_other_grids_keep_rocfft(Kd):
    """A prime factor beyond 7, axes out of range, one axis, and small grids."""
    A = _op(tuple(k // 2 for k in Kd), Kd, "single")
    assert not A.plan_info()["fused_fft"]
