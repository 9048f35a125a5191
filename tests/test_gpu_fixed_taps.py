"""Tap counts with compiled trip counts (J = 4, 5, 6 on every axis) and the
generic kernels beside them, against the oracle, and the trajectory gradient
against central differences.

The transforms are held to the parity bars (1e-5, 1e-12).  A difference
quotient of step h has an error of about eps / h relative to the samples
(1e-16 / 1e-7) and the two curvature-free sides of a linear interpolant agree
but for the points whose step crosses a table cell, so 1e-5 leaves room.
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from mrrt.nufft_amd.autograd import nufft
from oracle import nufft_oracle as O
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu

GEOMS = [((50,), (75,)), ((24, 31), (48, 62)), ((10, 12, 9), (20, 18, 18))]


@pytest.mark.parametrize("precision,tol", [("single", 1e-5), ("double", 1e-12)])
@pytest.mark.parametrize("phasing", ["real", "complex"])
@pytest.mark.parametrize("J", [3, 4, 5, 6, 7])
@pytest.mark.parametrize("Nd,Kd", GEOMS)
def test_transforms_vs_oracle(precision, tol, phasing, J, Nd, Kd):
    om = np.random.default_rng(1).uniform(-np.pi, np.pi, (700, len(Nd)))
    kw = dict(Jd=J, Kd=Kd, Ld=256, precision=precision, phasing=phasing, n_shift=np.asarray(Nd) / 2)
    A, B = NufftBase(Nd, om, device=torch.device("cuda", 0), **kw), O.NufftOracle(Nd, om, **kw)
    x = trj.complex_gaussian(Nd + (2,), seed=2)
    y = trj.complex_gaussian((700, 2), seed=3)
    assert rel_l2(A.fft(x), B.fft(x)) <= tol
    assert rel_l2(A.adj(y), B.adj(y)) <= tol


@pytest.mark.parametrize("J", [4, 5, 6, 7])
@pytest.mark.parametrize("Nd,Kd", GEOMS)
def test_gradient_vs_differences(J, Nd, Kd):
    m, h = 300, 1e-7
    om = torch.from_numpy(np.random.default_rng(4).uniform(-3, 3, (m, len(Nd)))).cuda()
    A = NufftBase(Nd, om, Jd=J, Kd=Kd, Ld=256, precision="double", device=om.device)
    x = torch.from_numpy(trj.complex_gaussian((3,) + Nd, seed=5)).cuda()
    w = torch.from_numpy(trj.complex_gaussian((3, m), seed=6)).cuda()
    o = om.clone().requires_grad_(True)
    (g,) = torch.autograd.grad(nufft(A, x, o), (o,), w)
    for d in range(len(Nd)):
        e = torch.zeros(len(Nd), dtype=torch.float64, device=om.device)
        e[d] = h
        dy = (nufft(A, x, om + e) - nufft(A, x, om - e)) / (2 * h)
        ref = (w.conj() * dy).real.sum(0)
        assert rel_l2(g[:, d].cpu().numpy(), ref.cpu().numpy()) <= 1e-5
