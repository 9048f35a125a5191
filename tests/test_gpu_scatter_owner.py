"""The 2-D scatter of several repetitions that owns its grid cells (no grid
atomics) against the float64-tile scatter and the oracle.

Rounding: a tap is rounded to a step of 2^-30 A cmax with A the largest sample
sum over 2 x 2 blocks of J - 1 cells, half a step at most, against cell sums of about
sqrt(n) c for the n taps of random phase that a cell collects; with the few
dozen samples per block and the coefficients (about a tenth of cmax)
of these inputs that is a few 1e-7, below the parity bar by more than ten.
"""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd import trajectories as trj
from oracle import nufft_oracle as O
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu


def dev():
    assert torch.cuda.is_available()
    return torch.device("cuda", 0)


def _points(kind, m, rng):
    if kind == "uniform":
        return rng.uniform(-np.pi, np.pi, (m, 2))
    if kind == "edge":      # first taps around the periodic seam and the tile edges
        k = rng.integers(-4, 5, (m, 2)) * (2 * np.pi / 8) * rng.choice([0.999, 1.0, 1.001], (m, 2))
        return np.clip(k, -np.pi, np.pi)
    om = rng.uniform(-np.pi, np.pi, (m, 2))  # half of the points in one bin: left to the atomic kernel
    om[: m // 2] = rng.uniform(0.1, 0.16, (m // 2, 2))
    return om


def _reps(Kd):
    """The smallest odd count whose grids together pass the size from which
    the path is taken."""
    return (320 << 20) // (8 * int(np.prod(Kd))) + 1 | 1


def _samples(reps, m, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn((reps, m), generator=g, device="cuda", dtype=torch.complex64)


@pytest.mark.parametrize("phasing", ["real", "complex"])
@pytest.mark.parametrize("kind,m", [("uniform", 2000), ("uniform", 3), ("edge", 2000), ("dense", 3000)])
@pytest.mark.parametrize("Nd,Kd,Jd,bins", [
    ((100, 100), (256, 256), 6, None),           # whole tiles
    ((120, 22), (240, 44), 6, None),             # partial tiles, the smallest range for J = 6
    ((100, 190), (250, 375), (4, 4), None),      # partial tiles and bins, J = 4
    ((140, 150), (300, 280), (5, 7), (8, 16)),   # unequal taps, other bins
    ((160, 100), (256, 200), (8, 8), (64, 32)),  # bins wider than a tile, the most taps
])
def test_owner_vs_float64_and_oracle(phasing, kind, m, Nd, Kd, Jd, bins):
    rng = np.random.default_rng(3)
    om = _points(kind, m, rng)
    kw = dict(Jd=Jd, Kd=Kd, Ld=256, phasing=phasing, n_shift=np.asarray(Nd) / 2)
    A = NufftBase(Nd, om, order="C", device=dev(), **kw)
    if bins:
        A.set_binning(bins)
    reps = _reps(Kd)
    y = _samples(reps, m, 4)
    got = A.adj(y)
    A.set_kernel_timing(True, count_atomics=True)
    again = A.adj(y)
    # no atomics on the grid but those of dense bins (more points than half their cells and than one batch)
    if kind != "edge":
        dense = kind == "dense" and m // 2 > max(256, int(np.prod(A.plan_info()["bin_size"])) // 2)
        assert (A.read_flush_atomics() > 0) == dense
    A.set_scatter("float64")
    ref = A.adj(y)
    for g in (got, again):
        d = (g - ref).reshape(reps, -1).norm(dim=1) / ref.reshape(reps, -1).norm(dim=1)
        assert d.max().item() <= 1e-6
    if kind == "edge" or m < 10:
        B = O.NufftOracle(Nd, om, **kw)
        for r in (0, reps - 1):
            assert rel_l2(got[r].cpu().numpy(), B.adj(y[r].cpu().numpy())) <= 1e-5


def test_owner_scales_and_nonfinite():
    """Samples of 2^-120 .. 2^100 keep the accuracy; a NaN sample shows in its
    own repetition only; zeros stay zero."""
    Nd, Kd, m = (128, 128), (256, 256), 3000
    A = NufftBase(Nd, trj.golden_angle_2d(30, 100)[:m], Jd=6, Kd=Kd, Ld=256, order="C", device=dev())
    reps = _reps(Kd)
    yn = _samples(reps, m, 5)
    s = torch.ones((reps, 1), dtype=torch.float64, device="cuda")
    s[:4, 0] = torch.tensor([2.0 ** -120, 1.0, 2.0 ** 100, 0.0])
    y = (yn.to(torch.complex128) * s).to(torch.complex64)
    x = A.adj(y)
    ref = A.adj(yn)
    for r in range(3):
        assert rel_l2((x[r].to(torch.complex128) / s[r]).cpu().numpy(), ref[r].cpu().numpy()) <= 1e-6
    assert (x[3] == 0).all()
    y[1, 17] = float("nan")
    x2 = A.adj(y)
    assert torch.isnan(x2[1].real).any() and torch.isfinite(x2[4:].real).all()
    assert rel_l2(x2[4:].cpu().numpy(), x[4:].cpu().numpy()) <= 1e-6


def test_owner_under_graph_and_between_single_adjoints():
    """Replays of a captured multi-repetition adjoint, with single ones (which
    need a cleared grid) between them, equal the eager results."""
    Nd, Kd, m = (256, 256), (512, 512), 4000
    A = NufftBase(Nd, trj.golden_angle_2d(40, 100), Jd=6, Kd=Kd, Ld=256, order="C", device=dev())
    y = _samples(_reps(Kd), m, 6)
    y0 = y[0].contiguous()
    ref, one = A.adj(y).clone(), A.adj(y0).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        A.adj(y), A.adj(y0)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g, g1 = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = A.adj(y)
    with torch.cuda.graph(g1):
        out1 = A.adj(y0)
    for k in range(4):
        (g if k % 2 else g1).replay()
        g.replay()
        g1.replay()
        torch.cuda.synchronize()
        for a, b in ((out, ref), (out1, one), (A.adj(y0), one), (A.adj(y), ref)):
            assert rel_l2(a.cpu().numpy(), b.cpu().numpy()) <= 1e-6
