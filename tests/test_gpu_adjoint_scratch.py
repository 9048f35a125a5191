"""Adjoints captured after eager ones of the same size that used the other
plan-owned grid (the scatter that owns its cells has one of its own): nothing
can be allocated while capturing, and either grid serves.

The replays are held to the float adds' order, as the tests of the owner
scatter are (1e-6)."""

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import NufftBase
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu

KD, M = (256, 256), 2000
REPS = (320 << 20) // (8 * 256 * 256) + 1  # grids beyond the size from which the owner scatter is taken


@pytest.mark.parametrize("warm,captured", [("float64", "auto"), ("auto", "float64")])
@pytest.mark.parametrize("fft", ["auto", "rocfft"])
def test_capture_after_the_other_scatter(warm, captured, fft):
    om = np.random.default_rng(0).uniform(-np.pi, np.pi, (M, 2))
    A = NufftBase((128, 128), om, Jd=6, Kd=KD, Ld=256, order="C", device=torch.device("cuda", 0))
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    y = torch.randn((REPS, M), generator=g, device="cuda", dtype=torch.complex64)
    B = NufftBase((128, 128), om, Jd=6, Kd=KD, Ld=256, order="C", device=y.device)
    B.set_scatter(captured)
    ref = B.adj(y).cpu().numpy()
    A.set_fft(fft)
    A.set_scatter(warm)
    A.adj(y)
    A.set_scatter(captured)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = A.adj(y)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert rel_l2(out.cpu().numpy(), ref) <= 1e-6
        A.set_scatter(warm)  # eager adjoints through the same grid between the replays
        assert rel_l2(A.adj(y).cpu().numpy(), ref) <= 1e-6
        A.set_scatter(captured)
    assert rel_l2(A.adj(y).cpu().numpy(), ref) <= 1e-6
