"""The most points that the static scratch of mi355nufft_table1_adjoint_noalloc
holds.  One line of 1,536 grid points in complex64: 20 bytes per point in five
sections of whole 256 bytes (a gate, tm twice, three int arrays, 35 ints per
bin of 512, and three ints per subproblem of 512 points and one), 3,351,457
points in 64 MiB exactly; one section more for 3,351,473."""

import ctypes

import numpy as np
import pytest
import torch

from mrrt.nufft_amd import _lib
from tests.test_zz_no_alloc import _call, _fn, _tables, _vp, dev

pytestmark = pytest.mark.gpu


def _total(M):
    up = lambda v: -(-v // 256) * 256  # noqa: E731
    o = 256
    for n in (4 * M, 12 * M, 35 * 3 * 4, (3 * (3 + -(-M // 512)) + 1) * 4, 4 * M):
        o = up(o + n)
    return o


def test_noalloc_takes_what_fills_the_scratch():
    lib, fn = _fn()
    Nd, Kd, Jd, L, M = (768,), (1536,), (4,), 64, 3351457
    assert _total(M) == 64 << 20
    hs, hd, hp = _tables(Nd, Jd, Kd, L, np.float32)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    tm = torch.rand((1, M), generator=g, device=dev()) * 1536 - 768
    fm = torch.randn((1, M), generator=g, device=dev(), dtype=torch.complex64)
    rc, got = _call(fn, Kd, Jd, L, np.float32, fm, hp, tm, 1)
    _lib.check(rc)
    ref = torch.empty_like(got)
    _lib.check(lib.mi355nufft_table1_adjoint(1, _lib.i64arr(Kd), _lib.i32arr(Jd), L, 0, 0, _vp(fm), hp, _vp(tm), M,
                                             _vp(ref), 1, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert ((got - ref).norm() / ref.norm()).item() <= 1e-5
    over = M + 16
    assert _total(over) > 64 << 20
    tm2, fm2 = torch.zeros((1, over), device=dev()), torch.zeros((1, over), device=dev(), dtype=torch.complex64)
    rc, _ = _call(fn, Kd, Jd, L, np.float32, fm2, hp, tm2, 1)
    assert rc != 0 and "scratch" in lib.mi355nufft_last_error().decode()
