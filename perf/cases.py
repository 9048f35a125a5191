"""The work that a user of this framework has it do, as cases to be timed and compared.

A case names one call pattern (``kind``) with its sizes:

transform  one forward and one adjoint transform of a ``NufftBase`` operator
           (one iteration of an iterative reconstruction): 1-D to 3-D, with
           one image or several coils, either precision, either kernel
points     a new trajectory set on an existing operator, then one adjoint
           (gridding reconstruction where the trajectory changes per frame)
frames     a dynamic multi-coil series: ``SenseOperator`` over ``NufftFrames``,
           forward and adjoint of every frame and coil
train      forward and backward through ``autograd.nufft`` with gradients of
           the coil images and of the trajectory
normal     the Toeplitz form of the multi-coil normal operator (one iteration
           of conjugate gradients)

``prepare`` makes the inputs on the GPU from the seed and builds the operator
that a program keeps; ``run`` is one pass through the public entry points;
``exact`` is the same sum as a float64 non-uniform DFT in plain torch.
"""

import math

import numpy as np
import torch

from mrrt.nufft_amd import NufftBase
from mrrt.nufft_amd.autograd import nufft
from mrrt.nufft_amd.batched import NufftFrames
from mrrt.nufft_amd.mri import SenseOperator

GOLDEN = math.pi * (math.sqrt(5.0) - 1.0) / 2.0
DEV = "cuda"


def _case(kind, n, over=2.0, j=6, m=0, traj="radial", reps=1, frames=1, precision="single", phasing="real", **kw):
    n = tuple(n) + (0, 0)
    return dict(kw, kind=kind, n0=n[0], n1=n[1], n2=n[2], over=over, j=j, m=m, traj=traj, reps=reps, frames=frames,
                precision=precision, phasing=phasing)


def listed():
    return [
        # the smallest call: one line through the complex-phase kernel, latency and launches only
        _case("transform", (512,), m=2000, traj="random", phasing="complex", name="line 512"),
        # a small 2-D image (48 spokes x 128), as in a preview or a low-resolution navigator
        _case("transform", (64, 64), m=48 * 128, name="radial 64x64"),
        # an ordinary single-coil slice: 402 golden-angle spokes x 512 readout
        _case("transform", (256, 256), m=402 * 512, name="radial 256x256"),
        # the same slice in double precision
        _case("transform", (256, 256), m=402 * 512, precision="double", name="radial 256x256 double"),
        # the constructor's own defaults (Kd = 1.5 Nd, Jd = 4) on a ragged matrix: no power of two anywhere
        _case("transform", (240, 200), over=1.5, j=4, m=90007, traj="spiral", name="spiral 240x200 defaults"),
        # a 12-coil slice at the common 320 matrix
        _case("transform", (320, 320), m=201 * 640, reps=12, name="radial 320x320 12 coils"),
        # a 3-D kooshball volume, 8,192 spokes x 256 readout
        _case("transform", (128, 128, 128), m=8192 * 256, traj="kooshball", name="kooshball 128^3"),
        # a ragged 3-D slab with five taps
        _case("transform", (96, 90, 60), j=5, m=500003, traj="kooshball", name="kooshball 96x90x60"),
        # a trajectory that changes before every gridding
        _case("points", (256, 256), m=402 * 512, name="new points 256x256"),
        # the largest: a dynamic series of 24 frames (13..89 spokes x 512) and 32 coils
        _case("frames", (256, 256), m=512, reps=32, frames=24, name="24 frames x 32 coils"),
        # a training step on 8 coils of a variable-density spiral
        _case("train", (256, 256), m=65536, traj="spiral", reps=8, name="train spiral 8 coils"),
        # one conjugate-gradient iteration on the same data
        _case("normal", (256, 256), m=65536, traj="spiral", reps=8, name="normal spiral 8 coils"),
    ]


def draw(rng):
    def size(lo, hi):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(8, v // 8 * 8) if rng.random() < 0.5 else v

    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["transform"] * 6 + ["points", "frames", "train", "normal"])
    precision = "double" if rng.random() < 0.2 else "single"
    over = rng.choice([2.0, 2.0, 1.5])
    j = rng.choice([4, 5, 6, 6, 6])
    if kind == "transform":
        phasing = "complex" if rng.random() < 0.2 else "real"
        nd = rng.choice([1, 2, 2, 3])
        if nd == 1:
            return _case(kind, (size(64, 4096),), over, j, logint(500, 100000), "random", logint(1, 16), 1, precision,
                         phasing)
        if nd == 2:
            a = size(32, 512)
            n = (a, max(32, min(512, int(a * rng.uniform(0.6, 1.5)))))
            return _case(kind, n, over, j, logint(2000, 400000), rng.choice(["radial", "spiral", "random"]),
                         logint(1, 16), 1, precision, phasing)
        a = size(24, 128)
        n = tuple(max(24, min(128, int(a * rng.uniform(0.6, 1.3)))) for _ in range(2))
        return _case(kind, (a,) + n, over, j, logint(20000, 2000000), rng.choice(["kooshball", "random"]), 1, 1,
                     precision, phasing)
    a = size(64, 256)
    n = (a, max(64, min(256, int(a * rng.uniform(0.7, 1.4)))))
    if kind == "points":
        return _case(kind, n, over, j, logint(2000, 400000), rng.choice(["radial", "spiral", "random"]), 1, 1,
                     precision)
    if kind == "frames":
        return _case(kind, n, over, j, 2 * a, "radial", logint(2, 32), logint(2, 24))
    return _case(kind, n, over, j, logint(4000, 100000), rng.choice(["radial", "spiral"]), logint(1, 8), 1, precision)


# ---------------------------------------------------------------- inputs


def _shape(case):
    return tuple(v for v in (case["n0"], case["n1"], case["n2"]) if v)


def _dtypes(case):
    return ((torch.float64, torch.complex128) if case["precision"] == "double" else (torch.float32, torch.complex64))


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)


def _gauss(g, *shape):
    return torch.complex(torch.randn(shape, generator=g, device=DEV, dtype=torch.float64),
                         torch.randn(shape, generator=g, device=DEV, dtype=torch.float64))


def _spokes(first, nspokes, nread):
    th = torch.remainder((first + torch.arange(nspokes, device=DEV, dtype=torch.float64)) * GOLDEN, math.pi)
    r = -math.pi + 2 * math.pi * torch.arange(nread, device=DEV, dtype=torch.float64) / nread
    return torch.stack([(r[None, :] * torch.cos(th[:, None])).reshape(-1),
                        (r[None, :] * torch.sin(th[:, None])).reshape(-1)], dim=1)


def _trajectory(case, g):
    """(m, ndim) float64 points in [-pi, pi): golden-angle radial, a spiral of
    16 interleaves, a randomly turned kooshball, or uniform random points."""
    nd, m, traj = len(_shape(case)), case["m"], case["traj"]
    if traj == "random":
        return (2 * _rand(g, m, nd) - 1) * math.pi * (1 - 1e-7)
    if traj == "radial":
        nread = 2 * case["n0"]
        return _spokes(1000 * float(_rand(g, 1)), -(-m // nread), nread)[:m].contiguous()
    if traj == "spiral":
        per = -(-m // 16)
        s = torch.arange(per, device=DEV, dtype=torch.float64) / per
        r = math.pi * 0.999 * s ** 1.5
        k = torch.arange(16, device=DEV, dtype=torch.float64)
        th = 2 * math.pi * (16 * s[None, :] + k[:, None] / 16 + float(_rand(g, 1)))
        om = torch.stack([(r * torch.cos(th)).reshape(-1), (r * torch.sin(th)).reshape(-1)], dim=1)[:m]
        om = om + 1e-3 * torch.randn(om.shape, generator=g, device=DEV, dtype=torch.float64)
        return om.clamp(-math.pi, math.pi * (1 - 1e-7))
    nread = 256
    ns = -(-m // nread)
    i = torch.arange(ns, device=DEV, dtype=torch.float64) + 0.5
    z = 1 - 2 * i / ns
    phi = math.pi * (1 + 5 ** 0.5) * i
    rxy = torch.sqrt(1 - z * z)
    rot = np.linalg.qr(np.random.default_rng(int(1e9 * float(_rand(g, 1)))).standard_normal((3, 3)))[0]
    d = torch.stack([rxy * torch.cos(phi), rxy * torch.sin(phi), z], dim=1) @ torch.from_numpy(rot).to(DEV)
    r = -math.pi + 2 * math.pi * torch.arange(nread, device=DEV, dtype=torch.float64) / nread
    return (r[None, :, None] * d[:, None, :]).reshape(-1, 3)[:m].contiguous()


def _images(g, count, shape):
    """Textured objects inside an ellipse, as in a slice of a body."""
    ax = [torch.linspace(-1, 1, s, device=DEV, dtype=torch.float64) for s in shape]
    r2 = sum(c ** 2 for c in torch.meshgrid(*ax, indexing="ij"))
    return ((r2 < 0.8) + 0.02) * (1 + 0.5 * _gauss(g, count, *shape))


def _coil_maps(g, ncoils, shape):
    ax = torch.meshgrid(*[torch.linspace(-1, 1, s, device=DEV, dtype=torch.float64) for s in shape], indexing="ij")
    c = 2 * _rand(g, ncoils, len(shape)) - 1
    out = []
    for k in range(ncoils):
        d2 = sum((a - 1.2 * c[k, i]) ** 2 for i, a in enumerate(ax))
        out.append(torch.polar(torch.exp(-d2), 2 * sum(a * c[k, -1 - i] for i, a in enumerate(ax))))
    return torch.stack(out)


def _samples(g, om, reps):
    """Samples whose size falls with |omega|, as those of an object do."""
    r = om.norm(dim=1)
    return _gauss(g, reps, om.shape[0]) * (0.05 + 1 / (1 + (r / 0.3) ** 2))


def _spoke_counts(case):
    """13..89 spokes per frame, uneven as in a gated series (the sizes belong to the case, not to the seed)."""
    return np.random.default_rng(case["frames"]).integers(13, 90, size=case["frames"])


def _inputs(case, seed):
    g, (rdt, cdt), nd = _gen(seed), _dtypes(case), _shape(case)
    d = {}
    if case["kind"] == "frames":
        counts = _spoke_counts(case)
        first = float(_rand(g, 1)) * 1000
        d["omegas"] = [_spokes(first + int(counts[:f].sum()), int(c), case["m"]) for f, c in enumerate(counts)]
        d["maps"] = _coil_maps(g, case["reps"], nd).to(cdt)
        d["x"] = _images(g, case["frames"], nd).to(cdt)
        d["y"] = _samples(g, torch.cat(d["omegas"]), case["reps"]).to(cdt)
        return d
    d["om"] = _trajectory(case, g).to(rdt)
    x = _images(g, case["reps"], nd).to(cdt)
    y = _samples(g, d["om"].double(), case["reps"]).to(cdt)
    one = case["reps"] == 1 and case["kind"] != "train"
    d["x"], d["y"] = (x[0], y[0]) if one else (x, y)
    if case["kind"] == "normal":
        d["maps"] = _coil_maps(g, case["reps"], nd).to(cdt)
        d["x"] = x[0].contiguous()
        w = d["om"].double().norm(dim=1) + 0.02
        d["w"] = (w / w.sum()).to(rdt)
    if case["kind"] == "points":
        d["om_before"] = _trajectory(case, g).to(rdt)
    return d


def _n_shift(case):
    return tuple(n // 2 for n in _shape(case))


def prepare(case, seed):
    nd = _shape(case)
    s = _inputs(case, seed)
    s["kind"] = case["kind"]
    kw = dict(Jd=case["j"], Kd=tuple(int(case["over"] * n) for n in nd), Ld=1024, precision=case["precision"],
              phasing=case["phasing"], n_shift=_n_shift(case))
    if case["kind"] == "frames":
        op = NufftFrames(nd, [o.cpu().numpy() for o in s["omegas"]], case["reps"], **kw)
        s["sense"] = SenseOperator(op, s["maps"])
    else:
        s["op"] = NufftBase(nd, s["om_before"] if case["kind"] == "points" else s["om"], order="C", **kw)
        if case["kind"] == "normal":
            s["sense"] = SenseOperator(s["op"], s["maps"], weights=s["w"])
            s["sense"].normal(s["x"], toeplitz=True)  # the operator's spectrum is made once, at its first use
        if case["kind"] == "train":
            s["x"].requires_grad_(True)
            s["om"].requires_grad_(True)
    return s


def run(s):
    kind = s["kind"]
    if kind == "transform":
        return s["op"].fft(s["x"]), s["op"].adj(s["y"])
    if kind == "points":
        s["op"].set_points(s["om"])
        return s["op"].adj(s["y"])
    if kind == "frames":
        return s["sense"].forward(s["x"]), s["sense"].adjoint(s["y"])
    if kind == "train":
        y = nufft(s["op"], s["x"], s["om"])
        gx, gom = torch.autograd.grad(y, (s["x"], s["om"]), s["y"])
        return y.detach(), gx, gom
    return s["sense"].normal(s["x"], toeplitz=True)


def work(case):
    """Inputs read once and outputs written once; the taps and the FFTs of the
    oversampled grid (the method's own operations)."""
    nd = _shape(case)
    r = 8 if case["precision"] == "double" else 4
    pix = math.prod(nd)
    nk = math.prod(int(case["over"] * n) for n in nd)
    reps = case["reps"]
    m = case["m"] * int(_spoke_counts(case).sum()) if case["kind"] == "frames" else case["m"]
    fft = 5 * nk * math.log2(nk)
    taps = 4 * m * case["j"] ** len(nd)
    samples, images = 2 * r * m * reps, 2 * r * pix * reps
    points = r * m * len(nd)
    if case["kind"] == "normal":
        full = math.prod(2 * n for n in nd)
        return {"bytes": 2 * r * (2 * pix + reps * pix + full), "flops": 2 * reps * 5 * full * math.log2(full)}
    if case["kind"] == "points":
        return {"bytes": samples + images + points, "flops": fft + taps}
    if case["kind"] == "frames":
        return {"bytes": 2 * (samples + points + 2 * r * pix * (case["frames"] + reps)),
                "flops": 2 * reps * (case["frames"] * fft + taps)}
    if case["kind"] == "train":
        return {"bytes": 2 * (samples + images) + 3 * points, "flops": 2 * reps * (fft + 3 * taps)}
    return {"bytes": 2 * (samples + images + points), "flops": 2 * reps * (fft + taps)}


# ---------------------------------------------------------------- float64 sums


def _phases(om, nd, shift, lo, hi):
    """exp(-i omega_d (n - shift_d)) of points lo..hi, one (points, N_d) matrix per axis."""
    out = []
    for d, n in enumerate(nd):
        k = torch.arange(n, device=DEV, dtype=torch.float64) - shift[d]
        a = om[lo:hi, d, None] * k[None, :]
        out.append(torch.complex(torch.cos(a), -torch.sin(a)))
    return out


def _chunk(reps, nd):
    return max(64, (1 << 26) // (reps * math.prod(nd[1:])))


def _sum_forward(om, x, shift):
    """(reps, m) samples of (reps,) + nd images."""
    om, x = om.double(), x.to(torch.complex128)
    reps, nd = x.shape[0], tuple(x.shape[1:])
    flat = x.movedim(0, 1).reshape(nd[0], -1)
    out = torch.empty((reps, om.shape[0]), dtype=torch.complex128, device=DEV)
    step = _chunk(reps, nd)
    for lo in range(0, om.shape[0], step):
        e = _phases(om, nd, shift, lo, min(lo + step, om.shape[0]))
        t = (e[0] @ flat).reshape((e[0].shape[0], reps) + nd[1:])
        for q in reversed(e[1:]):
            t = (t * q.reshape((q.shape[0],) + (1,) * (t.dim() - 2) + (q.shape[1],))).sum(-1)
        out[:, lo:lo + step] = t.t()
    return out


def _sum_adjoint(om, y, nd, shift):
    """(reps,) + nd images of (reps, m) samples."""
    om, y = om.double(), y.to(torch.complex128)
    reps = y.shape[0]
    acc = torch.zeros((nd[0], reps * math.prod(nd[1:])), dtype=torch.complex128, device=DEV)
    step = _chunk(reps, nd)
    for lo in range(0, om.shape[0], step):
        e = _phases(om, nd, shift, lo, min(lo + step, om.shape[0]))
        t = y[:, lo:lo + step].t()
        for q in e[1:]:
            t = t.unsqueeze(-1) * q.conj().reshape((q.shape[0],) + (1,) * (t.dim() - 1) + (q.shape[1],))
        acc += e[0].conj().t().contiguous() @ t.reshape(t.shape[0], -1)
    return acc.reshape((nd[0], reps) + nd[1:]).movedim(1, 0)


def exact(case, seed):
    nd, d, shift = _shape(case), _inputs(case, seed), _n_shift(case)
    kind = case["kind"]
    if kind == "frames":
        maps, m0, ys, xs = d["maps"].to(torch.complex128), 0, [], []
        for f, om in enumerate(d["omegas"]):
            ys.append(_sum_forward(om, maps * d["x"][f].to(torch.complex128), shift))
            y = d["y"][:, m0:m0 + om.shape[0]]
            xs.append((maps.conj() * _sum_adjoint(om, y, nd, shift)).sum(0))
            m0 += om.shape[0]
        return torch.cat(ys, dim=1), torch.stack(xs)
    if kind == "normal":
        maps, w = d["maps"].to(torch.complex128), d["w"].double()
        y = _sum_forward(d["om"], maps * d["x"].to(torch.complex128), shift)
        return (maps.conj() * _sum_adjoint(d["om"], y * w, nd, shift)).sum(0)
    one = d["x"].dim() == len(nd)
    x, y = (d["x"][None], d["y"][None]) if one else (d["x"], d["y"])
    xa = _sum_adjoint(d["om"], y, nd, shift)
    if kind == "points":
        return xa[0] if one else xa
    yf = _sum_forward(d["om"], x, shift)
    if kind == "transform":
        return (yf[0], xa[0]) if one else (yf, xa)
    grads = []
    for a, n in enumerate(nd):
        k = torch.arange(n, device=DEV, dtype=torch.float64) - shift[a]
        k = k.reshape((1,) + tuple(n if b == a else 1 for b in range(len(nd))))
        dy = _sum_forward(d["om"], -1j * k * x.to(torch.complex128), shift)
        grads.append((y.to(torch.complex128).conj() * dy).real.sum(0))
    return yf, xa, torch.stack(grads, dim=1)
