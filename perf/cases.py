"""Performance cases of the TGV-DCT deshade path.

Each case is one call (or one forward and backward pass) that a program makes
through the package's public entry points, with its inputs already in device
memory (`*_device` entry points) or in host arrays (the denoise cases).  One
native.Context serves the whole process, as a program that deshades one volume
after another keeps it.  Sizes are voxels: w x h x d, x fastest.

  kind           entry point
  denoise_host   Context.tgv2_denoise on host arrays, optionally with the energy trace
  deshade        Context.deshade_pipeline_device (3-D, masked or 2-D; FP32 or BF16 fields)
  tgvk           Context.tgvk_deshade_pipeline_device
  downsampled    Context.tgvk_deshade_downsampled_device
  poisson        Context.integrate_gradients_poisson_device
  adjoint        autograd.tgv2_l2_denoise, forward and backward
"""
import math

import numpy as np
import torch

from ambient_image_processor_amd import native
from ambient_image_processor_amd.autograd import tgv2_l2_denoise

DCT = {"reference": native.DCT_REFERENCE, "f32": native.DCT_F32, "bf16x3": native.DCT_BF16X3}
STEP = float(np.float32(1.0 / math.sqrt(20.0)))   # tau = sigma, the default parameters' value


def listed():
    return [
        # the smallest calls: a region of interest denoised from host memory; latency and
        # launches count, not bandwidth
        dict(name="denoise_host_32", kind="denoise_host", w=32, h=30, d=24, iterations=50,
             data="l2", energy=0),
        # a small volume run to convergence
        dict(name="deshade_64", kind="deshade", w=64, h=64, d=64, iterations=500, data="l2",
             storage="f32", dct="reference", mask=0.0),
        # the ordinary volume: FP32 fields, reference-numerics DCT
        dict(name="deshade_256", kind="deshade", w=256, h=256, d=256, iterations=200, data="l1",
             storage="f32", dct="reference", mask=0.0),
        # an odd-sized scan with its object masked (about 35% of the voxels)
        dict(name="deshade_masked_odd", kind="deshade", w=181, h=217, d=181, iterations=100,
             data="l1", storage="f32", dct="f32", mask=0.42),
        # an odd-sized volume from host memory with its convergence watched
        dict(name="denoise_host_energy_odd", kind="denoise_host", w=161, h=145, d=140,
             iterations=100, data="l1", energy=10),
        # the largest volume: BF16 fields and the split-precision DCT
        dict(name="deshade_bf16_384", kind="deshade", w=384, h=384, d=384, iterations=100,
             data="l2", storage="bf16", dct="bf16x3", mask=0.0),
        # a large 2-D image
        dict(name="deshade_image_2048", kind="deshade", w=2048, h=1500, d=1, iterations=200,
             data="l1", storage="f32", dct="f32", mask=0.0),
        # third-order smoothing above the TGV2 loop (order 4)
        dict(name="tgvk4_128", kind="tgvk", w=128, h=128, d=128, iterations=100, order=4,
             dct="reference"),
        # a large masked volume deshaded at half resolution (order 3) and resampled back
        dict(name="downsampled_512", kind="downsampled", w=512, h=512, d=256, iterations=50,
             order=3, factor=0.5, mask=0.46, dct="bf16x3"),
        # the bias solve alone: gradients of a large volume, split-precision DCT
        dict(name="poisson_512_bf16x3", kind="poisson", w=512, h=512, d=256, dct="bf16x3"),
        # the bias solve alone in the reference's numerics, sizes that are no power of two
        dict(name="poisson_ref_odd", kind="poisson", w=251, h=240, d=180, dct="reference"),
        # a training step through the unrolled denoiser: gradients of the volumes and weights
        dict(name="adjoint_128", kind="adjoint", w=128, h=128, d=128, batch=2, iterations=60,
             checkpoint=20),
    ]


def _extents(rng, low, high, cap):
    """Three extents, each spread over the logarithm of [low, high], at most `cap` voxels."""
    while True:
        e = [int(round(math.exp(rng.uniform(math.log(low), math.log(high))))) for _ in range(3)]
        if e[0] * e[1] * e[2] <= cap:
            return dict(w=e[0], h=e[1], d=e[2])


def draw(rng):
    """One more case: the listed kinds over 2e3 .. 5e7 voxels, odd and ragged sizes among them."""
    kind = rng.choice(["denoise_host", "deshade", "deshade", "masked", "bf16", "image", "tgvk",
                       "downsampled", "poisson", "poisson", "adjoint"])
    its = rng.randint(20, 100)
    data = rng.choice(["l1", "l2"])
    dct = rng.choice(sorted(DCT))
    if kind == "denoise_host":
        return dict(kind=kind, iterations=its, data=data, energy=rng.choice([0, 10, 25]),
                    **_extents(rng, 12, 192, 4e6))
    if kind == "deshade":
        return dict(kind="deshade", iterations=its, data=data, storage="f32", dct=dct, mask=0.0,
                    **_extents(rng, 16, 320, 1.6e7))
    if kind == "masked":
        return dict(kind="deshade", iterations=its, data=data, storage="f32", dct=dct,
                    mask=round(rng.uniform(0.2, 0.48), 3), **_extents(rng, 32, 256, 1.2e7))
    if kind == "bf16":
        return dict(kind="deshade", iterations=its, data=data, storage="bf16", dct="bf16x3",
                    mask=0.0, **_extents(rng, 32, 384, 3e7))
    if kind == "image":
        e = _extents(rng, 100, 3000, 1e12)
        return dict(kind="deshade", iterations=its, data="l1", storage="f32",
                    dct=rng.choice(["f32", "bf16x3"]), mask=0.0, w=e["w"], h=e["h"], d=1)
    if kind == "tgvk":
        return dict(kind=kind, iterations=rng.randint(20, 60), order=rng.randint(3, 5), dct=dct,
                    **_extents(rng, 24, 200, 4e6))
    if kind == "downsampled":
        return dict(kind=kind, iterations=rng.randint(20, 50), order=3,
                    factor=rng.choice([0.25, 0.4, 0.5, 0.7]), mask=round(rng.uniform(0.3, 0.5), 3),
                    dct="bf16x3", **_extents(rng, 64, 512, 5e7))
    if kind == "poisson":
        return dict(kind=kind, dct=dct, **_extents(rng, 24, 512, 2e7))
    return dict(kind=kind, batch=rng.randint(1, 2), iterations=rng.randint(20, 60),
                checkpoint=rng.choice([1, 10, 20]), **_extents(rng, 24, 144, 2.1e6))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _shape(case):
    return case["d"], case["h"], case["w"]


def _axes(shape):
    return [(torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) / n for n in shape]


def _phantom(shape, gen, noise=0.03):
    """Spheres of different intensity, a smooth bias of low cosine orders and noise."""
    z, y, x = _axes(shape)
    top = float(max(shape))
    f = torch.zeros(shape, device="cuda")
    for _ in range(24):
        c = torch.rand(3, generator=gen).tolist()
        r = 0.03 + 0.16 * float(torch.rand(1, generator=gen))
        val = 0.1 + 0.9 * float(torch.rand(1, generator=gen))
        dist = sum((((a - c[k]) * (shape[k] / top)) ** 2).reshape([-1 if j == k else 1 for j in range(3)])
                   for k, a in enumerate((z, y, x)))
        f.masked_fill_(dist <= r * r, val)
    for k in range(3):
        for j in range(3):
            for i in range(3):
                if i + j + k == 0:
                    continue
                a = 0.05 * float(torch.randn(1, generator=gen))
                f += a * (torch.cos(math.pi * k * z)[:, None, None] *
                          torch.cos(math.pi * j * y)[None, :, None] *
                          torch.cos(math.pi * i * x)[None, None, :])
    dev = torch.Generator(device="cuda").manual_seed(int(torch.randint(1 << 31, (1,), generator=gen)))
    f += noise * torch.randn(shape, generator=dev, device="cuda")
    return f


def _ball(shape, radius):
    """1 inside an ellipsoid of the given relative radius, 0 outside; None for radius 0."""
    if not radius:
        return None
    z, y, x = _axes(shape)
    d = ((z - 0.5) ** 2)[:, None, None] + ((y - 0.5) ** 2)[None, :, None] + ((x - 0.5) ** 2)[None, None, :]
    return (d <= radius * radius).to(torch.float32).contiguous()


def _smooth_gradients(shape, gen):
    """Forward differences of a field of low cosine modes (what the iteration's v looks like),
    with a little noise."""
    z, y, x = _axes(shape)
    phi = torch.zeros(shape, device="cuda")
    for _ in range(24):
        k = torch.randint(0, 12, (3,), generator=gen).tolist()
        phi += float(torch.randn(1, generator=gen)) * (
            torch.cos(math.pi * k[0] * z)[:, None, None] * torch.cos(math.pi * k[1] * y)[None, :, None] *
            torch.cos(math.pi * k[2] * x)[None, None, :])
    dev = torch.Generator(device="cuda").manual_seed(int(torch.randint(1 << 31, (1,), generator=gen)))
    out = []
    for axis in (2, 1, 0):
        v = torch.zeros(shape, device="cuda")
        n = shape[axis]
        v.narrow(axis, 0, n - 1).copy_(phi.narrow(axis, 1, n - 1) - phi.narrow(axis, 0, n - 1))
        out.append(v + 1e-3 * torch.randn(shape, generator=dev, device="cuda"))
    return out


def _inputs(case, seed):
    gen = torch.Generator().manual_seed(seed)
    shape = _shape(case)
    kind = case["kind"]
    if kind == "poisson":
        return dict(v=_smooth_gradients(shape, gen))
    if kind == "adjoint":
        f = torch.stack([_phantom(shape, gen, 0.05) for _ in range(case["batch"])])
        dev = torch.Generator(device="cuda").manual_seed(seed + 1)
        g = torch.randn(f.shape, generator=dev, device="cuda") / math.sqrt(f.numel())
        return dict(f=f, g=g)
    return dict(f=_phantom(shape, gen), mask=_ball(shape, case.get("mask", 0.0)))


def _alpha(case):
    return [1.0 + 3.0 * i for i in range(case["order"])]


def _params(case):
    flags = native.FLAG_SET_NEGATIVE_ZERO
    if case.get("mask"):
        flags |= native.FLAG_MASKED_ITERATION | native.FLAG_ADD_BACKGROUND_BACK
    if case["d"] == 1:
        flags |= native.FLAG_PLANAR
    return native.default_params(
        lam=0.5, alpha0=2.0, alpha1=1.0, iterations=case["iterations"],
        data_term=native.DATA_L2 if case.get("data") == "l2" else native.DATA_L1,
        storage=native.STORAGE_BF16 if case.get("storage") == "bf16" else native.STORAGE_F32,
        dct_precision=DCT[case.get("dct", "reference")], flags=flags)


_contexts = []


def _context():
    if not _contexts:
        _contexts.append(native.Context(torch.cuda.current_device()))
    return _contexts[0]


def prepare(case, seed):
    state = dict(case=case, **_inputs(case, seed))
    if case["kind"] == "adjoint":
        state["f"].requires_grad_(True)
        state["weights"] = [torch.tensor(a, requires_grad=True) for a in (2.0, 1.0, 1.0)]
        torch.cuda.synchronize()
        return state
    state["ctx"] = _context()
    if case["kind"] == "denoise_host":
        state["f"] = state["f"].cpu().numpy()
    else:
        n_out = 1 if case["kind"] == "poisson" else 3
        state["out"] = [torch.empty(_shape(case), device="cuda") for _ in range(n_out)]
    if case["kind"] != "poisson":
        state["params"] = _params(case)
    torch.cuda.synchronize()   # the context works on its own stream
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "adjoint":
        f, w = state["f"], state["weights"]
        u = tgv2_l2_denoise(f, *w, iterations=case["iterations"],
                            checkpoint_every=case["checkpoint"])
        grads = torch.autograd.grad(u, [f] + w, state["g"])
        return [u.detach(), *grads]
    ctx = state["ctx"]
    if kind == "denoise_host":
        ctx.set_energy_interval(case["energy"])
        u = ctx.tgv2_denoise(state["f"], state["params"])
        trace = ctx.energy_trace() if case["energy"] else None
        ctx.set_energy_interval(0)
        return [u] if trace is None else [u, trace]
    out = [o.data_ptr() for o in state["out"]]
    shape = _shape(case)
    if kind == "poisson":
        ctx.integrate_gradients_poisson_device(*[v.data_ptr() for v in state["v"]], shape, out[0],
                                               precision=DCT[case["dct"]])
        return state["out"]
    f, p = state["f"].data_ptr(), state["params"]
    mask = state["mask"].data_ptr() if state["mask"] is not None else None
    if kind == "deshade":
        ctx.deshade_pipeline_device(f, shape, p, *out, mask_dev=mask)
    elif kind == "tgvk":
        ctx.tgvk_deshade_pipeline_device(f, shape, p, _alpha(case), *out, mask_dev=mask)
    else:
        ctx.tgvk_deshade_downsampled_device(f, shape, p, case["factor"], _alpha(case), mask, *out)
    return state["out"]


def _small_shape(case):
    return native.resize_extents(_shape(case), case["factor"])


def work(case):
    """Bytes: inputs read and outputs written once, and per iteration every field of the state
    (u, v, p, q: 13 elements a voxel; 12 more per level of TGV-k) read and written and f read.
    Flops: the updates' operations per voxel, and 2.5 n log2(n) per transformed line."""
    shape = _shape(case)
    n = shape[0] * shape[1] * shape[2]
    solve = 5.0 * n * math.log2(max(n, 2))
    if case["kind"] == "poisson":
        return dict(bytes=16.0 * n, flops=solve + 7.0 * n)
    size = 2 if case.get("storage") == "bf16" else 4
    it = case["iterations"]
    if case["kind"] == "adjoint":
        n *= case["batch"]
        # forward, then per reverse iteration the state and its adjoint
        return dict(bytes=it * n * 4.0 * (27 + 13 + 27) + 16.0 * n, flops=it * n * (110.0 + 250.0))
    levels = max(0, case.get("order", 2) - 2)
    if case["kind"] == "downsampled":
        small = _small_shape(case)
        m = small[0] * small[1] * small[2]
        return dict(bytes=20.0 * n + it * m * 4.0 * (27 + 24 * levels),
                    flops=it * m * (110.0 + 70.0 * levels) + 2 * 128.0 * n +
                    5.0 * m * math.log2(max(m, 2)))
    if case["d"] == 1:
        per, ops = 2 * 8 + 1, 60.0    # no z components
    else:
        per, ops = 27, 110.0
    if case["kind"] == "denoise_host":
        return dict(bytes=8.0 * n + it * n * per * 4.0, flops=it * n * ops)
    return dict(bytes=16.0 * n + it * n * (size * (per - 1 + 24 * levels) + 4.0),
                flops=it * n * (ops + 70.0 * levels) + solve)


# ---------------------------------------------------------------------------
# the same results in 64 bits, from the definitions
# ---------------------------------------------------------------------------

def _fwd(a, axis):
    """D+: a[i + 1] - a[i], 0 at the end."""
    n = a.shape[axis]
    last = torch.zeros_like(a.narrow(axis, 0, 1))
    return torch.cat([a.narrow(axis, 1, n - 1) - a.narrow(axis, 0, n - 1), last], axis)


def _bwd(a, axis):
    """B: a[i - 1] - a[i], -a[0] at the start."""
    n = a.shape[axis]
    first = -a.narrow(axis, 0, 1)
    return torch.cat([first, a.narrow(axis, 0, n - 1) - a.narrow(axis, 1, n - 1)], axis)


X, Y, Z = 2, 1, 0
AXES = [(X, None), (Y, None), (Z, None), (X, Y), (X, Z), (Y, Z)]   # tensor components


def _project(t, alpha, weights):
    n2 = sum(w * c * c for w, c in zip(weights, t))
    # scale alpha / |t| outside the ball (no square root of 0, so gradients stay finite)
    scale = torch.where(n2 > alpha * alpha, alpha / torch.sqrt(n2.clamp_min(alpha * alpha)),
                        torch.ones_like(n2))
    return [c * scale for c in t]


def _tensor_op(t, diff, half):
    out = []
    for c, (a, b) in zip(t, AXES):
        d = diff(c, a)
        if b is not None:
            d = (d + diff(c, b)) * half
        out.append(d)
    return out


TENSOR_WEIGHTS = [1, 1, 1, 2, 2, 2]


def _tgv(f, iterations, lam, alpha, l2, active=None, planar=False):
    """The TGV-k iteration (k = len(alpha)); alpha[0] bounds p, alpha[1] q -> u, [vx, vy, vz]."""
    zero = torch.zeros_like(f)
    u = ub = f
    v = [zero] * 3
    vb = [zero] * 3
    p = [zero] * 3
    q = [zero] * 6
    levels = len(alpha) - 2
    w = [[zero] * 6 for _ in range(levels)]
    wb = [[zero] * 6 for _ in range(levels)]
    r = [[zero] * 6 for _ in range(levels)]
    tau = sigma = STEP
    tl = tau * lam
    no_z = l2 and f.shape[0] == 1

    def keep(new, old):
        return new if active is None else [torch.where(active, a, b) for a, b in zip(new, old)]

    def bz(a):
        return zero if planar else _bwd(a, Z)

    for _ in range(iterations):
        p = keep(_project([p[k] + sigma * (_fwd(ub, ax) - vb[k]) for k, ax in enumerate((X, Y, Z))],
                          alpha[0], [1, 1, 1]), p)
        div = _bwd(p[0], X) + _bwd(p[1], Y)
        if not no_z:
            div = div + _bwd(p[2], Z)
        un = u - tau * div
        if l2:
            un = (un + tl * f) / (1.0 + tl)
        else:
            un = torch.where(un - f > tl, un - tl, torch.where(un - f < -tl, un + tl, f))
        (un,), (ub,) = keep([un], [u]), keep([2.0 * un - u], [ub])
        u = un
        e = [_bwd(vb[0], X), _bwd(vb[1], Y), bz(vb[2]), 0.5 * (_bwd(vb[1], X) + _bwd(vb[0], Y)),
             0.5 * (_bwd(vb[2], X) + bz(vb[0])), 0.5 * (_bwd(vb[2], Y) + bz(vb[1]))]
        if levels:
            e = [a - b for a, b in zip(e, wb[0])]
        q = keep(_project([a + sigma * b for a, b in zip(q, e)], alpha[1], TENSOR_WEIGHTS), q)
        dq = [_fwd(q[0], X) + _fwd(q[3], Y) + _fwd(q[4], Z), _fwd(q[1], Y) + _fwd(q[3], X) + _fwd(q[5], Z),
              _fwd(q[2], Z) + _fwd(q[4], X) + _fwd(q[5], Y)]
        vn = keep([a - tau * (b - c) for a, b, c in zip(v, dq, p)], v)
        vb = keep([2.0 * a - b for a, b in zip(vn, v)], vb)
        v = vn
        for i in range(levels):
            g = _tensor_op(wb[i], _fwd if i % 2 else _bwd, 0.5)
            if i + 1 < levels:
                g = [a - b for a, b in zip(g, wb[i + 1])]
            r[i] = keep(_project([a + sigma * b for a, b in zip(r[i], g)], alpha[i + 2],
                                 TENSOR_WEIGHTS), r[i])
            hr = _tensor_op(r[i], _bwd if i % 2 else _fwd, 1.0)
            below = q if i == 0 else r[i - 1]
            wn = keep([a - tau * (b - c) for a, b, c in zip(w[i], hr, below)], w[i])
            wb[i] = keep([2.0 * a - b for a, b in zip(wn, w[i])], wb[i])
            w[i] = wn
    return u, v


def _cosines(n):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    return torch.cos(math.pi * k[:, None] * (k[None, :] + 0.5) / n)      # [k][m]


def _along(a, m, axis):
    return torch.movedim(torch.tensordot(m, a, dims=([1], [axis])), 0, axis).contiguous()


def _integrate(v):
    """Divergence, DCT-II, eigenvalue divide (its cosines in 32 bits, as the solve defines
    them), DCT-III."""
    g = _bwd(v[0], X) + _bwd(v[1], Y)
    shape = g.shape
    if shape[0] > 1:
        g = g + _bwd(v[2], Z)
    for axis in (X, Y, Z):
        g = _along(g, _cosines(shape[axis]), axis)
    g = g * 8.0
    c = [torch.cos(math.pi * torch.arange(n, device="cuda", dtype=torch.float64) / n).float().double()
         for n in shape]
    den = -2.0 * c[1][None, :, None] - 2.0 * c[2][None, None, :]
    den = den + 4.0 if shape[0] == 1 else den + 6.0 - 2.0 * c[0][:, None, None]
    den[0, 0, 0] = 1.0
    g = g / den
    g[0, 0, 0] = 0.0
    for axis in (X, Y, Z):
        m = _cosines(shape[axis]).t().clone()
        m[:, 1:] *= 2.0
        g = _along(g, m, axis)
    return g / (8.0 * g.numel())


def _tail(u, l, mask, r0=None):
    """r = u - l, the mask on l and r, clamp, background back (r0: the order of the downsampled
    tail, whose clamp comes last)."""
    if mask is None:
        return l, (u - l).clamp_min(0.0)
    if r0 is None:
        return l * mask, ((u - l) * mask).clamp_min(0.0) + u * (1.0 - mask)
    return l * mask, ((r0 * mask - l) * mask + r0 * (1.0 - mask)).clamp_min(0.0)


def _spline_matrix(n, new, pad):
    """Cubic B-spline resampling of a line of n samples to `new` ones, as a matrix."""
    if n == 1:
        return torch.ones(new, 1, dtype=torch.float64, device="cuda")
    interp = np.zeros((n, n))
    for i in range(n):   # samples from coefficients, mirrored about the first and last
        interp[i, i] += 4.0 / 6.0
        for j in (i - 1, i + 1):
            interp[i, -j if j < 0 else 2 * (n - 1) - j if j >= n else j] += 1.0 / 6.0
    spacing = 1.0 / float(np.float32(new + pad) / np.float32(n))
    out = np.zeros((new, n))
    for j in range(new):
        x = j * spacing
        if not -0.5 <= x < n - 0.5:
            continue
        i = math.floor(x)
        t = x - i
        wt = [(1 - t) ** 3 / 6, (3 * t ** 3 - 6 * t * t + 4) / 6,
              (-3 * t ** 3 + 3 * t * t + 3 * t + 1) / 6, t ** 3 / 6]
        for k in range(4):
            m = (i - 1 + k) % (2 * (n - 1))
            out[j, m if m < n else 2 * (n - 1) - m] += wt[k]
    return torch.from_numpy(np.linalg.solve(interp.T, out.T).T.copy()).cuda()


def _resize(a, shape):
    pad = 2 if any(s > t for s, t in zip(shape, a.shape)) else 0
    for axis in (X, Y, Z):
        a = _along(a, _spline_matrix(a.shape[axis], shape[axis], pad), axis)
    return a.float().double()   # a resized volume is stored in 32 bits


def _adjoint_exact(case, given):
    f = given["f"].double().requires_grad_(True)
    w = [torch.tensor(a, dtype=torch.float64, device="cuda", requires_grad=True) for a in (2.0, 1.0, 1.0)]
    us, grads = [], [torch.zeros_like(f)] + [torch.zeros((), dtype=torch.float64, device="cuda") for _ in w]
    for b in range(f.shape[0]):
        fb = given["f"][b].double().requires_grad_(True)
        u, _ = _tgv(fb, case["iterations"], w[2], [w[1], w[0]], True)
        got = torch.autograd.grad(u, [fb] + w, given["g"][b].double())
        us.append(u.detach())
        grads[0][b] = got[0]
        for k in range(3):
            grads[k + 1] += got[k + 1]
        del u, got
    return [torch.stack(us), *[g.detach() for g in grads]]


def exact(case, seed):
    given = _inputs(case, seed)
    if case["kind"] == "poisson":
        return [_integrate([v.double() for v in given["v"]])]
    if case["kind"] == "adjoint":
        # the tape of one volume holds about 90 fields an iteration
        n = case["w"] * case["h"] * case["d"]
        return _adjoint_exact(case, given) if 8.0 * 90 * n * case["iterations"] < 1.6e11 else None
    f = given["f"].double()
    mask = given["mask"].double() if given["mask"] is not None else None
    active = mask >= 1 if mask is not None else None
    l2 = case.get("data") == "l2"
    it = case["iterations"]
    if case["kind"] == "denoise_host":
        u, _ = _tgv(f, it, 0.5, [1.0, 2.0], l2)
        return [u.cpu().numpy(), None] if case["energy"] else [u.cpu().numpy()]
    if case["kind"] == "downsampled":
        small = _small_shape(case)
        fs = _resize((given["f"] * given["mask"]).double(), small)
        ms = _resize(mask, small)
        u, v = _tgv(fs, it, 0.5, _alpha(case), False, ms >= 1)
        l = _integrate(v) * ms
        u, l = _resize(u.float().double(), f.shape), _resize(l.float().double(), f.shape)
        return [u, *_tail(u, l, mask, r0=f)]
    alpha = _alpha(case) if case["kind"] == "tgvk" else [1.0, 2.0]
    u, v = _tgv(f, it, 0.5, alpha, l2, active, planar=case["d"] == 1)
    return [u, *_tail(u, _integrate(v), mask)]
