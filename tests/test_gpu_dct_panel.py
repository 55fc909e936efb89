"""GPU tests of the BF16x3 panel DCT passes (and the F32 ones over the same
shapes): every count of waves along the outputs (axes of up to 32, 64, 128, 256
and more values), several groups and stages, partial tiles and chunks, rows and
planes whose length is no multiple of four, axes of one voxel (no pass), and
enough columns for the widest panels.  Reference: scipy's FP64 DCT-II and its
inverse, whose scaling is the transforms' own, and the FP64 oracle for the
Poisson solve with the eigenvalue divide fused into the last pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b)) / np.max(np.abs(b)))


# (D, H, W)
SHAPES = [(1, 1, 5), (1, 1, 300), (1, 37, 1), (1, 33, 65), (3, 1, 17), (17, 31, 33), (32, 16, 15),
          (64, 63, 66), (5, 130, 127), (129, 7, 34), (9, 255, 20), (257, 3, 45), (4, 511, 6),
          (2, 6, 513), (600, 5, 7), (70, 250, 251), (128, 130, 300)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision,tol", [(1, 3e-6), (2, 4e-5)])
def test_transforms_against_scipy(ctx, shape, precision, tol):
    from scipy import fft
    print("panel", shape, precision, flush=True)
    x = np.random.default_rng(3).standard_normal(shape).astype(np.float32)
    x64 = x.astype(np.float64)
    assert _rel(ctx.cosine_transform(x, precision), fft.dctn(x64, type=2)) < tol
    assert _rel(ctx.inverse_cosine_transform(x, precision), fft.idctn(x64, type=2)) < tol


@pytest.mark.parametrize("shape", [(1, 1, 9), (1, 40, 1), (1, 33, 66), (6, 1, 21), (20, 18, 34),
                                   (70, 5, 17), (3, 520, 5)])
@pytest.mark.parametrize("precision,tol", [(1, 1e-5), (2, 1e-4)])
def test_poisson_solve_against_oracle(ctx, orc, shape, precision, tol):
    print("poisson", shape, precision, flush=True)
    rng = np.random.default_rng(4)
    phi = np.zeros(shape)
    for ks in rng.integers(0, 6, (12, 3)):
        z, y, x = np.ix_(*[np.cos(np.pi * k * (np.arange(n) + 0.5) / n) for k, n in zip(ks, shape)])
        phi += rng.standard_normal() * z * y * x
    v = [orc.forward_difference(phi, a).astype(np.float32) for a in range(3)]
    ref = orc.integrate_poisson(*[c.astype(np.float64) for c in v], dtype=np.float64)
    out = ctx.integrate_gradients_poisson(*v, precision=precision)
    assert _rel(out, ref) < tol


# axes whose split table goes to the device in several pieces (from 1025 values on)
@pytest.mark.parametrize("shape", [(1, 3, 2100), (1, 2065, 4), (4096, 1, 2)])
def test_long_axes_against_scipy(ctx, shape):
    test_transforms_against_scipy(ctx, shape, 2, 4e-5)
