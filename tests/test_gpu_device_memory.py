"""GPU tests of a card that is nearly full: what the fused TGV-k sweep keeps second
copies for runs as two launches where they do not fit (order 4 needs 448 bytes per
voxel with them, 236 without), and copies that an earlier call holds make room
for what a later one cannot do without.  Another context takes the rest of the
memory; every allocation that fails is answered on the host."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TAU = float(np.float32(1 / np.sqrt(20)))
GIB = 1 << 30
SHAPE = (256, 256, 256)          # state of order 4: 3.7 GiB, second copies: 3.3 GiB
ALPHA = (1.0, 2.0, 0.6, 0.4)


def _params(native, iterations, **kw):
    return native.default_params(lam=0.7, alpha0=2.0, alpha1=1.0, tau=TAU, sigma=TAU, theta=1.0,
                                 iterations=iterations, **kw)


def _denoise_adjoint(c, native, f):
    return c.tgv2_denoise_adjoint(f[:64], _params(native, 3, data_term=native.DATA_L2), f[64:128],
                                  checkpoint_every=2)


def test_order_4_on_a_nearly_full_card():
    from ambient_image_processor_amd import native
    f = (0.4 + 0.2 * np.random.default_rng(8).standard_normal(SHAPE)).astype(np.float32)
    with native.Context(0) as c:
        c.set_override("tgvk_fused", 0)
        ref = c.tgvk_deshade(f, _params(native, 4), ALPHA)
        c.tgvk_deshade(f, _params(native, 2), ALPHA)
        ref_state = c.get_state()
        ref_adjoint = _denoise_adjoint(c, native, f)
    with native.Context(0) as holder, native.Context(0) as c:
        pieces = [holder.alloc(5 * GIB // 2), holder.alloc(GIB + GIB // 16)]
        rest = []
        while True:   # all but 3.95 GiB
            take = torch.cuda.mem_get_info(0)[0] - int(3.95 * GIB)
            if take < 16 << 20:
                break
            rest.append(holder.alloc(min(take, 16 * GIB)))

        def fused_launches(masked):
            c.profile(True)
            c.profile_reset()
            out = (c.tgvk_deshade_masked(f, _params(native, 4), ALPHA, np.ones(SHAPE, np.uint8))
                   if masked else c.tgvk_deshade(f, _params(native, 4), ALPHA))
            for a, b in zip(out, ref):
                np.testing.assert_array_equal(a, b)
            return c.profile_counts()["tgvk_fused"]

        print("neither copy fits", flush=True)
        assert fused_launches(False) == 0
        holder.free(pieces.pop())
        print("one of the two fits", flush=True)
        assert fused_launches(False) == 0
        assert fused_launches(True) == 0
        holder.free(pieces.pop())
        print("both fit", flush=True)
        assert fused_launches(False) == 3

        print("room for another buffer, the state in the copies", flush=True)
        c.tgvk_deshade(f, _params(native, 2), ALPHA)   # one fused launch
        p = c.alloc(3 * GIB)
        np.testing.assert_array_equal(c.get_state(), ref_state)
        c.free(p)
        print("room for the adjoint's workspace", flush=True)
        c.tgvk_deshade(f, _params(native, 2), ALPHA)   # leaves 0.5 GiB
        for a, b in zip(_denoise_adjoint(c, native, f), ref_adjoint):   # six states of 0.27 GiB
            np.testing.assert_array_equal(a, b)
        for q in rest:
            holder.free(q)
