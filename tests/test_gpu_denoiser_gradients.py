"""The backward kernels of the denoiser against 64-bit sums over the tensors that
the library itself stores (ohpt_denoiser_read_tensor), so nothing but the kernel
under test lies between: sizes at the edges of its 16x16 tiles, one tile and one
pixel per level, several images, more tiles than blocks."""
import sys
from pathlib import Path

import numpy as np
import pytest

from ohao_engine_amd import ohpt

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import denoiser_ref as R  # noqa: E402

pytestmark = pytest.mark.gpu

INDEX = {n: i for i, (n, _, _) in enumerate(ohpt.DENOISER_TENSORS)}
SIZES = [(1, 16, 16), (2, 37, 72), (1, 17, 250), (5, 64, 96), (3, 144, 16)]


def trained_pass(B, H, W, seed=3):
    rng = np.random.default_rng(seed)
    f = lambda *s: rng.random(s, dtype=np.float32)
    dn = ohpt.Denoiser(seed=1)
    dn.set_params(R.init_params(seed))
    dn.forward_backward(f(B, H, W, 4) * 3, f(B, H, W, 4), f(B, H, W, 4) * 2 - 1, f(B, H, W) * 9, f(B, H, W, 4))
    return dn


def grad_of(dn, name):
    t = ohpt.TENSOR_LOGITS if name == "logits" else INDEX[name]
    return dn.read_tensor(ohpt.TENSOR_GRAD + t).astype(np.float64)


@pytest.mark.parametrize("size", SIZES)
def test_weight_gradients_are_the_sums_over_the_stored_tensors(size):
    dn = trained_pass(*size)
    grads = dn.get_grads().astype(np.float64)
    for li, (a, b, o, cout, _) in enumerate(R.LAYERS):
        x = dn.read_tensor(INDEX[a]).astype(np.float64)
        if b:
            x = np.concatenate([x, dn.read_tensor(INDEX[b]).astype(np.float64)], -1)
        g = grad_of(dn, o)[..., :cout]
        B, h, w, ci = x.shape
        xp = np.pad(x, ((0, 0), (1, 1), (1, 1), (0, 0)))
        ws, bs = R.layer_slices()[li]
        # FP32 sums of n products of two bf16 values (each product exact in FP32): every
        # addition rounds once, so the error is at most n 2^-24 of the sum of magnitudes
        n = B * h * w
        for t in range(9):
            xt = xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(n, ci)
            want = xt.T @ g.reshape(n, cout)
            bound = n * 2.0 ** -24 * (np.abs(xt).T @ np.abs(g).reshape(n, cout)) + 1e-30
            got = grads[ws].reshape(9, ci, cout)[t]
            assert np.all(np.abs(got - want) <= bound), (li, t, float(np.max(np.abs(got - want) / bound)))
        bound = n * 2.0 ** -24 * np.abs(g).sum((0, 1, 2)) + 1e-30
        assert np.all(np.abs(grads[bs] - g.sum((0, 1, 2))) <= bound), li
    dn.close()
