"""The persistent convolution (more than two tiles and channel groups per resident
block) against 64-bit sums over the tensors that the library stores: one chunk of
input channels with several tiles per block and ranges that cross into the next
image, one and two chunks with one tile per block, and the input gradient."""
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from ohao_engine_amd import ohpt

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import denoiser_ref as R  # noqa: E402
from test_gpu_denoiser_gradients import INDEX, trained_pass  # noqa: E402

pytestmark = pytest.mark.gpu


def conv(x, w):
    """x (B, H, W, ci), w (9, ci, co) in float64: the zero-padded sums, and of magnitudes."""
    t = torch.from_numpy(np.ascontiguousarray(x.transpose(0, 3, 1, 2)))
    k = torch.from_numpy(np.ascontiguousarray(w.transpose(2, 1, 0).reshape(w.shape[2], w.shape[1], 3, 3)))
    f = lambda a, b: torch.nn.functional.conv2d(a, b, padding=1).numpy().transpose(0, 2, 3, 1)
    return f(t, k), f(t.abs(), k.abs())


def bf16(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).bfloat16().double().numpy()


@pytest.mark.parametrize("size", [(2, 530, 545), (1, 1090, 290)])
def test_persistent_convolution(size):
    print(f"persistent convolution {size}", flush=True)
    dn = trained_pass(*size)
    params = dn.get_params().astype(np.float64)
    read = lambda n, g=0: dn.read_tensor(g + INDEX[n]).astype(np.float64)
    for li in (1, 2, 3):                       # a0 -> e0, p1 -> a1, a1 -> e1
        a, _, o, co, _ = R.LAYERS[li]
        ws, bs = R.layer_slices()[li]
        x = read(a)
        w = bf16(params[ws].reshape(9, x.shape[3], co))
        want, mag = conv(x, w)
        want = np.maximum(want + params[bs], 0.0)
        # FP32 sums of 9 ci products (each exact) and a bias, then one rounding to bf16
        bound = 2.0 ** -8 * np.abs(want) + (9 * x.shape[3] + 1) * 2.0 ** -24 * (mag + np.abs(params[bs])) + 1e-30
        assert np.all(np.abs(read(o) - want) <= bound), o
    ws, _ = R.layer_slices()[3]
    w = bf16(params[ws].reshape(9, 64, 64))
    want, mag = conv(read("e1", ohpt.TENSOR_GRAD), w[::-1].transpose(0, 2, 1))
    want *= read("a1") > 0                     # the stored gradient is masked by its own ReLU
    bound = 2.0 ** -8 * np.abs(want) + 9 * 64 * 2.0 ** -24 * mag + 1e-30
    assert np.all(np.abs(read("a1", ohpt.TENSOR_GRAD) - want) <= bound)
    dn.close()
