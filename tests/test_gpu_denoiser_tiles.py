"""The persistent convolution (more than two tiles and channel groups per resident
block) against 64-bit sums over the tensors that the library stores: one, two and
three or more chunks of input channels with several tiles per block, ranges that
cross into the next image, the fused 2x2 maximum, and the input gradient with and
without a mask; and bit for bit against the other convolutions."""
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


def conv_taps(x, w):
    """conv for many channels: a product per tap."""
    B, H, W, ci = x.shape
    xp = torch.nn.functional.pad(torch.from_numpy(x), (0, 0, 1, 1, 1, 1))
    s, m = 0.0, 0.0
    for t in range(9):
        xt = xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, ci)
        k = torch.from_numpy(np.ascontiguousarray(w[t]))
        s = s + xt @ k
        m = m + xt.abs() @ k.abs()
    shape = (B, H, W, w.shape[2])
    return s.reshape(shape).numpy(), m.reshape(shape).numpy()


def test_persistent_convolution_of_three_chunks_and_several_tiles():
    """2 x 530 x 545 (544 x 560 padded): layer 16 at full size reads three chunks in blocks of
    five tiles, layer 14's input gradient at half size two chunks in blocks of six, layer 3
    two chunks in blocks of three with the maximum for the next level; ranges cross the images."""
    dn = trained_pass(2, 530, 545)
    params = dn.get_params().astype(np.float64)
    read = lambda n, g=0: dn.read_tensor(g + INDEX[n])
    for e, p in (("e0", "p1"), ("e1", "p2"), ("e2", "p3"), ("e3", "p4")):
        y = read(e)
        B, H, W, c = y.shape
        assert np.array_equal(read(p), y.reshape(B, H // 2, 2, W // 2, 2, c).max((2, 4))), p
    print("pooled maxima equal", flush=True)
    ws, bs = R.layer_slices()[16]
    x = np.concatenate([read("u0"), read("e0")], -1).astype(np.float64)
    want, mag = conv_taps(x, bf16(params[ws].reshape(9, 96, 32)))
    want = np.maximum(want + params[bs], 0.0)
    bound = 2.0 ** -8 * np.abs(want) + (9 * 96 + 1) * 2.0 ** -24 * (mag + np.abs(params[bs])) + 1e-30
    assert np.all(np.abs(read("b0") - want) <= bound)
    print("three chunks within bounds", flush=True)
    ws, _ = R.layer_slices()[14]
    w = bf16(params[ws].reshape(9, 160, 64))
    want, mag = conv_taps(read("b1", ohpt.TENSOR_GRAD).astype(np.float64), w[::-1].transpose(0, 2, 1)[:, :, :96])
    bound = 2.0 ** -8 * np.abs(want) + 9 * 64 * 2.0 ** -24 * mag + 1e-30
    assert np.all(np.abs(read("u1", ohpt.TENSOR_GRAD) - want) <= bound)
    dn.close()


def test_streaming_inference_equals_the_persistent_training_forward():
    """2 x 300 x 475: 1140 full-resolution tiles, more than two per resident block, so training
    takes the persistent convolution where inference streams."""
    rng = np.random.default_rng(4)
    f = lambda *s: rng.random(s, dtype=np.float32)
    B, H, W = 2, 300, 475
    guides = f(B, H, W, 4) * 3, f(B, H, W, 4), f(B, H, W, 4) * 2 - 1, f(B, H, W) * 9
    dn = ohpt.Denoiser(seed=1)
    dn.set_params(R.init_params(12))
    names = ["a0", "e0", "p1", "b0", "d0"]
    dn.forward_backward(*guides, f(B, H, W, 4))
    train = {n: dn.read_tensor(INDEX[n]) for n in names}
    dn.infer(*guides)
    for n in names:
        got = dn.read_tensor(INDEX[n])
        assert np.array_equal(got.view(np.uint32), train[n].view(np.uint32)), n
        assert np.count_nonzero(got) > got.size // 8, n
    dn.close()
