"""The backward kernels of the denoiser against 64-bit sums over the tensors that
the library itself stores (ohpt_denoiser_read_tensor), so nothing but the kernel
under test lies between: sizes at the edges of its 16x16 tiles, one tile and one
pixel per level, several images (a tile per block), and one with several tiles per
block at every one of the four upper levels."""
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

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


def tiles_per_block(li, B, H, W):
    """16x16 tiles that a block of layer li's weight gradient walks: two blocks per compute
    unit over the combinations of 32 output and 32 (16 in the input layer) input channels."""
    a, b, o, cout, _ = R.LAYERS[li]
    level = [lv for n, lv, _ in ohpt.DENOISER_TENSORS if n == a][0]
    cin = R.CHAN[a] + (R.CHAN[b] if b else 0)
    up = lambda v, d: -(-v // d)
    tiles = B * up(R.pad16(H) >> level, 16) * up(R.pad16(W) >> level, 16)
    combos = up(cout, 32) * (1 if a == "x0" else cin // 32)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return up(tiles, max(1, 2 * cus // combos)), tiles


def test_weight_gradients_of_blocks_with_several_tiles():
    """Tiles of the next step are loaded while this one's are multiplied, ranges cross from one
    image (182 tiles) into the next and the last range is shorter. The bound is the depth of
    the sum and not its length, so that one tile dropped or taken twice exceeds it."""
    B, H, W = 5, 200, 216
    dn = trained_pass(B, H, W)
    grads = dn.get_grads().astype(np.float64)
    seen = set()
    for li, (a, b, o, cout, _) in enumerate(R.LAYERS):
        per, tiles = tiles_per_block(li, B, H, W)
        seen.add((per > 1, per > 2, tiles % per != 0))
        x = dn.read_tensor(INDEX[a])
        if b:
            x = np.concatenate([x, dn.read_tensor(INDEX[b])], -1)
        g = torch.from_numpy(grad_of(dn, o)[..., :cout])
        n, h, w, ci = x.shape
        xp = torch.nn.functional.pad(torch.from_numpy(x).double(), (0, 0, 1, 1, 1, 1))
        # additions that one product passes through: those of its wave's 64 pixels of each of
        # the block's tiles, of four waves, of every 16th block and of 16 threads. Each loses
        # at most 2^-23 of the partial sum, rounded or cut
        blocks = -(-tiles // per)
        depth = 64 * per + 4 + -(-blocks // 16) + 16
        ws, bs = R.layer_slices()[li]
        got = torch.from_numpy(grads[ws].reshape(9, ci, cout))
        gf = g.reshape(-1, cout)
        worst = 0.0
        for t in range(9):
            xt = xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(-1, ci)
            bound = depth * 2.0 ** -23 * (xt.abs().T @ gf.abs()) + 1e-30
            worst = max(worst, float(((got[t] - xt.T @ gf).abs() / bound).max()))
        bias = float((np.abs(grads[bs] - gf.sum(0).numpy()) / (depth * 2.0 ** -23 * gf.abs().sum(0).numpy() + 1e-30)).max())
        print(f"layer {li}: {per} tiles per block, {blocks} blocks, error / bound {worst:.3f}, bias {bias:.3f}", flush=True)
        assert worst <= 1.0 and bias <= 1.0, li
        if li == 1:   # the bound tells a tile: without one of the 910, many sums miss it
            drop = xp[1, 17:33, 17:33].reshape(-1, ci).T @ g[1, 16:32, 16:32].reshape(-1, cout)
            mag = xp[:, 1:-1, 1:-1].reshape(-1, ci).abs().T @ gf.abs()
            assert (drop.abs() > 4 * depth * 2.0 ** -23 * mag).float().mean() > 0.2
    assert {(True, False, True), (True, True, False)} & seen and {(True, True, True)} & seen, seen
    dn.close()
