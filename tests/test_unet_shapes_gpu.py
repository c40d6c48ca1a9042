"""The U-Net's tiled kernels at image sizes whose tiles are cut: one pixel at
the deepest level, widths that are no multiple of 16, heights below a tile,
batches that take the larger and the smaller tiles.  Against the CPU oracle
(oracle/unet_torch.py) with the tolerances of test_unet_gpu.py (BF16 operands,
2^-9 per product, FP32 sums), and against themselves (no atomics: the same
bits every time)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, 1), (8, 136, 2), (24, 104, 3), (40, 24, 5), (72, 200, 8)]


@pytest.mark.parametrize("H,W,B", SHAPES)
def test_cut_tiles_match_the_oracle(H, W, B):
    import torch
    from cffc_amd import unet as U
    from oracle.unet_torch import RefUNet
    rng = np.random.default_rng(H + W + B)
    net = U.UNet(H=H, W=W, max_batch=B + 1, seed=3)
    X = rng.normal(0, 1, (B, H, W, 8)).astype(np.float32)
    T = rng.normal(0, 0.5, (B, H, W, 4)).astype(np.float32)
    net.set_dataset(X, T)
    last = net.nlayers - 1
    w, b = net.get_weights(last)
    net.set_weights(last, w * 20.0, b + 0.1)
    shapes = [net.layer_shape(l) for l in range(net.nlayers)]
    ref = RefUNet([net.get_weights(l) for l in range(net.nlayers)], shapes)
    loss_ref, y_ref = ref.loss(X, T)
    loss_ref.backward()
    y = net.predict(X)
    yr = y_ref.detach()[..., :4].numpy()
    assert np.abs(y - yr).max() / np.abs(yr).max() < 2e-2
    idx = np.arange(B)
    for l in range(net.nlayers):
        loss, gw, gb = net.loss_grad(idx, l)
        gr, br = ref.w[l].grad.numpy(), ref.b[l].grad.numpy()
        # below a few hundred pixels the BF16 rounding of single gradients does
        # not average out over the weight gradient's sum
        tol = 5e-2 if H * W * B > 1000 else 1e-1
        assert np.linalg.norm(gw - gr) / np.linalg.norm(gr) < tol, l
        assert np.linalg.norm(gb - br) / max(np.linalg.norm(br), 1e-30) < tol, l
        assert abs(loss - float(loss_ref.detach())) / float(loss_ref.detach()) < 2e-2
        loss2, gw2, gb2 = net.loss_grad(idx, l)
        assert loss2 == loss and np.array_equal(gw, gw2) and np.array_equal(gb, gb2)
    net.close()


def test_training_steps_are_reproducible():
    from cffc_amd import unet as U
    out = []
    for _ in range(2):
        rng = np.random.default_rng(1)
        net = U.UNet(H=24, W=40, max_batch=4, seed=5)
        net.set_dataset(rng.normal(0, 1, (6, 24, 40, 8)).astype(np.float32),
                        rng.normal(0, 0.5, (6, 24, 40, 4)).astype(np.float32))
        losses = [net.train_step(np.array(i), 1e-3) for i in ([0, 1, 2, 3], [4, 5], [2, 0, 5])]
        out.append((losses, [net.get_weights(l) for l in range(net.nlayers)]))
        net.close()
    assert out[0][0] == out[1][0]
    for (w0, b0), (w1, b1) in zip(out[0][1], out[1][1]):
        assert np.array_equal(w0, w1) and np.array_equal(b0, b1)
