"""Weight and bias gradients on NHWC activations (levels at least 32 pixels wide), where the split
over rows, strips and images has edges: levels of two rows, strips at both borders of a row, units
that do not fill the last workgroup, and more units than waves."""
import numpy as np
import pytest

import unet_oracle as U
import ufomi
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _net(ctx, B, H, W, params):
    net = ufomi.Unet(ctx, B, H, W, training=True)
    flat = np.zeros(net.padded, dtype=np.float32)
    for name, off, dims in net.tensors:
        flat[off:off + int(np.prod(dims))] = params[name].reshape(-1)
    net.set_params(flat)
    return net


def _images(seed, B, H, W):
    rng = np.random.default_rng(seed)
    img = rng.standard_normal((B, H, W)).astype(np.float32)
    return img, (img + 0.5 * rng.standard_normal((B, H, W))).astype(np.float32)


# (3, 16, 256): the bottom level has 2 rows of one strip; (1, 16, 512): two strips; (3, 32, 64):
# only the upper two levels are wide enough, the others take the channel-major product
@pytest.mark.parametrize("B,H,W", [(3, 16, 256), (1, 16, 512), (3, 32, 64)])
def test_against_oracle(ctx, torch_dev, B, H, W):
    import torch
    params = U.random_params(np.random.default_rng(17))
    img, tgt = _images(18, B, H, W)
    net = _net(ctx, B, H, W, params)
    _, g = net.gradients(torch.from_numpy(img).to(torch_dev), torch.from_numpy(tgt).to(torch_dev))
    got = net.unpack(g)
    _, ref = U.UNet(params).gradients(img.astype(np.float64), tgt.astype(np.float64))
    _, r32 = U.UNet(params, acc=np.float32).gradients(img.astype(np.float64), tgt.astype(np.float64))
    for name, _ in U.layout():
        # three times the distance of float32 accumulation, with 3% of room for the bf16 rounding
        # flips that sums in another order cause; a missing row or strip is off by more than 10%
        assert rel_l2(got[name], ref[name]) < max(3 * rel_l2(r32[name], ref[name]) + 2e-3, 3e-2), name
    net.close()


# The loss is a mean over the batch, so a batch's gradient is the mean of its halves' (the factor 2
# is exact in bf16).  Halves and whole split differently: only float32 sums differ, 20 layers of
# them at 2^-24 each times the cancellation of random gradients.
@pytest.mark.parametrize("B,H,W", [(2, 16, 256), (6, 64, 256), (16, 16, 8192)])
def test_batch_is_mean_of_halves(ctx, torch_dev, B, H, W):
    import torch
    params = U.random_params(np.random.default_rng(19))
    img, tgt = (torch.from_numpy(a).to(torch_dev) for a in _images(20, B, H, W))
    net = _net(ctx, B, H, W, params)
    whole = net.unpack(net.gradients(img, tgt)[1])
    h = B // 2
    a = net.unpack(net.gradients(img[:h].contiguous(), tgt[:h].contiguous())[1])
    b = net.unpack(net.gradients(img[h:].contiguous(), tgt[h:].contiguous())[1])
    for name, _ in U.layout():
        assert rel_l2(whole[name], 0.5 * (a[name].astype(np.float64) + b[name])) < 2e-5, name
    net.close()
