"""The convolution's tile sizes: which one runs depends on how many workgroups the larger ones give."""
import numpy as np
import pytest

import unet_oracle as U
import ufomi
from conftest import rel_l2

pytestmark = pytest.mark.gpu


# 32 pixels wide: 32-channel tiles below 512 workgroups of 64-channel ones (1 x 256 x 32: 32 pixel
# tiles), 64-channel tiles above, the last with cout not a multiple of 64; 64 wide likewise
@pytest.mark.parametrize("B,cin,cout,H,W", [(1, 64, 64, 8, 32), (3, 32, 136, 16, 32), (1, 32, 1024, 128, 32),
                                            (1, 32, 1000, 128, 32), (1, 32, 512, 256, 64), (1, 32, 136, 8, 64)])
def test_conv3x3_tiles(ctx, torch_dev, B, cin, cout, H, W):
    import torch
    rng = np.random.default_rng(cin + cout + H)
    x = U.bf16(rng.standard_normal((B, H, W, cin)))
    w = U.bf16(rng.standard_normal((cout, 3, 3, cin)) / np.sqrt(9 * cin))
    b = rng.standard_normal(cout).astype(np.float32)

    def dev(a, shift):
        t = torch.empty(a.size + 8, dtype=torch.bfloat16, device=torch_dev)
        t[shift:shift + a.size] = torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).reshape(-1).to(torch_dev)
        return t[shift:shift + a.size]

    d_w, d_b = dev(w, 0), torch.from_numpy(b).to(torch_dev)
    got = []
    for shift in (0, 4) if W == 32 else (0,):  # 16-byte aligned tensors; 8-byte aligned ones take the generic product
        out = dev(np.zeros((B, H, W, cout)), shift)
        ctx.nn_conv3x3(dev(x, shift), B, H, W, cin, d_w, d_b, True, cout, out)
        got.append(out.float().cpu().numpy().reshape(B, H, W, cout))
    ref = np.maximum(U.conv3x3(x, w, b.astype(np.float64)), 0)
    for g in got:  # one bf16 rounding of a float32 sum
        assert rel_l2(g, ref) < 4e-3
        assert np.all(np.abs(g - ref) <= 2 * 2.0 ** -7 * np.abs(ref) + 1e-6)


def test_batches_take_other_tiles_and_agree(ctx, torch_dev):
    """Every tile size sums in the same order, so a batch (larger tiles, with the fused pool) gives
    the bits of its images alone (smaller ones)."""
    import torch
    B, H, W = 16, 256, 256
    img = torch.from_numpy(np.random.default_rng(23).standard_normal((B, H, W)).astype(np.float32)).to(torch_dev)
    out, one = torch.empty_like(img), torch.empty_like(img)
    net = ufomi.Unet(ctx, B, H, W, seed=3)
    for n in (16, 8, 4):
        net.forward(img[:n].contiguous(), out[:n])
        for i in range(n):
            net.forward(img[i:i + 1].contiguous(), one[i:i + 1])
        assert torch.equal(out[:n], one[:n]), n
    net.close()


# transposed convolutions whose pixels do not fill the tiles of 128 (20, 80 and 320 of them), cross
# images within a tile, and (8 x 64 x 64: 4096) take the XCD order
@pytest.mark.parametrize("B,H,W", [(5, 16, 16), (3, 16, 64), (8, 64, 64)])
def test_transposed_conv_tiles(ctx, torch_dev, B, H, W):
    import torch
    params = U.random_params(np.random.default_rng(29))
    net = ufomi.Unet(ctx, B, H, W)
    flat = np.zeros(net.padded, dtype=np.float32)
    for name, off, dims in net.tensors:
        flat[off:off + int(np.prod(dims))] = params[name].reshape(-1)
    net.set_params(flat)
    img = np.random.default_rng(30).standard_normal((B, H, W)).astype(np.float32)
    d_in = torch.from_numpy(img).to(torch_dev)
    out = torch.full((B + 1, H, W), 7.0, device=torch_dev)
    net.forward(d_in, out[:B])
    assert bool((out[B] == 7.0).all())
    ref, _ = U.UNet(params).forward(img.astype(np.float64))
    r32, _ = U.UNet(params, acc=np.float32).forward(img.astype(np.float64))
    # three times what float32 accumulation does through the bf16 layers
    assert rel_l2(out[:B].cpu().numpy() - img, ref - img) < 3 * rel_l2(r32 - img, ref - img) + 2e-3
    net.close()
