"""Axis passes of fft_nd / ifft_nd at the edges of their line lengths: every transform length from 16 to
8192, powers of two and the sizes around them (Bluestein lengths change there), along each axis, with
line counts off the lines of a workgroup, zero padding and cropping.

Bar: float32 butterflies over 2 log2(L) <= 26 levels of one rounding each (2^-24, independent) give
3e-7 relative L2, chirps and their tables three more; 1e-6 is three times that."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu
SIZES = [2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 255, 256, 257, 500, 512, 513, 1000, 1024, 1025,
         2047, 2048, 2049, 4095, 4096, 8192]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("m", SIZES)
def test_line_lengths(ctx, torch_dev, axis, m):
    import torch
    shape = [[5, 3], [3, 19], [2, 7]][axis]          # the other two axes, x before y before z
    n = list(shape)
    n.insert(axis, max(1, m - m // 3))               # zero padded to m
    full = list(n)
    full[axis] = m
    rng = np.random.default_rng(m + axis)
    x = rng.standard_normal(n[::-1]).astype(np.float32)
    spec = torch.empty(tuple(full[::-1]) + (2,), device=torch_dev)
    ctx.fft_nd(torch.from_numpy(x).to(torch_dev), n, 3, full, spec)
    got = torch.view_as_complex(spec).cpu().numpy()
    ref = np.fft.fftn(x.astype(np.float64), s=full[::-1], axes=(0, 1, 2))
    assert rel_l2(got, ref) < 1e-6
    back = torch.empty(tuple(full[::-1]), device=torch_dev)
    ctx.ifft_nd(spec, full, 3, back)
    want = np.zeros(full[::-1])
    want[tuple(slice(0, k) for k in n[::-1])] = x
    assert rel_l2(back.cpu().numpy(), want) < 2e-6   # both directions


def test_tables_of_many_sizes(ctx, torch_dev):
    """More sizes in turn than the context keeps Bluestein tables for, and back to the first."""
    import torch
    for m in list(range(90, 160)) + [90, 95]:
        x = np.random.default_rng(m).standard_normal((4, m, m + 1)).astype(np.float32)
        spec = torch.empty((4, m, m + 1, 2), device=torch_dev)
        ctx.fft_nd(torch.from_numpy(x).to(torch_dev), (m + 1, m, 4), 2, (m + 1, m, 4), spec)
        assert rel_l2(torch.view_as_complex(spec).cpu().numpy(), np.fft.fft2(x.astype(np.float64))) < 1e-6


def test_streams_with_many_sizes(torch_dev):
    """More tables than the context keeps, used on two streams in turn: one is replaced only when no stream
    reads it any more."""
    import torch
    import ufomi
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    c = ufomi.Context(0, streams[0])
    held = []
    for i, m in enumerate(list(range(300, 370)) + [300, 301]):
        st = streams[i % 2]
        c.set_stream(st)
        with torch.cuda.stream(st):
            x = torch.randn((40, m, m), device=torch_dev)
            spec = torch.empty((40, m, m, 2), device=torch_dev)
            c.fft_nd(x, (m, m, 40), 2, (m, m, 40), spec)
            held.append((x, spec))
    torch.cuda.synchronize()
    for x, spec in held:
        ref = np.fft.fft2(x[7].cpu().numpy().astype(np.float64))
        assert rel_l2(torch.view_as_complex(spec[7]).cpu().numpy(), ref) < 1e-6
    c.close()


def test_capture(torch_dev):
    """A transform with tables is refused under capture, first call or not; one without is captured."""
    import torch
    import ufomi
    st = torch.cuda.Stream()
    c = ufomi.Context(0, st)
    for m in (96, 100):
        x = torch.randn((3, 64, m), device=torch_dev)
        spec = torch.zeros((3, 64, m, 2), device=torch_dev)
        torch.cuda.synchronize()
        for known in (False, True):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=st):
                spec.zero_()
                with pytest.raises(ufomi.UfomiError):
                    c.fft_nd(x, (m, 64, 3), 2, (m, 64, 3), spec)
            if not known:
                c.fft_nd(x, (m, 64, 3), 2, (m, 64, 3), spec)
                torch.cuda.synchronize()
                assert rel_l2(torch.view_as_complex(spec).cpu().numpy(), np.fft.fft2(x.double().cpu().numpy())) < 1e-6
    x, spec = torch.randn((3, 64, 128), device=torch_dev), torch.zeros((3, 64, 128, 2), device=torch_dev)
    c.fft_nd(x, (128, 64, 3), 2, (128, 64, 3), spec)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        c.fft_nd(x, (128, 64, 3), 2, (128, 64, 3), spec)
    for k in range(3):
        x.normal_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(torch.view_as_complex(spec).cpu().numpy(), np.fft.fft2(x.double().cpu().numpy())) < 1e-6
    c.close()
