"""Pipelines whose stage batches are blocks the context keeps and whose last stage writes the
caller's memory: the results are those of the single calls for every kind of destination, and
batches of changing sizes and streams do not disturb each other."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
import ufo_tasks  # noqa: E402
import ufomi  # noqa: E402

pytestmark = pytest.mark.gpu
CHAIN = "fft dimensions=1 size-x=%d ! filter ! ifft dimensions=1 crop-width=%d"


def _text(W, last):
    N = 1 << (2 * W - 1).bit_length()
    chain = CHAIN % (N, W)
    return chain + {"ifft": "", "backproject": " ! backproject axis-pos=%r" % (W / 2.0),
                    "average": " ! average", "transpose": " ! transpose-projections number=7"}[last]


def _run(ctx, text, x, out_ptr, cap, req_hw=None):
    pl = ufo_tasks.Pipeline(text)
    req, oreq, err, n = ufo_tasks.Requisition(), ufo_tasks.Requisition(), ufo_tasks.Error(), ctypes.c_int()
    req.n_dims = 2
    req.dims[0], req.dims[1], req.dims[2] = x.shape[2], x.shape[1], 1
    rc = pl.L.ufomi_pipeline_run(pl.h, ctx.h, x.data_ptr(), ctypes.byref(req), x.shape[0], out_ptr, cap,
                                 ctypes.byref(n), ctypes.byref(oreq), ctypes.byref(err))
    elems = n.value * oreq.dims[0] * oreq.dims[1]
    return rc, elems


@pytest.mark.parametrize("last", ["ifft", "backproject", "average", "transpose"])
def test_destinations_agree(last):
    W, P, S = 65, 9, 5
    ctx = ufomi.Context(0, torch.cuda.current_stream())
    x = torch.randn(S, P, W, device="cuda")
    text = _text(W, last)
    cap = 4 * 9 * 7 * 65 * 65
    plain = torch.full((cap // 4 + 64,), 7.0, device="cuda")
    rc, n = _run(ctx, text, x, plain.data_ptr() + 4, cap)       # not aligned: the result is copied
    assert rc == 0 and n > 0 and plain[0] == 7.0 and bool((plain[1 + n:] == 7.0).all())
    want = plain[1:1 + n].clone()
    direct = torch.full((cap // 4,), 7.0, device="cuda")
    rc, m = _run(ctx, text, x, direct.data_ptr(), 4 * n)        # exactly large enough
    assert rc == 0 and m == n
    assert torch.equal(direct[:n], want) and bool((direct[n:] == 7.0).all())
    direct.fill_(7.0)
    rc, _ = _run(ctx, text, x, direct.data_ptr(), 4 * n - 4)    # too small: refused, nothing written
    assert rc != 0 and bool((direct == 7.0).all())
    host = torch.zeros(n, pin_memory=True)                      # not device memory
    rc, _ = _run(ctx, text, x, host.data_ptr(), 4 * n)
    assert rc == 0 and torch.equal(host, want.cpu())
    both = torch.zeros(max(n, x.numel()), device="cuda")        # the input's own memory
    both[:x.numel()] = x.flatten()
    rc, _ = _run(ctx, text, both[:x.numel()].view_as(x), both.data_ptr(), 4 * n)
    assert rc == 0 and torch.equal(both[:n], want)


@pytest.mark.parametrize("tail", [" ! backproject num-projections=5", " ! backproject ! ifft dimensions=1"])
def test_failures_leave_the_output(tail):
    """Arguments and sizes are checked before the stage that writes the caller's memory starts."""
    W, P, S = 65, 9, 5
    ctx = ufomi.Context(0, torch.cuda.current_stream())
    x = torch.randn(S, P, W, device="cuda")
    out = torch.full((4 * S * W * W,), 7.0, device="cuda")
    rc, _ = _run(ctx, _text(W, "ifft") + tail, x, out.data_ptr(), 4 * out.numel())
    torch.cuda.synchronize()
    assert rc != 0 and bool((out == 7.0).all())


def test_blocks_over_sizes_and_streams():
    """Batches that grow, shrink and exceed what the context keeps, on two streams in turn."""
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    ctx, fresh = ufomi.Context(0, a), None
    for i, (S, P, W) in enumerate([(1, 8, 32), (6, 40, 200), (1, 8, 32), (3, 700, 2048), (40, 900, 2048),
                                   (6, 40, 200), (2, 700, 2048), (1, 1, 1)]):
        st = (a, b)[i % 2]
        ctx.set_stream(st)
        with torch.cuda.stream(st):
            x = torch.randn(S, P, W, device="cuda")
            st.synchronize()
            text = _text(W, "ifft") + " ! fft dimensions=1 ! ifft dimensions=1 crop-width=%d" % W if W > 1 else "average"
            got, n, shape = ufo_tasks.Pipeline(text).run(ctx, x, out_bytes=4 * x.numel())
            fresh = ufomi.Context(0, st)
            ref, m, _ = ufo_tasks.Pipeline(text).run(fresh, x, out_bytes=4 * x.numel())
            st.synchronize()
            k = 4 * n * shape[0] * shape[1] if len(shape) == 2 else 4 * n
            assert n == m and torch.equal(got[:k], ref[:k])


def test_one_pipeline_on_two_contexts():
    """A pipeline's coefficients serve every context that runs it; its batches are the running one's."""
    W, P, S = 64, 9, 3
    x = torch.randn(S, P, W, device="cuda")
    a, b = (ufomi.Context(0, torch.cuda.current_stream()) for _ in range(2))
    pl = ufo_tasks.Pipeline(_text(W, "backproject"))
    want = pl.run(a, x, out_bytes=4 * S * W * W)[0].clone()
    for ctx in (b, a, b):
        assert torch.equal(pl.run(ctx, x, out_bytes=4 * S * W * W)[0], want)
    del pl
    other = ufo_tasks.Pipeline(_text(W, "backproject"))
    assert torch.equal(other.run(a, x, out_bytes=4 * S * W * W)[0], want)
    del other


def test_threads_with_their_own_contexts():
    """Contexts of several threads create, run and end at the same time: their lists of idle memory are apart."""
    import threading
    W, P, S = 320, 700, 24   # a stack for the matrix cores: blocks and a row workspace in every context
    xs = [torch.randn(S, P, W, device="cuda") for _ in range(3)]
    text = _text(W, "backproject")
    main = ufomi.Context(0, torch.cuda.current_stream())
    want = [ufo_tasks.Pipeline(text).run(main, x, out_bytes=4 * S * W * W)[0].clone() for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        try:
            st = torch.cuda.Stream()
            for _ in range(4):
                ctx = ufomi.Context(0, st)
                with torch.cuda.stream(st):
                    for _ in range(3):
                        got = ufo_tasks.Pipeline(text).run(ctx, xs[i], out_bytes=4 * S * W * W)[0]
                        if not torch.equal(got, want[i]):
                            bad.append(i)
                ctx.close()
        except Exception as e:  # reported by the main thread
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in threads)


def _fill(leave):
    """A buffer that leaves about `leave` bytes of the device free."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    return torch.empty(max(1, free - leave), dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("own", [True, False], ids=["same context", "another context"])
def test_idle_memory_is_given_back(own):
    """What a context keeps idle (1 GiB of rows after a stack, a pipeline's blocks) makes room for an allocation
    that does not fit beside it: a U-Net's, a transform's scratch memory, the next stack's rows."""
    GiB = 1 << 30
    st = torch.cuda.current_stream()
    ctx = ufomi.Context(0, st)
    user = ctx if own else ufomi.Context(0, st)
    S, P, W, r = 64, 1800, 2048, 448
    x = torch.randn(S, P, W, device="cuda")
    out = torch.empty(S, r, r, device="cuda")
    roi = dict(n_slices=S, roi_x=800, roi_y=800, roi_width=r, roi_height=r)
    ctx.bp_parallel(x, W, P, out, **roi)
    want = out.clone()
    n = 512
    img = torch.rand(1, n, n, device="cuda")
    small = ufomi.Unet(user, 1, n, n, seed=1)
    ref = torch.empty_like(img)
    small.forward(img, ref)
    small.close()
    # a U-Net of about free + 0.4 GiB: 610 bytes a pixel (float32 output, bf16 images and activations)
    fill = _fill(2 * GiB)
    batch = (torch.cuda.mem_get_info()[0] + int(0.4 * GiB)) // (610 * n * n) + 1
    net = ufomi.Unet(user, batch, n, n, seed=1)
    got = torch.empty_like(img)
    net.forward(img, got, batch=1)
    assert torch.equal(got, ref)
    net.close()
    ctx.bp_parallel(x, W, P, out, **roi)   # takes its rows again
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    # two intermediates of a 3-D transform: 1.5 GiB, with less than 1 GiB free
    del fill
    z = torch.randn(96, 1024, 1024, device="cuda")
    spec = torch.empty(96, 1024, 1024, 2, device="cuda")
    fill = _fill(int(0.8 * GiB))
    user.fft_nd(z, (1024, 1024, 96), 3, (1024, 1024, 96), spec)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(spec[::31, ::101]).all())
    del fill
    torch.cuda.empty_cache()
