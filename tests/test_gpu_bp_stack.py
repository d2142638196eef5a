"""Stacks of slices on the matrix cores (bp_mfma.hip) against the oracle and the interpolating kernel.

The path takes 12 and more slices with at least 1e9 updates (2.5e9 in f16 storage), in units of 64, 32
and 16 slices with up to 8 leftover ones on the interpolating kernel, four angles at a time on 32 x 32
tiles.  Bars: 1e-5 relative L2, the bar of the interpolating kernel (float32 coordinates of up to 512
pixels round at 3e-5 pixels); 16-bit storage is compared on the stored values, so the same bar holds.
"""
import numpy as np
import pytest

import oracle
import ufomi
from conftest import rel_l2

pytestmark = pytest.mark.gpu
DTYPES = {"f32": (ufomi.F32, "float32"), "f16": (ufomi.F16, "float16"), "bf16": (ufomi.BF16, "bfloat16")}


def _both(ctx, torch_dev, x, storage="f32", **props):
    """(matrix cores, interpolating kernel) results of stack x [S][P][W]."""
    import torch
    S, P, W = x.shape
    code = DTYPES[storage][0]
    rw, rh = props.get("roi_width") or W, props.get("roi_height") or W
    outs = []
    try:
        for config in ((0, 0, 0), (8, 8, -1)):
            ctx.bp_configure(*config)
            out = torch.full((S, rh, rw), float("nan"), device=torch_dev)
            ctx.bp_parallel(x, W, P, out, n_slices=S, dtype=code, **props)
            outs.append(out)
    finally:
        ctx.bp_configure(0, 0, 0)
    return outs


def _stack(torch_dev, S, P, W, storage="f32", seed=1):
    import torch
    x = np.random.default_rng(seed).standard_normal((S, P, W)).astype(np.float32)
    return torch.from_numpy(x).to(torch_dev).to(getattr(torch, DTYPES[storage][1]))


@pytest.mark.parametrize("S,P,W,storage", [
    (12, 401, 480, "f32"), (16, 402, 400, "f32"), (17, 403, 400, "f32"), (32, 300, 351, "f32"),
    (33, 300, 352, "f32"), (41, 260, 321, "f32"), (48, 200, 353, "f32"), (49, 200, 353, "f32"),
    (64, 129, 383, "f32"), (73, 1, 3800, "f32"), (130, 64, 512, "f32"),
    (20, 500, 511, "f16"), (64, 400, 320, "f16"), (40, 300, 333, "bf16"),
])
def test_units_vs_oracle(ctx, torch_dev, S, P, W, storage):
    """Full and padded units of 64, 32 and 16 slices, leftovers, angle counts off the fours, split and
    unsplit angles, widths off the tiles.  Against FP64 the bar is the rounding of the inputs of both kernels:
    the float32 (sin, cos) table is off by up to 3e-8, which at 0.7 W (360 pixels) moves a sample by up to 1e-5
    pixels, and white noise turns that into the same relative error; the axis is a float32 number."""
    x = _stack(torch_dev, S, P, W, storage, seed=S)
    got, ref = _both(ctx, torch_dev, x, storage, axis_pos=W / 2.0 + 0.25)
    got, ref = got.cpu().numpy(), ref.cpu().numpy()
    assert np.isfinite(got).all()
    assert not np.array_equal(got, ref)  # the matrix cores ran: they sum in another order
    for s in range(S):
        assert rel_l2(got[s], ref[s]) < 1e-5, s
    s = S // 2
    if W < 1000:
        exact = oracle.bp_texture_f64(x[s].float().cpu().numpy(), axis_pos=W / 2.0 + 0.25)
        assert rel_l2(got[s], exact) < 1e-5
        assert rel_l2(got[s], exact) < 1.2 * rel_l2(ref[s], exact) + 1e-7  # no less precise


@pytest.mark.parametrize("props", [
    dict(axis_pos=150.25, roi_x=33, roi_y=7, roi_width=301, roi_height=215, angle_offset=0.7),
    dict(angle_step=0.013, offset=11, num_projections=900),
    dict(axis_pos=1.5, roi_width=420, roi_height=300),   # most of the image off the detector
])
def test_geometry_and_pitches(ctx, torch_dev, props):
    import torch
    S, P, W = 24, 800, 300  # at least 1.2e9 updates
    x = _stack(torch_dev, S, P, W, seed=5)
    rw, rh = props.get("roi_width") or W, props.get("roi_height") or W
    wide = torch.zeros((S, P * W + 37), device=torch_dev)
    wide[:, :P * W] = x.view(S, -1)
    pitch = rw * rh + 3  # slices of the output off the 16-byte alignment
    got, ref = _both(ctx, torch_dev, x, "f32", **props)
    assert not torch.equal(got, ref)  # the matrix cores ran: they sum in another order
    exact = oracle.bp_texture_f64(x[7].cpu().numpy(), **props)
    assert rel_l2(got[7].cpu().numpy(), exact) < 1e-5
    flat = []
    for config in ((0, 0, 0), (8, 8, -1)):
        try:
            ctx.bp_configure(*config)
            out = torch.full((S, pitch), 7.0, device=torch_dev)
            ctx.bp_parallel(wide, W, P, out, n_slices=S, sino_pitch=P * W + 37, out_pitch=pitch, **props)
            flat.append(out.cpu().numpy())
        finally:
            ctx.bp_configure(0, 0, 0)
    assert (flat[0][:, rw * rh:] == 7.0).all()  # nothing past a slice
    assert rel_l2(flat[0][:, :rw * rh], flat[1][:, :rw * rh]) < 1e-5
    np.testing.assert_array_equal(flat[0][:, :rw * rh].reshape(S, rh, rw), got.cpu().numpy())


@pytest.mark.parametrize("S,P,W,roi,storage,matrix", [
    (16, 800, 2048, 320, "f32", False), (16, 800, 2048, 1024, "f32", True),
    (24, 900, 2048, 384, "f16", False), (24, 900, 2048, 768, "f16", True),
    (64, 720, 4096, 256, "bf16", False), (64, 720, 4096, 512, "bf16", True),
    (100, 180, 256, 256, "f32", False), (96, 180, 256, 256, "f32", True),  # leftovers' own launch, none
])
def test_small_work(ctx, torch_dev, S, P, W, roi, storage, matrix):
    """Regions too small to pay for laying out whole rows, and stacks too small to pay for a launch of leftover
    slices, stay with the interpolating kernel (f16: the one with half staging, as before)."""
    import torch
    x = _stack(torch_dev, S, P, W, storage, seed=14)
    props = dict(roi_x=(W - roi) // 2, roi_y=(W - roi) // 3, roi_width=roi, roi_height=roi)
    got, ref = _both(ctx, torch_dev, x, storage, **props)
    if storage == "f16" and not matrix:
        try:
            ctx.bp_configure(8, 8, 0)
            ctx.bp_parallel(x, W, P, ref, n_slices=S, dtype=ufomi.F16, **props)
        finally:
            ctx.bp_configure(0, 0, 0)
    assert torch.equal(got, ref) != matrix
    # float32 coordinates of the interpolating kernel: 2^-14 pixels at 1024 to 2048, the samples' difference is
    # 1.4 of their size and one of two roundings counts
    assert rel_l2(got.cpu().numpy(), ref.cpu().numpy()) < 2.0 ** -14


@pytest.mark.parametrize("S,P,W,roi,matrix", [
    (12, 65532, 16, 36, True),     # the largest angle count, rounded up to fours, of the layout's grid
    (12, 65533, 16, 36, False),
    (12, 70001, 16, 36, False),
    (65504, 16, 8, 32, True),      # the most slices of one chunk
    (65600, 16, 8, 32, True),      # and the first that take two
])
def test_launch_limits(ctx, torch_dev, S, P, W, roi, matrix):
    """A grid's second axis holds 65535 blocks: more slices go in chunks, more angles to the interpolating kernel."""
    import torch
    x = _stack(torch_dev, S, P, W, seed=13)
    got, ref = _both(ctx, torch_dev, x, roi_width=roi, roi_height=roi)
    assert torch.equal(got, ref) != matrix
    assert bool(torch.isfinite(got).all())
    err = (got - ref).double().norm(dim=(1, 2)) / ref.double().norm(dim=(1, 2))
    # float32 sums of P terms of order 1: both round at up to 2^-24 of the partial sums, whose size is that of
    # the result (a random walk) -> P^0.5 roundings
    assert float(err.max()) < 1e-5 + 2.0 ** -24 * P ** 0.5
    if not matrix or S < 100:
        exact = oracle.bp_texture_f64(x[S // 2].cpu().numpy(), axis_pos=W / 2.0, roi_width=roi, roi_height=roi)
        assert rel_l2(got[S // 2].cpu().numpy(), exact) < 1e-5 + 2.0 ** -24 * P ** 0.5


def test_chunks_of_the_workspace(ctx, torch_dev):
    """Rows above 1 GiB go in chunks: two of 64 slices here, and one of 41 as units of 32 and 16 (padded).  An
    Inf leaves out the second chunk's unit and a large sample the third one's first: the interpolating kernel's
    bits are there, and nowhere else."""
    import torch
    S, P, W, roi = 169, 3000, 1300, 260
    x = torch.randn((S, P, W), device=torch_dev, generator=torch.Generator(device=torch_dev).manual_seed(15))
    x[70, 5, 600] = float("inf")
    x[150, 7, 650] = 1e20
    got, ref = _both(ctx, torch_dev, x, roi_x=520, roi_y=515, roi_width=roi, roi_height=roi - 3)
    finite = torch.isfinite(ref)
    assert bool((torch.isfinite(got) == finite).all())
    got[~finite] = ref[~finite] = 0.0
    for s in range(S):
        # coordinates of 1300 pixels round at up to 2^-14 pixels there, a fifth of that on average
        assert rel_l2(got[s].cpu().numpy(), ref[s].cpu().numpy()) < 2e-5, s
        assert torch.equal(got[s], ref[s]) == (64 <= s < 160), s


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
def test_nonfinite_values_stay_local(ctx, torch_dev, storage):
    """An Inf or a NaN reaches the pixels whose samples touch it and no others, whichever unit it is in."""
    import torch
    x = _stack(torch_dev, 105, 300, 300, storage, seed=7)
    x[3, 150, 140] = float("inf")
    x[70, 0, 1] = float("nan")
    x[100, 299, 299] = float("-inf")
    got, ref = _both(ctx, torch_dev, x, storage)
    assert bool((torch.isfinite(got) == torch.isfinite(ref)).all())
    assert bool((torch.isnan(got) == torch.isnan(ref)).all())
    m = torch.isfinite(ref)
    assert float((got[m] - ref[m]).norm() / ref[m].norm()) < 1e-5


def test_scales(ctx, torch_dev):
    """Slices of very different size each keep their precision, denormal and all-zero ones too."""
    import torch
    x = _stack(torch_dev, 16, 400, 400, seed=9)
    scale = [1.0, 1e-30, 1e30, 1e-20, 0.0, 65504.0, 1e-38, 3e-41, 2.0 ** -14, 1e10, 1e-5, 1e5, 1.0, 1e35, 1e-36, 7.0]
    x *= torch.tensor(scale, device=torch_dev)[:, None, None]
    got, ref = _both(ctx, torch_dev, x)
    got, ref = got.cpu().numpy().astype(np.float64), ref.cpu().numpy().astype(np.float64)
    for s, v in enumerate(scale):
        if v == 0.0:
            assert (got[s] == 0.0).all()
        elif v >= 1e-36:
            assert rel_l2(got[s], ref[s]) < 1e-5, v
        else:  # results near the smallest normal float: half a denormal step (7e-46) per addition at most
            assert np.abs(got[s] - ref[s]).max() < 400 * 1.5e-45, v


@pytest.mark.parametrize("scale", [1e9, 1e12, 1e25])
def test_small_columns_at_the_axis(ctx, torch_dev, scale):
    """Voxels at the axis see only the 8 of 700 detector columns there, a share of 1/88, whatever the others hold."""
    x = _stack(torch_dev, 16, 300, 700, seed=17)
    x[3, :, :346] *= scale
    x[3, :, 354:] *= scale
    got, ref = (t[:, 348:352, 348:352].double().cpu().numpy() for t in _both(ctx, torch_dev, x, axis_pos=350.0))
    for s in range(16):
        assert rel_l2(got[s], ref[s]) < 1e-5, s


@pytest.mark.parametrize("storage,hot", [("f32", 3e4), ("f32", 1e6), ("f32", 1e8), ("f32", 1e20), ("f32", 3e38),
                                         ("bf16", 1e9), ("bf16", 1e14), ("f16", 65504.0)])
def test_large_sample_stays_local(ctx, torch_dev, storage, hot):
    """One large finite sample (angle 0, first detector entry) reaches the first column of voxels and leaves the
    precision of the others, in its slice and in its neighbours, as the interpolating kernel has it.  f16 storage
    holds denormals beside its largest value."""
    x = _stack(torch_dev, 33, 300, 512, storage, seed=11)
    if storage == "f16":
        x *= 2.0 ** -20
    x[5, 0, 0] = hot
    x[32, 0, 0] = -hot
    got, ref = (t[:, :, 2:].double().cpu().numpy() for t in _both(ctx, torch_dev, x, storage))
    for s in range(33):
        assert rel_l2(got[s], ref[s]) < 1e-5, s


@pytest.mark.parametrize("hot,matrix", [(2.0 ** 20 * 1.5, True), (2.0 ** 22 * 1.5, False)])
def test_range_of_the_matrix_cores(ctx, torch_dev, hot, matrix):
    """Samples of size 1 to 2 beside one of 2^20 stay on the matrix cores: their floor is 2^-40 of 2^21 at most,
    2^-19 of a sample, and the errors of the 4 P samples of a voxel have random signs; beside 2^22 they leave."""
    import torch
    x = _stack(torch_dev, 64, 300, 400, seed=16)  # enough tiles that neither kernel splits the angles
    x = torch.sign(x) * (1.0 + x.abs() % 1.0)
    x[9, 0, 0] = hot
    got, ref = _both(ctx, torch_dev, x, axis_pos=200.0)
    assert torch.equal(got, ref) != matrix
    exact = oracle.bp_texture_f64(x[9].cpu().numpy(), axis_pos=200.0)[:, 2:]
    assert rel_l2(got[9, :, 2:].cpu().numpy(), exact) < 2.0 ** -19 + rel_l2(ref[9, :, 2:].cpu().numpy(), exact)


def test_small_part_beside_large(ctx, torch_dev):
    """Voxels that see only the quarter of the detector with samples of order 1, beside 1e12 elsewhere (angles
    up to 0.4, so the left edge of the upper half stays on that quarter)."""
    W = 512
    x = _stack(torch_dev, 16, 400, W, seed=12)
    x[3, :, W // 4:] *= 1e12
    got, ref = (t[:, :W // 2, :W // 8].double().cpu().numpy() for t in _both(ctx, torch_dev, x, angle_step=0.001))
    for s in range(16):
        assert rel_l2(got[s], ref[s]) < 1e-5, s


def test_streams_share_a_context(ctx, torch_dev):
    """Calls of one context on two streams in turn: the second waits for the first one's workspace.  Both have
    the same angles, whose table stays as it is (a new one frees the last, which waits for every stream)."""
    import torch
    a, b = _stack(torch_dev, 64, 400, 512, seed=1), _stack(torch_dev, 48, 400, 400, seed=2)
    oa, ob = torch.empty((64, 512, 512), device=torch_dev), torch.empty((48, 400, 400), device=torch_dev)
    ctx.bp_parallel(a, 512, 400, oa, n_slices=64)
    ctx.bp_parallel(b, 400, 400, ob, n_slices=48)
    torch.cuda.synchronize()
    ra, rb = oa.clone(), ob.clone()
    side = torch.cuda.Stream()
    main = torch.cuda.current_stream(0)
    side.wait_stream(main)
    try:
        for _ in range(4):
            oa.zero_()
            ob.zero_()
            torch.cuda.synchronize()
            ctx.set_stream(main)
            ctx.bp_parallel(a, 512, 400, oa, n_slices=64)
            ctx.set_stream(side)
            with torch.cuda.stream(side):
                ctx.bp_parallel(b, 400, 400, ob, n_slices=48)
            torch.cuda.synchronize()
            assert torch.equal(oa, ra) and torch.equal(ob, rb)
    finally:
        ctx.set_stream(main)
