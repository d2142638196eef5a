"""Edges of the vector widths and item runs of flat-field-correct and cone-beam-projection-weight:
4-pixel and single-pixel accesses, runs of 8 items (4 projections) and their remainders, dark and flat
streams that end inside a run, and unaligned buffers."""
import numpy as np
import pytest

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _dev(x, torch_dev, shift=0):
    """A device copy whose data starts `shift` floats into its allocation."""
    import torch
    x = np.ascontiguousarray(x, dtype=np.float32)
    flat = torch.empty(x.size + shift, device=torch_dev)
    flat[shift:].copy_(torch.from_numpy(x.ravel()))
    return flat[shift:].view(x.shape)


@pytest.mark.parametrize("n,h,w,shift", [(1, 3, 8, 0), (7, 5, 4, 0), (8, 2, 6, 0), (9, 1, 1028, 0), (17, 3, 5, 0),
                                         (9, 4, 16, 1), (20, 2, 2, 0),
                                         # runs of 2, 4 and 8 items need 1024 workgroups at least
                                         (2047, 1, 6, 0), (4095, 1, 4, 0), (8190, 1, 5, 0), (8185, 1, 4, 0)])
@pytest.mark.parametrize("sino,nd,nf", [(False, 1, 1), (False, 3, 10), (True, 12, 2), (True, 1, 1),
                                        (False, 4091, 8188)])
def test_flat_field_runs(ctx, torch_dev, n, h, w, shift, sino, nd, nf):
    rng = np.random.default_rng(n * 100 + w)
    nd, nf = min(nd, n), min(nf, n)
    data = rng.uniform(0.2, 1.0, (n, h, w)).astype(np.float32)
    shape = (1, w) if sino else (h, w)
    dark = rng.uniform(0.0, 0.1, (nd,) + shape).astype(np.float32)
    flat = rng.uniform(1.0, 1.2, (nf,) + shape).astype(np.float32)
    out = _dev(np.full((n, h, w), np.nan), torch_dev, shift)
    ctx.flat_field_correct(_dev(data, torch_dev, shift), w, h, n, _dev(dark, torch_dev), nd, _dev(flat, torch_dev), nf,
                           out, sinogram_input=sino, absorption_correct=True, dark_scale=0.5, flat_scale=1.5)
    got = out.cpu().numpy()
    assert np.isfinite(got).all()
    for i in range(n) if n < 100 else [*range(20), *range(max(nd - 9, 0), min(nd + 9, n)), *range(n - 20, n)]:
        ref = oracle.flat_field_correct_ref32(data[i:i + 1], dark[min(i, nd - 1)], flat[min(i, nf - 1)], True, False,
                                              False, 0.5, 1.5)[0]
        assert rel_l2(got[i], ref) < 1e-6, i  # one rounding of logf (2 ulp) over the oracle's


@pytest.mark.parametrize("p,h,w,shift", [(1, 2, 4, 0), (4, 3, 260, 0), (5, 5, 62, 0), (9, 4, 8, 2), (6, 2, 7, 0)])
@pytest.mark.parametrize("per_projection", [False, True])
def test_cone_weight_runs(ctx, torch_dev, p, h, w, shift, per_projection):
    rng = np.random.default_rng(p + w)
    x = rng.uniform(0.5, 2.0, (p, h, w)).astype(np.float32)
    cx = list(w / 2.0 + 0.25 * np.arange(p)) if per_projection else w / 2.0
    sod = list(300.0 + np.arange(p)) if per_projection else 300.0
    out = _dev(np.full((p, h, w), np.nan), torch_dev, shift)
    ctx.cone_weight(_dev(x, torch_dev, shift), out, w, h, p, cx, h / 2.0, sod, 500.0, 0.0)
    got = out.cpu().numpy()
    for i in range(p):
        ref = oracle.cone_weight_ref32(x[i], cx[i] if per_projection else cx, h / 2.0,
                                       sod[i] if per_projection else sod, 500.0, 0.0)
        np.testing.assert_allclose(got[i], ref, rtol=2e-6)
