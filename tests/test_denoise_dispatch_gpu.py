"""The convolutions' and reductions' kernels at the sizes where their dispatch changes,
against the float64 oracle on bf16-rounded inputs (tolerances as in
tests/test_denoise_gpu.py: 2^-8 relative for a bf16 output, 1e-4 for float32 sums)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import conv_ref as cr
from tests.test_denoise_gpu import _bf, _close_bf16, _cm, _dev, _np, _rounded, dn  # noqa: F401

pytestmark = pytest.mark.gpu


# Weight gradients: rows of 64, 32 and 16 in whole tiles (several per split, one, and
# fewer tiles than splits: some partials are zeros), a tile height that does not divide h
# and short rows (the general kernel), with position counts off the splits' multiples.
@pytest.mark.parametrize("shape, cin, cout, splits", [
    ((1, 2, 4, 64), 16, 16, 1), ((1, 5, 8, 64), 16, 32, 3), ((2, 3, 4, 64), 32, 16, 16),
    ((1, 1, 8, 32), 16, 16, 1), ((2, 3, 16, 32), 32, 32, 5), ((1, 3, 16, 16), 64, 16, 2),
    ((2, 2, 32, 16), 16, 48, 7), ((1, 3, 6, 64), 16, 16, 4), ((1, 5, 8, 8), 16, 32, 3),
])
def test_weight_gradient_tiles(dn, shape, cin, cout, splits):  # noqa: F811
    import torch

    rng = np.random.default_rng(cin + cout + splits)
    n, d, h, w = shape
    x, dz = _rounded(rng.standard_normal(shape + (cin,))), _rounded(rng.standard_normal(shape + (cout,)))
    x_cm, dz_cm = _cm(_dev(_bf(x)), cin), _cm(_dev(_bf(dz)), cout)
    part = torch.full((splits, 27, cout, cin), float("nan"), dtype=torch.float32, device="cuda:0")
    gw = torch.empty((27, cout, cin), dtype=torch.float32, device="cuda:0")
    dn._call("hdn_conv3d_wgrad", x_cm.data_ptr(), dz_cm.data_ptr(), part.data_ptr(), splits, n, d, h, w, cin, cout,
             None)
    dn._call("hdn_reduce_splits", part.data_ptr(), gw.data_ptr(), gw.numel(), splits, None)
    ref = cr.conv_wgrad(x, dz)
    np.testing.assert_allclose(_np(gw), ref, rtol=1e-4, atol=1e-4 * np.abs(ref).max())


# Forward convolutions by wave count: single tiles, 2 x 2 tiles (whole and partly filled last
# workgroups) and, from 512 waves on, 64-position waves; taps shared by a k-step's lanes
# (input channels in whole 32s) and not; an output channel count off the pairs.
@pytest.mark.parametrize("shape, cin, cout", [
    ((1, 1, 4, 16), 128, 128), ((3, 5, 8, 8), 128, 64), ((1, 8, 8, 8), 16, 48), ((127, 1, 8, 8), 32, 32),
    ((16, 8, 8, 8), 64, 64), ((43, 3, 8, 8), 16, 32), ((25, 3, 8, 8), 32, 48),
    ((7, 73, 8, 8), 16, 16), ((8, 16, 16, 16), 16, 16),
])
def test_forward_by_wave_count(dn, shape, cin, cout):  # noqa: F811
    import torch

    rng = np.random.default_rng(cin + cout)
    n, d, h, w = shape
    x = _rounded(rng.standard_normal(shape + (cin,)))
    master = rng.standard_normal((27, cout, cin)).astype(np.float32) * 0.1
    bias = rng.standard_normal(cout).astype(np.float32)
    wq = _rounded(master)
    xd, wf, bd = _dev(_bf(x)), _dev(_bf(wq)), _dev(torch.from_numpy(bias))
    y = torch.empty(shape + (cout,), dtype=torch.bfloat16, device="cuda:0")
    y_cm = torch.empty((cout, n * d * h * w), dtype=torch.bfloat16, device="cuda:0")
    dn._call("hdn_conv3d_fwd", xd.data_ptr(), wf.data_ptr(), bd.data_ptr(), y.data_ptr(), y_cm.data_ptr(), n, d, h, w,
             cin, cout, 0.1, None)
    _close_bf16(_np(y), cr.leaky(cr.conv_fwd(x, wq, bias.astype(np.float64)), 0.1))
    np.testing.assert_array_equal(_np(y_cm), _np(y).reshape(-1, cout).T)


# Full-resolution rows of each channel pair: one slice to a workgroup (16 -> 16) or a tile
# (with 32), and from 3 slices a CU on two slices to a workgroup with a last one of one; the
# other kernels' shapes for the fused steps.
MARCHED = [((1, 1, 4, 64), 16, 16), ((2, 6, 4, 64), 16, 32), ((1, 7, 8, 64), 32, 16), ((1, 20, 4, 64), 16, 16),
           ((11, 7, 44, 64), 16, 16), ((6, 17, 32, 64), 16, 32), ((6, 17, 32, 64), 32, 16)]


@pytest.mark.parametrize("shape, cin, cout", MARCHED)
def test_forward_marched(dn, shape, cin, cout):  # noqa: F811
    test_forward_by_wave_count(dn, shape, cin, cout)


# An infinite activation gives the infinities that the oracle gives, in every build of the
# marching kernel and in the others: what pads the last k-step past the 27 taps multiplies
# zeros. (Positive weights: no sum meets infinities of both signs.)
@pytest.mark.parametrize("src", (0, 1, 3))
@pytest.mark.parametrize("shape, cin, cout", MARCHED + [((1, 2, 8, 32), 16, 32), ((1, 2, 4, 16), 16, 16),
                                                        ((9, 16, 16, 16), 16, 16)])
def test_an_infinity_stays_an_infinity(dn, shape, cin, cout, src):  # noqa: F811
    import torch

    n, d, h, w = shape
    d += d % 2 if src == 1 else 0
    rng = np.random.default_rng(cin + cout + src)
    x = _rounded(rng.random((n, d, h, w, cin)))
    if src == 1:
        x = x[:, ::2, ::2, ::2].copy()
    if src == 3:
        x[..., 8:] = 0.0
    x[0, 0, 0, 0, 3] = x[-1, -1, -1, -1, 5] = x[n // 2, x.shape[1] // 2, x.shape[2] // 2, x.shape[3] // 2, 0] = np.inf
    wq = _rounded(rng.uniform(0.1, 1.0, (27, cout, cin)).astype(np.float32))
    y = torch.empty((n, d, h, w, cout), dtype=torch.bfloat16, device="cuda:0")
    xd, wd = _dev(_bf(x)), _dev(_bf(wq))
    dn._call("hdn_conv3d_fwd_src", xd.data_ptr(), None, src, wd.data_ptr(), None, y.data_ptr(), None, n, d, h, w, cin,
             cout, 0.1, None)
    full = x.repeat(2, axis=1).repeat(2, axis=2).repeat(2, axis=3) if src == 1 else x
    want, got = cr.conv_fwd(full, wq), _np(y)
    assert np.isinf(want).any() and not np.isnan(want).any()
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    _close_bf16(got[finite], want[finite])


@pytest.mark.parametrize("shape, cin, cout", MARCHED[1:] + [((1, 2, 8, 32), 32, 32), ((1, 2, 8, 32), 64, 32),
                                                            ((1, 2, 4, 16), 64, 64), ((2, 16, 16, 16), 64, 64),
                                                            ((3, 16, 32, 32), 16, 16)])
@pytest.mark.parametrize("upsampled", (False, True))
def test_fused_steps_equal_separate_calls(dn, shape, cin, cout, upsampled):  # noqa: F811
    """The skip addition and the prediction made in a convolution's store, against hdn_add
    and hdn_loss on its stored output, bit for bit."""
    import torch

    n, d, h, w = shape
    d -= d % 2 if upsampled else 0
    shape = (n, d, h, w)
    P = n * d * h * w
    rng = np.random.default_rng(cin)
    src = (n, d // 2, h // 2, w // 2) if upsampled else shape
    x = _dev(_bf(rng.standard_normal(src + (cin,))))
    wt = _dev(_bf(rng.standard_normal((27, cout, cin)) * 0.1))
    bias = _dev(torch.from_numpy(rng.standard_normal(cout).astype(np.float32)))
    skip = _dev(_bf(rng.standard_normal(shape + (cout,))))
    y, want, got = (torch.zeros(shape + (cout,), dtype=torch.bfloat16, device="cuda:0") for _ in range(3))
    args = (n, d, h, w, cin, cout, 0.1, None)

    def fused(skip_ptr, inp, c_in, pred, out):
        dn._call("hdn_conv3d_fwd_fused", x.data_ptr(), None, int(upsampled), wt.data_ptr(), bias.data_ptr(), skip_ptr,
                 inp, c_in, pred, out, None, *args)

    dn._call("hdn_conv3d_fwd_src", x.data_ptr(), None, int(upsampled), wt.data_ptr(), bias.data_ptr(), y.data_ptr(),
             None, *args)
    dn._call("hdn_add", y.data_ptr(), skip.data_ptr(), want.data_ptr(), None, P, cout, None)
    fused(skip.data_ptr(), None, 0, None, got.data_ptr())
    assert torch.equal(got, want)
    pred, ref = (torch.zeros(P, device="cuda:0") for _ in range(2))
    if upsampled:
        with pytest.raises(ValueError):
            fused(None, skip.data_ptr(), cout, pred.data_ptr(), None)
        return
    dn._call("hdn_loss", y.data_ptr(), skip.data_ptr(), cout, cout, None, None, None, None, ref.data_ptr(), None, P,
             1.0, None)
    fused(None, skip.data_ptr(), cout, pred.data_ptr(), None)
    assert torch.equal(pred, ref)


@pytest.mark.parametrize("shape, cin, cout", MARCHED + [
    ((1, 2, 8, 32), 32, 32), ((1, 2, 8, 32), 64, 32),  # staged tiles
    ((1, 2, 4, 16), 64, 64), ((1, 8, 8, 8), 16, 48), ((16, 8, 8, 8), 64, 64), ((48, 8, 8, 8), 16, 32),  # small waves
    ((9, 16, 16, 16), 16, 16),  # 64-position waves
])
def test_added_input_equals_a_separate_addition(dn, shape, cin, cout):  # noqa: F811
    """src 2 (x + x2 read as the input) against hdn_add and src 0, bit for bit, in every
    forward kernel; no part of the network reads its input so any more."""
    import torch

    n, d, h, w = shape
    P = n * d * h * w
    rng = np.random.default_rng(cin + cout)
    x, x2 = (_dev(_bf(rng.standard_normal(shape + (cin,)))) for _ in range(2))
    wt = _dev(_bf(rng.standard_normal((27, cout, cin)) * 0.1))
    bias = _dev(torch.from_numpy(rng.standard_normal(cout).astype(np.float32)))
    added = torch.empty_like(x)
    want, got = (torch.zeros(shape + (cout,), dtype=torch.bfloat16, device="cuda:0") for _ in range(2))
    want_cm, got_cm = (torch.zeros((cout, P), dtype=torch.bfloat16, device="cuda:0") for _ in range(2))
    args = (n, d, h, w, cin, cout, 0.1, None)
    dn._call("hdn_add", x.data_ptr(), x2.data_ptr(), added.data_ptr(), None, P, cin, None)
    dn._call("hdn_conv3d_fwd", added.data_ptr(), wt.data_ptr(), bias.data_ptr(), want.data_ptr(), want_cm.data_ptr(),
             *args)
    dn._call("hdn_conv3d_fwd_src", x.data_ptr(), x2.data_ptr(), 2, wt.data_ptr(), bias.data_ptr(), got.data_ptr(),
             got_cm.data_ptr(), *args)
    assert torch.equal(got, want) and torch.equal(got_cm, want_cm)
    assert torch.count_nonzero(want.float()) > 0


@pytest.mark.parametrize("cin, cout", [(16, 16), (16, 32), (32, 16)])
@pytest.mark.parametrize("src", (0, 1, 2, 3))
def test_volumes_of_a_batch_equal_volumes_alone(dn, cin, cout, src):  # noqa: F811
    """Sixteen volumes of 21 (20 upsampled) slices march 6 to 11 slices to a workgroup, one
    alone takes a workgroup or tile per slice: the same bits, with and without a skip."""
    import torch

    n, d, h, w = 16, 20 if src == 1 else 21, 64, 64
    rng = np.random.default_rng(cin + src)
    dims = (d // 2, h // 2, w // 2) if src == 1 else (d, h, w)
    x, x2 = (_dev(_bf(rng.standard_normal((n,) + dims + (cin,), dtype=np.float32))) for _ in range(2))
    if src == 3:
        x[..., 8:] = 0
    wt, bias = _dev(_bf(rng.standard_normal((27, cout, cin)) * 0.1)), _dev(torch.zeros(cout))
    skip = _dev(_bf(rng.standard_normal((n, d, h, w, cout), dtype=np.float32)))
    for with_skip in (False, True) if src < 2 else (False,):
        batch, alone = (torch.zeros_like(skip) for _ in range(2))

        def call(y, first, count):
            dn._call("hdn_conv3d_fwd_fused", x[first].data_ptr(), x2[first].data_ptr() if src == 2 else None, src,
                     wt.data_ptr(), bias.data_ptr(), skip[first].data_ptr() if with_skip else None, None, 0, None,
                     y[first].data_ptr(), None, count, d, h, w, cin, cout, 0.1, None)

        call(batch, 0, n)
        for i in range(n):
            call(alone, i, 1)
        assert torch.equal(batch, alone)
        assert torch.count_nonzero(batch.float()) > 0


@pytest.mark.parametrize("splits, length", [(1, 5), (16, 64), (17, 65), (700, 6912), (1, 16383), (3, 16384), (5, 16385),
                                            (255, 20_000), (256, 20_000)])
def test_reduce_splits(dn, splits, length):  # noqa: F811
    import torch

    part = torch.rand((splits, length), device="cuda:0")
    out = torch.empty(length, device="cuda:0")
    dn._call("hdn_reduce_splits", part.data_ptr(), out.data_ptr(), length, splits, None)
    # float32 sums of positive terms: at most one rounding of each partial sum per term
    np.testing.assert_allclose(_np(out), part.double().sum(dim=0).cpu().numpy(), rtol=(splits + 1) * 2.0 ** -24)
