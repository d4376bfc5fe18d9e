"""The part products (three bf16 parts per operand, six products) of the fp32 LDS-staged and register-streaming
GEMMs: each product must hold fp32's precision at the operands' own exponents, and a result that is not finite
must be the fp32 convolution's.

Two float64 bars.  Elementwise, for every result, derived from the method: per product the dropped parts and the
roundings of the parts are below 2^-23 of |a w|, and the sum rounds once per 16 channels and part product, each
rounding at most 2^-24 of the largest partial sum: |error| <= (2 + 6 * 27 * cin / 16) * 2^-24 * sum |a w|.  Random
rounding errors grow with the square root of their number, so the bar used is (2 + sqrt(6 * 27 * cin / 16)) times
4 * 2^-24 -- four standard deviations.  It holds single results, and is too wide to see a lost part product; the
root mean square of ``part_products`` sees that."""

from __future__ import annotations


import numpy as np
import pytest
import torch

from part_products import RMS_BAR, normalised_rms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev(ctmr):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda")


def _conv64(x, w, pad=1):
    """Float64 3x3x3 convolution of NDHWC ``x`` on the CPU."""
    y = torch.nn.functional.conv3d(x.double().permute(0, 4, 1, 2, 3), w.double(), padding=pad)
    return y.permute(0, 2, 3, 4, 1)


def _bar(x, w):
    cin = int(x.shape[-1])
    return (2 + np.sqrt(6 * 27 * cin / 16)) * 4 * 2.0 ** -24 * _conv64(x.abs(), w.abs())


# (name, shape, second source's channels, cout, split)
CASES = [
    ("one full brick", (1, 4, 8, 8, 64), 0, 64, 1),
    ("ragged bricks", (2, 7, 15, 15, 80), 0, 64, 1),
    ("two column tiles", (1, 4, 8, 16, 64), 0, 128, 1),
    ("two sources", (1, 7, 8, 15, 64), 48, 64, 1),
    ("two wave sets", (1, 4, 16, 16, 128), 0, 64, 2),
    ("two sources, partial planes", (1, 4, 8, 8, 128), 112, 64, 3),
    ("32 outputs", (1, 4, 8, 16, 32), 0, 32, 1),
    ("32 outputs, ragged bricks, odd chunks", (2, 7, 15, 15, 48), 0, 32, 1),
]


@pytest.mark.parametrize(("name", "shape", "c2", "cout", "split"), CASES, ids=[c[0] for c in CASES])
def test_products_hold_fp32_at_every_scale(ctmr, dev, name, shape, c2, cout, split):
    """Channels of 2^-40 .. 2^40 against weights of the inverse scales: each product keeps its own precision."""
    f, L, ops = ctmr.fast_fp32, ctmr._lib, ctmr.ops
    g = torch.Generator().manual_seed(7)
    cin = shape[-1] + c2
    scale = torch.exp2(torch.randint(-40, 41, (cin,), generator=g).float())
    x = torch.randn(*shape[:-1], cin, generator=g) * scale
    w = torch.randn(cout, cin, 3, 3, 3, generator=g) / scale.reshape(1, -1, 1, 1, 1)
    first = x[..., :shape[-1]].contiguous().to(dev)
    xin = f.ChannelCat(first, x[..., shape[-1]:].contiguous().to(dev)) if c2 else first
    assert L.conv_kernel(ops.make_desc(tuple(shape), cout, 3, 1, 0, 0, L.DT_F32, split, c2)) == "lds"
    y = f.implicit_gemm_conv3d(xin, f.pack_weight(w.to(dev), dtype="fp32"), None, cout=cout, split=split)
    ref = _conv64(x, w)
    err = (y.cpu().double() - ref).abs()
    assert bool((err <= _bar(x, w)).all()), f"{name}: {(err / _bar(x, w)).max():.2f} of the bar"
    rms = normalised_rms(y.cpu(), ref, _conv64(x.double() ** 2, w.double() ** 2).sqrt())
    print(f"{name}: {rms:.2e}", flush=True)
    assert rms <= RMS_BAR


@pytest.mark.parametrize(("name", "shape", "c2", "cout", "split"), CASES, ids=[c[0] for c in CASES])
def test_results_that_are_not_finite(ctmr, dev, name, shape, c2, cout, split):
    """Infinities, NaN and values past bf16's largest in the input, an infinite weight: the fp32 pattern."""
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(11)
    cin, (n, d, h, wd) = shape[-1] + c2, shape[:-1]
    x, w = torch.randn(*shape[:-1], cin, generator=g), torch.randn(cout, cin, 3, 3, 3, generator=g) * 0.02
    x[0, 0, 0, 0, 3] = float("inf")
    x[n - 1, d - 1, h - 1, wd - 1, cin - 1] = float("-inf")
    x[0, 2, h - 2, 1, 5] = float("nan")
    x[0, d - 1, 0, wd - 1, 9] = 3.402e38  # rounds to infinity in bf16; finite here
    w[1, 2, 1, 1, 1] = float("inf")
    first = x[..., :shape[-1]].contiguous().to(dev)
    xin = f.ChannelCat(first, x[..., shape[-1]:].contiguous().to(dev)) if c2 else first
    y = f.implicit_gemm_conv3d(xin, f.pack_weight(w.to(dev), dtype="fp32"), None, cout=cout, split=split).cpu()
    ref = _conv64(x, w)
    # a sum in fp32 may overflow only where the float64 one passes fp32's range
    ref = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * float("inf"), ref)
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isposinf(), ref.isposinf())
    assert torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    xa, wa = torch.nan_to_num(x.abs(), 0.0, 0.0, 0.0), torch.nan_to_num(w.abs(), 0.0, 0.0, 0.0)
    # the recomputed results round once per product: 27 * cin fp32 steps
    bar = _bar(xa, wa) + np.sqrt(27 * cin) * 4 * 2.0 ** -24 * _conv64(xa, wa)
    assert bool(((y.double() - ref).abs() <= bar)[ok].all())
    assert bool((~ok).any()) and bool(ok.any())


def test_not_finite_through_the_norm_and_silu(ctmr, dev):
    """The staging transform of a recomputed result: one NaN voxel taints its 27 neighbours and nothing else."""
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(1, 4, 8, 8, 64, generator=g), torch.randn(64, 64, 3, 3, 3, generator=g) * 0.02
    affine = torch.stack([torch.rand(1, 64, generator=g) + 0.5, torch.randn(1, 64, generator=g)], dim=-1)
    x[0, 1, 3, 3, 7] = float("nan")
    y = f.implicit_gemm_conv3d(x.to(dev), f.pack_weight(w.to(dev), dtype="fp32"), None, cout=64,
                               affine=affine.to(dev), silu=True).cpu()
    taint = torch.zeros(1, 4, 8, 8, dtype=torch.bool)
    taint[0, 0:3, 2:5, 2:5] = True
    assert torch.equal(y.isnan().all(-1), taint) and torch.equal(y.isnan().any(-1), taint)


@pytest.mark.parametrize("groups", [1, 4, 32])
def test_statistics_of_32_outputs(ctmr, dev, groups):
    """The epilogue's group-norm partials of the 32-column form, with bias, residual, affine and SiLU."""
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(2, 7, 15, 16, 32, generator=g), torch.randn(32, 32, 3, 3, 3, generator=g) * 0.05
    bias, res = torch.randn(2, 32, generator=g), torch.randn(2, 7, 15, 16, 32, generator=g)
    affine = torch.stack([torch.rand(2, 32, generator=g) + 0.5, torch.randn(2, 32, generator=g)], dim=-1)
    a = affine[:, None, None, None]
    src = torch.nn.functional.silu(x.double() * a[..., 0] + a[..., 1])
    y = f.implicit_gemm_conv3d(x.to(dev), f.pack_weight(w.to(dev), dtype="fp32"), bias.to(dev), cout=32,
                               affine=affine.to(dev), silu=True, residual=res.to(dev), split=1, gn_groups=groups)
    ref = _conv64(src, w) + bias.double().reshape(2, 1, 1, 1, 32) + res.double()
    # SiLU within 1e-6, bias and residual one rounding each
    bar = _bar(src, w) + 1e-6 * _conv64(src.abs(), w.abs()) + 2.0 ** -23 * ref.abs()
    assert bool(((y.cpu().double() - ref).abs() <= bar).all())
    st = f.conv_output_stats(y, groups).cpu().sum(1)
    yy = y.cpu().double().reshape(2, -1, groups, 32 // groups)
    want = torch.stack([yy.sum((1, 3)), (yy * yy).sum((1, 3))], -1)
    # float64 sums of under 2^16 values in another order
    assert torch.allclose(st, want, rtol=1e-11, atol=1e-11 * float((yy * yy).sum()))


# The register-streaming GEMM (whole pairs of 16-channel blocks; an odd block count stays on FP32 MFMA):
# (name, shape, cout, options, kernel)
STREAM_CASES = [
    ("direct reads, one tile", (1, 3, 4, 5, 64), 64, {"stream_gemm": True, "split": 1}, "stream_direct"),
    ("direct, remainder rows and columns", (2, 5, 7, 9, 32), 48, {"stream_gemm": True, "split": 1}, "stream_direct"),
    ("two 16-column blocks", (1, 6, 9, 11, 32), 32, {"split": 1}, "stream_direct"),
    ("128-wide tiles, odd split of the steps", (1, 5, 6, 7, 96), 128, {"split": 7}, "stream_direct"),
    ("an odd block count", (1, 5, 6, 7, 48), 64, {"split": 1}, "stream_direct"),
    ("stride 2, ragged", (1, 7, 9, 10, 64), 96, {"stride": 2, "split": 1}, "stream_direct"),
    ("packed copy", (1, 4, 5, 6, 64), 64, {"stream_gemm": True, "split": 2, "silu": True}, "stream"),
    ("nearest-2x", (1, 3, 4, 5, 64), 64, {"upsample": True, "split": 1}, "stream"),
    ("nearest-2x, 128-wide", (2, 3, 5, 4, 128), 128, {"upsample": True}, "split_waves"),
    ("trilinear-2x", (1, 3, 4, 5, 64), 64, {"trilinear": True, "split": 1}, "stream"),
    ("split over four waves", (2, 8, 8, 4, 128), 128, {}, "split_waves"),
    ("split over four waves, two sets", (1, 18, 21, 11, 256), 256, {}, "split_waves"),
]


def _stream_conv(ctmr, dev, x, w, cout, options, kernel):
    """The op on the named route, and the float64 result with its bar (of |x|, |w|)."""
    f, L, ops = ctmr.fast_fp32, ctmr._lib, ctmr.ops
    opts = dict(options)
    mode = (L.MODE_NEAREST2X if opts.get("upsample") else L.MODE_TRILINEAR2X if opts.get("trilinear")
            else L.MODE_PLAIN)
    flags = (L.F_STREAM if opts.get("stream_gemm") else 0) | (L.F_SILU if opts.get("silu") else 0)
    desc = ops.make_desc(tuple(x.shape), cout, 3, opts.get("stride", 1), mode, flags, L.DT_F32, opts.get("split", 0))
    assert L.conv_kernel(desc) == kernel
    packed = (f.pack_upsample_weight if opts.get("upsample") else f.pack_weight)(w.to(dev), dtype="fp32")
    y = f.implicit_gemm_conv3d(x.to(dev), packed, None, cout=cout, **opts).cpu()
    xd = x.double()
    if opts.get("silu"):
        xd = xd * torch.sigmoid(xd)
    if opts.get("upsample"):
        for axis in (1, 2, 3):
            xd = xd.repeat_interleave(2, axis)
    if opts.get("trilinear"):
        xd = torch.nn.functional.interpolate(xd.permute(0, 4, 1, 2, 3), scale_factor=2, mode="trilinear",
                                             align_corners=False).permute(0, 2, 3, 4, 1)
    st = opts.get("stride", 1)
    sub = (slice(None), *(slice(None, None, st),) * 3)
    # the staging transform and the parity fold round once more each: 2e-6 of the operands together
    return y, _conv64(xd, w)[sub], lambda a, b: (_bar(a, b) + 2e-6 * _conv64(a.abs(), b.abs()))[sub], xd


@pytest.mark.parametrize(("name", "shape", "cout", "options", "kernel"), STREAM_CASES, ids=[c[0] for c in STREAM_CASES])
def test_streaming_products_hold_fp32(ctmr, dev, name, shape, cout, options, kernel):
    g = torch.Generator().manual_seed(23)
    wide = 0 if options.get("silu") else 30
    scale = torch.exp2(torch.randint(-wide, wide + 1, (shape[-1],), generator=g).float())
    x = torch.randn(*shape, generator=g) * scale
    w = torch.randn(cout, shape[-1], 3, 3, 3, generator=g) / scale.reshape(1, -1, 1, 1, 1)
    y, ref, bar, xd = _stream_conv(ctmr, dev, x, w, cout, options, kernel)
    err, limit = (y.double() - ref).abs(), bar(xd, w)
    assert bool((err <= limit).all()), f"{name}: {(err / limit).max():.2f} of the bar"
    st = options.get("stride", 1)
    size = _conv64(xd ** 2, w.double() ** 2)[(slice(None), *(slice(None, None, st),) * 3)].sqrt()
    rms = normalised_rms(y, ref, size)
    print(f"{name}: {rms:.2e}", flush=True)
    assert rms <= RMS_BAR


@pytest.mark.parametrize(("name", "shape", "cout", "options", "kernel"),
                         [c for c in STREAM_CASES if not c[3].get("trilinear")],
                         ids=[c[0] for c in STREAM_CASES if not c[3].get("trilinear")])
def test_streaming_results_that_are_not_finite(ctmr, dev, name, shape, cout, options, kernel):
    g = torch.Generator().manual_seed(29)
    x, w = torch.randn(*shape, generator=g), torch.randn(cout, shape[-1], 3, 3, 3, generator=g) * 0.02
    n, d, h, wd, c = shape
    x[n - 1, d - 1, h - 1, wd - 1, c - 1] = float("nan")
    if not options.get("silu"):  # the staged SiLU itself turns these into NaN
        x[0, 0, 0, 0, 3] = float("inf")
        x[0, d - 1, 0, wd - 1, 9] = 3.402e38  # rounds to infinity in bf16; finite here
    y, ref, bar, xd = _stream_conv(ctmr, dev, x, w, cout, options, kernel)
    ref = torch.where(ref.abs() > 3.4028235e38, torch.sign(ref) * float("inf"), ref)
    if options.get("upsample"):  # the parity fold adds weights before they meet an infinity
        assert torch.equal(y.isfinite(), ref.isfinite())
    else:
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isposinf(), ref.isposinf())
        assert torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    xa = torch.nan_to_num(xd.abs(), 0.0, 0.0, 0.0)
    limit = bar(xa, w) + np.sqrt(27 * c) * 4 * 2.0 ** -24 * ref.abs().nan_to_num(0.0, 0.0, 0.0).clamp(min=1e-3)
    assert bool(((y.double() - ref).abs() <= limit)[ok].all()) and bool((~ok).any())
