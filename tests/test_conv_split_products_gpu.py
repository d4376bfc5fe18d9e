"""The fp32 LDS-staged GEMM's part products (three bf16 parts per operand, six products): each product must
hold fp32's precision at the operands' own exponents, and a result that is not finite must be the fp32
convolution's.

The float64 bar is elementwise, derived from the method: per product the dropped parts and the roundings of
the parts are below 2^-23 of |a w|, and the sum rounds once per 16 channels and part product, each rounding at
most 2^-24 of the largest partial sum: |error| <= (2 + 6 * 27 * cin / 16) * 2^-24 * sum |a w|.  Random rounding
errors grow with the square root of their number, so the bar used is (2 + sqrt(6 * 27 * cin / 16)) times
4 * 2^-24 -- four standard deviations."""

from __future__ import annotations


import numpy as np
import pytest
import torch

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
    err = (y.cpu().double() - _conv64(x, w)).abs()
    assert bool((err <= _bar(x, w)).all()), f"{name}: {(err / _bar(x, w)).max():.2f} of the bar"


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
