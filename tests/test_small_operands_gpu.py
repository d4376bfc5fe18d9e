"""Operands near the lower end of fp32's range on the kernels that multiply in bf16 parts: a part below 2^-126 is a
bf16 subnormal, so an operand below 2^-110 would lose bits of its 24 (1.5e-5 of it at 2^-118, 6e-4 at 2^-124).

The bar is the one for operands of ordinary size: relative to the 2-norm, fp32 sums of up to 2000 products stay
within 2e-6 of float64 (measured 2e-7 .. 6e-7).  At 2^-124 a third of the operands are fp32 subnormals."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

CONVS = [
    ("LDS-staged GEMM", (1, 8, 8, 8, 64), 64, {"split": 1}, "lds"),
    ("two wave sets", (1, 4, 16, 16, 64), 64, {"split": 2}, "lds"),
    ("32 outputs", (1, 4, 8, 16, 32), 32, {"split": 1}, "lds"),
    ("direct reads", (1, 4, 5, 6, 64), 64, {"stream_gemm": True, "split": 1}, "stream_direct"),
    ("split over four waves", (2, 8, 8, 4, 128), 128, {}, "split_waves"),
    ("8 -> 8 plane by plane", (1, 16, 128, 160, 8), 8, {}, "march"),
    ("8 -> 32 plane by plane", (1, 40, 64, 128, 8), 32, {"stride": 2}, "march"),
]


@pytest.mark.parametrize("side", ["input", "weight"])
@pytest.mark.parametrize("exponent", [-108, -112, -118, -124])
@pytest.mark.parametrize(("name", "shape", "cout", "options", "kernel"), CONVS, ids=[c[0] for c in CONVS])
def test_conv(ctmr, dev, name, shape, cout, options, kernel, exponent, side):
    f, L = ctmr.fast_fp32, ctmr._lib
    g = torch.Generator().manual_seed(1)
    small = lambda *s: (torch.randn(*s, generator=g).double() * 2.0 ** exponent).float()
    plain = lambda *s: torch.randn(*s, generator=g)
    x = (small if side == "input" else plain)(*shape)
    w = (plain if side == "input" else small)(cout, shape[-1], 3, 3, 3)
    stride = options.get("stride", 1)
    flags = L.F_STREAM if options.get("stream_gemm") else 0
    assert L.conv_kernel(ctmr.ops.make_desc(shape, cout, 3, stride, L.MODE_PLAIN, flags, L.DT_F32,
                                            options.get("split", 0))) == kernel
    y = f.implicit_gemm_conv3d(x.to(dev), f.pack_weight(w.to(dev)), None, cout=cout, **options).cpu().double()
    ref = torch.nn.functional.conv3d(x.double().permute(0, 4, 1, 2, 3), w.double(), padding=1,
                                     stride=stride).permute(0, 2, 3, 4, 1)
    err = float((y - ref).norm() / ref.norm())
    print(f"{name} at 2^{exponent}: {err:.2e}", flush=True)
    assert err <= 2e-6


@pytest.mark.parametrize("exponent", [-108, -112, -118, -124])
@pytest.mark.parametrize("tokens", [60, 256, 700])
def test_attention_values(ctmr, dev, tokens, exponent):
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn(1, tokens, 64, generator=g) for _ in range(3))
    v = (v.double() * 2.0 ** exponent).float()
    y = f.flash_attention(q.to(dev), k.to(dev), v.to(dev), heads=2, scale=0.17).cpu().double()
    split = lambda t: t.double().reshape(1, tokens, 2, 32).transpose(1, 2)
    ref = (torch.softmax(split(q) @ split(k).transpose(-1, -2) * 0.17, -1) @ split(v)).transpose(1, 2)
    err = float((y - ref.reshape(1, tokens, 64)).norm() / ref.norm())
    print(f"{tokens} tokens at 2^{exponent}: {err:.2e}", flush=True)
    assert err <= 2e-6
