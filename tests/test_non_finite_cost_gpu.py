"""What NaN costs: the kernels that multiply in bf16 parts compute results that are not finite again on FP32 MFMA.

A NaN spreads to every voxel of its group through a group norm, and to every query of its head through one key,
so a pass over operands that are all NaN is an ordinary pass of a diverged sample.  FP32 MFMA has a sixteenth of
the bf16 rate against six products, 2.7 times their time, and the second pass reads its operands without LDS or
prefetch: at most 16 times the finite pass, where a scalar loop per result took several hundred."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# (name, input shape NDHWC, cout, options, kernel)
CONVS = [
    ("LDS-staged GEMM, norm and SiLU", (1, 32, 32, 32, 128), 128, {"silu": True, "affine": True}, "lds"),
    ("two wave sets", (1, 16, 32, 32, 128), 64, {"split": 2}, "lds"),
    ("32 outputs", (1, 64, 64, 32, 32), 32, {}, "lds"),
    ("nearest-2x", (1, 16, 16, 16, 128), 128, {"upsample": True, "split": 1}, "stream"),
    ("direct, stride 2", (1, 32, 32, 32, 128), 128, {"stride": 2, "split": 1}, "stream_direct"),
    ("split over four waves", (2, 8, 8, 4, 512), 512, {}, "split_waves"),
    ("8 -> 8 plane by plane", (1, 64, 96, 96, 8), 8, {"silu": True}, None),
    ("8 -> 32 plane by plane", (1, 96, 96, 96, 8), 32, {"stride": 2}, None),
]


def _time(fn):
    """Milliseconds of one call, the least of three runs of four."""
    fn()
    best = float("inf")
    for _ in range(3):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(4):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 4)
    return best


@pytest.mark.parametrize(("name", "shape", "cout", "options", "kernel"), CONVS, ids=[c[0] for c in CONVS])
def test_conv_of_nan(ctmr, dev, name, shape, cout, options, kernel):
    f, L = ctmr.fast_fp32, ctmr._lib
    opts = dict(options)
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(*shape, device=dev, generator=g)
    c = shape[-1]
    w = torch.randn(cout, c, 3, 3, 3, device=dev, generator=g) * (27 * c) ** -0.5
    if opts.pop("affine", False):
        opts["affine"] = torch.rand(shape[0], c, 2, device=dev, generator=g)
    mode = L.MODE_NEAREST2X if opts.get("upsample") else L.MODE_PLAIN
    flags = (L.F_AFFINE if "affine" in opts else 0) | (L.F_SILU if opts.get("silu") else 0)
    if kernel:
        assert L.conv_kernel(ctmr.ops.make_desc(shape, cout, 3, opts.get("stride", 1), mode, flags, L.DT_F32,
                                                opts.get("split", 0))) == kernel
    packed = (f.pack_upsample_weight if opts.get("upsample") else f.pack_weight)(w)
    run = lambda v: f.implicit_gemm_conv3d(v, packed, None, cout=cout, **opts)
    nan = torch.full_like(x, float("nan"))
    finite, taken = _time(lambda: run(x)), _time(lambda: run(nan))
    zero = _time(lambda: run(torch.zeros_like(x)))  # exact zeros are no reason to compute again
    print(f"{name}: finite {finite * 1e3:.1f} us, NaN {taken * 1e3:.1f} us, {taken / finite:.1f}x, zeros "
          f"{zero * 1e3:.1f} us", flush=True)
    assert bool(run(nan).isnan().all()) and bool(run(x).isfinite().all())
    assert zero <= 1.6 * finite + 0.02  # the fill and the exact test
    assert taken <= 16 * finite


@pytest.mark.parametrize(("n", "tokens", "heads"), [(2, 2048, 8), (1, 4158, 16)])
def test_attention_of_nan(ctmr, dev, n, tokens, heads):
    f = ctmr.fast_fp32
    g = torch.Generator(device=dev).manual_seed(2)
    q, k, v = (torch.randn(n, tokens, heads * 32, device=dev, generator=g) for _ in range(3))
    bad = k.clone()
    bad[:, tokens // 2] = float("nan")  # one key: every query of every head
    run = lambda keys: f.flash_attention(q, keys, v, heads=heads, scale=32 ** -0.5)
    finite, taken = _time(lambda: run(k)), _time(lambda: run(bad))
    print(f"{tokens} tokens: finite {finite * 1e3:.1f} us, NaN {taken * 1e3:.1f} us, {taken / finite:.1f}x", flush=True)
    assert bool(run(bad).isnan().all()) and bool(run(k).isfinite().all())
    assert taken <= 16 * finite
