"""The plane-marching conv of 8 input channels: stride 1 to 8 outputs, stride 2 to 17 .. 32.

Held against a float64 convolution on the GPU and against the streaming GEMM over im2col rows
(``CTMR_F_STREAM``), whose distance from float64 it must not exceed by more than rounding noise.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
import torch.nn.functional as F  # noqa: E402

pytestmark = pytest.mark.gpu

# (input shape NDHWC, cout, stride, options): whole tiles; remainders on every axis (tiles 16 x 32 outputs at
# stride 1, 8 x 16 at stride 2) and odd sizes; one tile a run; a batch with per-item bias, affine, residual
CASES = [
    ((1, 64, 64, 96, 8), 8, 1, {}),
    ((1, 65, 71, 75, 8), 8, 1, {"silu": True}),
    ((2, 97, 47, 77, 8), 8, 1, {"affine": True, "silu": True, "residual": True, "batch_bias": True}),
    ((1, 5, 270, 250, 8), 8, 1, {"affine": True, "gn": 4}),
    ((2, 97, 47, 77, 8), 8, 1, {"residual": True, "gn": 8}),
    ((1, 65, 71, 75, 8), 8, 1, {"silu": True, "gn": 1}),
    ((1, 64, 64, 64, 8), 32, 2, {"silu": True}),
    ((1, 75, 83, 101, 8), 32, 2, {}),
    ((2, 66, 57, 79, 8), 20, 2, {"affine": True, "silu": True, "residual": True, "batch_bias": True}),
    ((1, 9, 130, 251, 8), 32, 2, {"affine": True, "gn": 8}),
    ((2, 70, 64, 62, 8), 32, 2, {"gn": 16}),
]


def _inputs(shape, cout, stride, opts, dev):
    g = torch.Generator(device=dev).manual_seed(sum(shape) + cout)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g)
    n, c = shape[0], shape[-1]
    out = (n, *((v - 1) // stride + 1 for v in shape[1:4]), cout)
    return (2 * rand(*shape) + 0.5, rand(cout, c, 3, 3, 3) / (27 * c) ** 0.5,
            rand(n, cout) if opts.get("batch_bias") else rand(cout),
            torch.stack([1 + 0.3 * rand(n, c), 0.4 * rand(n, c)], -1) if opts.get("affine") else None,
            rand(*out) if opts.get("residual") else None)


def _reference(x, w, bias, affine, res, silu, stride):
    x = x.double()
    if affine is not None:
        a = affine.double()[:, None, None, None]
        x = x * a[..., 0] + a[..., 1]
    if silu:
        x = F.silu(x)
    n, d, h, wd, c = x.shape
    od, oh, ow = ((v - 1) // stride + 1 for v in (d, h, wd))
    p = F.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    y = torch.zeros(n, od, oh, ow, w.shape[0], device=x.device, dtype=torch.float64)
    for kd in range(3):
        for kh in range(3):
            for kw in range(3):
                s = p[:, kd:kd + stride * od:stride, kh:kh + stride * oh:stride, kw:kw + stride * ow:stride]
                y += (s[:, :od, :oh, :ow].reshape(-1, c) @ w.double()[:, :, kd, kh, kw].t()).reshape(y.shape)
    y = y + (bias.double().reshape(n, 1, 1, 1, -1) if bias.dim() == 2 else bias.double())
    return y if res is None else y + res.double()


@pytest.mark.parametrize(("shape", "cout", "stride", "opts"), CASES)
def test_against_float64_and_the_im2col_gemm(ctmr, dev, shape, cout, stride, opts):
    print(f"march {shape} -> {cout} stride {stride} {opts}", flush=True)
    f, L = ctmr.fast_fp32, ctmr._lib
    x, w, bias, affine, res = _inputs(shape, cout, stride, opts, dev)
    silu, groups = bool(opts.get("silu")), opts.get("gn", 0)
    desc = ctmr.ops.make_desc(shape, cout, 3, stride, L.MODE_PLAIN, 0, L.DT_F32, 0)
    assert L.conv_kernel(desc) == "march"
    assert L.workspace_bytes(desc) == 0  # x itself is read: no im2col rows
    run = lambda stream: f.implicit_gemm_conv3d(x, f.pack_weight(w), bias, cout=cout, affine=affine, silu=silu,
                                                stride=stride, residual=res, stream_gemm=stream, gn_groups=groups)
    y, y1 = run(False), run(True)
    ref = _reference(x, w, bias, affine, res, silu, stride)
    # Both sum 216 products in fp32: the streaming GEMM within 216 rounding steps of 2^-24 of the largest partial
    # sum, this kernel within 54 + 3 (the six part products of 9 or 7 MFMAs); SiLU adds 1e-6 relative to each.
    scale = float(ref.abs().max())
    err, err1 = (float((v.double() - ref).abs().max()) / scale for v in (y, y1))
    print(f"distance from float64 {err:.2e}, im2col GEMM {err1:.2e}", flush=True)
    assert err <= 216 * 2.0 ** -24 + 1e-6
    assert err <= 1.5 * err1 + 2.0 ** -23
    assert torch.equal(run(False), y)
    if groups:
        st = f.conv_output_stats(y, groups)
        assert st is not None
        yy = y.double().reshape(shape[0], -1, groups, cout // groups)
        want = torch.stack([yy.sum((1, 3)), (yy * yy).sum((1, 3))], -1)
        # float64 sums of fewer than 2^24 values in another order
        assert torch.allclose(st.sum(1), want, rtol=1e-11, atol=1e-11 * float((yy * yy).sum()))


@pytest.mark.parametrize(("shape", "cout", "stride"), [((1, 83, 65, 61, 8), 8, 1), ((1, 66, 70, 65, 8), 32, 2)])
def test_non_finite_values_reach_their_windows_only(ctmr, dev, shape, cout, stride):
    """An infinity or a NaN makes the outputs of its 3x3x3 windows what fp32 sums make them and no others (the
    zero weights beside a row's window must not spread it)."""
    f, L = ctmr.fast_fp32, ctmr._lib
    assert L.conv_kernel(ctmr.ops.make_desc(shape, cout, 3, stride, L.MODE_PLAIN, 0, L.DT_F32, 0)) == "march"
    x, w, bias, _, _ = _inputs(shape, cout, stride, {}, dev)
    x[0, 7, 11, 13, 2] = float("inf")
    x[0, 20, 0, 31, 5] = float("-inf")
    x[0, 31, 40, 50, 7] = float("nan")
    x[0, 15, 23, 33, 1] = 3.0e38
    y = f.implicit_gemm_conv3d(x, f.pack_weight(w), bias, cout=cout, stride=stride)
    y1 = f.implicit_gemm_conv3d(x, f.pack_weight(w), bias, cout=cout, stride=stride, stream_gemm=True)
    assert torch.equal(torch.isnan(y), torch.isnan(y1))
    inf = torch.isinf(y1)
    assert torch.equal(torch.isinf(y), inf) and torch.equal(y[inf], y1[inf])
    ok = torch.isfinite(y1)
    assert bool(((y[ok].double() - y1[ok].double()).abs() <= 1e-5 * (1 + y1[ok].double().abs())).all())


@pytest.mark.parametrize(("shape", "cout", "stride"), [((1, 5, 270, 250, 8), 8, 1), ((1, 64, 64, 64, 8), 32, 2)])
def test_input_at_any_four_byte_address(ctmr, dev, shape, cout, stride):
    """Volumes whose im2col rows would be packed (4x8x8 bricks under 3/4 full, or stride 2) take x at any 4-byte
    address, as the pack does: the aligned call's bits."""
    import ctypes

    f, L = ctmr.fast_fp32, ctmr._lib
    x, w, bias, _, _ = _inputs(shape, cout, stride, {}, dev)
    packed = f.pack_weight(w)
    desc = ctmr.ops.make_desc(shape, cout, 3, stride, L.MODE_PLAIN, 0, L.DT_F32, 0)
    assert L.conv_kernel(desc) == "march" and L.workspace_bytes(desc) == 0
    y = f.implicit_gemm_conv3d(x, packed, bias, cout=cout, stride=stride)
    odd = torch.empty(x.numel() + 1, device=dev)[1:].view(shape)
    odd.copy_(x)
    again = torch.zeros_like(y)
    L.check(L.lib().ctmr_conv3d(ctypes.byref(desc), odd.data_ptr(), packed.data_ptr(), bias.data_ptr(), None, None,
                                again.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream), "ctmr_conv3d")
    assert torch.equal(again, y)
