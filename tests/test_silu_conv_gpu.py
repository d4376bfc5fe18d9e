"""A conv that applies its input's SiLU itself equals the SiLU pass and the conv, bit for bit."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


# one shape per way the input is read: im2col rows, a brick halo, whole planes, a packed copy, the streaming GEMM
# (whose SiLU stays a pass) and the LDS-staged GEMM
@pytest.mark.parametrize("precision", ["fp32", "bf16", "f16x2"])
@pytest.mark.parametrize(("shape", "cout", "stride"), [
    ((1, 6, 9, 7, 8), 32, 2), ((2, 8, 16, 16, 8), 8, 1), ((1, 80, 64, 72, 8), 8, 1), ((1, 65, 64, 70, 8), 32, 2),
    ((1, 9, 12, 10, 32), 32, 1), ((1, 12, 9, 14, 32), 64, 2), ((1, 16, 32, 32, 64), 64, 1), ((1, 4, 8, 8, 20), 12, 1)])
def test_silu_conv_equals_silu_then_conv(ctmr, dev, precision, shape, cout, stride):
    print(f"silu conv {shape} -> {cout} stride {stride} {precision}", flush=True)
    f = ctmr.fast_fp32
    g = torch.Generator(device=dev).manual_seed(sum(shape))
    x = 3 * torch.randn(*shape, device=dev, generator=g)
    w = torch.randn(cout, shape[-1], 3, 3, 3, device=dev, generator=g) / (27 * shape[-1]) ** 0.5
    b = torch.randn(cout, device=dev, generator=g)
    with f.precision(precision):
        y = f._silu_conv3d(x, w, b, stride=stride)
        assert torch.equal(y, f.conv3d(f.silu(x), w, b, padding=1, stride=stride))
