"""Flash attention on shared, split key blocks: part and block boundaries, and operands that are not finite.

The bar against float64: scores are sums of 32 products held to 2^-23 each and rounded a dozen times, so a score
s carries an absolute error of at most 2^-20 * sum |q k| * scale, which scales its probability by as much; the
sums over keys round once per part product and block: 2e-6 of the largest |v| covers both at these sizes."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, heads, scale):
    n, lq, c = q.shape
    split = lambda t: t.double().reshape(n, t.shape[1], heads, 32).transpose(1, 2)
    p = torch.softmax(split(q) @ split(k).transpose(-1, -2) * scale, dim=-1)
    return (p @ split(v)).transpose(1, 2).reshape(n, lq, c)


# one key; a block less one / whole / plus one; the four-part split's edges (empty, one-key and full last parts);
# query tiles and groups less one / plus one
SHAPES = [(1, 1, 1, 1), (2, 15, 31, 2), (1, 16, 32, 1), (1, 17, 33, 3), (1, 65, 127, 2), (2, 64, 128, 1), (1, 63, 129, 2),
          (1, 129, 192, 1), (1, 128, 193, 2), (1, 40, 255, 1), (1, 300, 257, 2), (1, 128, 2049, 1), (3, 2048, 64, 16),
          # four parts to 256 workgroups of 32 queries, two to 1023 of 64, then one; the two-part split's edges
          (2, 256, 128, 16), (2, 257, 128, 16), (2, 288, 129, 16), (2, 300, 192, 16), (2, 300, 193, 16),
          (2, 270, 255, 16), (3, 1300, 300, 16), (1, 1023 * 64, 161, 1), (1, 1023 * 64 + 1, 161, 1)]


@pytest.mark.parametrize("precision", ["fp32", "f16x2"])
@pytest.mark.parametrize(("n", "lq", "lk", "heads"), SHAPES, ids=["-".join(map(str, s)) for s in SHAPES])
def test_key_parts_and_blocks(ctmr, dev, precision, n, lq, lk, heads):
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(lq * 7 + lk)
    q, k, v = (torch.randn(n, r, heads * 32, generator=g) * s for r, s in ((lq, 1.5), (lk, 1.5), (lk, 2.0)))
    with f.precision(precision):
        run = lambda: f.flash_attention(q.to(dev), k.to(dev), v.to(dev), heads=heads, scale=32 ** -0.5)
        y = run()
        assert torch.equal(y, run())
    ref = _reference(q, k, v, heads, 32 ** -0.5)
    err = (y.cpu().double() - ref).abs().max().item()
    assert err <= 2e-6 * v.abs().max().item(), err
    # A lost part product of P V is 2.4e-6 of a row's sqrt(sum (p v)^2), about its own size over many keys; one of
    # K Q^T, 2.4e-6 of sqrt(sum (q k)^2) * scale = 2.25 in the exponent, about 5e-6 of it.  fp32 sums leave 2e-7.
    norm = float((y.cpu().double() - ref).norm() / ref.norm())
    print(f"{norm:.2e}", flush=True)
    assert norm <= 8e-7


@pytest.mark.parametrize(("lq", "lk"), [(40, 70), (33, 300)])
def test_operands_that_are_not_finite(ctmr, dev, lq, lk):
    """The fp32 kernel's pattern: a key whose score overflows to -inf has no weight, a NaN or +inf score or an
    infinite value taints its rows, and every other row keeps its precision."""
    f = ctmr.fast_fp32
    g = torch.Generator().manual_seed(lk)
    q, k, v = (torch.randn(1, r, 64, generator=g) for r in (lq, lk, lk))
    q[..., 0] = q[..., 0].abs() + 0.5
    k[0, 3, :32] = 0.0
    k[0, 3, 0] = float("-inf")        # every score of head 0 with key 3 is -inf
    k[0, lk - 1, :32] = 0.0
    k[0, lk - 1, 0] = -3.402e38       # overflows in bf16, -inf as a score where the query's dim exceeds 1
    q[0, 5, 7] = float("nan")
    q[0, lq - 1, 40] = float("inf")   # head 1: +inf, -inf or NaN scores
    v[0, 2, 50] = float("inf")        # head 1, dim 18: that output of every row
    y = f.flash_attention(q.to(dev), k.to(dev), v.to(dev), heads=2, scale=32 ** -0.5).cpu()
    ref = _reference(q, k, v, 2, 32 ** -0.5)
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isposinf(), ref.isposinf())
    assert torch.equal(y.isneginf(), ref.isneginf())
    ok = ref.isfinite()
    assert bool(((y.double() - ref).abs()[ok] <= 1e-5).all()) and 64 < int((~ok).sum()) < ok.numel() // 2


@pytest.mark.parametrize("precision", ["fp32", "f16x2"])
def test_rows_a_gigabyte_apart(ctmr, dev, precision):
    """Rows of a key block past the last key whose byte offset exceeds 2^32: two keys, rows 2^30 - 256 bytes
    apart, so that row 5's offset wraps to the gap behind row 0.  The gap holds NaN, which no output may show."""
    f = ctmr.fast_fp32
    ld = (1 << 28) - 64
    buf = torch.full((2 * ld,), float("nan"), device=dev)
    rows = buf.as_strided((1, 2, 64), (2 * ld, ld, 1))
    g = torch.Generator().manual_seed(3)
    kv, q = torch.randn(1, 2, 64, generator=g), torch.randn(1, 20, 32, generator=g)
    rows.copy_(kv)
    with f.precision(precision):
        y = f.flash_attention(q.to(dev), rows[..., :32], rows[..., 32:], heads=1, scale=32 ** -0.5)
    err = (y.cpu().double() - _reference(q, kv[..., :32], kv[..., 32:], 1, 32 ** -0.5)).abs().max().item()
    assert err <= 2e-6 * kv.abs().max().item(), err
