"""How far sums of products in bf16 parts are from float64, in a measure that sees the loss of any one part product.

An fp32 operand is three bf16 parts; six of the nine part products are summed.  Against the root of the sum of
squared products -- the size of a sum of products of random signs -- the six leave a root mean square error of
6e-9 however many products a sum has, and without any one of the five small ones at least 2.4e-6
(``test_part_product_bar.py``).  fp32 accumulation adds 2e-7 .. 7e-7 (up to 7000 products): the bar is half the
least loss."""

from __future__ import annotations

import torch

RMS_BAR = 1.2e-6


def normalised_rms(y: torch.Tensor, ref: torch.Tensor, size: torch.Tensor) -> float:
    """Root mean square of ``(y - ref) / size`` over the results whose ``size`` is not zero."""
    ok = size > 0
    return float((((y.double() - ref)[ok] / size[ok]) ** 2).mean().sqrt())
