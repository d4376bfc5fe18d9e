"""The measure and bar of ``part_products``: six part products pass, five never do."""

from __future__ import annotations

import pytest
import torch

from part_products import RMS_BAR, normalised_rms

SIX = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]


def _parts(v):
    out, rest = [], v
    for _ in range(3):
        out.append(rest.bfloat16().float())
        rest = rest - out[-1]
    assert not rest.any()  # three parts hold fp32's 24 bits
    return [p.double() for p in out]


@pytest.mark.parametrize("products", [32, 1728])
def test_bar_sees_the_loss_of_any_part_product(products):
    g = torch.Generator().manual_seed(products)
    scale = torch.exp2(torch.randint(-40, 41, (products,), generator=g).float())
    a = torch.randn(200, products, generator=g) * scale
    b = torch.randn(products, 150, generator=g) / scale[:, None]
    pa, pb = _parts(a), _parts(b)
    ref, size = a.double() @ b.double(), ((a.double() ** 2) @ (b.double() ** 2)).sqrt()
    terms = {ij: pa[ij[0]] @ pb[ij[1]] for ij in SIX}
    rms = lambda keep: normalised_rms(sum(terms[k] for k in keep), ref, size)
    assert rms(SIX) < 0.01 * RMS_BAR
    for lost in SIX:
        assert rms([k for k in SIX if k != lost]) > 1.9 * RMS_BAR, lost
    swapped = pa[0] @ pb[0] + pa[0] @ pb[1] + pa[2] @ pb[0] + pa[1] @ pb[1] + pa[0] @ pb[2] + pa[2] @ pb[0]
    assert normalised_rms(swapped, ref, size) > RMS_BAR
