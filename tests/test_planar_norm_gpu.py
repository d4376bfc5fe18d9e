"""Group norm of NCDHW tensors as they lie (``ctmr_gn_planar``): both forms (one workgroup per run, chunked runs),
vector and scalar reads, against the NDHWC path and float64.

The bar: the statistics are fp64 on both paths, the apply is one fp32 fma (2^-24 relative of its larger term) on an
affine rounded to fp32 (two roundings), and the SiLU is within 1e-6: 4e-7 * (|x * scale| + |offset|) + 1e-6 |y|."""

from __future__ import annotations

import pytest
import torch

from oracle import reference_math as rm

pytestmark = pytest.mark.gpu

# (name, n, c, groups, (d, h, w), silu, floats of offset into the storage)
CASES = [
    ("one value a channel", 2, 32, 32, (1, 1, 1), True, 0),
    ("one odd plane, scalar reads", 1, 6, 3, (3, 5, 7), False, 0),
    ("the smallest vector run", 3, 64, 32, (1, 2, 2), True, 0),
    ("the deepest level", 2, 512, 32, (8, 8, 4), True, 0),
    ("the longest one-launch vector run", 1, 32, 1, (16, 16, 4), True, 0),
    ("past it", 1, 32, 1, (16, 16, 5), False, 0),
    ("the longest one-launch scalar run", 1, 8, 1, (1, 1, 1024), False, 1),
    ("chunked scalar run, ragged", 1, 4, 2, (17, 31, 29), True, 0),
    ("chunked vector run, remainder chunk", 2, 64, 32, (20, 22, 42), True, 0),
    ("one group of every channel, misaligned storage", 1, 48, 1, (12, 12, 12), True, 3),
    ("many channels a group", 1, 1024, 1, (2, 3, 2), True, 0),
    # past 2048 chunks of 4096 vectors: two of them a chunk, the last chunk in its first
    ("scalar run of more than 2^23 values", 1, 64, 1, (51, 51, 51), True, 0),
]


@pytest.mark.parametrize(("name", "n", "c", "groups", "grid", "silu", "offset"), CASES, ids=[c[0] for c in CASES])
def test_planar_group_norm(ctmr, dev, name, n, c, groups, grid, silu, offset):
    f = ctmr.fast_fp32
    d, h, w = grid
    g = torch.Generator().manual_seed(5)
    buf = torch.randn(n * c * d * h * w + offset, generator=g) * 1.7 + 2.5
    x = buf[offset:].view(n, c, d, h, w)
    gamma, beta = torch.randn(c, generator=g), torch.randn(c, generator=g)
    xg = buf.to(dev)[offset:].view(n, c, d, h, w)
    y = f.group_norm_ncdhw(xg, gamma.to(dev), beta.to(dev), num_groups=groups, eps=1e-6, apply_silu=silu)
    assert y.is_contiguous() and y.shape == x.shape
    assert torch.equal(y, f.group_norm_ncdhw(xg, gamma.to(dev), beta.to(dev), num_groups=groups, eps=1e-6,
                                             apply_silu=silu))
    nd = x.permute(0, 2, 3, 4, 1).contiguous().double().numpy()
    aff = rm.group_norm_affine(nd, gamma.double().numpy(), beta.double().numpy(), groups, 1e-6)
    ref = torch.from_numpy(rm.apply_affine(nd, aff, silu)).permute(0, 4, 1, 2, 3)
    scale, off = (torch.from_numpy(aff[..., k]).reshape(n, c, 1, 1, 1) for k in (0, 1))
    bar = 4e-7 * ((x.double() * scale).abs() + off.abs()) + 1e-6 * ref.abs()
    assert bool(((y.cpu().double() - ref).abs() <= bar).all()), name
    # a view that lies as NDHWC takes the other path, within the same bar of it
    nd_view = xg.permute(0, 2, 3, 4, 1).contiguous().permute(0, 4, 1, 2, 3)
    other = f.group_norm_ncdhw(nd_view, gamma.to(dev), beta.to(dev), num_groups=groups, eps=1e-6, apply_silu=silu)
    assert bool(((other - y).cpu().double().abs() <= 2 * bar).all())


def test_planar_group_norm_not_finite(ctmr, dev):
    """A NaN or an infinity taints its own (batch item, group) on both paths and nothing else."""
    f = ctmr.fast_fp32
    x = torch.randn(2, 64, 6, 6, 6, generator=torch.Generator().manual_seed(1)).to(dev)
    x[0, 5, 1, 2, 3] = float("nan")
    x[1, 40, 0, 0, 0] = float("inf")
    one, zero = torch.ones(64, device=dev), torch.zeros(64, device=dev)
    y = f.group_norm_ncdhw(x, one, zero, num_groups=32, eps=1e-6)
    other = f.group_norm_ncdhw(x.permute(0, 2, 3, 4, 1).contiguous().permute(0, 4, 1, 2, 3), one, zero, num_groups=32,
                               eps=1e-6)
    assert torch.equal(y.isnan(), other.isnan()) and int(y.isnan().any(dim=(2, 3, 4)).sum()) == 4
