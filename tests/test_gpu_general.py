"""GPU parity of the general kernels (fp64 layers, fp32 layers above degree 16)
at the sizes where their tilings change: each forward tile with its reduction
unsplit and split, the dx reduction in one and two groups, every chunk size of
the degree axis (one and several chunks), and row, input and output
remainders.  References: the oracles in fp64.

Tolerances: fp64 1e-11 norm-wise relative (both sides fp64, summation order
and acos/cos against the recurrence); fp32 1e-5 up to degree 40 and 3e-7 per
degree above: the three-term recurrence rounds at 2^-24 per step and its steps'
errors add up coherently for the Jacobi family (2.1e-5 at degree 100 for the
same recurrence run in plain fp32 FMAs)."""
import pytest
import torch

from oracle import chebykan_oracle as orc
from oracle import family_oracle as fo

pytestmark = pytest.mark.gpu


def _tol(dtype, deg):
    return 1e-11 if dtype == torch.float64 else max(1e-5, 3e-7 * deg)


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    n = b.norm().item()
    return (a - b).norm().item() / (n if n > 0 else 1.0)


def _check(dtype, B, I, O, deg, family=None):
    from kan_amd import functional as F
    from kan_amd import JacobiKANLayer
    print(f"general {dtype} B={B} I={I} O={O} deg={deg} {family}", flush=True)
    g = torch.Generator().manual_seed(B + 3 * I + 5 * O + 7 * deg)
    x = torch.randn(B, I, generator=g, dtype=dtype) * 1.5
    c = torch.randn(I, O, deg + 1, generator=g, dtype=dtype) / (I * (deg + 1))
    dy = torch.randn(B, O, generator=g, dtype=dtype)
    xd, cd = x.cuda().requires_grad_(True), c.cuda().requires_grad_(True)
    if family is None:
        ref = orc.layer_forward_backward(x.double(), c.double(), dy.double())
        y = F.chebykan(xd, cd)
    else:
        ref = fo.family_forward_backward(x.double(), c.double(), dy.double(), "jacobi", 0.5, -0.25)
        y = F.family_kan(xd, cd, JacobiKANLayer(I, O, deg, alpha=0.5, beta=-0.25).basis.spec())
    y.backward(dy.cuda())
    torch.cuda.synchronize()
    assert y.dtype == dtype
    for got, want in zip((y, xd.grad, cd.grad), ref):
        assert _rel(got, want) <= _tol(dtype, deg)


@pytest.mark.parametrize("B,I,O,deg", [
    (16400, 9, 250, 4),    # 32 x 64 forward tiles, unsplit
    (4100, 21, 250, 8),    # the same, reduction split in four
    (2049, 33, 100, 6),    # 32 x 32 tiles, split
    (65, 50, 18, 5),       # 16 x 16 tiles, eight reduction groups
    (1, 3, 1, 1), (3, 1, 17, 1), (15, 2, 16, 2), (17, 5, 33, 3),  # smaller than one tile
    (2050, 257, 20, 7),    # dx unsplit; odd widths
    (70, 250, 500, 8),     # dC on 32-output tiles
    (130, 100, 130, 2),    # dC on 64-output tiles
    (200, 30, 33, 4), (200, 33, 30, 3), (90, 20, 250, 17),  # even and odd degree counts of the staging
    (48, 40, 30, 9), (50, 20, 24, 10), (31, 17, 40, 12), (33, 24, 20, 14), (40, 18, 35, 27),  # chunks
])
@pytest.mark.parametrize("family", [None, "jacobi"])
def test_fp64_tilings(B, I, O, deg, family):
    _check(torch.float64, B, I, O, deg, family)


@pytest.mark.parametrize("B,I,O,deg", [
    (4100, 20, 250, 17), (2049, 33, 100, 24), (65, 50, 18, 20), (1, 3, 1, 17), (17, 5, 33, 33),
    (2050, 257, 20, 18), (70, 250, 500, 24), (70, 260, 500, 17),
    (300, 40, 33, 25), (2049, 17, 33, 26),  # dx in one chunk: row, input and output remainders
    (40, 18, 35, 28), (33, 24, 20, 30), (50, 20, 24, 40), (31, 17, 40, 100),
])
@pytest.mark.parametrize("family", [None, "jacobi"])
def test_fp32_tilings(B, I, O, deg, family):
    _check(torch.float32, B, I, O, deg, family)
