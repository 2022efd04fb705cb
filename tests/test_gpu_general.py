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
import math

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


def _hermite_case(scaling, domain, deg, low_only, B=90, I=18, O=21):
    """x, coefficients, dy of a Hermite layer whose every degree counts: H_n
    (He_n) grows as sqrt(2^n n!) (sqrt(n!)), so coefficient n is divided by it;
    low_only keeps the degrees below a third."""
    g = torch.Generator().manual_seed(deg + 100 * low_only)
    x = torch.randn(B, I, generator=g) * 1.5 if domain is None else torch.rand(B, I, generator=g) * 7 - 2
    n = torch.arange(deg + 1, dtype=torch.float64)
    norm = torch.exp(0.5 * (torch.lgamma(n + 1) + (n * math.log(2.0) if scaling == "physicist" else 0)))
    c = (torch.randn(I, O, deg + 1, generator=g, dtype=torch.float64) / norm).float()
    if low_only:
        c[..., deg // 3:] = 0
    return x, c, torch.randn(B, O, generator=g)


# every coefficient's gradient counts likewise: dC's degree n over its norm
def _hermite_dc_scaled(dc, scaling):
    n = torch.arange(dc.shape[-1], dtype=torch.float64)
    norm = torch.exp(0.5 * (torch.lgamma(n + 1) + (n * math.log(2.0) if scaling == "physicist" else 0)))
    return dc.detach().double().cpu() / norm


@pytest.mark.parametrize("deg", [17, 20, 24, 26, 27, 40])  # dx in one chunk to 26, several above
@pytest.mark.parametrize("scaling", ["physicist", "probabilist"])
@pytest.mark.parametrize("domain", [None, (-2.0, 5.0)])
@pytest.mark.parametrize("low_only", [False, True])
def test_fp32_hermite_every_degree_counts(deg, scaling, domain, low_only):
    """The Hermite bases are evaluated at 3 t, and dx carries that factor once
    for every degree.  Tolerance: the fp32 recurrence at |u| <= 3 alone (plain
    torch in fp32 against fp64, these inputs) is off by at most 9.2e-7."""
    from kan_amd import HermiteKANLayer
    print(f"general hermite {scaling} {domain} deg={deg} low={low_only}", flush=True)
    x, c, dy = _hermite_case(scaling, domain, deg, low_only)
    m = HermiteKANLayer(c.shape[0], c.shape[1], deg, scaling=scaling, domain=domain,
                        normalize_domain=True)
    with torch.no_grad():
        m.hermite_coeffs.copy_(c)
    m = m.cuda()
    xd = x.cuda().requires_grad_(True)
    y = m(xd)
    y.backward(dy.cuda())
    torch.cuda.synchronize()
    y_ref, dx_ref, dc_ref = fo.family_forward_backward(
        x.double(), c.double(), dy.double(), "hermite" if scaling == "physicist" else "hermite_e",
        domain=domain)
    assert _rel(y, y_ref) <= _tol(torch.float32, deg)
    assert _rel(xd.grad, dx_ref) <= _tol(torch.float32, deg)
    assert _rel(_hermite_dc_scaled(m.hermite_coeffs.grad, scaling),
                _hermite_dc_scaled(dc_ref, scaling)) <= _tol(torch.float32, deg)
