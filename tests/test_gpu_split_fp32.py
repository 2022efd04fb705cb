"""GPU parity of the fp32 layers' three-plane bf16 GEMMs (degrees 3-16) at the
sizes where their tilings change: row, input, output and degree remainders,
the 64- and 128-column forward tiles with the reduction whole and split, both
dC tile widths, split batches, and the input gradient's row blocks.

Tolerance against the oracle in fp64: 4e-6 norm-wise.  The plane products
dropped are below 2^-24 of each product and the planes are exact, so what
remains is fp32 accumulation (at most 16384 terms here, at 2^-24 per rounding
and the square root of their number: 1.5e-6 at 8192 terms) and the basis
recurrence's rounding."""
import pytest
import torch

from oracle import chebykan_oracle as orc

pytestmark = pytest.mark.gpu

TOL = 4e-6


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return (a - b).norm().item() / b.norm().item()


def _inputs(B, I, O, deg, seed=0):
    g = torch.Generator().manual_seed(B + 3 * I + 5 * O + 7 * deg + seed)
    x = torch.randn(B, I, generator=g) * 1.5
    c = torch.randn(I, O, deg + 1, generator=g) / (I * (deg + 1))
    dy = torch.randn(B, O, generator=g)
    return x, c, dy


def _run(x, c, dy):
    from kan_amd import functional as F
    xd, cd = x.cuda().requires_grad_(True), c.cuda().requires_grad_(True)
    y = F.chebykan(xd, cd, "fp32")
    y.backward(dy.cuda())
    torch.cuda.synchronize()
    return y.detach(), xd.grad, cd.grad


@pytest.mark.parametrize("B,I,O,deg", [
    (513, 40, 40, 3), (600, 33, 64, 4), (770, 100, 65, 4), (1025, 65, 130, 4),   # P = 4
    (513, 40, 40, 5), (600, 33, 64, 8), (770, 100, 65, 7), (1025, 65, 130, 8),   # P = 8
    (513, 40, 40, 9), (600, 33, 64, 16), (770, 100, 65, 12), (1025, 65, 130, 16),  # P = 16
    (4097, 96, 300, 5),     # dC's narrow tile, batch split
    (3000, 500, 257, 4),    # dC's wide and narrow tiles with remainders
    (16400, 40, 33, 8),     # many row tiles, one output pair
    (640, 1024, 128, 16),   # the forward reduction split over blocks
    # small batches: the 64 x 128 forward tile, its reduction whole, split and
    # split to one super-group, a row and a column of fragments past the end
    (65, 8, 65, 8), (130, 70, 500, 10), (300, 300, 96, 6), (257, 200, 129, 3), (512, 640, 1000, 7),
    (65, 8, 100, 16), (100, 16, 97, 4),
])
def test_split_fp32_tilings(B, I, O, deg):
    print(f"split fp32 B={B} I={I} O={O} deg={deg}", flush=True)
    x, c, dy = _inputs(B, I, O, deg)
    ref = orc.layer_forward_backward(x.double(), c.double(), dy.double())
    for got, want in zip(_run(x, c, dy), ref):
        assert _rel(got, want) <= TOL


@pytest.mark.parametrize("B", [300, 600])  # the 64 x 128 forward tile, the large ones
@pytest.mark.parametrize("deg", [4, 8, 16])
def test_non_finite_and_extreme_values_stay_where_they_were(B, deg):
    """An infinite coefficient or upstream gradient reaches exactly the results
    that the fp32 products reach, with their sign; values next to overflow and
    far below 1 keep their precision."""
    print(f"split fp32 non-finite B={B} deg={deg}", flush=True)
    I, O = 40, 70
    x, c, dy = _inputs(B, I, O, deg, 1)
    x = x.abs() * 0.3 + 0.05
    big = torch.finfo(torch.float32).max
    c[3, 5, 1], c[7, 9, 1], c[11, 20, 0] = float("inf"), float("-inf"), float("nan")
    c[:, 30] = 0
    c[2, 30, 1] = big            # t < 1: finite results
    c[:, 31] *= 1e-30
    dy[10, 4], dy[20, 6] = float("inf"), float("-inf")
    t = torch.tanh(x)
    y, dx, dc = (v.cpu() for v in _run(x, c, dy))
    basis = orc.basis_recurrence(t, deg)
    # one non-finite term per affected sum: its sign decides
    y_ref = torch.einsum("bid,iod->bo", basis.double(), c.double())
    for o in (5, 9, 20):
        assert torch.equal(torch.isnan(y[:, o]), torch.isnan(y_ref[:, o]))
        ok = ~torch.isnan(y_ref[:, o])
        assert torch.equal(y[ok, o], y_ref[ok, o].float())
    rest = [o for o in range(O) if o not in (5, 9, 20)]
    assert torch.isfinite(y[:, rest]).all()
    for o in (30, 31):
        assert _rel(y[:, o], y_ref[:, o]) <= TOL
    for b, o, sign in ((10, 4, 1.0), (20, 6, -1.0)):
        want = sign * basis[b] * float("inf")  # [I, D]: +-inf, nan where the basis is 0
        got = dc[:, o]
        sel = (basis[b].abs() > 0)
        assert torch.equal(got[sel], want[sel])
    assert torch.isfinite(dc[:, [o for o in range(O) if o not in (4, 6)]]).all()


@pytest.mark.parametrize("B", [90, 600])
@pytest.mark.parametrize("deg", [4, 8, 16])
def test_infinite_coefficient_meets_infinite_gradient(B, deg):
    """dx where an infinite coefficient meets an infinite upstream gradient:
    the product's sign and infinity, as the fp32 product gives them.  Every
    input is near 1 (U_{d-1} > 0 for all degrees there) and the coefficients of
    output 7 share one sign, so no sum holds two infinities of opposite sign."""
    print(f"split fp32 inf x inf B={B} deg={deg}", flush=True)
    I, O = 40, 70
    x, c, dy = _inputs(B, I, O, deg, 2)
    x = 2.7 + 0.3 * torch.rand(B, I, generator=torch.Generator().manual_seed(deg))
    for o, sign in ((7, 1.0), (33, -1.0)):
        c[:, o] = sign * (c[:, o].abs() + 1e-3)
        c[3, o, 2] = sign * float("inf")
    dy[10, 7], dy[20, 7] = float("inf"), float("-inf")
    dy[30, 33], dy[40, 33] = float("inf"), float("-inf")
    dy[:, 33] = torch.where(torch.isinf(dy[:, 33]), dy[:, 33], -dy[:, 7].sign() * (dy[:, 33].abs() + 1e-3))
    dy[[10, 20], 33] = 0.5 * torch.tensor([-1.0, 1.0])
    dy[[30, 40], 7] = 0.5 * torch.tensor([-1.0, 1.0])
    _, dx, _ = (v.cpu() for v in _run(x, c, dy))
    inf = float("inf")
    assert torch.equal(dx[10], torch.full((I,), inf)) and torch.equal(dx[20], torch.full((I,), -inf))
    assert torch.equal(dx[30], torch.full((I,), -inf)) and torch.equal(dx[40], torch.full((I,), inf))
    # input 3 of every other row: the infinite coefficients times a finite gradient
    assert torch.equal(dx[:, 3], dy[:, 7].sign() * inf)
    rest = [b for b in range(B) if b not in (10, 20, 30, 40)]
    assert torch.isfinite(dx[rest][:, [i for i in range(I) if i != 3]]).all()


# B, O: the 64 x 128 forward tile, the 128- and 64-column large ones, both dC tiles
@pytest.mark.parametrize("B,O", [(300, 70), (600, 70), (600, 40), (1100, 130)])
@pytest.mark.parametrize("deg,far", [(4, 1e10), (8, 1e5), (16, 140.0)])
def test_affine_map_basis_overflow(B, O, deg, far):
    """Under an affine map t is unbounded: at t = ``far`` T_deg alone
    overflows, and its products are infinite with their sign; where T_deg is
    finite but above the largest bf16, they are finite.  The same results at
    every batch size, and no other row or input is touched."""
    from kan_amd.functional import ChebyKANFunction
    print(f"split fp32 affine overflow B={B} O={O} deg={deg}", flush=True)
    I = 40
    x, c, dy = _inputs(B, I, O, deg, 3)
    x, dy = x * 0.5, dy.clamp(-1, 1) * 0.5
    c[4, 5, deg] = float("-inf")
    near = ((3.3995e38 / 2 ** (deg - 1)) ** (1 / deg))
    x[17, 4], x[50, 9] = far, near
    basis = orc.basis_recurrence(x, deg)  # fp32
    assert torch.isinf(basis[17, 4, deg]) and torch.isfinite(basis[17, 4, :deg]).all()
    assert 3.3962e38 < basis[50, 9, deg] < 3.4028e38
    xd, cd = x.cuda().requires_grad_(True), c.cuda().requires_grad_(True)
    y = ChebyKANFunction.apply(xd, cd, "fp32", None, (1.0, 0.0))  # t = x
    y.backward(dy.cuda())
    y, dc = y.detach().cpu(), cd.grad.cpu()
    cf = c.clone()
    cf[4, 5, deg] = 0
    b64 = orc.basis_recurrence(x.double(), deg)
    y_ref = torch.einsum("bid,iod->bo", b64, cf.double())
    inf = float("inf")
    want = c[4, :, deg].sign() * inf
    assert torch.equal(y[17], want)
    rows, cols = [b for b in range(B) if b != 17], [o for o in range(O) if o != 5]
    assert torch.equal(y[rows, 5], -torch.sign(basis[rows, 4, deg]) * inf)
    assert _rel(y[50][cols], y_ref[50][cols]) <= TOL
    rows.remove(50)
    assert _rel(y[rows][:, cols], y_ref[rows][:, cols]) <= TOL
    assert torch.equal(dc[4, :, deg], dy[17].sign() * inf)
    assert _rel(dc[9, :, deg], torch.einsum("b,bo->o", b64[:, 9, deg], dy.double())) <= TOL
    assert torch.isfinite(dc[4, :, :deg]).all() and torch.isfinite(dc[9]).all()
    ins = [i for i in range(I) if i not in (4, 9)]
    assert _rel(dc[ins], torch.einsum("bid,bo->iod", b64[:, ins], dy.double())) <= TOL
