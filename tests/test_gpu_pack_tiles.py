"""The packed operands at the pack's two tile widths (8 and 32 outputs per
block) and their edges: every packed value against a restatement of the
layout's formulas, through the GEMMs that read them (forward and input
gradient at a small and a large batch), for layers on both sides of the rule
that picks the width.

Tolerance 1e-5 (fp32) / 2e-2 (bf16) norm-wise, as every parity test of these
paths: a misplaced packed value is an error of order 1 in its column."""
import pytest
import torch

from oracle import chebykan_oracle as orc

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return (a - b).norm().item() / b.norm().item()


@pytest.mark.parametrize("I,O,deg", [
    (1, 1, 3), (31, 7, 4), (33, 8, 8), (40, 9, 7), (32, 33, 16), (65, 63, 12),   # 8-output blocks
    (500, 511, 8), (512, 512, 4), (480, 545, 6),                                   # 256 blocks of 32 outputs and fewer
    (520, 530, 2), (300, 90, 16),
])
@pytest.mark.parametrize("compute,tol", [("fp32", 1e-5), ("bf16", 2e-2)])
def test_pack_widths(I, O, deg, compute, tol):
    from kan_amd import functional as F
    print(f"pack I={I} O={O} deg={deg} {compute}", flush=True)
    g = torch.Generator().manual_seed(I + 3 * O + deg)
    c = torch.randn(I, O, deg + 1, generator=g) / (I * (deg + 1))
    if compute == "bf16":
        c = c.bfloat16().float()
    for B in (40, 600):
        x, dy = torch.randn(B, I, generator=g), torch.randn(B, O, generator=g)
        y_ref, dx_ref, _ = orc.layer_forward_backward(x.double(), c.double(), dy.double())
        xd = x.cuda().requires_grad_(True)
        y = F.chebykan(xd, c.cuda(), compute)
        y.backward(dy.cuda())
        for o in range(0, O, max(1, O // 9)):  # column by column: an edge column is not averaged away
            assert _rel(y[:, o], y_ref[:, o]) <= 3 * tol
        assert _rel(y, y_ref) <= tol
        assert _rel(xd.grad, dx_ref) <= tol
