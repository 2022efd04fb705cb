"""The workloads whose speed this framework is judged by, through its public entry points.

``listed()`` names them, ``draw()`` gives more of the same ranges; ``prepare()`` builds what a program has
in hand before the call, ``run()`` is one pass, ``work()`` what a pass cannot do without, ``exact()`` the
same results in 64 bits and ``tolerance()`` how far another correct implementation may be from them.
"""
import math

import torch

import kan_amd

# Learning rates small enough that thousands of passes on one state stay finite.
TRAIN_LR = 1e-5
FIT_LR = 0.01


def _layer(name, rows, in_dim, out_dim, degree, compute, kind="train", family="chebyshev", coeffs="fp32"):
    return {"name": name, "kind": kind, "family": family, "rows": rows, "in": in_dim, "out": out_dim,
            "degree": degree, "compute": compute, "coeffs": coeffs}


def _stack(name, kind, rows, widths, degree, compute, loss, steps):
    return {"name": name, "kind": kind, "rows": rows, "widths": "-".join(map(str, widths)),
            "degree": degree, "compute": compute, "loss": loss, "steps": steps}


def listed():
    return [
        # Serving one request through a wide layer with bf16 coefficients: the coefficient stream alone.
        _layer("infer_1_bf16", 1, 2048, 2048, 8, "bf16", "infer", coeffs="bf16"),
        # The same layer serving a small batch of requests.
        _layer("infer_64_bf16", 64, 2048, 2048, 8, "bf16", "infer", coeffs="bf16"),
        # Evaluating a default (fp32) layer on a batch and widths that are no powers of two.
        _layer("infer_300_fp32", 300, 500, 300, 6, "fp32", "infer"),
        # The benchmark's training layer in bf16, optimizer step included.
        _layer("train_8192_bf16", 8192, 1024, 1024, 8, "bf16"),
        # The same in the default precision.
        _layer("train_8192_fp32", 8192, 1024, 1024, 8, "fp32"),
        # A mini-batch of the same layer: one rank's share of a batch, or a small problem.
        _layer("train_512_bf16", 512, 1024, 1024, 8, "bf16"),
        # A Jacobi layer of odd widths and batch in the default precision.
        _layer("train_jacobi_odd_fp32", 3000, 500, 300, 5, "fp32", family="jacobi"),
        # A double-precision layer, as scientific fits use it.
        _layer("train_fp64", 2048, 256, 256, 8, "fp64"),
        # A high-degree layer (function approximation with few, rich inputs).
        _layer("train_degree24_fp32", 4096, 256, 128, 24, "fp32"),
        # The reference's training loop on a small classifier, written with the layers and torch's loss.
        _stack("module_classifier", "module", 256, (784, 64, 10), 4, "fp32", "ce", 1),
        # The same classifier trained by the resident executor: launch-bound.
        _stack("fit_classifier", "fit", 256, (784, 64, 10), 4, "fp32", "ce", 20),
        # One step of the deep regression stack at its full batch, and its weights read back.
        _stack("fit_deep", "fit", 65536, (512, 512, 512, 512, 64), 16, "bf16", "mse", 1),
    ]


def _size(rng, lo, hi):
    """Log-uniform in [lo, hi]; half of them as they fall, half multiples of 32 where that fits."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    v = int(round(v / 32) * 32) if rng.random() < 0.5 and v > 48 else int(round(v))
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["infer", "infer", "train", "train", "train", "train", "fp64", "high", "module", "fit"])
    while True:
        if kind == "infer":
            compute = rng.choice(["bf16", "fp32"])
            c = _layer("", _size(rng, 1, 4096), _size(rng, 64, 2048), _size(rng, 32, 2048),
                       rng.randint(2, 16), compute, "infer", rng.choice(["chebyshev", "jacobi", "hermite"]),
                       rng.choice(["bf16", "fp32"]) if compute == "bf16" else "fp32")
        elif kind == "train":
            c = _layer("", _size(rng, 128, 16384), _size(rng, 64, 2048), _size(rng, 32, 2048),
                       rng.randint(2, 16), rng.choice(["bf16", "fp32"]), "train",
                       rng.choice(["chebyshev", "chebyshev", "jacobi", "hermite"]))
        elif kind == "fp64":
            c = _layer("", _size(rng, 128, 8192), _size(rng, 16, 1024), _size(rng, 16, 1024),
                       rng.randint(2, 12), "fp64")
        elif kind == "high":
            c = _layer("", _size(rng, 128, 8192), _size(rng, 16, 512), _size(rng, 16, 512),
                       rng.randint(17, 64), "fp32")
        elif kind == "module":
            c = _stack("", "module", _size(rng, 32, 2048), (_size(rng, 64, 1024), _size(rng, 16, 256), 10),
                       rng.randint(2, 8), rng.choice(["fp32", "bf16"]), "ce", 1)
        else:
            c = _stack("", "fit", _size(rng, 64, 8192), (_size(rng, 16, 1024), _size(rng, 16, 512), _size(rng, 8, 64)),
                       rng.randint(2, 16), rng.choice(["fp32", "bf16"]), rng.choice(["ce", "mse"]), rng.randint(1, 20))
        # no more than the largest listed case: by flops, weighted by the rate that each precision can reach
        weight = 32.0 if c["compute"] == "fp64" or c["degree"] > 16 else 16.0 if c["compute"] == "fp32" else 1.0
        if work(c)["flops"] * weight <= 4.8e12:
            del c["name"]
            return c


# ---- what a program has before the call --------------------------------------

def _widths(case):
    return [int(w) for w in case["widths"].split("-")]


def _make_layer(family, in_dim, out_dim, degree, compute):
    if family == "jacobi":
        return kan_amd.JacobiKANLayer(in_dim, out_dim, degree, alpha=0.5, beta=0.5, compute=compute)
    if family == "hermite":
        # the Hermite polynomials of 3 tanh(x) grow with the degree: scaled down as a trained layer's would be
        top = max(1.0, math.sqrt(2.0 ** degree * math.factorial(degree)))
        return kan_amd.HermiteKANLayer(in_dim, out_dim, degree, init_scale=1.0 / (in_dim * (degree + 1) * top),
                                       compute=compute)
    return kan_amd.ChebyKANLayer(in_dim, out_dim, degree, compute=compute)


def _classifier_inputs(rows, width, classes, gen):
    """Images with most pixels dark, and their labels."""
    x = torch.rand(rows, width, device="cuda", generator=gen)
    x = x * (torch.rand(rows, width, device="cuda", generator=gen) >= 0.8)
    return x, torch.randint(0, classes, (rows,), device="cuda", generator=gen)


def _tensors(case, seed):
    """The case's seeded inputs: a layer's or stack's modules, x, and dy or the target."""
    torch.manual_seed(seed)
    gen = torch.Generator("cuda").manual_seed(seed + 1)
    compute = "fp32" if case["compute"] == "fp64" else case["compute"]
    if case["kind"] in ("infer", "train"):
        with torch.device("cuda"):
            layer = _make_layer(case["family"], case["in"], case["out"], case["degree"], compute)
        dtype = torch.float64 if case["compute"] == "fp64" else torch.float32
        x = torch.randn(case["rows"], case["in"], device="cuda", generator=gen).to(dtype)
        dy = torch.randn(case["rows"], case["out"], device="cuda", generator=gen).to(dtype) / case["rows"]
        if case["compute"] == "fp64":
            layer = layer.double()
        elif case["coeffs"] == "bf16":
            layer = layer.bfloat16()
        return layer, x, dy
    widths = _widths(case)
    with torch.device("cuda"):
        model = kan_amd.KANSequential(*[kan_amd.ChebyKANLayer(a, b, case["degree"], compute=compute)
                                        for a, b in zip(widths[:-1], widths[1:])])
    if case["loss"] == "ce":
        x, target = _classifier_inputs(case["rows"], widths[0], widths[-1], gen)
    else:
        x = torch.rand(case["rows"], widths[0], device="cuda", generator=gen) * 6 - 3
        w = torch.randn(widths[0], widths[-1], device="cuda", generator=gen) / math.sqrt(widths[0])
        target = x @ w + 0.1 * torch.randn(case["rows"], widths[-1], device="cuda", generator=gen)
    return model, x, target


def prepare(case, seed):
    module, x, other = _tensors(case, seed)
    state = {"kind": case["kind"], "module": module, "x": x, "other": other}
    if case["kind"] == "train":
        x.requires_grad_(True)
        state["opt"] = (torch.optim.SGD if case["compute"] == "fp64" else kan_amd.optim.SGD)(module.parameters(), lr=TRAIN_LR)
    elif case["kind"] == "module":
        state["opt"] = kan_amd.optim.SGD(module.parameters(), lr=FIT_LR)
    elif case["kind"] == "fit":
        state["ex"] = kan_amd.ResidentExecutor.from_sequential(
            module, case["rows"], compute=case["compute"], loss=case["loss"], optimizer="sgd", lr=FIT_LR)
        state["steps"] = case["steps"]
        state["layers"] = len(module)
    return state


# ---- one pass -----------------------------------------------------------------

def run(state):
    kind, module, x, other = state["kind"], state["module"], state["x"], state["other"]
    if kind == "infer":
        with torch.no_grad():
            return module(x)
    if kind == "train":
        state["opt"].zero_grad(set_to_none=True)
        x.grad = None
        y = module(x)
        y.backward(other)
        state["opt"].step()
        return {"y": y.detach(), "dx": x.grad, "dc": module.get_coefficients().grad}
    if kind == "module":
        state["opt"].zero_grad(set_to_none=True)
        logits = module(x)
        loss = torch.nn.functional.cross_entropy(logits, other)
        loss.backward()
        state["opt"].step()
        return {"loss": loss.detach(), "logits": logits.detach(),
                "dc": [m.get_coefficients().grad for m in module]}
    ex = state["ex"]
    # a mini-batch loop steps; full-batch epochs go in one call
    loss = ex.step(x, other) if state["steps"] == 1 else ex.fit(x, other, state["steps"])
    return {"loss": loss, "coeffs": [ex.get_coeffs(l) for l in range(state["layers"])]}


# ---- what a pass cannot do without --------------------------------------------

def work(case):
    d = case["degree"] + 1
    if case["kind"] in ("infer", "train"):
        b, i, o = case["rows"], case["in"], case["out"]
        size = 8 if case["compute"] == "fp64" else 4
        csize = 2 if case["coeffs"] == "bf16" else size
        if case["kind"] == "infer":
            return {"bytes": csize * i * o * d + size * b * (i + o), "flops": 2.0 * b * i * o * d}
        # forward: x, C -> y; backward: x, dy, C -> dx, dC; optimizer: dC, C -> C
        return {"bytes": size * (i * o * d * 4 + b * (i + o) * 2), "flops": 6.0 * b * i * o * d}
    widths, b = _widths(case), case["rows"]
    moved = flops = 0
    for l, (i, o) in enumerate(zip(widths[:-1], widths[1:])):
        moved += 4 * i * o * d * (4 if case["kind"] == "module" else 2)
        flops += 2.0 * b * i * o * d * (3 if l else 2)  # the first layer's inputs need no gradient
    moved += 4 * b * (widths[0] + widths[-1])
    return {"bytes": case["steps"] * moved, "flops": case["steps"] * flops}


# ---- the same results in 64 bits ----------------------------------------------

def _recurrence(family, n):
    """(a, b, c) of P_n(u) = (a u + b) P_{n-1}(u) - c P_{n-2}(u), n >= 1."""
    if family == "jacobi":
        al = be = 0.5
        if n == 1:
            return (al + be + 2) / 2, (al - be) / 2, 0.0
        s = 2 * n + al + be
        k = 2 * n * (n + al + be) * (s - 2)
        return (s - 1) * s * (s - 2) / k, (s - 1) * (al * al - be * be) / k, 2 * (n + al - 1) * (n + be - 1) * s / k
    if family == "hermite":
        return 2.0, 0.0, 2.0 * (n - 1)
    return (1.0, 0.0, 0.0) if n == 1 else (2.0, 0.0, 1.0)


def _basis(u, family, degree):
    """P_n(u) and P_n'(u), one degree at a time."""
    p1, p0 = torch.ones_like(u), torch.zeros_like(u)
    q1, q0 = torch.zeros_like(u), torch.zeros_like(u)
    yield p1, q1
    for n in range(1, degree + 1):
        a, b, c = _recurrence(family, n)
        p = (a * u + b) * p1 - c * p0
        q = a * p1 + (a * u + b) * q1 - c * q0
        yield p, q
        p1, p0, q1, q0 = p, p1, q, q1


def _exact_forward(x, c, family="chebyshev"):
    scale = 3.0 if family == "hermite" else 1.0
    y = torch.zeros(x.shape[0], c.shape[1], dtype=torch.float64, device=x.device)
    for n, (p, _) in enumerate(_basis(scale * torch.tanh(x), family, c.shape[2] - 1)):
        y += p @ c[:, :, n].contiguous()
    return y


def _exact_backward(x, c, dy, need_dx=True, family="chebyshev"):
    scale = 3.0 if family == "hermite" else 1.0
    t = torch.tanh(x)
    dx, dc = torch.zeros_like(x), torch.empty_like(c)
    for n, (p, q) in enumerate(_basis(scale * t, family, c.shape[2] - 1)):
        dc[:, :, n] = p.t().contiguous() @ dy
        if need_dx and n:
            dx += q * (dy @ c[:, :, n].t().contiguous())
    return dx * (1 - t * t) * scale if need_dx else None, dc


def _exact_step(x, coeffs, target, loss):
    """(loss, logits, coefficient gradients) of one training step on a stack of layers."""
    h = [x]
    for c in coeffs:
        h.append(_exact_forward(h[-1], c))
    y = h[-1]
    if loss == "ce":
        logp = torch.log_softmax(y, 1)
        value = -logp.gather(1, target[:, None]).mean()
        dy = logp.exp()
        dy[torch.arange(len(target), device=y.device), target] -= 1
        dy /= len(target)
    else:
        value = (y - target).square().mean()
        dy = 2 * (y - target) / y.numel()
    grads = [None] * len(coeffs)
    for l in range(len(coeffs) - 1, -1, -1):
        dy, grads[l] = _exact_backward(h[l], coeffs[l], dy, l > 0)
    return value, y, grads


def exact(case, seed):
    module, x, other = _tensors(case, seed)
    x = x.detach().double()
    if case["kind"] in ("infer", "train"):
        c = module.get_coefficients().detach().double()
        y = _exact_forward(x, c, case["family"])
        if case["kind"] == "infer":
            return y
        dx, dc = _exact_backward(x, c, other.double(), True, case["family"])
        return {"y": y, "dx": dx, "dc": dc}
    coeffs = [m.get_coefficients().detach().double() for m in module]
    target = other if case["loss"] == "ce" else other.double()
    if case["kind"] == "module":
        loss, logits, grads = _exact_step(x, coeffs, target, case["loss"])
        return {"loss": loss, "logits": logits, "dc": grads}
    losses = []
    for _ in range(case["steps"]):
        loss, _, grads = _exact_step(x, coeffs, target, case["loss"])
        losses.append(loss)
        coeffs = [c - FIT_LR * g for c, g in zip(coeffs, grads)]
    loss = losses[0] if case["steps"] == 1 else torch.stack(losses)
    return {"loss": loss, "coeffs": coeffs}


# ---- how far another correct implementation may be ----------------------------

def tolerance(case):
    """Relative 2-norm errors of results at each precision: about four times those against 64 bits."""
    if case["compute"] == "fp64":
        return {"rel": 1e-14}
    if case["compute"] == "bf16":
        # a stack's weights move little in a few steps, so their error is that much smaller
        return {"rel": 5e-4 if case["kind"] == "fit" else 1e-2}
    # above degree 16 the recurrence's own rounding grows with the degree
    return {"rel": 5e-6 if case["degree"] <= 16 else 3e-7 * case["degree"]}
