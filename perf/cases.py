"""Workloads by which the speed of this package is judged, through its public entry points.

``listed()`` gives twelve of them, ``draw(rng)`` more of the same kinds and ranges,
``prepare`` / ``run`` execute one, ``work`` says what it cannot do without and
``tolerance`` how far two correct implementations may lie apart.

A case is a flat dict.  ``op`` names what a pass does:

``loss``   ``SamplesLoss(...)`` on two clouds and the gradients a training step asks for
``hvp``    the same with a Hessian-vector product behind it (double backward in x)
``pots``   ``SamplesLoss(..., potentials=True)``: the dual potentials of a solve
``alt``    the alternating solver, called directly (the one with ``threshold``)
``map``    products with a known plan: barycentric map, plan-vector product both ways
``ctrans`` the hard c-transform of a dual potential, values and assignment

Sizes are those of the package's own five configurations, of its tests and of its documents
(2,000 x 3, 10,000 x 64, 50,000 x 64, 20,000 x 30,000 x 128, 8,192 x 1,536; 1,000 x 784 with
early stopping; products at n = 2,048), mini-batches, batches of point clouds, and odd sizes.
"""
import math

import torch

from flash_sinkhorn_amd import SamplesLoss, c_transform_fwd
from flash_sinkhorn_amd.kernels import (apply_plan_mat_flashstyle, apply_plan_vec_flashstyle,
                                        sinkhorn_flashstyle_alternating)

LOG2E = 1.4426950408889634
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}

# Every key of a case with its default: plain values only.
#   data     "normal" N(0, I) against N(shift, spread^2 I); "mixture" eight components with means
#            N(0, 4I), one mixture per cloud; "unit" N(0, I/d) (rows of length about one)
#   weights  "uniform" (none passed) or "dirichlet" (random masses, passed as a and b)
#   mass     total mass of b where weights are passed without normalisation
#   blur, scaling   the eps schedule; eps / n_iters instead of it where eps > 0
#   reach_x, reach_y  0: strict marginal
#   grad     which inputs the training step differentiates: "x", "xy" or ""
BASE = dict(op="loss", batch=0, n=0, m=0, d=0, dtype="f32", data="normal", shift=0.5, spread=1.0,
            weights="uniform", mass=1.0, blur=0.05, scaling=0.5, eps=0.0, n_iters=0,
            debias=False, half_cost=False, reach_x=0.0, reach_y=0.0, threshold=0.0, grad="x",
            cg=0)


def _case(name=None, **kw):
    c = dict(BASE)
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # A mini-batch of feature vectors inside a training step, with the default schedule:
        # the smallest calls, where the launches and the host are what the user waits for.
        _case("minibatch", n=256, m=256, d=16, debias=True, grad="xy"),
        # A batch of point clouds (registration, generative models of shapes): every item is a
        # solve of its own, all options at their defaults but the debiasing.
        _case("cloud batch", batch=8, n=1024, m=1024, d=3, debias=True),
        # Configuration 1: debiased loss and gradient of two small clouds at a fixed eps.
        _case("small clouds", n=2000, m=2000, d=3, shift=0.0, blur=0.1, eps=0.01, n_iters=100,
              half_cost=True, debias=True),
        # Odd and different sizes, random masses, both marginals relaxed, both gradients.
        _case("ragged unbalanced", n=3001, m=4567, d=33, weights="dirichlet", blur=0.1,
              reach_x=1.5, reach_y=1.5, grad="xy"),
        # Image-sized features in half precision, stopped early (1,000 x 784, threshold 1e-3).
        _case("early stopping", op="pots", n=1000, m=1000, d=784, dtype="bf16", data="unit",
              shift=0.0, eps=0.1, n_iters=100, threshold=1e-3, grad=""),
        # Configuration 2: debiased loss and gradient at 10,000 points.
        _case("medium debiased", n=10000, m=10000, d=64, blur=0.1, eps=0.01, n_iters=100,
              debias=True),
        # What a user who passes no options gets on large clouds, both gradients.
        _case("large schedule", n=30011, m=29989, d=64, grad="xy"),
        # Configuration 3: 100 iterations at 50,000 points, a peaked plan, and the gradient.
        _case("large peaked", n=50000, m=50000, d=64, data="mixture", blur=0.1, eps=0.01,
              n_iters=100),
        # Configuration 4: the alternating solver, unbalanced, ten iterations and one check.
        _case("alternating", op="alt", n=20000, m=30000, d=128, shift=0.0, spread=1.5,
              weights="dirichlet", mass=1.3, eps=0.0025, n_iters=10, reach_x=1.0, reach_y=1.0,
              threshold=1e-3, grad=""),
        # Configuration 5: wide rows; loss, gradient and one Hessian-vector product.
        _case("wide rows", op="hvp", n=8192, m=8192, d=1536, data="unit", shift=0.0, blur=0.5,
              eps=0.25, n_iters=50, cg=20),
        # A second-order step at the size the package's documents quote its CG loop for.
        _case("second order", op="hvp", n=2048, m=2048, d=64, data="unit", shift=0.0, blur=0.5,
              eps=0.25, n_iters=50, cg=50),
        # After a solve: the transport map and the marginals of a plan whose potentials are
        # kept (domain adaptation, label propagation), on new calls of the products.
        _case("transport map", op="map", n=20000, m=15013, d=32, data="unit", shift=0.0, eps=0.05,
              grad=""),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then sizes over the kind's whole range."""
    kind = rng.choice(["minibatch", "batch", "fixed", "schedule", "unbalanced", "features", "alt",
                       "hvp", "map", "ctrans"])
    near = lambda n, lo, hi: min(hi, max(lo, int(n * rng.uniform(0.6, 1.5))))  # noqa: E731
    if kind == "minibatch":
        n = _log_uniform(rng, 64, 1500)
        return _case(n=n, m=near(n, 64, 1500), d=_log_uniform(rng, 2, 128),
                     debias=rng.random() < 0.6, blur=rng.choice([0.05, 0.1, 0.3]),
                     grad=rng.choice(["x", "xy"]))
    if kind == "batch":
        n = _log_uniform(rng, 128, 2048)
        return _case(batch=rng.randint(2, 12), n=n, m=near(n, 128, 2048), d=rng.randint(2, 8),
                     debias=rng.random() < 0.6, blur=rng.choice([0.05, 0.1]))
    if kind == "fixed":  # a fixed eps, many iterations: small clouds to the largest
        n = _log_uniform(rng, 1000, 45000)
        return _case(n=n, m=near(n, 1000, 45000), d=_log_uniform(rng, 2, 64),
                     data=rng.choice(["normal", "mixture"]), blur=0.1, eps=0.01,
                     n_iters=rng.randint(20, 100), half_cost=rng.random() < 0.5,
                     debias=n <= 12000 and rng.random() < 0.5)
    if kind == "schedule":
        n = _log_uniform(rng, 1500, 40000)
        return _case(n=n, m=near(n, 1500, 40000), d=_log_uniform(rng, 2, 128),
                     debias=n <= 15000 and rng.random() < 0.5, blur=rng.choice([0.05, 0.1, 0.3]),
                     dtype=rng.choice(["f32", "f32", "f16"]), grad=rng.choice(["x", "xy"]))
    if kind == "unbalanced":
        n = _log_uniform(rng, 800, 15000)
        return _case(n=n, m=near(n, 800, 15000), d=_log_uniform(rng, 2, 100), weights="dirichlet",
                     blur=rng.choice([0.1, 0.2]), reach_x=rng.choice([0.0, 1.5]), reach_y=1.5,
                     grad=rng.choice(["x", "xy"]))
    if kind == "features":
        n = _log_uniform(rng, 500, 8192)
        return _case(op="pots", n=n, m=near(n, 500, 8192), d=_log_uniform(rng, 130, 1536),
                     dtype=rng.choice(["f32", "f16", "bf16"]), data="unit", shift=0.0, eps=0.1,
                     n_iters=rng.randint(20, 60), threshold=rng.choice([0.0, 1e-3]), grad="")
    if kind == "alt":
        n = _log_uniform(rng, 2000, 30000)
        return _case(op="alt", n=n, m=near(n, 2000, 30000), d=_log_uniform(rng, 8, 128), shift=0.0,
                     spread=1.5, weights="dirichlet", mass=1.3, eps=rng.choice([0.0025, 0.05, 0.5]),
                     n_iters=10, reach_x=rng.choice([0.0, 1.0]), reach_y=rng.choice([0.0, 1.0]),
                     threshold=rng.choice([0.0, 1e-3]), grad="")
    if kind == "hvp":
        n = _log_uniform(rng, 500, 8192)
        return _case(op="hvp", n=n, m=near(n, 500, 8192), d=_log_uniform(rng, 4, 1536),
                     data="unit", shift=0.0, blur=0.5, eps=0.25, n_iters=rng.randint(20, 50),
                     cg=rng.choice([20, 50]))
    n = _log_uniform(rng, 1000, 50000)
    sizes = dict(n=n, m=near(n, 1000, 50000), d=_log_uniform(rng, 2, 128), shift=0.0, grad="")
    if kind == "map":
        return _case(op="map", data="unit", eps=rng.choice([0.05, 0.2]), **sizes)
    return _case(op="ctrans", **sizes)


def _points(case, rows, gen, second):
    d, lead = case["d"], ((case["batch"],) if case["batch"] else ())
    p = torch.randn(lead + (rows, d), device="cuda", generator=gen)
    if case["data"] == "mixture":
        means = 2.0 * torch.randn(8, d, device="cuda", generator=gen)
        p += means[torch.randint(8, lead + (rows,), device="cuda", generator=gen)]
    elif second:
        p = case["spread"] * p + case["shift"]
    if case["data"] == "unit":
        p = p / math.sqrt(d)
    return p.to(DTYPES[case["dtype"]])


def _masses(case, rows, total, gen):
    if case["weights"] == "uniform":
        return torch.full((rows,), total / rows, device="cuda")
    w = -torch.log(torch.rand(rows, device="cuda", generator=gen).clamp_(min=1e-12))
    return total * w / w.sum()  # exponential variables over their sum: Dirichlet(1)


def _schedule(case):
    if case["eps"]:
        return dict(use_epsilon_scaling=False, eps=case["eps"], n_iters=case["n_iters"])
    return dict(blur=case["blur"], scaling=case["scaling"])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    state = {"case": case, "x": _points(case, case["n"], gen, False),
             "y": _points(case, case["m"], gen, True)}
    op = case["op"]
    if op in ("alt", "map") or case["weights"] != "uniform":
        state["a"] = _masses(case, case["n"], 1.0, gen)
        state["b"] = _masses(case, case["m"], case["mass"], gen)
    if op in ("loss", "hvp", "pots"):
        state["loss"] = SamplesLoss(
            debias=case["debias"], half_cost=case["half_cost"], potentials=op == "pots",
            reach_x=case["reach_x"] or None, reach_y=case["reach_y"] or None,
            threshold=case["threshold"] or None, hvp_max_cg_iter=case["cg"] or 300,
            **_schedule(case))
        state["x"].requires_grad_("x" in case["grad"])
        state["y"].requires_grad_("y" in case["grad"])
        if op == "hvp":
            state["v"] = torch.randn(case["n"], case["d"], device="cuda", generator=gen)
    if op == "map":
        # the potentials of a converged plan, as a program has them from its solve
        x, y, a, b = (state[k] for k in ("x", "y", "a", "b"))
        f, g = SamplesLoss(potentials=True, use_epsilon_scaling=False, eps=case["eps"],
                           n_iters=30)(a, x, b, y)
        state.update(f_hat=f - (x * x).sum(1), g_hat=g - (y * y).sum(1), log_a=a.log(),
                     log_b=b.log(), u=torch.rand(case["n"], device="cuda", generator=gen),
                     v=torch.rand(case["m"], device="cuda", generator=gen))
    if op == "ctrans":
        # a dual potential in the course of an optimisation: about the size of the costs
        state["psi"] = (0.1 * case["d"]) * torch.randn(case["m"], device="cuda", generator=gen)
    return state


def run(state):
    case, x, y = state["case"], state["x"], state["y"]
    op = case["op"]
    if op in ("loss", "hvp", "pots"):
        args = (x, y) if "a" not in state else (state["a"], x, state["b"], y)
        out = state["loss"](*args)
        if op == "pots":
            return {"f": out[0], "g": out[1]}
        total = out.sum() if case["batch"] else out
        if op == "hvp":
            (gx,) = torch.autograd.grad(total, x, create_graph=True)
            (hv,) = torch.autograd.grad((gx * state["v"]).sum(), x)
            return {"loss": out.detach(), "grad_x": gx.detach(), "hvp": hv}
        wanted = [t for t, k in ((x, "x"), (y, "y")) if k in case["grad"]]
        grads = torch.autograd.grad(total, wanted)
        return {"loss": out.detach(), **{"grad_%d" % i: g for i, g in enumerate(grads)}}
    if op == "alt":
        f, g = sinkhorn_flashstyle_alternating(
            x, y, state["a"], state["b"], eps=case["eps"], n_iters=case["n_iters"],
            reach_x=case["reach_x"] or None, reach_y=case["reach_y"] or None,
            threshold=case["threshold"] or None, check_every=10)
        return {"f": f, "g": g}
    if op == "map":
        plan = (x, y, state["f_hat"], state["g_hat"], state["log_a"], state["log_b"])
        return {"mapped": apply_plan_mat_flashstyle(*plan, y, eps=case["eps"], axis=1),
                "pv": apply_plan_vec_flashstyle(*plan, state["v"], eps=case["eps"], axis=1),
                "ptu": apply_plan_vec_flashstyle(*plan, state["u"], eps=case["eps"], axis=0)}
    values, assigned = c_transform_fwd(x, y, state["psi"])
    return {"values": values, "assigned": assigned}


def _steps(case):
    """Iterations of a solve (the first full one and the extrapolation included)."""
    if case["op"] == "alt":
        return case["n_iters"]
    if case["threshold"]:
        return min(case["n_iters"], 20) + 2  # what such a solve takes at the least: two checks
    if case["eps"]:
        return case["n_iters"] + 2
    diameter = 8.0 * math.sqrt(case["d"])  # of the joint bounding box, about
    return 2 + math.ceil(math.log(diameter / case["blur"]) / -math.log(case["scaling"])) + 2


def work(case):
    """Bytes: inputs read once, outputs written once.  Flops: one evaluation of the matrix of
    logits per iteration (2 d per pair; a pair of half-updates shares it in a symmetric step,
    not in an alternating one; a self problem's matrix is symmetric, half of it will do), and
    the products behind the solve."""
    n, m, d = case["n"], case["m"], case["d"]
    k = max(1, case["batch"])
    size = DTYPES[case["dtype"]].itemsize
    pairs, op = float(n) * m, case["op"]
    points = (n + m) * d
    passed = 4 * (n + m) if case["weights"] != "uniform" or op in ("alt", "map") else 0
    nbytes = points * size + passed
    if op == "ctrans":
        return {"bytes": nbytes + 4 * m + 12 * n, "flops": 2 * pairs * d}
    if op == "map":
        return {"bytes": nbytes + 8 * (n + m) + 4 * n * d + 4 * (n + m),
                "flops": (2 + 2) * pairs * d + 4 * pairs}
    steps = _steps(case)
    flops = steps * 2 * pairs * d * (2 if op == "alt" else 1)
    if case["debias"]:
        flops += steps * (float(n) * n + float(m) * m) * d
    if op in ("alt", "pots"):
        return {"bytes": nbytes + 4 * (n + m), "flops": flops}
    out = n * ("x" in case["grad"]) + m * ("y" in case["grad"])
    flops += 4 * pairs * d * len(case["grad"])
    if case["debias"]:
        flops += 4 * d * (float(n) * n * ("x" in case["grad"]) + float(m) * m * ("y" in case["grad"]))
    nbytes += out * d * size
    if op == "hvp":
        nbytes += 2 * n * d * 4
        flops += 5 * 4 * pairs * d  # matrix products and the second-order term; CG comes on top
    return {"bytes": k * nbytes + 4 * k, "flops": k * flops}


def tolerance(case):
    """32-bit sums give about 1e-5.  A gradient weighs points by 2^logit, and a logit of size L
    carries an error of the order of 2^-24 L whoever computes it; averaged over the points that
    share a weight about a quarter of that is left in a gradient, with single rows (one point
    against one other, nearly tied) far off the mean.  Differences of almost equal terms
    (debiasing, the Schur system of a Hessian-vector product) multiply what they inherit."""
    eps = case["eps"] or case["blur"] ** 2
    if case["op"] == "ctrans":  # two keys may tie to rounding
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
    if case["op"] == "pots" or case["op"] == "alt":
        return {"rel": 2e-5}
    scale = {"normal": 1.25 * case["d"], "mixture": 5.0 * case["d"], "unit": 1.0}[case["data"]]
    logit = 2.0 * (0.5 if case["half_cost"] else 1.0) * scale / eps * LOG2E
    rel = 2e-5 + logit * 2.0 ** -26
    if case["debias"]:
        rel *= 3
    if case["op"] == "hvp":
        rel += 3e-5
    if case["dtype"] != "f32":  # gradients come back in the inputs' type
        rel += 1e-3
    rel = min(rel, 0.01)
    return {"rel": rel, "max": min(100 * rel, 0.5)}
