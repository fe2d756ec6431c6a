"""Whole solves in one library call (small, medium and wide problems) and kept Hessian-vector products,
at the edges of their tiles and dispatch rules, against the fp64 oracle.

Tolerances: logits are formed from two fp16 planes a side (22 bits), so an inner product is off by
about 2^-21 |x| |y|, a potential by 2^-21 of the largest cost per step at most, which averaged
steps contract: 1e-5 of the largest potential.  A gradient multiplies the error of a logit (2^-21 of
the largest cost over eps, a few hundred here at most) with the spread of the cloud: 1e-4."""
import numpy as np
import pytest
import torch

import oracle
from tests.golden.recipe import inputs

pytestmark = pytest.mark.gpu
POT, GRAD = 1e-5, 1e-4


def dev(*arrs):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrs]


def rel_err(got, want):
    got = got.detach().cpu().numpy().astype(np.float64)
    want = np.asarray(want, dtype=np.float64)
    return float(np.abs(got - want).max() / max(np.abs(want).max(), 1e-30))


def check_symmetric(x, y, a, b, tol=POT, **kw):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    got = solve(*dev(x, y, a, b), return_prelast=True, **kw)
    want = oracle.sinkhorn_symmetric(x, y, a, b, return_prelast=True, **kw)
    for g, w in zip(got, want):
        assert rel_err(g, w) < tol


# ---- one launch per step: 32-row blocks, 16-column steps, eight or sixteen wavefronts ----
@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (1, 40, 3), (31, 33, 16), (32, 32, 17), (33, 257, 32),
                                   (255, 64, 33), (300, 1536, 64), (1537, 1505, 65),
                                   (70, 2100, 128), (4100, 100, 5)])
def test_small_steps(n, m, d):
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.3, n_iters=4)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.1, n_iters=3, rho_x=0.7, rho_y=2.0)


# schedules shorter than the steps that are enqueued before their length is known, and longer ones
@pytest.mark.parametrize("n,m,d", [(200, 300, 16), (130, 90, 100), (7100, 7050, 6)])
@pytest.mark.parametrize("cut", [1, 2, 3, 4, 5, 6, None])
def test_schedules_of_every_length(n, m, d, cut):
    if n > 1000 and cut not in (1, 5):
        pytest.skip("the oracle takes long; test_one_sweep_steps_of_a_full_schedule runs the full length")
    x, y, a, b = inputs(3, n, m, d, scale=0.5)
    for extrapolate in (True, False):
        from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
        kw = dict(blur=0.3, scaling=0.6, n_iters=cut, last_extrapolation=extrapolate)
        f, g = solve(*dev(x, y, a, b), **kw)
        wf, wg = oracle.sinkhorn_symmetric(x, y, a, b, **kw)
        assert rel_err(f, wf) < POT and rel_err(g, wg) < POT


# lengths of schedules, from boxes whose farthest corner lies in one block of rows and one column of either cloud (up to
# 64 blocks, sixteen threads a column or as many as 256 hold)
@pytest.mark.parametrize("n,m,d", [(2, 3, 1), (40, 33, 2), (300, 65, 3), (513, 290, 15), (260, 545, 16), (1100, 2049, 17),
                                   (2080, 700, 33), (90, 1000, 85), (333, 2100, 86), (2050, 100, 128), (4600, 4500, 5),
                                   (3073, 500, 128), (300, 5700, 69), (24600, 1000, 16)])
def test_lengths_of_schedules(n, m, d):
    from flash_sinkhorn_amd import SamplesLoss, _small
    rng = np.random.default_rng(n + d)
    base = [rng.uniform(-1, 1, (rows, d)).astype(np.float32) for rows in (n, m)]
    for cloud, row, col, far in [(0, 0, 0, 40.0), (0, -1, -1, -90.0), (1, 0, -1, 200.0), (1, -1, 0, -17.0), (0, n // 2, d // 2, 70.0)]:
        pts = [p.copy() for p in base]
        pts[cloud][row, col] = far
        boxes = [(p.min(0), p.max(0)) for p in pts]
        joint = (np.minimum(boxes[0][0], boxes[1][0]), np.maximum(boxes[0][1], boxes[1][1]))
        # (rounded otherwise than on the device by 2^-20 at most: a length that this changes would be seen as another seed's)
        diameters = [float(np.sqrt(((hi - lo).astype(np.float64) ** 2).sum())) for lo, hi in [joint] + boxes]
        want = [2 + max(0, int(np.ceil(2 * np.log(0.05 / D) / (2 * np.log(0.5))))) for D in diameters]
        loss = SamplesLoss(blur=0.05, scaling=0.5, debias=True)(*dev(*pts))
        assert torch.isfinite(loss) and _small._host_words(1)[:3].tolist() == want


# planes that are written anew for every eps, from rows by whole 16-byte words and one by one: the same bits
@pytest.mark.parametrize("n,m,d", [(4600, 4500, 36), (4600, 4500, 60), (4520, 4609, 64), (7200, 7100, 4), (7200, 7100, 20)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_planes_of_unaligned_rows(n, m, d, dtype):
    from flash_sinkhorn_amd import SamplesLoss
    x, y = (t.to(dtype) for t in dev(*inputs(7, n, m, d, scale=0.5)[:2]))
    def off(t):
        u = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view_as(t)
        return u.copy_(t)
    loss = SamplesLoss(blur=0.3, potentials=True)
    for got, want in zip(loss(off(x), off(y)), loss(x, y)):
        assert torch.equal(got, want)


# sums over one to several rows a thread and workgroup, of every combination of sides
@pytest.mark.parametrize("n,m", [(1, 1025), (1024, 3), (1030, 2049), (3073, 3072), (4500, 1000)])
@pytest.mark.parametrize("reach", [None, 1.3])
@pytest.mark.parametrize("debias", [False, True])
def test_losses_from_their_potentials(n, m, reach, debias):
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = dev(*inputs(5, n, m, 3, scale=0.5))
    kw = dict(use_epsilon_scaling=False, eps=0.2, n_iters=3, reach_x=reach, reach_y=reach)
    def cost(*clouds):
        f, g = (t.double() for t in SamplesLoss(potentials=True, **kw)(*clouds))
        if reach is None:
            return (clouds[0].double() * f).sum() + (clouds[2].double() * g).sum()
        rho = reach ** 2
        return (rho + 0.1) * ((clouds[0].double() * (1 - torch.exp(-f / rho))).sum() + (clouds[2].double() * (1 - torch.exp(-g / rho))).sum())
    want = cost(a, x, b, y)
    if debias:
        want = want - 0.5 * (cost(a, x, a, x) + cost(b, y, b, y))
    got = SamplesLoss(debias=debias, **kw)(a, x, b, y)
    # potentials are the same bits; sums of 4,500 terms in fp32 lie 1e-6 of their largest part apart
    assert abs(float(got) - float(want)) < 3e-6 * abs(float(cost(a, x, b, y)))


# ---- wide rows, one launch per step (up to 1e7 products and 4,096 keys): one and two rows a wavefront, pieces
# of 1,024 keys, and the sizes just past the line ----
@pytest.mark.parametrize("n,m,d", [(1, 1, 129), (5, 300, 130), (1023, 1025, 200), (1024, 1025, 140),
                                   (2400, 4096, 129), (30, 4097, 129), (2441, 4096, 131)])
def test_wide_steps_of_one_launch(n, m, d):
    x, y, a, b = inputs(n + d, n, m, d, scale=0.3)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.5, n_iters=4)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.2, n_iters=3, rho_x=0.7, rho_y=2.0)


# ---- narrower rows on kept products (8 steps and more; up to 3.4e7 bytes of them at d <= 64): planes of one to
# eight 16-column steps, blocks that are no multiple of the product's tiles, rows of 4,096 keys ----
@pytest.mark.parametrize("n,m,d", [(1, 1, 17), (31, 33, 33), (255, 257, 32), (1025, 769, 48), (2048, 2048, 64),
                                   (5, 4096, 65), (2050, 1023, 128)])
def test_steps_on_products_of_narrow_rows(n, m, d):
    x, y, a, b = inputs(n + d, n, m, d, scale=0.3)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.5, n_iters=8, rho_x=0.7, rho_y=2.0)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.5, n_iters=8)


@pytest.mark.parametrize("self_terms", [0, 1, 2])
@pytest.mark.parametrize("n,m,d,items", [(300, 257, 40, 3), (513, 200, 100, 1), (90, 300, 64, 2)])
def test_steps_on_products_equal_those_on_planes(n, m, d, items, self_terms):
    """The same call of the library with and without memory for the products: potentials of every problem, of every
    item of a batch, on a schedule by diameter."""
    import ctypes
    from flash_sinkhorn_amd import _lib, _small
    L, gen = _lib.lib(), torch.Generator(device="cuda").manual_seed(n + d)
    x, y = (0.4 * torch.randn(items, k, d, device="cuda", generator=gen) for k in (n, m))
    p = _small.Problem(x.data_ptr(), y.data_ptr(), None, None, None, n, m, d, items, 0.1, 0.5, 1.0, 0.0, 0.0, 1.5, 0.0,
                       0, 0, self_terms, 0, 1, 0, 0, 1, 1, 0)
    ref = ctypes.byref(p)
    size = L.fs_small_products_bytes(ref)
    assert size > 0
    results = []
    for kept in (0, size):
        ws = torch.empty(L.fs_small_workspace_bytes(ref), dtype=torch.uint8, device="cuda")
        # (what the memory held before shows in what is read past the end of a row)
        products = torch.full((max(kept, 4) // 4,), float("nan"), device="cuda")
        words = torch.empty(4 * items, dtype=torch.int32, pin_memory=True)
        rows = {0: n, 2: m, 4: n, 6: m}
        pots = {k: torch.zeros(items, r, device="cuda") for k, r in rows.items()
                if (self_terms < 2 if k < 4 else self_terms)}
        where = (ctypes.c_void_p * 8)(*[pots[k].data_ptr() if k in pots else None for k in range(8)])
        stream = torch.cuda.current_stream().cuda_stream
        assert L.fs_small_solve_products(ref, ws.data_ptr(), ws.numel(), products.data_ptr() if kept else None, kept,
                                         words.data_ptr(), None, None, stream) == 0
        assert L.fs_small_potentials(ref, ws.data_ptr(), ws.numel(), where, stream) == 0
        results.append(pots)
    # (a self problem's potentials are small differences of a shifted one and a norm, which is off by 2^-21 of
    # itself: the bound counts from the largest squared norm)
    norm = max(float((t * t).sum(-1).max()) for t in (x, y))
    for k, want in results[0].items():
        assert (results[1][k] - want).abs().max() <= 2.0 ** -21 * norm + POT * want.abs().max()
    if size > 4:  # memory too short for them is an error, not a write past its end
        assert L.fs_small_solve_products(ref, ws.data_ptr(), ws.numel(), products.data_ptr(), size - 1,
                                         words.data_ptr(), None, None, stream) != 0


@pytest.mark.parametrize("n,m,d,eps", [(300, 256, 17, 0.01), (1000, 1100, 33, 0.0625), (1500, 1400, 48, 0.01),
                                       (1000, 900, 100, 0.0625)])
def test_steps_on_products_are_as_exact_as_those_on_planes(monkeypatch, n, m, d, eps):
    """Forty steps on a peaked plan against fp64, where roundings that the two sides of a pair do not share add up.  With the cross
    products of every 16 columns added to hi * hi, and logits in base 2, errors are 1.12 to 1.6 times as large; formed alike they
    differ by the order of the sums alone, 0.2 % over eight seeds."""
    from flash_sinkhorn_amd import _graphs, _lib
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    clouds, want = [], []
    for seed in range(8):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        x, y = (torch.randn(k, d, device="cuda", generator=gen) + s for k, s in ((n, 0.0), (m, 0.5)))
        clouds.append((x, y, torch.full((n,), 1 / n, device="cuda"), torch.full((m,), 1 / m, device="cuda")))
        X, Y = x.double(), y.double()
        cost = ((X * X).sum(1)[:, None] + (Y * Y).sum(1)[None] - 2 * X @ Y.T) / eps
        f, g = torch.zeros_like(X[:, 0]), torch.zeros_like(Y[:, 0])
        for step in range(42):
            new = (-eps * torch.logsumexp(g[None] / eps - cost - np.log(m), 1),
                   -eps * torch.logsumexp(f[:, None] / eps - cost - np.log(n), 0))
            f, g = new if step in (0, 41) else ((f + new[0]) / 2, (g + new[1]) / 2)
        want.append((f, g))
    errors = []
    for planes in (False, True):
        _graphs.clear()  # (a replayed solve stays with the form it was captured in)
        if planes:
            monkeypatch.setattr(_lib.lib(), "fs_small_products_bytes", lambda p: 0)
        errors.append([float(sum((a - b).norm() / b.norm() for a, b in
                                 zip(solve(*c, use_epsilon_scaling=False, eps=eps, n_iters=40), w)))
                       for c, w in zip(clouds, want)])
    _graphs.clear()
    assert np.log(np.array(errors[0]) / errors[1]).mean() < 0.03


@pytest.mark.parametrize("n,m,d,far", [(1, 300, 33, 1e4), (300, 1, 70, 1e5), (1, 1, 20, 1e5), (1, 1500, 128, 1e6),
                                       (1, 700, 12, 1e5), (60, 1, 3, 1e6)])
@pytest.mark.parametrize("n_iters", [3, 10])  # (from 8 on, and from 17 columns, on kept products)
def test_small_steps_of_clouds_far_apart(n, m, d, far, n_iters):
    """Logits of 1e10 to 1e15, whose rounding in base 2 is past what an exponential holds: the largest of a row counts as one."""
    x, y, a, b = inputs(n + d, n, m, d, scale=0.3)
    if n == 1:
        x = x + np.float32(far)
    else:
        y = y + np.float32(far)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.25, n_iters=n_iters)
    check_symmetric(x, y, a, b, use_epsilon_scaling=True, blur=0.5, scaling=0.5)


# ---- both half-updates from one sweep (from 2e7 logits per step on): 256-row groups, chunks of
# 64-row tiles; eps at which steps go without running maxima, and at which the first ones may not ----
@pytest.mark.parametrize("n,m,d,eps", [(4481, 4703, 3, 0.5), (4608, 4352, 16, 0.01),
                                       (21000, 970, 33, 0.2), (900, 22400, 64, 0.002)])
def test_one_sweep_steps(n, m, d, eps):
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5)
    a[::7] = 0.0 if eps == 0.01 else a[::7]  # (rows without weight)
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=eps, n_iters=3)


# At a small fixed eps an averaged step halves how far the smallest sum lies below one, some hundreds of base-2 units at
# first, and relaxed marginals take every sum away from one: each of these ends in a step whose sums fit fp32 only
# with their logits shifted, or just before or behind one.
@pytest.mark.parametrize("n,m,d,eps,rho,mass", [(4513, 4481, 20, 0.01, None, 1.0), (4481, 4609, 9, 0.02, None, 1.0),
                                                (4700, 4650, 33, 0.02, 0.7, 1.3)])
@pytest.mark.parametrize("n_iters", [3, 4, 5, 6, 7])
def test_one_sweep_steps_whose_sums_need_a_shift(n, m, d, eps, rho, mass, n_iters):
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5, y_shift=0.2)
    check_symmetric(x, y, a, (mass * b).astype(b.dtype), use_epsilon_scaling=False, eps=eps, n_iters=n_iters,
                    rho_x=rho, rho_y=rho)


# ... and that a shift of either sign was taken off the last step's logits (small sums: units that end at coarse products, and
# every logit; large bounds: an eps that falls to a tenth from one step to the next).  Want: double precision.
@pytest.mark.parametrize("n,m,d,scale,rho,mass,kw,sign", [
    (4513, 4481, 20, 0.5, None, 1.3, dict(eps=0.003, entries=2, extrapolate=True), -1),
    (4513, 4481, 20, 0.5, 0.1, 1.0, dict(eps=0.005, entries=4, extrapolate=True), -1),
    (4513, 4481, 36, 0.5, None, 1.0, dict(blur=0.1, scaling=0.2, extrapolate=True), -1),
    (4513, 4481, 36, 0.5, None, 1.0, dict(blur=0.1, scaling=0.3, cut=5, extrapolate=False), 1),
    (4513, 4481, 36, 0.1, None, 1.0, dict(blur=0.1, scaling=0.25, cut=5, extrapolate=False), 1),
    (4513, 4481, 36, 0.5, 0.7, 1.0, dict(blur=0.1, scaling=0.3, cut=4, extrapolate=False), 1)])
def test_shifts_of_one_sweep_steps(n, m, d, scale, rho, mass, kw, sign):
    import ctypes

    from flash_sinkhorn_amd import _lib, _small
    from flash_sinkhorn_amd.kernels._common import epsilon_schedule, max_diameter
    x, y, a, b = inputs(n + d, n, m, d, scale=scale, y_shift=0.2)
    X, Y, A, B = dev(x, y, a, (mass * b).astype(b.dtype))
    eps = [kw["eps"]] * kw["entries"] if "eps" in kw else epsilon_schedule(
        max_diameter(X, Y), kw["blur"], kw["scaling"])[:kw.get("cut")]
    s = _small.solve(*_small.points(X, Y), A, B, items=1, cost_scale=1.0, rho_x=rho, rho_y=rho, normalize=False, self_terms=0,
                     want_values=False, want_loss=False, keep=True, **kw)
    at = _lib.lib().fs_small_last_step_offset(ctypes.byref(s.problem()), 0, 0)
    words = s.ws[at:at + 20].cpu().numpy()
    assert words[:4].view(np.int32)[0] == 1 and np.sign(words[16:].view(np.float32)[0]) == sign

    U, V = X.double(), Y.double()
    cost = (U * U).sum(1)[:, None] + (V * V).sum(1) - 2.0 * U @ V.T
    la, lb = A.double().log()[:, None], B.double().log()
    f, g = torch.zeros(n, 1, device="cuda").double(), torch.zeros(m, device="cuda").double()

    def halves(e):
        damp = 1.0 if rho is None else 1.0 / (1.0 + e / rho)
        return (-e * damp * torch.logsumexp((g - cost) / e + lb, 1, keepdim=True),
                -e * damp * torch.logsumexp((f - cost) / e + la, 0))
    f, g = halves(eps[0])
    for e in eps:
        new = halves(e)
        f, g = 0.5 * (f + new[0]), 0.5 * (g + new[1])
    if kw["extrapolate"]:
        f, g = halves(eps[-1])
    # (four steps' worth of 2^-21 of the largest cost each)
    off = 4.0 * 2.0 ** -21 * float(cost.max())
    for got, want in ((s.potentials("f")[0], f[:, 0]), (s.potentials("g")[0], g)):
        assert float((got.double() - want).abs().max()) < off


# ... of clouds so far from zero that a float's step at their potentials is 2 to 4 base-2 units: every cost is the same, so the
# bounds are as tight as they come, a few units below what fp32 holds
@pytest.mark.parametrize("rho", [None, 3.0])
@pytest.mark.parametrize("far,units", [(30.0, 200.0), (100.0, 600.0), (100.0, 1500.0), (250.0, 1000.0)])
def test_shifts_far_from_zero(far, units, rho):
    import ctypes

    from flash_sinkhorn_amd import _lib, _small
    n, m, d = 4500, 4480, 16
    per_unit = (2.8e7 - units) / (d * far * far)  # base-2 units per unit of cost
    x, y = torch.full((n, d), far, device="cuda"), torch.full((m, d), far - (units / per_unit / d) ** 0.5, device="cuda")
    a, b = torch.full((n,), 1 / n, device="cuda"), torch.full((m,), 1 / m, device="cuda")
    cost, eps = float(((x[0] - y[0]).double() ** 2).sum()), 1.0 / (per_unit * np.log(2.0))
    s = _small.solve(x, y, a, b, items=1, eps=eps, entries=1, cost_scale=1.0, rho_x=rho, rho_y=rho, normalize=False,
                     self_terms=0, want_values=False, extrapolate=False, want_loss=False, keep=True)
    at = _lib.lib().fs_small_last_step_offset(ctypes.byref(s.problem()), 0, 0)
    words = s.ws[at:at + 20].cpu().numpy()
    assert words[:4].view(np.int32)[0] == 1 and words[16:].view(np.float32)[0] != 0.0
    damp = 1.0 if rho is None else 1.0 / (1.0 + eps / rho)
    first = damp * cost
    want = 0.5 * first + 0.5 * damp * (cost - first)
    for which in "fg":  # (two steps; the logits of each are off by 2^-21 of the largest product, as everywhere)
        assert float((s.potentials(which)[0] - want).abs().max()) < 2.0 ** -19 * 2 * d * far * far


# a whole schedule on these kernels (planes written behind every step), as long as it is
def test_one_sweep_steps_of_a_full_schedule():
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(3, 4600, 4400, 36, scale=0.5)
    kw = dict(blur=0.5, scaling=0.5)
    want = oracle.sinkhorn_symmetric(x, y, a, b, return_prelast=True, **kw)
    X = dev(x, y, a, b)
    got = solve(*X, return_prelast=True, **kw) + solve(*X, last_extrapolation=False, **kw)
    for g, w in zip(got, want + want[2:]):
        assert rel_err(g, w) < POT


@pytest.mark.parametrize("n,m,d,eps", [(4700, 4650, 7, 0.05), (5100, 4209, 40, 0.01)])
def test_one_sweep_self_problems(n, m, d, eps):
    from flash_sinkhorn_amd.sinkhorn_solvers import sinkhorn_flashstyle_symmetric_self_pair as pair
    x, y, a, b = inputs(n, n, m, d, scale=0.5)
    X, Y, A, B = dev(x, y, a, b)
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=3)
    px, py = pair(X, A, Y, B, return_prelast=True, **kw)
    for got, (u, w) in ((px, (x, a)), (py, (y, b))):
        want = oracle.sinkhorn_symmetric(u, u, w, w, return_prelast=True, **kw)
        # (the potentials of a cloud against itself are far smaller than the costs, whose rounding is
        # what is left in them: absolute, 2^-21 of the largest cost in each of two sums)
        for p, q in ((got[0], want[0]), (got[2], want[2])):
            assert np.abs(p.cpu().numpy() - q).max() < 2.0 ** -20 * 4.0 * (u * u).sum(axis=1).max()


def symmetric_steps(x, y, a, b, eps, n_iters, rho=(None, None)):
    """The same updates in double precision on the GPU (more logits than numpy takes in good time)."""
    X, Y, A, B = (t.double() for t in dev(x, y, a, b))
    nx, ny = (X * X).sum(1), (Y * Y).sum(1)
    la, lb = A.clamp(min=1e-300).log(), B.clamp(min=1e-300).log()

    def half(u, v, pot, lw, norm, r):  # potentials of u's rows, without the norms
        damp = 1.0 if r is None else 1.0 / (1.0 + eps / r)
        out = torch.cat([torch.logsumexp((2.0 * p @ v.T + pot) / eps + lw, 1) for p in u.split(1024)])
        return -eps * damp * out - (1.0 - damp) * norm
    f, g = -nx, -ny
    f, g = half(X, Y, g, lb, nx, rho[0]), half(Y, X, f, la, ny, rho[1])
    for _ in range(n_iters):
        f, g = 0.5 * (f + half(X, Y, g, lb, nx, rho[0])), 0.5 * (g + half(Y, X, f, la, ny, rho[1]))
    last = half(X, Y, g, lb, nx, rho[0]), half(Y, X, f, la, ny, rho[1])
    return [t.cpu().numpy() for t in (last[0] + nx, last[1] + ny, f + nx, g + ny)]


# ---- peaked plans: units that end at their coarse products, then lists of those that do not.  Odd
# numbers of rows, one row group and one chunk, light rows, relaxed marginals, several clusters.  A
# step's error, 2^-21 of the largest cost for the logits and as much for what fp32 holds of norms and
# potentials, is halved by every averaged step: four of them at most ----
@pytest.mark.parametrize("n,m,d,eps,mixed,rho", [(4513, 4481, 64, 0.01, False, (None, None)),
                                                 (5003, 4201, 9, 0.002, False, (None, None)),
                                                 (4700, 4400, 33, 0.01, True, (2.0, 0.5)),
                                                 (250, 65000, 16, 0.003, True, (None, None)),
                                                 (65000, 310, 40, 0.02, False, (None, 1.0))])
def test_peaked_plans(n, m, d, eps, mixed, rho):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5, y_shift=0.2)
    if mixed:
        r = np.random.default_rng(d)
        means = r.standard_normal((6, d)).astype(np.float32)
        x, y = x + means[r.integers(6, size=n)], y + means[r.integers(6, size=m)]
        a[::7] *= 1e-3
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=30, rho_x=rho[0], rho_y=rho[1])
    got = solve(*dev(x, y, a, b), return_prelast=True, **kw)
    largest = sum(np.sqrt((t.astype(np.float64) ** 2).sum(1)).max() for t in (x, y)) ** 2
    for g, w in zip(got, symmetric_steps(x, y, a, b, eps, 30, rho)):
        assert np.abs(g.cpu().numpy() - w).max() < 4 * 2.0 ** -21 * largest


# ---- numbers that fp32 does not hold, or that the library would take for "none" ----
# One infinite weight leaves every key of its side as far away as the padding behind the last one, which then
# holds the largest logits of rows whose products are all negative: no such key may be kept (that every index
# stays inside is asserted where the kernel is compiled), and the next solve finds nothing of it.
def test_infinite_weights_on_opposite_clouds():
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(2, 8013, 7950, 20, scale=0.2)
    X, Y, A, B = dev(x + 1.0, y - 1.0, a, b)
    kw = dict(use_epsilon_scaling=False, eps=0.1, n_iters=12)
    want = solve(X, Y, A, B, **kw)
    W = A.clone()
    W[17] = float("inf")
    for weights in ((W, B), (A, W[:7950])):
        for t in solve(X, Y, *weights, **kw):
            assert not t.isfinite().all() or t.abs().max() > 1e3 * want[0].abs().max()
    assert all(torch.equal(g, w) for g, w in zip(solve(X, Y, A, B, **kw), want))


# A weight that is not a number is none, as one of zero is, and nothing is known of its side's mass: the steps take both sides
# apart then, whichever side it is on.
@pytest.mark.parametrize("of_x", [False, True])
def test_weights_that_are_no_numbers(of_x):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(5, 4620, 4513, 12, scale=0.5)
    X, Y, A, B = dev(x, y, a, b)
    heavy, at = (A, 17) if of_x else (B, 4400)
    heavy *= 2.0 ** 30
    kw = dict(use_epsilon_scaling=False, eps=0.05, n_iters=6)
    heavy[at] = 0.0
    want = solve(X, Y, A, B, **kw)
    heavy[at] = float("nan")
    for g, w in zip(solve(X, Y, A, B, **kw), want):
        assert rel_err(g, w.cpu().numpy()) < POT


@pytest.mark.parametrize("d", [4, 200])
def test_relaxations_of_zero_and_less_are_not_strict_marginals(d):
    from flash_sinkhorn_amd import SamplesLoss, sinkhorn_solvers as S
    from flash_sinkhorn_amd.hvp import hvp_x_sqeuclid_from_potentials as hvp
    x, y, a, b = inputs(2, 60, 50, d, scale=1.0 / np.sqrt(d))
    X, Y, A, B = dev(x, y, a, b)
    fixed = dict(use_epsilon_scaling=False, eps=0.2, n_iters=3)
    for rho in (dict(rho=0.0), dict(rho_x=0.0), dict(rho_y=0.0)):
        with pytest.raises(ZeroDivisionError):
            S.sinkhorn_flashstyle_symmetric(X, Y, A, B, **rho, **fixed)
        with pytest.raises(ZeroDivisionError):
            S.sinkhorn_flashstyle_alternating(X, Y, A, B, eps=0.2, n_iters=3, **rho)
    with pytest.raises(ZeroDivisionError):
        S.sinkhorn_flashstyle_symmetric_self_pair(X, A, Y, B, rho=0.0, **fixed)
    for rho in (dict(rho_x=0.0), dict(rho_y=0.0)):
        with pytest.raises(ZeroDivisionError):
            hvp(X, Y, A.log(), B.log(), X, eps=0.2, **rho)
    # (two launches a step and damping on the host: always the general path)
    for rho in (-0.7, 1e-50):
        f, g = S.sinkhorn_flashstyle_symmetric(X, Y, A, B, rho=rho, **fixed)
        u, v = S.sinkhorn_flashstyle_symmetric(X, Y, A, B, rho=rho, fused=False, **fixed)
        assert torch.allclose(f, u, atol=1e-5, rtol=1e-5) and torch.allclose(g, v, atol=1e-5, rtol=1e-5)
    assert SamplesLoss(reach=1e-25, **fixed)(X, Y).isnan()  # 0 * inf: rho is zero on the device
    for fn in (lambda: SamplesLoss(blur=1e-30)(X, Y), lambda: SamplesLoss(blur=1e-30, potentials=True)(X, Y),
               lambda: S.sinkhorn_flashstyle_symmetric(X, Y, A, B, blur=1e-30),
               lambda: S.sinkhorn_flashstyle_symmetric_self_pair(X, A, Y, B, blur=1e-30)):
        with pytest.raises(RuntimeError, match="bad argument"):
            fn()


# ---- kept products: 256-column strips, tiles of 64, 128 and 256, both shapes of the sweep ----
@pytest.mark.parametrize("n,m,d", [(1, 1, 129), (63, 257, 130), (256, 255, 144), (1000, 1000, 784),
                                   (2100, 4099, 200), (513, 2049, 1536)])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_kept_products(n, m, d, dtype):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    x, y = x.astype(dtype), y.astype(dtype)
    kw = dict(use_epsilon_scaling=False, eps=0.1, n_iters=4, rho_y=1.5)
    f, g = solve(*dev(x, y, a, b), **kw)
    wf, wg = oracle.sinkhorn_symmetric(x.astype(np.float64), y.astype(np.float64), a, b, **kw)
    assert rel_err(f, wf) < POT and rel_err(g, wg) < POT


# products in tiles of 64 with eight stages: odd and even numbers of 16-column steps, up to the number of tiles where four take over
@pytest.mark.parametrize("n,m,d", [(70, 90, 131), (65, 300, 160), (130, 64, 163), (300, 200, 192), (500, 129, 239), (90, 260, 300),
                                   (1400, 1500, 145), (1500, 1600, 150)])
def test_kept_products_of_small_tiles(n, m, d):
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.1, n_iters=3)


@pytest.mark.parametrize("threshold", [None, 1e-3])
def test_kept_products_of_a_batch(threshold):
    from flash_sinkhorn_amd import SamplesLoss
    rng = np.random.default_rng(5)
    # (the second item is spread out further and stops later)
    x, y = (rng.standard_normal((3, k, 200)).astype(np.float32) * np.float32([[[0.05]], [[0.1]], [[0.07]]])
            for k in (300, 530))
    kw = dict(use_epsilon_scaling=False, eps=0.1, n_iters=30)
    f, g = SamplesLoss(potentials=True, threshold=threshold, inner_iterations=3, **kw)(*dev(x, y))
    for i in range(3):
        a, b = (np.full(k, 1.0 / k, np.float32) for k in (300, 530))
        wf, wg = oracle.sinkhorn_symmetric(x[i], y[i], a, b, threshold=threshold, check_every=3, **kw)
        assert rel_err(f[i], wf) < POT and rel_err(g[i], wg) < POT


# rows that do not start at multiples of 16 bytes take the narrow loads
def test_kept_products_of_unaligned_rows():
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(5, 300, 200, 160, scale=0.1)
    kw = dict(use_epsilon_scaling=False, eps=0.1, n_iters=3)
    X, Y, A, B = dev(x, y, a, b)
    buf = torch.empty(X.numel() + 1, device="cuda")
    U = buf[1:].view(X.shape)
    U.copy_(X)
    assert all(torch.equal(p, q) for p, q in zip(solve(U, Y, A, B, **kw), solve(X, Y, A, B, **kw)))


# ---- early stopping on the device ----
@pytest.mark.parametrize("n,m,d", [(300, 200, 20), (400, 300, 200), (4700, 4500, 8)])
def test_early_stopping(n, m, d):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(9, n, m, d, scale=1.0 / np.sqrt(d))
    kw = dict(use_epsilon_scaling=False, eps=0.5, n_iters=60, threshold=1e-3, check_every=4,
              return_n_iters=True)
    *got, used = solve(*dev(x, y, a, b), **kw)
    *want, wused = oracle.sinkhorn_symmetric(x, y, a, b, **kw)
    assert used == wused < 62
    assert all(rel_err(p, q) < POT for p, q in zip(got, want))


# the host may look at a check only after the device has run the next one as well (here: always, every
# launch is waited for), and find there that everything has stopped
def test_early_stopping_seen_early():
    import os
    import subprocess
    import sys
    code = """
import sys
import torch
from tests import test_gpu_whole_solves as t
for n, m, d in ((300, 200, 20), (400, 300, 200), (4700, 4500, 8)):
    t.test_early_stopping(n, m, d)
for threshold in (None, 1e-3):
    t.test_alternating(333, 65, 16, threshold)
t.test_kept_products_of_a_batch(1e-3)
"""
    env = dict(os.environ, AMD_SERIALIZE_KERNEL="3", PYTHONPATH=os.getcwd())
    res = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stderr[-3000:]


@pytest.mark.parametrize("n,m,d", [(1, 5, 2), (333, 65, 16), (200, 1600, 40), (2100, 2000, 128)])
@pytest.mark.parametrize("threshold", [None, 1e-3])
def test_alternating(n, m, d, threshold):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_alternating as solve
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    kw = dict(eps=0.3, n_iters=7 if threshold is None else 50, rho_x=0.8, threshold=threshold,
              check_every=3, return_n_iters=True)
    *got, used = solve(*dev(x, y, a, b * 1.2), **kw)
    *want, wused = oracle.sinkhorn_alternating(x, y, a, b * 1.2, **kw)
    assert used == wused
    assert all(rel_err(p, q) < POT for p, q in zip(got, want))


# more rows than a whole solve takes, few enough logits for one: the general path
@pytest.mark.parametrize("n,m", [(65537, 200), (150, 70000)])
def test_alternating_of_long_and_thin_problems(n, m):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_alternating as solve
    x, y, a, b = inputs(1, n, m, 3, scale=0.5)
    f, g = solve(*dev(x, y, a, b), eps=0.3, n_iters=3)
    wf, wg = oracle.sinkhorn_alternating(x, y, a, b, eps=0.3, n_iters=3)
    assert rel_err(f, wf) < POT and rel_err(g, wg) < POT


# ---- the loss, its gradients, and what a training program does with them ----
def expected(x, y, a, b, debias, eps, n_iters):
    def one(u, v, wu, wv):
        f, g, fp, gp = oracle.sinkhorn_symmetric(u, v, wu, wv, use_epsilon_scaling=False, eps=eps,
                                                 n_iters=n_iters, return_prelast=True)
        gu, gv = oracle.grad_barycentric(u, v, wu, wv, fp, gp, eps)
        return oracle.sinkhorn_cost(wu, wv, f, g, eps), gu, gv
    c, gx, gy = one(x, y, a, b)
    if debias:
        cx, g1, g2 = one(x, x, a, a)
        cy, h1, h2 = one(y, y, b, b)
        c, gx, gy = c - 0.5 * (cx + cy), gx - 0.5 * (g1 + g2), gy - 0.5 * (h1 + h2)
    return c, gx, gy


@pytest.mark.parametrize("n,m,d", [(1, 3, 1), (33, 31, 16), (100, 129, 33), (257, 64, 65), (90, 1700, 128),
                                   (4600, 4400, 10)])
@pytest.mark.parametrize("debias", [False, True])
def test_loss_and_gradients(n, m, d, debias):
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5, y_shift=0.5)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_(), Y.requires_grad_()
    steps = 4 if n < 1000 else 1
    fn = SamplesLoss("sinkhorn", use_epsilon_scaling=False, eps=0.2, n_iters=steps, debias=debias,
                     half_cost=False)
    loss = fn(A, X, B, Y)
    assert loss.shape == ()
    gx, gy = torch.autograd.grad(loss, [X, Y])
    c, wx, wy = expected(x, y, a, b, debias, 0.2, steps)
    # (a debiased loss or gradient is a difference: its error is that of the parts)
    _, px, py = expected(x, y, a, b, False, 0.2, steps)
    assert abs(loss.item() - c) < 1e-4 * (abs(c) + (0.5 * d if debias else 0.0))
    for g, w, p in ((gx, wx, px), (gy, wy, py)):
        assert np.abs(g.cpu().numpy() - w).max() < GRAD * np.abs(p).max()


# ---- planes of 48 and 96 columns: the last one they hold and the first they do not, in every form ----
@pytest.mark.parametrize("n,m,d", [(33, 70, 33), (300, 257, 47), (65, 1600, 48), (300, 130, 49), (90, 129, 65),
                                   (257, 200, 95), (40, 300, 96), (130, 90, 97), (4500, 4471, 48)])
def test_columns_of_the_planes(n, m, d):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_alternating as alternating
    x, y, a, b = inputs(n + d, n, m, d, scale=0.5, y_shift=0.2)
    # (below eight steps on planes, from there on, where they fit, on kept products)
    for n_iters in (3, 9)[:1 if n > 1000 else 2]:
        check_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.1, n_iters=n_iters)
        got = alternating(*dev(x, y, a, b), eps=0.1, n_iters=n_iters)
        for g, w in zip(got, oracle.sinkhorn_alternating(x, y, a, b, eps=0.1, n_iters=n_iters)):
            assert rel_err(g, w) < POT
    for debias in (False, True)[:1 if n > 1000 else 2]:
        test_loss_and_gradients(n, m, d, debias)


# ---- medium problems: both directions of the one-sweep kernels at small eps ----
def gradient_bound(x, y, eps):
    """Largest error of a barycentre whose logits are off by delta: every weight by a factor e^(+-delta),
    so at most 2 delta times the cloud's extent.  delta: inner products of two planes a side (2^-21 of
    |x| |y|, twice over eps), potentials and norms that fp32 holds (2^-23 of the largest cost, over eps)."""
    nx, ny = (np.sqrt((t.astype(np.float64) ** 2).sum(1)).max() for t in (x, y))
    delta = (2.0 ** -21 * 2.0 * nx * ny + 2.0 ** -23 * 2.0 * (nx + ny) ** 2) / eps
    return 2.0 * delta * (nx + ny)


# (6 steps end in a two-sided one, 25 in one that goes along its lists)
@pytest.mark.parametrize("n,m,d,eps,n_iters", [(4500, 4470, 64, 0.01, 6), (5003, 4201, 9, 0.003, 6),
                                               (4513, 4490, 64, 0.01, 25), (310, 65000, 33, 0.01, 25),
                                               (65000, 290, 16, 0.003, 25)])
def test_one_sweep_gradients_at_small_eps(n, m, d, eps, n_iters):
    from flash_sinkhorn_amd import SamplesLoss
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(n, n, m, d, scale=0.5, y_shift=0.2)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_(), Y.requires_grad_()
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=n_iters)
    gx, gy = torch.autograd.grad(SamplesLoss("sinkhorn", normalize=False, **kw)(A, X, B, Y), [X, Y])
    # at the potentials of the same solve: what is left is the gradient's own error
    _, _, fp, gp = solve(X.detach(), Y.detach(), A, B, return_prelast=True, **kw)
    wx, wy = oracle.grad_barycentric(x, y, a, b, fp.cpu().numpy(), gp.cpu().numpy(), eps)
    bound = gradient_bound(x, y, eps)
    for got, want, w in ((gx, wx, a), (gy, wy, b)):
        off = np.abs(got.cpu().numpy() - want).max(axis=1)
        assert (off <= 2.0 * w * bound).all()


# Large clouds at a fixed eps: on either side of the line between these kernels and the general path both give
# the same.  (What two solves may lie apart: a potential by four steps' worth of 2^-21 of the largest cost
# each, a gradient by its own bound and by what such potentials do to the logits.)
@pytest.mark.parametrize("n,m,d,n_iters,small", [(25013, 26000, 40, 3, False), (25013, 26000, 40, 4, True),
                                                 (53000, 50007, 33, 30, True), (53000, 50007, 33, 20, False),
                                                 (53000, 50007, 32, 9, True), (53000, 50007, 16, 8, False)])
def test_both_routes_of_large_losses_agree(monkeypatch, n, m, d, n_iters, small):
    from flash_sinkhorn_amd import SamplesLoss, _small
    assert _small._size_ok(n, m, d, True, 0, False, 1, n_iters) == small
    assert _small._size_ok(n, m, d, True, 1, False, 1, n_iters) and _small._size_ok(n, m, d, False, 0, False)
    x, y, a, b = inputs(n, n, m, d, scale=0.5, y_shift=0.2)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_(), Y.requires_grad_()
    eps, out = 0.05, {}
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=n_iters, normalize=False)
    for route in (True, False):
        with monkeypatch.context() as forced:
            forced.setattr(_small, "_size_ok", lambda *_: route)
            loss = SamplesLoss("sinkhorn", **kw)(A, X, B, Y)
            out[route] = [loss.detach(), *torch.autograd.grad(loss, [X, Y]),
                          *SamplesLoss("sinkhorn", potentials=True, **kw)(A, X.detach(), B, Y.detach())]
    loss = SamplesLoss("sinkhorn", **kw)(A, X, B, Y)
    assert torch.equal(loss, out[small][0])
    largest = sum(np.sqrt((t.astype(np.float64) ** 2).sum(1)).max() for t in (x, y)) ** 2
    off = 4 * 2.0 ** -21 * largest
    (l0, gx0, gy0, f0, g0), (l1, gx1, gy1, f1, g1) = out[False], out[True]
    assert (f0 - f1).abs().max() < 2 * off and (g0 - g1).abs().max() < 2 * off and abs(l0 - l1) < 4 * off
    bound = 2 * gradient_bound(x, y, eps) + 2 * (4 * off / eps) * largest ** 0.5
    for u, v, w in ((gx0, gx1, A), (gy0, gy1, B)):
        assert ((u - v).abs().amax(1) <= 2.0 * w * bound).all()


# ... in every form that the line sends to these kernels above 2.6e9 logits
@pytest.mark.parametrize("form", ["debiased", "batch", "float16", "bfloat16", "relaxed", "no weights", "strided",
                                  "no extrapolation", "early stopping", "half cost"])
def test_both_routes_of_the_largest_losses_agree_in_every_form(monkeypatch, form):
    from flash_sinkhorn_amd import SamplesLoss, _small
    n, m, d, eps = 52001, 50400, 14, 0.05
    x, y, a, b = inputs(11, n, m, d, scale=0.5, y_shift=0.2)
    X, Y, A, B = dev(x, y, a, b)
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=16, normalize=False)
    if form == "debiased":
        kw.update(debias=True)
    if form in ("float16", "bfloat16"):
        X, Y = X.to(getattr(torch, form)), Y.to(getattr(torch, form))
    if form == "relaxed":
        kw.update(reach_x=1.5, reach_y=2.0)
    if form == "no extrapolation":
        kw.update(last_extrapolation=False)
    if form == "early stopping":
        kw.update(threshold=1e-2, inner_iterations=3)
    if form == "half cost":
        kw.update(half_cost=True)
    if form == "batch":
        X, Y, A, B = (torch.stack([t, t.roll(5, 0)]) for t in (X, Y, A, B))
    if form == "strided":
        X = X.t().contiguous().t()
    X.requires_grad_(), Y.requires_grad_()
    args = (X, Y) if form == "no weights" else (A, X, B, Y)
    runs, solve = [], _small.solve
    monkeypatch.setattr(_small, "solve", lambda *p, **q: runs.append(1) or solve(*p, **q))
    fn, out = SamplesLoss("sinkhorn", **kw), []
    for route in ("these", "general"):
        if route == "general":
            monkeypatch.setattr(_small, "_size_ok", lambda *_: False)
        loss = fn(*args)
        out.append([loss.detach(), *torch.autograd.grad(loss.sum(), [X, Y])])
        assert len(runs) == 1
    x, y = (t.detach().float().reshape(-1, d).cpu().numpy() for t in (X, Y))
    largest = sum(np.sqrt((t.astype(np.float64) ** 2).sum(1)).max() for t in (x, y)) ** 2
    off = 4 * 2.0 ** -21 * largest + (1e-2 if form == "early stopping" else 0.0)
    (l0, gx0, gy0), (l1, gx1, gy1) = out
    assert l0.shape == l1.shape and (l0 - l1).abs().max() < 12 * off
    bound = 3 * (2 * gradient_bound(x, y, eps) + 2 * (4 * off / eps) * largest ** 0.5)
    grain = {"float16": 2.0 ** -10, "bfloat16": 2.0 ** -7}.get(form, 0.0)
    for u, v, w in ((gx0, gx1, A), (gy0, gy1, B)):
        w = torch.full_like(w, 1.0 / w.shape[-1]) if form == "no weights" else w
        assert u.dtype == v.dtype
        u, v = u.float(), v.float()
        assert ((u - v).abs().amax(-1) <= 2.0 * w * bound + grain * u.abs().amax(-1) + (grain and 2.0 ** -24)).all()


def test_one_sweep_gradients_of_peaked_self_problems():
    from flash_sinkhorn_amd import SamplesLoss
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    from flash_sinkhorn_amd.sinkhorn_solvers import sinkhorn_flashstyle_symmetric_self_pair as pair
    n, m, d, eps = 3313, 3190, 20, 0.02
    x, y, a, b = inputs(n, n, m, d, scale=0.5, y_shift=0.2)
    x[1::2] = x[:-1:2] + 0.02 * x[1::2]  # (a point's own weight is not all of its row)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_(), Y.requires_grad_()
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=25)
    gx, gy = torch.autograd.grad(SamplesLoss("sinkhorn", normalize=False, debias=True, **kw)(A, X, B, Y), [X, Y])
    X, Y = X.detach(), Y.detach()
    _, _, fp, gp = (t.cpu().numpy() for t in solve(X, Y, A, B, return_prelast=True, **kw))
    (_, _, fx, _), (_, _, fy, _) = pair(X, A, Y, B, return_prelast=True, **kw)
    fx, fy = fx.cpu().numpy(), fy.cpu().numpy()
    wx, wy = oracle.grad_barycentric(x, y, a, b, fp, gp, eps)
    # (a self problem has its gradient once for either role of the points, and is taken off by half)
    wx = wx - oracle.grad_barycentric(x, x, a, a, fx, fx, eps)[0]
    wy = wy - oracle.grad_barycentric(y, y, b, b, fy, fy, eps)[0]
    for got, want, w, (u, v) in ((gx, wx, a, (x, x)), (gy, wy, b, (y, y))):
        off = np.abs(got.cpu().numpy() - want).max(axis=1)
        assert (off <= 2.0 * w * (gradient_bound(x, y, eps) + gradient_bound(u, v, eps))).all()


def test_one_sweep_debiased_schedule():
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(7, 3230, 3190, 36, scale=0.5, y_shift=0.5)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_(), Y.requires_grad_()
    kw = dict(blur=0.5, scaling=0.5)
    loss = SamplesLoss("sinkhorn", debias=True, normalize=False, **kw)(A, X, B, Y)
    gx, gy = torch.autograd.grad(loss, [X, Y])

    def one(u, v, wu, wv):
        f, g, fp, gp = oracle.sinkhorn_symmetric(u, v, wu, wv, return_prelast=True, **kw)
        return (oracle.sinkhorn_cost(wu, wv, f, g, 0.25),) + oracle.grad_barycentric(u, v, wu, wv, fp, gp, 0.25)
    c, px, py = one(x, y, a, b)
    cx, g1, g2 = one(x, x, a, a)
    cy, h1, h2 = one(y, y, b, b)
    assert abs(loss.item() - (c - 0.5 * (cx + cy))) < 1e-4 * abs(c)
    for got, w, p in ((gx, px - 0.5 * (g1 + g2), px), (gy, py - 0.5 * (h1 + h2), py)):
        assert np.abs(got.cpu().numpy() - w).max() < GRAD * np.abs(p).max()


@pytest.mark.parametrize("n,m,d,kw", [(4600, 4400, 10, dict(use_epsilon_scaling=False, eps=0.05, n_iters=5)),
                                      (3230, 3190, 36, dict(blur=0.5, debias=True))])
def test_one_sweep_batch_equals_its_items(n, m, d, kw):
    from flash_sinkhorn_amd import SamplesLoss
    gen = torch.Generator(device="cuda").manual_seed(3)
    X = 0.5 * torch.randn(2, n, d, device="cuda", generator=gen)
    X[1] *= 3.0  # (a longer schedule)
    Y = 0.5 * torch.randn(2, m, d, device="cuda", generator=gen)
    X.requires_grad_(), Y.requires_grad_()
    fn = SamplesLoss("sinkhorn", **kw)
    loss = fn(X, Y)
    grads = torch.autograd.grad(loss.sum(), [X, Y])
    for i in range(2):
        Xi, Yi = (t[i].detach().clone().requires_grad_() for t in (X, Y))
        li = fn(Xi, Yi)
        # (items of a batch are cut into other chunks: sums in another order)
        assert abs(loss[i].item() - li.item()) < 1e-5 * (1.0 + d * 3.0)
        for g, w in zip(grads, torch.autograd.grad(li, [Xi, Yi])):
            assert rel_err(g[i], w.cpu().numpy()) < GRAD


def test_gradients_of_double_precision_points_are_refused_at_every_size():
    from flash_sinkhorn_amd import SamplesLoss
    for n in (60, 30000):
        X = torch.rand(n, 24, device="cuda", dtype=torch.float64, requires_grad=True)
        W = torch.full((n,), 1.0 / n, device="cuda", requires_grad=True)
        fn = SamplesLoss("sinkhorn", blur=0.5, n_iters=1)
        with pytest.raises(ValueError, match="Unsupported dtype"):
            torch.autograd.grad(fn(X, X.detach() + 0.1), X)
        torch.autograd.grad(fn(W, X.detach(), W.detach(), X.detach() + 0.1), W)


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("types", [(torch.float64, torch.float64), (torch.float32, torch.float64),
                                   (torch.float16, torch.float32)])
def test_the_loss_keeps_the_type_that_its_weights_give_it(normalize, types):
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(8, 61, 50, 4)
    X, Y, A, B = dev(x, y, a, b)
    A, B = A.to(types[0]), B.to(types[1])
    loss = SamplesLoss("sinkhorn", normalize=normalize)(A, X, B, Y)
    assert loss.dtype == (torch.float32 if normalize else torch.promote_types(torch.float32,
                                                                             torch.promote_types(*types)))


def test_weights_elsewhere_are_refused():
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(8, 61, 50, 4)
    X, Y, A, B = dev(x, y, a, b)
    for kw in (dict(), dict(potentials=True), dict(debias=True),
               dict(backend="alternating", use_epsilon_scaling=False, eps=0.1, n_iters=3)):
        for w in ((A.cpu(), B), (A, B.cpu())):
            with pytest.raises(ValueError, match="same device"):
                SamplesLoss("sinkhorn", **kw)(w[0], X, w[1], Y)


def test_batch_equals_its_items():
    from flash_sinkhorn_amd import SamplesLoss
    rng = np.random.default_rng(4)
    x, y = (rng.standard_normal((5, k, 6)).astype(np.float32) * s for k, s in ((150, 0.5), (97, 0.7)))
    X, Y = dev(x, y)
    X.requires_grad_()
    fn = SamplesLoss("sinkhorn", debias=True, blur=0.1)  # items have schedules of their own
    loss = fn(X, Y)
    gx, = torch.autograd.grad(loss.sum(), X)
    for i in range(5):
        Xi = X[i].detach().clone().requires_grad_()
        li = fn(Xi, Y[i])
        gi, = torch.autograd.grad(li, Xi)
        assert abs(loss[i].item() - li.item()) < 1e-6 * 6
        assert rel_err(gx[i], gi.cpu().numpy()) < GRAD


def test_a_batch_of_one_and_a_single_problem_keep_graphs_of_their_own():
    from flash_sinkhorn_amd import SamplesLoss
    x, y, _, _ = inputs(8, 61, 50, 4)
    X, Y = dev(x, y)
    fn = SamplesLoss("sinkhorn", use_epsilon_scaling=False, eps=0.1, n_iters=10)
    for _ in range(3):  # (eager, captured, replayed)
        one, batch = fn(X, Y), fn(X[None], Y[None])
        assert one.shape == () and batch.shape == (1,) and one.item() == batch.item()


def test_batches_beyond_the_workspace_bound_go_item_by_item(monkeypatch):
    from flash_sinkhorn_amd import SamplesLoss, _small
    X = torch.randn(4, 70, 3, device="cuda").requires_grad_()
    Y = torch.rand(4, 60, 3, device="cuda")
    for kw in (dict(debias=True), dict(use_epsilon_scaling=False, eps=0.1, n_iters=9)):
        fn, pots = SamplesLoss(**kw), SamplesLoss(potentials=True, **kw)
        monkeypatch.setattr(_small, "MAX_BATCH_BYTES", 16 << 30)
        want, (wf, wg) = fn(X, Y), pots(X, Y)
        wx, = torch.autograd.grad(want.sum(), X)
        monkeypatch.setattr(_small, "MAX_BATCH_BYTES", 1000)
        got, (f, g) = fn(X, Y), pots(X, Y)
        gx, = torch.autograd.grad(got.sum(), X)
        # (two paths: 1e-5 of the costs, as above)
        assert (got - want).abs().max() < 1e-4 and rel_err(gx, wx.cpu().numpy()) < 10 * GRAD
        assert rel_err(f, wf.cpu().numpy()) < 2 * POT and rel_err(g, wg.cpu().numpy()) < 2 * POT


# (a schedule's table has the entries the schedule can have, and one more)
@pytest.mark.parametrize("blur,scaling,cut", [(0.05, 0.9, None), (0.05, 0.9, 1), (0.05, 0.9, 40), (3.0, 0.5, None),
                                              (10.0, 0.5, None), (1e-4, 0.97, None)])
@pytest.mark.parametrize("threshold", [None, 1e-2])
def test_tables_of_long_and_short_schedules(blur, scaling, cut, threshold):
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(6, 70, 90, 5, scale=0.5)
    kw = dict(blur=blur, scaling=scaling, n_iters=cut, threshold=threshold, check_every=3,
              return_n_iters=True)
    f, g, used = solve(*dev(x, y, a, b), **kw)
    wf, wg, wused = oracle.sinkhorn_symmetric(x, y, a, b, **kw)
    assert used == wused
    assert rel_err(f, wf) < 2 * POT and rel_err(g, wg) < 2 * POT


def test_graphs_of_batches_are_bounded_by_all_their_items(monkeypatch):
    from collections import OrderedDict
    from flash_sinkhorn_amd import SamplesLoss, _graphs
    monkeypatch.setattr(_graphs, "_cache", OrderedDict())
    fn = SamplesLoss("sinkhorn", use_epsilon_scaling=False, eps=0.1, n_iters=8)
    # one item has few logits; the batch has as many as a large problem, or as large a workspace
    for items, n, kept in ((3, 300, 1), (400, 300, 0), (8192, 16, 0)):
        _graphs.clear()
        x = torch.randn(items, n, 3, device="cuda").requires_grad_()
        want = None
        for _ in range(3):
            loss = fn(x, x.detach().flip(0))
            grad, = torch.autograd.grad(loss.sum(), x)
            assert want is None or torch.equal(grad, want)
            want = grad
        assert len(_graphs._cache) == kept


# every thread has a stream, clouds and graphs of its own; captures meet other threads' allocations and waits
def test_threads_on_streams_of_their_own():
    import threading
    from flash_sinkhorn_amd import SamplesLoss, _graphs

    def passes(x, y):
        out = []
        for kw in (dict(debias=True), dict(use_epsilon_scaling=False, eps=0.1, n_iters=20),
                   dict(use_epsilon_scaling=False, eps=0.3, n_iters=50, threshold=1e-3)):
            u = x.clone().requires_grad_()
            loss = SamplesLoss(**kw)(u, y)
            out += [loss.detach(), torch.autograd.grad(loss, u)[0]]
        return out

    clouds = [dev(*(a[0] for a in (inputs(k, 100 + 37 * k, 120, 5)[:1], inputs(k + 9, 90 + k, 120, 5)[:1])))
              for k in range(4)]
    want = [passes(x, y) for x, y in clouds]  # (eager: the first call with a shape)
    torch.cuda.synchronize()
    found, start = [], threading.Barrier(4)

    def run(k):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                start.wait(30)
                for _ in range(6):  # (eager, captured, replayed)
                    got = passes(*clouds[k])
                    stream.synchronize()
                    found.extend((k, i) for i, (u, v) in enumerate(zip(got, want[k])) if not torch.equal(u, v))
        except Exception as e:
            found.append((k, repr(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not found
    _graphs.clear()


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("fixed", [False, True])
def test_the_loss_may_be_changed_in_place(batched, fixed):
    from flash_sinkhorn_amd import SamplesLoss
    x, y, _, _ = inputs(8, 64, 50, 4)
    X, Y = dev(x, y) if not batched else dev(x[None], y[None])
    X.requires_grad_()
    fn = SamplesLoss("sinkhorn", **(dict(use_epsilon_scaling=False, eps=0.1, n_iters=10) if fixed else {}))
    for _ in range(3):  # (eager, captured, replayed)
        want, = torch.autograd.grad(fn(X, Y).sum(), X)
        loss = fn(X, Y)
        loss += 1.0
        loss *= 2.0
        got, = torch.autograd.grad(loss.sum(), X)
        assert torch.equal(got, 2.0 * want)


@pytest.mark.parametrize("d", [4, 200])
def test_potentials_are_tensors_of_their_own(d):
    from flash_sinkhorn_amd import SamplesLoss, sinkhorn_solvers as S
    x, y, a, b = inputs(8, 64, 50, d, scale=1.0 / np.sqrt(d))
    X, Y, A, B = dev(x, y, a, b)
    fixed = dict(use_epsilon_scaling=False, eps=0.1, n_iters=10)
    runs = [lambda: S.sinkhorn_flashstyle_symmetric(X, Y, A, B, return_prelast=True, **fixed),
            lambda: S.sinkhorn_flashstyle_symmetric(X, Y, A, B, threshold=1e-3, **fixed),
            lambda: S.sinkhorn_flashstyle_alternating(X, Y, A, B, eps=0.1, n_iters=10),
            lambda: [p[0] for p in S.sinkhorn_flashstyle_symmetric_self_pair(X, A, Y, B, **fixed)],
            lambda: SamplesLoss(potentials=True)(X, Y) if d < 129 else SamplesLoss(potentials=True, **fixed)(X, Y),
            lambda: SamplesLoss(potentials=True, **fixed)(X[None].expand(3, -1, -1), Y[None].expand(3, -1, -1))]
    for run in runs:
        for _ in range(3):  # (eager, captured, replayed)
            out = run()
            assert len({t.untyped_storage().data_ptr() for t in out}) == len(out)
            assert all(t.untyped_storage().nbytes() == 4 * t.numel() for t in out)
            w = torch.ones_like(out[1], requires_grad=True)
            total = (out[1] * w).sum()
            out[0].add_(1.0)
            total.backward()  # (out[1] has not been modified)


def test_saved_tensors_pass_through_hooks_and_version_checks():
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(8, 90, 50, 4)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_()
    fn = SamplesLoss("sinkhorn", normalize=False)
    want, = torch.autograd.grad(fn(A, X, B, Y), X)
    with torch.autograd.graph.save_on_cpu():
        loss = fn(A, X, B, Y)
    got, = torch.autograd.grad(loss, X, create_graph=True)
    assert torch.equal(got, want)
    assert torch.isfinite(torch.autograd.grad((got * Y[:1]).sum(), X)[0]).all()
    for t in (A, Y):  # changed between the passes: refused
        loss = fn(A, X, B, Y)
        with torch.no_grad():
            t.mul_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()


# The native autograd node against the Function that it stands for, to the bit; what only a Function serves or
# refuses still reaches one.
@pytest.mark.parametrize("form", ["x", "y", "both", "weights", "batch", "float16", "strided", "replayed", "scaled", "hooks"])
@pytest.mark.parametrize("debias", [False, True])
def test_native_node_equals_the_function(monkeypatch, form, debias):
    from flash_sinkhorn_amd import SamplesLoss, _small
    from types import SimpleNamespace
    x, y, a, b = inputs(21, 130, 97, 20, scale=0.5, y_shift=0.2)
    X, Y, A, B = dev(x, y, a, b)
    if form == "batch":
        X, Y, A, B = (torch.stack([t, t.flip(0)]) for t in (X, Y, A, B))
    if form == "float16":
        X, Y = X.half(), Y.half()
    if form == "strided":
        X = X.t().contiguous().t()
    kw = dict(use_epsilon_scaling=False, eps=0.1, n_iters=12) if form == "replayed" else dict(blur=0.2)
    fn = SamplesLoss("sinkhorn", debias=debias, **kw)
    wanted = {"x": [X], "y": [Y], "weights": [A, X, B, Y]}.get(form, [X, Y])
    for t in wanted:
        t.requires_grad_()
    native, grad = _small._native()
    out = []
    for ordinary in (True, False):
        with monkeypatch.context() as m:
            m.setattr(_small, "_NATIVE", (SimpleNamespace(ordinary=lambda _: ordinary, attach=native.attach), grad))
            for _ in range(3):
                if form == "hooks":
                    with torch.autograd.graph.save_on_cpu():
                        loss = fn(A, X, B, Y)
                else:
                    loss = fn(A, X, B, Y)
                seed = torch.full_like(loss, 3.0) if form == "scaled" else torch.ones_like(loss)
                grads = torch.autograd.grad(loss, wanted, seed, retain_graph=True)
                again = torch.autograd.grad(loss, wanted, seed)
            assert all(torch.equal(u, v) for u, v in zip(grads, again))
            with pytest.raises(RuntimeError, match="second time"):
                torch.autograd.grad(loss, wanted, seed)
            out.append((loss.detach(), *grads))
    assert all(u.dtype is v.dtype and torch.equal(u, v) for u, v in zip(*out))
    if form == "x" and not debias:
        with torch.no_grad():
            assert not fn(A, X, B, Y).requires_grad
        gx, = torch.autograd.grad(fn(A, X, B, Y), X, create_graph=True)
        assert torch.equal(gx.detach(), out[0][1])
        with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
            fn(torch.autograd.forward_ad.make_dual(X.detach(), torch.ones_like(X)), Y)
        with pytest.raises(RuntimeError, match="functorch"):
            torch.func.grad(lambda t: fn(t, Y))(X.detach())


# ---- gradients along lists read nothing but the workspace that the autograd node holds: behind other
# losses of the same replayed graph, behind a graph that is forgotten, at another address ----
@pytest.mark.parametrize("n,m,d,eps,debias", [(4513, 4490, 64, 0.01, False), (3300, 3290, 20, 0.02, True)])
@pytest.mark.parametrize("between", ["nothing", "graphs forgotten", "saved on the host"])
def test_gradients_along_lists_after_their_workspace_was_copied(monkeypatch, n, m, d, eps, debias, between):
    from flash_sinkhorn_amd import SamplesLoss, _graphs
    fn = SamplesLoss("sinkhorn", normalize=False, use_epsilon_scaling=False, eps=eps, n_iters=25, debias=debias)
    sets = [dev(*inputs(seed, n, m, d, scale=0.5, y_shift=0.2)) for seed in range(4)]
    for k, (x, y, _, _) in enumerate(sets):
        if debias:  # (partners at another distance in every set: other lists of a cloud with itself)
            x[n // 2:] = x[:n // 2].roll(300 * k, 0) + 0.02 * x[n // 2:]
        else:
            x[1::2] = x[:-1:2] + 0.02 * x[1::2]
        x.requires_grad_(), y.requires_grad_()
    with monkeypatch.context() as off:
        off.setattr(_graphs, "ENABLED", False)
        want = [torch.autograd.grad(fn(a, x, b, y), [x, y]) for x, y, a, b in sets]
    _graphs.clear()
    if between == "saved on the host":
        with torch.autograd.graph.save_on_cpu():
            losses = [fn(a, x, b, y) for x, y, a, b in sets]
    else:
        losses = [fn(a, x, b, y) for x, y, a, b in sets]  # (launch by launch, captured, replayed twice)
    if between != "nothing":
        _graphs.clear()
        torch.cuda.empty_cache()
    for i in (3, 2, 1, 0):
        got = torch.autograd.grad(losses[i], sets[i][:2])
        assert all(torch.equal(g, w) for g, w in zip(got, want[i]))


# ---- gradients and Hessian-vector products on the products that a solve of wide rows keeps (from 2^22
# of them on): odd sizes, columns that fill no step, one cloud far larger, half precision, relaxed ----
@pytest.mark.parametrize("n,m,d,dtype,rho,stop", [(2051, 2100, 129, torch.float32, None, None),
                                                  (600, 8001, 200, torch.float32, 1.5, None),
                                                  (8200, 515, 300, torch.float16, None, 0.02),
                                                  (2305, 1830, 1000, torch.bfloat16, None, None),
                                                  (2049, 2048, 130, torch.float32, 2.0, "scaling")])
def test_gradients_on_kept_products(n, m, d, dtype, rho, stop):
    from flash_sinkhorn_amd import SamplesLoss
    from flash_sinkhorn_amd.hvp import geomloss_to_ott_potentials, hvp_x_sqeuclid_from_potentials
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(n, n, m, d, scale=1.0 / np.sqrt(d), y_shift=0.3 / np.sqrt(d))
    X, Y, A, B = dev(x, y, a, b)
    X, Y = X.to(dtype).requires_grad_(), Y.to(dtype).requires_grad_()
    x, y = (t.detach().float().cpu().numpy() for t in (X, Y))
    eps = 0.1
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=4)
    if stop == "scaling":  # (a list of eps)
        kw = dict(blur=eps ** 0.5, scaling=0.5)
    elif stop:
        kw.update(n_iters=60, threshold=stop)
    fn = SamplesLoss("sinkhorn", normalize=False, reach_x=rho, reach_y=rho, **kw)
    gx, gy = torch.autograd.grad(2.0 * fn(A, X, B, Y), [X, Y])
    relaxed = dict(reach_x=rho, reach_y=rho)
    _, _, fp, gp = solve(X.detach(), Y.detach(), A, B, return_prelast=True, **relaxed, **kw)
    wx, wy = oracle.grad_barycentric(x, y, a, b, fp.cpu().numpy(), gp.cpu().numpy(), eps)
    # (a gradient comes back in the type of the points)
    tol = GRAD + (0.0 if dtype is torch.float32 else 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11)
    assert rel_err(gx.float(), 2.0 * wx) < tol and rel_err(gy.float(), 2.0 * wy) < tol
    if dtype is torch.float32:
        (gx,) = torch.autograd.grad(2.0 * fn(A, X, B, Y.detach()), X, create_graph=True)
        v = torch.randn(n, d, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
        (got,) = torch.autograd.grad((gx * v).sum(), X)
        ott = geomloss_to_ott_potentials(fp, gp, A, B, eps=eps)
        want, _ = hvp_x_sqeuclid_from_potentials(X.detach(), Y.detach(), *ott, v, eps=eps,
                                                 rho_x=rho and rho ** 2, rho_y=rho and rho ** 2)
        # (the same sums of the same products, formed once instead of twice)
        assert torch.equal(got, 2.0 * want)


# Features as they come (|x|^2 of 3.2e7) with a small reach: potentials are the norms and a little more, and
# say next to nothing of a row's sum.  The bound is that of logits, gradient_bound.
def test_gradients_on_kept_products_at_a_small_reach():
    from flash_sinkhorn_amd import SamplesLoss
    from flash_sinkhorn_amd.kernels import sinkhorn_flashstyle_symmetric as solve
    x, y, a, b = inputs(5, 2051, 2100, 200, scale=400.0, y_shift=100.0)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_()
    eps = 4e4
    kw = dict(use_epsilon_scaling=False, eps=eps, n_iters=4)
    gx, = torch.autograd.grad(SamplesLoss("sinkhorn", normalize=False, reach=0.4, **kw)(A, X, B, Y), X)
    _, _, fp, gp = solve(X.detach(), Y, A, B, return_prelast=True, rho_x=0.16, rho_y=0.16, **kw)
    want, _ = oracle.grad_barycentric(x, y, a, b, fp.cpu().numpy(), gp.cpu().numpy(), eps)
    off = np.abs(gx.cpu().numpy() - want).max(axis=1)
    assert (off <= 2.0 * a * gradient_bound(x, y, eps)).all()


# (the workspace comes back at another address; gradient and Hessian-vector product read nothing else)
def test_kept_products_pass_through_hooks():
    from flash_sinkhorn_amd import SamplesLoss
    x, y, a, b = inputs(9, 2051, 2100, 140, scale=0.1)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_()
    fn = SamplesLoss("sinkhorn", normalize=False, use_epsilon_scaling=False, eps=0.1, n_iters=4)

    def pass_through(loss):
        g, = torch.autograd.grad(loss, X, create_graph=True)
        return g, torch.autograd.grad((g * Y[:1]).sum(), X)[0]
    want = pass_through(fn(A, X, B, Y))
    with torch.autograd.graph.save_on_cpu():
        loss = fn(A, X, B, Y)
        assert all(torch.equal(g, w) for g, w in zip(pass_through(loss), want))


# Products are held only while half of the card stays free, and not at all where that is asked for: the
# gradient then forms them again.
@pytest.mark.parametrize("kept", ["as a rule", "declined", "card half full", "allocator idle"])
def test_products_are_kept_where_there_is_room(monkeypatch, kept):
    from flash_sinkhorn_amd import SamplesLoss, _small
    x, y, a, b = inputs(6, 2600, 2500, 140, scale=0.1)
    X, Y, A, B = dev(x, y, a, b)
    X.requires_grad_()
    fn = SamplesLoss("sinkhorn", normalize=False, use_epsilon_scaling=False, eps=0.1, n_iters=4)
    want, = torch.autograd.grad(fn(A, X, B, Y), X)
    if kept == "declined":
        monkeypatch.setattr(_small, "KEEP_PRODUCTS", False)
    elif kept != "as a rule":
        total = 100 << 30
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: ((50 << 30) + (1 << 20), total))
        idle = (1 << 30) if kept == "allocator idle" else 0
        monkeypatch.setattr(torch.cuda, "memory_reserved", lambda device: torch.cuda.memory_allocated(device) + idle)
    before = torch.cuda.memory_allocated()
    loss = fn(A, X, B, Y)
    held = torch.cuda.memory_allocated() - before
    assert (held >= 4 * 2600 * 2500) == (kept in ("as a rule", "allocator idle"))
    got, = torch.autograd.grad(loss, X)
    assert rel_err(got, want.cpu().numpy()) < GRAD


# ---- Hessian-vector products: whole rows in registers (2,048, 4,096, 8,192 columns) ----
@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (37, 2048, 64), (300, 2049, 5), (65, 4097, 130), (257, 200, 129),
                                   (40, 8192, 20)])
@pytest.mark.parametrize("rho", [None, 1.5])
def test_kept_hvp(n, m, d, rho):
    from flash_sinkhorn_amd.hvp import hvp_x_sqeuclid_from_potentials as hvp
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    eps = 0.25
    f, g = oracle.sinkhorn_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=eps, n_iters=20, rho_x=rho)
    f, g = oracle.geomloss_to_ott_potentials(f, g, a, b, eps)
    A = np.random.default_rng(1).standard_normal((n, d)).astype(np.float32)
    f, g = f.astype(np.float32), g.astype(np.float32)
    for iters in (0, 1, 200):
        kw = dict(eps=eps, rho_x=rho, max_cg_iter=iters, cg_rtol=1e-5, cg_atol=1e-12,
                  preconditioner="none")
        got, info = hvp(*dev(x, y, f, g, A), **kw)
        want, winfo = oracle.hvp_x_from_potentials(x, y, f, g, A, **kw)
        # conjugate gradients to 1e-5 of a right-hand side whose Schur complement is no smaller than
        # the gap of the plan (above 1e-1 at this eps): 1e-4 of the result
        assert rel_err(got, want) < 2e-4
        assert info.cg_iters <= iters and np.isfinite(info.cg_residual)
        if iters == 200:
            # (one point: the right-hand side is zero, and nothing is iterated)
            assert info.cg_converged or info.cg_initial_residual == 0.0
            assert info.cg_residual <= max(1e-5 * info.cg_initial_residual, 1e-12)
        elif not info.cg_converged and info.cg_initial_residual > 0.0:
            assert info.cg_iters == iters


# Potentials that leave the weights to the plan (uniform ones need no tensor; a point without mass), and a scaled result:
# the same numbers, formed by the kernel that reads the potentials and by the last one.
@pytest.mark.parametrize("n,m,d", [(1, 1, 1), (130, 257, 5), (65, 2049, 129), (2047, 300, 64)])
@pytest.mark.parametrize("uniform", [(False, False), (True, False), (False, True), (True, True)])
def test_kept_hvp_of_weighted_plans(n, m, d, uniform):
    from flash_sinkhorn_amd.hvp import geomloss_to_ott_potentials, hvp_x_sqeuclid_from_potentials as hvp
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    a, b = (np.full_like(w, 1.0 / len(w)) if u else w for w, u in zip((a, b), uniform))
    if n > 100 and not uniform[0]:
        a[3] = 0.0
    f, g = oracle.sinkhorn_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.25, n_iters=5)
    X, Y, A, B, F, G = dev(x, y, a, b, f.astype(np.float32), g.astype(np.float32))
    V = dev(np.random.default_rng(1).standard_normal((n, d)).astype(np.float32))[0]
    kw = dict(eps=0.25, cg_rtol=1e-5, cg_atol=1e-12, preconditioner="none")
    scale = torch.tensor(-1.7, device="cuda")
    want, _ = hvp(X, Y, *geomloss_to_ott_potentials(F, G, A, B, eps=0.25), V, **kw)
    got, _ = hvp(X, Y, F, G, V, _weights=tuple(None if u else w for u, w in zip(uniform, (A, B))), _scale=scale, **kw)
    if not any(uniform):
        assert torch.equal(got, want * scale)
    # (the logarithm of a uniform weight is the host's, 1e-7 of its 8 or less, and so 1e-7 of any entry of the plan: as far as
    # conjugate gradients to 1e-5 take that)
    assert rel_err(got, (want * scale).cpu().numpy()) < 2e-4


@pytest.mark.parametrize("n,m,d", [(37, 300, 64), (65, 130, 5), (100, 257, 136)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_kept_hvp_of_half_precision_points(n, m, d, dtype):
    from flash_sinkhorn_amd.hvp import hvp_x_sqeuclid_from_potentials as hvp
    x, y, a, b = inputs(n + d, n, m, d, scale=1.0 / np.sqrt(d))
    X, Y = (t.to(dtype) for t in dev(x, y))
    x, y = (t.float().cpu().numpy() for t in (X, Y))
    f, g = oracle.sinkhorn_symmetric(x, y, a, b, use_epsilon_scaling=False, eps=0.25, n_iters=20)
    f, g = (t.astype(np.float32) for t in oracle.geomloss_to_ott_potentials(f, g, a, b, 0.25))
    A = np.random.default_rng(1).standard_normal((n, d)).astype(np.float32)
    kw = dict(eps=0.25, cg_rtol=1e-5, cg_atol=1e-12, preconditioner="none")
    got, _ = hvp(X, Y, *dev(f, g, A), **kw)
    want, _ = oracle.hvp_x_from_potentials(x, y, f, g, A, **kw)
    assert rel_err(got, want) < 2e-4  # (as above: the points are exact in two fp16 planes)


def test_hvp_refuses_operands_elsewhere_and_of_other_lengths():
    from flash_sinkhorn_amd.hvp import (hvp_x_sqeuclid_from_potentials as hvp,
                                        inverse_hvp_x_sqeuclid_from_potentials as inverse)
    x, y, _, _ = inputs(3, 40, 30, 4)
    X, Y, F, G, A = dev(x, y, *(np.zeros(k, np.float32) for k in (40, 30)), x)
    for args in ((X, Y, F, G, A.cpu()), (X, Y, G, F, A), (X, Y, F[:7], G, A), (X, Y, F, G[:7], A)):
        for fn in (hvp, inverse):
            with pytest.raises((RuntimeError, ValueError, AssertionError)):
                fn(*args, eps=0.3)


# ---- the merge of the key splits: four wavefronts share them, two, four or eight at a time ----
@pytest.mark.parametrize("n,m", [(1, 40000), (63, 9000), (257, 20000), (1000, 3000), (5000, 5100), (20000, 700)])
def test_merge_of_key_splits(n, m):
    from flash_sinkhorn_amd.kernels import apply_plan_vec_flashstyle as apply
    rng = np.random.default_rng(n)
    x, y, a, b = inputs(n, n, m, 12, scale=0.3)
    f, g = (0.1 * rng.standard_normal(k).astype(np.float32) for k in (n, m))
    la, lb = np.log(a), np.log(b)
    for axis, k in ((1, m), (0, n)):
        v = rng.random(k).astype(np.float32)
        got = apply(*dev(x, y, f, g, la, lb, v), eps=0.2, axis=axis)
        want = oracle.apply_plan_vec(x, y, f, g, la, lb, v, 0.2, axis)
        # (positive terms: the error of a logit, 2^-21 of the largest cost over eps, is the whole error)
        assert rel_err(got, want) < GRAD
