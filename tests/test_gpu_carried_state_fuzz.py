"""Seeded random walks over the state that ``lse_coarse_kernel`` carries from launch to launch.

On prepared planes the kernel keeps, per row, the key of the row's largest logit, that logit,
the key biases of the last launch and, per 32-row block and 32-key sub-tile, a margin with a
generation tag; state words say which form of the kernel runs.  Whatever sequence of launches
touches that state, every launch must return what the plain kernel returns on the same inputs.
The walks below mix, in random order: Jacobi steps that let the potentials settle, small and
large disturbances of the potentials, changes of eps (each starts a new generation of margins:
the long walk passes the 255 generations an entry can name), the two clouds swapping roles,
key arrays overwritten with arbitrary numbers, and one-sided launches in either direction.
Every step is held to 2e-6 (max norm, relative to the largest potential) against the plain
launch, which the other tests hold to 1e-4 against the fp64 oracle; the walk stops at the first
step that fails and names it.

Rows of 65 to 128 columns carry lists of keys instead (``lse_coarse128_kernel``): the same walks, forced and with the
variant left to the device, and on one cloud against itself, whose two sides share their state.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _clouds(rng, n, m, d):
    centres = rng.standard_normal((6, d)) * 2.0
    x = (centres[rng.integers(0, 6, n)] + rng.standard_normal((n, d))).astype(np.float32)
    y = (centres[rng.integers(0, 6, m)] + rng.standard_normal((m, d))).astype(np.float32)
    return x, y


def _walk(seed, n, m, d, eps0, steps, p_eps, coarse=True, same=False):
    from flash_sinkhorn_amd import _lib
    from flash_sinkhorn_amd.kernels.sinkhorn_flashstyle_sqeuclid import (
        _symmetric_step_raw, flashsinkhorn_lse_fused)
    rng = np.random.default_rng(seed)
    x, y = _clouds(rng, n, m, d)
    X, Y = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    if same:
        Y, m = X, n
    b = (rng.random(m) + 0.5).astype(np.float32)
    LA = torch.full((n,), -float(np.log(n)), device="cuda")
    LB = torch.from_numpy(np.log(b / b.sum())).cuda()
    F, G = -(X * X).sum(1), -(Y * Y).sum(1)
    prep = _lib.PreparedOperands(X, Y, _lib.flags(True, False))
    kw = dict(cost_scale=1.0, alpha=0.5, damping_f=1.0, damping_g=1.0, allow_tf32=False)
    eps = eps0
    swapped = False
    by_lists = 0
    worst = 0.0
    counts = {}

    def noise(k, amp):
        return torch.from_numpy((amp * rng.standard_normal(k)).astype(np.float32)).cuda()

    for it in range(steps):
        u = rng.random()
        if u < p_eps:
            act = "eps"
            eps = eps0 * float(rng.choice([1.0, 1.5, 2.0, 0.75]))
        elif u < p_eps + 0.08:
            act = "small disturbance"  # a few base-2 units: margins are used up one by one
            amp = float(rng.uniform(1.0, 40.0)) * eps * np.log(2.0)
            F, G = F + noise(n, amp), G + noise(m, amp)
        elif u < p_eps + 0.12:
            act = "large disturbance"  # far past any margin
            F, G = F + noise(n, 10.0), G + noise(m, 10.0)
        elif u < p_eps + 0.17:
            act = "swap roles"
            swapped = not swapped
        elif u < p_eps + 0.21:
            act = "overwrite keys"
            prep.best_keys(0).copy_(torch.from_numpy(rng.integers(-5, m + 5, n).astype(np.int32)))
            if not same:
                prep.best_keys(1).copy_(torch.from_numpy(
                    rng.integers(-2**31, 2**31 - 1, m).astype(np.int32)))
        elif u < p_eps + 0.33:
            act = "one-sided f" if rng.random() < 0.5 else "one-sided g"
        else:
            act = "step"
        counts[act] = counts.get(act, 0) + 1
        if act.startswith("one-sided"):
            q, k, pot, lw = (X, Y, G, LB) if act.endswith("f") else (Y, X, F, LA)
            got = flashsinkhorn_lse_fused(q, k, pot, lw, eps, allow_tf32=False, _prepared=prep,
                                          _coarse=coarse)
            want = flashsinkhorn_lse_fused(q, k, pot, lw, eps, allow_tf32=False)
            err = float((got - want).abs().max() / want.abs().max())
            if act.endswith("f"):
                F = 0.5 * (F + got)
            else:
                G = 0.5 * (G + got)
        else:
            args = (Y, X, G, F, LB, LA) if swapped else (X, Y, F, G, LA, LB)
            o1, o2 = _symmetric_step_raw(*args, eps, coarse=coarse, prepared=prep, **kw)
            p1, p2 = _symmetric_step_raw(*args, eps, coarse=False, **kw)
            scale = max(float(p1.abs().max()), float(p2.abs().max()))
            err = max(float((o1 - p1).abs().max()), float((o2 - p2).abs().max())) / scale
            F, G = (o2, o1) if swapped else (o1, o2)
        worst = max(worst, err)
        by_lists += d > 64 and prep.variant_state()["by_lists"]
        assert err < 2e-6, (f"seed {seed}, shape {n} x {m} x {d}, step {it} ({act}, eps {eps:g}, "
                            f"roles swapped: {swapped}): differs from the plain launch by {err:.3e}")
    state = prep.variant_state()
    state["steps_by_lists"] = by_lists
    print(f"walk seed {seed} {n}x{m}x{d}: {steps} steps {counts}, largest difference to the plain "
          f"launch {worst:.2e}, units not visited {state['tiles_skipped']}, tested "
          f"{state['tiles_tested']}")
    return state


@pytest.mark.parametrize("seed,n,m,d,eps", [(1, 2600, 2200, 32, 0.02), (2, 1500, 3100, 64, 0.01),
                                            (3, 3000, 2900, 16, 0.05), (4, 700, 4200, 8, 0.05)])
def test_random_walks_over_the_carried_state(seed, n, m, d, eps):
    state = _walk(seed, n, m, d, eps, steps=160, p_eps=0.04)
    assert state["tiles_skipped"] > 0  # the sparse form ran, with margins that held


def test_random_walk_past_255_generations_of_margins():
    """An entry names its generation in 8 bits; after 255 generations on one set of planes the
    margins of that role must stay off rather than match a stale entry."""
    _walk(5, 1300, 1100, 32, 0.02, steps=640, p_eps=0.7)


@pytest.mark.parametrize("seed,n,d,eps", [(10, 2600, 48, 0.02), (11, 3100, 16, 0.05)])
def test_random_walks_over_the_margins_of_a_cloud_against_itself(seed, n, d, eps):
    """Two potentials on one matrix: the sides of a step have all they carry to themselves."""
    state = _walk(seed, n, n, d, eps, steps=120, p_eps=0.04, same=True)
    assert state["tiles_skipped"] > 0


@pytest.mark.parametrize("coarse", [True, "auto"])
@pytest.mark.parametrize("seed,n,m,d,eps,same", [
    (6, 2600, 5200, 96, 0.02, False), (7, 6100, 3100, 128, 0.01, False), (8, 1500, 6300, 70, 0.01, False),
    (9, 4100, 0, 100, 0.02, True)])
def test_random_walks_over_the_lists_of_rows_of_65_to_128_columns(seed, n, m, d, eps, same, coarse):
    state = _walk(seed, n, m or n, d, eps, steps=160, p_eps=0.05, coarse=coarse, same=same)
    # launches that went by lists, and lists that were there for a good part of the walk
    assert state["tiles_skipped"] > 0 and state["steps_by_lists"] > 40
