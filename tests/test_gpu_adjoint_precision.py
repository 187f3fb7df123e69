"""Rounding errors of the reverse pass, with the pieces side by side and turn
by turn, against the same linear maps in 80-bit arithmetic on the same states
(the exact build's forward pass, which NumPy repeats operation by operation on
a lattice of drifts and multipoles).  Pieces side by side reach their end
cotangents through products with their Jacobians; without the correction that
follows, element by element, the coordinates' gradients are twice as far off
as turn by turn."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from sixtracklib_amd import beam_elements as be, lattices  # noqa: E402
from sixtracklib_amd.cobject import get_object  # noqa: E402
from sixtracklib_amd.cobjects import CBuffer  # noqa: E402
from test_gpu_adjoint_plan import _turn_by_turn  # noqa: E402

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _lattice(seed):
    """996 elements, the sub-lattice of the gradient benchmark without its
    cavity, and its elements as (length,) or coefficients."""
    src = lattices.adjoint_sublattice(seed=seed)
    eb = CBuffer(max_slots=32000, max_objects=1100, max_pointers=1100)
    for i in range(src.n_objects):
        o = get_object(src, i)
        if src.get_object_typeid(i) == 2:
            be.Drift(cbuffer=eb, length=float(o.length))
        elif src.get_object_typeid(i) == 4:
            bal = np.array(o.bal)
            fact = np.array([math.factorial(k) for k in range(len(bal) // 2)], dtype=float)
            be.Multipole(cbuffer=eb, knl=bal[0::2] * fact, ksl=bal[1::2] * fact)
    elements = []
    for i in range(eb.n_objects):
        o = get_object(eb, i)
        elements.append(float(o.length) if eb.get_object_typeid(i) == 2 else np.array(o.bal))
    return eb, elements


def _states(elements, coords, turns, beta0):
    """(per turn and element the two coordinates its map's Jacobian needs, per
    turn the end state), rpp, rvv"""
    x, px, y, py, _, delta = (coords[:, k].copy() for k in range(6))
    db = delta * beta0
    rvv = (1.0 + delta) / np.sqrt(db * db + 2.0 * db * beta0 + 1.0)
    rpp = 1.0 / (1.0 + delta)
    states, ends = [], []
    for _ in range(turns):
        for el in elements:
            if isinstance(el, float):
                states.append((px, py))
                x, y = x + (px * rpp) * el, y + (py * rpp) * el
            else:
                states.append((x, y))
                re, im = np.full_like(x, el[-2]), np.full_like(x, el[-1])
                for k in range(len(el) - 4, -1, -2):
                    re, im = el[k] + (re * x - im * y), el[k + 1] + (re * y + im * x)
                px, py = px - re, py + im
        ends.append((x, px, y, py))
    return states, ends, rpp, rvv


def _reverse(elements, states, ends, rpp, delta, beta0, target, n_mp, width):
    c = [np.zeros(len(rpp), LD) for _ in range(6)]
    gk, gs = np.zeros((n_mp, width), LD), np.zeros((n_mp, width), LD)
    b2, rpp, delta = LD(beta0) * LD(beta0), rpp.astype(LD), delta.astype(LD)
    root = np.sqrt(b2 * (delta * delta + 2 * delta) + 1)
    drvv, drpp = (1 - b2) / root ** 3, -rpp * rpp
    at = len(states)
    for t in range(len(ends) - 1, -1, -1):
        for q in range(4):
            c[q] = c[q] + 2 * (ends[t][q].astype(LD) - LD(target[t, q]))
        m = n_mp
        for el in reversed(elements):
            at -= 1
            u, v = (s.astype(LD) for s in states[at])
            if isinstance(el, float):
                xp, yp = u * rpp, v * rpp
                c[5] = c[5] + LD(el) * (c[0] * u * drpp + c[2] * v * drpp +
                                        c[4] * (drvv - (xp * u + yp * v) * drpp))
                c[1] = c[1] + LD(el) * rpp * (c[0] - c[4] * xp)
                c[3] = c[3] + LD(el) * rpp * (c[2] - c[4] * yp)
                continue
            m -= 1
            order = len(el) // 2 - 1
            wr, wi = np.ones_like(u), np.zeros_like(u)
            for k in range(order + 1):
                gk[m, k] += (-c[1] * wr + c[3] * wi).sum() / LD(math.factorial(k))
                gs[m, k] += (c[1] * wi + c[3] * wr).sum() / LD(math.factorial(k))
                wr, wi = wr * u - wi * v, wr * v + wi * u
            dre, dim = np.zeros_like(u), np.zeros_like(u)
            for k in range(order, 0, -1):
                dre, dim = (dre * u - dim * v + k * LD(el[2 * k]), dre * v + dim * u + k * LD(el[2 * k + 1]))
            c[0] = c[0] - c[1] * dre + c[3] * dim
            c[2] = c[2] + c[1] * dim + c[3] * dre
    return np.stack(c, 1), gk, gs


def test_the_reverse_pass_rounds_no_more_than_turn_by_turn():
    from sixtracklib_amd.adjoint import AdjointTracker
    n, turns = 96, 4
    _, species = lattices.make_particles(1)
    beta0 = float(np.array(species.beta0)[0])
    off = {"side by side": [], "turn by turn": []}
    for seed in range(4):
        eb, elements = _lattice(seed)
        tr = AdjointTracker(eb, turns, species=species)
        rng = np.random.default_rng(seed)
        coords = rng.normal(size=(n, 6)) * np.array([3e-4, 3e-6, 3e-4, 3e-6, 0.05, 1e-4])
        target = rng.normal(size=(turns, 4)) * np.array([3e-5, 3e-7, 3e-5, 3e-7])
        X = torch.tensor(coords, device="cuda", requires_grad=True)
        tgt = tr.target_tensor(target)
        knl, ksl = tr.knl0.clone().requires_grad_(), tr.ksl0.clone().requires_grad_()
        loss = tr.loss(X, knl, ksl, target)
        got = torch.autograd.grad(loss, [X, knl, ksl])
        one = _turn_by_turn(tr, X.detach(), tr.knl0, tr.ksl0, tgt)[1:]
        assert tr.n_mp == sum(not isinstance(el, float) for el in elements)
        states, ends, rpp, rvv = _states(elements, coords, turns, beta0)
        want = _reverse(elements, states, ends, rpp, coords[:, 5], beta0, target, tr.n_mp, tr.max_order + 1)
        for name, grads in (("side by side", got), ("turn by turn", one)):
            off[name].append([float(np.linalg.norm((g.cpu().numpy() - w).astype(float)) /
                                    np.linalg.norm(w.astype(float))) for g, w in zip(grads, want)])
    rms = {k: np.sqrt((np.array(v) ** 2).mean(0)) for k, v in off.items()}
    print(rms)
    assert np.all(rms["turn by turn"] < 2e-14)         # the states are the kernels'
    # four lattices of 96 particles: the coordinates' ratio scatters by some
    # 10 %, those of the strengths, sums over the particles, by 30 %
    assert rms["side by side"][0] <= 1.3 * rms["turn by turn"][0]
    assert np.all(rms["side by side"][1:] <= 1.7 * rms["turn by turn"][1:])
