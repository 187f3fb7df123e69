"""Gradients over the checkpoint interval K: ranges that hold one piece of 64
elements, several, parts of pieces or the whole lattice, with the pieces side
by side and one after another; and their cost, which K must not multiply."""
import time

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from sixtracklib_amd import lattices  # noqa: E402
from test_gpu_adjoint_plan import _compare, _lattice  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [63, 65, 100, 127, 128, 129, 192, 399, 400, 401, 10**5])
@pytest.mark.parametrize("n_elem", [65, 129, 400])
def test_gradients_over_K(n_elem, K):
    eb = _lattice(n_elem, n_elem)
    for n, turns, fma in ((65, 2, False), (128, 1, True)):
        _compare(eb, n, turns, K, fma, default=False)


@pytest.mark.parametrize("K", [65, 100, 200, 1000])
def test_gradients_over_K_one_wave_through_all_pieces(K):
    _compare(_lattice(200, 5), 65601, 2, K, False, default=False)


def test_gradients_in_groups_that_do_not_divide_the_turns():
    """2,000 elements, 65,536 particles: a group of turns is two."""
    _compare(lattices.adjoint_sublattice(n_cells=40, tune=8.62), 65536, 3, 64, False, default=False)


def _backward_seconds(eb, n, turns, K):
    from sixtracklib_amd.adjoint import AdjointTracker
    rng = np.random.default_rng(1)
    _, species = lattices.make_particles(1)
    tr = AdjointTracker(eb, turns, species=species, K=K)
    scale = np.array([3e-4, 3e-6, 3e-4, 3e-6, 0.05, 1e-4])
    X = torch.tensor(rng.normal(size=(n, 6)) * scale, device="cuda", requires_grad=True)
    best = float("inf")
    for _ in range(5):
        loss = tr.loss(X)
        torch.cuda.synchronize()
        t = time.perf_counter()
        torch.autograd.grad(loss, [X])
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("n, turns", [(4096, 4), (70000, 1)])
def test_the_backward_pass_is_linear_in_K(n, turns):
    """4,000 elements and one checkpoint a turn: the range is gone through once
    more than with K = 64 (measured 1.6 and 1.2 times the time; 5.9 and 6.6
    when each of the 63 pieces went through what lies before it)."""
    eb = lattices.adjoint_sublattice(n_cells=80, tune=17.24)
    assert _backward_seconds(eb, n, turns, 4000) < 3.0 * _backward_seconds(eb, n, turns, 64)


@pytest.mark.parametrize("K", [64, 300])
def test_gradients_where_the_device_is_short_of_memory(K, monkeypatch):
    """Room for all turns at once, for a few and for none (the allocations
    that find no room are refused here)."""
    from sixtracklib_amd.adjoint import AdjointTracker
    n, turns = 4096, 10
    rng = np.random.default_rng(1)
    _, species = lattices.make_particles(1)
    tr = AdjointTracker(lattices.adjoint_sublattice(), turns, species=species, K=K)
    scale = np.array([3e-4, 3e-6, 3e-4, 3e-6, 0.05, 1e-4])
    X = torch.tensor(rng.normal(size=(n, 6)) * scale, device="cuda", requires_grad=True)
    knl, ksl = tr.knl0.clone().requires_grad_(), tr.ksl0.clone().requires_grad_()
    empty, made = torch.empty, []

    def within(room):
        def f(*size, **kw):
            if len(size) == 1 and isinstance(size[0], int):
                if 8 * size[0] > room:
                    raise torch.OutOfMemoryError("no room for %d bytes" % (8 * size[0]))
                made.append(8 * size[0])
            return empty(*size, **kw)
        return f

    grads, most = [], []
    for room in (1e12, 2.5e8, 2e7):
        loss = tr.loss(X, knl, ksl)
        del made[:]
        monkeypatch.setattr(torch, "empty", within(room))
        grads.append(torch.autograd.grad(loss, [X, knl, ksl]))
        monkeypatch.undo()
        most.append(max(made))
    assert most[0] > 2.5e8 >= most[1] > 2e7 >= most[2]
    for some in grads[1:]:
        for a, b in zip(some, grads[0]):
            assert float((a - b).norm()) <= 2e-12 * float(b.norm())
    loss = tr.loss(X, knl, ksl)
    monkeypatch.setattr(torch, "empty", within(1e5))
    with pytest.raises(torch.OutOfMemoryError):
        torch.autograd.grad(loss, [X, knl, ksl])
