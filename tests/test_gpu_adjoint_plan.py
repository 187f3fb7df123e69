"""Gradients for all turns in few launches (NS(Adjoint_loss),
NS(Adjoint_gradients): pieces of 64 elements side by side up to 65,536
particles, in groups of turns, one wave through all pieces above) against the
turn-by-turn entry points (NS(Adjoint_forward), NS(Adjoint_backward_turn),
NS(Adjoint_reduce_coefficients)): lattices around the lengths of a piece and
of its parts with every map and order, checkpoint intervals that do and do
not divide them, particle counts around a wave."""
import ctypes as ct

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from sixtracklib_amd import lattices, beam_elements as be  # noqa: E402
from sixtracklib_amd.cobjects import CBuffer  # noqa: E402

pytestmark = pytest.mark.gpu

# Both sides apply the same Jacobians to cotangents in double precision and
# differ in the order of sums and products only: a relative error of at most
# about (elements x turns) x 2^-53 = 4e-13 of each gradient's norm at 4,000
# element passes, 2e-12 at 16,000.
REL = 2e-12


def _lattice(n_elem, seed):
    rng = np.random.default_rng(seed)
    eb = CBuffer(max_slots=64 * n_elem + 64, max_objects=n_elem + 8, max_pointers=n_elem + 8)
    for k in range(n_elem):
        kind = rng.choice(["d", "d", "m", "m", "dm", "cav", "rot", "shift", "rect", "ell"])
        if k == 0 and n_elem == 1:
            kind = "m"
        if kind in ("d", "dm"):
            be.Drift(cbuffer=eb, length=float(rng.uniform(0.1, 2.0)))
        elif kind == "m":
            order = int(rng.integers(0, 11))
            scale = 1e-6 * np.array([float(np.prod(np.arange(1, q + 1))) / 0.01 ** q
                                     for q in range(order + 1)])
            be.Multipole(cbuffer=eb, knl=rng.normal(size=order + 1) * scale,
                         ksl=rng.normal(size=order + 1) * scale)
        elif kind == "cav":
            be.Cavity(cbuffer=eb, voltage=2e6, frequency=400e6, lag=180.0)
        elif kind == "rot":
            be.SRotation(cbuffer=eb, angle=float(rng.normal(0, 2.0)))
        elif kind == "shift":
            be.XYShift(cbuffer=eb, dx=rng.normal(0, 1e-5), dy=rng.normal(0, 1e-5))
        elif kind == "rect":
            be.LimitRect(cbuffer=eb, min_x=-0.5, max_x=0.5, min_y=-0.5, max_y=0.5)
        else:
            be.LimitEllipse(cbuffer=eb, a=0.5, b=0.5)
    return eb


def _turn_by_turn(tr, coords, knl, ksl, tgt):
    """loss per particle and gradients of its sum, through the C entry points
    that take one turn at a time."""
    from sixtracklib_amd import adjoint as A
    n, dev = coords.shape[0], coords.device
    tr.write_coefficients(knl, ksl)
    X = coords.t().contiguous()
    ckpt = torch.empty(tr.checkpoint_size(n), dtype=torch.float64, device=dev)
    loss = torch.empty(n, dtype=torch.float64, device=dev)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    pr = tr.problem(n, tgt, ckpt)
    s = A._stream()
    assert A._lib.st_Adjoint_forward(ct.byref(pr), tr.fma, X.data_ptr(), loss.data_ptr(),
                                     status.data_ptr(), s) == 0
    assert int(status.item()) == 0
    seg = torch.empty(int(A._lib.st_Adjoint_segment_doubles(ct.byref(pr))), dtype=torch.float64, device=dev)
    coef = torch.empty(max(tr.n_mp * 4 * n, 1), dtype=torch.float64, device=dev)
    cot = torch.zeros(6, n, dtype=torch.float64, device=dev)
    gbal = torch.zeros(max(tr.n_mp, 1), 22, dtype=torch.float64, device=dev)
    g = torch.ones(1, dtype=torch.float64, device=dev)
    for turn in range(tr.n_turns - 1, -1, -1):
        assert A._lib.st_Adjoint_backward_turn(ct.byref(pr), tr.fma, turn, g.data_ptr(), seg.data_ptr(),
                                               coef.data_ptr(), cot.data_ptr(), s) == 0
        if tr.n_mp:
            assert A._lib.st_Adjoint_reduce_coefficients(
                ct.byref(pr), tr.fma, tr.orders.data_ptr(), tr.n_mp, coef.data_ptr(),
                gbal.data_ptr(), 22, s) == 0
    no = tr.max_order + 1
    inv = torch.tensor([1.0 / float(np.prod(np.arange(1, k + 1))) for k in range(no)],
                       dtype=torch.float64, device=dev)
    gbal = gbal[:tr.n_mp]
    gk = torch.where(tr.mask, gbal[:, 0:2 * no:2] * inv, 0.0)
    gs = torch.where(tr.mask, gbal[:, 1:2 * no:2] * inv, 0.0)
    return loss, cot.t(), gk, gs


def _compare(eb, n, turns, K, fma, default, coords=None):
    from sixtracklib_amd.adjoint import AdjointTracker
    rng = np.random.default_rng(n + turns)
    _, species = lattices.make_particles(1)
    tr = AdjointTracker(eb, turns, species=species, K=K, fma=fma,
                        weights=(1.0, 2.0, 0.5, 1.0, 1e-6, 3.0))
    scale = np.array([3e-4, 3e-6, 3e-4, 3e-6, 0.05, 1e-4])
    X = torch.tensor(rng.normal(size=(n, 6)) * scale, device="cuda", requires_grad=True)
    tgt = torch.tensor(rng.normal(size=(turns, 6)) * scale, device="cuda")
    knl, ksl = tr.knl0, tr.ksl0
    if not default:
        knl, ksl = (t * (1 + 1e-3 * torch.rand_like(t)) for t in (knl, ksl))
    knl_in, ksl_in = (t if default else t.clone().requires_grad_() for t in (knl, ksl))
    loss = tr.loss(X, knl_in, ksl_in, tgt)
    grads = torch.autograd.grad(loss, [X] if default else [X, knl_in, ksl_in])
    per = tr.per_particle_loss(X, knl_in, ksl_in, tgt)
    wl, wc, wk, ws = _turn_by_turn(tr, X.detach(), knl, ksl, tgt)
    if fma:
        assert torch.allclose(per, wl, rtol=1e-12, atol=0.0)
    else:
        assert torch.equal(per, wl)
    for got, want in zip(grads, (wc, wk, ws)):
        assert got.shape == want.shape and torch.isfinite(got).all()
        assert float((got - want).norm()) <= REL * float(want.norm())


@pytest.mark.parametrize("n_elem", [1, 15, 16, 17, 63, 64, 65, 129, 250])
def test_gradients_around_the_length_of_a_piece(n_elem):
    eb = _lattice(n_elem, n_elem)
    for n, turns, K in ((1, 1, 64), (63, 2, 7), (65, 3, 1000), (64, 2, 1)):
        for fma in (False, True):
            _compare(eb, n, turns, K, fma, default=(n == 63))


def test_gradients_of_more_particles_than_run_side_by_side():
    _compare(_lattice(70, 3), 65601, 2, 64, False, default=False)


def test_gradients_in_groups_of_turns():
    """4,000 elements, 65,536 particles: a group of turns is one."""
    _compare(lattices.adjoint_sublattice(n_cells=80, tune=17.24), 65536, 4, 64, False, default=False)


def test_no_multipoles():
    from sixtracklib_amd.adjoint import AdjointTracker
    _, species = lattices.make_particles(1)
    eb = CBuffer()
    be.Drift(cbuffer=eb, length=1.0)
    tr = AdjointTracker(eb, 2, species=species)
    X = torch.zeros(5, 6, dtype=torch.float64, device="cuda", requires_grad=True)
    g, = torch.autograd.grad(tr.loss(X), [X])
    assert g.shape == (5, 6) and not g.any()
