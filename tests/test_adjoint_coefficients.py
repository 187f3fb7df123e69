"""AdjointTracker.write_coefficients and NS(Adjoint_coefficients): what they
take, what they refuse, and the words they write; the work memory of the
gradients (CPU, no kernel runs)."""
import ctypes as ct

import pytest

torch = pytest.importorskip("torch")

from sixtracklib_amd import adjoint, beam_elements as be, lattices  # noqa: E402
from sixtracklib_amd.cobjects import CBuffer  # noqa: E402


def _tracker(orders):
    eb = CBuffer()
    be.Drift(cbuffer=eb, length=1.5)
    for k, order in enumerate(orders):
        be.Multipole(cbuffer=eb, knl=[0.1 * (k + 1)] * (order + 1), ksl=[0.2] * (order + 1))
        be.Drift(cbuffer=eb, length=0.5)
    _, species = lattices.make_particles(1)
    return adjoint.AdjointTracker(eb, 2, species=species, device="cpu")


def test_a_lattice_without_multipoles_has_nothing_to_write():
    tr = _tracker([])
    plan = tr.plan(0, tr.knl0, tr.lat)         # knl0 is empty: no target
    none = tr.knl0.data_ptr()
    assert adjoint._lib.st_Adjoint_coefficients(ct.byref(plan), 0, none, none, 0, None) == 0
    plan.n_mp = 1                              # a multipole without its coefficients
    assert adjoint._lib.st_Adjoint_coefficients(ct.byref(plan), 0, none, none, 0, None) == -1


@pytest.mark.parametrize("shape", [(), (1,), (3,), (1, 3), (2, 2), (3, 3), (2, 3, 1), (1, 2, 3)])
def test_other_shapes_are_refused(shape):
    tr = _tracker([2, 1])                      # coefficients: (2, 3)
    for knl, ksl in ((torch.ones(shape, dtype=torch.float64), tr.ksl0),
                     (tr.knl0, torch.ones(shape, dtype=torch.float64))):
        with pytest.raises(ValueError, match="shape"):
            tr.write_coefficients(knl, ksl)


def test_complex_coefficients_are_refused():
    tr = _tracker([2, 1])
    with pytest.raises(ValueError, match="real"):
        tr.write_coefficients(tr.knl0.to(torch.complex128), tr.ksl0)


def test_a_tracker_on_the_cpu_writes_both_streams():
    """The packed lattice and the hot stream that a new lattice with these
    strengths packs to, and the lattice's own again with the defaults."""
    def tracker(a, b):
        eb = CBuffer()
        be.Drift(cbuffer=eb, length=1.5)
        be.Multipole(cbuffer=eb, knl=a[0], ksl=b[0])
        be.Multipole(cbuffer=eb, knl=a[1][:2], ksl=b[1][:2])
        be.Drift(cbuffer=eb, length=0.5)
        _, species = lattices.make_particles(1)
        return adjoint.AdjointTracker(eb, 2, species=species, device="cpu")

    knl = [[0.1, 0.2, 0.7, 0.9], [0.3, 0.4, 9.0, 9.0]]
    ksl = [[1.1, 1.2, 1.3, 1.7], [1.3, 1.4, 9.0, 9.0]]
    tr = tracker([[1.0, 2.0, 4.0, 6.0]] * 2, [[3.0, 5.0, 8.0, 3.0]] * 2)
    want = tracker(knl, ksl)
    lat, hot = tr.lat.clone(), tr.hot.clone()
    tr.write_coefficients(torch.tensor(knl, dtype=torch.float64), torch.tensor(ksl, dtype=torch.float64))
    assert torch.equal(tr.lat, want.lat) and torch.equal(tr.hot, want.hot)
    assert not torch.equal(tr.lat, lat) and not torch.equal(tr.hot, hot)
    tr.write_coefficients(tr.knl0, tr.ksl0)
    assert torch.equal(tr.lat, lat) and torch.equal(tr.hot, hot)
    tr = _tracker([])
    tr.write_coefficients(tr.knl0, tr.ksl0)


@pytest.mark.parametrize("n", [1, 64, 1000, 65536, 70000])
def test_work_memory_for_fewer_turns_at_a_time(n):
    """As many whole turns as fit, and below one turn what a single wave
    through all elements needs."""
    tr = _tracker([2, 1] * 50)
    tr.n_turns = 7
    plan = tr.plan(n, tr.knl0, tr.lat)
    within = adjoint._lib.st_Adjoint_gradient_doubles_within
    most = within(ct.byref(plan), 2**62)
    least = within(ct.byref(plan), 0)
    assert 0 < least <= most <= 2**29
    assert most == adjoint._lib.st_Adjoint_gradient_doubles(ct.byref(plan))
    if n > 65536:                              # the waves fill the chip one by one
        assert most == least
        return
    assert most % 7 == 0
    turn = most // 7
    assert least < turn
    for limit in (0, turn - 1, turn, turn + 1, 3 * turn - 1, 3 * turn, 6 * turn + 5, 7 * turn, 8 * turn):
        turns = min(limit // turn, 7)
        assert within(ct.byref(plan), limit) == (turns * turn if turns else least)
