"""AdjointTracker.write_coefficients and NS(Adjoint_coefficients): what they
take and what they refuse (CPU, no kernel runs)."""
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
