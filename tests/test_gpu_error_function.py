"""The complex error function of the beam fields (cerrf) where its loop
changes form: zero, arguments below 1e-100 and above 1e50, both sides of the
regions' border and of the border itself, waves that mix them; both
orientations of the ellipse.  Against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib
from helpers import particles_dict, assert_particles_equal
from sixtracklib_amd import beam_elements as be, lattices
from sixtracklib_amd.cobjects import CBuffer
from sixtracklib_amd.particles import particles_in
from sixtracklib_amd.trackjob import TrackJob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [(2e-3, 1e-3), (1e-3, 3e-3)])
def test_fields_match_the_oracle(sigma):
    scale = np.sqrt(2 * abs(sigma[0] ** 2 - sigma[1] ** 2))
    rng = np.random.default_rng(7)
    # in units of the error function's argument
    line = np.concatenate([[0.0], 10.0 ** np.arange(-130.0, -3.0, 9.0), rng.uniform(0.0, 6.0, 20),
                           5.33 * (1 + 1e-9 * np.array([-1e6, -1.0, -1e-6, 0.0, 1.0])),
                           4.29 * (1 + 1e-9 * np.array([-1e6, -1.0, -1e-6, 0.0, 1.0])),
                           [9.0, 40.0, 1e9, 1e49, 1e52]])
    a, b = (v.ravel() for v in np.meshgrid(line, line))
    order = rng.permutation(a.size)                  # waves that mix them
    a, b = np.concatenate([a, a[order]]) * scale, np.concatenate([b, b[order]]) * scale
    eb = CBuffer(max_slots=4096, max_objects=8, max_pointers=8)
    be.BeamBeam4D(cbuffer=eb, charge=1e11, sigma_x=sigma[0], sigma_y=sigma[1], beta_r=1.0,
                  min_sigma_diff=1e-10, x_bb=0.0, y_bb=0.0, d_px=0.0, d_py=0.0, enabled=1)
    pb, p = lattices.gaussian_beam(a.size, seed=3, sigma_x=1e-3, sigma_y=1e-3)
    p.x[:] = a * rng.choice([-1.0, 1.0], a.size)
    p.y[:] = b * rng.choice([-1.0, 1.0], a.size)
    ob, gb = CBuffer.frombytes(pb.tobytes()), CBuffer.frombytes(pb.tobytes())
    oracle_lib.track_until(ob, eb, 1)
    job = TrackJob(eb, gb, config_str="fma=0")
    job.track_until(1)
    job.collect()
    assert_particles_equal(particles_dict(particles_in(gb)), particles_dict(particles_in(ob)),
                           what="sigma %s" % (sigma,))
