"""The complex error function of the beam fields (cerrf) where its loop
changes form: zero, arguments below 1e-100 and above 1e50, both sides of the
regions' border and of the border itself, waves that mix them; both
orientations of the ellipse.  Against the oracle, bit for bit.

A wave takes the loop with the shared reciprocal only if none of its lanes in
a region has an argument outside that loop's range, so waves of ordinary
arguments are laid out for themselves (_wave_forms counts which form each
takes); the line of test_fields_match_the_oracle has an extreme argument in
almost every wave."""
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


def _wave_forms(re, im):
    """(waves that take the shared reciprocal, waves that take the division)
    per region, near and far, for arguments in particle order: the rule of
    cerrf on the waves of 64."""
    x, y = np.abs(re), np.abs(im)
    near = (y < 4.29) & (x < 5.33)
    with np.errstate(invalid="ignore"):
        q = (1.0 - y / 4.29) * np.sqrt(1.0 - (x / 5.33) * (x / 5.33))
    extreme = (x > 1e50) | (y > 1e50) | ((x < 1e-100) & (x != 0)) | ((y < 1e-100) & (y != 0))
    out = []
    for region, plain in ((near, extreme | (near & (q < 1e-10))), (~near, extreme)):
        waves = [(region[k:k + 64], plain[k:k + 64] & region[k:k + 64]) for k in range(0, x.size, 64)]
        out.append((sum(bool(r.any() and not p.any()) for r, p in waves), sum(bool(p.any()) for r, p in waves)))
    return out


def _waves(rng, scale):
    """Arguments (re, im), 64 a wave."""
    border = [5.33 * (1 + e) for e in (-1e-3, -1e-9, -1e-15, 0.0, 1e-9)]
    border_y = [4.29 * (1 + e) for e in (-1e-3, -1e-9, -1e-15, 0.0, 1e-9)]
    inner = 5.33 * (1 - 2e-5), 4.29 * (1 - 1e-5)      # q small, not below 1e-10
    waves = []
    for _ in range(24):                               # dense points of the two regions
        waves.append((rng.uniform(0, 5.3, 64), rng.uniform(0, 4.28, 64)))
        waves.append((rng.uniform(0, 12, 64), rng.uniform(4.3, 12, 64)))
        waves.append((rng.uniform(0, 11, 64), rng.uniform(0, 9, 64)))       # both
        lo = 10.0 ** rng.uniform(-100, 0.6, (2, 64))                        # all small sizes
        waves.append((lo[0], lo[1]))
        hi = 10.0 ** rng.uniform(0.8, 49.9, (2, 64))
        waves.append((hi[0], hi[1]))
        waves.append((rng.choice([0.0, 1.0, 1e-99, 3.0], 64), rng.choice([0.0, 2.0, 1e-99], 64)))
        waves.append((rng.choice(border + [0.0, 2.0], 64), rng.choice(border_y + [0.0, 1.0], 64)))
        waves.append((rng.choice([inner[0], 1.0], 64), rng.choice([inner[1], 1.0], 64)))
        tiny = 10.0 ** rng.uniform(-300, -100.1, (2, 64))                   # outside the range
        waves.append((tiny[0], tiny[1]))
        huge = 10.0 ** rng.uniform(50.1, 80, (2, 64))
        waves.append((huge[0], huge[1]))
        one = rng.uniform(0, 11, (2, 64))                                   # one lane of a wave
        one[rng.integers(2), rng.integers(64)] = rng.choice([1e-130, 1e52])
        waves.append((one[0], one[1]))
    re, im = (np.concatenate([w[k] for w in waves]) * scale for k in (0, 1))
    return re, im


@pytest.mark.parametrize("call", [1, 2])
@pytest.mark.parametrize("sigma", [(2e-3, 1e-3), (1e-3, 3e-3)])
def test_both_forms_of_the_loop_match_the_oracle(sigma, call):
    """Waves laid out for the field's first call of the error function, or for
    its second (whose arguments are the first's times ss / sl and sl / ss)."""
    large, small = max(sigma), min(sigma)
    S = np.sqrt(2.0 * (large * large - small * small))
    rng = np.random.default_rng(11 + call)
    re, im = _waves(rng, S)                           # l and s plane of the position
    if call == 2:
        re, im = re * (large / small), im * (small / large)
    forms = [_wave_forms(re / S, im / S),
             _wave_forms(small / large * re / S, large / small * im / S)]
    for region in forms[call - 1]:
        assert region[0] >= 40 and region[1] >= 20, forms
    for region in forms[2 - call]:
        assert region[0] >= 20 and region[1] >= 20, forms
    eb = CBuffer(max_slots=4096, max_objects=8, max_pointers=8)
    be.BeamBeam4D(cbuffer=eb, charge=1e11, sigma_x=sigma[0], sigma_y=sigma[1], beta_r=1.0,
                  min_sigma_diff=1e-10, x_bb=0.0, y_bb=0.0, d_px=0.0, d_py=0.0, enabled=1)
    pb, p = lattices.gaussian_beam(re.size, seed=3, sigma_x=1e-3, sigma_y=1e-3)
    x, y = (re, im) if sigma[0] > sigma[1] else (im, re)
    p.x[:] = x * rng.choice([-1.0, 1.0], x.size)
    p.y[:] = y * rng.choice([-1.0, 1.0], y.size)
    ob, gb = CBuffer.frombytes(pb.tobytes()), CBuffer.frombytes(pb.tobytes())
    oracle_lib.track_until(ob, eb, 1)
    job = TrackJob(eb, gb, config_str="fma=0")
    job.track_until(1)
    job.collect()
    assert_particles_equal(particles_dict(particles_in(gb)), particles_dict(particles_in(ob)),
                           what="sigma %s call %d" % (sigma, call))
