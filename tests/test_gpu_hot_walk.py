"""The scheduled record walk (track_hot.h, config token hot) against the
oracle (exact build, bit for bit) and against the compiled loop (both
builds, bit for bit): every record kind and multipole order it handles,
alone and behind a drift, records it leaves to the caller (orders above 10,
curvature, cavities, DriftExact, DipoleEdge) between them, losses at every
kind that can lose a particle, streams shorter and longer than the interval
of its read-ahead, and particle counts around a wave and a tile."""
import numpy as np
import pytest

import oracle_lib
from helpers import particles_dict, assert_particles_equal
from sixtracklib_amd.cobjects import CBuffer
from sixtracklib_amd.particles import particles_in
from sixtracklib_amd import lattices, beam_elements as be

pytestmark = pytest.mark.gpu


def _multipole(eb, rng, order, **kw):
    scale = 1e-7 * np.array([float(np.prod(np.arange(1, k + 1))) / 0.01 ** k
                             for k in range(order + 1)])
    be.Multipole(cbuffer=eb, knl=rng.normal(0.0, 1.0, order + 1) * scale,
                 ksl=rng.normal(0.0, 1.0, order + 1) * scale, **kw)


def _lattice(seed, n_blocks):
    """Every kind in a random order, ``n_blocks`` times over."""
    rng = np.random.default_rng(seed)
    eb = CBuffer(max_slots=4096 * n_blocks, max_objects=64 * n_blocks, max_pointers=64 * n_blocks)

    def aperture(kind):
        if kind == "rect":
            be.LimitRect(cbuffer=eb, min_x=-0.02, max_x=0.021, min_y=-0.019, max_y=0.02)
        elif kind == "ellipse":
            be.LimitEllipse(cbuffer=eb, a=0.021, b=0.02)
        else:
            be.LimitRectEllipse(cbuffer=eb, max_x=0.02, max_y=0.02, a_squ=4.2e-4, b_squ=4e-4)

    for _ in range(n_blocks):
        items = [("dm", k) for k in range(11)] + [("m", k) for k in range(11)]
        items += [("m", 11), ("dm", 14), ("curv", 3), ("dcurv", 1)] + [("d", 0)] * 4
        items += [(k, 0) for k in ("shift", "rot", "edge", "cavity", "exact", "rect", "ellipse",
                                   "rectellipse", "dd")]
        rng.shuffle(items)
        for kind, order in items:
            order = int(order)
            if kind in ("dm", "d", "dd", "dcurv"):
                be.Drift(cbuffer=eb, length=float(rng.uniform(0.05, 0.4)))
            if kind == "dd":
                be.Drift(cbuffer=eb, length=float(rng.uniform(0.05, 0.4)))
            if kind in ("dm", "m"):
                _multipole(eb, rng, order)
            elif kind in ("curv", "dcurv"):
                _multipole(eb, rng, order, hxl=1e-6, hyl=-2e-7, length=0.7)
            elif kind == "shift":
                be.XYShift(cbuffer=eb, dx=rng.normal(0, 1e-5), dy=rng.normal(0, 1e-5))
            elif kind == "rot":
                be.SRotation(cbuffer=eb, angle=float(rng.normal(0, 2.0)))
            elif kind == "edge":
                be.DipoleEdge(cbuffer=eb, r21=1e-4, r43=-1e-4)
            elif kind == "cavity":
                be.Cavity(cbuffer=eb, voltage=1e6, frequency=400e6, lag=180.0)
            elif kind == "exact":
                be.DriftExact(cbuffer=eb, length=0.2)
            elif kind in ("rect", "ellipse", "rectellipse"):
                aperture(kind)
    return eb


def _beam(n, seed, lost_at_drift):
    pb, p = lattices.gaussian_beam(n, seed=seed, sigma_x=6e-3, sigma_y=6e-3, sigma_px=1e-5,
                                   sigma_py=1e-5)
    if lost_at_drift:                         # beyond the 1 m global aperture, and NaN
        x, px = np.asarray(p.x), np.asarray(p.px)
        x[::7] = 0.015
        px[::7] = 9.0
        x[::11] = np.nan
    return pb


def _run(eb, pb, cfg, turns):
    from sixtracklib_amd.trackjob import TrackJob
    b = CBuffer.frombytes(pb.tobytes())
    job = TrackJob(eb, b, config_str=cfg)
    for t in turns:
        job.track_until(t)
    job.collect()
    return particles_dict(particles_in(b))


@pytest.mark.parametrize("n,n_blocks,lost_at_drift", [(1, 1, False), (63, 1, True), (64, 3, False),
                                                      (65, 8, True), (1000, 8, True)])
def test_hot_walk_is_the_loop_and_the_oracle(n, n_blocks, lost_at_drift):
    eb = _lattice(n_blocks, n_blocks)
    pb = _beam(n, 5 + n, lost_at_drift)
    turns = (1, 4)
    for fma in (0, 1):
        loop = _run(eb, pb, "fma=%d ppl=1 hot=0" % fma, turns)
        for cfg in ("fma=%d ppl=1 hot=1", "fma=%d", "fma=%d hot=1 ppl=1 balance=0",
                    "fma=%d hot=1 ppl=1 waves_per_cu=1 turns_per_launch=1"):
            assert_particles_equal(_run(eb, pb, cfg % fma, turns), loop, what=cfg % fma)
        if fma == 0:
            ob = CBuffer.frombytes(pb.tobytes())
            for t in turns:
                oracle_lib.track_until(ob, eb, t)
            assert_particles_equal(loop, particles_dict(particles_in(ob)), what="oracle")
            if n >= 63:
                alive = int(np.count_nonzero(loop["state"]))
                assert 0 < alive < n


def _run_lines(eb, pb, cfg, cuts, turns):
    from sixtracklib_amd.trackjob import TrackJob
    b = CBuffer.frombytes(pb.tobytes())
    job = TrackJob(eb, b, config_str=cfg)
    for _ in range(turns):
        for lo, hi in zip(cuts, cuts[1:]):
            job.track_line(lo, hi, finish_turn=hi == cuts[-1])
    job.collect()
    return particles_dict(particles_in(b))


@pytest.mark.parametrize("n,n_blocks,step", [(1, 1, 1), (65, 1, 2), (200, 2, 3), (1000, 3, 17),
                                             (1000, 3, 1000)])
def test_hot_lines_are_the_full_kernel_and_track_until(n, n_blocks, step):
    """track_line in pieces that cut records of a Drift and a Multipole in
    two, against the full kernel (hot=0); with a wave of particles that
    start at another path length (they keep their own), against it too."""
    eb = _lattice(20 + n_blocks, n_blocks)
    cuts = list(range(0, eb.n_objects, step)) + [eb.n_objects]
    pb = _beam(n, 50 + n, n >= 65)
    for fma in (0, 1):
        want = _run_lines(eb, pb, "fma=%d hot=0" % fma, cuts, 2)
        got = _run_lines(eb, pb, "fma=%d" % fma, cuts, 2)
        assert_particles_equal(got, want, what="lines, fma=%d" % fma)
        until = _run(eb, pb, "fma=%d" % fma, (2,))
        if fma == 0:
            assert_particles_equal(got, until, what="lines and track_until")
    p = particles_in(pb)
    np.asarray(p.s)[n // 2:] = 3.25
    got, want = (_run_lines(eb, pb, "fma=0 hot=%s" % h, cuts, 1) for h in ("auto", "0"))
    assert_particles_equal(got, want, what="lines from another path length")


def test_lines_with_out_of_line_maps_and_monitors():
    eb = lattices.kitchen_sink(with_monitor=True)
    pb, _ = lattices.gaussian_beam(300, seed=3, sigma_x=8e-3, sigma_y=8e-3)
    for step in (1, 2, 7):
        cuts = list(range(0, eb.n_objects, step)) + [eb.n_objects]
        for fma in (0, 1):
            want = _run_lines(eb, pb, "fma=%d hot=0" % fma, cuts, 2)
            assert_particles_equal(_run_lines(eb, pb, "fma=%d" % fma, cuts, 2), want, what="step %d" % step)


@pytest.mark.parametrize("at_turn", [0, -3, "mixed"])
def test_requests_end_with_every_particle_at_its_turn(at_turn):
    """A request that ends without a further select pass (one launch of
    small sets, or launches that hold every tile) leaves no particle
    behind, also where the particles start at different or negative turns."""
    eb = _lattice(31, 1)
    pb, p = lattices.gaussian_beam(700, seed=4, sigma_x=4e-3, sigma_y=4e-3, sigma_px=1e-5, sigma_py=1e-5)
    turns = np.asarray(p.at_turn)
    if at_turn == "mixed":
        turns[:] = np.random.default_rng(5).integers(-4, 4, turns.size)
        turns[:3] = (0, -2, 3)
    else:
        turns[:] = at_turn
    want = _run(eb, pb, "fma=0 compact=0", (3, 5))
    assert set(want["at_turn"][want["state"] == 1].tolist()) == {5}
    for cfg in ("fma=0", "fma=0 waves_per_cu=1", "fma=0 waves_per_cu=2 turns_per_launch=2",
                "fma=0 hot=0", "fma=0 ppl=2", "fma=0 staging=lds"):
        assert_particles_equal(_run(eb, pb, cfg, (3, 5)), want, what=cfg)


@pytest.mark.parametrize("n", [1, 64, 65, 127, 129, 1000])
def test_two_particles_per_lane_are_the_loop(n):
    """The walk with one register set, two particles per lane: every record
    kind, pairs of which one or both lanes are empty or lost."""
    eb = _lattice(40 + n, 3)
    pb = _beam(n, 90 + n, n > 1)
    for fma in (0, 1):
        want = _run(eb, pb, "fma=%d ppl=1 hot=0" % fma, (1, 3))
        for cfg in ("fma=%d ppl=2", "fma=%d ppl=2 balance=0", "fma=%d ppl=2 waves_per_cu=1 turns_per_launch=1"):
            assert_particles_equal(_run(eb, pb, cfg % fma, (1, 3)), want, what=cfg % fma)


@pytest.mark.parametrize("n,fma", [(64 * 4096 + 1, 1), (64 * 8192, 1), (64 * 8192 + 1, 1), (64 * 8192 + 1, 0),
                                   (700001, 1), (128 * 8192 - 64, 0)])
def test_launches_that_fill_the_chip_are_the_loop(n, fma):
    """The walk with one register set as the sizes select it: one particle
    per lane from more than four waves per SIMD (FMA build), and mixed
    launches of one and two per lane above eight."""
    eb = _lattice(60, 1)
    pb = _beam(n, 7, True)
    want = _run(eb, pb, "fma=%d ppl=1 hot=0" % fma, (1, 2))
    assert 0 < np.count_nonzero(want["state"]) < n
    for cfg in ("fma=%d", "fma=%d ppl=1"):
        assert_particles_equal(_run(eb, pb, cfg % fma, (1, 2)), want, what=cfg % fma)
