"""Configuration tokens of the schedulers: what the configuration string
tells and restores, and that a change of it reaches the next launch."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import assert_particles_equal, particles_dict  # noqa: E402
from sixtracklib_amd import beam_elements as be, lattices  # noqa: E402
from sixtracklib_amd.cobjects import CBuffer  # noqa: E402
from sixtracklib_amd.particles import particles_in  # noqa: E402

pytestmark = pytest.mark.gpu


def _tokens(batch):
    return dict(t.split("=") for t in batch.config.split() if "=" in t)


def test_batch_config_tells_and_restores_the_walk():
    """A captured graph is replayed for the configuration it was captured
    under; hot selects other kernels and launch shapes, so it is part of it."""
    from sixtracklib_amd.trackbatch import TrackBatch
    rings = lattices.lhc_like_ring_family(2, seed=0, n_cells=8, n_cavities=1)
    parts = [lattices.matched_gaussian_beam(n, seed=1)[0] for n in (100, 700)]
    start = [pb.words.copy() for pb in parts]
    batch = TrackBatch(rings, parts, config_str="fma=0 balance=0 graph=1 hot=1 ppl=auto mix=0")
    seen, first = [], None
    for hot in ("1", "0", "1"):
        batch.set_config("hot=" + hot)
        assert _tokens(batch)["hot"] == hot and _tokens(batch)["mix"] == "0"
        seen.append(batch.config)
        for pb, w in zip(parts, start):
            pb.words[:] = w
        batch.push()
        batch.track_until(3)
        batch.collect()
        got = [particles_dict(particles_in(CBuffer.frombytes(pb.tobytes()))) for pb in parts]
        first = first or got
        for g, w in zip(got, first):
            assert_particles_equal(g, w, what="hot=" + hot)
    assert seen[0] != seen[1] and seen[0] == seen[2]
    batch.set_config("fma=1 hot=0 ppl=2 mix=1")
    batch.set_config(seen[1])                      # the string restores what it tells
    assert batch.config == seen[1]


def _kernels(call, every=False):
    """names of the tracking kernels that ``call`` launches, one per launch;
    with ``every`` of all of the library's"""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return [e.name.split("(")[0] for e in prof.events()
            if "st_k_" in e.name and (every or "_track" in e.name)]


@pytest.mark.parametrize("n, cfg, walk", [
    (1000, "ppl=auto", {"hot"}),
    (530000, "ppl=auto", {"mix"}),             # more than one particle per resident lane
    (1000, "ppl=2", {"track2"}),
    (1000, "ppl=2 balance=0", {"track2"}),
])
def test_hot_0_runs_the_compiled_loop(n, cfg, walk):
    """At every number of particles per lane that the walk has a kernel for."""
    from sixtracklib_amd.trackjob import TrackJob
    eb = lattices.fodo_ring(n_cells=4)
    end = {}
    for hot in ("1", "0", "auto"):
        pb, p = lattices.gaussian_beam(n, seed=2, sigma_x=1e-4, sigma_y=1e-4)
        job = TrackJob(eb, pb, config_str="fma=1 hot=%s %s" % (hot, cfg))
        names = _kernels(lambda: job.track_until(2))
        assert names, "no tracking kernel seen"
        special = {k for k in ("hot", "mix", "track2") if any(k in name for name in names)}
        assert special == (set() if hot == "0" else walk), (hot, names)
        job.collect()
        end[hot] = np.stack([np.array(p.x), np.array(p.px), np.array(p.zeta), np.array(p.delta)])
    assert np.array_equal(end["0"], end["1"]) and np.array_equal(end["0"], end["auto"])


@pytest.mark.parametrize("hot, one, two", [(1, 4, 4), (0, 12, 0)])
def test_autotune_times_every_launch_form_once(hot, one, two):
    """Candidates of one and of two particles per lane that run other launches
    (a workgroup of the walk is one wave whatever block says), each timed with
    one launch of one turn, and the three fastest a second time."""
    from sixtracklib_amd.trackbatch import TrackBatch
    rings = lattices.lhc_like_ring_family(2, seed=0, n_cells=8, n_cavities=1)
    parts = [lattices.matched_gaussian_beam(n, seed=1)[0] for n in (100, 700)]
    batch = TrackBatch(rings, parts, config_str="fma=1 hot=%d" % hot)
    names = _kernels(lambda: batch.autotune(trial_turns=1, skip_turns=0))
    names = [k for k in names if "_lds" not in k]
    pairs = sum("track2" in k for k in names)
    assert one <= len(names) - pairs <= one + 3 and two <= pairs <= two + 3
    assert _tokens(batch)["block"] in (("256",) if hot else ("64", "128", "256"))


def _all_lost_at_once(heavy=False):
    """402 elements, or 3 with a space-charge map; no particle passes the first."""
    eb = CBuffer(max_slots=65536, max_objects=512, max_pointers=512)
    be.LimitRect(cbuffer=eb, min_x=-1e-12, max_x=1e-12, min_y=-1e-12, max_y=1e-12)
    if heavy:
        be.SCCoasting(cbuffer=eb, number_of_particles=1e10, circumference=1e3, sigma_x=1e-3,
                               sigma_y=1e-3, length=1.0, x_co=0.0, y_co=0.0, min_sigma_diff=1e-10,
                               enabled=1)
    for _ in range(1 if heavy else 401):
        be.Drift(cbuffer=eb, length=0.1)
    return eb


# one launch holds 2^24 element passes: 41,734 turns of 402 elements; a map out
# of line counts as many passes as it may take longer than one
@pytest.mark.parametrize("heavy, at_turn, until, one_launch", [
    (False, 0, 41734, True), (False, 0, 41735, False),
    (False, 10**6, 10**6 + 1, True), (False, 2**40, 2**40 + 41734, True),
    (False, -41000, 734, True), (False, -41000, 735, False),
    (True, 0, 1000, True), (True, 0, 2**24 // 3, False),
])
def test_one_launch_for_as_many_turns_as_are_to_go(heavy, at_turn, until, one_launch):
    from sixtracklib_amd.trackjob import TrackJob
    pb, p = lattices.gaussian_beam(100, seed=2, sigma_x=1e-4, sigma_y=1e-4)
    p.at_turn[:] = at_turn
    p.at_turn[7], p.state[7] = at_turn - 10**9, 0       # lost: not to be tracked
    job = TrackJob(_all_lost_at_once(heavy), pb)
    for _ in range(2):                                  # made with the job, and pushed
        names = _kernels(lambda: job.track_until(until), every=True)
        assert (len(names) == 1) == one_launch, names
        job.push_particles()


def test_one_launch_a_turn_far_from_turn_0():
    """The turns a job has tracked count as done: track_until, track_line."""
    from sixtracklib_amd.trackjob import TrackJob
    eb = lattices.fodo_ring(n_cells=100)
    pb, p = lattices.gaussian_beam(64, seed=2, sigma_x=1e-6, sigma_y=1e-6, sigma_px=1e-8, sigma_py=1e-8)
    p.at_turn[:] = 41730
    job = TrackJob(eb, pb)
    for turn in range(41731, 41740):
        names = _kernels(lambda: job.track_until(turn), every=True)
        assert len(names) == 1, (turn, names)
    for _ in range(3):
        job.track_line(0, eb.n_objects, finish_turn=True)
    names = _kernels(lambda: job.track_until(41743), every=True)
    assert len(names) == 1
    job.collect()
    assert np.all(np.array(p.state) == 1) and np.all(np.array(p.at_turn) == 41743)
