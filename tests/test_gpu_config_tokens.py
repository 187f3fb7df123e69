"""Configuration tokens of the schedulers: what the configuration string
tells and restores, and that a change of it reaches the next launch."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import assert_particles_equal, particles_dict  # noqa: E402
from sixtracklib_amd import lattices  # noqa: E402
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


def _kernels(call):
    """names of the tracking kernels that ``call`` launches, one per launch"""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return [e.name.split("(")[0] for e in prof.events() if "_track" in e.name and "st_k_" in e.name]


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
