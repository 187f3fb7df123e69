"""Configuration tokens of the schedulers: what the configuration string
tells and restores, and that a change of it reaches the next launch."""
import pytest

from helpers import assert_particles_equal, particles_dict
from sixtracklib_amd import lattices
from sixtracklib_amd.cobjects import CBuffer
from sixtracklib_amd.particles import particles_in

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
