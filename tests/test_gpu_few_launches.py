"""Recorded single-token passes on both sides of the line between a handful of launches, which go out one by one, and a graph:
every replay against the sums computed on the host, with the backend's own eager work and reads between the replays."""
import numpy as np
import pytest

from util import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ops", [1, 2, 7, 8, 9, 10, 11, 40])
def test_replays_of_short_and_long_passes(n_ops):
    import inferred_hip as ih
    be = ih.Hip(exact=True)
    try:
        r = rng(n_ops)
        n = 2048
        x, other = np.zeros(n, np.float32), np.zeros(n, np.float32)
        add = [r.integers(-50, 50, n).astype(np.float32) for _ in range(n_ops)]
        for turn in range(8):
            fresh = r.integers(-1000, 1000, n).astype(np.float32)
            x[:] = fresh
            be.begin_pass(1)
            be.host_wrote(x)
            for a in add:
                be.add_assign(x, a)
            be.end_pass()
            be.host_needs(x)
            be.raise_if_error()
            assert np.array_equal(x, fresh + sum(add)), turn       # whole numbers: every order gives the same
            if turn < 3:
                continue
            other[:] = fresh
            be.begin_pass(2)                                        # work that no recorded pass knows of
            be.host_wrote(other)
            be.add_assign(other, add[0])
            be.end_pass()
            be.host_needs(other)
            assert np.array_equal(other, fresh + add[0]), turn
            be.raise_if_error()
        stats = be.graph_stats()
        assert stats["captures"] >= 1 and stats["replays"] >= 3, stats
        assert be.launched_replays() == (stats["replays"] if n_ops <= 10 else 0), stats
    finally:
        be.take_error()
        be.close()
