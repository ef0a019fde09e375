"""Sizes at which the rebuild's cells and rows can go wrong: rows that end on,
before and after the 16 neighbours kept from the count, cylinders far apart and
on the negative side (cells that share buckets), cells whose indices saturate,
and cylinder counts around the block's. Pair list and tables equal the oracle's."""
import numpy as np
import pytest

from medyan_amd import mechanics, network
from test_gpu_parity import bits_equal

pytestmark = pytest.mark.gpu


def scattered(mid, seed):
    """One-cylinder filaments of 108 nm with these midpoints."""
    u = np.random.default_rng(seed).normal(size=mid.shape)
    u *= 54.0 / np.linalg.norm(u, axis=1, keepdims=True)
    return network.from_filaments([np.array([m - v, m + v]) for m, v in zip(mid, u)], 4000.0)


def check(net, oracle):
    ctx = mechanics.Context(0)
    ctx.set_network(net)
    ctx.build_neighbors()
    pairs = oracle.nl_pairs(net, net.coord)
    np.testing.assert_array_equal(ctx.pairs(), pairs)
    s = oracle.system(net, net.coord)
    bs, kr = ctx.exvol_table()
    np.testing.assert_array_equal(bs, s.ev_table[0])
    assert bits_equal(kr, s.ev_table[1] * s.ev_table[2][:, 0] * s.ev_table[2][:, 1])
    ctx.close()
    return pairs


@pytest.mark.parametrize("n", [2, 16, 17, 18, 33, 70])
def test_row_lengths(oracle, n):
    """All within reach of each other: rows of 0 to n - 1."""
    mid = 2000.0 + np.random.default_rng(n).uniform(-30.0, 30.0, size=(n, 3))
    assert len(check(scattered(mid, n), oracle)) == n * (n - 1) // 2


@pytest.mark.parametrize("n", [3, 255, 256, 257, 1025])
def test_negative_and_far_cells(oracle, n):
    """Clusters of three at random places within +-1e6 nm."""
    rng = np.random.default_rng(n)
    at = np.repeat(rng.uniform(-1e6, 1e6, size=((n + 2) // 3, 3)), 3, axis=0)[:n]
    assert len(check(scattered(at + rng.uniform(-40.0, 40.0, size=at.shape), n), oracle)) > 0


@pytest.mark.parametrize("far", [1e12, 1e15])
def test_cells_beyond_the_integers(oracle, far):
    """Midpoints past the cells' integer range share the last cell."""
    rng = np.random.default_rng(1)
    at = np.array([[far, 0, 0], [far, 0, 0], [-far, 0, 0], [-far, 0, 0], [0, far, -far], [0, far, -far], [0, 0, 0]])
    check(scattered(at + rng.uniform(-20.0, 20.0, size=at.shape), 2), oracle)
