"""Sizes at which the sweep's and the gather's lane arithmetic can go wrong:
excluded-volume pair counts around the wave (32 pairs), pairs at the coplanar
threshold, beads whose slot rows end on, before and after a group of 16, and a
cluster of one block that takes more turns than its block sums hold without
carrying. Bit for bit against the exact-mode oracle, or against the same
minimization on the whole device."""
import numpy as np
import pytest
import torch

from medyan_amd import _abi, mechanics, network
from test_gpu_parity import bits_equal

pytestmark = pytest.mark.gpu


@pytest.fixture
def exact(oracle):
    oracle.set_exact(1)
    yield oracle
    oracle.set_exact(0)


def couples(n, seed, third=None):
    """n couples of one-cylinder filaments crossing 20 to 60 nm apart, couples
    out of each other's reach: n excluded-volume pairs."""
    rng = np.random.default_rng(seed)
    fil = []
    for i in range(n):
        o = 400.0 + 600.0 * np.array([i % 8, (i // 8) % 8, i // 64])
        a, b = (v / np.linalg.norm(v) for v in rng.normal(size=(2, 3)))
        d = rng.normal(size=3)
        d *= rng.uniform(20.0, 60.0) / np.linalg.norm(d)
        fil.append(np.array([o - 54 * a, o + 54 * a]))
        fil.append(np.array([o + d - 54 * b, o + d + 54 * b]))
        if third is not None:
            third(i, fil[-2], fil[-1])
    return network.from_filaments(fil, 6000.0)


def check(net, exact):
    ctx = mechanics.Context(0)
    ctx.set_network(net)
    ctx.build_neighbors()
    s = exact.system(net)
    e, _ = ctx.energy(net.coord)
    assert bits_equal([e], [s.energy()[0]])
    assert bits_equal(ctx.forces(net.coord), s.forces())
    n = len(ctx.exvol_table()[1])
    ctx.close()
    return n


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 97])
def test_pair_counts_around_the_wave(exact, n):
    assert check(couples(n, n), exact) == n


def test_pairs_at_the_coplanar_threshold(exact):
    """The last bead placed at |cos| = 0.1 (1 + k 1e-14) from the plane of the
    other three, k = -40 .. 40: the quick test must leave those to the exact one."""
    def place(i, p, q):
        n = np.cross(p[1] - p[0], q[0] - p[0])
        n /= np.linalg.norm(n)
        u = q[1] - p[0]
        r = np.linalg.norm(u)
        t = u - (u @ n) * n
        t /= np.linalg.norm(t)
        c = 0.1 * (1.0 + (i - 40) * 1e-14)
        q[1] = p[0] + r * (c * n + np.sqrt(1.0 - c * c) * t)
    assert check(couples(81, 5, place), exact) == 81


@pytest.mark.parametrize("links", [3, 12, 13, 14, 15, 29, 30, 31, 61])
def test_row_lengths(exact, links):
    """A bead with `links` linkers besides its stretching term."""
    rng = np.random.default_rng(links)
    hub = np.array([[1500.0, 1500, 1500], [1608, 1500, 1500]])
    fil = [hub]
    items = []
    for i in range(links):
        v = rng.normal(size=3)
        o = hub[0] + 400.0 * v / np.linalg.norm(v)
        fil.append(np.array([o, o + 108.0 * v / np.linalg.norm(v)]))
        items.append((0, 0, rng.uniform(0.1, 0.9), i + 1, 0, rng.uniform(0.1, 0.9), 8.0, 300.0))
    check(network.from_filaments(fil, 3000.0, linkers=items), exact)


@pytest.mark.parametrize("precision", [_abi.MDY_PREC_FP64, _abi.MDY_PREC_MIXED])
def test_one_small_block_takes_many_turns(lib, precision):
    """Two networks share a launch by weights that leave the second one block
    (about 40 turns per sweep): the same bits as on its own."""
    nets = [network.generate(lib, "net500", seed=s, n_filaments=f, box=b) for s, f, b in ((3, 20, 1200.0),
                                                                                       (4, 900, 4000.0))]
    p = _abi.default_cg_params(0, force_call_limit=40)
    out = []
    for batch in (False, True):
        ctxs, xs, fs = [], [], []
        for n in nets:
            c = mechanics.Context(0, precision=precision)
            c.set_network(n)
            c.build_neighbors()
            ctxs.append(c)
            xs.append(torch.tensor(n.coord, device="cuda"))
            fs.append(torch.zeros_like(xs[-1]))
        torch.cuda.synchronize()
        if batch:
            res, _, _ = mechanics.minimize_batch(ctxs, p, [x.data_ptr() for x in xs], [f.data_ptr() for f in fs],
                                                 threads_per_block=64, weights=[1e12, 1.0])
        else:
            res = [c.minimize_dev(p, x.data_ptr(), f.data_ptr()) for c, x, f in zip(ctxs, xs, fs)]
        out.append([(x.cpu().numpy(), f.cpu().numpy(), r.energies_after[_abi.MDY_NFF], r.num_iter)
                    for x, f, r in zip(xs, fs, res)])
        for c in ctxs:
            c.close()
    for a, b in zip(*out):
        assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1]) and bits_equal([a[2]], [b[2]]) and a[3] == b[3]
