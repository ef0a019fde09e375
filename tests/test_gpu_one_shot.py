"""One-shot calls whose queue of quadrature fallbacks is empty, one, the tail
kernel's 64 blocks, one more, and more than two each; the next call after one
with fallbacks starts from an empty queue; the allocation-free form alike."""
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


def parallel_couples(n):
    """n couples of parallel one-cylinder filaments 30 nm apart."""
    fil = []
    for i in range(n):
        o = 400.0 + 600.0 * np.array([i % 8, (i // 8) % 8, i // 64])
        fil += [np.array([o, o + [0.0, 0.0, 108.0]]), np.array([o + [30.0, 0.0, 0.0], o + [30.0, 0.0, 108.0]])]
    return network.from_filaments(fil, 6000.0)


def context(net):
    ctx = mechanics.Context(0)
    ctx.set_network(net)
    ctx.build_neighbors()
    assert len(ctx.exvol_table()[1]) == net.n_cyl // 2
    return ctx


@pytest.mark.parametrize("n", [1, 64, 65, 130])
def test_energy_with_fallbacks(exact, n):
    net = parallel_couples(n)
    moved = net.coord + np.random.default_rng(n).uniform(-3.0, 3.0, size=net.coord.shape)
    ctx = context(net)
    for x in (net.coord, net.coord, moved, net.coord):
        # the pair list is that of the starting coordinates, in the oracle as here
        want = exact.system(net).energy(x)[0]
        assert bits_equal([ctx.energy(x)[0]], [want])
        d_x = torch.tensor(x, device="cuda")
        out = torch.zeros(_abi.MDY_NFF + 1, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ctx.energy_dev_noalloc(d_x.data_ptr(), out.data_ptr())
        ctx.energy(x)   # waits for the context's stream
        assert bits_equal(out.cpu().numpy()[-1:], [want])
    ctx.close()


def test_forces_with_fallbacks(exact):
    net = parallel_couples(2)
    moved = net.coord + np.random.default_rng(2).uniform(-3.0, 3.0, size=net.coord.shape)
    ctx = context(net)
    for x in (net.coord, moved, net.coord):
        start = np.linspace(-1.0, 1.0, x.size).reshape(x.shape)
        want = start + exact.system(net).forces(x)
        assert bits_equal(ctx.forces(x, accum=start.copy()), want)
    ctx.close()
