"""Force calls followed by energy calls on one context, with pairs whose
closed-form energy is invalid (exactly parallel cylinders): the force calls
leave nothing behind that a later energy counts, neither at coordinates where
the pairs are regular, nor after a rebuild or a smaller network renumbers the
pairs, nor after more force calls than the fallback queue has entries.

Energies and forces are compared bit for bit with the exact-mode oracle."""
import numpy as np
import pytest
import torch

from medyan_amd import _abi, mechanics
from test_gpu_one_shot import context, exact, parallel_couples  # noqa: F401  (exact is a fixture)
from test_gpu_parity import bits_equal

pytestmark = pytest.mark.gpu


def moved_apart(net, seed):
    return net.coord + np.random.default_rng(seed).uniform(-3.0, 3.0, size=net.coord.shape)


def energies(ctx, x):
    """The energy of every one-shot entry point at x."""
    d_x = torch.tensor(x, device="cuda")
    out = torch.zeros(2, _abi.MDY_NFF + 1, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.energy_dev(d_x.data_ptr(), out[0].data_ptr())
    ctx.energy_dev_noalloc(d_x.data_ptr(), out[1].data_ptr())
    e = ctx.energy(x)[0]   # waits for the context's stream
    return [e, *out.cpu().numpy()[:, -1]]


@pytest.mark.parametrize("precision", [_abi.MDY_PREC_FP64, _abi.MDY_PREC_MIXED])
@pytest.mark.parametrize("n", [1, 65, 130])
def test_energy_where_the_pairs_are_regular(exact, n, precision):  # noqa: F811
    net = parallel_couples(n)
    ctx = mechanics.Context(0, precision=precision)
    ctx.set_network(net)
    ctx.build_neighbors()
    moved = moved_apart(net, n)
    for x in (moved, net.coord, moved):
        ctx.forces(net.coord)
        f = ctx.forces(net.coord)
        if precision == _abi.MDY_PREC_FP64:
            assert bits_equal(f, exact.system(net).forces(net.coord))
        assert bits_equal(energies(ctx, x), [exact.system(net).energy(x)[0]] * 3)
    ctx.close()


def test_energy_after_a_rebuild(exact):  # noqa: F811
    """The couples of the first half drift apart beyond the cutoff: the list halves and is renumbered."""
    net = parallel_couples(64)
    ctx = context(net)
    x = moved_apart(net, 3).reshape(-1, 3)
    x[:x.shape[0] // 2].reshape(-1, 2, 2, 3)[:, 1] += [0.0, 250.0, 0.0]
    ctx.forces(net.coord)
    x = x.reshape(net.coord.shape)
    ctx.build_neighbors(x)
    assert len(ctx.exvol_table()[1]) == 32
    want = exact.system(net, coord=x).energy(x)[0]
    assert bits_equal(energies(ctx, x), [want] * 3)
    ctx.close()


def test_energy_after_a_smaller_network(exact):  # noqa: F811
    net, small = parallel_couples(130), parallel_couples(2)
    ctx = context(net)
    ctx.forces(net.coord)
    ctx.set_network(small)
    ctx.build_neighbors()
    for x in (moved_apart(small, 5), small.coord):
        assert bits_equal(energies(ctx, x), [exact.system(small).energy(x)[0]] * 3)
    ctx.close()


def test_more_force_calls_than_queue_entries(exact):  # noqa: F811
    net = parallel_couples(130)
    ctx = context(net)
    d_x = torch.tensor(net.coord, device="cuda")
    f = torch.zeros_like(d_x)
    torch.cuda.synchronize()
    for _ in range(4096 // 130 + 2):
        ctx.forces_dev(d_x.data_ptr(), f.data_ptr(), 0)
    ctx.sync_errors()
    for x in (moved_apart(net, 7), net.coord):
        assert bits_equal(energies(ctx, x), [exact.system(net).energy(x)[0]] * 3)
    ctx.close()
