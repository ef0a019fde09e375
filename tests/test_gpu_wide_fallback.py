"""Minimizations on a few blocks whose quadrature fallbacks move them to the
whole grid: where more energies are queued than there are blocks, and where a
force is queued (parallel cylinders in the exact mode, at the first
evaluation). Coordinates, forces, counts and trace are those of a
minimization on the whole grid from the start, bit for bit."""
import numpy as np
import pytest
import torch

from medyan_amd import _abi, mechanics, network
from test_gpu_one_shot import exact  # noqa: F401  (a fixture)
from test_gpu_parity import bits_equal

pytestmark = pytest.mark.gpu


def couples(n):
    """n couples of parallel filaments of two cylinders 30 nm apart: 2 n parallel pairs."""
    fil = []
    for i in range(n):
        o = 400.0 + 600.0 * np.array([i % 8, (i // 8) % 8, i // 64])
        z = np.array([0.0, 0.0, 108.0])
        fil += [np.array([o + k * z for k in range(3)]), np.array([o + [30.0, 0.0, 0.0] + k * z for k in range(3)])]
    return network.from_filaments(fil, 6000.0)


def minimized(net, params, **opts):
    ctx = mechanics.Context(0, **opts)
    ctx.set_network(net)
    ctx.build_neighbors()
    x, f, r = ctx.minimize(params, trace_cap=100)
    t = ctx.trace()
    out = (x, f, np.array([r.energies_before[_abi.MDY_NFF], r.energies_after[_abi.MDY_NFF], r.grad_inf_norm]),
           np.array([r.num_iter, r.num_energy_call, r.num_force_call, r.num_energy_eval, r.num_safe_mode,
                     r.num_recovery, r.error_flags]), [np.asarray(t[k]) for k in sorted(t)])
    ctx.close()
    return out


def equal(a, b):
    return (all(bits_equal(p, q) for p, q in zip(a[:3], b[:3])) and np.array_equal(a[3], b[3])
            and all(np.array_equal(p, q) for p, q in zip(a[4], b[4])))


# eight blocks: one queued energy, one turn, one more than a turn, two (on the small grid to the end)
# and eight turns (moved at the first iteration)
@pytest.mark.parametrize("ls", [_abi.MDY_LS_BACKTRACKING, _abi.MDY_LS_QUADRATIC])
@pytest.mark.parametrize("precision", [_abi.MDY_PREC_FP64, _abi.MDY_PREC_MIXED])
@pytest.mark.parametrize("n", [1, 4, 5, 8, 32])
def test_queued_energies(n, precision, ls):
    net = couples(n)
    p = _abi.default_cg_params(0, force_call_limit=30, energy_rel_tol=0.0, grad_tol=1e-9, line_search=ls)
    assert equal(minimized(net, p, precision=precision), minimized(net, p, precision=precision, blocks_per_cu=1))


def test_queued_energies_against_the_oracle(exact):  # noqa: F811
    net = couples(12)
    p = _abi.default_cg_params(0, force_call_limit=8, energy_rel_tol=0.0, grad_tol=1e-9)
    x, f, _, counts, _ = minimized(net, p)
    xo, fo, ro, _ = exact.system(net).minimize(p)
    assert bits_equal(x, xo) and bits_equal(f, fo)
    assert counts[:3].tolist() == [ro.num_iter, ro.num_energy_call, ro.num_force_call]


@pytest.mark.parametrize("n", [1, 3])
def test_queued_forces(n):
    net = couples(n)
    p = _abi.default_cg_params(0, force_call_limit=2, energy_rel_tol=0.0, grad_tol=1e-9)
    opts = dict(coplanar_mode=_abi.MDY_COPLANAR_EXACT)
    assert equal(minimized(net, p, **opts), minimized(net, p, blocks_per_cu=1, **opts))


def test_queued_forces_take_the_whole_grid():
    """A force quadrature (6e8 nodes) on eight of the 256 blocks takes about 30 times as long."""
    net = couples(1)
    p = _abi.default_cg_params(0, force_call_limit=2, energy_rel_tol=0.0, grad_tol=1e-9)
    ms = []
    for blocks in (0, 1):
        ctx = mechanics.Context(0, coplanar_mode=_abi.MDY_COPLANAR_EXACT, blocks_per_cu=blocks)
        ctx.set_network(net)
        ctx.build_neighbors()
        ctx.minimize(p)
        ctx.minimize(p)
        ms.append(ctx.last_ms())
        ctx.close()
    print(f"[gpu] {ms[0]:.1f} ms, {ms[1]:.1f} on the whole grid from the start")
    assert ms[0] < 3.0 * ms[1]


def in_batch(nets, p, passes, **opts):
    ctxs = []
    for net in nets:
        c = mechanics.Context(0, **opts)
        c.set_network(net)
        c.build_neighbors()
        ctxs.append(c)
    xs = [torch.tensor(net.coord, device="cuda") for net in nets]
    fs = [torch.zeros_like(x) for x in xs]
    torch.cuda.synchronize()
    res, _, ms = mechanics.minimize_batch(ctxs, p, [x.data_ptr() for x in xs], [f.data_ptr() for f in fs],
                                          first_pass_calls=passes)
    out = [(x.cpu().numpy(), f.cpu().numpy(),
            np.array([r.energies_before[_abi.MDY_NFF], r.energies_after[_abi.MDY_NFF], r.grad_inf_norm]),
            np.array([r.num_iter, r.num_energy_call, r.num_force_call, r.num_energy_eval, r.num_safe_mode,
                      r.num_recovery, r.error_flags]), []) for x, f, r in zip(xs, fs, res)]
    for c in ctxs:
        c.close()
    return out, ms


@pytest.mark.parametrize("precision", [_abi.MDY_PREC_FP64, _abi.MDY_PREC_MIXED])
@pytest.mark.parametrize("passes", [0, 5, -2])
def test_queued_energies_in_a_batch(lib, passes, precision):
    """Networks with and without queued energies, and more of them than may run uncapped: the ones that want
    blocks suspend the launch for all."""
    nets = [couples(n) if i % 3 == 0 else network.generate(lib, "net500", n_filaments=20, seed=30 + i % 5)
            for i, n in enumerate([32, 0, 0, 1, 0, 0, 4, 0, 0, 12, 0, 0] * 3)]
    p = _abi.default_cg_params(0, force_call_limit=40, energy_rel_tol=0.0, grad_tol=1e-9)
    got, _ = in_batch(nets, p, passes, precision=precision)
    want = {}
    for i, (net, g) in enumerate(zip(nets, got)):
        key = (net.n_cyl, i % 3 == 0, float(net.coord[0]))
        if key not in want:
            want[key] = minimized(net, p, precision=precision, blocks_per_cu=1)[:4] + ([],)
        assert equal(g, want[key]), i


@pytest.mark.parametrize("n", [1, 2, 5])
def test_queued_forces_in_a_batch(lib, n):
    """The first network's forces go by quadrature: on more blocks than its lanes need (one), so that the
    batch takes about 230 ms (7300 on that one)."""
    p = _abi.default_cg_params(0, force_call_limit=2, energy_rel_tol=0.0, grad_tol=1e-9)
    opts = dict(coplanar_mode=_abi.MDY_COPLANAR_EXACT)
    nets = [couples(1)] + [network.generate(lib, "net500", n_filaments=20, seed=30 + i) for i in range(n - 1)]
    got, ms = in_batch(nets, p, 0, **opts)
    for net, g in zip(nets, got):
        assert equal(g, minimized(net, p, **opts)[:4] + ([],))
    assert ms < 1000.0
