"""The device solve where it meets a direction of non-positive curvature, on
enough blocks that some start after others have ended: the iterate, the
residual and the direction it leaves are those of conjugate gradients before
that direction, and the same bits every time.

Tolerance: a dot product over n = 6000 entries carries n 2^-53 = 7e-13 of
|p||Hp|; the shifts leave p.(H + shift I)p between a tenth and all of that in
the first step, and the few steps before the stop amplify it by less than a
thousand: 1e-8 of the largest entry, on runs of at most ten iterations whose
curvatures are further than 1e-4 |p||Hp| from zero."""
import pytest
import torch

from medyan_amd import _abi, autodiff, mechanics, network

pytestmark = pytest.mark.gpu
TOL = 1e-8


def reference(ctx, x, b, shift):
    w, r, p = torch.zeros_like(b), b.clone(), b.clone()
    rr, it = float(r @ r), 0
    while True:
        hp = autodiff.hvp(ctx, x, p) + shift * p
        php = float(p @ hp)
        assert abs(php) > 1e-4 * float(p.norm() * hp.norm())
        if not php > 0.0:
            return w, r, p, it, php, rr
        a = rr / php
        w, r = w + a * p, r - a * hp
        new = float(r @ r)
        p, rr = r + (new / rr) * p, new
        it += 1
        assert it <= 10


@pytest.mark.parametrize("mode", [_abi.MDY_COPLANAR_EXACT, _abi.MDY_COPLANAR_QUADRATURE])
@pytest.mark.parametrize("part", [0.5, 0.9, 1.1])
def test_stop_at_negative_curvature(lib, mode, part):
    net = network.generate(lib, None, seed=9, n_filaments=400, cyl_per_filament=4, box=2500.0, n_linkers=400,
                           n_motors=40)
    ctx = mechanics.Context(0, coplanar_mode=mode)
    ctx.set_network(net)
    ctx.build_neighbors()
    x = torch.tensor(net.coord, device="cuda")
    b = torch.randn(x.numel(), generator=torch.Generator().manual_seed(3), dtype=torch.float64).to("cuda")
    # from 1 on the first direction already has the curvature b.(H + shift I)b <= 0
    shift = -part * float(b @ autodiff.hvp(ctx, x, b)) / float(b @ b)
    w0, r0, p0, it0, php0, rr0 = reference(ctx, x, b, shift)
    print(f"[gpu] {net.n_beads} beads, stop after {it0} iterations", flush=True)
    assert (it0 == 0) == (part > 1.0)
    rr, runs = float(b @ b), []
    for _ in range(5):
        w, r, p, hp = torch.zeros_like(b), b.clone(), b.clone(), torch.empty_like(b)
        torch.cuda.synchronize()
        res = ctx.solve_hessian_dev(x.data_ptr(), w.data_ptr(), r.data_ptr(), p.data_ptr(), hp.data_ptr(), rr,
                                    1e-20 * rr, 100, shift)
        runs.append((w, r, p))
        assert res.not_positive == 1 and res.iterations == it0
        assert res.residual_sq == pytest.approx(rr0, rel=TOL)
        assert res.curvature == pytest.approx(php0, rel=TOL / 1e-4)
    for got, want in zip(runs[0], (w0, r0, p0)):
        assert (got - want).abs().max() <= TOL * want.abs().max()
    for other in runs[1:]:
        assert all(torch.equal(a, c) for a, c in zip(runs[0], other))
    ctx.close()
