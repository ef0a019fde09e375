"""The quadrature mode's split of a pair's nodes into tiles (a panel of s times
a panel of t): pairs of up to 8 x 8 panels go to waves, 4 tiles each, larger
ones to blocks, at least 64 tiles and at most 16 pieces. Isolated pairs of parallel coplanar cylinders
at distances that give the panel counts around those limits, against an
independent numpy quadrature (tests/ev_quadrature.py) of each pair.

Tolerances: the separations are differences of coordinates up to 64 times
their size, raised to at most the eighth power: 8 * 64 * 2^-53, about 6e-14,
times the terms that cancel; bounds a hundred times that."""
import numpy as np
import pytest
import torch

import ev_quadrature as evq
from medyan_amd import _abi, autodiff, mechanics, network

pytestmark = pytest.mark.gpu
L = 100.0


def pairs_network(panels):
    x, b1, b2 = [], [], []
    for i, m in enumerate(panels):
        d = 120.0 if m == 1 else L / (m - 0.5)   # ceil(L / d) = m
        y = 1000.0 * i
        for off, yy in ((0.0, y), (3.0, y + d)):
            b1.append(3 * len(x)); x.append((off, yy, 0.0))
            b2.append(3 * len(x)); x.append((off + L, yy, 0.0))
    n = len(b1)
    z, zi = np.zeros(0), np.zeros(0, np.int32)
    b1, b2 = np.array(b1, np.int32), np.array(b2, np.int32)
    return network.Network(
        coord=np.array(x).ravel(), n_beads=len(x), cyl_bead1=b1, cyl_bead2=b2, cyl_id=np.arange(n, dtype=np.int64),
        cyl_filament=np.arange(n, dtype=np.int32), cyl_position=np.zeros(n, np.int32), cyl_type=np.zeros(n, np.int16),
        cyl_eq_length=np.full(n, L), cyl_exvol_k=np.full(n, 100.0), cyl_branch_child=np.full(n, -1, np.int32),
        cyl_minus_end=np.ones(n, np.uint8), fs_beadset=np.stack([b1, b2], 1).ravel(), fs_k=np.zeros(n),
        fs_l0=np.full(n, L), fb_beadset=zi, fb_k=z, fb_theta0=z, ls_beadset=zi, ls_k=z, ls_l0=z, ls_pos1=z, ls_pos2=z,
        ms_beadset=zi, ms_k=z, ms_l0=z, ms_pos1=z, ms_pos2=z, bs_beadset=zi, bs_k=z, bs_l0=z, bs_pos=z,
        bb_beadset=zi, bb_k=z, bb_theta0=z, plane=z, plane_k=z, plane_screen=z, boundary_enabled=0, box=1000.0,
        exvol_cutoff=150.0)


@pytest.mark.parametrize("panels", [(1,), (64,), (1, 2, 3, 4, 7, 8, 9), (15, 16, 17), (2, 8, 9, 32, 33) + (2,) * 300,
                                    (2, 3, 8, 12, 33) + (1,) * 8400])
def test_panel_counts(panels):
    net = pairs_network(panels)
    ctx = mechanics.Context(0, coplanar_mode=_abi.MDY_COPLANAR_QUADRATURE)
    ctx.set_network(net)
    ctx.build_neighbors()
    x = net.coord
    bs = ctx.exvol_table()[0]
    bs = np.asarray(bs).reshape(-1, 4)
    bs = bs[np.argsort(x.reshape(-1, 3)[bs[:, 0] // 3, 1])]
    assert len(bs) == len(panels) and ctx.quadrature_pair_count(x) == len(panels)
    v = np.random.default_rng(3).normal(size=x.size)
    X, V = x.reshape(-1, 3), v.reshape(-1, 3)
    dx, dv = (torch.tensor(a, device="cuda") for a in (x, v))
    total, per = ctx.energy(x)
    F = ctx.forces(x).reshape(-1, 3)
    H = autodiff.hvp(ctx, dx, dv).cpu().numpy().reshape(-1, 3)
    jvp = autodiff.energy_jvp(ctx, dx, dv).cpu().numpy()
    e = j = jabs = 0.0
    energies = {}
    for row in bs:
        b = row // 3
        c = X[b]
        i = int(c[0, 1] // 1000.0)
        m = panels[i]
        if i >= 400:   # enough of the same kind: their energies only
            e += energies[m]
            continue
        E, f, h = evq.pair(*c, 100.0 * L * L, V[b], n=16)
        energies[m] = E
        e += E
        j -= (f * V[b]).sum()
        jabs += np.abs(f * V[b]).sum()
        assert np.abs(F[b] - f).max() <= 1e-11 * np.abs(f).max(), m
        assert np.abs(H[b] - h).max() <= 1e-11 * np.abs(h).max(), m
    assert per[_abi.MDY_FF_EV] == pytest.approx(e, rel=1e-12) and total == pytest.approx(e, rel=1e-12)
    if len(panels) <= 400:
        assert abs(jvp[_abi.MDY_FF_EV] - j) <= 1e-11 * jabs
    # the same bits again, and after the totals were taken by a count
    ctx.quadrature_pair_count(x)
    assert np.array_equal(autodiff.hvp(ctx, dx, dv).cpu().numpy().reshape(-1, 3), H)
    assert np.array_equal(ctx.forces(x).reshape(-1, 3), F) and ctx.energy(x)[0] == total
    ctx.close()
