"""Minimizations suspended and resumed many times in blocks of eight waves: a
resumed minimization starts its kernel with control flow alone, which one
thread of every block advances while the others have still to read the state
it changes. Results equal those of one pass, bit for bit."""
import numpy as np
import pytest
import torch

from medyan_amd import _abi, mechanics, network
from test_gpu_batch import ctx_for, same

pytestmark = pytest.mark.gpu
N = 40   # more networks than get 4096 threads each (those run uncapped), fewer than blocks of 512 threads


@pytest.mark.parametrize("precision", [_abi.MDY_PREC_FP64, _abi.MDY_PREC_MIXED])
@pytest.mark.parametrize("ls", [_abi.MDY_LS_BACKTRACKING, _abi.MDY_LS_QUADRATIC])
def test_resumed_equals_one_pass(lib, precision, ls):
    """Caps of 1, 4, 16, ... force calls (1: suspended before the first
    iteration), and passes that end with every completion, against one pass."""
    nets = [network.generate(lib, "net500", n_filaments=20 + 10 * (i % 4), seed=50 + i % 8) for i in range(N)]
    ctxs = [ctx_for(net, precision) for net in nets]
    params = [_abi.default_cg_params(net.n_beads, line_search=ls, force_call_limit=200) for net in nets]
    out = []
    for passes in (0, 1, -N):
        xs = [torch.tensor(net.coord, device="cuda") for net in nets]
        fs = [torch.zeros_like(x) for x in xs]
        torch.cuda.synchronize()
        res, _, _ = mechanics.minimize_batch(ctxs, params, [x.data_ptr() for x in xs], [f.data_ptr() for f in fs],
                                             first_pass_calls=passes)
        out.append([(x.cpu().numpy(), f.cpu().numpy(), np.array([r.energies_after[_abi.MDY_NFF], r.grad_inf_norm]),
                     np.array([r.num_iter, r.num_energy_call, r.num_force_call, r.num_energy_eval, r.error_flags]))
                    for x, f, r in zip(xs, fs, res)])
    for got in out[1:]:
        for i, (a, b) in enumerate(zip(out[0], got)):
            assert all(same(p, q) for p, q in zip(a[:3], b[:3])) and np.array_equal(a[3], b[3]), i
    for c in ctxs:
        c.close()
