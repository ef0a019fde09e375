"""The batched launch's shape: threads_per_block as the caller gives it (64:
the library's choice), and more networks than blocks fit at once, which take
several launches. Results are those of single minimizations, bit for bit."""
import pytest
import torch

from medyan_amd import _abi, mechanics, network
from test_gpu_batch import ctx_for, same

pytestmark = pytest.mark.gpu


def minimize(ctxs, nets, **kw):
    xs = [torch.tensor(net.coord, device="cuda") for net in nets]
    torch.cuda.synchronize()
    res, ms, _ = mechanics.minimize_batch(ctxs, _abi.default_cg_params(0, force_call_limit=100),
                                          [x.data_ptr() for x in xs], **kw)
    return res, ms, [x.cpu().numpy() for x in xs]


@pytest.mark.parametrize("kw,threads", [({}, 512), (dict(threads_per_block=64), 512), (dict(threads_per_block=0), 512),
                                        (dict(threads_per_block=128), 128), (dict(threads_per_block=256), 256)])
@pytest.mark.parametrize("passes", [0, -1])
def test_threads_per_block(lib, kw, threads, passes):
    nets = [network.generate(lib, "net500", n_filaments=20, seed=30 + i) for i in range(3)]
    ctxs = [ctx_for(net, _abi.MDY_PREC_FP64) for net in nets]
    assert ctxs[0].last_launch() == (0, 0)
    _, _, got = minimize(ctxs, nets, first_pass_calls=passes, **kw)
    for c, x, net in zip(ctxs, got, nets):
        blocks, t = c.last_launch()
        assert t == threads and blocks >= 1
        assert same(x, c.minimize(_abi.default_cg_params(0, force_call_limit=100), net.coord)[0])
        assert c.last_launch()[1] == 512


@pytest.mark.parametrize("passes", [0, 3, -2])
def test_several_launches(lib, passes):
    """Networks are added until the last ones, among them the quickest kind,
    end after all of the first 256: one launch runs them side by side."""
    base = [network.generate(lib, None, seed=100 + i, n_filaments=3, cyl_per_filament=3, box=700.0, n_linkers=2,
                             n_motors=0, n_branches=0) for i in range(4)]
    single = [ctx_for(b, _abi.MDY_PREC_FP64).minimize(_abi.default_cg_params(0, force_call_limit=100)) for b in base]
    its = [r.num_iter for _, _, r in single]
    assert 2 * min(its) < max(its)
    ctxs, n = [], 264
    while True:
        ctxs += [ctx_for(base[i % 4], _abi.MDY_PREC_FP64) for i in range(len(ctxs), n)]
        nets = [base[i % 4] for i in range(n)]
        ms = minimize(ctxs, nets, threads_per_block=256)[1]
        if ms[-4:].min() > ms[:256].max():
            break
        n *= 2
        assert n <= 8 * 264   # eight blocks of 256 threads are all that a CU can hold
    print(f"[gpu] {n} networks, passes {passes}", flush=True)
    res, _, got = minimize(ctxs, nets, threads_per_block=256, first_pass_calls=passes)
    for i in range(n):
        x, _, r = single[i % 4]
        assert res[i].status == 0 and same(got[i], x)
        assert (res[i].num_iter, res[i].num_force_call) == (r.num_iter, r.num_force_call)
