"""The batched launch's shape: threads_per_block as the caller gives it (64:
the library's choice). Results are those of single minimizations, bit for bit."""
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
