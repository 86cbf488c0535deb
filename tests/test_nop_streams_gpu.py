"""GPU check of backward passes on two streams, each with its own workspace, that add to one gradient."""
import numpy as np
import pytest
import torch

from oracle import nop_ref as R
from tests.test_nop_bricks_gpu import SCALES, _bits, _case

pytestmark = pytest.mark.gpu


def test_two_streams_add_to_one_gradient():
    from allscale_ipic3d_amd import field_operator as FO
    n = (12, 20, 48)
    nets, inputs = [], []
    for seed in (31, 32):
        u, p = _case(n, 31)
        u = np.roll(u, seed, 0)
        rng = np.random.default_rng(seed)
        dout = np.zeros((u.size // 16, 16), dtype=np.float32)
        dout[:, :6] = R.bf(torch.as_tensor(rng.normal(size=(len(dout), 6)).astype(np.float32))).numpy()
        net = FO.Network(n, SCALES, params=p, train=True, stream=torch.cuda.Stream().cuda_stream)
        du = FO.Dev(2 * u.size)
        du.upload(_bits(u))
        net.dout.upload(_bits(dout))
        net.forward(du.ptr, train=True)
        net.sync()
        nets.append(net)
        inputs.append(du)

    def backward(net, u, grad):
        FO._chk(FO.nop_lib().ipic_nop_backward(net.n3, u.ptr, net.wb.ptr, net.params.ptr, net.ws.ptr, net.dout.ptr,
                                               grad.ptr, net.stream))

    def run(which):
        grad = nets[0].grad
        grad.zero()
        torch.cuda.synchronize()
        for net, u in which:
            backward(net, u, grad)
        torch.cuda.synchronize()
        return grad.download(np.float32)

    pairs = list(zip(nets, inputs))
    alone = [run([q]) for q in pairs]
    for _ in range(10):
        # two terms added to zero round once, in either order
        np.testing.assert_array_equal(run(pairs), alone[0] + alone[1])
