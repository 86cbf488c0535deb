"""GPU checks of the operator's convolutions and weight gradients over many bricks and at the
smallest grid, against the torch CPU reference (oracle/nop_ref.py) and through the periodic
grid's shift symmetry: rolling the input and the output gradient rolls the activations and leaves
the parameter gradient as it is, so a brick that is left out, done twice or read at a wrong
offset shows at full size."""
import numpy as np
import pytest
import torch

from oracle import nop_ref as R

pytestmark = pytest.mark.gpu

SCALES = {"in_E": 1.0, "in_B": 1.0, "in_J": 1.0, "out_E": 0.7, "out_P": 0.3}


def _bits(a):
    return (np.ascontiguousarray(a, dtype=np.float32).view(np.uint32) >> 16).astype(np.uint16)


def _case(n, seed):
    """BF16-valued network input of 9 channels and parameters whose every layer carries signal."""
    rng = np.random.default_rng(seed)
    u = np.zeros((*n, 16), dtype=np.float32)
    u[..., :9] = R.bf(torch.as_tensor(rng.normal(size=(*n, 9)).astype(np.float32))).numpy()
    p = R.init_params(seed, out_gain=1.0, res_gain=1.0)
    for l, (wo, bo, ci, co) in enumerate(R.OFFSETS):
        p[bo:bo + R.REAL_IO[l][1]] = rng.normal(0, 0.1, size=R.REAL_IO[l][1]).astype(np.float32)
    return u, p


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _passes(FO, net, u, dout):
    """Output of the inference pass, output of the training pass, parameter gradient for dout."""
    V = net.V
    du = FO.Dev(2 * 16 * V)
    du.upload(_bits(u))
    net.forward(du.ptr, train=False)
    o_inf = net.out.download(np.float32)
    net.forward(du.ptr, train=True)
    o = net.out.download(np.float32)
    net.dout.upload(_bits(dout))
    net.grad.zero()
    FO._chk(FO.nop_lib().ipic_nop_backward(net.n3, du.ptr, net.wb.ptr, net.params.ptr, net.ws.ptr, net.dout.ptr,
                                           net.grad.ptr, net.stream))
    net.sync()
    return o_inf, o, net.grad.download(np.float32)


@pytest.mark.parametrize("n", [(4, 4, 16), (12, 20, 48)], ids=["one brick", "45 bricks"])
def test_gradient_of_a_small_grid_matches_reference(n):
    from allscale_ipic3d_amd import field_operator as FO
    u, p = _case(n, 5)
    V = n[0] * n[1] * n[2]
    rng = np.random.default_rng(6)
    dout = np.zeros((V, 16), dtype=np.float32)
    dout[:, :6] = R.bf(torch.as_tensor(rng.normal(size=(V, 6)).astype(np.float32))).numpy()
    net = FO.Network(n, SCALES, params=p, train=True)
    o_inf, o, g = _passes(FO, net, u, dout)
    np.testing.assert_array_equal(o_inf, o)

    pt = torch.tensor(p.astype(np.float64), requires_grad=True)
    W = []
    for wo, bo, ci, co in R.OFFSETS:
        W.append((R.bf(pt[wo:bo].reshape(3, 3, 3, co, ci).permute(3, 4, 0, 1, 2)), pt[bo:bo + co]))
    ref = R.forward(None, u.reshape(V, 16).astype(np.float64), n, bf16=True, bf16_grads=True, weights=W)
    (R.from_grid(ref) * torch.as_tensor(dout.astype(np.float64))).sum().backward()
    gr = pt.grad.numpy()
    # the bounds of the other gradient test: BF16 values near a rounding tie go either way
    assert _rel(o.reshape(V, 16), R.from_grid(ref).detach().numpy()) < 6e-3
    for l, (wo, bo, ci, co) in enumerate(R.OFFSETS):
        assert _rel(g[wo:bo], gr[wo:bo]) < 3e-2 and _rel(g[bo:bo + co], gr[bo:bo + co]) < 3e-2, l


def test_shifted_inputs_give_the_same_gradient_over_many_bricks():
    from allscale_ipic3d_amd import field_operator as FO
    n = (36, 32, 80)  # 360 bricks: some blocks take two, and the blocks do not divide among the XCDs
    u, p = _case(n, 8)
    rng = np.random.default_rng(9)
    dout = np.zeros((*n, 16), dtype=np.float32)
    dout[2, 1, 3, :6] = 1.0
    dout[..., :6] += R.bf(torch.as_tensor(rng.normal(size=(*n, 6)).astype(np.float32))).numpy() * \
        (rng.random((*n, 1)) < 1e-4)
    dout = R.bf(torch.as_tensor(dout)).numpy()
    net = FO.Network(n, SCALES, params=p, train=True)
    o_inf, o0, g0 = _passes(FO, net, u, dout)
    np.testing.assert_array_equal(o_inf, o0)
    for shift in ((1, 0, 0), (0, 3, 0), (0, 0, 7), (35, 31, 79), (18, 5, 33)):
        s_inf, o, g = _passes(FO, net, np.roll(u, shift, (0, 1, 2)), np.roll(dout, shift, (0, 1, 2)))
        # every voxel's sums have a fixed order, so the outputs are the same bits
        np.testing.assert_array_equal(o, s_inf)
        np.testing.assert_array_equal(o.reshape(*n, 16), np.roll(o0.reshape(*n, 16), shift, (0, 1, 2)))
        # the gradient sums over the voxels in another order: FP32 rounding, below 1e-5 of each
        # layer's norm
        for wo, bo, ci, co in R.OFFSETS:
            assert _rel(g[wo:bo + co], g0[wo:bo + co]) < 1e-5
