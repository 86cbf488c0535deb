"""GPU checks of the operator's training pass in convolution bricks of 1 to 5 rows (forward with saved
activations, data gradients with the silu' factors and the residual stream): the inference and the
training output in the same bits, the gradient against the torch reference, and the same
gradient for inputs rolled along the rows, which moves every row through every place in a brick."""
import numpy as np
import pytest
import torch

from oracle import nop_ref as R
from tests.test_nop_bricks_gpu import SCALES, _case, _passes, _rel

pytestmark = pytest.mark.gpu


def _rows(n, cus):
    """Rows of a brick that the launcher takes: the least rounds of bricks, times rows and two."""
    planes = n[0] // 4 * (n[2] // 16)
    cost = {r: -(-planes * -(-n[1] // r) // (2 * cus)) * (r + 2) for r in (4, 5, 3, 2, 1)}
    return min(cost, key=cost.get)


@pytest.mark.parametrize("rows, n", [(1, (28, 24, 48)), (2, (32, 28, 64)), (3, (40, 40, 48)), (4, (48, 48, 48)),
                                     (5, (44, 52, 64)), (1, (4, 4, 16))],
                         ids=["1 row", "2", "3, last 1", "4", "5, last 2", "smallest"])
def test_training_pass_in_bricks_of_rows(rows, n):
    import allscale_ipic3d_amd as G
    from allscale_ipic3d_amd import field_operator as FO
    if G.device_info()["cu_count"] != 256:
        pytest.skip("the grids are chosen for the rows that 256 CUs take")
    assert _rows(n, 256) == rows
    u, p = _case(n, 21)
    V = n[0] * n[1] * n[2]
    rng = np.random.default_rng(22)
    dout = np.zeros((*n, 16), dtype=np.float32)
    dout[..., :6] = R.bf(torch.as_tensor(rng.normal(size=(*n, 6)).astype(np.float32))).numpy()
    net = FO.Network(n, SCALES, params=p, train=True)
    o_inf, o, g = _passes(FO, net, u, dout)
    np.testing.assert_array_equal(o_inf, o)

    pt = torch.tensor(p, requires_grad=True)
    W = []
    for wo, bo, ci, co in R.OFFSETS:
        W.append((R.bf(pt[wo:bo].reshape(3, 3, 3, co, ci).permute(3, 4, 0, 1, 2)), pt[bo:bo + co]))
    ref = R.forward(None, u.reshape(V, 16), n, dtype=torch.float32, bf16_grads=True, weights=W)
    (R.from_grid(ref) * torch.as_tensor(dout.reshape(V, 16))).sum().backward()
    gr = pt.grad.numpy()
    # the bounds of the other gradient tests: BF16 values near a rounding tie go either way
    assert _rel(o.reshape(V, 16), R.from_grid(ref).detach().numpy()) < 6e-3
    for l, (wo, bo, ci, co) in enumerate(R.OFFSETS):
        assert _rel(g[wo:bo], gr[wo:bo]) < 3e-2 and _rel(g[bo:bo + co], gr[bo:bo + co]) < 3e-2, l

    for shift in (1, 2, 3):
        _, os, gs = _passes(FO, net, np.roll(u, shift, 1), np.roll(dout, shift, 1))
        np.testing.assert_array_equal(os.reshape(*n, 16), np.roll(o.reshape(*n, 16), shift, 1))
        # the sums over the voxels in another order: FP32 rounding, below 1e-5 of each layer's norm
        for wo, bo, ci, co in R.OFFSETS:
            assert _rel(gs[wo:bo + co], g[wo:bo + co]) < 1e-5
