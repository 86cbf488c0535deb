"""GPU checks of the operator's convolutions in bricks of 1 to 5 rows, the last brick of a column shorter
where the rows do not divide the side: the output against the torch CPU reference, and the same bits for
inputs rolled along the rows, which moves every row through every place in a brick."""
import numpy as np
import pytest
import torch

from oracle import nop_ref as R
from tests.test_nop_bricks_gpu import SCALES, _bits, _case, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(28, 24, 48), (32, 28, 64), (40, 40, 48), (48, 48, 48), (44, 52, 64), (4, 4, 16)],
                         ids=["1 row", "2", "3, last 1", "4", "5, last 2", "smallest"])
def test_bricks_of_rows(n):
    from allscale_ipic3d_amd import field_operator as FO
    u, p = _case(n, 11)
    V = n[0] * n[1] * n[2]
    net = FO.Network(n, SCALES, params=p, train=True)

    def out(v):
        du = FO.Dev(2 * 16 * V)
        du.upload(_bits(v))
        net.forward(du.ptr, train=False)
        return net.out.download(np.float32).reshape(*n, 16)

    o = out(u)
    ref = R.from_grid(R.forward(p, u.reshape(V, 16).astype(np.float32), n, dtype=torch.float32)).detach().numpy()
    # the bound of the other output test: BF16 values near a rounding tie go either way
    assert _rel(o.reshape(V, 16), ref) < 6e-3
    for shift in (1, 2, 3):
        np.testing.assert_array_equal(out(np.roll(u, shift, 1)), np.roll(o, shift, 1))
