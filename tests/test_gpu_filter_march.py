"""The 3D filter pass over every march length its launch chooses, with
remainders in all three directions, bit for bit against the oracle (strict
build: the expression is evaluated in the oracle's order without contraction)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(9, 7, 5),          # 2 planes a workgroup
                               (65, 602, 23),      # 4
                               (10, 1030, 33),     # 8
                               (10, 2101, 17)])    # 16, the last of 1
def test_filter_march(hip, oracle, n):
    from entity_amd.containers import GridShape
    from entity_amd.kernels import DigitalFilter_kernel
    shape = GridShape(3, n)
    rng = np.random.default_rng(7)
    J = rng.standard_normal(shape.tensor_shape(3)).astype(np.float32)
    oracle.communicate(J, 0, 3, dim=3)
    buf = torch.from_numpy(J.copy()).cuda()
    got = buf.clone()
    DigitalFilter_kernel(got, buf, shape, strict=True)()
    oracle.filter_pass(J, J.copy(), dim=3)
    np.testing.assert_array_equal(got.cpu().numpy(), J)
