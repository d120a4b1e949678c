"""Training batches that leave waves or workgroups without a chunk of 32 pixels, or
give some one more than others: gradient and loss against the BF16-emulating
oracle, and the same bits from run to run."""
import numpy as np
import pytest

from tests import test_gpu_mlp as T
from tests.test_gpu_mlp import M

pytestmark = pytest.mark.gpu


# 256 workgroups of 8 waves: 8,192 pixels are one chunk a workgroup, 65,536 one a wave
@pytest.mark.parametrize("n", [1, 31, 32, 33, 8191, 8193, 16385, 65535, 65537])
def test_gradient(cpt, n):
    m = cpt.Mlp(1)
    p = T._params(5)
    m.set_params(p)
    X, t = T._data(n, n)
    loss = m.train_step(X, t, apply=False)
    g = m.grad()
    l_ref, g_ref = M.loss_grad(p, X, t, exact=False)
    # three operands of a product are rounded to BF16, where the oracle may round the other way: 3 * 2^-9
    assert abs(loss - l_ref) <= 3 * 2.0 ** -9 * max(1.0, l_ref)
    assert np.linalg.norm(g - g_ref) <= 2 * 3 * 2.0 ** -9 * np.linalg.norm(g_ref)
    assert m.train_step(X, t, apply=False) == loss
    assert np.array_equal(m.grad(), g)
