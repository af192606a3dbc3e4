"""The loss bound of tests/test_rows_gpu.py sees a block's partial sum that is left out."""
import numpy as np
import pytest

from tests.conftest import rng
from tests.test_rows_gpu import loss_bound


# (rows, columns, rows that a block takes at once)
@pytest.mark.parametrize("batch,classes,per_block", [(17000, 66, 4), (70000, 3, 64), (4500, 10, 64),
                                                     (2100, 1000, 4)])
def test_a_missing_block_exceeds_the_bound(batch, classes, per_block):
    g = rng(batch * 7 + classes)
    z = (g.standard_normal((batch, classes)) * 3).astype(np.float32)
    lab = g.integers(0, classes, batch).astype(np.int64)
    lab[::5] = -1
    shares, tol = loss_bound(z, lab)
    whole = len(shares) // per_block * per_block
    blocks = shares[:whole].reshape(-1, per_block).sum(1) / batch
    # (a block of rows that the network gets right adds next to nothing)
    assert np.mean(blocks > 2 * tol) > 0.99, (np.sort(blocks)[:5], tol)
    assert tol < 2e-5 * shares.sum() / batch
