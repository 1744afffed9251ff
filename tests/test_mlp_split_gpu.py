"""Weight and bias gradients of the guess network split over the batch, at the edges of the split."""
import numpy as np
import pytest

from oracle import mlp as orc
from tests.test_mlp import _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('m', [1, 63, 65, 257, 1023])
def test_gradient_of_ragged_batches(m):
    """Blocks of the gradient against the float64 oracle; the same bound as for whole batches (bf16 inputs:
    a product rounds to 2^-8, sums of m of them stay below it relative to the block's largest)."""
    from veloxchem_amd.densitynet import DensityNet
    n_in, nh, n_out, bc = 70, 128, 196, 14
    x, t, shape, params = _problem(m, n_in, nh, n_out, bc, 5)
    net = DensityNet(n_in, nh, n_out, bc, max_batch=1024)
    net.set_params(params)
    loss, g = net.loss_grad(x, t, shape, want_grad=True)
    loss_ref, g_ref, _ = orc.loss_grad(params.astype(np.float64), x, t, shape, n_in, nh, n_out, bc)
    assert abs(loss - loss_ref) < 1e-3 * loss_ref
    off = 0
    for fi, fo in [(n_in, nh), (nh, nh), (nh, n_out)]:
        for n in (fi * fo, fo):
            blk, ref = g[off:off + n], g_ref[off:off + n]
            assert np.max(np.abs(blk - ref)) / np.max(np.abs(ref)) < 2e-2
            off += n
