"""GPU tests of the U-Net's weight gradients at the edges of their layout: rows
padded to 8 elements and copied 128 elements at a time, the reduction over 32-element
chunks split over waves and workgroups (4 and more chunks per wave). Against
the CPU oracle, with test_gpu_unet.py's tolerances (set before the first
run): the operands are the same BF16 values there and the sums in float64."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_unet import B, GRAD_RTOL, U, rel_l2, sample  # noqa: E402

pytestmark = pytest.mark.gpu


# the smallest grid (coarsest level one voxel), rows over half a copied run and
# just over a whole one, grids with three different sides, and one whose waves
# take more than four chunks
@pytest.mark.parametrize("shape", [(3, 4, 4, 4), (1, 4, 8, 68), (1, 4, 8, 132), (2, 12, 4, 20), (1, 20, 12, 8), (2, 32, 32, 32)])
def test_gradients_at_layout_edges(shape):
    print(f"[unet] gradients {shape}", flush=True)
    net = B.Net(seed=13)
    x, t = sample(4, shape)
    loss = net.train_step(x, t, update=False)
    g = net.grads()
    lo, go, _ = U.backward(net.params().astype(np.float64), x, t, quant=True)
    assert abs(loss - lo) <= 1e-2 * abs(lo)
    off, _ = U.offsets()
    for a, b, name in zip(off, list(off[1:]) + [len(go)], list(U.NAMES) + ["head"]):
        e = rel_l2(g[a:b], go[a:b])
        print(f"[unet] grad {name} rel L2 {e:.2e}", flush=True)
        assert e <= GRAD_RTOL, name
    # no atomics: a second pass gives the same bits
    net.train_step(x, t, update=False)
    assert np.array_equal(g, net.grads())
