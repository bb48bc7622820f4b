"""The training kernel (loss and gradients in one launch) at the edges of its tiling: 16-row tiles,
32 rows per workgroup, and one row past what 256 workgroups take in a single trip."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp as mlp_oracle  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 31, 33, 256 * 32 + 1])
def test_loss_and_gradients_match_oracle(m):
    """Tolerances: products agree to FP32 rounding except where an activation within 1e-7 of a
    BF16 midpoint rounds the other way (about 2 % of rows have one such element of 384); a flip
    moves one of a dot product's 128 terms by 2^-8, so the loss by less than 1e-3 and a gradient
    by less than 1e-2 in L2 even if every row had one."""
    import assist_amd.learned as L
    from assist_amd.batch import DeviceArray
    rng = np.random.default_rng(100 + m)
    net = L.StepModel(max_batch=m, seed=2)
    p = rng.normal(0, 0.2, L.num_params()).astype(np.float32)
    w = np.linspace(0.2, 1.0, 32).astype(np.float32)
    net.set_params(p)
    net.set_output_weights(w)
    X, T = (rng.normal(0, 1, (m, k)).astype(np.float32) for k in (16, 32))
    d_X, d_T = DeviceArray(X), DeviceArray(T)
    loss, g = net.loss_grad(d_X, d_T, m, want_grad=True)
    ref_loss, ref_g = mlp_oracle.loss_grad(p, X, T, w, bf16_ops=True)
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
    assert np.linalg.norm(g - ref_g) <= 1e-2 * np.linalg.norm(ref_g)
    again = net.loss_grad(d_X, d_T, m, want_grad=True)
    assert again[0] == loss
    np.testing.assert_array_equal(again[1], g)  # fixed summation order
