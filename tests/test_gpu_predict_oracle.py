"""The prediction kernel of the learned start against the CPU oracle, on ragged row counts, fewer and more
tiles than its grid has waves, and with the shipped network; and against the training kernel, which
evaluates the network in code of its own: the loss of the predicted outputs is the loss it returns."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp as mlp_oracle  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shipped", [False, True])
@pytest.mark.parametrize("m", [1, 301, 4096, 70001])
def test_predict_matches_oracle_and_training_loss(gpu, m, shipped):
    """Tolerances: both round the same operands to BF16 and differ in FP32 rounding, so an output moves
    only where an activation lies at a BF16 midpoint and goes the other way (about 2% of rows have one of
    384).  One such element of the second layer moves an output by at most 2^-8 |W3 row| |W4 column|,
    1.5e-2 for the shipped network (row and column norms of 2), against outputs up to 2.7: 1e-2 of the
    largest output; the mean over all rows is 50 times below that.  The loss is an FP32 sum of at most
    300 terms a thread: 2e-5, and 1e-4 is asked."""
    import assist_amd.learned as L
    from assist_amd.batch import DeviceArray
    rng = np.random.default_rng(140 + m)
    if shipped:
        net = L.StepModel.load(L.default_model_path(), max_batch=m)
    else:
        net = L.StepModel(max_batch=m, seed=7)
        net.set_params(rng.normal(0, 0.2, L.num_params()).astype(np.float32))
    w = np.linspace(0.2, 1.0, 32).astype(np.float32)
    net.set_output_weights(w)
    X, T = (rng.normal(0, 1, (m, k)).astype(np.float32) for k in (16, 32))
    d_X, d_T, d_Y = DeviceArray(X), DeviceArray(T), DeviceArray(np.zeros((m, 32), np.float32))
    net.predict(d_X, m, d_Y)
    y = d_Y.download()
    ref, _ = mlp_oracle.forward(net.params(), X, bf16_ops=True)
    scale, err = np.abs(ref).max(), np.abs(y - ref)
    print("predict: max |err| / max |y| = %.3g, mean %.3g" % (err.max() / scale, err.mean() / scale))
    assert err.max() <= 1e-2 * scale and err.mean() <= 2e-4 * scale
    loss = float((w.astype(np.float64) * (y.astype(np.float64) - T) ** 2).sum() / m)
    assert abs(net.loss_grad(d_X, d_T, m) - loss) <= 1e-4 * loss
