"""GPU kernels at the edges of the sizes they serve (tile and wave remainders,
the smallest and largest of a range), against the CPU oracle.

Tolerance of a training step: rel 1e-4 / abs 1e-5 per element after a few SGD
steps, as the parity tests state it for fp32.
"""
import numpy as np
import pytest

from tests.oracle_lib import load_oracle
from tests.test_gpu_parity import assert_params_close, close_enough, run_steps, say
from volta_amd import DeviceArray, data, load_hip
from volta_amd.abi import STATUS_BAD_ARGUMENT, STATUS_NONFINITE_LOSS, MlpSpec, Trainer

pytestmark = pytest.mark.gpu


def against_oracle(spec, B, lr=0.01, steps=3, seed=7):
    """Losses and parameters after `steps` steps on fresh batches, HIP against oracle."""
    ws, bs = data.he_uniform(seed, spec.sizes)
    batches = [data.batch(seed + 1 + s, spec.sizes, B, spec.loss) for s in range(steps)]
    lh, wh, bh, st = run_steps(load_hip(), spec, B, ws, bs, batches, lr, steps)
    lo, wo, bo, _ = run_steps(load_oracle(), spec, B, ws, bs, batches, lr, steps)
    assert st == 0, f"status {st}"
    ok, mx, _ = close_enough(lh, lo)
    assert ok, f"losses differ, max abs {mx:.3e}\n hip={lh}\n ora={lo}"
    assert_params_close(wh, bh, wo, bo, spec.text())


# Stand-alone loss heads (more than 64 outputs): one wave per row, rows of up
# to 64, 128, 256 and 1024 columns in registers and longer ones read again;
# four rows per block, several rows per wave above 4096 rows.
@pytest.mark.parametrize("loss,C,B", [("ce", c, b) for c in (65, 128, 129, 1024, 1025) for b in (1, 5)] +
                         [("ce", 100, 4099), ("ce", 257, 66), ("mse", 65, 1), ("mse", 100, 41), ("mse", 67, 4099)])
def test_wide_loss_head(loss, C, B):
    say(f"wide loss head {loss} C={C} B={B}")
    against_oracle(MlpSpec([9, 12, C], "tanh", "sgd", loss), B)


def test_wide_loss_head_special_values():
    """A label outside the classes and an infinite logit: the loss is NaN, the
    label is reported, and the other rows' gradients are what they are without it."""
    say("wide loss head special values")
    lib, C, B = load_hip(), 100, 8
    spec = MlpSpec([4, C], "relu", "sgd", "ce")
    ws, bs = data.he_uniform(1, spec.sizes)
    X, Y = data.batch(2, spec.sizes, B, "ce")
    bad = Y.copy()
    bad[3] = C
    got = []
    for y in (Y, bad):
        t = Trainer(lib, spec, B)
        t.set_all_params(ws, bs)
        dx, dy = DeviceArray(X), DeviceArray(y)
        assert t.step_device(dx.ptr, dy.ptr, 0.0) == 0
        got.append((t.debug_buffer(1, 0).reshape(B, C), t.loss(), t.status()))
        t.close()
    (d0, l0, s0), (d1, l1, s1) = got
    assert s0 == 0 and np.isfinite(l0)
    assert s1 == STATUS_BAD_ARGUMENT | STATUS_NONFINITE_LOSS and np.isnan(l1)
    np.testing.assert_array_equal(np.delete(d0, 3, 0), np.delete(d1, 3, 0))
    X[2, 0] = np.inf
    t = Trainer(lib, spec, B)
    t.set_all_params(ws, bs)
    t.step(X, Y, 0.0)
    assert np.isnan(t.loss()) and t.status() == STATUS_NONFINITE_LOSS
    np.testing.assert_array_equal(np.delete(t.debug_buffer(1, 0).reshape(B, C), 2, 0), np.delete(d0, 2, 0))
    t.close()
