"""SiLU where e^-z lies near the top of the single-precision range: z / (1 + e^-z)
is a normal number of about -1e-37 there, in inference, in the fused training kernels
and in the layer-by-layer ones (hidden width 64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Z = np.array([-80.0, -86.5, -87.0, -87.5, -88.0, -88.5, -89.0, -120.0], np.float32)   # exact in bf16
GAIN = 121   # the outputs are the activations times 2^GAIN


@pytest.mark.parametrize("hidden", (256, 64))
def test_activation_near_the_top_of_the_exponential(hidden):
    from geliosphere_amd.surrogate import Surrogate
    s = Surrogate(0, n_members=1, n_hidden_layers=1, n_inputs=1, hidden=hidden, batch=64)
    s.set_normalization([0.0], [1.0], [-1e3], [1e3])
    pm, ((w0, _, _, n_in), (w1, _, _, n_hid)) = s.layout()
    p = np.zeros(pm, np.float32)
    p[w0] = 1.0            # unit 0: z = x
    p[w1] = 2.0 ** GAIN    # output 0: unit 0
    s.set_params(p)
    mean = s.predict(Z[:, None])[0][:, 0].astype(np.float64)
    z = Z.astype(np.float64)
    want = z / (1.0 + np.exp(-z)) * 2.0 ** GAIN
    want[z < -88.73] = 0.0   # e^-z beyond single precision
    # bf16 rounding 2^-9, e^-z to 2^-17
    assert np.all(np.abs(mean - want) <= 2.0 ** -8 * np.abs(want)), (mean, want)
    # the training kernels' forward pass: no loss on these outputs
    y = np.zeros((len(z), 30), np.float32)
    y[:, 0] = mean
    assert s.gradients(Z[:, None], y, np.ones_like(y))[1][0] == 0.0
