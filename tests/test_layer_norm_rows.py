"""LayerNorm at the edges of the pieces that a wavefront keeps of a row, few rows and many."""
import numpy as np
import pytest

from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("cols", [4, 252, 512, 516, 768, 772, 1021, 1024, 1028, 2048, 2052])
@pytest.mark.parametrize("rows", [1, 3, 1025])
def test_layer_norm_row_lengths(gpu_lib, rows, cols):
    print("layer_norm", rows, cols, flush=True)
    a, b = synth.normal_f32(61, (rows, cols)), synth.normal_f32(62, (rows, cols)) + f32(0.5)
    scale, bias = synth.normal_f32(63, (cols,)), synth.normal_f32(64, (cols,))
    x = (a + b).astype(np.float64)
    d = x - x.mean(1, keepdims=True)
    exp = d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5) * scale + bias
    got, q = H.add_layer_norm(a, b, scale, bias, q_scale=0.02, q_zp=3)
    np.testing.assert_allclose(got, exp, rtol=1e-5, atol=1e-5)
    assert np.array_equal(q, H.quantize(got, f32(0.02), 3, "i8"))
    plain, _, _ = H.layer_norm(a + b, keep_stats=False)
    np.testing.assert_allclose(plain, d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5), rtol=1e-5, atol=1e-5)
