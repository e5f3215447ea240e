"""Quantize and Dequantize where a group of four elements reaches into the next row of the scale table."""
import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


# (outer, scales, inner): rows of 1, 2, 3, just above 4, around a workgroup's step of 1024 elements, the count's remainders
@pytest.mark.parametrize("shape", [(1, 7, 1), (3, 5, 2), (2, 9, 3), (5, 3, 5), (4, 6, 7), (3, 2, 1023), (2, 3, 1025), (1, 4, 1026), (3, 1, 1027), (2, 2, 5003), (1, 1, 3), (7, 11, 238), (1, 3, 12345)])
def test_quantize_rows_of_any_length(gpu_lib, shape):
    print("quantize ragged", shape, flush=True)
    x = synth.normal_f32(71, shape) * np.float32(20)
    scale = synth.uniform_f32(72, (shape[1],), 0.05, 1.5)
    for qt, mode in (("i8", H.RNE), ("u8", H.RNE), ("i8", 0)):
        zp = synth.uniform_int(73, (shape[1],), 0, 40, H.NP_OF[H.dtype_code(qt)])
        got, exp = H.quantize(x, scale, zp, qt, (1,), mode), O.quantize(x, scale, zp, qt, (1,), mode)
        assert np.array_equal(got, exp)
        assert H.last_kernel() == "quantize_ragged"
        dq = H.dequantize(got, scale, zp, "f32", (1,))
        assert H.last_kernel() == "dequantize_ragged"
        assert np.array_equal(dq, O.dequantize(exp, scale, zp, "f32", (1,)))


# (more than eight steps a compute unit, where a lane takes several groups: rows of whole steps, of whole groups, of
# one step and more, of some groups, of less than one; the last step and the last group partly filled)
@pytest.mark.parametrize("shape,kernel", [((2, 261, 4096), "vec4"), ((3, 85, 8228), "vec4"), ((2, 1043, 1027), "ragged"), ((200, 1543, 7), "ragged"), ((401, 1807, 3), "ragged")])
def test_quantize_large(gpu_lib, shape, kernel):
    print("quantize large", shape, flush=True)
    x = synth.normal_f32(74, shape) * np.float32(20)
    scale = synth.uniform_f32(75, (shape[1],), 0.05, 1.5)
    for qt, mode in (("i8", H.RNE), ("u8", H.RNE), ("i8", 0), ("u8", 0)):
        zp = synth.uniform_int(76, (shape[1],), 0, 40, H.NP_OF[H.dtype_code(qt)])
        got, exp = H.quantize(x, scale, zp, qt, (1,), mode), O.quantize(x, scale, zp, qt, (1,), mode)
        assert H.last_kernel() == "quantize_" + kernel
        assert np.array_equal(got, exp)
        dq = H.dequantize(got, scale, zp, "f32", (1,))
        assert H.last_kernel() == "dequantize_" + kernel
        assert np.array_equal(dq, O.dequantize(exp, scale, zp, "f32", (1,)))
