"""The one-kernel attention at sequence lengths around the edges of its tiles, against the three ops."""
import numpy as np
import pytest

from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu
f32 = np.float32


# (lengths around 16 rows, a chunk of 128 keys and the largest; few heads and, the last five, enough for items of 32
# rows with one to four chunks)
@pytest.mark.parametrize("B,S,nh", [(2, 1, 3), (1, 15, 2), (3, 17, 4), (2, 63, 2), (1, 64, 1), (3, 64, 5), (25, 64, 12), (1, 65, 2), (24, 100, 12), (2, 127, 3), (9, 129, 8), (1, 197, 4), (2, 256, 1), (8, 257, 12), (1, 385, 2),
                                    (1, 509, 3), (25, 96, 12), (25, 128, 12), (10, 256, 12), (12, 384, 8), (16, 512, 4)])
def test_attention_of_any_length_equals_the_three_ops(gpu_lib, B, S, nh):
    print("attention", B, S, nh, flush=True)
    hd = 64
    h = nh * hd
    qkv = synth.normal_f32(52, (B * S, 3 * h)) * f32(1.5)
    v_scores = H.MatmulView(nh, S * 3 * h, hd, 3 * h, S * 3 * h, hd, 3 * h, nh * S * S, S * S, S)
    v_ctx = H.MatmulView(nh, nh * S * S, S * S, S, S * 3 * h, hd, 3 * h, S * h, hd, h)
    v_att = H.AttentionView(nh, S * 3 * h, hd, 3 * h, S * 3 * h, hd, 3 * h, S * 3 * h, hd, 3 * h, S * h, hd, h)
    scores, _ = H.batch_matmul_view(qkv, 0, qkv, h, B * nh * S * S, 0, v_scores, B * nh, S, hd, S, False, True)
    probs = H.softmax_scaled(scores.reshape(B * nh * S, S), 0.125)
    s_c = 0.4 / 127.0
    exp, exp_q = H.batch_matmul_view(probs, 0, qkv, 2 * h, B * S * h, 0, v_ctx, B * nh, S, S, hd, False, False, q_scale=s_c)
    got, q = H.attention(qkv, 0, h, 2 * h, B * S * h, v_att, B * nh, S, S, hd, factor=0.125, q_scale=s_c)
    assert H.last_kernel() == "attention_f32"
    assert np.array_equal(got.view(np.uint32), exp.view(np.uint32))
    assert np.array_equal(q, exp_q)


@pytest.mark.parametrize("cols", [1, 3, 31, 33, 63, 65, 127, 130, 255, 257, 381, 385, 511, 513, 1022, 1025, 2048, 2051])
def test_softmax_row_lengths(gpu_lib, cols):
    """every split of a row over lanes and pieces, aligned or not, against the same sums in f64"""
    x = synth.normal_f32(53, (37, cols)) * f32(3.0)
    e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    np.testing.assert_allclose(H.softmax(x, (1,)), e / e.sum(1, keepdims=True), rtol=2e-6, atol=1e-12)
