"""GPU parity of the fused attention at every head dimension class: on both
sides of the padded widths and of the step counts that they run (48 and 80),
multiples of 8 (float4 loads, the last chunk of a padded row past the head) and
others (element loads), causal or not, both output types; the bar of
test_gpu_attention.py, and a bf16 output equal to the rounded fp32 one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [8, 33, 40, 45, 48, 49, 56, 64, 65, 72, 80, 81, 88, 96, 120, 127, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_head_dimensions(be, orc, d, causal):
    import sdhip
    from oracle import f32_to_bf16

    N, Sq, Skv, heads, kvh = 2, 131, 200, 4, 2
    q, k, v = (orc.randn(s, 7700 + d + i) for i, s in enumerate(((N, Sq, heads * d), (N, Skv, kvh * d), (N, Skv, kvh * d))))
    dq, dk, dv, out = be.array(q), be.array(k), be.array(v), be.empty((N, Sq, heads * d))
    be.attention(dq, dk, dv, out, N, Sq, Skv, heads, kvh, d, causal)
    got = out.download()
    assert float(np.max(np.abs(got - orc.attention(q, k, v, heads, causal, kvh)))) <= 1e-4
    o16 = sdhip.DArray(be, (N, Sq, heads * d), dtype=np.uint16)
    be.attention_bf16(dq, dk, dv, o16, N, Sq, Skv, heads, kvh, d, causal)
    assert np.array_equal(o16.download().ravel(), f32_to_bf16(got).ravel())
