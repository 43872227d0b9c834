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


@pytest.mark.parametrize("N,Sq,Skv,heads,kvh,d,causal", [
    (1, 2048, 2048, 2, 2, 128, False),  # 32 tiles over four waves, one round
    (1, 1990, 1990, 8, 4, 40, True),    # two rounds, some waves without a tile
    (2, 33, 1601, 3, 1, 64, False), (1, 40, 129, 5, 5, 80, True), (1, 1, 190, 2, 2, 128, False),
    (1, 256, 100, 30, 30, 128, False),  # on both sides of one round
    (1, 288, 100, 30, 30, 128, False),
])
@pytest.mark.parametrize("fp16", [False, True])
def test_few_queries(be, orc, N, Sq, Skv, heads, kvh, d, causal, fp16):
    """The form whose waves share a head's key tiles, and its neighbours; values
    from one key tile far above the others, so that the waves' references differ."""
    q, k, v = (orc.randn(s, 7900 + d + i) for i, s in enumerate(((N, Sq, heads * d), (N, Skv, kvh * d), (N, Skv, kvh * d))))
    k[:, 64:128] *= 3
    out = be.empty((N, Sq, heads * d))
    call = be.attention_fp16 if fp16 else be.attention
    call(be.array(q), be.array(k), be.array(v), out, N, Sq, Skv, heads, kvh, d, causal)
    rows = np.unique(np.concatenate([np.arange(0, Sq, max(1, Sq // 60)), [Sq - 1]]))
    want = orc.attention(q, k, v, heads, causal, kvh, rows=rows)
    # fp16 operands: scores of spread 3 sqrt(d) with 2^-11 relative operands move a weight by about
    # 2^-10 of the score, at most 12 here
    assert float(np.max(np.abs(out.download()[:, rows] - want))) <= (0.05 if fp16 else 1e-4)
