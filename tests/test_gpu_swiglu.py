"""GPU tests of sdh_linear_swiglu's routes (k_gemm.hip) against the float64 oracle,
within the summation bound of the two products carried through SwiGLU: the one
launch (one tile and a full round of them, one row and a partial band, column
remainders) and both sides of the limits to the library's GEMMs."""
import numpy as np
import pytest

from test_gpu_gemm import _swiglu_bound

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,H,K", [
    (1, 64, 64), (300, 514, 256), (257, 8192, 128), (256, 16384, 64),  # one launch, up to a full round
    (257, 8196, 128), (1, 16388, 64),                                  # one column of tiles more: library
    (65, 130, 1024), (65, 132, 1024), (65, 132, 1088), (65, 130, 1088),  # either side of the limit on K
])
def test_linear_swiglu_routes(be, orc, M, H, K):
    from oracle import f32_to_bf16

    x = orc.randn((M, K), 8100 + M)
    w1 = f32_to_bf16(orc.randn((H, K), 8200 + H, 0.0, 1.0 / np.sqrt(K))).reshape(H, K)
    w3 = f32_to_bf16(orc.randn((H, K), 8300 + K, 0.0, 1.0 / np.sqrt(K))).reshape(H, K)
    guard = be.array(np.full((M * H + 64,), 7.0, np.float32))
    be.linear_swiglu(be.array(x), be.array(w1), be.array(w3), guard, M, K, H)
    got = guard.download()
    assert np.all(got[M * H:] == 7.0)
    _, g, u, sg, su = orc.linear_swiglu(x, w1, w3)
    bound, want = _swiglu_bound(g, u, sg, su, K + 1)
    err = np.abs(got[:M * H].reshape(M, H).astype(np.float64) - want)
    assert np.all(err <= bound + 1e-30), f"linear_swiglu {M}x{H}x{K}: {float(np.max(err / (bound + 1e-30))):.2f} x bound"
