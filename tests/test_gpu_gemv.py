"""GPU tests of the linear layers of a few rows (k_gemv.hip), fp32 and bf16
weights, against the float64 oracle within the rigorous fp32 summation bound:
every row count, sizes on both sides of the rules for columns per wave and for
cutting K, remainders of a wave's turn, unaligned rows, bias, accumulation."""
import numpy as np
import pytest

from tolerances import assert_gemm

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 7), (5, 256), (257, 260), (1024, 256), (1885, 650), (63, 1023), (70, 1024), (300, 2056), (2049, 1028),
         (4097, 96), (4099, 1288)]


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", SIZES)
def test_few_rows(be, orc, M, N, K):
    from oracle import f32_to_bf16

    lda = K + (4 if K % 8 == 0 else 3)
    A, W = orc.randn((M, lda), 6000 + K), orc.randn((N, K), 6001 + N, 0.0, 1.0 / np.sqrt(K))
    b, c0 = orc.randn((N,), 6002), orc.randn((M, N), 6003)
    dA, db = be.array(A), be.array(b)
    more = {True: np.abs(c0), False: np.abs(b)}  # the bound's sum is over every term, C or bias among them
    for acc in (False, True):
        dC = be.array(c0) if acc else be.empty((M, N))
        be.gemm_nt_f32(M, N, K, dA, lda, be.array(W), K, dC, N, None if acc else db, acc)
        want, S = orc.gemm_nt_f32(A[:, :K], W, None if acc else b, c0 if acc else None, acc)
        assert_gemm(dC.download(), want, S + more[acc], K + 2, f"fp32 {M}x{N}x{K} acc={acc}")
        W16 = f32_to_bf16(W).reshape(N, K)
        dC = be.array(c0) if acc else be.empty((M, N))
        be.gemm_nt_bf16(M, N, K, dA, lda, be.array(W16), K, dC, N, None if acc else db, acc)
        want, S = orc.gemm_nt_bf16(A[:, :K], W16, None if acc else b, c0 if acc else None, acc)
        assert_gemm(dC.download(), want, S + more[acc], K + 2, f"bf16 {M}x{N}x{K} acc={acc}")


@pytest.mark.parametrize("M", [1, 3, 8, 9])
@pytest.mark.parametrize("N,lda", [(256, 256), (1024, 1024), (4104, 4104), (512, 520)])
def test_bf16_rows_in_place(be, orc, M, N, lda):
    """C on A: every value of A is read (and rounded) before C is stored. C
    within A's rows (lda > N) too, with and without accumulation."""
    from oracle import f32_to_bf16

    A = orc.randn((M, lda), 6100 + N)
    W16 = f32_to_bf16(orc.randn((N, N), 6101 + N, 0.0, 1.0 / np.sqrt(N))).reshape(N, N)
    dW = be.array(W16)
    for acc in (False, True):
        dA = be.array(A)
        be.gemm_nt_bf16(M, N, N, dA, lda, dW, N, dA, lda, None, acc)
        want, S = orc.gemm_nt_bf16(A[:, :N], W16, None, A[:, :N] if acc else None, acc)
        got = dA.download()
        assert_gemm(got[:, :N], want, S + np.abs(A[:, :N]), N + 2, f"in place {M}x{N} acc={acc}")
        assert np.array_equal(got[:, N:], A[:, N:])
