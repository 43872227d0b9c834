// k_gemv.hip - linear layers of a few rows (M <= 8): the timestep MLP, the adaLN
// modulations and the UNet's time projections, whose one or two rows meet each
// weight once. C[M,N] = A[M,K] B[N,K]^T (+ C) (+ bias[N]) with fp32 or bf16 B
// (backend_cuda.h:38-43), fp32 FMAs on the vector ALUs; with bf16 weights A is
// rounded to bf16 first, as gemm_nt_bf16 does.
//
// Bound by launch and by the weights' bytes: no tile of a GEMM has M rows to
// share them. A wave takes one weight row, 16 bytes per lane and load, four
// loads in flight, keeps M sums per lane and adds them over the lanes at the
// end; four rows per wave above N = 4096, where there are waves enough and A is
// then read from the caches a quarter as often. Long rows (K >= 1024) of large
// layers are cut over the four waves of a workgroup, four columns each: A is
// read a quarter as often again. Measured on MI355X, us per call queued back to
// back (the host's 4 us per call is the floor; the library's plan look-up and
// launch take 10), library / one wave per row / cut: fp32 [1,256] x [1024,256]
// 10.5 / 4.2 / 4.7, [2,1280] x [5120,1280] 10.8 / 5.4 / 4.5, [8,1280] x [1280,1280]
// 10.9 / 6.5 / 5.9, [8,4096] x [4096,4096] 13.5 / 35.6 / 17.9, [8,650] x [1885,650] (rows not
// a multiple of 16 bytes) 48 / 4.8 / 5.7; bf16 [1,256] x [15360,256] 13.4 / 4.4 / 4.9,
// [1,3840] x [3840,3840] 13.7 / 12.9 / 6.8.
#include "sdh_internal.hpp"

namespace sdh {
namespace {

using dev::f4;
typedef unsigned short u16;
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

constexpr int kWaves = 4;

__device__ __forceinline__ float bf16_value(u16 b) { return __uint_as_float((unsigned)b << 16); }

// VE consecutive values of a row of A or B from k on.
template <int VE, bool VEC>
__device__ __forceinline__ void take(const float* p, float* v) {
    if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < VE; i += 4) {
            const f4 x = *(const f4*)(p + i);
            v[i] = x.x; v[i + 1] = x.y; v[i + 2] = x.z; v[i + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < VE; ++i) v[i] = p[i];
    }
}
template <int VE, bool VEC>
__device__ __forceinline__ void take(const u16* p, float* v) {
    if constexpr (VEC) {
        const us8 x = __builtin_nontemporal_load((const us8*)p);
#pragma unroll
        for (int i = 0; i < VE; ++i) v[i] = bf16_value(x[i]);
    } else {
#pragma unroll
        for (int i = 0; i < VE; ++i) v[i] = bf16_value(p[i]);
    }
}

// B: float or u16 (bf16). VEC: K a multiple of VE, rows 16-byte aligned; else
// VE = 1. Rows past m repeat the last one.
template <class B, int M, int COLS, int PARTS, bool VEC>
__global__ __launch_bounds__(64 * kWaves) void k_gemv(const float* __restrict__ A, int64_t lda,
                                                     const B* __restrict__ W, int64_t ldb, float* __restrict__ C,
                                                     int64_t ldc, const float* __restrict__ bias, int m, int64_t N,
                                                     int K, int accumulate) {
    constexpr bool BF = sizeof(B) == 2;
    constexpr int VE = !VEC ? 1 : BF ? 8 : 4, TURN = 64 * VE;
    __shared__ float sums[PARTS > 1 ? kWaves : 1][PARTS > 1 ? M * COLS : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n0 = ((int64_t)blockIdx.x * (kWaves / PARTS) + (PARTS > 1 ? 0 : wave)) * COLS;
    if (n0 >= N) return;  // a whole wave; with PARTS the whole workgroup
    const B* w[COLS];
    const float* a[M];
#pragma unroll
    for (int c = 0; c < COLS; ++c) w[c] = W + (n0 + c < N ? n0 + c : N - 1) * ldb;
#pragma unroll
    for (int i = 0; i < M; ++i) a[i] = A + (int64_t)min(i, m - 1) * lda;
    float acc[M][COLS];
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) acc[i][c] = 0.f;
    auto turn = [&](int k) __attribute__((always_inline)) {
        float b[COLS][VE];
#pragma unroll
        for (int c = 0; c < COLS; ++c) take<VE, VEC>(w[c] + k, b[c]);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            float x[VE];
            take<VE, VEC>(a[i] + k, x);
#pragma unroll
            for (int e = 0; e < VE; ++e) {
                const float v = BF ? bf16_value(dev::bf16_rne(x[e])) : x[e];
#pragma unroll
                for (int c = 0; c < COLS; ++c) acc[i][c] = fmaf(v, b[c][e], acc[i][c]);
            }
        }
    };
    constexpr int STEP = TURN * PARTS;  // with PARTS the waves take turns along K
    int k = (PARTS > 1 ? wave * TURN : 0) + lane * VE;
    for (; k + 3 * STEP < K; k += 4 * STEP) {
#pragma unroll
        for (int u = 0; u < 4; ++u) turn(k + u * STEP);
    }
    for (; k < K; k += STEP) turn(k);
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < M; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const float s = dev::wave_sum(acc[i][c]);
            if (lane == i * COLS + c) v = s;
        }
    if constexpr (PARTS > 1) {
        if (lane < M * COLS) sums[wave][lane] = v;
        __syncthreads();
        if (wave) return;
        v = 0.f;
        if (lane < M * COLS) v = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
    }
    const int i = lane / COLS;
    const int64_t n = n0 + lane % COLS;
    if (i < m && i < M && n < N) {
        float* p = C + i * ldc + n;
        if (accumulate) v += *p;
        if (bias) v += bias[n];
        *p = v;
    }
}

template <class B, int M>
void launch(const float* A, int64_t lda, const B* W, int64_t ldb, float* C, int64_t ldc, const float* bias, int m,
            int64_t N, int K, bool accumulate) {
    constexpr int VE = sizeof(B) == 2 ? 8 : 4;
    const bool vec = K % VE == 0 && ldb % VE == 0 && lda % 4 == 0 && aligned16(A) && aligned16(W);
    const int parts = K >= 1024 && (M * K > 4096 || N > 2048) ? 4 : 1, cols = parts > 1 || N > 4096 ? 4 : 1;
    auto go = parts == 4   ? (vec ? k_gemv<B, M, 4, 4, true> : k_gemv<B, M, 4, 4, false>)
              : cols == 4 ? (vec ? k_gemv<B, M, 4, 1, true> : k_gemv<B, M, 4, 1, false>)
                          : (vec ? k_gemv<B, M, 1, 1, true> : k_gemv<B, M, 1, 1, false>);
    go<<<blocks_for(N, kWaves / parts * cols), 64 * kWaves, 0, stream()>>>(A, lda, W, ldb, C, ldc, bias, m, N, K,
                                                                  accumulate ? 1 : 0);
}

template <class B>
bool run(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const B* W, int64_t ldb, float* C, int64_t ldc,
         const float* bias, bool accumulate) {
    // the library's tiles take large layers of five to eight rows (see above), and very large
    // bf16 ones of three or four ([4,1024] x [151936,1024] 58 us there, 106 here; [4,11008] x
    // [4096,11008] 23 and 28; [4,4096] x [4096,4096] still gains)
    if (M > 8 || (M > 4 && N * K > (int64_t(1) << 22)) || (M > 2 && sizeof(B) == 2 && N * K > (int64_t(1) << 25)) || K >= (1 << 30) || N * 64 >= kMaxGridItems) return false;
    const int m = (int)M;
    if (m == 1) launch<B, 1>(A, lda, W, ldb, C, ldc, bias, m, N, (int)K, accumulate);
    else if (m == 2) launch<B, 2>(A, lda, W, ldb, C, ldc, bias, m, N, (int)K, accumulate);
    else if (m <= 4) launch<B, 4>(A, lda, W, ldb, C, ldc, bias, m, N, (int)K, accumulate);
    else launch<B, 8>(A, lda, W, ldb, C, ldc, bias, m, N, (int)K, accumulate);
    return true;
}

}  // namespace

bool gemv_f32(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
              int64_t ldc, const float* bias, bool accumulate) {
    return run<float>(M, N, K, A, lda, B, ldb, C, ldc, bias, accumulate);
}
bool gemv_bf16(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const uint16_t* B, int64_t ldb, float* C,
               int64_t ldc, const float* bias, bool accumulate) {
    return run<u16>(M, N, K, A, lda, (const u16*)B, ldb, C, ldc, bias, accumulate);
}

}  // namespace sdh
