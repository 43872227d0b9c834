// k_gemm_f32.hip - the linear layer with fp32 weights: C[M,N] = A[M,K] * B[N,K]^T
// (+ C) (+ bias[N]) in fp32 (backend_cuda.h:38-40, gemm_nt_f32; the reference's
// device path is an fp32 SGEMM, backend_cuda.cu:453-464, its CPU path fp32
// micro-kernels, tensor.cpp:354-406): every linear of SD 1.x's UNet and text
// encoder and of the VAE, and Z-Image's weights under 2^20 elements
// (safetensors.cpp:110-116 with keep_bf16, pipeline.cpp:113). Large products run
// on split fp16 operands (k_gemm_split.hip), small ones on the library's fp32
// GEMM; what neither takes on the kernel below, a plain register-blocked fp32
// FMA kernel on the vector ALUs: 64 x 64 output tile per 256-thread workgroup,
// 4 x 4 per thread, K in steps of 16 through LDS (A and B tiles stored k-major,
// so a thread's four rows or columns are one float4 read).
//
// Also sdh_to_bf16: float32 -> bf16 bits on the device with the reference's
// rounding (nearest even; inf and NaN keep their top bits; tensor.cpp:114-121).
#include <algorithm>

#include "sdh_internal.hpp"

namespace sdh {
namespace {

using dev::f4;
constexpr int kT = 64, kKS = 16, kThreads = 256;

// VEC: K % 4 == 0, lda % 4 == 0, ldb % 4 == 0 and 16-B aligned A and B.
template <bool VEC>
__global__ __launch_bounds__(kThreads) void k_gemm_f32(const float* __restrict__ A, int64_t lda,
                                                       const float* __restrict__ B, int64_t ldb, float* __restrict__ C,
                                                       int64_t ldc, const float* __restrict__ bias, int64_t M,
                                                       int64_t N, int64_t K, int accumulate) {
    __shared__ float sA[kKS][kT + 4];
    __shared__ float sB[kKS][kT + 4];
    const int t = threadIdx.x, tx = t & 15, ty = t >> 4;
    const int64_t m0 = (int64_t)blockIdx.y * kT, n0 = (int64_t)blockIdx.x * kT;
    // loader mapping: thread t loads row (t >> 2) of the tile, k quad (t & 3)
    const int lr = t >> 2, lk = (t & 3) * 4;
    const int64_t am = m0 + lr, bn = n0 + lr;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int64_t k0 = 0; k0 < K; k0 += kKS) {
        f4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
        if constexpr (VEC) {
            if (am < M && k0 + lk < K) a = *(const f4*)(A + am * lda + k0 + lk);
            if (bn < N && k0 + lk < K) b = *(const f4*)(B + bn * ldb + k0 + lk);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t k = k0 + lk + e;
                if (am < M && k < K) a[e] = A[am * lda + k];
                if (bn < N && k < K) b[e] = B[bn * ldb + k];
            }
        }
        __syncthreads();  // every thread is done with the previous tiles
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sA[lk + e][lr] = a[e];
            sB[lk + e][lr] = b[e];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kKS; ++kk) {
            const f4 av = *(const f4*)&sA[kk][ty * 4];
            const f4 bv = *(const f4*)&sB[kk][tx * 4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float* cp = C + m * ldc + n;
            float v = acc[i][j];
            if (bias) v += bias[n];
            if (accumulate) v += *cp;
            *cp = v;
        }
    }
}

// Nearest-even float -> bf16 bits; inf and NaN keep their top 16 bits.
__device__ __forceinline__ unsigned short to_bf16_bits(float f) {
    const unsigned b = __float_as_uint(f);
    if ((b & 0x7F800000u) == 0x7F800000u) return (unsigned short)(b >> 16);
    return (unsigned short)((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}

__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ x, unsigned short* __restrict__ y,
                                                 int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) y[i] = to_bf16_bits(x[i]);
}

bool aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

void run_gemm_f32(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                  int64_t ldc, const float* bias, bool accumulate) {
    const char* op = "sdh_gemm_nt_f32";
    need(M >= 0 && N >= 0 && K >= 0, op, "negative size");
    need(lda >= K && ldb >= K && ldc >= N, op, "leading dimension smaller than the row");
    if (M == 0 || N == 0) return;
    ensure_init();
    if (K > 0) {
        check_range(A, (size_t)((M - 1) * lda + K) * 4, op, "A");
        check_range(B, (size_t)((N - 1) * ldb + K) * 4, op, "B");
    }
    check_range(C, (size_t)((M - 1) * ldc + N) * 4, op, "C");
    if (bias) check_range(bias, (size_t)N * 4, op, "bias");
    const bool lt = K > 0 && lda % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0 && aligned(A, 16) && aligned(B, 16) &&
                    aligned(C, 16) && (!bias || aligned(bias, 16));
    // C on A or B: the routes below that were always there
    const size_t cbytes = (size_t)((M - 1) * ldc + N) * 4;
    const bool apart = K == 0 || (!overlaps(C, cbytes, A, (size_t)((M - 1) * lda + K) * 4) &&
                                  !overlaps(C, cbytes, B, (size_t)((N - 1) * ldb + K) * 4));
    if (apart && gemv_f32(M, N, K, A, lda, B, ldb, C, ldc, bias, accumulate)) {  // a few rows
        launched(op);
        if (lt) reserve_blaslt();
        return;
    }
    // Split operands from the size where their pack and second launch pay
    // (MI355X, us, the library's fp32 GEMM in front): [512,640] x [5120,640] 36 / 31,
    // [256,2560] x [3840,2560] 44 / 42, [256,1280] x [4608,1280] 41 / 27, [8192,320] x
    // [2560,320] 107 / 67, [4224,2560] x [3840,2560] 583 / 231; with fewer rows the
    // weights' pack is not won back ([231,2560] x [3840,2560] 41 / 43). From 2.4 GFLOP
    // only tall ones, whose packed weights many rows share: [6400,320] x [640,320]
    // 24.5 / 23.9, [2400,512] x [1024,512] 35 / 21, [4800,512] x [512,512] 36 / 23 to 29;
    // below, [4096,512] x [512,512] 19.5 / 21.4, [1024,1024] x [1024,1024] 18.8 / 22.8,
    // [330,640] x [5120,640] 23 / 28. Not with under 256 columns ([8192,2048] x [128,2048]
    // 38 / 47) or a K that the pack cannot hold in registers ([512,65536] x [128,65536] 74 /
    // 223), nor a short one of few rows ([300,128] x [40000,128] 37 / 42) or, from 2.4 GFLOP, one
    // longer than the row that it makes ([2048,1200] x [512,1200] 26 / 29). Operands that the library
    // path does not take: from the size where the kernel below is slower ([130,33] x [70,33]
    // 8.6 / 9.3, [257,321] x [300,321] 31.6 / 10.8).
    const double flops = 2.0 * (double)M * (double)N * (double)K;
    const bool large = N >= 256 && K <= 16384 &&
                       ((flops >= 3e9 && M >= 256 && (M >= 512 || K >= 256)) || (flops >= 2.4e9 && M >= 2048 && K <= N));
    if (K > 0 && apart && (lt ? large : K >= 64 && M >= 16 && N >= 16) &&
        split_gemm(M, N, K, A, lda, B, ldb, C, ldc, bias, accumulate)) {
        launched(op);
        if (lt) reserve_blaslt();
        return;
    }
    // the library GEMM for aligned operands (fp32 products, fp32 accumulation)
    if (lt && blaslt_gemm(true, M, N, K, A, lda, B, ldb, C, ldc, bias, accumulate)) {
        launched(op);
        return;
    }
    const int64_t gx = (N + kT - 1) / kT, gy = (M + kT - 1) / kT;
    need(gy <= 65535 && gx * kThreads <= kMaxGridItems, op, "matrix too large for one launch");
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && aligned(A, 16) && aligned(B, 16);
    const dim3 grid((unsigned)gx, (unsigned)gy);
    if (vec)
        k_gemm_f32<true><<<grid, kThreads, 0, stream()>>>(A, lda, B, ldb, C, ldc, bias, M, N, K, accumulate ? 1 : 0);
    else
        k_gemm_f32<false><<<grid, kThreads, 0, stream()>>>(A, lda, B, ldb, C, ldc, bias, M, N, K, accumulate ? 1 : 0);
    launched(op);
}

}  // namespace

void to_bf16_device(const char* op, const float* x, uint16_t* y, int64_t n) {
    (void)op;
    if (n <= 0) return;
    const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, (int64_t)num_cus() * 32);
    k_to_bf16<<<grid, 256, 0, stream()>>>(x, y, n);
}

}  // namespace sdh

using namespace sdh;

extern "C" {

int sdh_gemm_nt_f32(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb,
                    float* C, int64_t ldc, const float* bias, int accumulate) {
    return guarded([&] { run_gemm_f32(M, N, K, A, lda, B, ldb, C, ldc, bias, accumulate != 0); });
}

int sdh_to_bf16(const float* x, uint16_t* y, int64_t n) {
    return guarded([&] {
        const char* op = "sdh_to_bf16";
        need(n >= 0, op, "negative size");
        if (n == 0) return;
        ensure_init();
        check_range(x, (size_t)n * 4, op, "x");
        check_range(y, (size_t)n * 2, op, "y");
        const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, (int64_t)num_cus() * 32);
        k_to_bf16<<<grid, 256, 0, stream()>>>(x, y, n);
        launched(op);
    });
}

}  // extern "C"
