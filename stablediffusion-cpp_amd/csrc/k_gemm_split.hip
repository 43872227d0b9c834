// k_gemm_split.hip - fp32 matrix products on the fp16 matrix cores: the linear
// layer with fp32 weights (backend_cuda.h:38-40, gemm_nt_f32) and conv2d
// (backend_cuda.h:45-47; tensor.cpp:520-560) as an implicit GEMM.
//
// What bounds these: gfx950's fp32 MFMA runs at 157 TFLOP/s, 1/16 of the fp16
// rate. Every operand is therefore split as in the attention kernels: a block
// of values is scaled by a power of two 2^-e that brings its largest magnitude
// into [2^14, 2^15), each scaled value x becomes hi = rne16(x) and
// lo = rne16(x - hi), and a product is lo_a hi_b + hi_a lo_b + hi_a hi_b with
// fp32 accumulation: three fp16 MFMAs per fp32 product. |x - hi - lo| is at most
// 2^-23 |x| while |x| >= 2^-16 of the block's largest value and at most 2^-39
// of that value below it; the dropped lo_a lo_b is at most 2^-24 of the product.
// Where the values that lose bits this way could matter, fp32 takes over: the
// pack counts, row by row, the values below 2^-19 of the row's largest that were
// not held exactly, and a result stands only if its magnitude is at least 2^20
// times the most that they can have cost it (kPerTail; as a rule they cost a
// tenth of that); else it is computed by fp32 FMAs from the original operands.
// Few ordinary rows have such a value, and about one result in 10^8 is computed
// again; a row of unlike groups of channels met by weights that ignore the
// large ones gives what fp32 gives.
// Against 64-bit results the products come out closer than the fp32 MFMA's,
// whose K additions round one by one where these round once per 16 products.
//   linear  a block is one row of A, one row of B (one output feature)
//   conv2d  a block is one output channel's weights, or 32 channels of a sample
//           of x (whose scale the weights take over, see the pack)
// The exponents are exact and are applied to the accumulators at the end.
// A result whose row or column (conv2d: one of its pixels) holds an infinity or a
// NaN is computed by those FMAs too, so such inputs give what fp32 gives.
//
// Packed operands (library scratch): K is cut into steps of 32; a step of a row
// is 128 bytes, 32 hi halves then 32 lo halves, and all rows of a step lie
// together (a plane). For conv2d a row is a pixel and a step 32 input channels
// under one kernel tap: the planes of x hold each pixel once and a step reads
// them at the tap's offset (one more row of zeros stands for the padding), so
// no patch matrix is written; the weights are packed in the steps' order
// (channels slowest, so that the nine taps of 32 channels follow each other
// and find the same pixels in L2).
//
// Product kernel: BM x BN tile, operands from global memory straight into LDS
// (buffer loads, two stages), rows of 128 bytes with 16-byte chunk c of row r at
// c ^ ((r >> 1) & 7): fragment reads of 16 consecutive rows hit 16 distinct chunks.
// v_mfma_f32_32x32x16_f16: lane l holds row l % 32 of A and of B, k (l / 32) * 8 .. + 7;
// result column l % 32, rows (i / 4) * 8 + (l / 32) * 4 + i % 4.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "sdh_internal.hpp"

namespace sdh {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;
using dev::f4;

constexpr int kStep = 32;            // K per step
constexpr int kRowBytes = 128;       // one row of one step: 32 hi, 32 lo
constexpr int kBad = 1 << 20;        // exponent of a row that holds an infinity or a NaN
constexpr unsigned kInf = 0x7F800000u;
constexpr unsigned kNotFinite = 1u << 31;  // in a row's count: it holds an infinity or a NaN
// A scaled value is off by at most 2^-25, which for one below kSmall can be more than 2^-20 of it.
// It meets one below 2^15: 2^-10 of a result before the exponents, and 2^20 times that must be reached.
constexpr float kSmall = 0x1p-5f, kPerTail = 1024.f;
constexpr int kBufferWord3 = 0x00020000;  // raw buffer resource, 32-bit data format

__device__ __forceinline__ unsigned absbits(float x) { return __float_as_uint(x) & 0x7FFFFFFFu; }

// The exponent of a block whose largest magnitude has these bits: scaled by
// 2^-e it lies in [2^14, 2^15). kBad if it is not finite.
__device__ __forceinline__ int exp_of(unsigned bits) {
    if (bits >= kInf) return kBad;
    if (bits == 0) return 0;
    return max((int)(bits >> 23), 1) - 141;
}

__device__ __forceinline__ unsigned wave_umax(unsigned v) {
#pragma unroll
    for (int o = 32; o; o >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, o, 64));
    return v;
}

__device__ __forceinline__ unsigned wave_usum(unsigned v) {
#pragma unroll
    for (int o = 32; o; o >>= 1) v += (unsigned)__shfl_xor((int)v, o, 64);
    return v;
}

// Eight values scaled by 2^s and split; how many of them are small (see kPerTail)
// and not held exactly, which few waves have to count.
__device__ __forceinline__ int split8(const float* x, int s, h8& hi, h8& lo) {
    float least = INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float v = __builtin_amdgcn_ldexpf(x[e], s);
        least = fminf(least, fabsf(v));
        hi[e] = (_Float16)v;
        lo[e] = (_Float16)(v - (float)hi[e]);
    }
    int n = 0;
    if (__any(least < kSmall)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = __builtin_amdgcn_ldexpf(x[e], s);
            const float back = (float)hi[e] + (float)lo[e];  // exact for small v; v may have vanished in the scaling
            n += fabsf(v) < kSmall && (back != v || (v == 0.f) != (x[e] == 0.f));
        }
    }
    return n;
}

// What a row's count asks of a result's magnitude.
__device__ __forceinline__ float limit_of(unsigned tail) { return tail >= kNotFinite ? INFINITY : (float)tail * kPerTail; }

// ---------------------------------------------------------------------------
// Pack of dense rows: X [rows, K] (ld) -> planes, exps. One wave per row: the
// row's largest magnitude first, then (from L1/L2) eight values per lane and turn.
// ---------------------------------------------------------------------------
struct PackRows {
    const float* X;
    int64_t ld;
    u16* P;
    int* exps;
    unsigned* tails;  // see kPerTail
    int rows, K;
    // further matrices of the same sizes: matrix i starts at X + (i / inner) outer_ld + (i % inner) inner_ld
    int inner;
    int64_t outer_ld, inner_ld;
};

__device__ __forceinline__ unsigned umax4(const f4& v) {
    return max(max(absbits(v.x), absbits(v.y)), max(absbits(v.z), absbits(v.w)));
}
__device__ __forceinline__ int store_split(u16* o, const float* v, int s) {
    h8 hi, lo;
    const int n = split8(v, s, hi, lo);
    *(h8*)o = hi;
    *(h8*)(o + kStep) = lo;
    return n;
}
// A row of LANES threads' values to steps. TURNS > 0: float4 loads (K, ld and X
// aligned for them) of at most 8 LANES TURNS values, all in flight at once and
// kept in registers. TURNS = 0: any row, read twice.
template <int LANES, int TURNS>
__device__ __forceinline__ void pack_row(const PackRows& a, const float* x, u16* P, int* exps, unsigned* tails, int row,
                                         int lane, unsigned* red) {
    const int kp = (a.K + kStep - 1) / kStep * kStep;
    auto out = [&](int k) __attribute__((always_inline)) {
        return P + ((int64_t)(k / kStep) * a.rows + row) * (kRowBytes / 2) + (k % kStep);
    };
    bool bad = false;
    auto exponent = [&](unsigned m) __attribute__((always_inline)) {
        m = wave_umax(m);
        if constexpr (LANES > 64) {
            if ((lane & 63) == 0) red[lane >> 6] = m;
            __syncthreads();
            m = max(max(red[0], red[1]), max(red[2], red[3]));
        }
        const int e = exp_of(m);
        if (lane == 0) exps[row] = e;
        bad = e == kBad;
        return bad ? 0 : -e;
    };
    unsigned m = 0;
    int n = 0;
    if constexpr (TURNS > 0) {
        f4 v[TURNS][2];
#pragma unroll
        for (int j = 0; j < TURNS; ++j) {  // past the row: its last four values, dropped below
            const int k = (j * LANES + lane) * 8;
            v[j][0] = *(const f4*)(x + min(k, a.K - 4));
            v[j][1] = *(const f4*)(x + min(k + 4, a.K - 4));
        }
#pragma unroll
        for (int j = 0; j < TURNS; ++j) m = max(m, max(umax4(v[j][0]), umax4(v[j][1])));
        const int e = exponent(m);
#pragma unroll
        for (int j = 0; j < TURNS; ++j) {
            const int k = (j * LANES + lane) * 8;
            if (k >= kp) continue;
            float f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = k + i < a.K ? v[j][i / 4][i % 4] : 0.f;
            n += store_split(out(k), f, e);
        }
    } else {
#pragma unroll 4
        for (int k = lane; k < a.K; k += LANES) m = max(m, absbits(x[k]));
        const int e = exponent(m);
        for (int k = lane * 8; k < kp; k += LANES * 8) {
            float f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = k + i < a.K ? x[k + i] : 0.f;
            n += store_split(out(k), f, e);
        }
    }
    unsigned tail = __any(n) ? wave_usum((unsigned)n) : 0u;
    if constexpr (LANES > 64) {
        if ((lane & 63) == 0) red[4 + (lane >> 6)] = tail;
        __syncthreads();
        tail = (red[4] + red[5]) + (red[6] + red[7]);
    }
    if (lane == 0) tails[row] = bad ? kNotFinite : tail;
}

// Two operands in one launch: the first ba workgroups take a's rows, the rest
// b's. Four rows per workgroup, a wave each, or (LANES 256) one. grid.y: the matrices.
template <int LANES, int TURNS>
__global__ __launch_bounds__(256, TURNS < 4 ? 8 : 4) void k_split_pack(PackRows a, PackRows b, int ba) {
    constexpr int ROWS = 256 / LANES;
    __shared__ unsigned red[8];
    const bool first = (int)blockIdx.x < ba;
    const PackRows& p = first ? a : b;
    const int row = ((int)blockIdx.x - (first ? 0 : ba)) * ROWS + (int)threadIdx.x / LANES;
    if (row >= p.rows) return;  // a whole wave or workgroup
    const int i = blockIdx.y;
    const int64_t steps = (p.K + kStep - 1) / kStep;
    const float* x = p.X + (i / p.inner) * p.outer_ld + (i % p.inner) * p.inner_ld + (int64_t)row * p.ld;
    pack_row<LANES, TURNS>(p, x, p.P + i * steps * p.rows * (kRowBytes / 2), p.exps + (int64_t)i * p.rows,
                           p.tails + (int64_t)i * p.rows, row, threadIdx.x % LANES, red);
}

// ---------------------------------------------------------------------------
// conv2d's pack. Launch 1: the weights, and the largest values of x per sample, 32
// channels and part of the pixels. Every workgroup of launch 2 reads all of these,
// so there are at most kMaxima, or kTable where samples and channels alone are
// more. Launch 2: the exponents, then the pixels, and the weights once more where
// they take over some of x's scale.
// Channels of unlike scale: chunk c of 32 channels has an exponent ec of its own
// besides the sample's es, and the weights of these channels take 2^ec before
// their row's exponent is found, so that x w keeps its value. With f the largest
// over the samples of (chunk's exponent - sample's), ec is f / 2 from -kNear on: x
// and w share the spread, and neither loses bits while it is below 2^34, whether the
// weights are alike, reciprocal to it, or zero where x is large. Chunks nearer to
// their sample, as a rule all of them, leave the weights as launch 1 packed them:
// packing them after the maxima, or reading them twice, took 3 to 9 us more
// ([1280,1280,3,3]: 59 MB).
// ---------------------------------------------------------------------------
constexpr int kTable = 2048, kMaxima = 256, kNear = 8;

struct ConvPack {
    const float* x;       // [N, Cin, HW]
    const float* w;       // [Cout, Cin, taps]
    unsigned* maxima;     // [N, chunks, parts], of finite values
    u16* X;               // planes of N * HW + 1 pixels
    u16* Wp;              // planes of Cout rows
    int* ex;              // [N]
    int* ew;              // [Cout]
    unsigned* tx;         // [N * HW + 1]: counts of the pixels, see kPerTail
    unsigned* tw;         // [Cout]
    int N, Cin, HW, Cout, taps;
    int chunks, parts;    // 32-channel steps; parts of the pixels, a power of two
    int per, groups;      // steps that a workgroup of launch 2 packs; such groups of steps
    int tiles, run, runs; // 64-pixel tiles of a sample; tiles that a workgroup packs; such runs
};

// One output channel's weights: [Cin][taps] -> steps (32 channels, tap), through
// LDS where there is room for them at `row`. FOLD: with 2^ec.
template <bool FOLD>
__device__ __forceinline__ void conv_pack_weights(const ConvPack& a, int co, const int* ec, float* row, unsigned* red) {
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, K = a.Cin * a.taps, chunk = kStep * a.taps;
    const float* w = a.w + (int64_t)co * K;
    // the largest |w| 2^ec by its bits with ec added to the exponent: floor(that / 2^23) bounds the
    // magnitude also where the exponent falls below 1, or the weight is subnormal or zero
    int m = INT_MIN, top = 0;
    int c = t / chunk, r = t - c * chunk;  // FOLD: the weight's chunk, its place there
    const int dc = 256 / chunk, dr = 256 - dc * chunk;
    constexpr int U = 8;
    for (int k0 = t; k0 < K; k0 += U * 256) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = w[min(k0 + u * 256, K - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u * 256 >= K) break;
            if (row) row[k0 + u * 256] = v[u];
            const int b = (int)absbits(v[u]);
            top = max(top, b);
            if constexpr (FOLD) {
                m = max(m, b + ec[c] * (1 << 23));
                r += dr;
                const int over = r >= chunk ? 1 : 0;
                c += dc + over;
                r -= over ? chunk : 0;
            }
        }
    }
    if constexpr (!FOLD) m = top;
#pragma unroll
    for (int o = 32; o; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    if (lane == 0) red[wv] = (unsigned)m;
    const bool bad = __syncthreads_or(top >= (int)kInf);
    m = max(max((int)red[0], (int)red[1]), max((int)red[2], (int)red[3]));
    const int e = (m >> 23) - 141;  // scaled by 2^(ec - e) the largest lies below 2^15
    if (t == 0) a.ew[co] = bad ? kBad : e;
    const int tasks = a.chunks * a.taps * 4;
    unsigned tail = 0;
    for (int i = t; i < tasks; i += 256) {  // eight channels of one step
        const int g = i & 3, step = i >> 2, cc = step / a.taps, tap = step - cc * a.taps, c0 = cc * kStep + g * 8;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = min((c0 + j) * a.taps + tap, K - 1);
            const float x = row ? row[k] : w[k];
            v[j] = c0 + j < a.Cin ? x : 0.f;
        }
        const int shift = (FOLD ? ec[cc] : 0) - e;
        tail += store_split(a.Wp + ((int64_t)step * a.Cout + co) * (kRowBytes / 2) + g * 8, v, bad ? 0 : shift);
    }
    tail = __any(tail != 0) ? wave_usum(tail) : 0u;
    if (lane == 0) red[4 + wv] = tail;
    __syncthreads();
    if (t == 0) a.tw[co] = bad ? kNotFinite : (red[4] + red[5]) + (red[6] + red[7]);
}

__global__ __launch_bounds__(256) void k_conv_prep(ConvPack a, int in_lds) {
    extern __shared__ float row[];
    __shared__ unsigned red[8];
    const int t = threadIdx.x, nx = gridDim.x - a.Cout, b = (int)blockIdx.x - a.Cout;
    if (b < 0) {
        if (in_lds) conv_pack_weights<false>(a, blockIdx.x, nullptr, row, red);
        else conv_pack_weights<false>(a, blockIdx.x, nullptr, nullptr, red);
        return;
    }
    for (int i = b * 256 + t; i <= a.N * a.HW; i += nx * 256) a.tx[i] = 0;
    const int part = b % a.parts, c0 = b / a.parts % a.chunks * kStep, n = b / (a.parts * a.chunks);
    const float* x = a.x + ((int64_t)n * a.Cin + c0) * a.HW;
    unsigned m = 0;
    for (int64_t p0 = part * 256; p0 < a.HW; p0 += a.parts * 256) {
        const int p = min((int)p0 + t, a.HW - 1);  // past the last pixel: that one again
        float v[kStep];
#pragma unroll
        for (int c = 0; c < kStep; ++c) v[c] = x[(int64_t)min(c, a.Cin - 1 - c0) * a.HW + p];  // likewise
#pragma unroll
        for (int c = 0; c < kStep; ++c) {
            const unsigned b = absbits(v[c]);
            m = max(m, b < kInf ? b : 0u);
        }
    }
    m = wave_umax(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    if (t == 0) a.maxima[b] = max(max(red[0], red[1]), max(red[2], red[3]));
}

// Exponents from the maxima: E [N, chunks], the chunks' biased ones (bits >> 23, at
// least 1; 0: all zero), and ec [chunks]; S [N]: the samples'. By the whole workgroup.
__device__ __forceinline__ int wave_imax(int v) { return (int)dev::wave_max((float)v); }  // |v| < 2^24
__device__ __forceinline__ void conv_scales(const ConvPack& a, int* E, int* S, int* ec) {
    constexpr int kNone = -1000;
    const int t = threadIdx.x, lane = t & 63, words = a.N * a.chunks * a.parts;
    if (a.parts > 64) {  // at most kMaxima / 128 entries
        if (t < a.N * a.chunks) E[t] = 0;
        __syncthreads();
    }
    for (int i0 = t - lane; i0 < words; i0 += 256) {
        const int i = i0 + lane;
        unsigned m = i < words ? a.maxima[i] : 0u;
        for (int o = 1; o < min(a.parts, 64); o <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
        const int e = m ? max((int)(m >> 23), 1) : 0;
        if (a.parts <= 64) {
            if (lane % a.parts == 0 && i < words) E[i / a.parts] = e;
        } else if (lane == 0) {
            atomicMax(E + i / a.parts, e);
        }
    }
    if (a.chunks < a.N)
        for (int c = t; c < a.chunks; c += 256) ec[c] = kNone;
    __syncthreads();
    // f, a chunk's largest (own - sample's) over the samples
    auto folded = [](int f) __attribute__((always_inline)) { return f == kNone || f > -kNear ? 0 : f / 2; };  // from -126 on
    if (a.chunks < a.N) {  // a lane per sample, at most 45 chunks (kTable)
        for (int n0 = t - lane; n0 < a.N; n0 += 256) {
            const int n = min(n0 + lane, a.N - 1);
            int whole = 0;
            for (int c = 0; c < a.chunks; ++c) whole = max(whole, E[n * a.chunks + c]);
            for (int c = 0; c < a.chunks; ++c) {
                const int own = E[n * a.chunks + c], f = wave_imax(own ? own - whole : kNone);
                if (lane == 0) atomicMax(ec + c, f);
            }
        }
        __syncthreads();
        for (int c = t; c < a.chunks; c += 256) ec[c] = folded(ec[c]);
    } else {  // a thread per chunk; a wave finds every fourth sample's, of one sample each wave for itself
        for (int n = a.N > 1 ? t >> 6 : 0; n < a.N; n += 4) {
            int whole = 0;
            for (int c = lane; c < a.chunks; c += 64) whole = max(whole, E[n * a.chunks + c]);
            S[n] = wave_imax(whole);  // the same from every lane
        }
        if (a.N > 1) __syncthreads();
        for (int c = t; c < a.chunks; c += 256) {
            int f = kNone;
#pragma unroll 4
            for (int n = 0; n < a.N; ++n) {
                const int own = E[n * a.chunks + c];
                f = max(f, own ? own - S[n] : kNone);
            }
            ec[c] = folded(f);
        }
    }
    __syncthreads();
}
// A sample's exponent beside those: its scaled values lie below 2^15.
__device__ __forceinline__ int conv_sample_exp(const ConvPack& a, const int* E, const int* ec, int n) {
    constexpr int kNone = -1000;
    int e = kNone;
    for (int c = threadIdx.x & 63; c < a.chunks; c += 64) {
        const int own = E[n * a.chunks + c];
        e = max(e, own ? own - 141 - ec[c] : kNone);
    }
    e = wave_imax(e);
    return e == kNone ? 0 : e;
}

// `run` times 64 pixels of a sample, `per` steps of 32 channels; each step through
// LDS, so that x is read in runs of 64 pixels and a step of 64 pixels is written
// as 8 KB in a row.
template <class Scales>
__device__ __forceinline__ void conv_pack_pixels(const ConvPack& a, int b, const int* E, const int* ec, u16* tile,
                                                 Scales&& scales) {
    const int t = threadIdx.x, lane = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
    const int run = b % a.runs, group = b / a.runs % a.groups, n = b / (a.runs * a.groups);
    const int s0 = group * a.per, s1 = min(a.chunks, s0 + a.per);
    float v[8];
    auto load = [&](int p, int s) __attribute__((always_inline)) {  // channels past the last: that one again, dropped below
        const int c0 = s * kStep + g * 8;
        const float* x = a.x + (int64_t)n * a.Cin * a.HW;
        const int pix = min(p * 64 + lane, a.HW - 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[(int64_t)min(c0 + j, a.Cin - 1) * a.HW + pix];
    };
    load(run * a.run, s0);
    scales();  // behind the first loads
    const int e = conv_sample_exp(a, E, ec, n);
    if (run == 0 && group == 0 && t == 0) a.ex[n] = e;
    const int64_t prows = (int64_t)a.N * a.HW + 1;
    const int p1 = min(a.tiles, (run + 1) * a.run);
    for (int p = run * a.run; p < p1; ++p) {
        const int p0 = p * 64, pix = p0 + lane;
        unsigned tail = 0;
        for (int s = s0; s < s1; ++s) {
            const int c0 = s * kStep + g * 8;
            unsigned m = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                v[j] = c0 + j < a.Cin ? v[j] : 0.f;
                m = max(m, absbits(v[j]));
            }
            h8 hi, lo;
            const unsigned c = split8(v, -(e + ec[s]), hi, lo);
            tail = (tail + c) | (m >= kInf ? kNotFinite : 0u);  // the count stays far below the mark
            const bool last = s + 1 == s1;
            if (!last || p + 1 < p1) load(last ? p + 1 : p, last ? s0 : s + 1);
            __syncthreads();  // the previous step's tile is read
            *(h8*)(tile + lane * 64 + ((g ^ (lane & 7)) << 3)) = hi;
            *(h8*)(tile + lane * 64 + (((g + 4) ^ (lane & 7)) << 3)) = lo;
            __syncthreads();
            u16* out = a.X + ((int64_t)s * prows + (int64_t)n * a.HW + p0) * 64;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int i = t + j * 256, r = i >> 3, k = i & 7;
                if (p0 + r < a.HW) *(h8*)(out + i * 8) = *(const h8*)(tile + r * 64 + ((k ^ (r & 7)) << 3));
            }
            if (n == a.N - 1 && p0 + 64 >= a.HW && t < 8)  // the row of zeros
                *(u32x4*)(a.X + ((int64_t)s * prows + prows - 1) * 64 + t * 8) = u32x4{0, 0, 0, 0};
        }
        if (tail && pix < a.HW) {  // rare; whole numbers, so that the order does not matter
            unsigned* at = a.tx + (int64_t)n * a.HW + pix;
            if (tail >= kNotFinite) atomicOr(at, kNotFinite);
            else atomicAdd(at, tail);
        }
    }
}

__global__ __launch_bounds__(256) void k_conv_pack(ConvPack a) {
    extern __shared__ int lds[];
    __shared__ unsigned red[8];
    __shared__ __attribute__((aligned(16))) u16 tile[64 * 64];
    int *E = lds, *ec = E + a.N * a.chunks, *S = ec + a.chunks;
    auto scales = [&]() __attribute__((always_inline)) { conv_scales(a, E, S, ec); };
    const int pixels = a.runs * a.groups * a.N;
    if ((int)blockIdx.x < pixels) {
        conv_pack_pixels(a, blockIdx.x, E, ec, tile, scales);
        return;
    }
    scales();
    bool fold = false;
    for (int c = threadIdx.x; c < a.chunks; c += 256) fold |= ec[c] != 0;
    if (__syncthreads_or(fold)) conv_pack_weights<true>(a, blockIdx.x - pixels, ec, nullptr, red);
}

// ---------------------------------------------------------------------------
// The product
// ---------------------------------------------------------------------------
enum Kind { kDense = 0, kConv = 1, kWeights = 2 };  // kWeights: A holds softmax weights, packed row by row

struct SplitArgs {
    const u16* A;
    const u16* B;
    int64_t planeA, planeB;  // bytes from one step's rows to the next's
    int rowA;                // bytes from one row of A's step to the next
    const int* ea;           // per row
    const int* eb;           // per column; conv2d: per sample
    const unsigned* ta;      // counts per row (not kWeights), per column; conv2d: per pixel: see kPerTail
    const unsigned* tb;
    float* C;
    int64_t ldc;
    const float* bias;       // per column; conv2d: per row
    int M, N, K;
    int steps, accumulate;
    int tm, tn, splits;      // tiles, parts of K
    float* part;             // splits > 1: [splits][tm * BM][tn * BN] sums without the exponents
    float* limc;             // conv2d, splits > 1: the columns' limits
    // further products of the same sizes (splits = 1): product i = (o, h) = (i / inner, i % inner)
    // takes A's matrix i, B's matrix o * kv + h / group and stores at C + o outC + h inC
    int batches, inner, group, kv;
    int64_t matA, matB, outC, inC, outA0, inA0, outB0, inB0;
    int causal, row0;        // kWeights: row r's weights end at column row0 + r
    // the original operands
    const float* A0;
    const float* B0;
    int64_t lda, ldb;
    // conv2d
    int H, W, Wo, HWo, kh, kw, stride, pad, taps, Cin, Cout, zero;
};

// Where element (row, col) lies, and what is added to it.
template <bool CONV>
__device__ __forceinline__ float* place(const SplitArgs& p, int row, int col) {
    if constexpr (CONV) {
        const int n = col / p.HWo;
        return p.C + ((int64_t)n * p.Cout + row) * p.HWo + (col - n * p.HWo);
    } else {
        return p.C + (int64_t)row * p.ldc + col;
    }
}
template <bool CONV>
__device__ __forceinline__ void store(const SplitArgs& p, int row, int col, float* cp, float v) {
    if (p.accumulate) v += *cp;
    if (p.bias) v += p.bias[CONV ? row : col];
    *cp = v;
}

// ---------------------------------------------------------------------------
// The fp32 path: elements by fp32 FMAs from the original operands.
// ---------------------------------------------------------------------------
// Where column col's patch lies (conv2d): its sample, and its first pixel.
struct Patch {
    const float* x;
    int iy, ix;
};
__device__ __forceinline__ Patch patch_of(const SplitArgs& p, int col) {
    const int n = col / p.HWo, q = col - n * p.HWo, oy = q / p.Wo, ox = q - oy * p.Wo;
    return Patch{p.B0 + (int64_t)n * p.Cin * p.H * p.W, oy * p.stride - p.pad, ox * p.stride - p.pad};
}
__device__ __forceinline__ float patch_value(const SplitArgs& p, const Patch& a, int ci, int ky, int kx) {
    const int iy = a.iy + ky, ix = a.ix + kx;
    const bool in = (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W;
    const float v = a.x[((int64_t)ci * p.H + (in ? iy : 0)) * p.W + (in ? ix : 0)];  // no load under a mask
    return in ? v : 0.f;
}
// Softmax weight k of a row as it was packed, with the row's exponent; one too small to be
// held counts as tiny, so that it still meets an infinity of B as fp32 has it.
__device__ __forceinline__ float packed_weight(const SplitArgs& p, int row, int e, int k) {
    const _Float16* h = (const _Float16*)((const char*)p.A + (int64_t)row * p.rowA + (k / kStep) * p.planeA) + k % kStep;
    return fmaxf(__builtin_amdgcn_ldexpf((float)h[0] + (float)h[kStep], e), 1e-38f);
}
__device__ __forceinline__ int weights_of(const SplitArgs& p, int row) {  // how many a row has
    return p.causal ? min(p.K, p.row0 + row + 1) : p.K;
}

// Thread t of T's share of one element.
template <Kind KIND>
__device__ __forceinline__ float dot_share(const SplitArgs& p, int row, int col, int t, int T) {
    float s = 0.f;
    if constexpr (KIND == kConv) {
        const Patch at = patch_of(p, col);
        const float* w = p.A0 + (int64_t)row * p.K;
#pragma unroll 4
        for (int k = t; k < p.K; k += T) {
            const int ci = k / p.taps, tap = k - ci * p.taps, ky = tap / p.kw;
            s = fmaf(w[k], patch_value(p, at, ci, ky, tap - ky * p.kw), s);
        }
    } else if constexpr (KIND == kWeights) {
        const int e = p.ea[row], end = weights_of(p, row);
        if (e == kBad) return __builtin_nanf("");
        const float* b = p.B0 + (int64_t)col * p.ldb;
#pragma unroll 4
        for (int k = t; k < end; k += T) s = fmaf(packed_weight(p, row, e, k), b[k], s);
    } else {
        const float* a = p.A0 + (int64_t)row * p.lda;
        const float* b = p.B0 + (int64_t)col * p.ldb;
#pragma unroll 8
        for (int k = t; k < p.K; k += T) s = fmaf(a[k], b[k], s);
    }
    return s;
}

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // four floats at any float's address

// Sixteen elements' sums over [k0, k1), K cut over the waves: rows row[], columns col[].
template <Kind KIND>
__device__ __forceinline__ void dot16(const SplitArgs& p, const int* row, const int* col, int k0, int k1,
                                      float (&s)[4][4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) s[r][c] = 0.f;
    auto add = [&](const float* a, const float* b) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) s[r][c] = fmaf(a[r], b[c], s[r][c]);
    };
    float a[4], b[4];
    if constexpr (KIND == kConv) {
        Patch at[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) at[c] = patch_of(p, col[c]);
        int ci = k0 / p.taps, ky = (k0 - ci * p.taps) / p.kw, kx = k0 - ci * p.taps - ky * p.kw;
        constexpr int U = 4;  // so many k's loads on their way at once; past k1: the last one again, not added
        for (int k = k0; k < k1; k += U) {
            float va[U][4], vb[U][4];
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int r = 0; r < 4; ++r) va[u][r] = p.A0[(int64_t)row[r] * p.K + min(k + u, k1 - 1)];
#pragma unroll
                for (int c = 0; c < 4; ++c) vb[u][c] = patch_value(p, at[c], ci, ky, kx);
                if (k + u + 1 < k1 && ++kx == p.kw) {
                    kx = 0;
                    if (++ky == p.kh) ky = 0, ++ci;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k + u < k1) add(va[u], vb[u]);
        }
    } else if constexpr (KIND == kWeights) {
        int e[4], end[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            e[r] = p.ea[row[r]];
            end[r] = weights_of(p, row[r]);
        }
        for (int k = k0; k < k1; ++k) {
#pragma unroll
            for (int c = 0; c < 4; ++c) b[c] = p.B0[(int64_t)col[c] * p.ldb + k];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float w = e[r] == kBad ? __builtin_nanf("") : packed_weight(p, row[r], e[r], k);
#pragma unroll
                for (int c = 0; c < 4; ++c) s[r][c] = k < end[r] ? fmaf(w, b[c], s[r][c]) : s[r][c];
            }
        }
    } else {
        const float *pa[4], *pb[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pa[r] = p.A0 + (int64_t)row[r] * p.lda;
            pb[r] = p.B0 + (int64_t)col[r] * p.ldb;
        }
        int k = k0;
#pragma unroll 2
        for (; k + 4 <= k1; k += 4) {
            f4u va[4], vb[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                va[r] = *(const f4u*)(pa[r] + k);
                vb[r] = *(const f4u*)(pb[r] + k);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int r = 0; r < 4; ++r) a[r] = va[r][i], b[r] = vb[r][i];
                add(a, b);
            }
        }
        for (; k < k1; ++k) {
#pragma unroll
            for (int r = 0; r < 4; ++r) a[r] = pa[r][k], b[r] = pb[r][k];
            add(a, b);
        }
    }
}

// One element by the workgroup's T threads; `sums`: T / 64 floats of LDS.
template <Kind KIND, int T>
__device__ __forceinline__ void element_fp32(const SplitArgs& p, int row, int col, float* sums) {
    const int t = threadIdx.x;
    const float s = dev::wave_sum(dot_share<KIND>(p, row, col, t, T));
    if ((t & 63) == 0) sums[t >> 6] = s;
    __syncthreads();
    if (t == 0) {
        float v = sums[0];
#pragma unroll
        for (int i = 1; i < T / 64; ++i) v += sums[i];
        store<KIND == kConv>(p, row, col, place<KIND == kConv>(p, row, col), v);
    }
    __syncthreads();
}

// 32 x 32 elements from (row0, col0) on by the workgroup: each wave sums a part
// of K for all of them, sixteen per lane; `sums`: 1024 floats of LDS.
template <Kind KIND, int T>
__device__ __forceinline__ void block_fp32(const SplitArgs& p, int row0, int col0, float* sums) {
    constexpr int NW = T / 64;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    auto row_of = [&](int l, int r) __attribute__((always_inline)) { return row0 + (l >> 3) + 8 * r; };
    auto col_of = [&](int l, int c) __attribute__((always_inline)) { return col0 + (l & 7) + 8 * c; };
    int row[4], col[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        row[r] = min(row_of(lane, r), p.M - 1);
        col[r] = min(col_of(lane, r), p.N - 1);
    }
    float s[4][4];
    dot16<KIND>(p, row, col, (int)((int64_t)p.K * w / NW), (int)((int64_t)p.K * (w + 1) / NW), s);
    for (int i = 0; i < NW; ++i) {
        if (w == i) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float* q = sums + (r * 4 + c) * 64 + lane;
                    *q = i ? *q + s[r][c] : s[r][c];
                }
        }
        __syncthreads();
    }
    for (int i = t; i < 1024; i += T) {
        const int rr = row_of(i & 63, i >> 8), cc = col_of(i & 63, (i >> 6) & 3);
        if (rr < p.M && cc < p.N) store<KIND == kConv>(p, rr, cc, place<KIND == kConv>(p, rr, cc), sums[i]);
    }
    __syncthreads();
}

// COUNT loads of 64 x 16 bytes into LDS, one after the other from dst on: lane l
// of load j reads base + v[j] (a buffer of `bytes` bytes) for dst + 512 j + 8 l.
template <int COUNT>
__device__ __forceinline__ void load_lds(const char* base, int bytes, const int* v, u16* dst) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, kBufferWord3);
#pragma unroll
    for (int j = 0; j < COUNT; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(dst + j * 512), 16, v[j],
                                                 0, 0, 0);
}

template <int BM, int BN, int WM, int WN, int STAGES, Kind KIND>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN), BM * BN > 128 * 128 ? 1 : BM * BN == 128 * 128 ? 2 : 3) void k_split_mm(SplitArgs p) {
    constexpr bool CONV = KIND == kConv;
    static_assert(STAGES == 2 || STAGES == 3, "LDS stages");
    constexpr int NW = (BM / WM) * (BN / WN), T = 64 * NW;
    constexpr int AI = BM / 8 / NW, BI = BN / 8 / NW;  // loads per wave and stage: 8 rows each
    constexpr int RA = WM / 32, RB = WN / 32;
    __shared__ __attribute__((aligned(1024))) u16 sA0[BM * 64];
    __shared__ __attribute__((aligned(1024))) u16 sA1[BM * 64];
    __shared__ __attribute__((aligned(1024))) u16 sA2[STAGES > 2 ? BM * 64 : 8];
    __shared__ __attribute__((aligned(1024))) u16 sB0[BN * 64];
    __shared__ __attribute__((aligned(1024))) u16 sB1[BN * 64];
    __shared__ __attribute__((aligned(1024))) u16 sB2[STAGES > 2 ? BN * 64 : 8];
    __shared__ __attribute__((aligned(16))) int sea[BM];  // exponents of the rows, of the columns
    __shared__ int seb[BN];
    __shared__ float sbias[CONV ? BM : BN];
    // A result stands if its magnitude before the exponents reaches its row's and its column's
    // limit together; else the fp32 path computes it: one by one from `alone`, or by whole
    // blocks of 32 x 32 where a block has more than kAlone of them.
    __shared__ __attribute__((aligned(16))) float slr[BM];
    __shared__ float slc[BN];
    constexpr int NB = (BM / 32) * (BN / 32), kAlone = 16;
    __shared__ int alone[NB * kAlone], whole[NB], nalone, nwhole;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = w / (BN / WN), wn = w % (BN / WN);
    const int fr = lane & 31, fh = lane >> 5;
    // Workgroups go to the 8 XCDs round robin: renumbered so that each XCD runs
    // one contiguous range of tiles; within it, eight row tiles by all columns.
    const int nblk = gridDim.x, xcd = blockIdx.x & 7, per = nblk >> 3, rem = nblk & 7;
    const int lb = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
    const int tiles = p.tm * p.tn, lt = lb % tiles;
    int z = lb / tiles;
    if (!CONV && p.batches > 1) {
        const int o = z / p.inner, h = z - o * p.inner, b = o * p.kv + h / p.group;
        p.A = (const u16*)((const char*)p.A + z * p.matA);
        p.B = (const u16*)((const char*)p.B + b * p.matB);
        p.ea += (int64_t)z * p.M;
        p.eb += (int64_t)b * p.N;
        if (KIND == kDense) p.ta += (int64_t)z * p.M;
        p.tb += (int64_t)b * p.N;
        p.C += o * p.outC + h * p.inC;
        if (KIND == kDense) p.A0 += o * p.outA0 + h * p.inA0;
        p.B0 += o * p.outB0 + (h / p.group) * p.inB0;
        z = 0;
    }
    const int gsz = 8 * p.tn, grp = lt / gsz, in = lt - grp * gsz, gm = min(8, p.tm - grp * 8);
    const int mt = grp * 8 + in % gm, nt = in / gm;
    const int m0 = mt * BM, n0 = nt * BN;

    // this lane's source row in each of the wave's loads; rows past the matrix
    // read its last row (their results are not stored)
    const int lr = lane >> 3;
    int va[AI], vb[BI];
    int iy0[CONV ? BI : 1], ix0[CONV ? BI : 1];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const int r = (w * AI + j) * 8 + lr;
        va[j] = min(m0 + r, p.M - 1) * p.rowA + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int j = 0; j < BI; ++j) {
        const int r = (w * BI + j) * 8 + lr, col = min(n0 + r, p.N - 1);
        const int chunk = ((lane & 7) ^ ((r >> 1) & 7)) << 4;
        if constexpr (CONV) {
            const int n = col / p.HWo, q = col - n * p.HWo, oy = q / p.Wo, ox = q - oy * p.Wo;
            iy0[j] = oy * p.stride - p.pad;
            ix0[j] = ox * p.stride - p.pad;
            vb[j] = (n * p.H * p.W + iy0[j] * p.W + ix0[j]) * kRowBytes + chunk;  // may lie before the sample
        } else {
            vb[j] = col * kRowBytes + chunk;
        }
    }
    const int bytesA = (p.M - 1) * p.rowA + kRowBytes, bytesB = (CONV ? p.zero + 1 : p.N) * kRowBytes;
    // this part's steps, and the one whose stage is issued next: its planes and
    // (conv2d) its tap, counted on without divisions
    const int s0 = (int)((int64_t)p.steps * z / p.splits), s1 = (int)((int64_t)p.steps * (z + 1) / p.splits);
    int left = s1 - s0, ky = 0, kx = 0;  // steps not issued yet
    const char* pa = (const char*)p.A + s0 * p.planeA;
    const char* pb = (const char*)p.B + (CONV ? s0 / p.taps : s0) * p.planeB;
    if (CONV) {
        const int tap = s0 % p.taps;
        ky = tap / p.kw;
        kx = tap - ky * p.kw;
    }
    int src[BI];  // the next stage's offsets into B's plane
    auto aim = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < BI; ++j) {
            src[j] = vb[j];
            if constexpr (CONV) {
                const bool ok = (unsigned)(iy0[j] + ky) < (unsigned)p.H && (unsigned)(ix0[j] + kx) < (unsigned)p.W;
                const int pad = p.zero * kRowBytes + (vb[j] & 127), at = vb[j] + (ky * p.W + kx) * kRowBytes;
                src[j] = pad + ((at - pad) & -(int)ok);
            }
        }
    };
    auto issue = [&](u16* dA, u16* dB) __attribute__((always_inline)) {
        load_lds<AI>(pa, bytesA, va, dA + w * AI * 512);
        load_lds<BI>(pb, bytesB, src, dB + w * BI * 512);
        --left;
        pa += p.planeA;
        if (!CONV) {
            pb += p.planeB;
        } else if (++kx == p.kw) {
            kx = 0;
            if (++ky == p.kh) {
                ky = 0;
                pb += p.planeB;
            }
        }
    };
    // the first stage is on its way while the tile's rows and columns are looked at
    aim();
    issue(sA0, sB0);

    // the rows' and columns' exponents and limits
    bool watch = false;
    auto limit = [&](unsigned tail) __attribute__((always_inline)) {
        watch |= tail != 0;
        return limit_of(tail);
    };
    if (t == 0) nalone = nwhole = 0;
    for (int i = t; i < BM; i += T) {
        const int row = min(m0 + i, p.M - 1), e = p.ea[row];
        sea[i] = e;
        if (CONV) sbias[i] = p.bias ? p.bias[row] : 0.f;
        slr[i] = limit(KIND == kWeights ? (e == kBad ? kNotFinite : 0u) : p.ta[row]);
    }
    for (int i = t; i < BN; i += T) {
        const int col = min(n0 + i, p.N - 1);
        if constexpr (CONV) {
            const int n = col / p.HWo, q = col - n * p.HWo, oy = q / p.Wo, ox = q - oy * p.Wo;
            seb[i] = p.eb[n];
            unsigned tail = 0, bad = 0;  // of all pixels that the column sees
            int ky = 0, kx = 0;
#pragma unroll 4
            for (int tap = 0; tap < p.taps; ++tap) {
                const int iy = oy * p.stride - p.pad + ky, ix = ox * p.stride - p.pad + kx;
                const bool in = (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W;
                const unsigned c = p.tb[in ? (n * p.H + iy) * p.W + ix : p.zero];
                tail += c & ~kNotFinite;
                bad |= c & kNotFinite;
                if (++kx == p.kw) kx = 0, ++ky;
            }
            slc[i] = limit(bad ? kNotFinite : tail);
            if (p.splits > 1 && z == 0 && mt == 0 && n0 + i < p.N) p.limc[col] = slc[i];
        } else {
            const int e = p.eb[col];
            seb[i] = e;
            sbias[i] = p.bias ? p.bias[col] : 0.f;
            slc[i] = limit(p.tb[col]);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    watch = __syncthreads_or(watch);  // the first stage is in LDS behind this

    f32x16 acc[RA][RB];
#pragma unroll
    for (int a = 0; a < RA; ++a)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

    // Fragment addresses: rows 32 apart share their swizzle, so a lane has one
    // chunk offset for each (slice, hi or lo).
    const int offA = (wm * WM + fr) * 64, offB = (wn * WN + fr) * 64;
    int at[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int l = 0; l < 2; ++l) at[s][l] = ((s * 2 + l * 4 + fh) ^ ((fr >> 1) & 7)) << 3;
    // A step is 2 RA turns (slice of 16 k, 32 rows of A) of 3 RB MFMAs; the
    // fragments of a turn are read one turn ahead. Before the last turn's MFMAs,
    // when every fragment of the step is in registers, the workgroup meets: the
    // next step's stage has landed, its first fragments are read behind those
    // MFMAs, and the buffer just read takes the stage STAGES steps on. Not
    // __syncthreads(), which waits for every copy into LDS.
    h8 ah[2], al[2], bh[2][RB], bl[2][RB];
    auto fragA = [&](const u16* tA, int i) __attribute__((always_inline)) {
        ah[i & 1] = *(const h8*)(tA + offA + (i % RA) * 2048 + at[i / RA][0]);
        al[i & 1] = *(const h8*)(tA + offA + (i % RA) * 2048 + at[i / RA][1]);
    };
    auto fragB = [&](const u16* tB, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            bh[s][b] = *(const h8*)(tB + offB + b * 2048 + at[s][0]);
            bl[s][b] = *(const h8*)(tB + offB + b * 2048 + at[s][1]);
        }
    };
    // The step's buffers; nA, nB: the next step's. TAIL: among the last steps, where
    // the next stages may not exist.
    auto step = [&](auto tail, int s, u16* cA, u16* cB, u16* nA, u16* nB) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail)::value;
        constexpr int AHEAD = (STAGES - 2) * (AI + BI);  // loads of the stage after the next one
#pragma unroll
        for (int i = 0; i < 2 * RA; ++i) {
            const int sl = i / RA, a = i % RA, q = i & 1;
            if (i + 1 < 2 * RA) {
                fragA(cA, i + 1);
                if (i + 1 == RA) fragB(cB, 1);
            } else if (!TAIL || s + 1 < s1) {
                const bool more = !TAIL || s + STAGES < s1;
                if (more) aim();
                if (!TAIL || s + 2 < s1)
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AHEAD) : "memory");
                else
                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (more) issue(cA, cB);
                fragA(nA, 0);
                fragB(nB, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < RB; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[q], bh[sl][b], acc[a][b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < RB; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], bl[sl][b], acc[a][b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < RB; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], bh[sl][b], acc[a][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (left > 0) {
        aim();
        issue(sA1, sB1);
    }
    if (STAGES == 3 && left > 0) {
        aim();
        issue(sA2, sB2);
    }
    fragA(sA0, 0);
    fragB(sB0, 0);
    int s = s0;
    std::false_type body;
    std::true_type tail;
    if constexpr (STAGES == 3) {
        for (; s + 6 <= s1; s += 3) {
            step(body, s, sA0, sB0, sA1, sB1);
            step(body, s, sA1, sB1, sA2, sB2);
            step(body, s, sA2, sB2, sA0, sB0);
        }
        step(tail, s, sA0, sB0, sA1, sB1);
        if (s + 1 < s1) step(tail, s + 1, sA1, sB1, sA2, sB2);
        if (s + 2 < s1) step(tail, s + 2, sA2, sB2, sA0, sB0);
        if (s + 3 < s1) step(tail, s + 3, sA0, sB0, sA1, sB1);
        if (s + 4 < s1) step(tail, s + 4, sA1, sB1, sA2, sB2);
    } else {
        for (; s + 4 <= s1; s += 2) {
            step(body, s, sA0, sB0, sA1, sB1);
            step(body, s, sA1, sB1, sA0, sB0);
        }
        step(tail, s, sA0, sB0, sA1, sB1);
        if (s + 1 < s1) step(tail, s + 1, sA1, sB1, sA0, sB0);
        if (s + 2 < s1) step(tail, s + 2, sA0, sB0, sA1, sB1);
    }

    if (p.splits > 1) {
        float* o = p.part + ((int64_t)z * p.tm * BM + m0 + wm * WM) * ((int64_t)p.tn * BN) + n0 + wn * WN + fr;
#pragma unroll
        for (int a = 0; a < RA; ++a)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = a * 32 + (i >> 2) * 8 + fh * 4 + (i & 3);
#pragma unroll
                for (int b = 0; b < RB; ++b) o[(int64_t)r * p.tn * BN + b * 32] = acc[a][b][i];
            }
        return;
    }
    // the elements that the fp32 path takes: one bit for each of a lane's
    unsigned low[RA * RB] = {};
    bool look = false;
    if (watch) {
        // most waves' smallest result reaches the largest limits that they have
        float top = 0.f, topc = 0.f, least = INFINITY;
#pragma unroll
        for (int i = 0; i < WM; i += 64) top = fmaxf(top, slr[wm * WM + (i + lane) % WM]);
#pragma unroll
        for (int i = 0; i < WN; i += 64) topc = fmaxf(topc, slc[wn * WN + (i + lane) % WN]);
        top = dev::wave_max(top) + dev::wave_max(topc);
#pragma unroll
        for (int a = 0; a < RA; ++a)
#pragma unroll
            for (int b = 0; b < RB; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) least = fminf(least, fabsf(acc[a][b][i]));
        look = __any(!(least >= top));
#pragma unroll
        for (int b = 0; b < RB && look; ++b) {
            const float lc = slc[wn * WN + b * 32 + fr];
#pragma unroll
            for (int a = 0; a < RA; ++a) {
                const int rl = wm * WM + a * 32;
                unsigned m = 0;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f4 lr = *(const f4*)(slr + rl + g * 8 + fh * 4);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        m |= (unsigned)!(fabsf(acc[a][b][g * 4 + i]) >= lr[i] + lc) << (g * 4 + i);
                }
                if (!__any(m != 0)) continue;
                if (wave_usum(__builtin_popcount(m)) > kAlone) {
                    low[a * RB + b] = 0xFFFFu;
                    if (lane == 0) whole[atomicAdd(&nwhole, 1)] = (rl << 16) | (wn * WN + b * 32);
                } else if (m) {
                    low[a * RB + b] = m;
                    int at = atomicAdd(&nalone, __builtin_popcount(m));
                    for (; m; m &= m - 1) {
                        const int i = __builtin_ctz(m);
                        alone[at++] = ((rl + (i >> 2) * 8 + fh * 4 + (i & 3)) << 16) | (wn * WN + b * 32 + fr);
                    }
                }
            }
        }
    }
    auto store_all = [&](auto some) __attribute__((always_inline)) {
        constexpr bool SOME = decltype(some)::value;
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int cl = wn * WN + b * 32 + fr, col = n0 + cl;
            if (col >= p.N) continue;
            const int ec = seb[cl];
            const float bc = CONV ? 0.f : sbias[cl];
            float* cp = place<CONV>(p, m0 + wm * WM + fh * 4, col);
            const int64_t ld = CONV ? p.HWo : p.ldc;
#pragma unroll
            for (int a = 0; a < RA; ++a)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int rl = wm * WM + a * 32 + g * 8 + fh * 4;  // four rows from here
                    const int4 er = *(const int4*)(sea + rl);
                    f4 v = {__builtin_amdgcn_ldexpf(acc[a][b][g * 4], er.x + ec),
                            __builtin_amdgcn_ldexpf(acc[a][b][g * 4 + 1], er.y + ec),
                            __builtin_amdgcn_ldexpf(acc[a][b][g * 4 + 2], er.z + ec),
                            __builtin_amdgcn_ldexpf(acc[a][b][g * 4 + 3], er.w + ec)};
                    float* q = cp + (a * 32 + g * 8) * ld;
                    const int left = p.M - m0 - rl;
                    if (!CONV && p.accumulate) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] += q[min(i, max(left - 1, 0)) * ld];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i < left && !(SOME && low[a * RB + b] >> (g * 4 + i) & 1)) q[i * ld] = v[i] + (CONV ? sbias[rl + i] : bc);
                }
        }
    };
    if (look)
        store_all(std::true_type());
    else
        store_all(std::false_type());
    if (!watch) return;
    __syncthreads();
    if (nalone + nwhole == 0) return;
    float* sums = (float*)sA0;  // every fragment has been read
    for (int i = 0; i < nalone; ++i) {
        const int row = m0 + (alone[i] >> 16), col = n0 + (alone[i] & 0xFFFF);
        if (row < p.M && col < p.N) element_fp32<KIND, T>(p, row, col, sums);
    }
    for (int i = 0; i < nwhole; ++i) {
        const int row0 = m0 + (whole[i] >> 16), col0 = n0 + (whole[i] & 0xFFFF);
        if (row0 < p.M && col0 < p.N) block_fp32<KIND, T>(p, row0, col0, sums);
    }
}

// The sum of the parts of K, in their order, with the exponents, bias and C:
// one column and four rows per thread (grid: columns / 256, rows / 4).
template <Kind KIND>
__global__ __launch_bounds__(256) void k_split_sum(SplitArgs p, int BM, int BN) {
    constexpr bool CONV = KIND == kConv;
    __shared__ float sums[4];
    __shared__ uint64_t left[4][4];  // the lanes of wave w whose row i the fp32 path takes
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, row0 = blockIdx.y * 4, mine = blockIdx.x * 256 + threadIdx.x;
    const int col = min(mine, p.N - 1);
    const int64_t ld = (int64_t)p.tn * BN, plane = (int64_t)p.tm * BM * ld;
    const float* s = p.part + row0 * ld + col;  // whole tiles: rows past the matrix are there
    float v[4] = {s[0], s[ld], s[2 * ld], s[3 * ld]};
#pragma unroll 4
    for (int z = 1; z < p.splits; ++z)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += s[z * plane + i * ld];
    const int ec = p.eb[CONV ? col / p.HWo : col];
    const float lc = CONV ? p.limc[col] : limit_of(p.tb[col]);
    float* q = place<CONV>(p, row0, col);
    const int64_t ldo = CONV ? p.HWo : p.ldc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + i, at = min(row, p.M - 1), er = p.ea[at];
        const float lr = limit_of(KIND == kWeights ? (er == kBad ? kNotFinite : 0u) : p.ta[at]);
        const bool in = mine < p.N && row < p.M, low = !(fabsf(v[i]) >= lr + lc);
        if (in && !low) store<CONV>(p, row, col, q + i * ldo, __builtin_amdgcn_ldexpf(v[i], er + ec));
        const uint64_t b = __ballot(in && low);
        if (lane == 0) left[wv][i] = b;
    }
    __syncthreads();
    if (!__any(lane < 16 && left[lane >> 2 & 3][lane & 3])) return;
    for (int w = 0; w < 4; ++w)
        for (int i = 0; i < 4; ++i)
            for (uint64_t b = left[w][i]; b; b &= b - 1)
                element_fp32<KIND, 256>(p, row0 + i, (int)blockIdx.x * 256 + w * 64 + __builtin_ctzll(b), sums);
}

// ---------------------------------------------------------------------------
// Row softmax whose result is the next product's packed operand, in place:
// a row of cols scores (ld a multiple of 32) becomes ld / 32 steps of weights
// (128 bytes take the place of 32 scores), with the row's exponent; the
// arithmetic is k_softmax.hip's. One workgroup per row, eight consecutive
// values per thread and turn; every score is read before any is overwritten.
// Row r's causal mask ends at column row0 + r % period.
// ---------------------------------------------------------------------------
template <int TPB, int TURNS>
__global__ __launch_bounds__(TPB) void k_softmax_split(float* __restrict__ S, int* __restrict__ exps, int cols, int ld,
                                                      float scale, int causal, int row0, int period) {
    constexpr int W = TPB / 64;
    __shared__ float sh[2 * W];
    const int t = threadIdx.x, row = blockIdx.x;
    float* x = S + (int64_t)row * ld;
    const int valid = causal ? min(cols, row0 + row % period + 1) : cols;
    float v[TURNS][8];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < TURNS; ++j) {
        const int k = (j * TPB + t) * 8, kc = min(k, ld - 8);
        const f4 a = *(const f4*)(x + kc), b = *(const f4*)(x + kc + 4);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[j][i] = k + i < valid ? (i < 4 ? a[i & 3] : b[i & 3]) * scale : -INFINITY;
            m = fmaxf(m, v[j][i]);
        }
    }
    m = dev::wave_max(m);
    if constexpr (W > 1) {
        if ((t & 63) == 0) sh[t >> 6] = m;
        __syncthreads();
        m = sh[0];
#pragma unroll
        for (int k = 1; k < W; ++k) m = fmaxf(m, sh[k]);
    }
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < TURNS; ++j) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = expf(v[j][i] - m);
        s += ((v[j][0] + v[j][1]) + (v[j][2] + v[j][3])) + ((v[j][4] + v[j][5]) + (v[j][6] + v[j][7]));
    }
    s = dev::wave_sum(s);
    if constexpr (W > 1) {
        if ((t & 63) == 0) sh[W + (t >> 6)] = s;
        __syncthreads();
        s = sh[W];
#pragma unroll
        for (int k = 1; k < W; ++k) s += sh[W + k];
    }
    const float inv = 1.0f / s;  // the largest weight; not finite where a score is not
    const int e = exp_of(absbits(inv));
    if (t == 0) exps[row] = e;
#pragma unroll
    for (int j = 0; j < TURNS; ++j) {
        const int k = (j * TPB + t) * 8;
        if (k >= ld) continue;
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) p[i] = v[j][i] * inv;
        store_split((u16*)x + (k / kStep) * (kRowBytes / 2) + (k % kStep), p, e == kBad ? 0 : -e);
    }
}

size_t up(size_t n) { return (n + 255) / 256 * 256; }

// The tiles of k_split_mm, with what a launch of it costs on MI355X. A CU holds
// `cu` workgroups of a tile; a round of workgroups takes `full` us per step with
// every CU full, `idle` us with few workgroups, and `once` us to start and to
// store; parts of K add a launch and the traffic of their sums. The constants are
// a fit to timings of every tile with 1 to 8 parts, M and N from 64 to 262144 and
// 3 to 720 steps. Measured at the ends of the range, best tile in
// front: [4096,320] x [320,320] 14.6 us with 64 x 64, 20.0 with 128 x 128;
// conv [1,256,256,256] to 256 channels 226 us with 256 x 256, 246 with 128 x 256,
// 273 with 128 x 128; conv [2,2560,8,8] to 1280 channels 119 us with 64 x 64 in
// 8 parts, 307 in one.
struct Tile {
    int bm, bn, cu;
    float full, idle, once;
};
constexpr Tile kTiles[] = {
    {256, 256, 1, 1.52f, 1.52f, 5.6f}, {128, 256, 1, 0.90f, 0.90f, 5.3f}, {128, 128, 2, 0.88f, 0.58f, 3.5f},
    {64, 64, 3, 0.52f, 0.27f, 2.3f}};
constexpr int kParts[] = {1, 2, 3, 4, 6, 8, 12, 16};

struct Plan {
    int tile;
    int tm, tn, splits;
    int bm() const { return kTiles[tile].bm; }
    int bn() const { return kTiles[tile].bn; }
    size_t part_bytes() const { return splits > 1 ? up((size_t)splits * tm * tn * bm() * bn() * 4) : 0; }
};
Plan plan_of(int64_t M, int64_t N, int64_t steps, int64_t batches = 1) {
    Plan best{};
    double least = 0;
    for (int i = 0; i < 4; ++i) {
        const Tile& t = kTiles[i];
        const int64_t tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn, slots = (int64_t)num_cus() * t.cu;
        for (const int parts : kParts) {
            // a part has at least four steps; parts only where one round of workgroups is not full
            if (parts > 1 && (batches > 1 || steps < 4 * parts || tm * tn >= slots)) break;
            const int64_t n = tm * tn * parts * batches, rest = n % slots;
            const double k = (double)steps / parts;
            double us = (double)(n / slots) * (k * t.full + t.once);
            if (rest) us += k * (t.idle + (t.full - t.idle) * rest / slots) + t.once;
            if (parts > 1) us += 3.0 + (double)(parts + 1) * tm * t.bm * tn * t.bn * 4 / 4.4e6;
            if (least == 0 || us < least) {
                least = us;
                best = Plan{i, (int)tm, (int)tn, parts};
            }
        }
    }
    return best;
}

template <Kind KIND>
void launch_mm(const Plan& q, SplitArgs& p) {
    const unsigned grid = (unsigned)(q.tm * q.tn * q.splits * std::max(1, p.batches));
    if (q.tile == 0)
        k_split_mm<256, 256, 128, 64, 2, KIND><<<grid, 512, 0, stream()>>>(p);
    else if (q.tile == 1)
        k_split_mm<128, 256, 64, 64, 3, KIND><<<grid, 512, 0, stream()>>>(p);
    else if (q.tile == 2)
        k_split_mm<128, 128, 64, 64, 2, KIND><<<grid, 256, 0, stream()>>>(p);
    else
        k_split_mm<64, 64, 32, 32, 3, KIND><<<grid, 256, 0, stream()>>>(p);
    if (q.splits > 1)
        k_split_sum<KIND><<<dim3((unsigned)((p.N + 255) / 256), (unsigned)((p.M + 3) / 4)), 256, 0, stream()>>>(
            p, q.bm(), q.bn());
}

bool vec_rows(const PackRows& a) {
    return a.K % 4 == 0 && a.ld % 4 == 0 && a.outer_ld % 4 == 0 && a.inner_ld % 4 == 0 && aligned16(a.X);
}
// Packs a and b (of the same K; b.rows may be 0), `batches` matrices of each.
void launch_pack(const PackRows& a, const PackRows& b, int64_t batches) {
    const bool vec = vec_rows(a) && (!b.rows || vec_rows(b)), wide = a.K > 4096;
    const int turns = !vec || a.K > 16384 ? 0 : a.K > (wide ? 8192 : 2048) ? 8 : wide || a.K > 1024 ? 4 : a.K > 512 ? 2 : 1;
    const unsigned ba = blocks_for(a.rows, wide ? 1 : 4), bb = b.rows ? blocks_for(b.rows, wide ? 1 : 4) : 0;
    auto go = wide ? (turns == 8 ? k_split_pack<256, 8> : turns == 4 ? k_split_pack<256, 4> : k_split_pack<256, 0>)
                   : (turns == 8   ? k_split_pack<64, 8>
                      : turns == 4 ? k_split_pack<64, 4>
                      : turns == 2 ? k_split_pack<64, 2>
                      : turns == 1 ? k_split_pack<64, 1>
                                   : k_split_pack<64, 0>);
    go<<<dim3(ba + bb, (unsigned)batches), 256, 0, stream()>>>(a, b, (int)ba);
}

constexpr size_t kRowLds = 48 << 10;  // weights of one output channel that k_conv_prep takes through LDS
constexpr int64_t kMost = int64_t(1) << 31;

}  // namespace

// C = A B^T (+ C) (+ bias), all fp32, on the split operands. Checked arguments.
// False where the general path has to take it (scratch, or sizes past 32-bit
// offsets or one launch's grid).
bool split_gemm(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                int64_t ldc, const float* bias, bool accumulate) {
    const int64_t steps = (K + kStep - 1) / kStep;
    if (M * kRowBytes >= kMost || N * kRowBytes >= kMost || K >= kMost) return false;
    const Plan q = plan_of(M, N, steps);
    if ((int64_t)q.tm * q.tn * q.splits * 512 >= kMost) return false;
    const size_t pa = up((size_t)steps * M * kRowBytes), pb = up((size_t)steps * N * kRowBytes);
    const size_t ea = up((size_t)M * 4), eb = up((size_t)N * 4);
    char* s = (char*)try_scratch(pa + pb + 2 * (ea + eb) + q.part_bytes());
    if (!s) return false;
    SplitArgs p{};
    char* const x = s + pa + pb;
    const PackRows ra{A, lda, (u16*)s, (int*)x, (unsigned*)(x + ea + eb), (int)M, (int)K, 1, 0, 0};
    const PackRows rb{B, ldb, (u16*)(s + pa), (int*)(x + ea), (unsigned*)(x + 2 * ea + eb), (int)N, (int)K, 1, 0, 0};
    launch_pack(ra, rb, 1);
    p.A = ra.P;
    p.B = rb.P;
    p.planeA = M * kRowBytes;
    p.planeB = N * kRowBytes;
    p.rowA = kRowBytes;
    p.ea = ra.exps;
    p.eb = rb.exps;
    p.ta = ra.tails;
    p.tb = rb.tails;
    p.C = C;
    p.ldc = ldc;
    p.bias = bias;
    p.M = (int)M;
    p.N = (int)N;
    p.K = (int)K;
    p.steps = (int)steps;
    p.accumulate = accumulate ? 1 : 0;
    p.tm = q.tm;
    p.tn = q.tn;
    p.splits = q.splits;
    p.part = (float*)(x + 2 * (ea + eb));
    p.A0 = A;
    p.B0 = B;
    p.lda = lda;
    p.ldb = ldb;
    launch_mm<kDense>(q, p);
    return true;
}

// conv2d of checked arguments; false as above.
bool split_conv(const float* x, int64_t N, int64_t Cin, int64_t H, int64_t W, const float* w, int64_t Cout, int64_t kh,
                int64_t kw, const float* bias, int stride, int pad, float* out, int64_t Ho, int64_t Wo) {
    const int64_t HW = H * W, HWo = Ho * Wo, taps = kh * kw, chunks = (Cin + kStep - 1) / kStep, steps = chunks * taps;
    const int64_t cols = N * HWo;
    if (HW == 0) return false;  // outputs that see padding only
    // 32-bit offsets, also of a padded tile's first pixel
    if ((N * HW + (int64_t)pad * (W + 1) + 1) * kRowBytes >= kMost || cols >= kMost - 256 || Cout * kRowBytes >= kMost ||
        steps >= kMost || Cin * taps >= kMost || N > 65535 || N * Cin * HW >= kMost * 64)
        return false;
    // samples at a time: the exponents' table of one call of the pack is bounded
    const int64_t most = std::min(N, kTable / chunks);
    if (most == 0) return false;
    const auto plan = [&](int64_t ns) { return plan_of(Cout, ns * HWo, steps); };
    const auto grid = [](const Plan& q) { return (int64_t)q.tm * q.tn * q.splits; };
    const Plan whole = plan(most), rest = plan(N % most ? N % most : most);
    if (std::max(grid(whole), grid(rest)) * 512 >= kMost) return false;
    const int64_t prows = most * HW + 1;
    const size_t px = up((size_t)chunks * prows * kRowBytes), pw = up((size_t)steps * Cout * kRowBytes);
    const size_t mx = up((size_t)kTable * 4), tx = up((size_t)prows * 4), ex = up((size_t)most * 4);
    const size_t ew = up((size_t)Cout * 4), lc = up((size_t)most * HWo * 4);
    char* s = (char*)try_scratch(px + pw + mx + tx + ex + 2 * ew + lc + std::max(whole.part_bytes(), rest.part_bytes()));
    if (!s) return false;
    ConvPack a{};
    a.w = w;
    a.X = (u16*)s;
    a.Wp = (u16*)(s += px);
    a.maxima = (unsigned*)(s += pw);
    a.tx = (unsigned*)(s += mx);
    a.ex = (int*)(s += tx);
    a.ew = (int*)(s += ex);
    a.tw = (unsigned*)(s += ew);
    float* const limc = (float*)(s += ew);
    float* const part = (float*)(s + lc);
    a.Cin = (int)Cin;
    a.HW = (int)HW;
    a.Cout = (int)Cout;
    a.taps = (int)taps;
    a.chunks = (int)chunks;
    a.tiles = (int)((HW + 63) / 64);
    in_pieces(N, most, [&](int64_t n0, int64_t ns) {
        const Plan& q = ns == most ? whole : rest;
        a.x = x + n0 * Cin * HW;
        a.N = (int)ns;
        a.parts = 1;
        while (a.parts * 256 < HW && ns * chunks * a.parts * 2 <= kMaxima) a.parts *= 2;
        // all channels of a pixel tile in one workgroup where that leaves at least four workgroups per
        // CU, and several tiles where it leaves sixteen rounds of those
        const int64_t pt = a.tiles * ns;
        a.groups = (int)std::min<int64_t>(chunks, std::max<int64_t>(1, (4 * num_cus() + pt - 1) / pt));
        a.per = (int)((chunks + a.groups - 1) / a.groups);
        a.groups = (int)((chunks + a.per - 1) / a.per);
        a.run = (int)std::max<int64_t>(1, pt * a.groups / (64 * num_cus()));
        a.runs = (a.tiles + a.run - 1) / a.run;
        const size_t row = (size_t)(Cin * taps) * 4;
        const bool in_lds = row <= kRowLds;
        k_conv_prep<<<(unsigned)(Cout + ns * chunks * a.parts), 256, in_lds ? row : 0, stream()>>>(a, in_lds ? 1 : 0);
        k_conv_pack<<<(unsigned)(Cout + (int64_t)a.runs * a.groups * ns), 256, (size_t)(ns * chunks + chunks + ns) * 4, stream()>>>(a);
        SplitArgs p{};
        p.A = a.Wp;
        p.B = a.X;
        p.planeA = Cout * kRowBytes;
        p.planeB = (ns * HW + 1) * kRowBytes;
        p.rowA = kRowBytes;
        p.ea = a.ew;
        p.eb = a.ex;
        p.ta = a.tw;
        p.tb = a.tx;
        p.C = out + n0 * Cout * HWo;
        p.bias = bias;
        p.M = (int)Cout;
        p.N = (int)(ns * HWo);
        p.K = (int)(Cin * taps);
        p.steps = (int)steps;
        p.tm = q.tm;
        p.tn = q.tn;
        p.splits = q.splits;
        p.limc = limc;
        p.part = part;
        p.A0 = w;
        p.B0 = a.x;
        p.H = (int)H;
        p.W = (int)W;
        p.Wo = (int)Wo;
        p.HWo = (int)HWo;
        p.kh = (int)kh;
        p.kw = (int)kw;
        p.stride = stride;
        p.pad = pad;
        p.taps = (int)taps;
        p.Cin = (int)Cin;
        p.Cout = (int)Cout;
        p.zero = (int)(ns * HW);
        launch_mm<kConv>(q, p);
    });
    return true;
}

// Attention through the score matrix (backend_cuda.cu:550-586), for the head
// dimensions that the fused kernel's registers do not hold: q [N, Sq, heads d],
// k and v [N, Skv, kv_heads d], fp32, out [N, Sq, heads d] fp32 or bf16, all
// checked. Per round as many heads, or as many rows of one head, as `budget`
// bytes of scores hold: S = q k^T, the softmax, which leaves the weights as the
// packed operand of O = P v, and that product against v^T, packed once. False,
// with nothing queued, where scratch or sizes do not allow it.
bool split_attention(const float* q, const float* k, const float* v, void* out, bool out16, int64_t N, int64_t Sq,
                     int64_t Skv, int heads, int kv_heads, int64_t d, bool causal, float scale, int64_t budget) {
    const int64_t inner = heads * d, kvi = kv_heads * d, skp = (Skv + kStep - 1) / kStep * kStep;
    const int64_t dsteps = (d + kStep - 1) / kStep, ssteps = skp / kStep;
    if (skp > 32768 || Sq * kRowBytes >= kMost || N * heads > 65535) return false;
    const int group = heads / kv_heads;
    const int64_t one = Sq * skp * 4, qn = N * heads, kn = N * kv_heads;
    // heads of a round (whole samples, or groups of one sample's) and rows of a round
    int64_t nb = 1, rb = Sq;
    if (one > budget)
        rb = std::min(Sq, std::max<int64_t>(256, budget / (skp * 4) / 256 * 256));
    else if (budget / one >= heads)
        nb = std::min(qn, budget / one / heads * heads);
    else
        nb = std::max<int64_t>(1, budget / one / group * group);
    const Plan p1 = plan_of(rb, Skv, dsteps, nb), p2 = plan_of(rb, d, ssteps, nb);
    const int64_t most = std::max((int64_t)p1.tm * p1.tn * p1.splits, (int64_t)p2.tm * p2.tn * p2.splits);
    if (rb * skp * 4 >= kMost || nb * rb >= kMost / 1024 || most * nb * 512 >= kMost) return false;
    const size_t pq = up((size_t)qn * dsteps * Sq * kRowBytes), pk = up((size_t)kn * dsteps * Skv * kRowBytes);
    const size_t pv = up((size_t)kn * ssteps * d * kRowBytes), vt = up((size_t)N * kvi * Skv * 4);
    const size_t sc = up((size_t)nb * rb * skp * 4);
    const size_t eq = up((size_t)qn * Sq * 4), ek = up((size_t)kn * Skv * 4), ev = up((size_t)kn * d * 4);
    const size_t ep = up((size_t)qn * Sq * 4);  // for any round, so that the budget alone decides what a call holds
    const size_t parts = std::max(p1.part_bytes(), p2.part_bytes()), o16 = out16 ? up((size_t)N * Sq * inner * 4) : 0;
    char* s = (char*)try_scratch(pq + pk + pv + vt + sc + 2 * (eq + ek + ev) + ep + o16 + parts);
    if (!s) return false;
    auto take = [&](size_t n) {
        char* r = s;
        s += n;
        return r;
    };
    const PackRows rq{q, inner, (u16*)take(pq), (int*)take(eq), (unsigned*)take(eq), (int)Sq, (int)d, heads, Sq * inner, d};
    const PackRows rk{k, kvi, (u16*)take(pk), (int*)take(ek), (unsigned*)take(ek), (int)Skv, (int)d, kv_heads, Skv * kvi, d};
    float* const tv = (float*)take(vt);
    const PackRows rv{tv, Skv, (u16*)take(pv), (int*)take(ev), (unsigned*)take(ev), (int)d, (int)Skv, 1, d * Skv, 0};
    float* const S = (float*)take(sc);
    int* const exps = (int*)take(ep);
    float* const o = out16 ? (float*)take(o16) : (float*)out;
    transpose_device("sdh_attention", v, tv, N, Skv, kvi);
    const PackRows none{};
    if (qn == kn) {
        launch_pack(rq, rk, qn);
    } else {
        launch_pack(rq, none, qn);
        launch_pack(rk, none, kn);
    }
    launch_pack(rv, none, kn);
    auto sized = [](Plan plan, SplitArgs& p) {  // the round's plan, for p's rows
        p.tm = plan.tm = (p.M + plan.bm() - 1) / plan.bm();
        p.tn = plan.tn;
        p.splits = plan.splits;
        return plan;
    };
    int64_t b = 0;
    for (int64_t b0 = 0; b0 < qn; b0 += b) {
        const int64_t n0 = b0 / heads, h0 = b0 % heads, kb = n0 * kv_heads + h0 / group;
        b = nb >= heads ? std::min(nb, qn - b0) : std::min(nb, heads - h0);
        for (int64_t r0 = 0; r0 < Sq; r0 += rb) {
            const int64_t m = std::min(rb, Sq - r0);
            SplitArgs p{};
            p.batches = (int)b;
            p.inner = b > 1 ? heads : 1;
            p.group = b > 1 ? group : 1;
            p.kv = b > 1 ? kv_heads : 1;
            p.A = rq.P + (b0 * dsteps * Sq + r0) * (kRowBytes / 2);
            p.matA = dsteps * Sq * kRowBytes;
            p.B = rk.P + kb * dsteps * Skv * (kRowBytes / 2);
            p.matB = dsteps * Skv * kRowBytes;
            p.planeA = Sq * kRowBytes;
            p.planeB = Skv * kRowBytes;
            p.rowA = kRowBytes;
            p.ea = rq.exps + b0 * Sq + r0;
            p.eb = rk.exps + kb * Skv;
            p.ta = rq.tails + b0 * Sq + r0;
            p.tb = rk.tails + kb * Skv;
            p.C = S;
            p.ldc = skp;
            p.outC = heads * m * skp;
            p.inC = m * skp;
            p.A0 = q + (n0 * Sq + r0) * inner + h0 * d;
            p.lda = inner;
            p.outA0 = Sq * inner;
            p.inA0 = d;
            p.B0 = k + n0 * Skv * kvi + h0 / group * d;
            p.ldb = kvi;
            p.outB0 = Skv * kvi;
            p.inB0 = d;
            p.M = (int)m;
            p.N = (int)Skv;
            p.K = (int)d;
            p.steps = (int)dsteps;
            p.part = (float*)s;
            launch_mm<kDense>(sized(p1, p), p);
            auto soft = skp <= 512    ? k_softmax_split<64, 1>
                        : skp <= 2048 ? k_softmax_split<256, 1>
                        : skp <= 4096 ? k_softmax_split<512, 1>
                        : skp <= 8192 ? k_softmax_split<1024, 1>
                        : skp <= 16384 ? k_softmax_split<1024, 2>
                                       : k_softmax_split<1024, 4>;
            const unsigned tpb = skp <= 512 ? 64 : skp <= 2048 ? 256 : skp <= 4096 ? 512 : 1024;
            soft<<<(unsigned)(b * m), tpb, 0, stream()>>>(S, exps, (int)Skv, (int)skp, scale, causal ? 1 : 0, (int)r0,
                                                         (int)m);
            p.A = (const u16*)S;
            p.matA = m * skp * 4;
            p.planeA = kRowBytes;
            p.rowA = (int)(skp * 4);
            p.ea = exps;
            p.B = rv.P + kb * ssteps * d * (kRowBytes / 2);
            p.matB = ssteps * d * kRowBytes;
            p.planeB = d * kRowBytes;
            p.eb = rv.exps + kb * d;
            p.tb = rv.tails + kb * d;
            p.C = o + (n0 * Sq + r0) * inner + h0 * d;
            p.ldc = inner;
            p.outC = Sq * inner;
            p.inC = d;
            p.B0 = tv + kb * d * Skv;
            p.ldb = Skv;
            p.outB0 = kvi * Skv;
            p.inB0 = d * Skv;
            p.N = (int)d;
            p.K = (int)Skv;
            p.steps = (int)ssteps;
            p.causal = causal ? 1 : 0;
            p.row0 = (int)r0;
            launch_mm<kWeights>(sized(p2, p), p);
        }
    }
    if (out16) to_bf16_device("sdh_attention", o, (uint16_t*)out, N * Sq * inner);
    return true;
}

}  // namespace sdh
