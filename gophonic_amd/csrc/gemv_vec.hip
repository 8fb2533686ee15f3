// Multi-vector GEMV: y[v] = dequant(W) . x[v] for V input vectors that share
// one read of the weights (qwen3lm gemvQ8BVector<V>, gpu.metal:239-314, the
// decode-lane kernels of gpu_darwin.go:1121-1281), for any V up to
// kMaxVecLanes and the Q8, Q8B, Q8B_F32 and Q4 formats, with the decode
// step's prologue (PRO_NORM) and epilogues (store, residual add, SwiGLU).
//
// Design: with fp32 VALU arithmetic every extra vector costs one FMA per
// weight, so 16 lanes would be VALU-bound. Here the vectors go through MFMA:
//   * vec_prep_blocks_kernel scales each 32-value block of each vector by an
//     exact power of two 2^e (its max into [2^14, 2^15)) and splits it into
//     FP16 hi + lo parts (x*2^e = hi + lo + r, |r| <= 2^-22 |x*2^e|), laid out
//     as MFMA A fragments;
//   * vecs_kernel, or vecd_kernel for small products (vecd_rows), widens each
//     32-value block of 16 weight rows to FP16 (int8 and 4-bit codes are exact
//     in FP16), runs v_mfma_f32_16x16x32_f16 on it (products exact in fp32),
//     and folds the block result into fp32 accumulators with the weight block
//     scale and the activation block's 2^-e: acc = fma(d*2^-e, C, acc), the
//     per-block scaling of the qwen3lm kernels;
//   * K is split over wavefronts; partial sums meet in LDS in a fixed order;
//     y[v][n] = acc_hi + acc_lo (Q8: times the row scale; PRO_NORM: times
//     1/sqrt(mean(x^2) + eps) from the prep pass's block sums of squares).
// 8-bit formats with up to 16 vectors and K a multiple of 512 take
// vech_kernel (one scale per vector).
// VALU work per weight does not grow with V.
#include "common.h"

namespace gphq {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Eight codes (two dwords) to FP16, exactly: each byte b, biased to
// u = b + 128 (8-bit codes) or taken as a nibble, is placed under the FP16
// exponent of 1024 (bits 0x64uu = 1024 + u) by one v_perm_b32 per pair, and
// one packed FP16 subtraction removes 1024 + bias.
__device__ __forceinline__ f16x8 bytes_to_f16x8(uint32_t u0, uint32_t u1, _Float16 bias) {
    const f16x2 b2 = {bias, bias};
    const f16x2 p0 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u)) - b2;
    const f16x2 p1 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u)) - b2;
    const f16x2 p2 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u)) - b2;
    const f16x2 p3 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)) - b2;
    return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
__device__ __forceinline__ f16x8 i8x8_to_f16(u32x2 w) {
    return bytes_to_f16x8(w.x ^ 0x80808080u, w.y ^ 0x80808080u, (_Float16)1152.0f);
}
// Nibbles (sh = 0 low, 4 high) of eight bytes, minus 8.
__device__ __forceinline__ f16x8 u4x8_to_f16(u32x2 w, int sh) {
    return bytes_to_f16x8((w.x >> sh) & 0x0F0F0F0Fu, (w.y >> sh) & 0x0F0F0F0Fu, (_Float16)1032.0f);
}

// 2^e for |e| <= 100 and the e placing m (>= 0) in [2^14, 2^15), from the
// float's exponent bits (m = 0, NaN, Inf and denormals clamp to +-100).
__device__ __forceinline__ int pow2_exponent(float m) {
    const int biased = (int)(__builtin_bit_cast(uint32_t, m) >> 23);
    return min(max(141 - biased, -100), 100);
}
__device__ __forceinline__ float pow2f(int e) { return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23); }


enum { VEC_STORE = 0, VEC_ADD = 1, VEC_SWIGLU = 2 };

constexpr int kMaxVecLanes = 32;

// A fragments for block kb of M-tile t: 1 KiB = 64 lanes x 8 FP16; lane l
// holds A row t*16 + l%16, values kb*32 + (l/16)*8 .. +8.
__host__ __device__ inline size_t vec_a_offset(int t, int kb, int KB, int lane) {
    return ((size_t)t * KB + kb) * 512 + (size_t)lane * 8;
}

// ---- multi-vector GEMV with per-block activation scales ----------------------
// The A tiles of V vectors: 8 vectors a tile, hi and lo of vector v in rows 2v
// and 2v + 1 (mod 16); for vecs_kernel from 9 to 16 vectors a hi tile and a lo
// tile with vector v in row v (PAIR, half the result registers).
__host__ __device__ inline bool vec_pair(int V) { return V > 8 && V <= 16; }

// vec_prep_blocks_kernel: four threads per (vector v, 32-value block kb), 8
// values each. The block's values are scaled by 2^e (its max into [2^14,
// 2^15)) and split into FP16 hi + lo, written as the MFMA A fragments;
// inv[v][kb] = 2^-e and ssq[v][kb] = the block's sum of squares (for
// PRO_NORM). Every block is independent, so the pass takes one short launch
// for any vector count.
__global__ __launch_bounds__(256) void vec_prep_blocks_kernel(const float *__restrict__ x, long stride, int V, int KB,
                                                              _Float16 *__restrict__ A, float *__restrict__ inv,
                                                              float *__restrict__ ssq, bool pair) {
    const long t4 = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int gq = (int)(t4 & 3);
    const long idx = min(t4 >> 2, (long)V * KB - 1);  // the last block's extra threads repeat its work
    const int v = (int)(idx / KB), kb = (int)(idx - (long)v * KB);
    const float4 *xp = (const float4 *)(x + (size_t)v * stride + (size_t)kb * 32 + gq * 8);
    const float4 q0 = xp[0], q1 = xp[1];
    const float xs[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
    float mx = 0.0f, ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        mx = fmaxf(mx, fabsf(xs[i]));
        ss += xs[i] * xs[i];
    }
    // The block's other three quarters sit in the neighbouring lanes.
#pragma unroll
    for (int off = 1; off < 4; off <<= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
        ss += __shfl_xor(ss, off);
    }
    const int e = pow2_exponent(mx);
    const float sc = pow2f(e);
    f16x8 hi, lo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float y = xs[i] * sc;  // exact: a power-of-two scaling
        const _Float16 h = (_Float16)y;
        hi[i] = h;
        lo[i] = (_Float16)(y - (float)h);
    }
    const int th = pair ? 0 : v >> 3, tl = pair ? 1 : th;
    const int rh = pair ? v : (2 * v) & 15, rl = pair ? v : rh + 1;
    *(f16x8 *)(A + vec_a_offset(th, kb, KB, gq * 16 + rh)) = hi;
    *(f16x8 *)(A + vec_a_offset(tl, kb, KB, gq * 16 + rl)) = lo;
    if (gq == 0) {
        inv[idx] = pow2f(-e);
        ssq[idx] = ss;
    }
}

struct Vec2Args {
    const void *codes;
    const void *scales;
    const _Float16 *A;
    const float *inv;  // [V][KB]
    const float *ssq;  // [V][KB]
    float *y;
    long ystride;
    int V, K, N, KB;
    float eps;
    float *part;  // K-split stationary path: [parts][V][N] partial sums
};

// Small products over prepared A fragments, operands straight from global
// memory: each wavefront applies its A fragments to RT tiles of 16 weight rows, U blocks at a time. All U*RT*MT
// MFMAs of a step are issued before their results are scaled and summed
// (acc += d * 2^-e_v * C), which keeps the MFMA latency off the critical path.
// VALU work per weight is the code conversion (v_perm + packed FP16
// subtract). K is split over the SK wavefronts of the block; partial sums meet
// in a fixed LDS tree, and PRO_NORM's sum of squares is read from the prep
// pass's block sums in block order.
template <int FMT, int MT, int SK, int RT, int U, int EPI, bool NORM>
__global__ __launch_bounds__(64 * SK) void vecd_kernel(const Vec2Args a) {
    static_assert((SK & (SK - 1)) == 0, "SK is a power of two");
    __shared__ f32x4 red[(SK > 1 ? SK / 2 : 1) * RT * MT * 64];
    const int lane = threadIdx.x & 63;
    const int ks = threadIdx.x >> 6;
    const int g = lane >> 4, m = lane & 15;
    const int n0 = blockIdx.x * (RT * 16);
    const int KB = a.KB;
    const int per = ((KB + SK - 1) / SK + U - 1) / U * U;  // whole U-groups per wavefront
    const int kb0 = ks * per, kb1 = min(KB, kb0 + per);
    const int8_t *wrow[RT];
    const uint8_t *srow[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = min(n0 + rt * 16 + m, a.N - 1);
        wrow[rt] = FMT == GPHQ_FMT_Q4 ? (const int8_t *)a.codes + (size_t)row * (a.K >> 1) + (g & 1) * 8
                                      : (const int8_t *)a.codes + (size_t)row * a.K + g * 8;
        srow[rt] = (const uint8_t *)a.scales + (size_t)row * KB * (FMT == GPHQ_FMT_Q8B_F32 ? 4 : 2);
    }
    // The lane's C rows 4g..4g+3 of tile t are vectors t*8 + 2g (hi, lo) and t*8 + 2g + 1.
    const float *invp[MT][2];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int p = 0; p < 2; ++p) invp[t][p] = a.inv + (size_t)min(t * 8 + 2 * g + p, a.V - 1) * KB;
    f32x4 acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int kbs = kb0; kbs < kb1; kbs += U) {
        f16x8 av[U][MT];
        u32x2 w[U][RT];
        float d[U][RT], iv[U][MT][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kb = min(kbs + u, KB - 1);
            const bool ok = kbs + u < kb1;
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                av[u][t] = *(const f16x8 *)(a.A + vec_a_offset(t, kb, KB, lane));
                iv[u][t][0] = ok ? invp[t][0][kb] : 0.0f;
                iv[u][t][1] = ok ? invp[t][1][kb] : 0.0f;
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                w[u][rt] = *(const u32x2 *)(wrow[rt] + (size_t)kb * (FMT == GPHQ_FMT_Q4 ? 16 : 32));
                if constexpr (FMT == GPHQ_FMT_Q8B || FMT == GPHQ_FMT_Q4)
                    d[u][rt] = half_bits_to_float(((const uint16_t *)srow[rt])[kb]);
                else if constexpr (FMT == GPHQ_FMT_Q8B_F32)
                    d[u][rt] = ((const float *)srow[rt])[kb];
                else
                    d[u][rt] = 1.0f;
            }
        }
        f32x4 c[U][RT][MT];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const f16x8 b = FMT == GPHQ_FMT_Q4 ? u4x8_to_f16(w[u][rt], (g >> 1) * 4) : i8x8_to_f16(w[u][rt]);
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    c[u][rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[u][t], b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const float d0 = d[u][rt] * iv[u][t][0], d1 = d[u][rt] * iv[u][t][1];
                    acc[rt][t][0] = fmaf(d0, c[u][rt][t][0], acc[rt][t][0]);
                    acc[rt][t][1] = fmaf(d0, c[u][rt][t][1], acc[rt][t][1]);
                    acc[rt][t][2] = fmaf(d1, c[u][rt][t][2], acc[rt][t][2]);
                    acc[rt][t][3] = fmaf(d1, c[u][rt][t][3], acc[rt][t][3]);
                }
    }
#pragma unroll
    for (int half = SK / 2; half >= 1; half >>= 1) {
        if (ks >= half && ks < 2 * half) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < MT; ++t) red[(((ks - half) * RT + rt) * MT + t) * 64 + lane] = acc[rt][t];
        }
        __syncthreads();
        if (ks < half) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[rt][t] += red[((ks * RT + rt) * MT + t) * 64 + lane];
        }
        __syncthreads();
    }
    if (ks != 0) return;
    float nf[MT][2];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int p = 0; p < 2; ++p) nf[t][p] = 1.0f;
    if constexpr (NORM) {
        // Each vector's block sums of squares, added by the whole wavefront in
        // a fixed order; lane group g keeps vectors t*8 + 2g + {0, 1}.
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int vv = 0; vv < 8; ++vv) {
                const float *q = a.ssq + (size_t)min(t * 8 + vv, a.V - 1) * KB;
                float part = 0.0f;
                for (int kb = lane; kb < KB; kb += 64) part += q[kb];
                const float tot = wave_sum(part);
                if ((vv >> 1) == g) nf[t][vv & 1] = 1.0f / sqrtf(tot / (float)a.K + a.eps);
            }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int col = n0 + rt * 16 + m;
        float rs = 1.0f;
        if constexpr (FMT == GPHQ_FMT_Q8) rs = ((const float *)a.scales)[min(col, a.N - 1)];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int v = t * 8 + 2 * g + p;
                float val = (acc[rt][t][2 * p] + acc[rt][t][2 * p + 1]) * nf[t][p];
                if constexpr (FMT == GPHQ_FMT_Q8) val *= rs;
                if constexpr (EPI == VEC_SWIGLU) {
                    const float up = __shfl_xor(val, 1);  // lane l^1 holds column col^1
                    if (v < a.V && col < a.N && (col & 1) == 0)
                        a.y[(size_t)v * a.ystride + (col >> 1)] = val / (1.0f + expf(-val)) * up;
                } else if (v < a.V && col < a.N) {
                    if constexpr (EPI == VEC_ADD)
                        a.y[(size_t)v * a.ystride + col] += val;
                    else
                        a.y[(size_t)v * a.ystride + col] = val;
                }
            }
        }
    }
}

// How a vecs_kernel launch cuts K: `parts` passes over the block's row tiles,
// each over SK wavefronts' slices of nb 32-value blocks.
struct VecsShape {
    int iters, SK, nb, parts;
    int svec;  // block scales load as one aligned vector per lane
};

// NB: 32-value blocks per slice, at most (their A fragments stay in registers).
template <int FMT, int T, bool PAIR, int NB>
struct VecsTraits {
    static constexpr bool Q4 = FMT == GPHQ_FMT_Q4;
    // Wavefronts of a block, at most: what the registers leave per SIMD (4, 3 or 2).
    static constexpr int kMaxSK = !PAIR && T == 1 ? 16 : (PAIR ? 2 : T) * NB <= 16 ? 12 : 8;
    static constexpr int WB = Q4 ? 16 : 32;                    // code bytes per block and row
    static constexpr int STEPS = NB * WB / 128;                // 128-byte lines per row and slice
    static constexpr int SB = FMT == GPHQ_FMT_Q8 ? 0 : FMT == GPHQ_FMT_Q8B_F32 ? 4 : 2;  // scale bytes per block
    static constexpr int VC = PAIR ? 16 : 8 * T;               // vectors the tiles hold
    static constexpr int CH = T > 2 ? 2 : 4;                   // tiles whose slice sums are reduced together
    static constexpr int kStage = STEPS * 128 * 16, kScale = 16 * NB * SB, kInv = NB * VC * 4;
    static constexpr int kWave = kStage + kScale + kInv;       // LDS bytes per wavefront
    static constexpr int ch(int SK) { return SK < CH ? SK : CH; }
    static int lds(int SK, int parts, int iters) {
        return SK * kWave + (SK > 1 ? ch(SK) * SK * T * 1024 : 0) + (parts > 1 ? iters * T * 1024 : 0) +
               (VC + 3) / 4 * 16;
    }
};

// Multi-vector GEMV over prepared A fragments, any K a multiple of 32. What
// bounds it is the weight stream together with the A fragments every CU reads
// from L2 (V = 8, K = 4096: 128 KB beside 225 KB of 4-bit weights for 24576
// rows), and for 4-bit codes the VALU work of widening them (12 instructions
// per 16 x 32 codes). So each wavefront keeps its K slice's A fragments in
// registers and walks 16-row tiles over a persistent grid; weights load as
// 8 rows x 128 bytes per instruction (whole lines: 8 bytes per lane straight
// into operands touch 16 lines per instruction and were address-bound) and
// turn into B fragments through the wavefront's LDS, the next tile's loads in
// flight meanwhile. Slices meet in LDS, a few tiles at a time. K past one
// pass's slices takes further passes over the same tiles, whose sums wait in
// LDS. 8 vectors, Q4, K = 4096, N = 24576: 65.6 -> 18.5 us with its preparation
// (VALU busy 34%, 3.5 TB/s); 32 vectors 102 -> 46.4, 8 vectors at K = 12288, N =
// 4096 35.1 -> 16.4.
template <int FMT, int T, bool PAIR, int NB, int EPI, bool NORM>
__global__ __launch_bounds__((64 * VecsTraits<FMT, T, PAIR, NB>::kMaxSK)) void vecs_kernel(const Vec2Args a,
                                                                                             const VecsShape sh) {
    using X = VecsTraits<FMT, T, PAIR, NB>;
    constexpr bool Q4 = X::Q4;
    constexpr int WB = X::WB, STEPS = X::STEPS, SB = X::SB, VC = X::VC;
    constexpr int AT = PAIR ? 2 : T;     // A tiles
    constexpr int NI = PAIR ? 4 : 2;     // vectors of one result tile in a lane
    constexpr int QB = NB / 4;           // scales per lane and tile
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int ks = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int g = lane >> 4, m = lane & 15;
    const int KB = a.KB, SK = sh.SK, nb = sh.nb, iters = sh.iters, CH = X::ch(SK);
    u32x4 *const st = (u32x4 *)(smem + ks * X::kWave);
    uint8_t *const ssc = smem + ks * X::kWave + X::kStage;
    float *const siv = (float *)(ssc + X::kScale);
    f32x4 *const part = (f32x4 *)(smem + SK * X::kWave);                      // [slot][slice][T][lane]
    f32x4 *const held = part + (SK > 1 ? CH * SK * T * 64 : 0);               // [iteration][T][lane]
    float *const nf = (float *)(held + (sh.parts > 1 ? iters * T * 64 : 0));  // [VC]
    const int tiles = (a.N + 15) / 16;
    const int rowBytes = KB * WB;
    if constexpr (NORM) {
        // Each vector's block sums of squares, added by one wavefront in a fixed order.
        for (int v = ks; v < VC; v += SK) {
            const float *q = a.ssq + (size_t)min(v, a.V - 1) * KB;
            float s = 0.0f;
            for (int kb = lane; kb < KB; kb += 64) s += q[kb];
            s = wave_sum(s);
            if (lane == 0) nf[v] = 1.0f / sqrtf(s / (float)a.K + a.eps);
        }
        __syncthreads();
    }
    u32x4 R[STEPS][2];
    uint32_t S[SB ? QB : 1];
    int kb0 = 0;
    auto gload = [&](int t2) {
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
            const int mm = h2 * 8 + (lane >> 3);
            const int c = (lane & 7) ^ (mm >> 1);
            const int row = min(t2 * 16 + mm, a.N - 1);
            const uint8_t *src = (const uint8_t *)a.codes + (size_t)row * rowBytes;
#pragma unroll
            for (int s = 0; s < STEPS; ++s)  // past the row's end: its last chunk, times a zero activation
                R[s][h2] = __builtin_nontemporal_load(
                    (const u32x4 *)(src + min(kb0 * WB + s * 128 + c * 16, rowBytes - 16)));
        }
        if constexpr (SB > 0) {
            // Lane l: row l / 4, QB blocks from (l % 4) QB.
            const size_t base = (size_t)min(t2 * 16 + (lane >> 2), a.N - 1) * KB;
            const int kq = kb0 + (lane & 3) * QB;
            if (sh.svec) {
                const uint8_t *p = (const uint8_t *)a.scales + (base + min(kq, KB - QB)) * SB;
                if constexpr (QB * SB == 16) {
                    const u32x4 w = *(const u32x4 *)p;
                    S[0] = w.x, S[1] = w.y, S[2] = w.z, S[3] = w.w;
                } else if constexpr (QB * SB == 8) {
                    const u32x2 w = *(const u32x2 *)p;
                    S[0] = w.x, S[1] = w.y;
                } else {
                    S[0] = *(const uint32_t *)p;
                }
            } else if constexpr (SB == 4) {
#pragma unroll
                for (int i = 0; i < QB; ++i) S[i] = ((const uint32_t *)a.scales)[base + min(kq + i, KB - 1)];
            } else {
#pragma unroll
                for (int i = 0; i < QB; i += 2) {
                    const uint32_t lo = ((const uint16_t *)a.scales)[base + min(kq + i, KB - 1)];
                    const uint32_t hi = ((const uint16_t *)a.scales)[base + min(kq + i + 1, KB - 1)];
                    S[i / 2] = lo | hi << 16;
                }
            }
        }
    };
    auto lwrite = [&]() {
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) st[s * 128 + h2 * 64 + lane] = R[s][h2];
        if constexpr (SB > 0) {
            uint8_t *d = ssc + ((lane >> 2) * NB + (lane & 3) * QB) * SB;
#pragma unroll
            for (int i = 0; i < QB * SB / 4; ++i) {
                // Blocks past K scale by 0 (their codes are another block's).
                const int kb = kb0 + (lane & 3) * QB + i * (4 / (SB ? SB : 1));
                uint32_t w = S[i];
                if (SB == 4) w = kb < KB ? w : 0;
                else w = kb + 1 < KB ? w : kb < KB ? w & 0xFFFFu : 0;
                __builtin_memcpy(d + 4 * i, &w, 4);
            }
        }
    };
    for (int part_i = 0; part_i < sh.parts; ++part_i) {
        kb0 = min((part_i * SK + ks) * nb, KB);
        const int mine = min(nb, KB - kb0);  // blocks of this slice (0: none left)
        int tt = blockIdx.x;
        gload(tt);
        // All of the slice's activation loads are issued before the first is used.
        constexpr int IV = NB * VC / 64;  // block factors per lane
        static_assert(IV * 64 == NB * VC, "whole wavefronts of block factors");
        float iv[IV];
#pragma unroll
        for (int i = 0; i < IV; ++i) {
            const int b = (lane + 64 * i) / VC, v = (lane + 64 * i) % VC;
            iv[i] = a.inv[(size_t)min(v, a.V - 1) * KB + min(kb0 + b, KB - 1)];
        }
        f16x8 av[NB][AT];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int t = 0; t < AT; ++t) {
                if (b < mine) av[b][t] = *(const f16x8 *)(a.A + vec_a_offset(t, kb0 + b, KB, lane));
                else av[b][t] = f16x8{};
            }
#pragma unroll
        for (int i = 0; i < IV; ++i) siv[lane + 64 * i] = (lane + 64 * i) / VC < mine ? iv[i] : 0.0f;
        lwrite();
        for (int it = 0; it < iters; ++it, tt += gridDim.x) {
            const bool more = it + 1 < iters;
            if (more) gload(tt + gridDim.x);  // past the last tile: its last row again
            f32x4 acc[T];
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            uint32_t sw[SB ? NB * SB / 4 : 1];  // the scales of this lane's row
            if constexpr (SB > 0) __builtin_memcpy(sw, __builtin_assume_aligned(ssc + m * NB * SB, 8), NB * SB);
#pragma unroll
            for (int b4 = 0; b4 < NB; b4 += 4) {
                if (b4 >= mine) break;
#pragma unroll
                for (int b = b4; b < b4 + 4; ++b) {
                    constexpr int PER = 128 / WB;  // blocks per line
                    const int c = Q4 ? b % PER : 2 * (b % PER) + (g >> 1);
                    const u32x2 wv = *(const u32x2 *)((const uint32_t *)(st + (b / PER) * 128 + m * 8 + (c ^ (m >> 1))) +
                                                      (g & 1) * 2);
                    const f16x8 bf = Q4 ? u4x8_to_f16(wv, (g >> 1) * 4) : i8x8_to_f16(wv);
                    float d = 1.0f;
                    if constexpr (SB == 2) d = half_bits_to_float((uint16_t)((b & 1) ? sw[b / 2] >> 16 : sw[b / 2]));
                    else if constexpr (SB == 4) d = __builtin_bit_cast(float, sw[b]);
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        const f32x4 zero{0.f, 0.f, 0.f, 0.f};
                        f32x4 cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[b][t], bf, zero, 0, 0, 0);
                        // Added outside: an MFMA with a sum to start from rounds worse.
                        if constexpr (PAIR) cc += __builtin_amdgcn_mfma_f32_16x16x32_f16(av[b][1], bf, zero, 0, 0, 0);
                        const float *iv = siv + b * VC + (PAIR ? 4 * g : 8 * t + 2 * g);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float f = iv[PAIR ? i : i >> 1];
                            acc[t][i] = fmaf(SB ? d * f : f, cc[i], acc[t][i]);
                        }
                    }
                }
            }
            if (more) lwrite();  // after this tile's LDS reads (LDS operations of a wavefront run in order)
            // Result i of lane (g, m): row tile * 16 + m; PAIR: vector 4g + i; else
            // hi and lo of vector 8t + 2g + i/2.
            auto epilogue = [&](int ti, int tile, f32x4 (&r)[T]) {
                if (part_i) {
#pragma unroll
                    for (int t = 0; t < T; ++t) r[t] = held[(ti * T + t) * 64 + lane] + r[t];
                }
                if (part_i + 1 < sh.parts) {
#pragma unroll
                    for (int t = 0; t < T; ++t) held[(ti * T + t) * 64 + lane] = r[t];
                    return;
                }
                if (tile >= tiles) return;
                const int col = tile * 16 + m;
                float rs = 1.0f;
                if constexpr (FMT == GPHQ_FMT_Q8) rs = ((const float *)a.scales)[min(col, a.N - 1)];
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int i = 0; i < NI; ++i) {
                        const int v = PAIR ? 4 * g + i : 8 * t + 2 * g + i;
                        float val = PAIR ? r[t][i] : r[t][2 * i] + r[t][2 * i + 1];
                        if constexpr (NORM) val *= nf[v];
                        if constexpr (FMT == GPHQ_FMT_Q8) val *= rs;
                        if constexpr (EPI == VEC_SWIGLU) {
                            const float up = __shfl_xor(val, 1);  // lane m^1 holds column col^1
                            if (v < a.V && col < a.N && (col & 1) == 0)
                                a.y[(size_t)v * a.ystride + (col >> 1)] = val / (1.0f + expf(-val)) * up;
                        } else if (v < a.V && col < a.N) {
                            if constexpr (EPI == VEC_ADD)
                                a.y[(size_t)v * a.ystride + col] += val;
                            else
                                a.y[(size_t)v * a.ystride + col] = val;
                        }
                    }
            };
            if (SK == 1) {
                epilogue(it, tt, acc);
                continue;
            }
            const int slot = it % CH;
#pragma unroll
            for (int t = 0; t < T; ++t) part[((slot * SK + ks) * T + t) * 64 + lane] = acc[t];
            if (slot != CH - 1 && it != iters - 1) continue;  // the same for every wavefront
            __syncthreads();
            if (ks <= slot) {
                // Wavefront ks adds slot ks's slices (T == 1: the even and the
                // odd ones apart): the tile slot - ks blocks back.
                f32x4 r[T];
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const f32x4 *ps = part + (ks * SK * T + t) * 64 + lane;
                    r[t] = ps[0];
                    if constexpr (T == 1) {
                        f32x4 odd = ps[64];
                        for (int k2 = 2; k2 < SK; k2 += 2) {
                            r[t] += ps[k2 * 64];
                            if (k2 + 1 < SK) odd += ps[(k2 + 1) * 64];
                        }
                        r[t] += odd;
                    } else {
                        for (int k2 = 1; k2 < SK; ++k2) r[t] += ps[k2 * T * 64];
                    }
                }
                epilogue(it - (slot - ks), tt - (slot - ks) * (int)gridDim.x, r);
            }
            __syncthreads();
        }
    }
}

// K = 0: every product is an empty sum.
template <int FMT>
__global__ __launch_bounds__(256) void vec_empty_kernel(const Vec2Args a, bool store) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)a.V * a.N || !store) return;
    const int v = (int)(idx / a.N), col = (int)(idx - (long)v * a.N);
    a.y[(size_t)v * a.ystride + col] = FMT == GPHQ_FMT_Q8 ? 0.0f * ((const float *)a.scales)[col] : 0.0f;
}

// ---- stationary activations: up to 16 vectors, 8-bit formats -------------------
// For V <= 16 vectors and K a multiple of 512 up to 4096 the activations stay
// in registers and the weights are transposed through LDS:
//   * vech_prep_kernel (one block per A row, 16 blocks, x read once) scales
//     each vector by one power of two 2^e (its max into [2^14, 2^15)) and
//     splits it into
//     FP16 hi + lo, as two 16-row A tiles (tile 0 hi, tile 1 lo; row v =
//     vector v, rows past V zero). Against the per-block split above, values
//     smaller than 2^-17 of the vector's maximum lose relative precision, but
//     their error stays below 2^-38 max|x| per product;
//   * vech_kernel: each wavefront of a block owns one K slice of 16 blocks and
//     keeps that slice's A fragments (hi and lo) in registers for the whole
//     launch. It walks 16-row tiles (persistent grid): weights are loaded as
//     8 rows x 128 bytes per instruction (whole cache lines; lane l of row
//     r takes 16-byte chunk (l & 7) ^ (r >> 1)), written to the wavefront's
//     LDS region and read back as MFMA B fragments (slot m*8 + (c ^ (m >> 1))
//     is bank-conflict free), while the next tile's loads are in flight. Per
//     block: hi and lo MFMAs accumulate into one 16x16 result (16 vectors x
//     16 rows), scaled by the weight block scale into fp32 accumulators; the
//     K slices meet in LDS in slice order. Each wavefront parks a tile's
//     partial sums in one of kVechCH LDS slots and moves on; every kVechCH
//     tiles one barrier pair lets wavefront w add up slot w's slices and run
//     that tile's epilogue, instead of two barriers and a one-wavefront
//     epilogue per tile.
// Measured on MI355X with 16 vectors (Qwen3-8B shapes, Q8B): the head 154 us
// (was 383 us with the per-block kernel), gate/up 34 us (was 83), qkv 16.5 us
// (was 33), o 13 us (was 20).
constexpr int kVechNB = 16;        // K blocks of 32 values per wavefront slice
constexpr int kVechMaxSlices = 8;  // 512 threads; the kernel holds ~230 VGPRs
constexpr int kVechCH = 8;         // tiles whose slice sums are reduced together

// One block of 1024 threads per vector; thread t holds float4 units t, t +
// 1024, .. of the vector (K <= 4 * 1024 * kPrepUnits), so the vector is read
// once: the maximum and the sum of squares come from registers, and the same
// registers are split into hi and lo.
constexpr int kPrepUnits = 8;
__global__ __launch_bounds__(1024) void vech_prep_kernel(const float *__restrict__ x, long stride, int V, int K,
                                                         _Float16 *__restrict__ A, float *__restrict__ inv,
                                                         float *__restrict__ ssq, const VecFold f) {
    typedef _Float16 f16x4v __attribute__((ext_vector_type(4)));
    __shared__ float red[2][16];
    const int v = blockIdx.x;  // 16 blocks; rows v >= V are written as zero
    const bool live = v < V;
    const float *xv = x + (size_t)min(v, V - 1) * stride;
    const int U = K / 4;
    float4 q[kPrepUnits];
#pragma unroll
    for (int j = 0; j < kPrepUnits; ++j) {
        const int u = threadIdx.x + j * 1024;
        q[j] = (live && u < U) ? *(const float4 *)(xv + 4 * u) : float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (f.parts) {
        // The pending residual add of a K-split GEMV: x += (sum of its parts
        // in order) * its vector scale (* the Q8 row scale), in
        // vech_finish_kernel's order, written back to x.
        const float pinv = live ? f.inv[v] : 0.0f;
#pragma unroll
        for (int j = 0; j < kPrepUnits; ++j) {
            const int u = threadIdx.x + j * 1024;
            if (!live || u >= U) continue;
            float4 sum = float4{0.0f, 0.0f, 0.0f, 0.0f};
            for (int pp = 0; pp < f.parts; ++pp) {
                const float4 t = *(const float4 *)(f.part + ((size_t)pp * V + v) * K + 4 * u);
                sum.x += t.x, sum.y += t.y, sum.z += t.z, sum.w += t.w;
            }
            float4 val{__fmul_rn(sum.x, pinv), __fmul_rn(sum.y, pinv), __fmul_rn(sum.z, pinv), __fmul_rn(sum.w, pinv)};
            if (f.rowScale) {
                const float4 rs = *(const float4 *)(f.rowScale + 4 * u);
                val = float4{__fmul_rn(val.x, rs.x), __fmul_rn(val.y, rs.y), __fmul_rn(val.z, rs.z), __fmul_rn(val.w, rs.w)};
            }
            q[j] = float4{__fadd_rn(q[j].x, val.x), __fadd_rn(q[j].y, val.y), __fadd_rn(q[j].z, val.z),
                          __fadd_rn(q[j].w, val.w)};
            *(float4 *)(const_cast<float *>(xv) + 4 * u) = q[j];
        }
    }
    float mx = 0.0f, ss = 0.0f;
#pragma unroll
    for (int j = 0; j < kPrepUnits; ++j) {
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(q[j].x), fabsf(q[j].y)), fmaxf(fabsf(q[j].z), fabsf(q[j].w))));
        ss += q[j].x * q[j].x + q[j].y * q[j].y + q[j].z * q[j].z + q[j].w * q[j].w;
    }
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[0][threadIdx.x >> 6] = mx, red[1][threadIdx.x >> 6] = ss;
    __syncthreads();
    mx = red[0][0];
#pragma unroll
    for (int w = 1; w < 16; ++w) mx = fmaxf(mx, red[0][w]);
    const int e = pow2_exponent(mx);
    const float sc = live ? pow2f(e) : 0.0f;
    const int KB = K / 32;
#pragma unroll
    for (int j = 0; j < kPrepUnits; ++j) {
        const int u = threadIdx.x + j * 1024;
        if (u >= U) break;
        // Unit u: block u / 8, 8-value group (u % 8) / 2, half u % 2.
        const int kb = u >> 3, gq = (u >> 1) & 3, half = u & 1;
        const float xs[4] = {q[j].x, q[j].y, q[j].z, q[j].w};
        f16x4v hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float y = xs[i] * sc;  // exact: a power-of-two scaling (or zero)
            const _Float16 h = (_Float16)y;
            hi[i] = h;
            lo[i] = (_Float16)(y - (float)h);
        }
        *(f16x4v *)(A + vec_a_offset(0, kb, KB, gq * 16 + v) + half * 4) = hi;
        *(f16x4v *)(A + vec_a_offset(1, kb, KB, gq * 16 + v) + half * 4) = lo;
    }
    if (threadIdx.x == 0 && live) {
        inv[v] = pow2f(-e);
        float t = red[1][0];
#pragma unroll
        for (int w = 1; w < 16; ++w) t += red[1][w];
        ssq[v] = t;
    }
}

template <int FMT, int SK, int EPI, bool NORM, bool SPLIT>
__global__ __launch_bounds__(64 * SK) void vech_kernel(const Vec2Args a, int iters) {
    constexpr int NB = kVechNB, STEPS = NB / 4;
    // Scale bytes per row and slice in 16-byte loads (Q8's row scale is applied at the end).
    constexpr int SC = FMT == GPHQ_FMT_Q8B ? NB * 2 / 16 : FMT == GPHQ_FMT_Q8B_F32 ? NB * 4 / 16 : 1;
    __shared__ u32x4 stage[SK][STEPS * 128];
    constexpr int CH = SK < kVechCH ? SK : kVechCH;
    __shared__ f32x4 part[SK > 1 ? CH * SK * 64 : 1];  // [slot][slice][lane]
    const int lane = threadIdx.x & 63;
    const int ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, m = lane & 15;
    const int KB = a.KB;
    // SPLIT: blockIdx.y picks which SK slices of K this block holds.
    const int kb0 = ((SPLIT ? (int)blockIdx.y * SK : 0) + ks) * NB;
    const int tiles = (a.N + 15) / 16;
    u32x4 *st = stage[ks];
    u32x4 R[STEPS][2];
    uint32_t S[SC * 4], Sn[SC * 4];  // the slice's block scales of this lane's row, as words
    auto gload = [&](int t2, uint32_t (&sd)[SC * 4]) {
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
            const int mm = h2 * 8 + (lane >> 3);
            const int c = (lane & 7) ^ (mm >> 1);
            const int row = min(t2 * 16 + mm, a.N - 1);
            const int8_t *src = (const int8_t *)a.codes + (size_t)row * a.K + kb0 * 32 + c * 16;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) R[s][h2] = __builtin_nontemporal_load((const u32x4 *)(src + s * 128));
        }
        if constexpr (FMT != GPHQ_FMT_Q8) {
            const int row = min(t2 * 16 + m, a.N - 1);
            const uint8_t *sr = (const uint8_t *)a.scales + ((size_t)row * KB + kb0) * (FMT == GPHQ_FMT_Q8B ? 2 : 4);
#pragma unroll
            for (int q = 0; q < SC; ++q) {
                const u32x4 w4 = *(const u32x4 *)(sr + q * 16);
                sd[4 * q] = w4.x, sd[4 * q + 1] = w4.y, sd[4 * q + 2] = w4.z, sd[4 * q + 3] = w4.w;
            }
        }
    };
    auto lwrite = [&]() {
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) st[s * 128 + h2 * 64 + lane] = R[s][h2];
    };
    int tt = blockIdx.x;
    if (tt < tiles) {
        gload(tt, S);
        lwrite();
    }
    f16x8 ah[NB], al[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        ah[b] = *(const f16x8 *)(a.A + vec_a_offset(0, kb0 + b, KB, lane));
        al[b] = *(const f16x8 *)(a.A + vec_a_offset(1, kb0 + b, KB, lane));
    }
    // The scale of each of the lane's 4 vectors (with the RMSNorm factor),
    // read once: read in the epilogue, each would wait for the previous
    // tile's stores as well.
    float vscale[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int vc = min(4 * g + i, a.V - 1);
        vscale[i] = a.inv[vc];
        if constexpr (NORM) vscale[i] = vscale[i] * (1.0f / sqrtf(a.ssq[vc] / (float)a.K + a.eps));
    }
    for (int it = 0; it < iters; ++it, tt += gridDim.x) {
        const bool valid = tt < tiles;
        const bool more = tt + (int)gridDim.x < tiles;
        if (more) gload(tt + gridDim.x, Sn);
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        if (valid) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int c = 2 * (b & 3) + (g >> 1);
                const u32x2 wv =
                    *(const u32x2 *)((const uint32_t *)(st + (b >> 2) * 128 + m * 8 + (c ^ (m >> 1))) + (g & 1) * 2);
                float d = 1.0f;
                if constexpr (FMT == GPHQ_FMT_Q8B) {
                    const uint32_t sw = S[b / 2];
                    d = half_bits_to_float((uint16_t)((b & 1) ? sw >> 16 : sw));
                } else if constexpr (FMT == GPHQ_FMT_Q8B_F32) {
                    d = __builtin_bit_cast(float, S[b]);
                }
                const f16x8 bf = i8x8_to_f16(wv);
                f32x4 cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[b], bf, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                cc = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[b], bf, cc, 0, 0, 0);
                if constexpr (FMT == GPHQ_FMT_Q8) {
                    acc += cc;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = fmaf(d, cc[i], acc[i]);
                }
            }
        }
        if (more) {
            lwrite();  // after this tile's LDS reads (LDS operations of a wavefront run in order)
#pragma unroll
            for (int q = 0; q < SC * 4; ++q) S[q] = Sn[q];
        }
        // Lane (g, m) holds vectors 4g..4g+3 of row t*16 + m.
        auto epilogue = [&](int t, const f32x4 &r) {
            const int col = t * 16 + m;
            if constexpr (SPLIT) {  // this part's sums; vech_finish_kernel applies the rest
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int v = 4 * g + i;
                    if (v < a.V && col < a.N) a.part[((size_t)blockIdx.y * a.V + v) * a.N + col] = r[i];
                }
                return;
            }
            float rs = 1.0f;
            if constexpr (FMT == GPHQ_FMT_Q8) rs = ((const float *)a.scales)[min(col, a.N - 1)];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int v = 4 * g + i;
                // inv is a power of two, so r * (inv * f) rounds like (r * inv) * f.
                float val = r[i] * vscale[i];
                if constexpr (FMT == GPHQ_FMT_Q8) val *= rs;
                if constexpr (EPI == VEC_SWIGLU) {
                    const float up = __shfl_xor(val, 1);  // lane m^1 holds row col^1
                    if (v < a.V && col < a.N && (col & 1) == 0)
                        a.y[(size_t)v * a.ystride + (col >> 1)] = val / (1.0f + expf(-val)) * up;
                } else if (v < a.V && col < a.N) {
                    if constexpr (EPI == VEC_ADD)
                        a.y[(size_t)v * a.ystride + col] += val;
                    else
                        a.y[(size_t)v * a.ystride + col] = val;
                }
            }
        };
        if constexpr (SK > 1) {
            const int slot = it % CH;
            part[(slot * SK + ks) * 64 + lane] = acc;
            if (slot != CH - 1 && it != iters - 1) continue;  // the same for every wavefront
            __syncthreads();
            if (ks <= slot) {
                // Wavefront ks reduces slot ks (tile tt - (slot - ks) blocks
                // back) in slice order, as one wavefront adding the others'.
                const f32x4 *ps = part + ks * SK * 64 + lane;
                f32x4 r = ps[0];
                for (int k2 = 1; k2 < SK; ++k2) r += ps[k2 * 64];
                const int t = tt - (slot - ks) * (int)gridDim.x;
                if (t < tiles) epilogue(t, r);
            }
            __syncthreads();
        } else {
            if (!valid) break;
            epilogue(tt, acc);
        }
    }
}

// The K-split stationary path's finish: thread (v, row) sums the parts in
// order, then applies the vector's scale, the norm, the Q8 row scale and the
// epilogue as vech_kernel does (SwiGLU: one thread per row pair).
template <int FMT, int EPI, bool NORM>
__global__ __launch_bounds__(256) void vech_finish_kernel(const Vec2Args a, int parts) {
    const int per = EPI == VEC_SWIGLU ? a.N / 2 : a.N;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.V * per) return;
    const int v = idx / per, r = idx - v * per;
    auto row_value = [&](int col) {
        float sum = 0.0f;
        for (int p = 0; p < parts; ++p) sum += a.part[((size_t)p * a.V + v) * a.N + col];
        float val = __fmul_rn(sum, a.inv[v]);
        if constexpr (NORM) val = __fmul_rn(val, 1.0f / sqrtf(a.ssq[v] / (float)a.K + a.eps));
        if constexpr (FMT == GPHQ_FMT_Q8) val = __fmul_rn(val, ((const float *)a.scales)[col]);
        return val;
    };
    if constexpr (EPI == VEC_SWIGLU) {
        const float gate = row_value(2 * r), up = row_value(2 * r + 1);
        a.y[(size_t)v * a.ystride + r] = gate / (1.0f + expf(-gate)) * up;
    } else if constexpr (EPI == VEC_ADD) {
        float *yp = a.y + (size_t)v * a.ystride + r;
        *yp = __fadd_rn(*yp, row_value(r));  // the same rounding as a folded add (vech_prep_kernel)
    } else {
        a.y[(size_t)v * a.ystride + r] = row_value(r);
    }
}

// Whether the stationary-activation kernel takes this GEMV.
static bool vech_takes(int fmt, int V, int K) {
    return fmt != GPHQ_FMT_Q4 && V >= 1 && V <= 16 && K % (32 * kVechNB) == 0 &&
           K / (32 * kVechNB) <= kVechMaxSlices;
}

// K parts of the split stationary path (K above one block's kVechMaxSlices
// slices, split evenly), or 0 when it does not apply.
static int vech_split_parts(int fmt, int V, int K) {
    if (fmt == GPHQ_FMT_Q4 || V < 1 || V > 16 || K % (32 * kVechNB)) return 0;
    const int slices = K / (32 * kVechNB);
    if (slices <= kVechMaxSlices) return 0;
    const int parts = (slices + kVechMaxSlices - 1) / kVechMaxSlices;
    return slices % parts == 0 && parts <= 8 && K <= 4 * 1024 * kPrepUnits ? parts : 0;
}

size_t gemv_vec_split_bytes(int V, int K, int N) {
    const int parts = vech_split_parts(GPHQ_FMT_Q8B, V, K);
    return parts ? (size_t)parts * V * N * 4 : 0;
}

template <int FMT, int SK, int EPI, bool NORM>
static int go_vech(const Vec2Args &a, hipStream_t stream) {
    const int tiles = (a.N + 15) / 16;
    const int perCu = std::max(1, 8 / SK);  // about 8 wavefronts per CU
    const int blocks = std::max(1, std::min(tiles, device_cus() * perCu));
    const int iters = (tiles + blocks - 1) / blocks;
    hipLaunchKernelGGL((vech_kernel<FMT, SK, EPI, NORM, false>), dim3((unsigned)blocks), dim3(64 * SK), 0, stream, a,
                       iters);
    return launch_status();
}

// K-split stationary path: blocks of kVechMaxSlices slices, one grid row per
// K part (about 8 wavefronts per CU in all), then the ordered finish.
template <int FMT, int EPI, bool NORM>
static int go_vech_split(const Vec2Args &a, int parts, hipStream_t stream, bool finish) {
    constexpr int SK = kVechMaxSlices;
    const int tiles = (a.N + 15) / 16;
    const int blocks = std::max(1, std::min(tiles, device_cus() / parts));
    const int iters = (tiles + blocks - 1) / blocks;
    hipLaunchKernelGGL((vech_kernel<FMT, SK, VEC_STORE, false, true>), dim3((unsigned)blocks, (unsigned)parts),
                       dim3(64 * SK), 0, stream, a, iters);
    GPHQ_TRY(launch_status());
    if (!finish) return GPHQ_OK;  // the next preparation adds the parts (VecFold)
    const int per = EPI == VEC_SWIGLU ? a.N / 2 : a.N;
    hipLaunchKernelGGL((vech_finish_kernel<FMT, EPI, NORM>), dim3((unsigned)((a.V * per + 255) / 256)), dim3(256), 0,
                       stream, a, parts);
    return launch_status();
}

template <int EPI, bool NORM>
static int launch_vech_split(int fmt, const Vec2Args &a, int parts, hipStream_t stream, bool finish = true) {
    switch (fmt) {
    case GPHQ_FMT_Q8: return go_vech_split<GPHQ_FMT_Q8, EPI, NORM>(a, parts, stream, finish);
    case GPHQ_FMT_Q8B: return go_vech_split<GPHQ_FMT_Q8B, EPI, NORM>(a, parts, stream, finish);
    case GPHQ_FMT_Q8B_F32: return go_vech_split<GPHQ_FMT_Q8B_F32, EPI, NORM>(a, parts, stream, finish);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

template <int FMT, int EPI, bool NORM>
static int launch_vech_sk(const Vec2Args &a, hipStream_t stream) {
    switch (a.K / (32 * kVechNB)) {
    case 1: return go_vech<FMT, 1, EPI, NORM>(a, stream);
    case 2: return go_vech<FMT, 2, EPI, NORM>(a, stream);
    case 3: return go_vech<FMT, 3, EPI, NORM>(a, stream);
    case 4: return go_vech<FMT, 4, EPI, NORM>(a, stream);
    case 5: return go_vech<FMT, 5, EPI, NORM>(a, stream);
    case 6: return go_vech<FMT, 6, EPI, NORM>(a, stream);
    case 7: return go_vech<FMT, 7, EPI, NORM>(a, stream);
    case 8: return go_vech<FMT, 8, EPI, NORM>(a, stream);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

template <int EPI, bool NORM>
static int launch_vech(int fmt, const Vec2Args &a, hipStream_t stream) {
    switch (fmt) {
    case GPHQ_FMT_Q8: return launch_vech_sk<GPHQ_FMT_Q8, EPI, NORM>(a, stream);
    case GPHQ_FMT_Q8B: return launch_vech_sk<GPHQ_FMT_Q8B, EPI, NORM>(a, stream);
    case GPHQ_FMT_Q8B_F32: return launch_vech_sk<GPHQ_FMT_Q8B_F32, EPI, NORM>(a, stream);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

size_t gemv_vec_workspace_bytes(int V, int K) {
    const int MT = std::max(2, (2 * V + 15) / 16);  // the stationary path uses two tiles
    const int KB = (K + 31) / 32;
    return (size_t)MT * KB * 1024 + 2 * (size_t)V * KB * 4 + 256;
}

// The slices of K: as few passes as hold KB blocks, each over as few wavefronts
// as hold a pass's share (twice the wavefronts at half the blocks each took
// 8 vectors, K = 1376, N = 24000, Q8B 17.7 us, 14.4 with this), or as many more
// as leave as many blocks on a CU (16 vectors, K = 4128, N = 20000, Q8B, six
// slices of 12 blocks instead of five of 16: 46.7 -> 44.5 us). Where the tiles'
// sums of a further pass would not fit in LDS, more blocks walk fewer tiles.
template <int FMT, int T, bool PAIR, int NB, int EPI, bool NORM>
static int go_vecs(const Vec2Args &a, hipStream_t stream) {
    using X = VecsTraits<FMT, T, PAIR, NB>;
    constexpr int kMaxSK = X::kMaxSK, kLds = 160 << 10;
    VecsShape sh{};
    sh.parts = (a.KB + kMaxSK * NB - 1) / (kMaxSK * NB);
    const int per = (a.KB + sh.parts - 1) / sh.parts;  // blocks of one pass
    const int line = X::Q4 ? 8 : 4;  // blocks per 128-byte line
    constexpr int kWaves = T == 1 && !PAIR ? kMaxSK : 8;  // wavefronts per CU
    const int least = (per + NB - 1) / NB, perCu = std::max(1, kWaves / least);
    sh.nb = std::min(NB, ((per + kWaves / perCu - 1) / (kWaves / perCu) + line - 1) / line * line);
    if (least > kWaves) sh.nb = NB;
    sh.SK = (per + sh.nb - 1) / sh.nb;
    sh.svec = X::SB && a.KB % 4 == 0 && (uintptr_t)a.scales % 16 == 0;
    const int tiles = (a.N + 15) / 16;
    int blocks = std::max(1, std::min(tiles, device_cus() * perCu));
    sh.iters = (tiles + blocks - 1) / blocks;
    const int room = (kLds - X::lds(sh.SK, 1, 0)) / (T * 1024);
    if (sh.parts > 1 && sh.iters > room) sh.iters = room;
    blocks = (tiles + sh.iters - 1) / sh.iters;
    const int lds = X::lds(sh.SK, sh.parts, sh.iters);
    if (lds > (64 << 10))
        GPHQ_TRY(hip_status(hipFuncSetAttribute((const void *)vecs_kernel<FMT, T, PAIR, NB, EPI, NORM>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, lds)));
    hipLaunchKernelGGL((vecs_kernel<FMT, T, PAIR, NB, EPI, NORM>), dim3((unsigned)blocks), dim3(64 * sh.SK), lds, stream,
                       a, sh);
    return launch_status();
}

template <int FMT, int EPI, bool NORM>
static int launch_vecs_tiles(const Vec2Args &a, hipStream_t stream) {
    if (vec_pair(a.V)) {
        // Slices of 8 blocks leave three wavefronts per SIMD instead of two but
        // hold K <= 3072 in one pass; a second pass costs more than they gain
        // (V = 9, K = 1984, N = 17374, Q8: 19.3 us with 16 blocks, 15.9 with 8).
        return a.KB <= 96 ? go_vecs<FMT, 1, true, 8, EPI, NORM>(a, stream)
                          : go_vecs<FMT, 1, true, 16, EPI, NORM>(a, stream);
    }
    switch ((a.V + 7) / 8) {
    case 1: return go_vecs<FMT, 1, false, 8, EPI, NORM>(a, stream);
    case 3: return go_vecs<FMT, 3, false, 8, EPI, NORM>(a, stream);
    case 4: return go_vecs<FMT, 4, false, 8, EPI, NORM>(a, stream);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

// Weight rows per block of vecd_kernel for this product (16 or 64), or 0 when
// vecs_kernel takes it. vecd_kernel is the faster where vecs_kernel's slices are
// few or fill only in part, so that its LDS round trip and barriers are most of
// its time, and where few blocks read the A fragments (each block of 16 rows
// reads all of them). Per vectors (<= 8, <= 16, more) and format: at most onePass
// blocks of K where vecs_kernel needs one pass, or perPass in each of two or
// three, at most `work` tiles x blocks and at most maxTiles tiles of 16 rows. Fitted on MI355X to K = 32 to 4128 and N =
// 64 to 24000, vecd / vecs in us: 16 vectors, Q8B, 480 -> 3000 5.7 / 7.0, 928 ->
// 5000 8.7 / 8.6, 1632 -> 5000 11.5 / 10.6, 480 -> 24000 11.0 / 10.7; 1 vector,
// Q8, 928 -> 5000 6.4 / 6.9, 2080 -> 6144 10.6 / 9.8; 8 vectors, Q4, 480 -> 3000
// 5.1 / 5.8, 928 -> 6144 7.3 / 6.8; 32 vectors, Q8B, 928 -> 4096 8.8 / 10.0,
// 3168 -> 5000 35.8 / 25.5; 17 vectors, Q4, one whole pass, 2048 -> 6144 16.7 /
// 12.2, one block more, 2080 -> 5000 15.0 / 16.4. 64-row blocks of eight slices:
// 17-24 vectors just past one pass (Q4, 2080 -> 16000: 21.8 / 26.1), and row-
// scaled codes, whose widening and adding is most of vecs_kernel's time when the
// weights come from the 256 MB cache (Q8, 31 vectors, 12288 -> 14000: 80 / 106 us
// cached, 101 / 106 not; 6208 -> 14000 59.5 / 66.0 not), except where its passes
// are nearly full and the rows few (8192 -> 11822: 59.1 / 61.6 cached, 72.1 / 62.5
// not), as long as they are one round of the chip (Q4, 2080 -> 24000: 36.5 / 35.6;
// Q8B_F32, 2336 -> 16000: 28.6 / 24.8).
static int vecd_rows(int fmt, int V, int KB, int N) {
    static constexpr struct {
        int onePass, perPass, work, maxTiles;
    } kRules[3][3] = {{{52, 0, 20000, INT32_MAX}, {26, 0, 10000, INT32_MAX}, {18, 0, 6000, INT32_MAX}},
                      {{30, 0, 18000, 1024}, {36, 0, 18000, 1024}, {16, 0, 6000, 1024}},
                      {{52, 52, 22000, 600}, {44, 44, 18000, 600}, {30, 37, 26000, 400}}};
    const auto &r = kRules[V <= 8 ? 0 : V <= 16 ? 1 : 2][fmt == GPHQ_FMT_Q8 ? 0 : fmt == GPHQ_FMT_Q4 ? 2 : 1];
    const long tiles = ((long)N + 15) / 16;
    const int pass = V > 16 ? 64 : 128, parts = (KB + pass - 1) / pass;
    const bool oneRound = tiles > 2 * device_cus() && tiles <= 4 * device_cus();  // of 64-row blocks
    if (V > 16 && KB > pass && oneRound &&
        (fmt == GPHQ_FMT_Q8 ? KB <= 56 * parts || parts > 4 || tiles > 3 * device_cus()
                            : V <= 24 && KB <= 88 && fmt != GPHQ_FMT_Q8B_F32))
        return 64;
    const bool few = parts == 1 ? KB <= r.onePass : parts <= 3 && KB <= r.perPass * parts;
    return few && KB * tiles <= r.work && tiles <= r.maxTiles ? 16 : 0;
}

template <int FMT, int MT, int EPI, bool NORM>
static int go_vecd(const Vec2Args &a, int rows, hipStream_t stream) {
    if constexpr (MT == 3 || (MT == 4 && FMT == GPHQ_FMT_Q8)) {
        if (rows == 64) {
            hipLaunchKernelGGL((vecd_kernel<FMT, MT, 8, 4, 2, EPI, NORM>), dim3((unsigned)((a.N + 63) / 64)), dim3(512),
                               0, stream, a);
            return launch_status();
        }
    }
    hipLaunchKernelGGL((vecd_kernel<FMT, MT, 4, 1, 4, EPI, NORM>), dim3((unsigned)((a.N + 15) / 16)), dim3(256), 0,
                       stream, a);
    return launch_status();
}

template <int FMT, int EPI, bool NORM>
static int launch_vecs_fmt(const Vec2Args &a, int rows, hipStream_t stream) {
    if (!rows) return launch_vecs_tiles<FMT, EPI, NORM>(a, stream);
    switch ((2 * a.V + 15) / 16) {
    case 1: return go_vecd<FMT, 1, EPI, NORM>(a, rows, stream);
    case 2: return go_vecd<FMT, 2, EPI, NORM>(a, rows, stream);
    case 3: return go_vecd<FMT, 3, EPI, NORM>(a, rows, stream);
    case 4: return go_vecd<FMT, 4, EPI, NORM>(a, rows, stream);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

template <int EPI, bool NORM>
static int launch_vecs(int fmt, const Vec2Args &a, int rows, hipStream_t stream) {
    switch (fmt) {
    case GPHQ_FMT_Q8: return launch_vecs_fmt<GPHQ_FMT_Q8, EPI, NORM>(a, rows, stream);
    case GPHQ_FMT_Q8B: return launch_vecs_fmt<GPHQ_FMT_Q8B, EPI, NORM>(a, rows, stream);
    case GPHQ_FMT_Q8B_F32: return launch_vecs_fmt<GPHQ_FMT_Q8B_F32, EPI, NORM>(a, rows, stream);
    case GPHQ_FMT_Q4: return launch_vecs_fmt<GPHQ_FMT_Q4, EPI, NORM>(a, rows, stream);
    }
    return GPHQ_ERR_UNSUPPORTED;
}

// Multi-vector GEMV, optionally with the decode step's prologue and epilogue:
// norm (0/1) selects PRO_NORM, epi is VEC_STORE, VEC_ADD or VEC_SWIGLU (y then
// holds N/2 values per vector). V <= kMaxVecLanes, K % 32 == 0, x rows 16-byte
// aligned; work holds gemv_vec_workspace_bytes(V, K). Validated by the caller.
// Whether a preparation for (fmt, V, K) goes through vech_prep_kernel, so a
// pending K-split residual add (VecFold) can be handed to it.
bool gemv_vec_prep_folds(int fmt, int V, int K) {
    return vech_split_parts(fmt, V, K) != 0 || vech_takes(fmt, V, K);
}

// fold: a K-split GEMV's residual add into x left pending by an earlier call
// (applied by this call's preparation, before it reads x); defer: when this
// call is a K-split residual add without a norm, its finish is left to the
// caller's next preparation and described in *defer (parts 0 otherwise).
int gemv_vec_fused_launch(int fmt, int norm, int epi, const void *codes, const void *scales, const float *x,
                          long xstride, float *y, long ystride, int V, int K, int N, float eps, void *work,
                          hipStream_t stream, float *split, size_t split_bytes, const VecFold &fold, VecFold *defer) {
    if (defer) *defer = VecFold{};
    if (N == 0 || V == 0) return fold.parts ? GPHQ_ERR_UNSUPPORTED : GPHQ_OK;
    const int KB = K / 32;
    const int parts = vech_split_parts(fmt, V, K);
    if (fold.parts && !gemv_vec_prep_folds(fmt, V, K)) return GPHQ_ERR_UNSUPPORTED;
    if (parts && split && split_bytes >= (size_t)parts * V * N * 4 && (epi != VEC_SWIGLU || N % 2 == 0)) {
        _Float16 *A = (_Float16 *)work;
        float *inv = (float *)((char *)work + (size_t)2 * KB * 1024);
        float *ssq = inv + V;
        hipLaunchKernelGGL(vech_prep_kernel, dim3(16), dim3(1024), 0, stream, x, xstride, V, K, A, inv, ssq, fold);
        GPHQ_TRY(launch_status());
        Vec2Args a{codes, scales, A, inv, ssq, y, ystride, V, K, N, KB, eps};
        a.part = split;
        if (epi == VEC_ADD && !norm && defer) {
            const int rc = launch_vech_split<VEC_ADD, false>(fmt, a, parts, stream, false);
            if (rc != GPHQ_OK) return rc;
            *defer = VecFold{split, inv, fmt == GPHQ_FMT_Q8 ? (const float *)scales : nullptr, parts};
            return GPHQ_OK;
        }
        if (epi == VEC_ADD) return norm ? launch_vech_split<VEC_ADD, true>(fmt, a, parts, stream)
                                        : launch_vech_split<VEC_ADD, false>(fmt, a, parts, stream);
        if (epi == VEC_SWIGLU) return norm ? launch_vech_split<VEC_SWIGLU, true>(fmt, a, parts, stream)
                                           : launch_vech_split<VEC_SWIGLU, false>(fmt, a, parts, stream);
        return norm ? launch_vech_split<VEC_STORE, true>(fmt, a, parts, stream)
                    : launch_vech_split<VEC_STORE, false>(fmt, a, parts, stream);
    }
    if (vech_takes(fmt, V, K)) {
        _Float16 *A = (_Float16 *)work;
        float *inv = (float *)((char *)work + (size_t)2 * KB * 1024);
        float *ssq = inv + V;
        hipLaunchKernelGGL(vech_prep_kernel, dim3(16), dim3(1024), 0, stream, x, xstride, V, K, A, inv, ssq, fold);
        GPHQ_TRY(launch_status());
        const Vec2Args a{codes, scales, A, inv, ssq, y, ystride, V, K, N, KB, eps};
        if (epi == VEC_ADD) return norm ? launch_vech<VEC_ADD, true>(fmt, a, stream)
                                        : launch_vech<VEC_ADD, false>(fmt, a, stream);
        if (epi == VEC_SWIGLU) return norm ? launch_vech<VEC_SWIGLU, true>(fmt, a, stream)
                                           : launch_vech<VEC_SWIGLU, false>(fmt, a, stream);
        return norm ? launch_vech<VEC_STORE, true>(fmt, a, stream) : launch_vech<VEC_STORE, false>(fmt, a, stream);
    }
    const int MT = (2 * V + 15) / 16;
    _Float16 *A = (_Float16 *)work;
    float *inv = (float *)((char *)work + (size_t)MT * KB * 1024);
    float *ssq = inv + (size_t)V * KB;
    const Vec2Args a{codes, scales, A, inv, ssq, y, ystride, V, K, N, KB, eps};
    if (KB == 0) {  // an empty sum: stored, or added as nothing
        const dim3 grid((unsigned)(((long)V * N + 255) / 256));
        if (fmt == GPHQ_FMT_Q8) hipLaunchKernelGGL(vec_empty_kernel<GPHQ_FMT_Q8>, grid, dim3(256), 0, stream, a, epi == VEC_STORE);
        else hipLaunchKernelGGL(vec_empty_kernel<GPHQ_FMT_Q8B>, grid, dim3(256), 0, stream, a, epi == VEC_STORE);
        return launch_status();
    }
    const int rows = vecd_rows(fmt, V, KB, N);
    // A rows past the vectors are never written; they only feed results that
    // are never stored.
    hipLaunchKernelGGL(vec_prep_blocks_kernel, dim3((unsigned)(((long)V * KB * 4 + 255) / 256)), dim3(256), 0, stream,
                       x, xstride, V, KB, A, inv, ssq, !rows && vec_pair(V));
    GPHQ_TRY(launch_status());
    if (epi == VEC_ADD) return norm ? launch_vecs<VEC_ADD, true>(fmt, a, rows, stream)
                                    : launch_vecs<VEC_ADD, false>(fmt, a, rows, stream);
    if (epi == VEC_SWIGLU) return norm ? launch_vecs<VEC_SWIGLU, true>(fmt, a, rows, stream)
                                       : launch_vecs<VEC_SWIGLU, false>(fmt, a, rows, stream);
    return norm ? launch_vecs<VEC_STORE, true>(fmt, a, rows, stream) : launch_vecs<VEC_STORE, false>(fmt, a, rows, stream);
}

// y[v*ystride + j] for v < V (gphq_gemv_vec). Arguments were validated by the caller.
int gemv_vec_launch(int fmt, const void *codes, const void *scales, const float *x, long xstride, float *y,
                    long ystride, int V, int K, int N, void *work, hipStream_t stream) {
    return gemv_vec_fused_launch(fmt, 0, VEC_STORE, codes, scales, x, xstride, y, ystride, V, K, N, 0.0f, work,
                                 stream, nullptr, 0, VecFold{}, nullptr);
}

}  // namespace gphq
