// GPTQ producer on MI355X: the core of cmd/qwen3-gptq, qwen3lm quantizeGroup
// (gptq.go:604-666) with gptqInverseFactor (gptq_linalg.go:68-223) and
// gptqRound (gptq.go:671-796), for one group of projections sharing their
// calibration inputs.
//
//   factor: H = X^T X over the calibration rows; dead channels (H[i][i] == 0)
//     get H[i][i] = 1; H += 0.01 * mean(diag) * I; U = J chol(J H J)^-1 J, the
//     upper factor with H^-1 = U^T U. The factorization and the factor's
//     inverse advance together in 64-column panels, two launches each (the
//     diagonal block and the products with its inverse in float64, the
//     trailing products fp32).
//   round: per 128-column block, one wavefront per weight row quantizes the
//     block's columns in order (code = clamp(rne(w / s)), error
//     e = (w - q s) / U[c][c], the block's later columns w[j] -= e U[c][j]),
//     choosing each 4-bit group's scale (q4GroupScale) from the current values
//     at the group's first column; then the columns after the block take the
//     lazy update W -= E U (an fp32 product).
// Storage is fp32, as the reference's. The Gram matrix adds each 16-row chunk's
// fp32 sum in float64, the factorization works within a panel in float64 (the
// reference's substitutions sum in float64), the trailing products and the lazy
// updates are fp32 products with fp32 sums.
#include <math.h>

#include <algorithm>
#include <vector>

#include "common.h"

using namespace gphq;

namespace {

constexpr int kPanel = 64;      // Cholesky / inverse panel width
constexpr int kRoundBlock = 128;  // gptqBlock (gptq.go:37)
constexpr int kRowsPerBlock = 8;  // weight rows (wavefronts) per rounding workgroup

// ---- fp32 product: C = [C +] alpha * op(A) op(B) ---------------------------
// A(i,p) = a[i*lda + p] (TA 0) or a[p*lda + i] (TA 1); B(p,j) = b[p*ldb + j]
// (TB 0) or b[j*ldb + p] (TB 1). BM x BN tiles, four wavefronts as 2 x 2, each
// on 32 x 32 tiles of v_mfma_f32_32x32x2_f32 (fp32 products and sums). 16-deep
// K chunks, double-buffered in LDS, the next chunk's loads in flight during
// the MFMAs, one barrier per chunk. An operand whose memory runs along K lies
// in LDS as [i][16 + 4] (one 16-byte read feeds four MFMAs), the other kind as
// [p][BM + 8] (four 4-byte reads); both conflict-free. Of each 8 K values lane
// half h multiplies 4h .. 4h + 3, so an MFMA pairs p with p + 4. With
// accumulate the full sum is formed first and added once.
using f32x16 = __attribute__((ext_vector_type(16))) float;

enum SgemmMode {
    kFull,
    // j >= i only, stored at C[M-1-i][N-1-j]: the Gram matrix J H J, its lower
    // triangle (M == N).
    kUpperReversed,
};

struct SgemmArgs {
    int M, N, K;
    float alpha;
    const float *a, *b;
    float *c;
    long lda, ldb, ldc;
    int accumulate;
    int vecA, vecB;  // 16-byte loads: base aligned, stride a multiple of 4
};

inline int vec16(const float *p, long ld) { return ((uintptr_t)p % 16 == 0 && ld % 4 == 0) ? 1 : 0; }

// Rows [i0, i0 + BM) x K chunk [p0, p0 + 16) of an operand with `rows` rows and
// K values, as BM/64 float4 per thread; zero past the edges.
template <int T, int BM>
__device__ __forceinline__ void sgemm_fetch(float4 (&v)[BM / 64], const float *x, long ld, int rows, int K, int i0,
                                            int p0, bool vec) {
#pragma unroll
    for (int e = 0; e < BM / 64; ++e) {
        const int idx = (int)threadIdx.x + 256 * e;
        const int i = i0 + (T == 0 ? idx >> 2 : (idx % (BM / 4)) * 4);
        const int p = p0 + (T == 0 ? (idx & 3) * 4 : idx / (BM / 4));
        const int left = T == 0 ? (i < rows ? K - p : 0) : (p < K ? rows - i : 0);
        float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (left > 0) {
            const float *src = T == 0 ? x + (size_t)i * ld + p : x + (size_t)p * ld + i;
            if (vec && left >= 4) {
                const float4 q = *(const float4 *)src;
                r[0] = q.x, r[1] = q.y, r[2] = q.z, r[3] = q.w;
            } else {
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    if (d < left) r[d] = src[d];
            }
        }
        v[e] = make_float4(r[0], r[1], r[2], r[3]);
    }
}

template <int T, int BM>
__device__ __forceinline__ void sgemm_stash(float *lds, const float4 (&v)[BM / 64]) {
#pragma unroll
    for (int e = 0; e < BM / 64; ++e) {
        const int idx = (int)threadIdx.x + 256 * e;
        float *d = T == 0 ? lds + (idx >> 2) * 20 + (idx & 3) * 4
                          : lds + (idx / (BM / 4)) * (BM + 8) + (idx % (BM / 4)) * 4;
        *(float4 *)d = v[e];
    }
}

// Four MFMAs' operand values of one 32-row tile: K values 8g + 4h .. + 3 of row i.
template <int T, int BM>
__device__ __forceinline__ void sgemm_frag(float (&f)[4], const float *lds, int i, int g, int h) {
    if (T == 0) {
        const float4 q = *(const float4 *)(lds + i * 20 + g * 8 + h * 4);
        f[0] = q.x, f[1] = q.y, f[2] = q.z, f[3] = q.w;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = lds[(g * 8 + h * 4 + e) * (BM + 8) + i];
    }
}

// LDS floats of one K chunk of an operand of kind T (0: runs along K).
template <int T, int BM>
constexpr int sgemm_lds() {
    return T == 0 ? BM * 20 : 16 * (BM + 8);
}

// The lower-triangle pair (row >= col) numbered t, row by row.
__device__ __forceinline__ void tri_pair(int t, int &row, int &col) {
    row = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while ((long)row * (row + 1) / 2 > t) --row;
    while ((long)(row + 1) * (row + 2) / 2 <= t) ++row;
    col = t - (int)((long)row * (row + 1) / 2);
}

template <int TA, int TB, int BM, int BN, int MODE>
__global__ __launch_bounds__(256) void sgemm_kernel(SgemmArgs g) {
    constexpr int MT = BM / 64, NT = BN / 64;  // 32 x 32 tiles per wavefront
    __shared__ __attribute__((aligned(16))) float As[2][sgemm_lds<TA, BM>()], Bs[2][sgemm_lds<TB ^ 1, BN>()];
    const int M = g.M, N = g.N, K = g.K;
    int ti, tj;
    if (MODE == kUpperReversed) {
        tri_pair((int)blockIdx.x, tj, ti);
    } else {
        const int tn = (N + BN - 1) / BN;
        ti = (int)blockIdx.x / tn;
        tj = (int)blockIdx.x - ti * tn;
    }
    const int bi = ti * BM, bj = tj * BN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, h = lane >> 5;
    const int wi = (wave >> 1) * (BM / 2), wj = (wave & 1) * (BN / 2);
    f32x16 acc[MT][NT] = {};
    // The Gram matrix's sums run over thousands of rows and its inverse
    // amplifies their rounding: each chunk's fp32 sum is added in float64.
    using f64x16 = __attribute__((ext_vector_type(16))) double;
    f64x16 sum[MODE == kUpperReversed ? MT : 1][MODE == kUpperReversed ? NT : 1] = {};
    float4 va[BM / 64], vb[BN / 64];
    sgemm_fetch<TA, BM>(va, g.a, g.lda, M, K, bi, 0, g.vecA);
    sgemm_fetch<TB ^ 1, BN>(vb, g.b, g.ldb, N, K, bj, 0, g.vecB);
    sgemm_stash<TA, BM>(As[0], va);
    sgemm_stash<TB ^ 1, BN>(Bs[0], vb);
    __syncthreads();
    int buf = 0;
    // Chunks are counted: K may be INT32_MAX, and a position past the last chunk would not fit.
    const int chunks = (int)(((uint32_t)K + 15) / 16);
    for (int chunk = 1; chunk <= chunks; ++chunk) {
        const bool more = chunk < chunks;
        if (more) {
            sgemm_fetch<TA, BM>(va, g.a, g.lda, M, K, bi, chunk * 16, g.vecA);
            sgemm_fetch<TB ^ 1, BN>(vb, g.b, g.ldb, N, K, bj, chunk * 16, g.vecB);
        }
#pragma unroll
        for (int gr = 0; gr < 2; ++gr) {
            float fa[MT][4], fb[NT][4];
#pragma unroll
            for (int x = 0; x < MT; ++x) sgemm_frag<TA, BM>(fa[x], As[buf], wi + 32 * x + li, gr, h);
#pragma unroll
            for (int y = 0; y < NT; ++y) sgemm_frag<TB ^ 1, BN>(fb[y], Bs[buf], wj + 32 * y + li, gr, h);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int x = 0; x < MT; ++x)
#pragma unroll
                    for (int y = 0; y < NT; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[x][e], fb[y][e], acc[x][y], 0, 0, 0);
        }
        if constexpr (MODE == kUpperReversed) {
#pragma unroll
            for (int x = 0; x < MT; ++x)
#pragma unroll
                for (int y = 0; y < NT; ++y) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[x][y][r] += (double)acc[x][y][r];
                    acc[x][y] = f32x16{};
                }
        }
        if (more) {
            sgemm_stash<TA, BM>(As[buf ^ 1], va);
            sgemm_stash<TB ^ 1, BN>(Bs[buf ^ 1], vb);
        }
        __syncthreads();
        buf ^= 1;
    }
    // Result register r of lane l: row (r & 3) + 8 (r >> 2) + 4 h, column l % 32.
#pragma unroll
    for (int x = 0; x < MT; ++x)
#pragma unroll
        for (int y = 0; y < NT; ++y) {
            if constexpr (MODE == kUpperReversed) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int i = bi + wi + 32 * x + (r & 3) + 8 * (r >> 2) + 4 * h, j = bj + wj + 32 * y + li;
                    if (i < M && j < N && j >= i)
                        g.c[(size_t)(M - 1 - i) * g.ldc + (N - 1 - j)] = (float)sum[x][y][r];
                }
                continue;
            }
            const int i0 = bi + wi + 32 * x + 4 * h, j = bj + wj + 32 * y + li;
            float own[16];
            if (g.accumulate) {
                // All 16 requested before the first store (clamped: what lies past an edge is not stored).
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    own[r] = g.c[(size_t)min(i0 + (r & 3) + 8 * (r >> 2), M - 1) * g.ldc + min(j, N - 1)];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = i0 + (r & 3) + 8 * (r >> 2);
                if (i >= M || j >= N) continue;
                const float v = g.alpha * acc[x][y][r];
                g.c[(size_t)i * g.ldc + j] = g.accumulate ? own[r] + v : v;
            }
        }
}

template <int TA, int TB>
int sgemm(int M, int N, int K, float alpha, const float *a, long lda, const float *b, long ldb, float *c, long ldc,
          bool accumulate, hipStream_t st) {
    if (M <= 0 || N <= 0) return GPHQ_OK;
    const SgemmArgs g{M, N, K, alpha, a, b, c, lda, ldb, ldc, accumulate ? 1 : 0, vec16(a, lda), vec16(b, ldb)};
    // 128 x 128 tiles halve the operand reads; below two rounds of the chip
    // the 64 x 64 tiles' four times as many blocks matter more.
    const long big = (long)((M + 127) / 128) * ((N + 127) / 128);
    if (big >= 2L * device_cus())
        hipLaunchKernelGGL((sgemm_kernel<TA, TB, 128, 128, kFull>), dim3((unsigned)big), dim3(256), 0, st, g);
    else
        hipLaunchKernelGGL((sgemm_kernel<TA, TB, 64, 64, kFull>),
                           dim3((unsigned)((M + 63) / 64) * (unsigned)((N + 63) / 64)), dim3(256), 0, st, g);
    return launch_status();
}

// Dead channels and damping (gptq.go:623-637) on A = J H J (A[i][i] is channel
// n-1-i): one block; the diagonal's mean in float64. Clears *bad.
__global__ __launch_bounds__(1024) void gptq_damp_kernel(float *a, int n, uint8_t *dead, int *bad) {
    __shared__ double part[16];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += (double)a[(size_t)i * n + i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    if (threadIdx.x == 0) *bad = 0;
    __syncthreads();
    double mean = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) mean += part[w];
    mean /= (double)n;
    const float add = (float)(0.01 * mean);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float d = a[(size_t)i * n + i];
        const bool isDead = d == 0.0f;
        dead[n - 1 - i] = isDead ? 1 : 0;
        if (isDead) d = 1.0f;
        a[(size_t)i * n + i] = d + add;
    }
}

// ---- Cholesky of A = J H J and the inverse of its factor ---------------------
// What the factor of an n x n matrix cannot do without is n^3 multiply-adds
// (half of H, a third each for L and L^-1), but its columns form a chain, one
// step per 64-column panel. Both factors advance in the same step, as an
// elimination on [A | I], so a step is two launches whatever n: with the
// diagonal block's inverse at hand chol_panel_kernel forms the panel below the
// block and the inverse's rows beside it (products in float64, where a
// substitution would be 64 dependent divisions), and chol_update_kernel takes
// the panel's products off the trailing tiles of A and adds them to the sums
// S = L X of the inverse's later rows. Its first block, which owns the next
// diagonal block, goes on to factor and invert that block while the others
// update. X's rows come from the sums over all rows above them, as in a
// substitution, so L X = I holds to fp32 rounding of |L||X| (products of
// inverted blocks, X21 = -X22 (L21 X11), have no such bound). K = 4096 from
// 4096 rows: 53.5 -> 2.91 ms (separate launches for the block, the panel's
// substitution and the update, then one thin product and a substitution per 64
// rows of the inverse, took 84 + 207 + 21 + 357 + 137 us a panel).

// The packed lower triangle of a 64 x 64 block: row r, column c <= r.
__device__ __forceinline__ int packed(int r, int c) { return r * (r + 1) / 2 + c; }

using f64x4 = __attribute__((ext_vector_type(4))) double;

// Lane N's value in each row of 16 lanes (DPP row_newbcast).
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + N, 0xF, 0xF, true));
}
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x150 + N, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x150 + N, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// A value of the diagonal block. An infinite pivot (an overflowed Gram matrix) is
// the reference's sqrt(Inf): Inf on the diagonal, zeros below it and in the
// inverse. As 1e300, from which updates take nothing, it gives the same float32
// values without Inf * 0 on the way (an infinity off the diagonal still ends in a
// pivot that is not positive, and a NaN stays one).
__device__ __forceinline__ double diag_value(float v) { return v > 3.4028235e38f ? 1e300 : (double)v; }

// The diagonal block's working storage: D's lower 16 x 16 blocks hold A, then
// L; an upper block (c, r) holds block (r, c) of S, then of L^-1, transposed;
// V the diagonal blocks of L^-1.
struct DiagLds {
    double D[64][66];
    double V[4][16][18];
};

// a[c] -= li L[c][J] for c = C .. 15, l holding L[.][J] by lane.
template <int J, int C>
__device__ __forceinline__ void chol16_row(double (&a)[16], double l, double li) {
    if constexpr (C < 16) {
        a[C] = fma(-li, row_bcast<C>(l), a[C]);
        // Kept here: sunk to their use, 15 columns of broadcasts spill.
        asm volatile("" : "+v"(a[C]));
        chol16_row<J, C + 1>(a, l, li);
    }
}

template <int J>
__device__ __forceinline__ void chol16_steps(double (&a)[16], double (&w)[4], int i, bool &fail) {
    if constexpr (J < 16) {
        double d = row_bcast<J>(a[J]);
        const bool positive = d > 0.0;
        fail = fail || !positive;
        d = positive ? d : 1.0;
        // sqrt(d) and its reciprocal from the hardware's estimate, two Goldschmidt steps.
        double r = __builtin_amdgcn_rsq(d), piv = d * r, hr = 0.5 * r;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const double e = fma(-piv, hr, 0.5);
            piv = fma(piv, e, piv);
            hr = fma(hr, e, hr);
        }
        r = 2.0 * hr;
        // choleskyLower's column (gptq_linalg.go:73-93), stored as float32.
        const float lf = i == J ? (float)piv : (float)(a[J] * r);
        const double l = (double)lf;
        a[J] = l;
        const double li = i > J ? l : 0.0;
        chol16_row<J, J + 1>(a, l, li);
        // The reciprocal of the stored pivot; row J of the inverse is final.
        const double ljj = (double)fminf(row_bcast<J>(lf), 3.4028235e38f);  // finite
#pragma unroll
        for (int n = 0; n < 2; ++n) r = fma(r, fma(-ljj, r, 1.0), r);
        const double lr = li * r;
#pragma unroll
        for (int k = 0; k <= J / 4; ++k) {
            const double t = row_bcast<J>(w[k]);
            w[k] = i == J ? t * r : fma(-lr, t, w[k]);
            asm volatile("" : "+v"(w[k]));
        }
        chol16_steps<J + 1>(a, w, i, fail);
    }
}

// Factors D's 16 x 16 diagonal block kb and inverts the factor into V, on one
// wavefront: lane l holds row l % 16 of the block (a copy in each row of 16
// lanes) and columns 4k + l / 16 of that row of the inverse.
__device__ __forceinline__ void chol16(DiagLds &s, int kb, int *bad) {
    const int i = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4, o = 16 * kb;
    double a[16], w[4];
#pragma unroll
    for (int c = 0; c < 16; ++c) a[c] = s.D[o + i][o + c];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = 4 * k + g == i ? 1.0 : 0.0;
    bool fail = false;
    chol16_steps<0>(a, w, i, fail);
    if (fail && threadIdx.x == 0) *bad = 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) s.V[kb][i][4 * k + g] = w[k];
    if (g == 0) {
#pragma unroll
        for (int c = 0; c < 16; ++c) s.D[o + i][o + c] = a[c];
    }
}

// acc +- the 16 x 16 x 16 product of A (rows [i][p] at pa, stride lda) and B
// ([j][p] at pb). Result register r of lane l: row 4 r + l / 16, column l % 16.
__device__ __forceinline__ f64x4 mma16(const double *pa, int lda, const double *pb, int ldb, f64x4 acc) {
    const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int p = 0; p < 16; p += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[li * lda + p + lk], pb[li * ldb + p + lk], acc, 0, 0, 0);
    return acc;
}

// Factors the b x b (b <= 64) diagonal block whose lower triangle D holds
// (identity past b) and inverts the factor, with 256 threads, float64
// throughout, L rounded to float32 as it is formed. L goes to l (row stride
// ld), L^-1 to x as float32 (row stride ld) and, unless inv is null (no panel
// follows), to inv as packed float64 for the panel product. 16 columns at a
// time: wavefront 0 factors the 16 x 16 block in registers while the others
// finish the previous columns' products on v_mfma_f64_16x16x4_f64. A chain of
// 64 columns, each a float64 root and its broadcasts: 16.5 us with the launch
// (52 us as one loop over LDS with a root, two divisions and a barrier a column).
__device__ __forceinline__ void chol_diag(DiagLds &s, int b, float *l, float *x, long ld, double *inv, int *bad) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int li = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    for (int kb = 0; kb < 4; ++kb) {
        // The products of block column kb - 1: tile 0 is the diagonal block that
        // wavefront 0 goes on to factor.
        const int q = kb - 1, trail = kb ? (4 - kb) * (5 - kb) / 2 : 0, tiles = kb ? trail + (4 - kb) * kb : 0;
        for (int t = wave; t < tiles; t += wave ? 3 : 1000) {
            int rb, cb;
            if (t < trail) {
                int row = 0, rest = t;
                while (rest > row) rest -= ++row;
                rb = kb + row;
                cb = kb + rest;
            } else {
                rb = kb + (t - trail) / kb;
                cb = (t - trail) % kb;
            }
            const bool minus = t < trail, fresh = !minus && cb == q;
            f64x4 acc = {};
            if (fresh) {
#pragma unroll
                for (int p = 0; p < 16; p += 4)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(s.D[16 * rb + li][16 * q + p + lk], s.V[q][p + lk][li],
                                                               acc, 0, 0, 0);
            } else {
                acc = mma16(&s.D[16 * rb][16 * q], 66, &s.D[16 * cb][16 * q], 66, acc);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double *d = minus ? &s.D[16 * rb + 4 * r + lk][16 * cb + li] : &s.D[16 * cb + li][16 * rb + 4 * r + lk];
                *d = minus ? *d - acc[r] : fresh ? acc[r] : *d + acc[r];
            }
        }
        if (wave == 0) chol16(s, kb, bad);
        __syncthreads();
        // Column kb of L below its diagonal block, row kb of L^-1 beside its own.
        if (wave < 3) {
            const int t = wave < kb ? wave : wave + 1;
            if (t > kb) {
                const f64x4 acc = mma16(&s.D[16 * t][16 * kb], 66, &s.V[kb][0][0], 18, f64x4{});
#pragma unroll
                for (int r = 0; r < 4; ++r) s.D[16 * t + 4 * r + lk][16 * kb + li] = (double)(float)acc[r];
            } else {
                const f64x4 acc = mma16(&s.V[kb][0][0], 18, &s.D[16 * t][16 * kb], 66, f64x4{});
#pragma unroll
                for (int r = 0; r < 4; ++r) s.D[16 * t + li][16 * kb + 4 * r + lk] = -acc[r];
            }
        }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
        const int r = e >> 6, c = e & 63;
        if (r >= b || c > r) continue;
        const double v = (r >> 4) == (c >> 4) ? s.V[r >> 4][r & 15][c & 15] : s.D[c][r];
        l[(size_t)r * ld + c] = (float)s.D[r][c];
        x[(size_t)r * ld + c] = (float)v;
        if (inv) inv[packed(r, c)] = v;
    }
}

// The first diagonal block.
__global__ __launch_bounds__(256, 3) void chol_first_kernel(float *a, int n, float *x, double *inv, int *bad) {
    __shared__ DiagLds d;
    const int b = min(64, n);
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        v[u] = a[(size_t)min(e >> 6, b - 1) * n + min(e & 63, b - 1)];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = (int)threadIdx.x + 256 * u, r = e >> 6, c = e & 63;
        d.D[r][c] = r < b && c <= r ? diag_value(v[u]) : r == c ? 1.0 : 0.0;
    }
    __syncthreads();
    chol_diag(d, b, a, x, n, inv, bad);
}

// The step at j0, on v_mfma_f64_16x16x4_f64. Blocks below `below`: 32 panel
// rows each, L21 = A21 L11^-T (gptq_linalg.go:97-110). The others: 32 columns
// each of the inverse's rows j0 .. j0+63, X = -L11^-1 S.
__global__ __launch_bounds__(256) void chol_panel_kernel(float *a, float *x, int n, int j0, int below,
                                                         const double *__restrict__ inv) {
    __shared__ double Li[64][66];  // L11^-1, zero above the diagonal
    __shared__ float Ar[64][36];   // the panel's 32 rows as [p][row], or S's 32 columns as [p][column]
    const bool rows = (int)blockIdx.x < below;
    const int i0 = rows ? j0 + 64 + (int)blockIdx.x * 32 : ((int)blockIdx.x - below) * 32;
    // Every load unconditional (clamped; what lies past an edge feeds only
    // results that are not stored): a guarded load is waited for on its own.
    double lv[16];
    float av[8];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = (int)threadIdx.x + 256 * u, r = e >> 6, c = e & 63;
        lv[u] = inv[packed(r, min(c, r))];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        av[u] = rows ? a[(size_t)min(i0 + (e >> 6), n - 1) * n + j0 + (e & 63)]
                     : x[(size_t)min(j0 + (e >> 5), n - 1) * n + i0 + (e & 31)];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = (int)threadIdx.x + 256 * u, r = e >> 6, c = e & 63;
        Li[r][c] = c <= r ? lv[u] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int e = (int)threadIdx.x + 256 * u;
        if (rows) Ar[e & 63][e >> 6] = av[u];
        else Ar[e >> 5][e & 31] = av[u];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    // Wavefront w: L11^-1's rows 16w .. 16w+15, which need p <= 16w + 15.
    f64x4 acc[2] = {};
    for (int p0 = 0; p0 <= 16 * wave; p0 += 16)
#pragma unroll
        for (int p = p0; p < p0 + 16; p += 4) {
            const double lr = Li[16 * wave + li][p + lk];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const double v = (double)Ar[p + lk][16 * t + li];
                acc[t] = rows ? __builtin_amdgcn_mfma_f64_16x16x4f64(v, lr, acc[t], 0, 0, 0)
                              : __builtin_amdgcn_mfma_f64_16x16x4f64(lr, v, acc[t], 0, 0, 0);
            }
        }
    // Result register r of lane l: row 4 r + l / 16, column l % 16.
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (rows) {
                const int i = i0 + 16 * t + 4 * r + lk;
                if (i < n) a[(size_t)i * n + j0 + 16 * wave + li] = (float)acc[t][r];
            } else {
                const int i = j0 + 16 * wave + 4 * r + lk;
                if (i < n) x[(size_t)i * n + i0 + 16 * t + li] = (float)-acc[t][r];
            }
        }
}

// The rest of the step at j0, in 64 x 64 tiles (fp32 products and sums, the
// whole 64-deep sum added once). Blocks below `tri`: A22 -= L21 L21^T on the
// lower triangle; block 0 then factors and inverts the diagonal block it has
// just updated, the next step's. The others: S += L21 X[j0 .. j0+63], the
// columns of the diagonal block for the first time.
__global__ __launch_bounds__(256, 3) void chol_update_kernel(float *a, int n, int j0, int tri, float *x, double *inv,
                                                          int *bad, int vec) {
    __shared__ union {
        struct {
            __attribute__((aligned(16))) float A[64][68], B[64][72];
        } p;
        DiagLds d;
    } sh;
    const int j1 = j0 + 64;
    const bool trailing = (int)blockIdx.x < tri;
    int ti, tj;
    if (trailing) {
        tri_pair((int)blockIdx.x, ti, tj);
    } else {
        const int cols = j1 / 64, t = (int)blockIdx.x - tri;
        ti = t / cols;
        tj = t - ti * cols;
    }
    const int bi = j1 + ti * 64, bj = trailing ? j1 + tj * 64 : tj * 64;
    float *const c = trailing ? a : x;
    const bool fresh = !trailing && bj == j0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 31, h = lane >> 5;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    // Every load unconditional, rows and columns past the edge clamped (they
    // feed only results that are not stored), the tile's own values among them.
    float4 va[4], vb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int idx = (int)threadIdx.x + 256 * e, r = idx >> 4, q = (idx & 15) * 4;
        const float *pa = a + (size_t)min(bi + r, n - 1) * n + j0 + q;
        // L21's rows [j][p], or the inverse's rows [p][j] (its diagonal block is lower).
        const float *pb = trailing ? a + (size_t)min(bj + r, n - 1) * n + j0 + q : x + (size_t)(j0 + r) * n + bj + q;
        if (vec) {
            va[e] = *(const float4 *)pa;
            vb[e] = *(const float4 *)pb;
        } else {
            va[e] = make_float4(pa[0], pa[1], pa[2], pa[3]);
            vb[e] = make_float4(pb[0], pb[1], pb[2], pb[3]);
        }
    }
    float own[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = bi + wi + (r & 3) + 8 * (r >> 2) + 4 * h, j = bj + wj + li;
        own[r] = c[(size_t)min(i, n - 1) * n + min(j, n - 1)];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int idx = (int)threadIdx.x + 256 * e, r = idx >> 4, q = (idx & 15) * 4;
        if (fresh)
            vb[e] = make_float4(q <= r ? vb[e].x : 0.0f, q + 1 <= r ? vb[e].y : 0.0f, q + 2 <= r ? vb[e].z : 0.0f,
                                q + 3 <= r ? vb[e].w : 0.0f);
        *(float4 *)&sh.p.A[r][q] = va[e];
        *(float4 *)&sh.p.B[r][q] = vb[e];
    }
    __syncthreads();
    f32x16 acc = {};
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const float4 fa = *(const float4 *)&sh.p.A[wi + li][8 * g + 4 * h];
        float4 fb;
        if (trailing) {
            fb = *(const float4 *)&sh.p.B[wj + li][8 * g + 4 * h];
        } else {
            const float *b = &sh.p.B[8 * g + 4 * h][wj + li];
            fb = make_float4(b[0], b[72], b[144], b[216]);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.x, fb.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.y, fb.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.z, fb.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa.w, fb.w, acc, 0, 0, 0);
    }
    const bool diag = blockIdx.x == 0;
    if (diag) __syncthreads();  // every wavefront has read its operands
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int lr = wi + (r & 3) + 8 * (r >> 2) + 4 * h, lc = wj + li;
        const float v = trailing ? own[r] - acc[r] : fresh ? acc[r] : own[r] + acc[r];
        // Past the matrix's edge the diagonal block continues as the identity.
        if (diag) sh.d.D[lr][lc] = bi + lr < n ? diag_value(v) : lr == lc ? 1.0 : 0.0;
        else if (bi + lr < n && bj + lc <= bi + lr) c[(size_t)(bi + lr) * n + bj + lc] = v;
    }
    if (!diag) return;
    __syncthreads();
    chol_diag(sh.d, min(64, n - j1), a + (size_t)j1 * n + j1, x + (size_t)j1 * n + j1, n, inv, bad);
}

// U[r][c] = X[n-1-r][n-1-c] for c >= r, else 0 (gptq_linalg.go:208-221).
__global__ void u_from_x_kernel(const float *__restrict__ x, float *__restrict__ u, int n) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)n * n) return;
    const int r = (int)(idx / n), c = (int)(idx - (size_t)r * n);
    u[idx] = c < r ? 0.0f : x[(size_t)(n - 1 - r) * n + (n - 1 - c)];
}

// ---- rounding ----------------------------------------------------------------

// Zero the dead columns of w [n][k] (gptq.go:643-651).
__global__ void zero_dead_kernel(float *w, int n, int k, const uint8_t *dead) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)n * k) return;
    if (dead[idx % k]) w[idx] = 0.0f;
}

// 8-bit row scales max|row| / 127 (gptq.go:675-680), NaN propagating like
// q8gemm.MaxAbs; fp32, also stored little-endian as the row's scale bytes.
__global__ __launch_bounds__(256) void row_scale_kernel(const float *__restrict__ w, int k, float *__restrict__ s) {
    __shared__ float part[4];
    __shared__ int nanp[4];
    const float *row = w + (size_t)blockIdx.x * k;
    float m = 0.0f;
    int nan = 0;
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        const float v = row[i];
        nan |= v != v;
        m = fmaxf(m, fabsf(v));
    }
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off));
        nan |= __shfl_xor(nan, off);
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6] = m;
        nanp[threadIdx.x >> 6] = nan;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float mm = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
        if (nanp[0] | nanp[1] | nanp[2] | nanp[3]) mm = __builtin_nanf("");
        s[blockIdx.x] = mm / 127.0f;
    }
}

__device__ __forceinline__ float f16r(float x) {
    asm volatile("" : "+v"(x));
    return (float)(_Float16)x;
}

// q4GroupScale (gptq.go:764-791) of the 32 values held one per lane by lanes
// g .. g+31 of the wavefront (the caller's x is the lane's value): peak = the
// value of largest magnitude, lowest column on ties; 16 FP16 candidates
// f16(peak / -8 * (1 - 0.02 step)); the candidate with the smallest float64
// sum of squared errors, the first on ties. Every lane returns the result.
__device__ float q4_group_scale_wave(float x, int g) {
    const int lane = threadIdx.x & 63;
    const bool in = lane >= g && lane < g + 32;
    float pv = in ? x : 0.0f;
    int pi = in ? lane : 64;
    for (int off = 1; off < 64; off <<= 1) {
        const float ov = __shfl_xor(pv, off);
        const int oi = __shfl_xor(pi, off);
        if (fabsf(ov) > fabsf(pv) || (fabsf(ov) == fabsf(pv) && oi < pi)) {
            pv = ov;
            pi = oi;
        }
    }
    const float peak = pv;  // the same on every lane
    if (peak == 0.0f) return 0.0f;
    float best = 0.0f;
    double bestErr = INFINITY;
    for (int step = 0; step < 16; ++step) {
        const float d = f16r(peak / -8.0f * (1.0f - 0.02f * (float)step));
        if (d == 0.0f) continue;
        double e = 0.0;
        if (in) {
            const float qv = fminf(7.0f, fmaxf(-8.0f, rintf(x / d)));
            const double diff = (double)x - (double)qv * (double)d;
            e = diff * diff;
        }
        for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
        if (e < bestErr) {
            best = d;
            bestErr = e;
        }
    }
    return best;
}

struct RoundArgs {
    float *w;              // [n][k], updated in place
    const float *u;        // [k][k]
    float *errs;           // [n][kRoundBlock]
    uint8_t *codes;        // 8-bit: int8 [n][k]; 4-bit: [n][k/2]
    uint8_t *scales;       // 8-bit: fp32 [n]; 4-bit: fp16 [n][k/32]
    const float *rowScale; // 8-bit row scales
    int n, k, i1, b, bits;
};

// One 128-column block of gptqRound (gptq.go:686-745): wavefront w of the
// workgroup takes weight row blockIdx.x * 8 + w; lane l holds block columns l
// and l + 64. The block's U rows sit in LDS.
__global__ __launch_bounds__(64 * kRowsPerBlock) void gptq_round_block_kernel(const RoundArgs a) {
    __shared__ float Ub[kRoundBlock][kRoundBlock + 1];
    const int b = a.b, i1 = a.i1, k = a.k;
    for (int e = threadIdx.x; e < b * b; e += blockDim.x) {
        const int p = e / b, q = e - p * b;
        Ub[p][q] = a.u[(size_t)(i1 + p) * k + i1 + q];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (r >= a.n) return;  // whole wavefronts: the row is wave-uniform
    float *row = a.w + (size_t)r * k + i1;
    float v[2];
    int code[2] = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h) v[h] = lane + 64 * h < b ? row[lane + 64 * h] : 0.0f;
    float s = a.bits == 8 ? a.rowScale[r] : 0.0f;
    for (int c = 0; c < b; ++c) {
        const int slot = c >> 6, owner = c & 63;
        if (a.bits == 4 && (c & 31) == 0) {
            s = q4_group_scale_wave(slot ? v[1] : v[0], owner);
            if (lane == 0)
                ((uint16_t *)a.scales)[(size_t)r * (k / 32) + (i1 + c) / 32] =
                    __builtin_bit_cast(uint16_t, (_Float16)s);
        }
        const float lo = a.bits == 8 ? -127.0f : -8.0f, hi = a.bits == 8 ? 127.0f : 7.0f;
        // The owner lane's value, the same on every lane.
        const float wc = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, slot ? v[1] : v[0]), owner));
        const float q = s != 0.0f ? fminf(hi, fmaxf(lo, rintf(wc / s))) : 0.0f;
        const float qv = __fmul_rn(q, s);
        const float e = __fsub_rn(wc, qv) / Ub[c][c];
        if (lane == owner) {
            if (slot) {
                v[1] = qv;
                code[1] = (int)q;
            } else {
                v[0] = qv;
                code[0] = (int)q;
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = lane + 64 * h;
            if (j > c && j < b) v[h] = __fsub_rn(v[h], __fmul_rn(e, Ub[c][j]));
        }
        if (lane == 0) a.errs[(size_t)r * kRoundBlock + c] = e;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int j = lane + 64 * h;
        if (j < b) row[j] = v[h];
        if (a.bits == 8) {
            if (j < b) a.codes[(size_t)r * k + i1 + j] = (uint8_t)(int8_t)code[h];
        } else {
            // Byte (col/32)*16 + col%16 holds col (low nibble) and col+16
            // (high nibble), both stored plus 8.
            const int up = __shfl_down(code[h], 16);
            const int col = i1 + j;
            if (j < b && (col & 31) < 16)
                a.codes[(size_t)r * (k / 2) + (col / 32) * 16 + (col & 15)] =
                    (uint8_t)((code[h] + 8) | ((up + 8) << 4));
        }
    }
}

}  // namespace

namespace gphq {

// C [M][N] (row stride ldc) = A [M][K] . B^T for B [N][K] (row-major, strides
// lda / ldb), fp32 with fp32 sums; with accumulate, C += the product (the
// whole sum formed first and added once, as `c[i] += d[i]` after a separate
// product). The calibration pass's projections and residual adds.
int sgemm_abt(int M, int N, int K, const float *a, long lda, const float *b, long ldb, float *c, long ldc,
              bool accumulate, hipStream_t st) {
    return sgemm<0, 1>(M, N, K, 1.0f, a, lda, b, ldb, c, ldc, accumulate, st);
}

}  // namespace gphq

extern "C" {

int64_t gphq_gptq_work_bytes(int64_t k) {
    if (k <= 0 || k > 65536) return GPHQ_ERR_DIMENSIONS;
    return 4 * k * k + 4 * (int64_t)kPanel * k + 256;
}

int gphq_gptq_factor(const float *x_dev, int64_t rows, int64_t k, float *u_dev, uint8_t *dead_dev, void *work_dev,
                     int64_t work_bytes, void *stream) {
    if (!x_dev || !u_dev || !dead_dev || !work_dev || rows < 1 || k < 1 || k > 65536 || rows > INT32_MAX)
        return GPHQ_ERR_DIMENSIONS;
    if (work_bytes < gphq_gptq_work_bytes(k)) return GPHQ_ERR_DIMENSIONS;
    hipStream_t st = (hipStream_t)stream;
    const int n = (int)k;
    const size_t nn = (size_t)n * n;
    const unsigned eb = (unsigned)((nn + 255) / 256);
    float *x = (float *)work_dev;  // X = L^-1
    // L11^-1 of the current panel: 2080 doubles (only read when n > 64, where
    // they fit the 64 n floats here with the alignment's 4 bytes).
    double *inv = (double *)(((uintptr_t)(x + nn) + 7) & ~(uintptr_t)7);
    int *bad = (int *)((char *)work_dev + gphq_gptq_work_bytes(k) - 64);
    float *A = u_dev;
    // A = J H J, H = X^T X (gptq.go:606-622), its lower triangle; dead channels and damping.
    const SgemmArgs g{n, n, (int)rows, 1.0f, x_dev, x_dev, A, n, n, n, 0, vec16(x_dev, n), vec16(x_dev, n)};
    const long t64 = (n + 63) / 64;
    hipLaunchKernelGGL((sgemm_kernel<1, 0, 64, 64, kUpperReversed>), dim3((unsigned)(t64 * (t64 + 1) / 2)), dim3(256),
                       0, st, g);
    GPHQ_TRY(launch_status());
    hipLaunchKernelGGL(gptq_damp_kernel, dim3(1), dim3(1024), 0, st, A, n, dead_dev, bad);
    GPHQ_TRY(launch_status());
    // Lower Cholesky in place (gptq_linalg.go:68-132), the inverses of the
    // diagonal blocks into x on the way.
    hipLaunchKernelGGL(chol_first_kernel, dim3(1), dim3(256), 0, st, A, n, x,
                       n > kPanel ? inv : nullptr, bad);
    GPHQ_TRY(launch_status());
    for (int j0 = 0; j0 < n; j0 += kPanel) {
        const int m = std::max(0, n - j0 - kPanel);
        const int below = (m + 31) / 32, left = j0 / 32;
        if (below + left > 0)
            hipLaunchKernelGGL(chol_panel_kernel, dim3((unsigned)(below + left)), dim3(256), 0, st, A, x, n, j0,
                               below, inv);
        GPHQ_TRY(launch_status());
        if (m == 0) break;
        const long tiles = (m + 63) / 64, tri = tiles * (tiles + 1) / 2;
        hipLaunchKernelGGL(chol_update_kernel, dim3((unsigned)(tri + tiles * (j0 / 64 + 1))), dim3(256), 0, st, A, n,
                           j0, (int)tri, x, inv, bad, vec16(A, n) & vec16(x, n));
        GPHQ_TRY(launch_status());
    }
    hipLaunchKernelGGL(u_from_x_kernel, dim3(eb), dim3(256), 0, st, x, u_dev, n);
    GPHQ_TRY(launch_status());
    int flag = 0;
    GPHQ_TRY(hip_status(hipMemcpyAsync(&flag, bad, sizeof(int), hipMemcpyDeviceToHost, st)));
    GPHQ_TRY(hip_status(hipStreamSynchronize(st)));
    return flag ? GPHQ_ERR_NOT_POSITIVE_DEFINITE : GPHQ_OK;
}

int64_t gphq_gptq_round_work_bytes(int64_t n, int64_t k) {
    if (n <= 0 || k <= 0) return GPHQ_ERR_DIMENSIONS;
    return 4 * n * kRoundBlock + 4 * n;
}

int gphq_gptq_round(float *w_dev, int64_t n, int64_t k, const float *u_dev, const uint8_t *dead_dev, int bits,
                    void *codes_dev, void *scales_dev, void *work_dev, int64_t work_bytes, void *stream) {
    if (bits != 8 && bits != 4) return GPHQ_ERR_UNSUPPORTED;
    if (!w_dev || !u_dev || !dead_dev || !codes_dev || !scales_dev || !work_dev || n < 1 || k < 1 ||
        n > INT32_MAX || k > 65536 || (bits == 4 && k % 32))
        return GPHQ_ERR_DIMENSIONS;
    if (work_bytes < gphq_gptq_round_work_bytes(n, k)) return GPHQ_ERR_DIMENSIONS;
    hipStream_t st = (hipStream_t)stream;
    float *errs = (float *)work_dev;
    float *rs = errs + (size_t)n * kRoundBlock;
    const size_t nk = (size_t)n * k;
    hipLaunchKernelGGL(zero_dead_kernel, dim3((unsigned)((nk + 255) / 256)), dim3(256), 0, st, w_dev, (int)n, (int)k,
                       dead_dev);
    GPHQ_TRY(launch_status());
    if (bits == 8) {
        hipLaunchKernelGGL(row_scale_kernel, dim3((unsigned)n), dim3(256), 0, st, w_dev, (int)k, rs);
        GPHQ_TRY(launch_status());
        GPHQ_TRY(hip_status(hipMemcpyAsync(scales_dev, rs, (size_t)n * 4, hipMemcpyDeviceToDevice, st)));
    }
    RoundArgs ra{};
    ra.w = w_dev;
    ra.u = u_dev;
    ra.errs = errs;
    ra.codes = (uint8_t *)codes_dev;
    ra.scales = (uint8_t *)scales_dev;
    ra.rowScale = rs;
    ra.n = (int)n;
    ra.k = (int)k;
    ra.bits = bits;
    for (int i1 = 0; i1 < k; i1 += kRoundBlock) {
        const int b = (int)std::min<int64_t>(kRoundBlock, k - i1), i2 = i1 + b;
        ra.i1 = i1;
        ra.b = b;
        hipLaunchKernelGGL(gptq_round_block_kernel, dim3((unsigned)((n + kRowsPerBlock - 1) / kRowsPerBlock)),
                           dim3(64 * kRowsPerBlock), 0, st, ra);
        GPHQ_TRY(launch_status());
        if (i2 < k)  // W[:, i2:] -= E U[i1:i2, i2:] (gptq.go:746-760)
            GPHQ_TRY((sgemm<0, 0>((int)n, (int)(k - i2), b, -1.0f, errs, kRoundBlock, u_dev + (size_t)i1 * k + i2, k,
                                 w_dev + i2, k, true, st)));
    }
    return GPHQ_OK;
}

}  // extern "C"
