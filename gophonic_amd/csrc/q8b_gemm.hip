// Block-32 int8 GEMM on MI355X: benchmark configuration 2 as worded there
// (activations and weights each with one fp32 scale per 32-value block). The
// reference has no such function: its q8gemm int8 path scales per row
// (int8.go:106-211, gphq_q8gemm_*). Each 32-value block is quantized with
// WorkspaceI8's per-row rule (int8.go:106-168), and the product sums, per
// output and in block order, acc = fmaf(float(dot_b), da[r][b] * dw[c][b], acc)
// with dot_b the exact int32 block product, so results are bit-exact against
// the oracle's restatement of that sum.
//
// One v_mfma_i32_16x16x32_i8 (q8b_tile_kernel, up to 16 rows q8b_small_kernel)
// or v_mfma_i32_32x32x32_i8 (q8b_gemm_kernel, the 128 x 192 tiles) takes exactly
// one 32-value block, so every block's int32 products come out of one MFMA with
// a zero accumulator; the fp32 scale-accumulate that follows is VALU work (three
// instructions per output and block), which bounds these kernels well below the
// int8 MFMA rate. One row takes sdot4 chains (q8b_gemv_kernel).
#include <type_traits>

#include "common.h"

using namespace gphq;

namespace {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Scale = max/127 and inverse = 127/max per (row, 32-value block), both 0
// unless 0 < max < inf (int8.go:106-119), codes RNE(x * inverse) saturated to
// int8 (int8.go:163-168). Latency-bound: eight lanes share a block, one float4
// each, so a wavefront reads 1 KiB in one load and all of it is in flight at
// once (one lane per block read lines in eight passes, 128 bytes apart). The
// maximum is taken over the bits of |x|, where infinities and NaN order above
// every finite value. Float4s are numbered through all rows (codes and scales
// have no gaps between rows), PER a thread, 256 apart, so rows of any length
// fill the wavefronts.
template <int PER>
__global__ __launch_bounds__(256) void q8b_quantize_kernel(const float *__restrict__ x, long units, uint32_t perRow,
                                                           uint32_t rcp, long stride, int8_t *__restrict__ q,
                                                           float *__restrict__ d) {
    const long u0 = (long)blockIdx.x * (256 * PER) + threadIdx.x;
    float4 f[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const long u = min(u0 + 256 * i, units - 1);
        long at = u * 4;
        if (stride != perRow * 4L) {
            long r = units <= UINT32_MAX ? (long)__umulhi((uint32_t)u, rcp) : u / perRow;
            r += u - r * perRow >= perRow;
            at = r * stride + (u - r * perRow) * 4;
        }
        f[i] = *(const float4 *)(x + at);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const long u = u0 + 256 * i;
        if (u >= units) return;  // whole groups of eight lanes: units is a multiple of 8
        const float v[4] = {f[i].x, f[i].y, f[i].z, f[i].w};
        uint32_t mb = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) mb = max(mb, __float_as_uint(v[j]) & 0x7fffffffu);
        mb = max(mb, (uint32_t)__builtin_amdgcn_mov_dpp((int)mb, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
        mb = max(mb, (uint32_t)__builtin_amdgcn_mov_dpp((int)mb, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
        mb = max(mb, (uint32_t)__builtin_amdgcn_mov_dpp((int)mb, 0x141, 0xF, 0xF, true));  // row_half_mirror
        float s = 0.0f, inv = 0.0f;
        if (mb > 0 && mb < 0x7f800000u) {
            const float mx = __uint_as_float(mb);
            s = __fdiv_rn(mx, 127.0f);
            inv = __fdiv_rn(127.0f, mx);
        }
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float p = __fmul_rn(v[j], inv);
            float c = p != p ? 0.0f : rintf(p);
            c = fminf(127.0f, fmaxf(-128.0f, c));
            word |= (uint32_t)(uint8_t)(int8_t)(int)c << (8 * j);
        }
        *(uint32_t *)(q + u * 4) = word;
        if ((u & 7) == 0) d[u >> 3] = s;
    }
}

struct Q8bArgs {
    const int8_t *qa;
    const float *da;
    const int8_t *qw;
    const float *dw;
    float *y;
    int m, k, n, gridM, gridN;
};

// 16-byte chunk c of a row of KSB*32 bytes in LDS, swizzled within each
// 128-byte half by the row (big_swz), so fragment reads of consecutive rows
// at one chunk hit distinct banks.
__device__ __forceinline__ int q8b_swz(int row, int c) { return (c & ~7) | big_swz(row, c & 7); }

// BM x BN output tiles, WGM x WGN wavefronts of (BM/WGM) x (BN/WGN) as 32x32
// MFMA tiles. Per K step of KSB blocks (KSB*32 bytes) both code tiles pass
// through LDS in rows of 16-byte chunks (q8b_swz), the step's block scales as
// [block][row] floats; double buffered, the next step's global loads one step
// ahead in registers. Rows past m or n load row m-1 / n-1 and are not
// stored; blocks past k are skipped, and so are the scale-accumulates of a
// tile's rows 16..31 when they are all past m.
//
// Per block the wavefront issues the MFMAs of block b+1 before the
// scale-accumulate of block b (two sets of int32 results), so the matrix
// cores run beside the VALU chain; the chain itself keeps block order.
template <int BM, int BN, int WGM, int WGN, int KSB>
__global__ __launch_bounds__(64 * WGM * WGN) void q8b_gemm_kernel(const Q8bArgs a) {
    constexpr int NT = 64 * WGM * WGN;
    constexpr int TI = BM / WGM / 32, TJ = BN / WGN / 32;
    constexpr int CH = 2 * KSB;                          // 16-byte chunks per row and step
    constexpr int AL = BM * CH / NT, BL = BN * CH / NT;  // chunks per thread and step
    constexpr int SU = (BM + BN) * (KSB / 4);            // float4 scale units per step
    constexpr int SL = (SU + NT - 1) / NT;
    static_assert(AL * NT == BM * CH && BL * NT == BN * CH && KSB % 4 == 0, "loader split");
    __shared__ i32x4 As[2][BM * CH];
    __shared__ i32x4 Bs[2][BN * CH];
    __shared__ float Sa[2][KSB][BM];
    __shared__ float Sb[2][KSB][BN];
    int bm, bn;
    tile_order(blockIdx.x, a.gridM, a.gridN, bm, bn);
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wv / WGN, wn = wv % WGN;
    const int m0 = bm * BM, n0 = bn * BN;
    const int kb = a.k >> 5, steps = (kb + KSB - 1) / KSB;

    // Loader: unit u = i*NT + t is row u/CH, 16-byte chunk u%CH of the
    // step's bytes; chunks past k load zeros. Scale unit v = i*NT + t is one
    // float4 (four blocks) of A's row v (v < BM*KSB/4 ordering: row-major over
    // rows, then quads) or of B's row.
    // A full step (every chunk inside k, the usual case) loads without
    // per-chunk conditions. first marks the loads of step 1, which stay in
    // registers across the first step: relaxed atomic loads, so that the
    // compiler does not merge them with the in-loop loads of the same
    // registers into one load at the top of the loop (which would wait for
    // each step's codes as they are stored).
    i32x4 ar[AL], br[BL];
    float4 sr[SL];
    auto ld = [&](const int8_t *p, bool first) -> i32x4 {
        if (!first) return *(const i32x4 *)p;
        const long lo = __hip_atomic_load((const long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const long hi = __hip_atomic_load((const long *)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return i32x4{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
    };
    auto gload = [&](int st, bool first) {
        const int kbyte = st * KSB * 32;
        if (kbyte + KSB * 32 <= a.k) {
#pragma unroll
            for (int i = 0; i < AL; ++i) {
                const int u = i * NT + t, row = u / CH, ch = u % CH;
                ar[i] = ld(a.qa + (long)min(m0 + row, a.m - 1) * a.k + kbyte + ch * 16, first);
            }
#pragma unroll
            for (int i = 0; i < BL; ++i) {
                const int u = i * NT + t, row = u / CH, ch = u % CH;
                br[i] = ld(a.qw + (long)min(n0 + row, a.n - 1) * a.k + kbyte + ch * 16, first);
            }
        } else {
#pragma unroll
            for (int i = 0; i < AL; ++i) {
                const int u = i * NT + t, row = u / CH, ch = u % CH;
                const int gr = min(m0 + row, a.m - 1);
                ar[i] = kbyte + ch * 16 < a.k ? ld(a.qa + (long)gr * a.k + kbyte + ch * 16, first) : i32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (int i = 0; i < BL; ++i) {
                const int u = i * NT + t, row = u / CH, ch = u % CH;
                const int gr = min(n0 + row, a.n - 1);
                br[i] = kbyte + ch * 16 < a.k ? ld(a.qw + (long)gr * a.k + kbyte + ch * 16, first) : i32x4{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const int v = i * NT + t;
            float4 f = float4{0.f, 0.f, 0.f, 0.f};
            if (v < SU) {
                const int quad = v % (KSB / 4), row = v / (KSB / 4);
                const int b0 = st * KSB + quad * 4;
                float sv[4];
                if (row < BM) {
                    const float *sp = a.da + (long)min(m0 + row, a.m - 1) * kb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) sv[e] = b0 + e < kb ? sp[b0 + e] : 0.0f;
                } else {
                    const float *sp = a.dw + (long)min(n0 + row - BM, a.n - 1) * kb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) sv[e] = b0 + e < kb ? sp[b0 + e] : 0.0f;
                }
                f = float4{sv[0], sv[1], sv[2], sv[3]};
            }
            sr[i] = f;
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int u = i * NT + t, row = u / CH;
            As[buf][row * CH + q8b_swz(row, u % CH)] = ar[i];
        }
#pragma unroll
        for (int i = 0; i < BL; ++i) {
            const int u = i * NT + t, row = u / CH;
            Bs[buf][row * CH + q8b_swz(row, u % CH)] = br[i];
        }
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const int v = i * NT + t;
            if (v < SU) {
                const int quad = v % (KSB / 4), row = v / (KSB / 4);
                float *dst = row < BM ? &Sa[buf][quad * 4][row] : &Sb[buf][quad * 4][row - BM];
                const int stride = row < BM ? BM : BN;
                dst[0] = sr[i].x, dst[stride] = sr[i].y, dst[2 * stride] = sr[i].z, dst[3 * stride] = sr[i].w;
            }
        }
    };

    f32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16{};
    // Row tile i's rows 16..31 hold rows of the matrix (else their
    // scale-accumulates are skipped; the wave takes the branch as one).
    bool hi[TI], allhi = true;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        hi[i] = m0 + wm * (32 * TI) + 32 * i + 16 < a.m;
        allhi = allhi && hi[i];
    }
    gload(0, false);
    lstore(0);
    if (steps > 1) gload(1, true);
    __syncthreads();
    const int fr = lane & 31, fh = lane >> 5;
    for (int st = 0; st < steps; ++st) {
        const int cur = st & 1;
        const int nb = min(KSB, kb - st * KSB);
        // The step's MFMAs run in units (block b, row tile i, column tile j),
        // block-major; unit u+1's MFMA is issued before unit u's
        // scale-accumulate, so the matrix cores work beside the VALU chain.
        constexpr int UN = KSB * TI * TJ;
        auto issue = [&](int u, i32x16 &d) {
            const int b = u / (TI * TJ), i = (u / TJ) % TI, j = u % TJ;
            const int c = 2 * b + fh;
            const int ra = wm * (32 * TI) + 32 * i + fr, rb = wn * (32 * TJ) + 32 * j + fr;
            d = __builtin_amdgcn_mfma_i32_32x32x32_i8(As[cur][ra * CH + q8b_swz(ra, c)],
                                                     Bs[cur][rb * CH + q8b_swz(rb, c)], i32x16{}, 0, 0, 0);
        };
        // acc = fmaf(float(dot), da * dw, acc) for unit u. This lane's 16
        // results of a tile are 4 runs of 4 consecutive rows; its column's
        // weight scale is one float. FULL: a whole step of blocks and every
        // row tile's rows 16..31 inside m (no conditions in the loop).
        auto apply = [&](auto full_c, int u, const i32x16 &d) {
            constexpr bool FULL = decltype(full_c)::value;
            const int b = u / (TI * TJ), i = (u / TJ) % TI, j = u % TJ;
            const float sb = Sb[cur][b][wn * (32 * TJ) + 32 * j + fr];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (!FULL && q >= 2 && !hi[i]) continue;
                const float4 s4 = *(const float4 *)&Sa[cur][b][wm * (32 * TI) + 32 * i + 8 * q + 4 * fh];
                const float sa[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float s = __fmul_rn(sa[e], sb);
                    acc[i][j][4 * q + e] = __builtin_fmaf((float)d[4 * q + e], s, acc[i][j][4 * q + e]);
                }
            }
        };
        auto units = [&](auto full_c) {
            constexpr bool FULL = decltype(full_c)::value;
            const int un = FULL ? UN : nb * TI * TJ;
            i32x16 d0, d1;
            issue(0, d0);
#pragma unroll
            for (int u = 0; u < UN; u += 2) {
                if (FULL || u < un) {
                    if (FULL || u + 1 < un) issue(u + 1, d1);
                    apply(full_c, u, d0);
                }
                if (FULL || u + 1 < un) {
                    if (u + 2 < UN && (FULL || u + 2 < un)) issue(u + 2, d0);
                    apply(full_c, u + 1, d1);
                }
            }
        };
        if (nb == KSB && allhi)
            units(std::true_type{});
        else
            units(std::false_type{});
        if (st + 1 < steps) {
            lstore(cur ^ 1);
            if (st + 2 < steps) gload(st + 2, false);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int col = n0 + wn * (32 * TJ) + 32 * j + fr;
            if (col >= a.n) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm * (32 * TI) + 32 * i + 8 * (e >> 2) + 4 * fh + (e & 3);
                if (row < a.m) a.y[(long)row * a.n + col] = acc[i][j][e];
            }
        }
}

// BM x BN output tiles, WGM x WGN wavefronts of 16 TI x 16 TJ outputs, one
// v_mfma_i32_16x16x32_i8 per 16 x 16 outputs and 32-value block. The
// scale-accumulate is three VALU instructions per output and block (128 x
// 12288 outputs at K = 4096: 15 us if every SIMD had the same share), so the
// tile decides how evenly the SIMDs share it: 32 x 32 MFMAs in 64 x 64 tiles gave
// half the CUs twice the others' work there, 64 x 96 tiles of these give every
// SIMD six 16 x 16 tiles (44.6 -> 36.8 us).
// Codes pass through LDS in rows of KSB * 32 bytes, 16-byte chunks
// XOR-swizzled (swz) so that the 8-byte fragment reads of 16 rows at one chunk
// cover all 64 banks; weight scales stay [row][block] (one float4 read per
// four blocks), activation scales [block][row]. Two LDS buffers; the next
// step's loads are issued before a step's products and stored after them.
// Rows past m or n and chunks past k repeat the last one: their rows are not
// stored and their blocks are skipped, and so are 16-row tiles past m. The
// chain per output is in block order, the same bits as the other kernels.
template <int TI, int TJ, int WGM, int WGN, int KSB>
__global__ __launch_bounds__(64 * WGM * WGN) void q8b_tile_kernel(const Q8bArgs a) {
    constexpr int NT = 64 * WGM * WGN, BM = 16 * TI * WGM, BN = 16 * TJ * WGN;
    constexpr int CH = 2 * KSB, UNITS = (BM + BN) * CH, LU = (UNITS + NT - 1) / NT;
    constexpr int SU = (BM + BN) * (KSB / 4), SL = (SU + NT - 1) / NT, SBS = KSB + 4;
    static_assert((KSB == 4 || KSB == 8) && BM * CH % 64 == 0, "swizzle; whole wavefronts load one operand");
    __shared__ __align__(16) int8_t cs[2][(BM + BN) * KSB * 32];
    __shared__ __align__(16) float Sa[2][KSB][BM];
    __shared__ __align__(16) float Sb[2][BN][SBS];
    int bm, bn;
    tile_order(blockIdx.x, a.gridM, a.gridN, bm, bn);
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wv / WGN, wn = wv % WGN, m0 = bm * BM, n0 = bn * BN;
    const int kb = a.k >> 5, steps = (kb + KSB - 1) / KSB;
    auto swz = [](int row, int c) { return KSB == 8 ? c ^ (row & 15) : c ^ ((row >> 1) & 7); };
    // Unit u = i * NT + t: 16-byte chunk u % CH of row u / CH, A's rows first.
    const int8_t *src[LU];
    int dst[LU];
#pragma unroll
    for (int i = 0; i < LU; ++i) {
        const int u = min(i * NT + t, UNITS - 1), row = u / CH, ch = u % CH;
        src[i] = row < BM ? a.qa + (size_t)min(m0 + row, a.m - 1) * a.k : a.qw + (size_t)min(n0 + row - BM, a.n - 1) * a.k;
        dst[i] = row * (KSB * 32) + swz(row, ch) * 16;
    }
    const float *ssrc[SL];
#pragma unroll
    for (int i = 0; i < SL; ++i) {
        const int row = min(i * NT + t, SU - 1) / (KSB / 4);
        ssrc[i] = row < BM ? a.da + (size_t)min(m0 + row, a.m - 1) * kb : a.dw + (size_t)min(n0 + row - BM, a.n - 1) * kb;
    }
    i32x4 cr[LU];
    f32x4 sr[SL];
    auto gload = [&](int st) {
#pragma unroll
        for (int i = 0; i < LU; ++i) {
            const int u = min(i * NT + t, UNITS - 1);
            cr[i] = *(const i32x4 *)(src[i] + min(st * (KSB * 32) + (u % CH) * 16, a.k - 16));
        }
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const int b0 = st * KSB + min(i * NT + t, SU - 1) % (KSB / 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) sr[i][e] = ssrc[i][min(b0 + e, kb - 1)];
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LU; ++i)
            if ((i + 1) * NT <= UNITS || i * NT + t < UNITS) *(i32x4 *)&cs[buf][dst[i]] = cr[i];
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const int v = i * NT + t;
            if (v >= SU) continue;
            const int quad = v % (KSB / 4), row = v / (KSB / 4);
            if (row < BM) {
#pragma unroll
                for (int e = 0; e < 4; ++e) Sa[buf][quad * 4 + e][row] = sr[i][e];
            } else {
                *(f32x4 *)&Sb[buf][row - BM][quad * 4] = sr[i];
            }
        }
    };
    const int c = lane & 15, g = lane >> 4;
    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{};
    int ti = 0;  // the wavefront's 16-row tiles that hold rows of the matrix
#pragma unroll
    for (int i = 0; i < TI; ++i) ti += m0 + (wm * TI + i) * 16 < a.m;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int st = 0; st < steps; ++st) {
        const int cur = st & 1, nb = min(KSB, kb - st * KSB);
        if (st + 1 < steps) gload(st + 1);
        auto frag = [&](int row, int b) {
            return *(const long *)&cs[cur][row * (KSB * 32) + swz(row, 2 * b + (g >> 1)) * 16 + (g & 1) * 8];
        };
        // Block b + 1's MFMAs are issued before block b's scale-accumulates.
        auto issue = [&](int b, i32x4(&d)[TI][TJ]) {
            long av[TI], bv[TJ];
#pragma unroll
            for (int i = 0; i < TI; ++i) av[i] = frag((wm * TI + i) * 16 + c, b);
#pragma unroll
            for (int j = 0; j < TJ; ++j) bv[j] = frag(BM + (wn * TJ + j) * 16 + c, b);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    d[i][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[i], bv[j], i32x4{}, 0, 0, 0);
        };
        f32x4 sb[TJ];
        auto apply = [&](int b, const i32x4(&d)[TI][TJ]) {
            if (b % 4 == 0)
#pragma unroll
                for (int j = 0; j < TJ; ++j) sb[j] = *(const f32x4 *)&Sb[cur][(wn * TJ + j) * 16 + c][b];
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const f32x4 sa = *(const f32x4 *)&Sa[cur][b][(wm * TI + i) * 16 + 4 * g];
#pragma unroll
                for (int j = 0; j < TJ; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[i][j][e] = __builtin_fmaf((float)d[i][j][e], __fmul_rn(sa[e], sb[j][b % 4]), acc[i][j][e]);
            }
        };
        i32x4 d[2][TI][TJ];
        if (ti > 0 && nb == KSB) {
            issue(0, d[0]);
#pragma unroll
            for (int b = 0; b < KSB; ++b) {
                if (b + 1 < KSB) issue(b + 1, d[(b + 1) & 1]);
                apply(b, d[b & 1]);
            }
        } else if (ti > 0) {
#pragma unroll
            for (int b = 0; b < KSB; ++b)
                if (b < nb) {
                    issue(b, d[0]);
                    apply(b, d[0]);
                }
        }
        if (st + 1 < steps) lstore(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int col = n0 + (wn * TJ + j) * 16 + c;
            if (col >= a.n) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + (wm * TI + i) * 16 + 4 * g + e;
                if (row < a.m) a.y[(size_t)row * a.n + col] = acc[i][j][e];
            }
        }
}

// M <= 16: one wavefront (and block) per 16 weight rows, all activation rows
// in one tile. A step is 128 bytes of K (four
// blocks): the wavefront loads its 16 weight rows and 16 activation
// rows with 16-byte loads, eight lanes per row (whole 128-byte lines), their
// block scales with one float per lane, and keeps D steps of loads in
// flight in a register ring. Each step passes through the wavefront's own
// LDS (rows padded to 144 bytes), from which every block is one
// v_mfma_i32_16x16x32_i8 (lane l supplies bytes
// 8(l/16)..+8 of the block for row or column l%16 and receives rows
// 4(l/16)..+3 of column l%16). The chain per output is the tiled kernel's,
// in block order: acc = fmaf(float(dot_b), da * dw, acc), so the results
// are the same bit for bit.
template <int D>
__global__ __launch_bounds__(64) void q8b_small_kernel(const Q8bArgs a) {
    constexpr int RS = 144;             // LDS row stride of the code tiles, bytes
    static_assert(D % 2 == 0, "the ring pairs with two LDS buffers");
    __shared__ __align__(16) int8_t wl[2][16 * RS];
    __shared__ __align__(16) int8_t al[2][16 * RS];
    __shared__ float swl[2][16][4];                // [buffer][weight row][block of the step]
    __shared__ __align__(16) float sal[2][4][16];  // [buffer][block of the step][activation row]
    const int lane = threadIdx.x, kb = a.k >> 5, steps = kb >> 2;
    const int n0 = blockIdx.x * 16;
    const int lr = lane >> 3, lc = lane & 7;  // loader: row lr (+8h), 16-byte chunk lc
    const int c = lane & 15, g = lane >> 4;   // MFMA lane: row/column c, byte group g
    const int8_t *wp[2];
    wp[0] = a.qw + (size_t)min(n0 + lr, a.n - 1) * a.k + lc * 16;
    wp[1] = a.qw + (size_t)min(n0 + lr + 8, a.n - 1) * a.k + lc * 16;
    const int8_t *ap[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) ap[h] = a.qa + (size_t)min(lr + 8 * h, a.m - 1) * a.k + lc * 16;
    // Scales: lane l takes block l%4 of the step of weight and activation row l/4.
    const float *dwp = a.dw + (size_t)min(n0 + (lane >> 2), a.n - 1) * kb + (lane & 3);
    const float *dap = a.da + (size_t)min(lane >> 2, a.m - 1) * kb + (lane & 3);
    i32x4 wr[D][2], ar[D][2];
    float sw[D], sa[D];
    auto load = [&](int p, int st, bool first) {
        const size_t off = (size_t)st * 128;
        auto ld = [&](const int8_t *q, bool stream) -> i32x4 {
            if (!first) return stream ? __builtin_nontemporal_load((const i32x4 *)q) : *(const i32x4 *)q;
            // Relaxed atomic loads for the first fill: with plain loads at
            // both the ring's entry and its refill the compiler merges them
            // into one load at the top of the loop, which waits for each
            // step as it is used.
            const long lo = __hip_atomic_load((const long *)q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const long hi = __hip_atomic_load((const long *)q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return i32x4{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
        };
        auto lf = [&](const float *q) -> float {
            return first ? __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : *q;
        };
        wr[p][0] = ld(wp[0] + off, true);
        wr[p][1] = ld(wp[1] + off, true);
#pragma unroll
        for (int h = 0; h < 2; ++h) ar[p][h] = ld(ap[h] + off, false);
        sw[p] = lf(dwp + 4 * st);
        sa[p] = lf(dap + 4 * st);
    };
    // Ring slot p to LDS buffer buf (this wavefront alone reads it back).
    auto stage = [&](int p, int buf) {
        *(i32x4 *)&wl[buf][lr * RS + lc * 16] = wr[p][0];
        *(i32x4 *)&wl[buf][(lr + 8) * RS + lc * 16] = wr[p][1];
#pragma unroll
        for (int h = 0; h < 2; ++h) *(i32x4 *)&al[buf][(lr + 8 * h) * RS + lc * 16] = ar[p][h];
        swl[buf][lane >> 2][lane & 3] = sw[p];
        sal[buf][lane & 3][lane >> 2] = sa[p];
    };
    f32x4 acc = f32x4{};
#pragma unroll
    for (int p = 0; p < D; ++p) load(p, min(p, steps - 1), true);
    stage(0, 0);
    load(0, min(D, steps - 1), false);
    // Step st is computed from LDS buffer st&1 while step st+1 is staged
    // into the other one, so the LDS round trip of a step overlaps the MFMAs
    // and scale-accumulates of the one before.
    for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
        for (int p = 0; p < D; ++p) {
            const int st = s0 + p, cur = p & 1;  // D is even, so st&1 == p&1
            const int pn = (p + 1) % D;
            stage(pn, cur ^ 1);
            load(pn, min(st + 1 + D, steps - 1), false);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const long wv = *(const long *)&wl[cur][c * RS + 32 * b + 8 * g];
                const float w1 = swl[cur][c][b];
                const long av = *(const long *)&al[cur][c * RS + 32 * b + 8 * g];
                const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, wv, i32x4{}, 0, 0, 0);
                const float4 s4 = *(const float4 *)&sal[cur][b][4 * g];
                const float s_[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf((float)d[e], __fmul_rn(s_[e], w1), acc[e]);
            }
            __builtin_amdgcn_wave_barrier();
            if (st + 1 >= steps) break;
        }
    }
    const int col = n0 + c;
    if (col < a.n) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 4 * g + e;
            if (row < a.m) a.y[(size_t)row * a.n + col] = acc[e];
        }
    }
}

// M = 1, K = 1024 KS: one wavefront per RG weight rows, streamed as whole
// rows (lane l takes bytes 16 l..+16 of each 1 KiB segment, so a load
// instruction covers 1 KiB of one row), RB rows of loads per batch and up to
// 128 VGPRs of them in flight (at K = 4096 all four rows at once). A row's
// block products are two lanes' sdot4 chains (exact int32) added by a lane
// swap; float(dot_b) and the scale product da[b] * dw[r][b] go to LDS, formed
// by the lanes that hold them, and once the RG rows are in, lane r runs
// output r's chain in block order, acc = fmaf(float(dot_b), da[b] * dw[r][b],
// acc): the same arithmetic as the tiled kernels, so the same bits. Measured
// on MI355X at config 2's shape (K = 4096, N = 12288, 56.6 MB a launch):
// 12.9-13.0 us with 4 rows per wavefront (3072 wavefronts), 13.2 with 8,
// 14.1 with 16, 13.4 with 2, against 19.3-19.8 us for q8b_small_kernel, whose
// wavefronts read 128 bytes of 16 rows per step.
template <int KS, int RG>
__global__ __launch_bounds__(64) void q8b_gemv_kernel(const Q8bArgs a) {
    constexpr int KB = 32 * KS;                                  // blocks per row
    constexpr int RB0 = KS >= 16 ? 1 : 16 / KS;
    constexpr int RB = RB0 < RG ? RB0 : RG;                      // rows per batch (RB * KS 16-byte loads)
    constexpr int NB = RG / RB;                                  // batches
    constexpr int NBUF0 = 32 / (RB * KS) > 0 ? 32 / (RB * KS) : 1;  // at most 128 VGPRs of codes in flight
    constexpr int NBUF = NB < NBUF0 ? NB : NBUF0;                // batches in flight
    static_assert(NB * RB == RG, "whole batches");
    constexpr int SPL = KB / 64;            // scale floats per lane and row
    static_assert(KS % 2 == 0 && KS <= 16, "whole 64-lane scale rows");
    __shared__ float dots[RG][KB + 1];      // float(dot); +1: lane r's chain reads stride KB + 1 words
    __shared__ float sw[RG][KB + 1];
    const int lane = threadIdx.x;
    const int n0 = blockIdx.x * RG;
    // The activation row: lane l's bytes of each segment, then its scales.
    i32x4 xa[KS];
#pragma unroll
    for (int j = 0; j < KS; ++j) xa[j] = *(const i32x4 *)(a.qa + 1024 * j + 16 * lane);
    i32x4 wr[NBUF][RB][KS];
    float sr[NBUF][RB][SPL];
    auto load = [&](int buf, int bt) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int row = min(n0 + bt * RB + r, a.n - 1);
            const int8_t *wp = a.qw + (size_t)row * a.k + 16 * lane;
#pragma unroll
            for (int j = 0; j < KS; ++j) wr[buf][r][j] = __builtin_nontemporal_load((const i32x4 *)(wp + 1024 * j));
            const float *sp = a.dw + (size_t)row * KB + SPL * lane;
#pragma unroll
            for (int i = 0; i < SPL; ++i) sr[buf][r][i] = sp[i];
        }
    };
#pragma unroll
    for (int b = 0; b < NBUF; ++b) load(b, b);
    float dar[SPL];  // the activation's block scales of this lane's scale slots
#pragma unroll
    for (int i = 0; i < SPL; ++i) dar[i] = a.da[SPL * lane + i];
#pragma unroll
    for (int bt = 0; bt < NB; ++bt) {
        const int buf = bt % NBUF;
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int rr = bt * RB + r;
#pragma unroll
            for (int j = 0; j < KS; ++j) {
                int d = __builtin_amdgcn_sdot4(wr[buf][r][j][0], xa[j][0], 0, false);
                d = __builtin_amdgcn_sdot4(wr[buf][r][j][1], xa[j][1], d, false);
                d = __builtin_amdgcn_sdot4(wr[buf][r][j][2], xa[j][2], d, false);
                d = __builtin_amdgcn_sdot4(wr[buf][r][j][3], xa[j][3], d, false);
                // Lanes 2t and 2t + 1 hold the halves of block 32 j + t.
                d += __builtin_amdgcn_mov_dpp(d, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
                if (!(lane & 1)) dots[rr][32 * j + (lane >> 1)] = (float)d;
            }
            // The chain's scale products da[b] * dw[r][b], formed here in parallel.
#pragma unroll
            for (int i = 0; i < SPL; ++i) sw[rr][SPL * lane + i] = __fmul_rn(dar[i], sr[buf][r][i]);
        }
        if (bt + NBUF < NB) load(buf, bt + NBUF);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < RG && n0 + lane < a.n) {
        float acc = 0.0f;
#pragma unroll 8
        for (int b = 0; b < KB; ++b) acc = __builtin_fmaf(dots[lane][b], sw[lane][b], acc);
        a.y[n0 + lane] = acc;
    }
}

template <int KS, int RG = 4>
int go_gemv(const Q8bArgs &a, hipStream_t st) {
    hipLaunchKernelGGL((q8b_gemv_kernel<KS, RG>), dim3((unsigned)((a.n + RG - 1) / RG)), dim3(64), 0, st, a);
    return launch_status();
}

template <int D>
int go_small(const Q8bArgs &a, hipStream_t st) {
    hipLaunchKernelGGL((q8b_small_kernel<D>), dim3((unsigned)((a.n + 15) / 16)), dim3(64), 0, st, a);
    return launch_status();
}

template <int BM, int BN, int WGM, int WGN, int KSB>
int launch_q8b(Q8bArgs a, hipStream_t st) {
    a.gridM = (a.m + BM - 1) / BM;
    a.gridN = (a.n + BN - 1) / BN;
    hipLaunchKernelGGL((q8b_gemm_kernel<BM, BN, WGM, WGN, KSB>), dim3((unsigned)(a.gridM * a.gridN)),
                       dim3(64 * WGM * WGN), 0, st, a);
    return launch_status();
}

template <int TI, int TJ, int WGM, int WGN, int KSB>
int launch_tile(Q8bArgs a, hipStream_t st) {
    constexpr int BM = 16 * TI * WGM, BN = 16 * TJ * WGN;
    a.gridM = (a.m + BM - 1) / BM;
    a.gridN = (a.n + BN - 1) / BN;
    hipLaunchKernelGGL((q8b_tile_kernel<TI, TJ, WGM, WGN, KSB>), dim3((unsigned)(a.gridM * a.gridN)),
                       dim3(64 * WGM * WGN), 0, st, a);
    return launch_status();
}

// The tile with the least time at rounds r = ceil(blocks / CUs), each tile
// with its least time (one block alone on a CU waits for its own loads), a
// fixed time and a time per round, in tenths of a microsecond at K = 4096,
// fitted to 33-512 rows at N = 600, 1000, 3396 and 12288 (K changes all
// of them alike). Over 17-768 rows and 22 shapes of K = 64 to 8192 and N = 594
// to 12288 with weights that no cache holds the tile taken is on average 0.2%
// behind the fastest of the five, at most 11% (384 x 64 -> 4000: 4.8 / 4.3 us). Measured at K = 4096 on MI355X, 32 x 32 / 64 x 48 / 64 x 64 /
// 64 x 96 / 128 x 192: 64 rows, N = 3396 (one round of each) 15.8 / 31.3 /
// 38.0 / 35.2 / - us; N = 12288, 64 rows 24.4 / 32.1 / 38.2 / 36.2 / -, 128 rows
// 43.6 / 39.2 / 44.6 / 36.8 / -, 160 rows 56.6 / 47.9 / 55.5 / 66.6 / -, 256
// rows 81.6 / 63.2 / 60.6 / 73.7 / 87.3, 512 rows 159 / 118 / 114 / 137 / 95.
// Small tiles win while several of them share a CU and hide each other's loads;
// large ones once LDS reads and not latency set the time. 32 rows, N = 12288 /
// 3396 and K = 8192, N = 600: 27.3 / 21.4 / 40.3 us with one wavefront per 16
// weight rows (q8b_small_kernel, kept for up to 16 rows: 18.9 / 12.8 / 22.0 us),
// 20.2 / 15.1 / 26.3 us in 32 x 32 tiles.
enum Tile { kTile32x32, kTile64x48, kTile64x64, kTile64x96, kTile128x192 };

Tile tile_for(int64_t m, int64_t n) {
    static constexpr struct {
        int bm, bn, least, fixed, round;
    } kTiles[] = {{32, 32, 160, 40, 66},
                  {64, 48, 320, 100, 140},
                  {64, 64, 380, 100, 170},
                  {64, 96, 345, 20, 345},
                  {128, 192, 870, 0, 920}};
    int best = 0;
    int64_t shortest = INT64_MAX;
    const int64_t cus = device_cus();
    for (int i = 0; i < 5; ++i) {
        const int64_t blocks = ((m + kTiles[i].bm - 1) / kTiles[i].bm) * ((n + kTiles[i].bn - 1) / kTiles[i].bn);
        const int64_t t = kTiles[i].fixed + (blocks + cus - 1) / cus * kTiles[i].round;
        const int64_t time = t < kTiles[i].least ? kTiles[i].least : t;
        if (time < shortest) shortest = time, best = i;
    }
    return (Tile)best;
}

}  // namespace

extern "C" {

int gphq_q8b_quantize(const float *x_dev, int64_t rows, int64_t k, int64_t x_stride, int8_t *q_dev, float *d_dev,
                      void *stream) {
    if (rows < 0 || k < 0 || k % 32 || x_stride < k || x_stride % 4 || rows > INT32_MAX || k > INT32_MAX)
        return GPHQ_ERR_DIMENSIONS;
    if (rows == 0 || k == 0) return GPHQ_OK;
    if (!x_dev || !q_dev || !d_dev) return GPHQ_ERR_DIMENSIONS;
    const uint32_t perRow = (uint32_t)(k / 4);
    const uint32_t rcp = (uint32_t)((1ull << 32) / perRow);
    const long units = (long)rows * perRow;
    // Two loads a thread once there are several rounds of the chip's wavefronts
    // (16384 x 4096: 59.8 us with one, 56.5 with two; 512 x 4096: 3.0 / 3.3).
    auto launch = [&](auto kernel, int per) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((units + 256 * per - 1) / (256 * per))), dim3(256), 0,
                           (hipStream_t)stream, x_dev, units, perRow, rcp, (long)x_stride, q_dev, d_dev);
    };
    if (units < 2 << 20) launch(q8b_quantize_kernel<1>, 1);
    else launch(q8b_quantize_kernel<2>, 2);
    return launch_status();
}

int gphq_q8b_gemm(const int8_t *qa_dev, const float *da_dev, const int8_t *qw_dev, const float *dw_dev, float *y_dev,
                  int64_t m, int64_t k, int64_t n, void *stream) {
    if (m < 0 || k < 0 || n < 0 || k % 32 || m > INT32_MAX || k > INT32_MAX || n > INT32_MAX)
        return GPHQ_ERR_DIMENSIONS;
    if (m == 0 || n == 0) return GPHQ_OK;
    if (!qa_dev || !da_dev || !qw_dev || !dw_dev || !y_dev) return GPHQ_ERR_DIMENSIONS;
    if (k == 0) return fill_f32(y_dev, (size_t)m * n, 0.0f, (hipStream_t)stream);
    Q8bArgs a{qa_dev, da_dev, qw_dev, dw_dev, y_dev, (int)m, (int)k, (int)n, 0, 0};
    hipStream_t st = (hipStream_t)stream;
    // Up to 16 rows with k a multiple of 128: one row at K = 2048, 4096, 8192 or
    // 12288 streams whole weight rows per wavefront, the others one wavefront
    // per 16 weight rows with a ring of steps in flight. Everything else takes
    // the tile of tile_for.
    if (m > 16 || k % 128) {
        switch (tile_for(m, n)) {
        case kTile32x32: return launch_tile<1, 1, 2, 2, 8>(a, st);
        case kTile64x48: return launch_tile<1, 3, 4, 1, 4>(a, st);
        case kTile64x64: return launch_tile<2, 2, 2, 2, 4>(a, st);
        case kTile64x96: return launch_tile<1, 3, 4, 2, 8>(a, st);
        case kTile128x192: return launch_q8b<128, 192, 4, 2, 4>(a, st);
        }
    }
    if (m == 1) {
        switch (k) {
        case 2048: return go_gemv<2>(a, st);
        case 4096: return go_gemv<4>(a, st);
        case 8192: return go_gemv<8>(a, st);
        case 12288: return go_gemv<12>(a, st);
        }
    }
    return go_small<8>(a, st);  // a ring of eight steps in flight
}

}  // extern "C"
