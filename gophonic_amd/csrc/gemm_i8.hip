// int8 x int8 GEMM with exact int32 accumulation (q8gemm MulPanelsI8 /
// MulStripsI8 semantics, q8gemm/int8.go:170-253):
//   dst[m*stride + n] = (float32(sum_k qa[m,k]*qw[n,k]) * colScale[n]) * rowScale[m]
// and the per-row activation quantizer of WorkspaceI8 (int8.go:100-168).
//
// Device layout ("tile layout"): an R x K int8 matrix is stored as
// [ceil(R/16)][ceil(K/64)][64 lanes][16 bytes]; lane l of group (rt, kt) holds
// row rt*16 + l%16, columns kt*64 + (l/16)*16 .. +16. One 1 KiB group is one
// operand fragment of v_mfma_i32_16x16x64_i8 for both A (rows = activation
// rows) and B (rows = weight rows / output columns), so every fragment load is
// a single contiguous 1 KiB wavefront load. Padding (rows past R, K past the
// logical K) is zero in the weights, so padded K never changes a sum.
//
// GEMM kernels, all exact in int32 and with one epilogue (int32 -> fp32 rounded
// to nearest even, like Go's float32(int32), then the two scale multiplies in the
// reference's order), so any of them gives the same bits:
//   * i8gemm_kernel (up to 16 rows): fragments straight from HBM / L2 into
//     registers, K split over a block's wavefronts, whose int32 partial tiles are
//     added in LDS;
//   * i8gemm_roles_kernel: tiles of 16 x 16 to 128 x 192, loading and multiplying
//     wavefronts apart, operands direct to a ring of LDS stages; tile layout or
//     the batched pass's row tiles and row-major weights;
//   * i8gemm_pp_kernel (tile layout) and i8gemm_rows_kernel (batched pass): 256-row
//     tiles, two groups of wavefronts half a K-step apart.
// i8gemm_launch and lm_i8_mm choose by rounds of the chip. Blocks are renumbered
// (tile_order, and by hand in i8gemm_kernel) so that consecutive blocks of one XCD
// share weight columns, which that XCD's L2 then reads once.
#include "common.h"

namespace gphq {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline size_t tile_offset(long r, long k, long kt) {
    return ((size_t)(r >> 4) * kt + (k >> 6)) * 1024 + (size_t)((((k & 63) >> 4) << 4) + (r & 15)) * 16 + (k & 15);
}

// The batched pass's int8 activations ("row tiles"): the same 1 KiB groups of
// 16 rows x 64 bytes, each row's 64 bytes contiguous inside the group, so a
// row-at-a-time packer writes 64-byte pieces. The direct-to-LDS GEMM gathers
// a group into the tile layout's lane order within its own 1 KiB.
__host__ __device__ inline size_t rowtile_offset(long r, long k, long kt) {
    return ((size_t)(r >> 4) * kt + (k >> 6)) * 1024 + (size_t)(r & 15) * 64 + (k & 63);
}

// ---- weight packing: row-major int8 [rows][K] -> tile layout ---------------
// One thread per 16-byte lane chunk of the destination; rows past `rows`
// (inside the last 16-row tile) and K padding are written as zero.
__global__ void i8_pack_tiles_kernel(const int8_t *__restrict__ src, int8_t *__restrict__ dst, int rows, int K,
                                     int row0, int rowTiles, int kt) {
    const size_t chunk = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // 16-byte chunk index
    const size_t total = (size_t)rowTiles * kt * 64;
    if (chunk >= total) return;
    const int lane = (int)(chunk & 63);
    const size_t g = chunk >> 6;
    const int ktile = (int)(g % kt);
    const int rtile = (int)(g / kt) + (row0 >> 4);
    const int r = rtile * 16 + (lane & 15);  // absolute row
    const int kbase = ktile * 64 + (lane >> 4) * 16;
    int8_t v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int k = kbase + i;
        const int rr = r - row0;
        v[i] = (rr >= 0 && rr < rows && k < K) ? src[(size_t)rr * K + k] : (int8_t)0;
    }
    int8_t *d = dst + ((size_t)rtile * kt + ktile) * 1024 + (size_t)lane * 16;
    // Rows outside [row0, row0+rows) of a shared tile keep their bytes.
    const int rr = r - row0;
    if (rr >= 0 && rr < rows) {
#pragma unroll
        for (int i = 0; i < 16; ++i) d[i] = v[i];
    }
}

// ---- activation quantizer ---------------------------------------------------
// Workspace Pack fused: per row (one block each), MaxAbs with NaN propagation
// (gemm.go:138-150), SetRowScale, then quantize every column into the tile
// layout (and zero the row's K padding).
__global__ __launch_bounds__(256) void i8_pack_rows_kernel(const float *__restrict__ x, long stride, int K, int kt,
                                                           int8_t *__restrict__ act, float *__restrict__ rowScale,
                                                           float *__restrict__ rowInv) {
    __shared__ float smax[4];
    __shared__ int snan[4];
    const int row = blockIdx.x;
    const float *xr = x + (size_t)row * stride;
    float m = 0.0f;
    int nan = 0;
    // Eight independent loads per thread per trip, so a row's reads are in
    // flight together instead of one L2 round trip after another.
    constexpr int UNR = 8;
    for (int k0 = 0; k0 < K; k0 += 256 * UNR) {
        float v[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int k = k0 + u * 256 + (int)threadIdx.x;
            v[u] = k < K ? xr[k] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            nan |= (v[u] != v[u]);
            m = fmaxf(m, fabsf(v[u]));
        }
    }
    // wave max / nan-any
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off));
        nan |= __shfl_xor(nan, off);
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smax[wv] = m;
        snan[wv] = nan;
    }
    __syncthreads();
    float mm = 0.0f;
    int anyNan = 0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) {
        mm = fmaxf(mm, smax[i]);
        anyNan |= snan[i];
    }
    if (anyNan) mm = __builtin_nanf("");
    float scale, inv;
    i8_row_scale(mm, scale, inv);
    if (threadIdx.x == 0) {
        rowScale[row] = scale;
        rowInv[row] = inv;
    }
    // Quantize: each thread takes 16 consecutive columns (one 16-byte lane
    // chunk of the tile layout) and stores them with one 128-bit write.
    for (int c = threadIdx.x; c < kt * 4; c += blockDim.x) {
        const int kb = c * 16;
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t packed = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = kb + 4 * j + i;
                const int8_t q = k < K ? quantize_i8(__fmul_rn(xr[k], inv)) : (int8_t)0;
                packed |= (uint32_t)(uint8_t)q << (8 * i);
            }
            w[j] = packed;
        }
        *(uint4 *)(act + tile_offset(row, kb, kt)) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// The same Pack for K a multiple of 16 and 16-byte aligned rows: the row is
// read once, as 16-byte pieces, into registers (CPT chunks of 16 values per
// thread, thread t holding columns 16 (t + 256 c) .. + 15, the chunks past K
// zero), reduced for MaxAbs, and quantized from the registers. Rows with a
// finite positive 127/max quantize without quantize_i8's NaN test (rint,
// v_med3 clamp, v_perm byte packing); the others take quantize_i8 itself: the
// same bytes either way. The 8 rows whose 16-byte pieces share a 128-byte line
// of the tile layout (rows 8q .. 8q + 7) go to blocks b, b + 8, .., b + 56,
// which the dispatcher places on one XCD (round robin over 8), so each line is
// completed in one L2.
template <int CPT>
__global__ __launch_bounds__(256) void i8_pack_rows_vec_kernel(const float *__restrict__ x, long stride, int K,
                                                               int kt, int8_t *__restrict__ act,
                                                               float *__restrict__ rowScale,
                                                               float *__restrict__ rowInv, int rows) {
    __shared__ float smx[4];
    __shared__ int snan[4];
    const int bx = blockIdx.x, row = (bx & ~63) + 8 * (bx & 7) + ((bx >> 3) & 7);
    if (row >= rows) return;
    float4 v[CPT][4];
    load_row_chunks<CPT>(v, x + (size_t)row * stride, K);
    zero_past_end<CPT>(v, K);
    float mx = 0.0f;
    int nan = 0;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            mx = fmaxf(fmaxf(fmaxf(mx, fabsf(v[c][q].x)), fmaxf(fabsf(v[c][q].y), fabsf(v[c][q].z))), fabsf(v[c][q].w));
            nan |= (v[c][q].x != v[c][q].x) | (v[c][q].y != v[c][q].y) | (v[c][q].z != v[c][q].z) |
                   (v[c][q].w != v[c][q].w);
        }
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
        nan |= __shfl_xor(nan, off);
    }
    if ((threadIdx.x & 63) == 0) {
        smx[threadIdx.x >> 6] = mx;
        snan[threadIdx.x >> 6] = nan;
    }
    __syncthreads();
    float m = fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3]));
    if (snan[0] | snan[1] | snan[2] | snan[3]) m = __builtin_nanf("");
    float scale, inv;
    i8_row_scale(m, scale, inv);
    if (threadIdx.x == 0) {
        rowScale[row] = scale;
        rowInv[row] = inv;
    }
    const bool plain = inv > 0.0f && inv < INFINITY;  // the same for the whole block
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        const int kb = 16 * ((int)threadIdx.x + 256 * c);
        if (kb >= kt * 64) continue;
        uint32_t w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float e[4] = {v[c][q].x, v[c][q].y, v[c][q].z, v[c][q].w};
            if (plain) {
                int b[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    b[i] = (int)__builtin_amdgcn_fmed3f(rintf(__fmul_rn(e[i], inv)), -128.0f, 127.0f);
                w[q] = __builtin_amdgcn_perm((uint32_t)b[1], (uint32_t)b[0], 0x0c0c0400u) |
                       __builtin_amdgcn_perm((uint32_t)b[3], (uint32_t)b[2], 0x04000c0cu);
            } else {
                uint32_t packed = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) packed |= (uint32_t)(uint8_t)quantize_i8(__fmul_rn(e[i], inv)) << (8 * i);
                w[q] = packed;
            }
        }
        *(uint4 *)(act + tile_offset(row, kb, kt)) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// PackRange (int8.go:116-163) with row scales already set: quantize columns
// [k0, k1) of every prepared row; k1 == K also zeroes the K padding.
__global__ __launch_bounds__(256) void i8_pack_range_kernel(const float *__restrict__ x, long stride, int K, int kt,
                                                            int k0, int k1, int8_t *__restrict__ act,
                                                            const float *__restrict__ rowInv) {
    const int row = blockIdx.x;
    const float inv = rowInv[row];
    const float *xr = x + (size_t)row * stride;
    const int kend = (k1 == K) ? kt * 64 : k1;
    for (int k = k0 + threadIdx.x; k < kend; k += blockDim.x) {
        const int8_t q = k < K ? quantize_i8(__fmul_rn(xr[k], inv)) : (int8_t)0;
        act[tile_offset(row, k, kt)] = q;
    }
}

// The qwen3lm batched pass's int8 activations, the CPU provider's int8 route
// (qwen3lm/ops.go:96-147: the row is normalized, SetRowScale(MaxAbs), then
// PackRange) over the GPU layer formats: per row v = x * f with f the RMSNorm
// factor (MODE 2, the FP16 packer's sum order) or 1 (MODE 1); SetRowScale of
// max|v| (NaN-propagating); q = quantize(v * inv) written as row tiles
// (rowtile_offset, K a multiple of 64); rowScale[r] = max / 127. One block per row, the row in
// registers (CPT chunks of 16 values per thread). ROT first rotates the row
// as the down projection's input (the online Hadamard, gpu.metal:339-367;
// the CPU path's scaleRow, qwen3lm/ops.go:111-122): x * signs (signs carry
// the 1/sqrt(block) scale), then the butterfly network of each block in LDS
// (K floats of dynamic LDS), the same arithmetic as the decode step's
// rotation kernel.
template <int MODE, int CPT, bool ROT>
__global__ __launch_bounds__(256) void i8_act_rows_kernel(const float *__restrict__ x, long stride, int K, float eps,
                                                          const float *__restrict__ signs, int block,
                                                          int8_t *__restrict__ act, float *__restrict__ rowScale,
                                                          int rows) {
    __shared__ float sss[4], smx[4];
    __shared__ int snan[4];
    // The 2 rows whose 64-byte pieces share a 128-byte line of the row tiles
    // go to blocks b and b + 8, which the dispatcher places on one XCD (round
    // robin over 8), so each line is completed in one L2.
    const int bx = blockIdx.x, row = (bx & ~15) + 2 * (bx & 7) + ((bx >> 3) & 1);
    if (row >= rows) return;
    const float *xr = x + (size_t)row * stride;
    float4 v[CPT][4];
    float ss = 0.0f, mx = 0.0f;
    int nan = 0;
    float4 sg[4];
    if constexpr (ROT) {
        rot_signs(sg, signs, 16 * (int)threadIdx.x, K);
        __builtin_amdgcn_sched_barrier(0);  // the signs are requested first
    }
    load_row_chunks<CPT>(v, xr, K);
    if constexpr (ROT) rotate_row_lds<CPT>(v, sg, K, signs, block);
    zero_past_end<CPT>(v, K);
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (MODE == 2)
                ss += v[c][q].x * v[c][q].x + v[c][q].y * v[c][q].y + v[c][q].z * v[c][q].z + v[c][q].w * v[c][q].w;
            mx = fmaxf(fmaxf(fmaxf(mx, fabsf(v[c][q].x)), fmaxf(fabsf(v[c][q].y), fabsf(v[c][q].z))), fabsf(v[c][q].w));
            nan |= (v[c][q].x != v[c][q].x) | (v[c][q].y != v[c][q].y) | (v[c][q].z != v[c][q].z) |
                   (v[c][q].w != v[c][q].w);
        }
    }
    if constexpr (MODE == 2) ss = wave_sum(ss);
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
        nan |= __shfl_xor(nan, off);
    }
    if ((threadIdx.x & 63) == 0) {
        sss[threadIdx.x >> 6] = ss;
        smx[threadIdx.x >> 6] = mx;
        snan[threadIdx.x >> 6] = nan;
    }
    __syncthreads();
    const float f = MODE == 2 ? 1.0f / sqrtf(((sss[0] + sss[1]) + (sss[2] + sss[3])) / (float)K + eps) : 1.0f;
    // max |x * f| is (max |x|) * f: rounding is monotonic.
    float m = __fmul_rn(fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3])), f);
    if (snan[0] | snan[1] | snan[2] | snan[3]) m = __builtin_nanf("");
    float scale, inv;
    i8_row_scale(m, scale, inv);
    if (threadIdx.x == 0) rowScale[row] = scale;
    // A row with a finite, nonzero 127/max has only finite products, so
    // quantize_i8's NaN test can go: rint, clamp (v_med3) and convert, the
    // four bytes packed by v_perm. Other rows (NaN, infinite, zero or
    // denormal-range maxima) take quantize_i8 itself. The same bytes either way.
    const bool plain = inv > 0.0f && inv < INFINITY;  // the same for the whole block
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        const int k = 16 * ((int)threadIdx.x + 256 * c);
        if (k >= K) continue;
        uint32_t w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float e[4] = {v[c][q].x, v[c][q].y, v[c][q].z, v[c][q].w};
            if (plain) {
                int b[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float y = MODE == 2 ? __fmul_rn(e[i], f) : e[i];
                    b[i] = (int)__builtin_amdgcn_fmed3f(rintf(__fmul_rn(y, inv)), -128.0f, 127.0f);
                }
                w[q] = __builtin_amdgcn_perm((uint32_t)b[1], (uint32_t)b[0], 0x0c0c0400u) |
                       __builtin_amdgcn_perm((uint32_t)b[3], (uint32_t)b[2], 0x04000c0cu);
            } else {
                uint32_t packed = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float y = MODE == 2 ? __fmul_rn(e[i], f) : e[i];
                    packed |= (uint32_t)(uint8_t)quantize_i8(__fmul_rn(y, inv)) << (8 * i);
                }
                w[q] = packed;
            }
        }
        *(uint4 *)(act + rowtile_offset(row, k, K >> 6)) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// ---- GEMM ------------------------------------------------------------------
struct I8GemmArgs {
    const int8_t *A;      // activations, tile layout, MT x KT groups (row tiles for the batched pass)
    const int8_t *B;      // weights, tile layout, NT x KT groups (row-major [N][K] for the batched pass)
    const float *rowScale;  // [M]
    const float *colScale;  // [N]
    float *dst;
    long stride;
    int M, N, KT, NT;
    int c0, c1;  // output columns [c0, c1)
    int tileN0;  // first 16-column tile covered by the grid
    int gridM, gridN;  // blocks along M and N
    int K;             // row length in bytes of row-major weights (a multiple of 64)
};

// Epilogues: store, fp32 add into dst, SwiGLU of interleaved columns.
enum { I8_EPI_STORE = 0, I8_EPI_ADD = 1, I8_EPI_SWIGLU = 2 };

// A block is WM x WN x SK wavefronts; wavefront (wm, wn, ks) owns a (16 TM) x (16
// TN) output tile and the ks-th slice of the K tiles. It loads U K-steps of A and
// B fragments into registers, then issues TM TN MFMAs per step.
template <int TM, int TN, int WM, int WN, int SK, int U>
__global__ __launch_bounds__(64 * WM * WN * SK) void i8gemm_kernel(const I8GemmArgs a) {
    constexpr int NW = WM * WN * SK;
    __shared__ i32x4 red[(SK > 1) ? (NW * TM * TN * 64) : 1];
    // XCD-aware renumbering: hardware places block b on XCD b % 8. Give the
    // blocks of one XCD consecutive logical ids, M fastest, so they share
    // weight column tiles.
    const int G = a.gridM * a.gridN;
    const int b = blockIdx.x;
    int logical = b;
    if (G % 8 == 0) logical = (b % 8) * (G / 8) + b / 8;
    const int bm = logical % a.gridM, bn = logical / a.gridM;

    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int ks = wv % SK;
    const int wn = (wv / SK) % WN;
    const int wm = wv / (SK * WN);
    const int mt0 = (bm * WM + wm) * TM;                      // first 16-row tile
    const int nt0 = a.tileN0 + (bn * WN + wn) * TN;           // first 16-col tile
    const int MT = (a.M + 15) >> 4;
    const int KT = a.KT;
    const int per = (KT + SK - 1) / SK;
    const int kt0 = ks * per, kt1 = min(KT, kt0 + per);

    size_t aoff[TM], boff[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) aoff[i] = (size_t)min(mt0 + i, MT - 1) * KT * 1024 + (size_t)lane * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) boff[j] = (size_t)min(nt0 + j, a.NT - 1) * KT * 1024 + (size_t)lane * 16;

    i32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = i32x4{0, 0, 0, 0};

    // Two register buffers: the fragments of batch b+1 are requested before the
    // MFMAs of batch b, so memory latency overlaps the matrix work. Fragments
    // past the slice end are zero and add nothing.
    auto load = [&](i32x4 (&fa)[U][TM], i32x4 (&fb)[U][TN], int kt) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool ok = kt + u < kt1;
            const size_t ko = (size_t)(kt + u) * 1024;
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[u][i] = ok ? *(const i32x4 *)(a.A + aoff[i] + ko) : i32x4{0, 0, 0, 0};
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[u][j] = ok ? __builtin_nontemporal_load((const i32x4 *)(a.B + boff[j] + ko)) : i32x4{0, 0, 0, 0};
        }
    };
    auto mma = [&](const i32x4 (&fa)[U][TM], const i32x4 (&fb)[U][TN]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[u][i], fb[u][j], acc[i][j], 0, 0, 0);
    };
    i32x4 fa0[U][TM], fb0[U][TN], fa1[U][TM], fb1[U][TN];
    int kt = kt0;
    if (kt < kt1) load(fa0, fb0, kt);
    while (kt < kt1) {
        if (kt + U < kt1) load(fa1, fb1, kt + U);
        mma(fa0, fb0);
        kt += U;
        if (kt >= kt1) break;
        if (kt + U < kt1) load(fa0, fb0, kt + U);
        mma(fa1, fb1);
        kt += U;
    }

    if constexpr (SK > 1) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) red[((wv * TM + i) * TN + j) * 64 + lane] = acc[i][j];
        __syncthreads();
        if (ks != 0) return;
#pragma unroll
        for (int s = 1; s < SK; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += red[(((wv + s) * TM + i) * TN + j) * 64 + lane];
    }

    // Epilogue. Lane l of a 16x16 output tile holds rows 4*(l/16)+e, column
    // l%16. The scales are read first, unconditionally (clamped indices;
    // outputs outside the matrix are not written): scales read between
    // stores would each wait for the stores too.
    float rsc[TM][4], csc[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) rsc[i][e] = a.rowScale[min((mt0 + i) * 16 + 4 * (lane >> 4) + e, a.M - 1)];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = (nt0 + j) * 16 + (lane & 15);
        csc[j] = a.colScale[col >= a.c0 && col < a.c1 ? col : a.c0];
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = (nt0 + j) * 16 + (lane & 15);
        if (col < a.c0 || col >= a.c1) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (mt0 + i) * 16 + 4 * (lane >> 4) + e;
                if (row < a.M)
                    a.dst[(size_t)row * a.stride + col] = __fmul_rn(__fmul_rn((float)acc[i][j][e], csc[j]), rsc[i][e]);
            }
        }
    }
}

// The stores of dma_epilogue with the column-tile pairs starting at tile P
// of the wavefront (P = nt0 % 2, so that each pair's 32 columns are one
// 128-byte line of every row): v_permlane16_swap exchanges lanes 16-31 of
// tile j's values with lanes 0-15 of tile j + 1's (and 48-63 with 32-47), so
// each store covers 32 consecutive columns of two rows (two whole 128-byte
// lines) instead of 16 columns of four rows. After the swap, lane l holds
// column (j + bit 4 of l) * 16 + l % 16; the first value is row 8 (l / 32) + e,
// the second row 4 more. The tiles left out of the pairs (the first when P is
// 1, an odd last one) are stored as they are, and their half lines meet the
// neighbouring wavefront's in L2.
template <int TI, int TJ, int EPI, int P>
__device__ __forceinline__ void dma_epilogue_stores(const I8GemmArgs &a, const i32x4 (&acc)[TI][TJ], int mt0,
                                                    int nt0, int lane, const float (&rsc)[TI][4],
                                                    const float (&csc)[TJ]) {
    constexpr int PE = EPI == I8_EPI_SWIGLU ? 0 : P + ((TJ - P) & ~1);  // pairs cover tiles [P, PE)
    if constexpr (PE > P) {
#pragma unroll
        for (int j = P; j < PE; j += 2) {
            const int col = (nt0 + j + ((lane >> 4) & 1)) * 16 + (lane & 15);
            const bool colOk = col >= a.c0 && col < a.c1;
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v0 = __fmul_rn(__fmul_rn((float)acc[i][j][e], csc[j]), rsc[i][e]);
                    const float v1 = __fmul_rn(__fmul_rn((float)acc[i][j + 1][e], csc[j + 1]), rsc[i][e]);
                    const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v0),
                                                                     __builtin_bit_cast(uint32_t, v1), false, false);
                    const int row = (mt0 + i) * 16 + 8 * (lane >> 5) + e;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int r = row + 4 * h;
                        const float v = __builtin_bit_cast(float, h ? sw[1] : sw[0]);
                        if (!colOk || r >= a.M) continue;
                        if constexpr (EPI == I8_EPI_STORE)
                            a.dst[(size_t)r * a.stride + col] = v;
                        else
                            __builtin_amdgcn_global_atomic_fadd_f32(a.dst + (size_t)r * a.stride + col, v);
                    }
                }
        }
    }
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        if (PE > P && j >= P && j < PE) continue;  // stored as a pair
        const int col = (nt0 + j) * 16 + (lane & 15);
        const bool colOk = col >= a.c0 && col < a.c1;
        if constexpr (EPI != I8_EPI_SWIGLU) {
            if (!colOk) continue;
        }
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (mt0 + i) * 16 + 4 * (lane >> 4) + e;
                const float v = __fmul_rn(__fmul_rn((float)acc[i][j][e], csc[j]), rsc[i][e]);
                if constexpr (EPI == I8_EPI_STORE) {
                    if (row < a.M) a.dst[(size_t)row * a.stride + col] = v;
                } else if constexpr (EPI == I8_EPI_ADD) {
                    if (row < a.M) __builtin_amdgcn_global_atomic_fadd_f32(a.dst + (size_t)row * a.stride + col, v);
                } else {
                    // Every lane runs the exchange (DPP quad_perm [1,0,3,2]: lane l ^ 1 holds column col ^ 1).
                    const float u = __builtin_bit_cast(
                        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
                    if (colOk && !(col & 1) && row < a.M)
                        a.dst[(size_t)row * a.stride + (col >> 1)] = v / (1.0f + expf(-v)) * u;
                }
            }
    }
}

// Epilogue of the direct-to-LDS kernels, as in i8gemm_kernel: lane l of a
// 16 x 16 tile holds rows 4 (l / 16) + e, column l % 16; scales first, then
// the stores. mt0 / nt0: the wavefront's first row and column tile.
// Measured on MI355X (config 2, M = 512): stores of 16 columns per row wrote
// 1.32x the output's bytes to HBM (WRITE_SIZE); column-tile pairs from the
// wavefront's first tile 1.19x (wavefronts of 48 columns starting at an odd
// tile paired across lines); pairs that start on a line once.
template <int TI, int TJ, int EPI>
__device__ __forceinline__ void dma_epilogue(const I8GemmArgs &a, const i32x4 (&acc)[TI][TJ], int mt0, int nt0,
                                             int lane) {
    float rsc[TI][4], csc[TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) rsc[i][e] = a.rowScale[min((mt0 + i) * 16 + 4 * (lane >> 4) + e, a.M - 1)];
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const int col = (nt0 + j) * 16 + (lane & 15);
        csc[j] = a.colScale[col >= a.c0 && col < a.c1 ? col : a.c0];
    }
    if (EPI != I8_EPI_SWIGLU && TJ > 2 && (nt0 & 1))
        dma_epilogue_stores<TI, TJ, EPI, 1>(a, acc, mt0, nt0, lane, rsc, csc);
    else
        dma_epilogue_stores<TI, TJ, EPI, 0>(a, acc, mt0, nt0, lane, rsc, csc);
}

// The direct-to-LDS kernels below: BM x BN block tiles, WGM x WGN wavefronts
// each with a grid of 16 x 16 v_mfma_i32_16x16x64_i8 tiles, a ring of NS LDS
// stages. Every operand fragment (the tile layout's 1 KiB group of 16 rows x
// 64 bytes) loads with one global_load_lds_dwordx4 and is read back by the
// lanes that own it (lane l at byte 16 l: no bank conflicts). BROWS (the
// batched pass) takes A as row tiles (rowtile_offset) and B from row-major
// rows (a.K bytes each, K a multiple of 64): each fragment is gathered into
// the same LDS image, lane l reading row l % 16 at byte 16 (l / 16) of the
// step (for A inside one 1 KiB group). Loads return in issue order, so a wait
// is a count of the loads issued after the stage it waits for; the barrier is
// s_barrier with compiler-only fences around it (ring_barrier; a
// __syncthreads fence would wait for every load in flight). When the
// fragments of a stage do not split evenly over the wavefronts that load
// them, the first ones issue one more. Epilogue (float32(sum) * colScale) *
// rowScale, then a store, an fp32 atomic add into dst (I8_EPI_ADD: one owner
// per element, so exactly dst + v) or the SwiGLU of interleaved gate/up
// columns into dst[row][col / 2] (I8_EPI_SWIGLU, the neighbouring column's
// value by DPP).

// vmcnt(PER * min(after, MAXA)) and lgkmcnt(0).
template <int PER, int MAXA>
__device__ __forceinline__ void wait_stages_n(int after) {
    if constexpr (MAXA <= 0) {
        wait_vm_lgkm0<0>();
    } else {
        if (after >= MAXA)
            wait_vm_lgkm0<PER * MAXA>();
        else
            wait_stages_n<PER, MAXA - 1>(after);
    }
}

// Ping-pong schedule, one 64-deep K-step per stage (8 wavefronts, two per
// SIMD: a probe of the hardware wave id on MI355X places wavefronts w and w + 4
// of a 512-thread block on one SIMD). The wavefronts of group 0 (0-3) and
// group 1 (4-7) run half a K step apart: while one group issues its MFMAs for a
// step (at raised wave priority), the other requests the ring stage NS - 1
// ahead, reads its fragments of the step from LDS and waits for its share of
// the next stage; a barrier ends each half. Group 1 starts one barrier late and
// group 0 ends with one extra, so every wavefront passes the same number of
// barriers (2 KT + 2). Ordering: a wavefront's share of stage s + 1 is
// complete, and its reads of stage s returned, before the barrier that ends
// its memory half of step s; so both groups' shares of a stage are in LDS
// before the barrier after which group 0 reads it, and the slot that stage
// s + NS - 1 overwrites (stage s - 1's) was last read before the barrier
// preceding the memory half that requests it. 256 x 256 tiles of the tile
// layout, NS = 5, K = 4096, N = 12288, M = 4096: 160 us (2.58 POPS; 387 us with
// both operands staged through registers).
template <int BM, int BN, int WGM, int WGN, int NS>
__global__ __launch_bounds__(64 * WGM * WGN) void i8gemm_pp_kernel(const I8GemmArgs a) {
    constexpr int NW = WGM * WGN;
    static_assert(NW == 8, "two groups of four wavefronts");
    constexpr int FA = BM / 16, FB = BN / 16, F = FA + FB;
    constexpr int DMAX = (F + NW - 1) / NW, DREM = F % NW;
    constexpr int TI = BM / 16 / WGM, TJ = BN / 16 / WGN;
    static_assert(TI * 16 * WGM == BM && TJ * 16 * WGN == BN, "wave grid");
    static_assert(NS >= 3 && DMAX * (NS - 2) < 64, "ring depth");
    __shared__ i32x4 ring[NS][F][64];
    int bm, bn;
    tile_order(blockIdx.x, a.gridM, a.gridN, bm, bn);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wv >> 2;
    const int wm = wv / WGN, wn = wv % WGN;
    const int rt0 = bm * FA, ct0 = a.tileN0 + bn * FB;
    const int MT = (a.M + 15) >> 4, KT = a.KT;
    const bool full = DREM == 0 || wv < DREM;
    const int8_t *src[DMAX];
    int dst[DMAX];
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {
        const int f = min(wv + NW * d, F - 1);
        dst[d] = f;
        if (f < FA) {
            src[d] = a.A + (size_t)min(rt0 + f, MT - 1) * KT * 1024 + (size_t)lane * 16;
        } else {
            src[d] = a.B + (size_t)min(ct0 + (f - FA), a.NT - 1) * KT * 1024 + (size_t)lane * 16;
        }
    }
    auto stage_load = [&](int s) {
        const int slot = s % NS;
#pragma unroll
        for (int d = 0; d < DMAX; ++d)
            if (d < DMAX - 1 || full)
                lds_dma16(src[d] + (size_t)s * 1024, &ring[slot][dst[d]][0]);
    };
    auto wait_stages = [&](int after) {
        if (full)
            wait_stages_n<DMAX, NS - 2>(after);
        else
            wait_stages_n<DMAX - 1, NS - 2>(after);
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        ring_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    i32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
        if (p < KT) stage_load(p);
    wait_stages(min(KT - 1, NS - 2));
    barrier();
    if (grp == 1) barrier();
    i32x4 fa[TI], fb[TJ];
    for (int s = 0; s < KT; ++s) {
        // Memory half: the stage NS - 1 ahead (its slot held stage s - 1, which
        // every wavefront finished reading before the barrier that ended its
        // previous memory half), this step's fragments, then a wait for this
        // wavefront's share of stage s + 1 and for the fragment reads.
        if (s + NS - 1 < KT) stage_load(s + NS - 1);
        const int slot = s % NS;
#pragma unroll
        for (int i = 0; i < TI; ++i) fa[i] = ring[slot][wm * TI + i][lane];
#pragma unroll
        for (int j = 0; j < TJ; ++j) fb[j] = ring[slot][FA + wn * TJ + j][lane];
        wait_stages(min(KT - 2 - s, NS - 2));
        barrier();
        // MFMA half.
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        barrier();
    }
    if (grp == 0) barrier();
    dma_epilogue<TI, TJ, I8_EPI_STORE>(a, acc, rt0 + wm * TI, ct0 + wn * TJ, lane);
}

// The ping-pong schedule for row-major weights (the batched pass): a 64-deep
// step takes half a 128-byte line of each weight row, and loads of half lines
// (16 rows x 64 bytes an instruction) held the schedule to 1.75 POPS (472 us, Qwen3-
// 8B gate/up at 4096 rows, SwiGLU; the tile layout's whole groups run 2.58 with a
// plain store). Whole lines: 445 us, 1.85 POPS; with the activation pack (26 us)
// 498 -> 463 us. MFMA busy 41%, VALU busy 43%. B comes in pieces
// of two K-steps: 8 rows x 128 bytes an instruction, lane l taking chunk (l % 8)
// ^ ((row / 2) % 8) of row l / 8, so that a fragment's 16 rows at one chunk sit on distinct
// banks. LDS holds four A stages and three B pieces; a step requests A's stage
// three ahead and, when even, B's piece two ahead (the slot of the piece
// before this one, whose last reads precede the barrier before the request, as
// in i8gemm_pp_kernel). At the end of a memory half the wavefront's loads older
// than A's stage s + 1 are complete, so may remain in flight: for an even step
// B's piece of step s - 2, A's of s - 1, and both of s; for an odd one A's and
// B's of s - 1 and A's of s. The last steps, whose requests run out, wait for
// all. A piece past K (an odd step count) reads its row's first half twice.
template <int BN, int EPI>
__global__ __launch_bounds__(512) void i8gemm_rows_kernel(const I8GemmArgs a) {
    constexpr int BM = 256, WGM = 4, WGN = 2;
    constexpr int TI = BM / 16 / WGM, TJ = BN / 16 / WGN;
    constexpr int LA = BM / 16 / 8, LB = BN / 8 / 8;  // loads per wavefront: A per step, B per piece
    constexpr int NA = 4, NB = 3;
    // One array: with two the compiler waits for every direct-to-LDS load into
    // either before it reads from one.
    __shared__ i32x4 lds[NA * BM * 4 + NB * BN * 8];
    i32x4 *const As = lds, *const Bs = lds + NA * BM * 4;  // [NA][BM / 16][64]; [NB][row][8 chunks, swizzled]
    int bm, bn;
    tile_order(blockIdx.x, a.gridM, a.gridN, bm, bn);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wv >> 2;
    const int wm = wv / WGN, wn = wv % WGN;
    const int rt0 = bm * (BM / 16), ct0 = a.tileN0 + bn * (BN / 16);
    const int MT = (a.M + 15) >> 4, KT = a.KT;
    const int pieces = (KT + 1) / 2;
    const int8_t *asrc[LA], *bsrc[LB];
    const int brow = lane >> 3;
    int bchunk[LB];
#pragma unroll
    for (int d = 0; d < LA; ++d)
        asrc[d] = a.A + (size_t)min(rt0 + wv + 8 * d, MT - 1) * KT * 1024 + (size_t)(lane & 15) * 64 + (lane >> 4) * 16;
#pragma unroll
    for (int d = 0; d < LB; ++d) {
        const int r = 8 * (wv + 8 * d) + brow;  // row of the block's tile
        bchunk[d] = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
        bsrc[d] = a.B + (size_t)min(ct0 * 16 + r, a.N - 1) * a.K;
    }
    auto aload = [&](int s) {
#pragma unroll
        for (int d = 0; d < LA; ++d) lds_dma16(asrc[d] + (size_t)s * 1024, &As[(s % NA) * (BM * 4) + 64 * (wv + 8 * d)]);
    };
    auto bload = [&](int p) {
        const bool half = 2 * p + 1 >= KT;
#pragma unroll
        for (int d = 0; d < LB; ++d)
            lds_dma16(bsrc[d] + (size_t)p * 128 + (half ? bchunk[d] & 63 : bchunk[d]), &Bs[(p % NB) * (BN * 8) + 64 * (wv + 8 * d)]);
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        ring_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    i32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = i32x4{0, 0, 0, 0};
    bload(0);
    aload(0);
    if (pieces > 1) bload(1);
    if (KT > 1) aload(1);
    if (KT > 2) aload(2);
    wait_vm_lgkm0<0>();
    barrier();
    if (grp == 1) barrier();
    const int fr = lane & 15, fg = lane >> 4;
    i32x4 fa[TI], fb[TJ];
    auto step = [&](int s, int odd) {
        // Memory half.
        if (s + 3 < KT) aload(s + 3);
        if (!odd && s / 2 + 2 < pieces) bload(s / 2 + 2);
#pragma unroll
        for (int i = 0; i < TI; ++i) fa[i] = As[(s % NA) * (BM * 4) + 64 * (wm * TI + i) + lane];
        const int slot = (s / 2) % NB;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int r = (wn * TJ + j) * 16 + fr;
            fb[j] = Bs[slot * (BN * 8) + r * 8 + ((4 * odd + fg) ^ ((r >> 1) & 7))];
        }
        if (s + 4 < KT) {
            if (odd) wait_vm_lgkm0<2 * LA + LB>();
            else wait_vm_lgkm0<2 * LA + 2 * LB>();
        } else {
            wait_vm_lgkm0<0>();
        }
        barrier();
        // MFMA half.
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        barrier();
    };
    for (int s = 0; s < KT; s += 2) {
        step(s, 0);
        if (s + 1 < KT) step(s + 1, 1);
    }
    if (grp == 0) barrier();
    dma_epilogue<TI, TJ, EPI>(a, acc, rt0 + wm * TI, ct0 + wn * TJ, lane);
}

template <int BN, int EPI>
static int launch_i8gemm_rows(I8GemmArgs a, hipStream_t stream) {
    const int tiles = (a.c1 + 15) / 16 - a.tileN0;
    a.gridN = (tiles * 16 + BN - 1) / BN;
    a.gridM = (a.M + 255) / 256;
    hipLaunchKernelGGL((i8gemm_rows_kernel<BN, EPI>), dim3((unsigned)(a.gridM * a.gridN)), dim3(512), 0, stream, a);
    return launch_status();
}

template <int BM, int BN, int WGM, int WGN, int NS>
static int launch_i8gemm_pp(I8GemmArgs a, hipStream_t stream) {
    const int tiles = (a.c1 + 15) / 16 - a.tileN0;
    a.gridN = (tiles * 16 + BN - 1) / BN;
    a.gridM = (a.M + BM - 1) / BM;
    hipLaunchKernelGGL((i8gemm_pp_kernel<BM, BN, WGM, WGN, NS>), dim3((unsigned)(a.gridM * a.gridN)),
                       dim3(64 * WGM * WGN), 0, stream, a);
    return launch_status();
}

// BM x BN block tiles with the roles split: NP wavefronts only issue
// direct-to-LDS loads (a ring of NS stages of SB 64-deep K-steps), WGM x WGN
// wavefronts only multiply. A CU takes 60 bytes a clock from L2 (measured: 125-
// 143 GB/s, by direct-to-LDS or register loads, from 64 KB in flight), but a
// wavefront that both issues a stage's loads (16 clocks each on the address
// path) and multiplies it does one after the other, and kernels built so moved
// 16 bytes a clock at any M and N (M = 100, K = 4096: 18 us for N = 600 and for
// N = 3396; 9.9 and 12.1 here). Here the
// issue, the fragment reads (one K-step ahead, in a second register set) and
// the MFMAs run beside each other. Every wavefront passes one barrier before
// the loop and one per stage. Ordering: at the barrier that ends stage s,
// stage s + 2 is complete (the loaders' wait) and every read of stage s has
// returned (lgkmcnt(0)); during stage s the multipliers read stage s and the
// first step of s + 1, and the loaders refill the slot of stage s - 1. K-steps
// past KT in the last stage load the last step again and are not multiplied.
template <int BM, int BN, int WGM, int WGN, int NP, int SB, int NS, bool BROWS, int EPI>
__global__ __launch_bounds__(64 * (WGM * WGN + NP)) void i8gemm_roles_kernel(const I8GemmArgs a) {
    constexpr int NC = WGM * WGN;
    constexpr int FA = BM / 16, FB = BN / 16, F = FA + FB;  // fragments per K-step
    constexpr int FS = F * SB;                              // per stage
    constexpr int DMAX = (FS + NP - 1) / NP, DREM = FS % NP;
    constexpr int TI = BM / 16 / WGM, TJ = BN / 16 / WGN;
    static_assert(TI * 16 * WGM == BM && TJ * 16 * WGN == BN, "wave grid");
    static_assert(NS >= 4 && DMAX * (NS - 3) < 64, "ring depth");
    __shared__ i32x4 ring[NS][FS][64];
    int bm, bn;
    tile_order(blockIdx.x, a.gridM, a.gridN, bm, bn);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rt0 = bm * FA, ct0 = a.tileN0 + bn * FB;
    const int MT = (a.M + 15) >> 4, KT = a.KT;
    const int S = (KT + SB - 1) / SB;
    if (wv >= NC) {
        const int pw = wv - NC;
        const bool full = DREM == 0 || pw < DREM;
        const int8_t *src[DMAX];
        int dst[DMAX];
#pragma unroll
        for (int d = 0; d < DMAX; ++d) {
            dst[d] = min(pw + NP * d, FS - 1);
            const int f = dst[d] % F;
            if (f < FA) {
                src[d] = a.A + (size_t)min(rt0 + f, MT - 1) * KT * 1024 +
                         (BROWS ? (size_t)(lane & 15) * 64 + (lane >> 4) * 16 : (size_t)lane * 16);
            } else if constexpr (BROWS) {
                src[d] = a.B + (size_t)min((ct0 + (f - FA)) * 16 + (lane & 15), a.N - 1) * a.K + (lane >> 4) * 16;
            } else {
                src[d] = a.B + (size_t)min(ct0 + (f - FA), a.NT - 1) * KT * 1024 + (size_t)lane * 16;
            }
        }
        int slot = 0;
        auto stage_load = [&](int s) {
#pragma unroll
            for (int d = 0; d < DMAX; ++d)
                if (d < DMAX - 1 || full) {
                    const int st = min(s * SB + dst[d] / F, KT - 1);
                    lds_dma16(src[d] + (size_t)st * (BROWS && dst[d] % F >= FA ? 64 : 1024), &ring[slot][dst[d]][0]);
                }
            slot = slot + 1 == NS ? 0 : slot + 1;
        };
        auto wait_stages = [&](int after) {
            if (full)
                wait_stages_n<DMAX, NS - 3>(after);
            else
                wait_stages_n<DMAX - 1, NS - 3>(after);
        };
        for (int p = 0; p < NS - 1; ++p)
            if (p < S) stage_load(p);
        wait_stages(min(S - 2, NS - 3));  // stages 0 and 1
        ring_barrier();
        for (int s = 0; s < S; ++s) {
            if (s + NS - 1 < S) stage_load(s + NS - 1);
            wait_stages(min(S - 3 - s, NS - 3));
            ring_barrier();
        }
        return;
    }
    const int wm = wv / WGN, wn = wv % WGN;
    i32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = i32x4{0, 0, 0, 0};
    i32x4 fa[2][TI], fb[2][TJ];
    int rslot = 0, rstep = 0;  // where the next K-step's fragments are
    auto frags = [&](int set) {
        const i32x4(*r)[64] = &ring[rslot][rstep * F];
#pragma unroll
        for (int i = 0; i < TI; ++i) fa[set][i] = r[wm * TI + i][lane];
#pragma unroll
        for (int j = 0; j < TJ; ++j) fb[set][j] = r[FA + wn * TJ + j][lane];
        if (++rstep == SB) {
            rstep = 0;
            rslot = rslot + 1 == NS ? 0 : rslot + 1;
        }
    };
    ring_barrier();
    frags(0);
    auto step = [&](int k, int set) {
        if (k + 1 < KT) frags(set ^ 1);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[set][i], fb[set][j], acc[i][j], 0, 0, 0);
        if ((k + 1) % SB == 0 || k + 1 == KT) {
            wait_vm_lgkm0<63>();
            ring_barrier();
        }
    };
    for (int k = 0; k < KT; k += 2) {
        step(k, 0);
        if (k + 1 < KT) step(k + 1, 1);
    }
    dma_epilogue<TI, TJ, EPI>(a, acc, rt0 + wm * TI, ct0 + wn * TJ, lane);
}

template <int BM, int BN, int WGM, int WGN, int NP, int SB, int NS, bool BROWS = false, int EPI = I8_EPI_STORE>
static int launch_i8gemm_roles(I8GemmArgs a, hipStream_t stream) {
    const int tiles = (a.c1 + 15) / 16 - a.tileN0;
    a.gridN = (tiles * 16 + BN - 1) / BN;
    a.gridM = (a.M + BM - 1) / BM;
    hipLaunchKernelGGL((i8gemm_roles_kernel<BM, BN, WGM, WGN, NP, SB, NS, BROWS, EPI>),
                       dim3((unsigned)(a.gridM * a.gridN)), dim3(64 * (WGM * WGN + NP)), 0, stream, a);
    return launch_status();
}

template <int TM, int TN, int WM, int WN, int SK, int U>
static int launch_i8gemm(I8GemmArgs a, hipStream_t stream) {
    const int tiles = (a.c1 + 15) / 16 - a.tileN0;
    a.gridN = (tiles + TN * WN - 1) / (TN * WN);
    a.gridM = (a.M + 16 * TM * WM - 1) / (16 * TM * WM);
    const unsigned blocks = (unsigned)(a.gridM * a.gridN);
    hipLaunchKernelGGL((i8gemm_kernel<TM, TN, WM, WN, SK, U>), dim3(blocks), dim3(64 * WM * WN * SK), 0, stream, a);
    return launch_status();
}

// Columns [c0, c1) of dst for M activation rows. Chooses a tile shape by M;
// every shape gives identical bits (exact int32 sums, same epilogue).
int i8gemm_launch(const int8_t *A, const int8_t *B, const float *rowScale, const float *colScale, float *dst,
                  long stride, int M, int N, int KT, int c0, int c1, hipStream_t stream) {
    if (M == 0 || c0 >= c1) return GPHQ_OK;
    I8GemmArgs a{};
    a.A = A;
    a.B = B;
    a.rowScale = rowScale;
    a.colScale = colScale;
    a.dst = dst;
    a.stride = stride;
    a.M = M;
    a.N = N;
    a.KT = KT;
    a.NT = (N + 15) / 16;
    a.c0 = c0;
    a.c1 = c1;
    a.tileN0 = c0 / 16;
    // Up to 16 rows the weights alone bound the product: 32 columns a block, K
    // split over its wavefronts (M = 8, N = 12288, K = 4096: 10.7 us; 16.8 in
    // 16 x 16 tiles below).
    if (M <= 16) return launch_i8gemm<1, 2, 1, 2, 4, 4>(a, stream);
    // Above, one tile per CU at a time, and a tile's time follows its K steps
    // whatever the rest of the chip does: the tile with the least rounds of
    // the chip x (steps x time per step + fill and stores) is the fastest.
    // Nanoseconds per 64-deep step measured on MI355X (KT 12 against 64).
    // K = 4096, N = 12288, M = 24 / 50 / 100 / 200 / 500 / 1000 / 4096: 13.5 /
    // 14.2 / 19.6 / 23.8 / 35.9 / 75.3 / 387 us before (tiles chosen by M
    // alone, each wavefront loading what it multiplies), 12.5 / 13.0 / 15.9 /
    // 20.0 / 30.8 / 47.7 / 160 with this; N = 3396: 12.2 / 12.9 / 18.1 / 21.8 /
    // 31.4 / 41.0 / 122 before, 9.3 / 9.4 / 12.1 / 12.8 / 16.2 / 22.1 / 55.6
    // (weights from the 256 MB cache). With weights that no cache holds, over 506
    // sizes (17-1500 rows, K = 64 to 8192, N = 594 to 12288) the tile taken is 0.9%
    // behind the fastest on average; 25 sizes lose more than 6%, most at 896 x
    // 7040 -> 10234 (107 us in 128 x 96, 68 in 256 x 256); 20 rows, 4096 ->
    // 12288, take 12.7 us (12.3 before).
    struct Tile {
        int bm, bn, ns;
    };
    static constexpr Tile tiles[] = {{64, 16, 87},   {64, 32, 92},   {32, 48, 95},   {64, 48, 108},
                                     {128, 32, 112}, {64, 64, 123},  {128, 48, 133}, {128, 64, 163},
                                     {128, 96, 177}, {128, 128, 190}, {128, 192, 325}, {256, 256, 560}};
    int best = 0;
    long cost = 0;
    for (int i = 0; i < (int)(sizeof(tiles) / sizeof(tiles[0])); ++i) {
        const long width = ((c1 + 15) / 16 - a.tileN0) * 16L;
        const long blocks = ((M + tiles[i].bm - 1) / tiles[i].bm) * ((width + tiles[i].bn - 1) / tiles[i].bn);
        const long rounds = (blocks + device_cus() - 1) / device_cus();
        const long c = rounds * ((long)KT * tiles[i].ns + 1500);
        if (i == 0 || c < cost) cost = c, best = i;
    }
    switch (best) {
    case 0: return launch_i8gemm_roles<64, 16, 4, 1, 4, 4, 7>(a, stream);
    case 1: return launch_i8gemm_roles<64, 32, 4, 1, 4, 2, 9>(a, stream);
    case 2: return launch_i8gemm_roles<32, 48, 2, 1, 4, 4, 6>(a, stream);
    case 3: return launch_i8gemm_roles<64, 48, 4, 1, 4, 2, 8>(a, stream);
    case 4: return launch_i8gemm_roles<128, 32, 4, 1, 4, 2, 7>(a, stream);
    case 5: return launch_i8gemm_roles<64, 64, 2, 2, 4, 2, 9>(a, stream);
    case 6: return launch_i8gemm_roles<128, 48, 4, 1, 4, 2, 7>(a, stream);
    case 7: return launch_i8gemm_roles<128, 64, 4, 2, 4, 2, 6>(a, stream);
    case 8: return launch_i8gemm_roles<128, 96, 4, 2, 4, 1, 10>(a, stream);
    case 9: return launch_i8gemm_roles<128, 128, 2, 4, 4, 1, 9>(a, stream);
    case 10: return launch_i8gemm_roles<128, 192, 2, 4, 4, 1, 8>(a, stream);
    }
    return launch_i8gemm_pp<256, 256, 4, 2, 5>(a, stream);
}

template <int MODE, bool ROT>
static int launch_i8_act_rows(const float *x, long stride, int rows, int K, float eps, const float *signs, int block,
                              int8_t *act, float *rowScale, hipStream_t stream) {
    const int chunks = K / 16;
    const size_t lds = ROT ? rot_lds_bytes(K) : 0;
#define GPHQ_I8ACT(CPT)                                                                                                \
    do {                                                                                                               \
        if (lds > 65536)                                                                                               \
            (void)hipFuncSetAttribute((const void *)i8_act_rows_kernel<MODE, CPT, ROT>,                                \
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                           \
        hipLaunchKernelGGL((i8_act_rows_kernel<MODE, CPT, ROT>), dim3((unsigned)((rows + 15) & ~15)), dim3(256), lds,  \
                           stream, x, stride, K, eps, signs, block, act, rowScale, rows);                              \
    } while (0)
    if (chunks <= 256)
        GPHQ_I8ACT(1);
    else if (chunks <= 512)
        GPHQ_I8ACT(2);
    else if (chunks <= 768)
        GPHQ_I8ACT(3);
    else
        GPHQ_I8ACT(4);
#undef GPHQ_I8ACT
    return launch_status();
}

// int8 activations of the batched pass (see i8_act_rows_kernel): x rows
// `stride` floats apart and 16-byte aligned, K % 64 == 0, K <= 16384; act is
// in row tiles (rowtile_offset: ceil(rows / 16) * 16 rows of K bytes; rows
// past `rows` in the last tile are not written). signs (device, K values with the
// rotation's scale folded in) rotate each row first, in blocks of `block`;
// null for none.
int lm_i8_act(const float *x, long stride, int rows, int K, bool norm, float eps, const float *signs, int block,
              int8_t *act, float *rowScale, hipStream_t stream) {
    if (rows == 0) return GPHQ_OK;
    if (signs) {
        if (norm) return GPHQ_ERR_UNSUPPORTED;  // no pass normalizes a rotated input
        return launch_i8_act_rows<1, true>(x, stride, rows, K, eps, signs, block, act, rowScale, stream);
    }
    if (norm) return launch_i8_act_rows<2, false>(x, stride, rows, K, eps, nullptr, 0, act, rowScale, stream);
    return launch_i8_act_rows<1, false>(x, stride, rows, K, eps, nullptr, 0, act, rowScale, stream);
}

// The batched pass's int8 GEMM over columns [a.c0, a.c1) in 256 x BN tiles.
template <int BN>
static int lm_i8_mm_rows(int epi, const I8GemmArgs &a, hipStream_t stream) {
    if (epi == 0) return launch_i8gemm_rows<BN, I8_EPI_STORE>(a, stream);
    if (epi == 1) return launch_i8gemm_rows<BN, I8_EPI_ADD>(a, stream);
    return launch_i8gemm_rows<BN, I8_EPI_SWIGLU>(a, stream);
}

template <int BM, int BN, int WGM, int WGN, int NP, int SB, int NS>
static int lm_i8_mm_roles(int epi, const I8GemmArgs &a, hipStream_t stream) {
    if (epi == 0) return launch_i8gemm_roles<BM, BN, WGM, WGN, NP, SB, NS, true, I8_EPI_STORE>(a, stream);
    if (epi == 1) return launch_i8gemm_roles<BM, BN, WGM, WGN, NP, SB, NS, true, I8_EPI_ADD>(a, stream);
    return launch_i8gemm_roles<BM, BN, WGM, WGN, NP, SB, NS, true, I8_EPI_SWIGLU>(a, stream);
}

// One projection of the batched pass on the int8 route: y = (float32(A W^T)
// * w_scale) * a_scale for int8 activations A in row tiles (lm_i8_act)
// and row-major Q8 codes W [N][K] (one fp32 scale per weight row), then epi 0
// stores y[M][N], 1 adds it into y, 2 stores the SwiGLU of interleaved gate/up
// columns into y[M][N/2]; y rows are y_stride floats apart. K % 64 == 0.
int lm_i8_mm(int epi, const int8_t *act, const float *a_scale, const int8_t *codes, const float *w_scale, float *y,
             long y_stride, int M, int K, int N, hipStream_t stream) {
    if (M == 0 || N == 0) return GPHQ_OK;
    I8GemmArgs a{};
    a.A = act;
    a.B = codes;
    a.rowScale = a_scale;
    a.colScale = w_scale;
    a.dst = y;
    a.stride = y_stride;
    a.M = M;
    a.N = N;
    a.K = K;
    a.KT = (K + 63) / 64;
    a.NT = (N + 15) / 16;
    a.c0 = 0;
    a.c1 = N;
    a.tileN0 = 0;
    // The tile with the least rounds of the chip x (K steps x time per step +
    // fill and stores), as in i8gemm_launch; nanoseconds per 64-deep step
    // measured on MI355X, K = 1024 to 12288. Columns past whole rounds of 256 x
    // 256 tiles may take 256 x 128 ones. With their activation packs, rows 4 /
    // 50 / 300 / 1500: Qwen3-8B down 128 / 130 / 136 / 163 us in 256-row tiles,
    // 30.8 / 37.9 / 65.9 / 129 with this; O 47 / 48 / 53 / 68, 12.0 / 15.0 /
    // 26.1 / 57.6; gate/up 52 / 60 / 72 / 199, 31 / 33 / 65 / 199.
    struct Tile {
        int bm, bn, ns, perCu;
    };
    static constexpr Tile tiles[] = {{16, 16, 118, 2},   {64, 32, 150, 1},   {64, 64, 207, 1},  {128, 64, 266, 1},
                                     {128, 128, 385, 1}, {256, 128, 470, 1}, {256, 256, 700, 1}};
    constexpr int kWide = 6, kSplit = 7;
    auto time = [&](const Tile &t, long width) {
        const long blocks = ((M + t.bm - 1L) / t.bm) * ((width + t.bn - 1) / t.bn), at_once = (long)device_cus() * t.perCu;
        return (blocks + at_once - 1) / at_once * ((long)a.KT * t.ns + 1500);
    };
    int best = 0;
    long cost = time(tiles[0], N);
    for (int i = 1; i <= kWide; ++i) {
        const long c = time(tiles[i], N);
        if (c < cost) cost = c, best = i;
    }
    const long full = whole_round_cols256((M + 255) / 256, (N + 255) / 256);
    if (full > 0 && time(tiles[kWide], full * 256) + time(tiles[kWide - 1], N - full * 256) < cost) best = kSplit;
    switch (best) {
    case 0: return lm_i8_mm_roles<16, 16, 1, 1, 2, 4, 8>(epi, a, stream);
    case 1: return lm_i8_mm_roles<64, 32, 4, 1, 4, 2, 9>(epi, a, stream);
    case 2: return lm_i8_mm_roles<64, 64, 2, 2, 4, 2, 9>(epi, a, stream);
    case 3: return lm_i8_mm_roles<128, 64, 4, 2, 4, 2, 6>(epi, a, stream);
    case 4: return lm_i8_mm_roles<128, 128, 2, 4, 4, 1, 9>(epi, a, stream);
    case 5: return lm_i8_mm_rows<128>(epi, a, stream);
    case kWide: return lm_i8_mm_rows<256>(epi, a, stream);
    }
    I8GemmArgs b = a;
    b.c1 = (int)(full * 256);
    GPHQ_TRY(lm_i8_mm_rows<256>(epi, b, stream));
    a.c0 = b.c1;
    a.tileN0 = a.c0 / 16;
    return lm_i8_mm_rows<128>(epi, a, stream);
}

int i8_pack_tiles(const int8_t *src, int8_t *dst, int rows, int K, int row0, int kt, hipStream_t stream) {
    if (rows == 0) return GPHQ_OK;
    const int rowTiles = ((row0 + rows + 15) >> 4) - (row0 >> 4);
    const size_t chunks = (size_t)rowTiles * kt * 64;
    hipLaunchKernelGGL(i8_pack_tiles_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, stream, src, dst,
                       rows, K, row0, rowTiles, kt);
    return launch_status();
}

int i8_pack_rows(const float *x, long stride, int rows, int K, int kt, int8_t *act, float *rowScale, float *rowInv,
                 hipStream_t stream) {
    if (rows == 0) return GPHQ_OK;
    // Rows whose values can be read as 16-byte pieces are held in registers
    // (one read of the row); other shapes take the two-pass kernel.
    if (K % 16 == 0 && stride % 4 == 0 && (uintptr_t)x % 16 == 0 && kt <= 256) {
        switch ((kt + 63) / 64) {
#define GPHQ_PACK_VEC(C)                                                                                              \
    case C:                                                                                                           \
        hipLaunchKernelGGL(i8_pack_rows_vec_kernel<C>, dim3((unsigned)((rows + 63) & ~63)), dim3(256), 0, stream, x,  \
                           stride, K, kt, act, rowScale, rowInv, rows);                                               \
        return launch_status();
            GPHQ_PACK_VEC(1)
            GPHQ_PACK_VEC(2)
            GPHQ_PACK_VEC(3)
            GPHQ_PACK_VEC(4)
#undef GPHQ_PACK_VEC
        }
    }
    hipLaunchKernelGGL(i8_pack_rows_kernel, dim3(rows), dim3(256), 0, stream, x, stride, K, kt, act, rowScale, rowInv);
    return launch_status();
}

int i8_pack_range(const float *x, long stride, int rows, int K, int kt, int k0, int k1, int8_t *act,
                  const float *rowInv, hipStream_t stream) {
    if (rows == 0 || (k0 == k1 && k1 != K)) return GPHQ_OK;
    hipLaunchKernelGGL(i8_pack_range_kernel, dim3(rows), dim3(256), 0, stream, x, stride, K, kt, k0, k1, act, rowInv);
    return launch_status();
}

}  // namespace gphq
