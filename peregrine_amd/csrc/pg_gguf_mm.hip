// Skinny / grouped product over GGUF block-quantised weights on the int8 matrix cores:
//   y[pair, n] = sum_b  d[n, b] * xs[tok, b] * sum_{k in block b} q[n, k] * X[tok, k]
// for up to 32 activation rows ("tokens") per workgroup, so the weights are read from HBM
// once per group of tokens instead of once per token (M > 1 dequant-matmul of models::llama,
// src/models/llama/model.rs:243-257 + src/tensor.rs:1342-1353, and the per-expert products
// of the MoE FFN, examples/grok1/moe.rs:91-104).
//
// A GGUF block is 32 consecutive k, exactly the K of one v_mfma_i32_32x32x32_i8: per block
// and 32x32 (weight rows x tokens) tile, two MFMAs give the exact integer dots of the
// weights with the high and the low byte digit of the fixed-point activations
// X = 256 * hi + lo (|X| <= 32639, per-block scale xs = absmax / 32639), and the tile is scaled by
// d[n, b] * xs[tok, b] and accumulated in f32.  Weight rows sit on the accumulator
// registers, tokens on lanes.
//
// Workgroup = 4 wavefronts = 128 weight rows x 32 tokens x one K chunk.  Everything is
// staged through LDS with direct global->LDS loads, two stages of 4 blocks ahead of the one
// being consumed: each wavefront's own 32 weight rows and their f16 block scales, and the
// token digits and scales of the stage, which the four wavefronts share.
#include <limits.h>
#include <type_traits>
#include "pg_internal.h"
#include "pg_stream_addr.h"
#include "pg_digits.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef const void __attribute__((address_space(1))) *gptr_t;
typedef void __attribute__((address_space(3))) *lptr_t;
typedef const v4i __attribute__((address_space(1))) *gv4i_ptr;

inline unsigned grid_for(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }

constexpr int NBU = 4;                              // blocks per stage
// LDS stage layout.  Every fill is arranged so that neighbouring lanes fetch neighbouring
// 16-byte chunks of global memory (whole 64- or 128-byte runs per request); the chunk order
// inside a run is XOR-swizzled so that the 128-bit LDS reads of 16 neighbouring lanes fall
// into 16 different 16-byte bank groups (gfx950 serves a 128-bit read over 256 bytes of banks a
// pass: with 8 distinct groups per 8 lanes only, lanes l and l + 8 collided and every such read
// took 8 cycles instead of 4).  For the digits that means: tokens 8 .. 15 (mod 16) keep their two
// planes in swapped places.
constexpr int DIG_STAGE = 64 * 128;                 // [token][plane] units of 128 B: 4 blocks x 2 halves  8 KiB
constexpr int D_STAGE = 4 * 256;                    // [wave][row group of 8][j][8 f16]                     1 KiB
constexpr int XS_STAGE = 32 * 16;                   // [token][4 block scales]                              512 B
constexpr int OFF_D = DIG_STAGE, OFF_XS = OFF_D + D_STAGE, OFF_W = OFF_XS + XS_STAGE;
template <int QT> struct MMCfg {
    static constexpr int W_WAVE = QT == 8 ? 64 * 64 : 32 * 64;  // per wavefront: [stream][4 blocks][16 B]
    static constexpr int W_FILLS = W_WAVE / 1024;               // weight fills per wavefront and stage
    static constexpr int STAGE = OFF_W + 4 * W_WAVE;            // 25.5 KiB (Q8_0) / 17.5 KiB (Q4_0)
    // Two LDS stages (one in flight beyond the one consumed), so that THREE workgroups share a CU (three wavefronts
    // a SIMD, 168 registers each).  Against two workgroups of three stages the expert products ran 2 % faster, the
    // 16-row product 6 % and the 1024-row o projection 7 %: a third wavefront fills the issue slots the other two
    // leave while they wait, which counts for more than the deeper ring.  (Three stages of the smaller Q4_0 stage,
    // 3 x 52.5 KiB a CU, measured like two workgroups: they do not fit three at a time.)
    static constexpr int RING = 2;
    static constexpr int AHEAD = RING - 1;
    static constexpr int LPS = 2 + 1 + 1 + W_FILLS;             // LDS fills per wavefront and stage
};

// ---- activation rows -> two byte-digit planes (pg_emit_mm_digits, pg_digits.h) ----------
template <bool NIB>
__global__ __launch_bounds__(256) void x_to_mm_digits_kernel(const float *__restrict__ x, int nb, int nbp,
                                                             int8_t *__restrict__ digits, float *__restrict__ xs,
                                                             float *__restrict__ xsum) {
    const size_t row = blockIdx.y;
    const int b = blockIdx.x * 32 + (threadIdx.x >> 3), sub = threadIdx.x & 7;
    if (b >= nb) return;  // whole 8-thread groups leave together
    const float4 v = reinterpret_cast<const float4 *>(x + (row * nb + b) * 32)[sub];
    const float f[4] = {v.x, v.y, v.z, v.w};
    pg_emit_mm_digits<NIB>(f, row, b, sub, nb, nbp, digits, xs, xsum);
}

// The rows' block sums alone (where the first term of Q4_1 runs on the f16 matrix cores).
__global__ __launch_bounds__(256) void block_sums_kernel(const float *__restrict__ x, int nb, int nbp, float *__restrict__ xsum) {
    const size_t row = blockIdx.y;
    const int b = blockIdx.x * 32 + (threadIdx.x >> 3), sub = threadIdx.x & 7;
    if (b >= nb) return;  // whole 8-thread groups leave together
    const float4 v = reinterpret_cast<const float4 *>(x + (row * nb + b) * 32)[sub];
    const float f[4] = {v.x, v.y, v.z, v.w};
    const float t = pg_block_sum(f);
    if (sub == 0) xsum[row * nbp + b] = t;
}

// Q4_1's second term on many rows: y[t][n] = first term + sum_b (8 d[n][b] + m[n][b]) * xsum[t][b]; the first,
// d sum (q - 8) x, is the Q4_0 product on the same nibbles, in y or (ks > 1) in the planes of its K chunks at part.
//
// Up to 64 tokens: workgroup = 16 weight rows x 16 tokens, thread = (row, one of 16 runs of blocks), 16 tokens in
// registers, eight blocks' scales requested at a time; the tokens' block sums wait in LDS as [b][16]; the runs are added
// in ascending order, a thread an output.  It is latency: a workgroup per 16 rows gives every CU one from 4096 rows on
// (64 rows a workgroup, one block's scales at a time and the planes added by a launch of their own took 17 us for
// 40 x 4096 -> 4096, this 8.7).
constexpr int Q41_TT = 16, Q41_NQ = 16;
__device__ __forceinline__ float q41_first_term(const float *part, int ks, size_t stride, const float *y, size_t i) {
    float v = ks > 1 ? part[i] : y[i];
    for (int s = 1; s < ks; ++s) v += part[(size_t)s * stride + i];
    return v;
}
__global__ __launch_bounds__(256) void q41_offset_kernel(const uint16_t *__restrict__ d, const uint16_t *__restrict__ m, int n_out,
                                                         int nb, const float *__restrict__ xsum, int nbp, int rows,
                                                         const float *__restrict__ part_in, int ks, size_t stride, float *y) {
    constexpr int RPW = 256 / Q41_NQ, AHEAD = 8;
    static_assert(RPW * Q41_TT == 256, "a thread adds one output's runs");
    extern __shared__ __attribute__((aligned(16))) float s_tile[];  // [nb][Q41_TT], then [Q41_NQ][RPW][Q41_TT + 1] partial sums
    const int t0 = blockIdx.y * Q41_TT, lrow = threadIdx.x % RPW, run = threadIdx.x / RPW;
    const int n = blockIdx.x * RPW + lrow;
    for (int i = threadIdx.x; i < nb * Q41_TT; i += 256) {
        const int t = i / nb, b = i - t * nb;  // (consecutive threads: consecutive blocks of one token)
        s_tile[b * Q41_TT + t] = t0 + t < rows ? xsum[(size_t)(t0 + t) * nbp + b] : 0.0f;
    }
    __syncthreads();
    float acc[Q41_TT];
#pragma unroll
    for (int t = 0; t < Q41_TT; ++t) acc[t] = 0.0f;
    const int nc = n < n_out ? n : n_out - 1;
    const size_t tile = (size_t)(nc >> 3) * nb * 8 + (nc & 7);
    const int per = (nb + Q41_NQ - 1) / Q41_NQ, b_lo = run * per, b_hi = b_lo + per < nb ? b_lo + per : nb;
    for (int b0 = b_lo; b0 < b_hi; b0 += AHEAD) {
        uint16_t db[AHEAD], mb[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const size_t at = tile + (size_t)(b0 + u < b_hi ? b0 + u : b_hi - 1) * 8;
            db[u] = d[at];
            mb[u] = m[at];
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (b0 + u >= b_hi) break;
            _Float16 dh, mh;
            __builtin_memcpy(&dh, &db[u], 2);
            __builtin_memcpy(&mh, &mb[u], 2);
            const float c = fmaf(8.0f, (float)dh, (float)mh);
#pragma unroll
            for (int t4 = 0; t4 < Q41_TT / 4; ++t4) {
                const float4 sv = *reinterpret_cast<const float4 *>(s_tile + (b0 + u) * Q41_TT + 4 * t4);
                acc[4 * t4] = fmaf(c, sv.x, acc[4 * t4]); acc[4 * t4 + 1] = fmaf(c, sv.y, acc[4 * t4 + 1]);
                acc[4 * t4 + 2] = fmaf(c, sv.z, acc[4 * t4 + 2]); acc[4 * t4 + 3] = fmaf(c, sv.w, acc[4 * t4 + 3]);
            }
        }
    }
    float *part = s_tile + nb * Q41_TT;
#pragma unroll
    for (int t = 0; t < Q41_TT; ++t) part[(run * RPW + lrow) * (Q41_TT + 1) + t] = acc[t];
    __syncthreads();
    const int t = run;  // (consecutive threads store consecutive rows)
    float sum = 0.0f;
#pragma unroll
    for (int qv = 0; qv < Q41_NQ; ++qv) sum += part[(qv * RPW + lrow) * (Q41_TT + 1) + t];
    if (n < n_out && t0 + t < rows) {
        const size_t i = (size_t)(t0 + t) * n_out + n;
        y[i] = q41_first_term(part_in, ks, stride, y, i) + sum;
    }
}

// From 65 tokens on it is a product like any other, over K = the blocks: v_mfma_f32_32x32x2_f32 (the vector form was
// bound by its own FMAs and LDS reads: 140 of 374 us at 1000 x 4096 -> 14336).  A wavefront takes 32 weight rows
// x 64 tokens.  The order in which blocks meet the instruction's k-slots is free, so lane half h takes blocks
// 8 i + 4 h .. + 3 for four instructions: one 128-bit load of a token's sums, and of a weight row's scales one 64-byte run
// per 8 rows.  Result lane = weight row: the read-modify-write of y goes in 128-byte runs.
//
// A step waits for memory and multiplies little, so where few tiles leave the chip idle the chain of steps is what counts.
// RUNS: a workgroup's four wavefronts share ONE tile, a quarter of the blocks each, and add their sums up through LDS in order
// of the blocks; else they take four tiles side by side, whose tokens' sums they read in common.
typedef float v16f __attribute__((ext_vector_type(16)));
template <bool RUNS>
__global__ __launch_bounds__(256) void q41_offset_mfma_kernel(const uint16_t *__restrict__ d, const uint16_t *__restrict__ m, int n_out,
                                                              int nb, const float *__restrict__ xsum, int nbp, int rows,
                                                              const float *__restrict__ part, int ks, size_t stride, float *y) {
    const int lane = threadIdx.x & 63, l31 = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = (RUNS ? blockIdx.x : blockIdx.x * 4 + wave) * 32 + l31, t0 = blockIdx.y * 64;
    if (n - l31 >= n_out) return;  // (with RUNS: none)
    const int nc = n < n_out ? n : n_out - 1;
    const size_t tile = (size_t)(nc >> 3) * nb * 8 + (nc & 7);
    const float *xt[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) xt[j] = xsum + (size_t)(t0 + 32 * j + l31 < rows ? t0 + 32 * j + l31 : rows - 1) * nbp;
    v16f acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
    uint16_t db[2][4], mb[2][4];
    float4 xv[2][2];
    auto load = [&](int buf, int i) {  // blocks past the end: the last one, its sum taken as zero
        const int b = 8 * i + 4 * h;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const size_t at = tile + (size_t)(b + c < nb ? b + c : nb - 1) * 8;
            db[buf][c] = d[at];
            mb[buf][c] = m[at];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float4 v = *reinterpret_cast<const float4 *>(xt[j] + (b < nbp ? b : 0));
            if (b + 3 >= nb) {
                v.x = b < nb ? v.x : 0.0f;
                v.y = b + 1 < nb ? v.y : 0.0f;
                v.z = b + 2 < nb ? v.z : 0.0f;
                v.w = 0.0f;
            }
            xv[buf][j] = v;
        }
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            _Float16 dh, mh;
            __builtin_memcpy(&dh, &db[buf][c], 2);
            __builtin_memcpy(&mh, &mb[buf][c], 2);
            const float w = fmaf(8.0f, (float)dh, (float)mh);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 v = xv[buf][j];
                const float a = c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, w, acc[j], 0, 0, 0);  // rows = tokens, columns = weight rows
            }
        }
    };
    const int all = (nb + 7) / 8, per = RUNS ? (all + 3) / 4 : all;
    const int begin = RUNS ? per * wave : 0, steps = RUNS ? min(all, begin + per) : all;
    if (begin < steps) load(0, begin);
    for (int i = begin; i < steps; i += 2) {
        if (i + 1 < steps) load(1, i + 1);
        multiply(0);
        if (i + 2 < steps) load(0, i + 2);
        if (i + 1 < steps) multiply(1);
    }
    if constexpr (RUNS) {  // register 16 j + r of all four runs is added up and stored by wavefront (16 j + r) / 8
        __shared__ float sums[4][32][64];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[wave][16 * j + r][lane] = acc[j][r];
        __syncthreads();
        if (n >= n_out) return;
        const int j = wave >> 1;
        auto at = [&](int u) { const int r = 8 * (wave & 1) + u; return 32 * j + 8 * (r >> 2) + 4 * h + (r & 3); };
        float first[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) first[u] = 0.0f;
        for (int s = 0; s < (ks > 1 ? ks : 1); ++s) {
            const float *p = (ks > 1 ? part + (size_t)s * stride : y) + (size_t)t0 * n_out + n;
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = t0 + at(u) < rows ? p[(size_t)at(u) * n_out] : 0.0f;
#pragma unroll
            for (int u = 0; u < 8; ++u) first[u] += v[u];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            float sum = sums[0][8 * wave + u][lane];
#pragma unroll
            for (int q = 1; q < 4; ++q) sum += sums[q][8 * wave + u][lane];
            if (t0 + at(u) < rows) y[(size_t)(t0 + at(u)) * n_out + n] = first[u] + sum;
        }
        return;
    }
    if (n >= n_out) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float first[16];  // every plane's sixteen loads together, and all of them before the stores
        auto at = [&](int r) { return 32 * j + 8 * (r >> 2) + 4 * h + (r & 3); };
#pragma unroll
        for (int r = 0; r < 16; ++r) first[r] = 0.0f;
        for (int s = 0; s < (ks > 1 ? ks : 1); ++s) {
            const float *p = (ks > 1 ? part + (size_t)s * stride : y) + (size_t)t0 * n_out + n;
            float v[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = t0 + at(r) < rows ? p[(size_t)at(r) * n_out] : 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) first[r] += v[r];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (t0 + at(r) < rows) y[(size_t)(t0 + at(r)) * n_out + n] = first[r] + acc[j][r];
    }
}

// Two's-complement nibbles (as stored at upload) of one dword -> four signed bytes holding
// 16 * (q - 8): a nibble moved to the top of its byte IS that value, no sign extension
// needed.  left = 4 takes the low nibble of every byte, left = 0 the high one.
__device__ __forceinline__ int nibbles_to_i8x16(int v, int left) {
    return (int)(((unsigned)v << left) & 0xF0F0F0F0u);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
    _Float16 v;
    const uint16_t hb = (uint16_t)h;
    __builtin_memcpy(&v, &hb, 2);
    return (float)v;
}

// Tiles of `slots` pairs that experts' lists fill at most, T pairs each and P together: a launch over experts x ceil(T / slots) of them is
// mostly workgroups that read a count and leave, a round of the chip each 768 of them (256 tokens, top 1 of 16 experts of 1024 x 4096,
// Q4_0: 98.8 -> 67.5 us; 2000, 2 of 8, Q8_0: 444 -> 418; 64, 2 of 8 of 3072 x 8192: 155 -> 150; 81 to 2048 tokens 7 % in the mean).
inline size_t expert_tiles_bound(size_t experts, size_t T, size_t P, size_t slots) {
    return std::min(std::min(P, (P + experts * (slots - 1)) / slots), experts * ((T + slots - 1) / slots));
}
// The expert that tile `tile` of all experts' tiles belongs to (-1: past the last), its number among that expert's and the expert's pairs.
// By a wavefront, 64 experts at a time: sums of their tiles up to each lane's, within rows of 16 lanes and then across them.
__device__ __forceinline__ int expert_of_tile(const int *__restrict__ counts, int experts, int slots, int lane, int &tile, int &count) {
    for (int e0 = 0; e0 < experts; e0 += 64) {
        const int c = e0 + lane < experts ? counts[e0 + lane] : 0, mine = (int)((unsigned)(c + slots - 1) / (unsigned)slots);
        int sum = mine;
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x111, 0xf, 0xf, false);  // row_shr:1, 2, 4, 8
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x112, 0xf, 0xf, false);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x114, 0xf, 0xf, false);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x118, 0xf, 0xf, false);
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
        sum += __builtin_amdgcn_update_dpp(0, sum, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
        const unsigned long long past = __ballot(sum > tile);
        if (past) {
            const int l = __builtin_ctzll(past);
            tile -= __builtin_amdgcn_readlane(sum - mine, l);
            count = __builtin_amdgcn_readlane(c, l);
            return e0 + l;
        }
        tile -= __builtin_amdgcn_readlane(sum, 63);
    }
    return -1;
}

// grid: x = tiles of 128 weight rows, y = token tile (with lists, of all experts: expert_of_tile), z = K chunk.
// `chunk` (blocks per K chunk) is a multiple of NBU and no chunk is empty.
// out: [K chunks][total pairs][n_out] (plain y with one chunk).
// (Three wavefronts per SIMD, 168 registers each: the MFMA results are written to ordinary VGPRs,
// not to accumulation registers that would have to be copied out first.)
// NT: the weight fills carry the non-temporal hint.  Right for the expert products, where a
// weight byte is used by one or two workgroups and 1.7 GB of them per launch would otherwise
// push the activations, digits and partial sums of the neighbouring kernels out of the caches
// (MoE step 1.22 -> 1.17 ms); wrong for a prefill, where 32 token tiles re-read every weight.
template <int QT, bool NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void gguf_mm_kernel(const uint8_t *__restrict__ qs0, const uint16_t *__restrict__ d0,
                                                      pg_mm_group grp, int n_out_arg, int nb, int nbp, int chunk,
                                                      const int8_t *__restrict__ digits, const float *__restrict__ xs,
                                                      float *__restrict__ out_arg, size_t part_stride_arg) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];  // RING * STAGE bytes
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l31 = lane & 31, hh = lane >> 5;

    // Which 128 weight rows (bx) and which token tile (by).  With many token tiles (a prefill)
    // the launch is one-dimensional and XCD-aware: workgroup id = 8 * j + xcd, and the j-th
    // workgroup of an XCD is member j % 32 of super-tile (j / 32) * 8 + xcd, a super-tile being
    // 4 row groups x 8 token tiles whose weights and digits (about 3 MB) stay in that XCD's L2
    // while its 32 workgroups run: each weight row group is fetched once per 8 token tiles
    // instead of once per tile.
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (grp.xcd_ks) {
        // K chunks dealt to XCDs (workgroup id % 8 = XCD): chunk z runs on the 8 / ks XCDs with
        // id % ks == z, so an XCD's L2 holds only its chunk of the activation digits, and the
        // workgroups of an XCD walk the row groups of one token tile after another.
        const int xcd = blockIdx.x & 7, per = 8 / grp.xcd_ks;
        const int j = (blockIdx.x >> 3) * per + xcd / grp.xcd_ks;
        if (j >= grp.remap_rg * grp.remap_tiles) return;
        bz = xcd % grp.xcd_ks;
        bx = j % grp.remap_rg;
        by = j / grp.remap_rg;
    } else if (grp.remap_rg) {
        const int nrgb = (grp.remap_rg + 3) / 4, ntb = (grp.remap_tiles + 7) / 8;
        const int jj = blockIdx.x >> 3, st = (jj >> 5) * 8 + (blockIdx.x & 7), w = jj & 31;
        if (st >= nrgb * ntb) return;
        bx = (st % nrgb) * 4 + (w & 3);
        by = (st / nrgb) * 8 + (w >> 2);
        if (bx >= grp.remap_rg || by >= grp.remap_tiles) return;
    }
    int e = 0, tt = by, count = grp.max_count;
    if (grp.counts) {
        e = expert_of_tile(grp.counts, grp.num_experts, 32, lane, tt, count);
        if (e < 0) return;  // the same for every thread of the workgroup
    } else if (tt * 32 >= count) return;
    int n_out = n_out_arg;
    float *__restrict__ out = out_arg;
    const uint8_t *const *qs_table = grp.qs_table;
    const uint16_t *const *d_table = grp.d_table;
    if (grp.nseg < 0 && bx >= (n_out_arg + 127) / 128) {  // the expert's second tensor
        bx -= (n_out_arg + 127) / 128;
        qs_table = grp.qs_table2;
        d_table = grp.d_table2;
        out = grp.out2;
    }
    const uint8_t *qs_any = qs_table ? qs_table[e] : qs0;
    const uint16_t *d_any = d_table ? d_table[e] : d0;
    size_t part_stride = part_stride_arg;
    if (grp.nseg > 0) {  // which tensor of the launch this row group belongs to
        int t = 0;
        while (t + 1 < grp.nseg && bx >= grp.seg_first[t + 1]) ++t;
        bx -= grp.seg_first[t];
        qs_any = grp.seg_qs[t];
        d_any = grp.seg_d[t];
        n_out = grp.seg_n[t];
        out = grp.seg_out[t];
        part_stride = grp.seg_stride[t];
    }

    constexpr int STAGE = MMCfg<QT>::STAGE, W_WAVE = MMCfg<QT>::W_WAVE, W_FILLS = MMCfg<QT>::W_FILLS;
    // Activation row of a token slot of this tile (spare slots shadow the tile's first token).
    auto xrow_of = [&](int tok) -> size_t {
        const int slot = tt * 32 + tok;
        const int slot_c = slot < count ? slot : tt * 32;
        const int pr = grp.lists ? grp.lists[(size_t)e * grp.list_stride + slot_c] : slot_c;
        return (size_t)(pr / grp.x_row_div);
    };
    // Orientation of the 32x32 result tile: TOKENS on the accumulator-register axis (register r
    // of lanes with hh = lane/32 holds token slot 8*(r/4) + 4*hh + r%4), WEIGHT ROWS on the lanes.
    // A tile with few tokens then needs only the first NR registers scaled and accumulated:
    // NR = 4 covers 8 token slots, 8 covers 16, 16 all 32.
    const int ntok = count - tt * 32 < 32 ? count - tt * 32 : 32;

    // Fill duties of this lane.
    // digits: fill n = 2*wave + u covers units 8n .. 8n+7, unit = 2*token + plane; the lane
    // fetches chunk (lane & 7) ^ (token & 7) of the unit's 128 bytes, chunk = 2*block + half.
    const int8_t *dig_src[2];
    int dig_jb[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int unit = (2 * wave + u) * 8 + (lane >> 3), tok = unit >> 1, pl = (unit & 1) ^ ((tok >> 3) & 1);
        const int ch = (lane & 7) ^ (tok & 7);
        dig_jb[u] = ch >> 1;
        dig_src[u] = digits + xrow_of(tok) * pg_mm_row_bytes(nb) + (size_t)pl * nb * 32 + (ch & 1) * 16;
    }
    // xs: lanes 0..7 of wavefront w fetch the 4 block scales of tokens 8w .. 8w+7
    const float *xs_src = xs + xrow_of(8 * wave + (lane & 7)) * (size_t)nbp;
    // weights: fill q covers streams 16q .. 16q+15 (Q8_0: stream = 32*half + row, Q4_0: stream = row);
    // the lane fetches block (lane & 3) ^ swizzle of the stream's 4 blocks.
    const int row0 = bx * 128 + wave * 32;
    const int w_jb = (lane & 3) ^ ((lane >> 4) & 3);  // (stream >> 2) & 3, stream = 16q + (lane >> 2)
    const int8_t *w_src[W_FILLS];
#pragma unroll
    for (int q = 0; q < W_FILLS; ++q) {
        const int st = 16 * q + (lane >> 2);
        const int wrow = row0 + (st & 31) < n_out ? row0 + (st & 31) : n_out - 1;  // clamped; masked at the store
        w_src[q] = reinterpret_cast<const int8_t *>(qs_any) +
                   (QT == 8 ? ((size_t)wrow * 2 + (st >> 5)) * nb * 16 : (size_t)wrow * nb * 16);
        // Tile-major copy: [row group][4 blocks][wavefront][fill][lane] 16-byte chunks, the very
        // order of the fills below, padded with zero rows and blocks: a stage of a workgroup is
        // 4 * W_WAVE contiguous bytes (row groups pg_tiled_group_bytes apart).
        if (grp.tiled)
            w_src[q] = reinterpret_cast<const int8_t *>(qs_any) +
                       (size_t)bx * pg_tiled_group_bytes(nb, QT == 8) + wave * W_WAVE + q * 1024 + lane * 16;
    }
    // f16 scales of this wavefront's 32 rows: lane -> (group lane/16, block (lane/4)%4, dword lane%4)
    const int ngroups = (n_out + 7) / 8;
    int dg = (row0 >> 3) + (lane >> 4);
    dg = dg < ngroups ? dg : ngroups - 1;
    const char *d_grp = reinterpret_cast<const char *>(d_any) + (size_t)dg * nb * 16 + (lane & 3) * 4;
    const int d_jb = (lane >> 2) & 3;

    const int b_begin = bz * chunk;
    const int b_end = b_begin + chunk < nb ? b_begin + chunk : nb;
    const int nst = (b_end - b_begin + NBU - 1) / NBU;

    // Every load of the K loop is a direct global->LDS fill, so the only memory waits in the
    // loop are the explicit ones below (two stages stay in flight across the barrier).
    // (The ring slot is a compile-time constant everywhere so that the compiler can tell the
    // stage being filled from the stage being read and adds no waits of its own.)
    auto issue = [&](auto ring_slot, int s) {
        const int b0 = b_begin + s * NBU;
        char *base = lds + decltype(ring_slot)::value * STAGE;
        auto blk = [&](int j) { return (size_t)(b0 + j < b_end ? b0 + j : b_end - 1); };  // past the end: a valid, unused block
#pragma unroll
        for (int u = 0; u < 2; ++u)
            __builtin_amdgcn_global_load_lds((gptr_t)(dig_src[u] + blk(dig_jb[u]) * 32), (lptr_t)(base + (2 * wave + u) * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(d_grp + blk(d_jb) * 16), (lptr_t)(base + OFF_D + wave * 256), 4, 0, 0);
        if (lane < 8)
            __builtin_amdgcn_global_load_lds((gptr_t)(xs_src + b0), (lptr_t)(base + OFF_XS + wave * 128), 16, 0, 0);
        const size_t w_off = grp.tiled ? (size_t)(b0 >> 2) * (4 * W_WAVE) : blk(w_jb) * 16;
#pragma unroll
        for (int q = 0; q < W_FILLS; ++q)
            __builtin_amdgcn_global_load_lds((gptr_t)(w_src[q] + w_off), (lptr_t)(base + OFF_W + wave * W_WAVE + q * 1024), 16, 0, NT ? 2 : 0);
    };

    float acc[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;

    // One block of the stage at `base`: operands from LDS, two MFMAs, scale-and-accumulate.
    // Split into three phases so that the full-stage path can overlap them across blocks.
    const int w_rd = OFF_W + wave * W_WAVE + (QT == 8 ? lane : l31) * 64, w_sw = ((QT == 8 ? lane : l31) >> 2) & 3;
    const int dig_rd = l31 * 256, dig_sw = l31 & 7, dig_hi = ((l31 >> 3) & 1) * 128;  // tokens 8 .. 15 (mod 16) keep their planes swapped
    const int d_rd = OFF_D + wave * 256 + (l31 >> 3) * 64 + (l31 & 7) * 2;  // this lane's weight row: [group of 8][j][8 f16]
    auto read_ab = [&](const char *base, int j, v4i (&ab)[3]) {
        ab[0] = *reinterpret_cast<const v4i *>(base + w_rd + ((j ^ w_sw) * 16));
        ab[1] = *reinterpret_cast<const v4i *>(base + dig_rd + dig_hi + (((2 * j + hh) ^ dig_sw) * 16));
        ab[2] = *reinterpret_cast<const v4i *>(base + dig_rd + (128 - dig_hi) + (((2 * j + hh) ^ dig_sw) * 16));
    };
    // the block's weight scale of this lane's row
    // (read as integers: a float-typed LDS read makes the compiler wait for every fill in flight)
    auto read_d = [&](const char *base, int j, unsigned &dbits) {
        dbits = *reinterpret_cast<const unsigned short *>(base + d_rd + j * 16);
    };
    auto mfmas = [&](const v4i (&ab)[3], v16i &ihi, v16i &ilo) {
        v4i a = ab[0];
        if constexpr (QT == 4) {
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = nibbles_to_i8x16(a[t], 4 - 4 * hh);
        }
        v16i zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0;
        ihi = __builtin_amdgcn_mfma_i32_32x32x32_i8(ab[1], a, zero, 0, 0, 0);  // rows = tokens, columns = weight rows
        ilo = __builtin_amdgcn_mfma_i32_32x32x32_i8(ab[2], a, zero, 0, 0, 0);
    };
    auto scale_acc = [&](auto nr, const v16i &ihi, const v16i &ilo, unsigned dbits, const int (&sx)[16][4], int j) {
        float dv = half_bits_to_float(dbits);
        if constexpr (QT == 4) dv *= 0.0625f;  // the weight operand was 16 * (q - 8)
#pragma unroll
        for (int r = 0; r < decltype(nr)::value; ++r) {
            // |integer| < 2^31: rounded to 24 bits, then scaled (two roundings of 2^-24, far below the digit step)
            const float fx = (float)(ihi[r] * 256 + ilo[r]) * __int_as_float(sx[r][j]);
            acc[r] = fmaf(dv, fx, acc[r]);
        }
    };
    auto compute = [&](auto nr, auto ring_slot, int s) {
        const int b0 = b_begin + s * NBU;
        const char *base = lds + decltype(ring_slot)::value * STAGE;
        // activation scales of this lane's NR token slots for the stage's four blocks
        // (vector element -> named int: a bit cast applied directly to a vector element
        // expression was compiled as a cast of element 0)
        int sx[16][4];
#pragma unroll
        for (int r = 0; r < decltype(nr)::value; ++r) {
            const v4i t = *reinterpret_cast<const v4i *>(base + OFF_XS + (8 * (r >> 2) + 4 * hh + (r & 3)) * 16);
            const int t0 = t[0], t1 = t[1], t2 = t[2], t3 = t[3];
            sx[r][0] = t0; sx[r][1] = t1; sx[r][2] = t2; sx[r][3] = t3;
        }
        v4i ab[2][3];
        unsigned dd[2];
        v16i ihi[2], ilo[2];
        if (b0 + NBU <= b_end) {  // full stage (wavefront-uniform)
            // Software pipeline over the 4 blocks: while block j is scaled and accumulated on
            // the vector ALU, the MFMAs of block j+1 run and the LDS reads of block j+2 return.
            read_ab(base, 0, ab[0]);
            read_d(base, 0, dd[0]);
            read_ab(base, 1, ab[1]);
            mfmas(ab[0], ihi[0], ilo[0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NBU; ++j) {
                if (j + 1 < NBU) {
                    mfmas(ab[(j + 1) & 1], ihi[(j + 1) & 1], ilo[(j + 1) & 1]);
                    __builtin_amdgcn_sched_barrier(0);  // younger LDS reads must not be waited for here
                    read_d(base, j + 1, dd[(j + 1) & 1]);
                }
                if (j + 2 < NBU) read_ab(base, j + 2, ab[j & 1]);
                __builtin_amdgcn_sched_barrier(0);
                scale_acc(nr, ihi[j & 1], ilo[j & 1], dd[j & 1], sx, j);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NBU - 1; ++j)
                if (b0 + j < b_end) {
                    read_ab(base, j, ab[0]);
                    read_d(base, j, dd[0]);
                    mfmas(ab[0], ihi[0], ilo[0]);
                    scale_acc(nr, ihi[0], ilo[0], dd[0], sx, j);
                }
        }
    };

    // ---- the other orientation, for tiles with more than 16 tokens: weight rows on the
    // accumulator-register axis (register r <-> row 8*(r/4) + 4*hh + r%4), tokens on the lanes.
    // All 16 registers are needed either way, and this way round the activation scales are one
    // LDS read per stage instead of sixteen.
    auto read_d_rows = [&](const char *base, int j, v2i (&dd)[4]) {
#pragma unroll
        for (int g = 0; g < 4; ++g)  // rows 8g + 4*hh + {0..3}  <->  accumulator registers 4g .. 4g+3
            dd[g] = *reinterpret_cast<const v2i *>(base + OFF_D + wave * 256 + (g * 4 + j) * 16 + hh * 8);
    };
    auto mfmas_rows = [&](const v4i (&ab)[3], v16i &ihi, v16i &ilo) {  // rows = weight rows, columns = tokens
        v4i a = ab[0];
        if constexpr (QT == 4) {
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = nibbles_to_i8x16(a[t], 4 - 4 * hh);
        }
        v16i zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0;
        ihi = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, ab[1], zero, 0, 0, 0);
        ilo = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, ab[2], zero, 0, 0, 0);
    };
    auto scale_acc_rows = [&](const v16i &ihi, const v16i &ilo, const v2i (&dd)[4], float sj) {
        if constexpr (QT == 4) sj *= 0.0625f;  // the weight operand was 16 * (q - 8)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = 4 * g + q;
                const uint32_t pairbits = (uint32_t)dd[g][q >> 1];
                const float dv = half_bits_to_float((q & 1) ? pairbits >> 16 : pairbits & 0xFFFFu);
                // |integer| < 2^31: rounded to 24 bits, then scaled (two roundings of 2^-24, far below the digit step)
                const float fx = (float)(ihi[r] * 256 + ilo[r]) * sj;
                acc[r] = fmaf(dv, fx, acc[r]);
            }
    };
    auto compute_rows = [&](auto ring_slot, int s) {
        const int b0 = b_begin + s * NBU;
        const char *base = lds + decltype(ring_slot)::value * STAGE;
        // Read as integers: a float-typed LDS read makes the compiler wait for every LDS fill in
        // flight (it cannot tell the stages apart), an int-typed one leaves the waits to us.
        const v4i sxi = *reinterpret_cast<const v4i *>(base + OFF_XS + l31 * 16);
        // (element -> named int -> float: a bit cast applied directly to a vector element
        // expression was compiled as a cast of element 0)
        const int sx0 = sxi[0], sx1 = sxi[1], sx2 = sxi[2], sx3 = sxi[3];
        const float sx[4] = {__int_as_float(sx0), __int_as_float(sx1), __int_as_float(sx2), __int_as_float(sx3)};
        v4i ab[2][3];
        v2i dd[2][4];
        v16i ihi[2], ilo[2];
        if (b0 + NBU <= b_end) {  // full stage (wavefront-uniform)
            // Software pipeline over the 4 blocks: while block j is scaled and accumulated on
            // the vector ALU, the MFMAs of block j+1 run and the LDS reads of block j+2 return.
            read_ab(base, 0, ab[0]);
            read_d_rows(base, 0, dd[0]);
            read_ab(base, 1, ab[1]);
            mfmas_rows(ab[0], ihi[0], ilo[0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NBU; ++j) {
                if (j + 1 < NBU) {
                    mfmas_rows(ab[(j + 1) & 1], ihi[(j + 1) & 1], ilo[(j + 1) & 1]);
                    __builtin_amdgcn_sched_barrier(0);  // younger LDS reads must not be waited for here
                    read_d_rows(base, j + 1, dd[(j + 1) & 1]);
                }
                if (j + 2 < NBU) read_ab(base, j + 2, ab[j & 1]);
                __builtin_amdgcn_sched_barrier(0);
                scale_acc_rows(ihi[j & 1], ilo[j & 1], dd[j & 1], sx[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NBU - 1; ++j)
                if (b0 + j < b_end) {
                    read_ab(base, j, ab[0]);
                    read_d_rows(base, j, dd[0]);
                    mfmas_rows(ab[0], ihi[0], ilo[0]);
                    scale_acc_rows(ihi[0], ilo[0], dd[0], sx[j]);
                }
        }
    };

    auto wait_barrier = [&](bool one_ahead) {
        if (one_ahead) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n s_barrier" ::"n"(MMCfg<QT>::LPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
    };

    constexpr int RING = MMCfg<QT>::RING, AHEAD = MMCfg<QT>::AHEAD;
    issue(std::integral_constant<int, 0>{}, 0);
    if (AHEAD > 1 && nst > 1) issue(std::integral_constant<int, 1 % RING>{}, 1);
    auto k_loop = [&](auto nr) {
        for (int s0 = 0; s0 < nst; s0 += RING) {
#define PG_MM_STEP(U)                                                                     \
            if (s0 + U < nst) {                                                           \
                const int s = s0 + U;                                                     \
                wait_barrier(AHEAD > 1 && s + 1 < nst);                                   \
                if (s + AHEAD < nst) issue(std::integral_constant<int, (U + AHEAD) % RING>{}, s + AHEAD); \
                compute(nr, std::integral_constant<int, U>{}, s);                         \
            }
            PG_MM_STEP(0)
            PG_MM_STEP(1)
            if constexpr (RING > 2) { PG_MM_STEP(2) }
#undef PG_MM_STEP
        }
    };
    if (ntok > 16) {  // the same choice for the whole workgroup
        for (int s0 = 0; s0 < nst; s0 += RING) {
#define PG_MM_STEP(U)                                                                     \
            if (s0 + U < nst) {                                                           \
                const int s = s0 + U;                                                     \
                wait_barrier(AHEAD > 1 && s + 1 < nst);                                   \
                if (s + AHEAD < nst) issue(std::integral_constant<int, (U + AHEAD) % RING>{}, s + AHEAD); \
                compute_rows(std::integral_constant<int, U>{}, s);                        \
            }
            PG_MM_STEP(0)
            PG_MM_STEP(1)
            if constexpr (RING > 2) { PG_MM_STEP(2) }
#undef PG_MM_STEP
        }
        const bool tok_ok = tt * 32 + l31 < count;  // the token whose outputs this lane accumulated
        if (!tok_ok) return;
        const int pair = grp.lists ? grp.lists[(size_t)e * grp.list_stride + tt * 32 + l31] : tt * 32 + l31;
        float *y = out + bz * part_stride + (size_t)pair * n_out;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int r0 = row0 + 8 * g + 4 * hh;
            if (r0 + 3 < n_out && (n_out & 3) == 0) {
                *reinterpret_cast<float4 *>(y + r0) = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (r0 + q < n_out) y[r0 + q] = acc[4 * g + q];
            }
        }
        return;
    }
    if (ntok <= 8) k_loop(std::integral_constant<int, 4>{});
    else k_loop(std::integral_constant<int, 8>{});

    // lanes hold consecutive weight rows: each token's 32 outputs leave as one 128-byte run
    const int row = row0 + l31;
    if (row >= n_out) return;
    float *ybase = out + bz * part_stride + row;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int tok = 8 * (r >> 2) + 4 * hh + (r & 3);
        if (tok < ntok) {
            const int slot = tt * 32 + tok;
            const int pair = grp.lists ? grp.lists[(size_t)e * grp.list_stride + slot] : slot;
            ybase[(size_t)pair * n_out] = acc[r];
        }
    }
}

// ---- up to 8 activation rows over a Q4_0 or Q8_0 tensor in one launch after the digits --------------------------
// The product above splits K between workgroups where one token tile meets a wide tensor, and a third launch adds
// the planes.  Here a workgroup owns 16 NB weight rows and all of K: its NW wavefronts take one run of K each, every
// wavefront with an LDS ring of its own (no barrier in the loop: it reads only what it loaded itself), and their
// f32 tiles are added through LDS in a fixed order at the end.  A unit of the ring is 8 blocks (256 k): the weight
// tiles as whole 128-byte lines per row (8 rows an instruction, 16-byte chunk p of row r at position
// p ^ ((r >> 1) & 7)), their f16 scales, the two digit planes of the MT token rows (256 bytes a row and plane,
// chunk c of token t at position c ^ t) and the tokens' block scales; NST - 1 units are in flight while one is
// consumed.  The weights are read in the row-major planes every tensor has (no tile-major copy).  Each workgroup starts its
// walk through K at its own unit.
// MT: token rows the ring holds (4 or 8: the digits are most of a unit, and the fewer there are the more units
// fit in flight); token slots from MT on read the rows of slots 0 .. MT - 1 again and are never stored.
// QT = 8 (Q8_0): a weight row is two streams (bytes 0 .. 15 and 16 .. 31 of its blocks, as the upload splits them), 32
// streams a tile, kept in LDS half-major (stream slot 16 half + row) so that the fragment reads of 16 rows and one
// half stay free of bank conflicts; no nibbles to unpack.
// Up to three tensors of equal K in one launch (q|k|v, gate|up of models::llama): tensor g owns the workgroups
// wg0[g] .. wg0[g + 1] - 1 (unused slots hold INT_MAX).
template <int QT, int NB, int MT, int NW, int NST>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 4))) void gguf_skinny_kernel(const int8_t *__restrict__ digits, const float *__restrict__ xs,
                                                                    const pg_skinny_group grp, int nb, int nbp, int m) {
    int tg = 0;
#pragma unroll
    for (int i = 1; i < 3; ++i) tg = (int)blockIdx.x >= grp.wg0[i] ? i : tg;
    const uint8_t *__restrict__ qs = grp.qs[tg];
    const uint16_t *__restrict__ dsc = grp.d[tg];
    float *__restrict__ y = grp.y[tg];
    const float *__restrict__ res = grp.res[tg];
    const int n_out = grp.n[tg];
    constexpr int WF = QT == 8 ? 4 : 2, W_T = WF * 1024, D_T = 256, DIG = MT * 512, XS_B = 512, GQ = MT / 2;  // WF, GQ: weight, digit fills per unit
    constexpr int OFF_DS = NB * W_T, OFF_DG = OFF_DS + NB * D_T, OFF_X = OFF_DG + DIG, UNIT = OFF_X + XS_B;
    constexpr int LPS = WF * NB + 1 + GQ + 1;  // fills per unit
    static_assert(MT == 4 || MT == 8, "tokens in quads");
    static_assert((NST - 1) * LPS < 64 && NST <= 6 && NB <= 2, "the wait counter holds 63");
    extern __shared__ __attribute__((aligned(1024))) char lds[];  // NW rings of NST units; afterwards the wavefronts' tiles
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = ((int)blockIdx.x - grp.wg0[tg]) * 16 * NB;
    const int units = nb / 8, per = (units + NW - 1) / NW;
    const int u_begin = wave * per, u_end = u_begin + per < units ? u_begin + per : units;
    const int cnt = u_end - u_begin;
    char *ring = lds + (size_t)wave * NST * UNIT;
    const size_t row_bytes = pg_mm_row_bytes(nb);

    // fill duties of this lane
    const uint8_t *w_src[NB][WF];  // stream slot 8 j + lane / 8 of tile c (Q4_0: slot = row; Q8_0: slot = 16 half + row), chunk (lane % 8) ^ ((row >> 1) & 7); rows past the end: the last
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int j = 0; j < WF; ++j) {
            const int slot = 8 * j + (lane >> 3), r = slot & 15, half = slot >> 4, ch = (lane & 7) ^ ((r >> 1) & 7);
            const int row = pg_gemv_clamp_row(n0 + 16 * c + r, n_out);
            w_src[c][j] = qs + pg_gskinny_weight_offset(QT == 8 ? (size_t)row * 2 + half : (size_t)row, nb, 0, ch);
        }
    // scales: lanes 0 .. 16 NB - 1: scale tile (n0 / 8 + lane / 8), blocks of the unit lane % 8 (16 bytes = 8 rows x f16)
    const int ntile = (n_out + 7) / 8;
    const int dt = pg_gskinny_scale_tile(n0, lane, ntile);
    const char *d_src = reinterpret_cast<const char *>(dsc) + pg_gskinny_scale_offset(dt, nb, 0, lane);
    // digits: instruction q covers runs 4 q .. 4 q + 3, run = 2 token + plane; lane -> run 4 q + lane / 16, position lane % 16
    const int8_t *g_src[GQ];
#pragma unroll
    for (int q = 0; q < GQ; ++q) {
        const int run = 4 * q + (lane >> 4), tok = run >> 1, pl = run & 1;
        const int ch = (lane & 15) ^ tok;
        g_src[q] = digits + (size_t)(tok < m ? tok : 0) * row_bytes + (size_t)pl * nb * 32 + ch * 16;
    }
    // token scales: lanes 0 .. 2 MT - 1: token lane / 2, blocks 4 (lane % 2) .. + 3 of the unit
    const float *x_src = xs + (size_t)((lane >> 1) < m ? (lane >> 1) : 0) * nbp + 4 * (lane & 1);

    const int rot = cnt > 0 ? (int)((blockIdx.x * 5u) % (unsigned)cnt) : 0;
    auto issue = [&](auto slot, int t) {
        const size_t unit = (size_t)pg_skinny_walk_unit(u_begin, cnt, t, rot);
        char *base = ring + decltype(slot)::value * UNIT;
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int j = 0; j < WF; ++j)
                __builtin_amdgcn_global_load_lds((gptr_t)(w_src[c][j] + unit * 128), (lptr_t)(base + c * W_T + j * 1024), 16, 0, 2);
        if (lane < 16 * NB) __builtin_amdgcn_global_load_lds((gptr_t)(d_src + unit * 128), (lptr_t)(base + OFF_DS), 16, 0, 0);
#pragma unroll
        for (int q = 0; q < GQ; ++q)
            __builtin_amdgcn_global_load_lds((gptr_t)(g_src[q] + unit * 256), (lptr_t)(base + OFF_DG + q * 1024), 16, 0, 0);
        if (lane < 2 * MT) __builtin_amdgcn_global_load_lds((gptr_t)(x_src + unit * 8), (lptr_t)(base + OFF_X), 16, 0, 0);
    };

    // fragment reads of this lane
    const int fr = lane & 15, g4 = lane >> 4;
    const int w_sw = (fr >> 1) & 7;
    const int ds_rd = OFF_DS + (fr >> 3) * 128 + (fr & 7) * 2;              // + tile c * 256 + j * 16: this lane's weight row

    // v_mfma_i32_4x4x4_i8: sixteen independent 4 x 4 x 4 products an instruction.
    // Product b of a lane quad takes weight rows 4 (b % 4) .. + 3 against four tokens for FOUR DIFFERENT blocks of K
    // (block lane / 16 of a group of four): lane -> weight row lane % 16 of block lane / 16, its eight operand
    // dwords the block's 32 k; the token operand comes from lane % 4's token (one more set of instructions for
    // tokens 4 .. 7).  The result registers are the four tokens of the lane's own row and block, so nothing of the
    // 16 x 16 tile is padding.  A lane sums blocks lane / 16, + 4, ...; the four partial sums of a
    // row meet in the final pass through LDS.
    constexpr int NQ = MT / 4, NS = NB * NQ;  // accumulator sets: weight tiles x token quads
    float acc[NS][4];
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[c][i] = 0.0f;

    auto consume = [&](auto slot) {
        const char *base = ring + decltype(slot)::value * UNIT;
        const int tq = lane & 3;  // the token (of each set) whose digits this lane hands to its quad
#pragma unroll
        for (int J = 0; J < 2; ++J) {
            const int blk = 4 * J + g4;
            // the lane's rows (one a tile) and block: 32 weight bytes each as eight dwords in the order of the digit halves
            int wk[NB][8];
            float dv[NB];
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const char *wt = base + c * W_T;
                if constexpr (QT == 4) {
                    const v4i wr = *reinterpret_cast<const v4i *>(wt + fr * 128 + ((blk ^ w_sw) * 16));
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        wk[c][p] = nibbles_to_i8x16(wr[p], 4);      // low nibbles: the even elements (digit half 0)
                        wk[c][4 + p] = nibbles_to_i8x16(wr[p], 0);  // high nibbles: the odd ones (half 1)
                    }
                } else {
                    const v4i w0 = *reinterpret_cast<const v4i *>(wt + fr * 128 + ((blk ^ w_sw) * 16));
                    const v4i w1 = *reinterpret_cast<const v4i *>(wt + (16 + fr) * 128 + ((blk ^ w_sw) * 16));
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        wk[c][p] = w0[p];
                        wk[c][4 + p] = w1[p];
                    }
                }
                dv[c] = half_bits_to_float(*reinterpret_cast<const unsigned short *>(base + ds_rd + c * D_T + blk * 16));
            }
#pragma unroll
            for (int s2 = 0; s2 < NQ; ++s2) {
                const int tok = 4 * s2 + tq;
                const char *dg = base + OFF_DG + tok * 512;
                const v4i h0 = *reinterpret_cast<const v4i *>(dg + (((2 * blk) ^ tok) * 16));
                const v4i h1 = *reinterpret_cast<const v4i *>(dg + (((2 * blk + 1) ^ tok) * 16));
                const v4i l0 = *reinterpret_cast<const v4i *>(dg + 256 + (((2 * blk) ^ tok) * 16));
                const v4i l1 = *reinterpret_cast<const v4i *>(dg + 256 + (((2 * blk + 1) ^ tok) * 16));
                int sx[4];  // the scales of tokens 4 s2 .. + 3 for this lane's block (read as integers: see gguf_mm_kernel)
#pragma unroll
                for (int i = 0; i < 4; ++i) sx[i] = *reinterpret_cast<const int *>(base + OFF_X + (4 * s2 + i) * 32 + blk * 4);
#pragma unroll
                for (int c = 0; c < NB; ++c) {
                    v4i ihi = {0, 0, 0, 0}, ilo = {0, 0, 0, 0};
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        ihi = __builtin_amdgcn_mfma_i32_4x4x4i8(h0[p], wk[c][p], ihi, 0, 0, 0);  // rows = tokens, columns = weight rows
                        ilo = __builtin_amdgcn_mfma_i32_4x4x4i8(l0[p], wk[c][p], ilo, 0, 0, 0);
                    }
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        ihi = __builtin_amdgcn_mfma_i32_4x4x4i8(h1[p], wk[c][4 + p], ihi, 0, 0, 0);
                        ilo = __builtin_amdgcn_mfma_i32_4x4x4i8(l1[p], wk[c][4 + p], ilo, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float fx = (float)(ihi[i] * 256 + ilo[i]) * __int_as_float(sx[i]);
                        acc[c * NQ + s2][i] = fmaf(dv[c], fx, acc[c * NQ + s2][i]);
                    }
                }
            }
        }
    };

    if (cnt > 0) {
#define PG_GS_PRO(U) if (U < NST - 1 && U < cnt) issue(std::integral_constant<int, (U < NST ? U : 0)>{}, U);
        PG_GS_PRO(0) PG_GS_PRO(1) PG_GS_PRO(2) PG_GS_PRO(3) PG_GS_PRO(4)
#undef PG_GS_PRO
        for (int t0 = 0; t0 < cnt; t0 += NST) {
#define PG_GS_STEP(U)                                                                                          \
            if (U < NST && t0 + U < cnt) {                                                                     \
                const int t = t0 + U;                                                                          \
                /* unit t is the oldest of those in flight: all but the NST - 2 younger ones have landed */   \
                if (t + NST - 2 < cnt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LPS) : "memory");  \
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                          \
                if (t + NST - 1 < cnt) issue(std::integral_constant<int, (U + NST - 1) % NST>{}, t + NST - 1); \
                __builtin_amdgcn_sched_barrier(0);                                                             \
                consume(std::integral_constant<int, (U < NST ? U : 0)>{});                                     \
                __builtin_amdgcn_sched_barrier(0);                                                             \
            }
            PG_GS_STEP(0) PG_GS_STEP(1) PG_GS_STEP(2) PG_GS_STEP(3) PG_GS_STEP(4) PG_GS_STEP(5)
#undef PG_GS_STEP
        }
    }
    __syncthreads();  // the rings are done with: their space takes the wavefronts' tiles
    float *red = reinterpret_cast<float *>(lds);  // [NW][NS][4][64]
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((wave * NS + c) * 4 + i) * 64 + lane] = acc[c][i];
    __syncthreads();
    for (int e = threadIdx.x; e < NS * 4 * 16; e += 64 * NW) {
        const int r = e & 15, i = (e >> 4) & 3, c = e >> 6;  // c = tile * NQ + token quad
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w)  // ascending runs of K, within a run the four block classes in order
#pragma unroll
            for (int q = 0; q < 4; ++q) sum += red[((w * NS + c) * 4 + i) * 64 + 16 * q + r];
        const int tok = 4 * (c % NQ) + i, row = n0 + 16 * (c / NQ) + r;
        if (tok < m && row < n_out) {
            const float v = QT == 4 ? sum * 0.0625f : sum;  // (Q4_0: the weight operand was 16 * (q - 8))
            y[(size_t)tok * n_out + row] = res ? res[(size_t)tok * n_out + row] + v : v;
        }
    }
}

// ---- 2 and more activation rows over a small product in one launch after the digits, any K -------------------------
// gguf_mm_kernel's 32 x 32 tile with gguf_skinny_kernel's split of K: a workgroup owns 32 weight rows x MT tokens and all of
// K, its NW wavefronts take one run of K each with an LDS ring of their own (no barrier in the loop), and their f32 tiles
// are added through LDS in a fixed order.  Nothing is left for a third launch, and a small tensor has as many wavefronts as its
// blocks can feed.  A unit of the ring is four blocks: the tile-major copy's run of the 32 rows (2 or 4 KiB), their f16 scales,
// the digit planes and block scales of the tokens.  Blocks past the end of K are not added.  UPLOADED: the weights' 16-byte chunks
// come from the planes as uploaded instead, 64 bytes of a row to four lanes, into the same places (see pg_launch_gguf_one_launch).
// More than MT tokens: groups of MT, a weight tile's groups behind each other on one XCD.
// MT = 8, 16: tokens on the accumulator registers (half of MT of them), weight rows on the lanes; MT = 32 the other way
// round, as gguf_mm_kernel.
// Q41 (with QT = 4): Q4_1, whose value q d + m is (q - 8) d + (8 d + m): besides the Q4_0 product every block adds 8 d + m times
// the block's plain sum of x, one FMA more per output; a unit holds the blocks' f16 m and the tokens' block sums too.
// Q4_1's offsets and block sums are arguments of its kernels alone: in everybody's they cost the other formats 0.1 to 0.5 us
// a launch.
template <bool Q41> struct ktile_args : pg_skinny_group {
    void set(const pg_gguf_tensor *const *, int, const pg_mmdigits &) {}
};
template <> struct ktile_args<true> : pg_skinny_group {
    const uint16_t *mo[3];
    const float *xsum;
    void set(const pg_gguf_tensor *const *w, int count, const pg_mmdigits &md) {
        for (int i = 0; i < 3; ++i) mo[i] = i < count ? w[i]->m : nullptr;
        xsum = md.xsum;
    }
};

// Experts' products: tile blockIdx.y of all experts' tiles of MT pairs, 32 rows of one of up to two tensors; pair p reads activation row
// p / div and writes output row p.
struct ktile_experts {
    const uint8_t *const *qs[2];
    const uint16_t *const *d[2];
    float *y[2];
    const int *lists, *counts;
    int list_stride, div, experts, n, wgs1;  // wgs1: 32-row tiles of one tensor
};

template <int QT, int MT, bool Q41> struct KTCfg {
    static constexpr int W_T = QT == 8 ? 4096 : 2048, OFF_D = W_T, OFF_M = OFF_D + 256, OFF_DG = OFF_M + (Q41 ? 256 : 0);
    static constexpr int OFF_X = OFF_DG + MT * 256, OFF_S = OFF_X + MT * 16, UNIT = OFF_S + (Q41 ? MT * 16 : 0);
};
template <int QT, int MT, int NW, bool Q41, typename ARGS = ktile_args<Q41>, bool UPLOADED = false>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 4))) void gguf_ktile_kernel(const int8_t *__restrict__ digits, const float *__restrict__ xs, const ARGS grp,
                                                                int nb, int nbp, int m, int groups, int wgs) {
    using C = KTCfg<QT, MT, Q41>;
    static_assert(!Q41 || QT == 4, "Q4_1 is the Q4_0 product and its offsets");
    constexpr bool EXPERTS = std::is_same_v<ARGS, ktile_experts>;
    int wg = blockIdx.x, t0 = 0, n0, n_out;
    const uint8_t *__restrict__ qs;
    const uint16_t *__restrict__ dsc;
    float *__restrict__ y;
    const float *__restrict__ res = nullptr;
    const int *__restrict__ list = nullptr;  // pairs of this tile's tokens
    int tg = 0;
    if constexpr (EXPERTS) {
        int tile = blockIdx.y;
        const int e = expert_of_tile(grp.counts, grp.experts, MT, threadIdx.x & 63, tile, m);
        if (e < 0) return;  // the same for every thread of the workgroup
        t0 = tile * MT;
        tg = wg >= grp.wgs1;
        qs = grp.qs[tg][e];
        dsc = grp.d[tg][e];
        y = grp.y[tg];
        n_out = grp.n;
        n0 = (wg - tg * grp.wgs1) * 32;
        list = grp.lists + (size_t)e * grp.list_stride + t0;
    } else {
        if (groups > 1) {
            const int j = blockIdx.x >> 3;
            wg = j / groups * 8 + (blockIdx.x & 7);
            t0 = j % groups * MT;
            if (wg >= wgs) return;
        }
#pragma unroll
        for (int i = 1; i < 3; ++i) tg = wg >= grp.wg0[i] ? i : tg;
        qs = grp.qs[tg];
        dsc = grp.d[tg];
        y = grp.y[tg];
        res = grp.res[tg];
        n_out = grp.n[tg];
        n0 = (wg - grp.wg0[tg]) * 32;
    }
    auto row_of = [&](int tok) -> size_t {  // activation row of a token of this tile
        if constexpr (EXPERTS) return (size_t)(list[tok] / grp.div);
        else return (size_t)(t0 + tok);
    };
    extern __shared__ __attribute__((aligned(1024))) char lds[];  // NW rings of two units; afterwards the wavefronts' tiles
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l31 = lane & 31, hh = lane >> 5;
    const int mt = m - t0 < MT ? m - t0 : MT;
    const int units = (nb + 3) / 4, per = (units + NW - 1) / NW;
    const int u_begin = wave * per, u_end = u_begin + per < units ? u_begin + per : units;
    const int cnt = u_end - u_begin;
    char *ring = lds + (size_t)wave * 2 * C::UNIT;

    // fill duties of this lane
    const char *w_src[UPLOADED ? 2 : 1];  // UPLOADED: of fill q's row (lane / 4 of 16, q odd the second 16), else of the tile-major copy
    const int w_jb = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
    for (int i = 0; i < (UPLOADED ? 2 : 1); ++i) {
        const int row = n0 + 16 * i + (lane >> 2);
        w_src[i] = reinterpret_cast<const char *>(qs) +
                   (UPLOADED ? (size_t)(row < n_out ? row : n_out - 1) * (QT == 8 ? 2 : 1) * nb * 16  // (rows past the end: never stored)
                             : (size_t)(n0 >> 7) * pg_tiled_group_bytes(nb, QT == 8) + ((n0 >> 5) & 3) * C::W_T + lane * 16);
    }
    const int ngroups = (n_out + 7) / 8;
    const int dg8 = (n0 >> 3) + (lane >> 4) < ngroups ? (n0 >> 3) + (lane >> 4) : ngroups - 1;
    const size_t d_at = (size_t)dg8 * nb * 16 + (lane & 3) * 4;
    const int d_jb = (lane >> 2) & 3;
    const char *d_src = reinterpret_cast<const char *>(dsc) + d_at;
    const char *m_src = nullptr;
    if constexpr (Q41) m_src = reinterpret_cast<const char *>(grp.mo[tg]) + d_at;
    // digits: fill q covers runs 8 q .. 8 q + 7 of 128 bytes, run = 2 token + plane (tokens 8 .. 15 (mod 16) keep their planes swapped)
    const int8_t *g_src[MT / 4];
    int g_jb[MT / 4];
#pragma unroll
    for (int q = 0; q < MT / 4; ++q) {
        const int run = 8 * q + (lane >> 3), tok = run >> 1, pl = (run & 1) ^ ((tok >> 3) & 1), ch = (lane & 7) ^ (tok & 7);
        g_jb[q] = ch >> 1;
        g_src[q] = digits + row_of(tok < mt ? tok : 0) * pg_mm_row_bytes(nb) + (size_t)pl * nb * 32 + (ch & 1) * 16;
    }
    const size_t x_at = row_of(lane < mt ? lane : 0) * nbp;

    const int rot = cnt > 0 ? (int)((wg * 5u) % (unsigned)cnt) : 0;
    auto issue = [&](auto slot, int t) {
        const int unit = pg_skinny_walk_unit(u_begin, cnt, t, rot), b0 = 4 * unit;
        char *base = ring + decltype(slot)::value * C::UNIT;
        auto blk = [&](int j) { return (size_t)(b0 + j < nb ? b0 + j : nb - 1); };  // past the end: a valid block, never added
#pragma unroll
        for (int q = 0; q < C::W_T / 1024; ++q)
            __builtin_amdgcn_global_load_lds((gptr_t)(UPLOADED ? w_src[q & 1] + (blk(w_jb) + (size_t)(q >> 1) * nb) * 16 : w_src[0] + (size_t)unit * (4 * C::W_T) + q * 1024),
                                             (lptr_t)(base + q * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(d_src + blk(d_jb) * 16), (lptr_t)(base + C::OFF_D), 4, 0, 0);
        if constexpr (Q41) __builtin_amdgcn_global_load_lds((gptr_t)(m_src + blk(d_jb) * 16), (lptr_t)(base + C::OFF_M), 4, 0, 0);
#pragma unroll
        for (int q = 0; q < MT / 4; ++q)
            __builtin_amdgcn_global_load_lds((gptr_t)(g_src[q] + blk(g_jb[q]) * 32), (lptr_t)(base + C::OFF_DG + q * 1024), 16, 0, 0);
        if (lane < MT) {
            __builtin_amdgcn_global_load_lds((gptr_t)(xs + x_at + b0), (lptr_t)(base + C::OFF_X), 16, 0, 0);
            if constexpr (Q41) __builtin_amdgcn_global_load_lds((gptr_t)(grp.xsum + x_at + b0), (lptr_t)(base + C::OFF_S), 16, 0, 0);
        }
    };

    constexpr bool ROWS = MT == 32;      // weight rows on the registers
    constexpr int NR = ROWS ? 16 : MT / 2;
    float acc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = 0.0f;
    const int ws = QT == 8 ? lane : l31, w_rd = ws * 64, w_sw = (ws >> 2) & 3;
    const int tok = l31 & (MT - 1), dig_rd = C::OFF_DG + tok * 256, dig_sw = tok & 7, dig_hi = ((tok >> 3) & 1) * 128;
    auto read = [&](const char *base, int j, v4i (&ab)[3]) {
        ab[0] = *reinterpret_cast<const v4i *>(base + w_rd + ((j ^ w_sw) * 16));
        ab[1] = *reinterpret_cast<const v4i *>(base + dig_rd + dig_hi + (((2 * j + hh) ^ dig_sw) * 16));
        ab[2] = *reinterpret_cast<const v4i *>(base + dig_rd + (128 - dig_hi) + (((2 * j + hh) ^ dig_sw) * 16));
    };
    auto mfmas = [&](const v4i (&ab)[3], v16i &ihi, v16i &ilo) {
        v4i a = ab[0];
        if constexpr (QT == 4) {
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = nibbles_to_i8x16(a[t], 4 - 4 * hh);
        }
        v16i zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0;
        ihi = ROWS ? __builtin_amdgcn_mfma_i32_32x32x32_i8(a, ab[1], zero, 0, 0, 0) : __builtin_amdgcn_mfma_i32_32x32x32_i8(ab[1], a, zero, 0, 0, 0);
        ilo = ROWS ? __builtin_amdgcn_mfma_i32_32x32x32_i8(a, ab[2], zero, 0, 0, 0) : __builtin_amdgcn_mfma_i32_32x32x32_i8(ab[2], a, zero, 0, 0, 0);
    };
    auto quad = [&](const char *base, int off, int (&v)[4]) {  // four ints at once (read as integers: see gguf_mm_kernel)
        const v4i t = *reinterpret_cast<const v4i *>(base + off);
        const int a0 = t[0], a1 = t[1], a2 = t[2], a3 = t[3];
        v[0] = a0; v[1] = a1; v[2] = a2; v[3] = a3;
    };
    auto consume = [&](auto slot, int t) {
        const char *base = ring + decltype(slot)::value * C::UNIT;
        const int left = nb - 4 * pg_skinny_walk_unit(u_begin, cnt, t, rot);
        // the scales (and Q4_1's block sums) of the tokens for the unit's four blocks: of this lane's token, or of its NR tokens
        int sx[ROWS ? 1 : NR][4], sm[Q41 ? (ROWS ? 1 : NR) : 1][4];
#pragma unroll
        for (int r = 0; r < (ROWS ? 1 : NR); ++r) {
            const int at = (ROWS ? l31 : 8 * (r >> 2) + 4 * hh + (r & 3)) * 16;
            quad(base, C::OFF_X + at, sx[r]);
            if constexpr (Q41) quad(base, C::OFF_S + at, sm[r]);
        }
        v4i ab[2][3];
        v16i ihi[2], ilo[2];
        auto scale = [&](int j, const v16i &hi, const v16i &lo) {
            if constexpr (ROWS) {
                const float sj = __int_as_float(sx[0][j]) * (QT == 4 ? 0.0625f : 1.0f);  // (Q4_0: the weight operand was 16 * (q - 8))
#pragma unroll
                for (int g = 0; g < 4; ++g) {  // rows 8 g + 4 hh + {0 .. 3}  <->  registers 4 g .. 4 g + 3
                    const v2i dd = *reinterpret_cast<const v2i *>(base + C::OFF_D + (g * 4 + j) * 16 + hh * 8);
                    v2i mm = {0, 0};
                    if constexpr (Q41) mm = *reinterpret_cast<const v2i *>(base + C::OFF_M + (g * 4 + j) * 16 + hh * 8);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int r = 4 * g + q;
                        const uint32_t bits = (uint32_t)dd[q >> 1];
                        const float dv = half_bits_to_float((q & 1) ? bits >> 16 : bits & 0xFFFFu);
                        const float fx = (float)(hi[r] * 256 + lo[r]) * sj;
                        acc[r] = fmaf(dv, fx, acc[r]);
                        if constexpr (Q41) {
                            const uint32_t mbits = (uint32_t)mm[q >> 1];
                            const float cv = fmaf(8.0f, dv, half_bits_to_float((q & 1) ? mbits >> 16 : mbits & 0xFFFFu));
                            acc[r] = fmaf(cv, __int_as_float(sm[0][j]), acc[r]);
                        }
                    }
                }
            } else {
                const int at = (l31 >> 3) * 64 + j * 16 + (l31 & 7) * 2;
                float dv = half_bits_to_float(*reinterpret_cast<const unsigned short *>(base + C::OFF_D + at)), cv = 0.0f;
                if constexpr (Q41) cv = fmaf(8.0f, dv, half_bits_to_float(*reinterpret_cast<const unsigned short *>(base + C::OFF_M + at)));
                if constexpr (QT == 4) dv *= 0.0625f;
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const float fx = (float)(hi[r] * 256 + lo[r]) * __int_as_float(sx[r][j]);
                    acc[r] = fmaf(dv, fx, acc[r]);
                    if constexpr (Q41) acc[r] = fmaf(cv, __int_as_float(sm[r][j]), acc[r]);
                }
            }
        };
        read(base, 0, ab[0]);
        read(base, 1, ab[1]);
        mfmas(ab[0], ihi[0], ilo[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // while block j is scaled the MFMAs of block j + 1 run and the reads of block j + 2 return
            if (j + 1 < 4) mfmas(ab[(j + 1) & 1], ihi[(j + 1) & 1], ilo[(j + 1) & 1]);
            if (j + 2 < 4) read(base, j + 2, ab[j & 1]);
            __builtin_amdgcn_sched_barrier(0);
            if (j < left) scale(j, ihi[j & 1], ilo[j & 1]);  // (the same for the whole wavefront)
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (cnt > 0) {
        issue(std::integral_constant<int, 0>{}, 0);
        auto step = [&](auto slot, int t) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (t + 1 < cnt) issue(std::integral_constant<int, 1 - decltype(slot)::value>{}, t + 1);
            __builtin_amdgcn_sched_barrier(0);
            consume(slot, t);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int t = 0; t < cnt; t += 2) {
            step(std::integral_constant<int, 0>{}, t);
            if (t + 1 < cnt) step(std::integral_constant<int, 1>{}, t + 1);
        }
    }
    __syncthreads();  // the rings are done with: their space takes the wavefronts' tiles
    float *red = reinterpret_cast<float *>(lds);  // [NW][NR][64], a lane's registers 65 apart
#pragma unroll
    for (int r = 0; r < NR; ++r) red[(wave * NR + r) * 65 + lane] = acc[r];
    __syncthreads();
    for (int e = threadIdx.x; e < NR * 64; e += 64 * NW) {
        // ROWS: consecutive threads take consecutive weight rows of one token; otherwise a register's 64 lanes
        const int r = ROWS ? (e & 3) + 4 * ((e >> 3) & 3) : e >> 6;
        const int l = ROWS ? (e >> 5) + 32 * ((e >> 2) & 1) : e & 63;
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += red[(w * NR + r) * 65 + l];
        const int at = 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);
        const int token = ROWS ? l & 31 : at, row = n0 + (ROWS ? at : l & 31);
        if (token < mt && row < n_out) {
            size_t o = (size_t)(t0 + token) * n_out + row;
            if constexpr (EXPERTS) o = (size_t)list[token] * n_out + row;
            y[o] = res ? res[o] + sum : sum;
        }
    }
}

// y[i] = part[0][i] + part[1][i] + ... in a fixed order.
__global__ void sum_parts_kernel(const float *__restrict__ part, size_t n, int ks, size_t stride, float *__restrict__ y) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float acc = part[i];
    for (int s = 1; s < ks; ++s) acc += part[(size_t)s * stride + i];
    y[i] = acc;
}

}  // namespace

pg_status pg_launch_sum_parts(pg_ctx *ctx, const float *part, size_t n, int ks, size_t stride, float *y) {
    if (n == 0) return PG_OK;
    return pg_launch(ctx, "gguf_mm_sum_parts", sum_parts_kernel, dim3(grid_for(n, 256)), dim3(256), 0, part, n, ks, stride, y);
}

size_t pg_mmdigits_bytes(size_t rows, size_t k) {
    const size_t nb = k / 32, nbp = pg_round_up(nb, 4);
    return rows * pg_mm_row_bytes(nb) + 2 * pg_round_up(rows * nbp * sizeof(float), 256);
}

pg_mmdigits pg_mmdigits_carve(void *base, size_t rows, size_t k) {
    const size_t nb = k / 32;
    pg_mmdigits md;
    char *p = static_cast<char *>(base);
    md.digits = reinterpret_cast<int8_t *>(p);
    p += rows * pg_mm_row_bytes(nb);
    md.xs = reinterpret_cast<float *>(p);
    p += pg_round_up(rows * pg_round_up(nb, 4) * sizeof(float), 256);
    md.xsum = reinterpret_cast<float *>(p);
    md.rows = rows;
    md.k = k;
    return md;
}

pg_status pg_launch_x_to_mm_digits(pg_ctx *ctx, const float *x_dev, size_t rows, size_t k, int ggml_type,
                                   const pg_mmdigits &md) {
    if (rows == 0) return PG_OK;
    if (rows > 65535) return pg_fail(PG_EUNSUPPORTED, "x_to_mm_digits: more than 65535 activation rows");
    const int nb = (int)(k / 32), nbp = (int)pg_round_up(nb, 4);
    const dim3 grid(grid_for(nb, 32), (unsigned)rows);
    if (ggml_type == PG_GGML_Q4_0 || ggml_type == PG_GGML_Q4_1)
        return pg_launch(ctx, "x_to_mm_digits", x_to_mm_digits_kernel<true>, grid, dim3(256), 0, x_dev, nb, nbp, md.digits, md.xs,
                         ggml_type == PG_GGML_Q4_1 ? md.xsum : (float *)nullptr);
    return pg_launch(ctx, "x_to_mm_digits", x_to_mm_digits_kernel<false>, grid, dim3(256), 0, x_dev, nb, nbp, md.digits, md.xs,
                     (float *)nullptr);
}

pg_status pg_launch_block_sums(pg_ctx *ctx, const float *x_dev, size_t rows, size_t k, float *xsum) {
    if (rows > 65535) return pg_fail(PG_EUNSUPPORTED, "gguf_matmul: too many activation rows");
    const int nb = (int)(k / 32);
    return pg_launch(ctx, "gguf_block_sums", block_sums_kernel, dim3((unsigned)((nb + 31) / 32), (unsigned)rows), dim3(256), 0, x_dev, nb,
                     (int)pg_round_up(nb, 4), xsum);
}

pg_status pg_launch_q41_offset(pg_ctx *ctx, const pg_gguf_tensor *w, const float *xsum, size_t rows, const float *part, int ks, float *y) {
    const int nb = (int)(w->k_in / 32), nbp = (int)pg_round_up(nb, 4);
    const size_t stride = rows * w->n_out;
    if (rows > 64) {
        if ((rows + 63) / 64 > 65535) return pg_fail(PG_EUNSUPPORTED, "gguf_matmul: too many activation rows");
        // Few tiles and steps enough to share out; the more tiles there are, the more steps it takes, since what four runs of a tile add is
        // their sums' way through LDS and four times the reads of the rows' sums.  Both timed on 2900 products: to 128 workgroups (half
        // the CUs) from 4 steps on 0.95 of the time and less, to 192 from 5 on none longer (4: 1.04), beyond, at 4 to 6 steps 1.07 to 1.12, at 9 to 16 about
        // even, from 17 on 0.97 and less, past 384 no rule.  us of the whole product, side by side : RUNS, 70 x 9760 -> 2282 (36 workgroups, 39 steps)
        // 61.8 : 38.5, 129 x 14336 -> 4096 (96, 56) 100.5 : 78.8, 514 x 7040 -> 1330 (99, 28) 73.3 : 62.2, 256 x 4096 -> 4096 (128, 16) 47.4 : 41.1,
        // 1008 x 1216 -> 972 (128, 5) 28.3 : 27.0, 1024 x 14336 -> 3072 (384, 56) 293 : 286; but 171 x 960 -> 13241 (312, 4) 37.0 : 41.3, 413 x 1184 ->
        // 5268 (294, 5) 37.0 : 40.0, 512 x 4096 -> 8192 (512, 16) 118.7 : 119.8, 1000 x 4096 -> 14336 (1792, 16) 297 : 304, and of two steps 200 x 512 ->
        // 14336 (448) 25.8 : 29.4.
        const size_t wgs = (size_t)grid_for(w->n_out, 128) * ((rows + 63) / 64), cus = (size_t)ctx->num_cu;
        const bool runs = 2 * wgs <= cus ? nb > 24 : 4 * wgs <= 3 * cus ? nb > 32 : 2 * wgs <= 3 * cus && nb > 128;
        return pg_launch(ctx, "gguf_q4_1_offsets", runs ? q41_offset_mfma_kernel<true> : q41_offset_mfma_kernel<false>,
                         dim3(grid_for(w->n_out, runs ? 32 : 128), (unsigned)((rows + 63) / 64)), dim3(256), 0,
                         (const uint16_t *)w->d, (const uint16_t *)w->m, (int)w->n_out, nb, xsum, nbp, (int)rows, part, ks, stride, y);
    }
    const size_t lds = ((size_t)nb * Q41_TT + 256 * (Q41_TT + 1)) * sizeof(float);
    if (lds > 128 * 1024) return pg_fail(PG_EUNSUPPORTED, "gguf_matmul: Q4_1 rows of %zu on the matrix-core route", w->k_in);
    PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)q41_offset_kernel, 128 * 1024));
    return pg_launch(ctx, "gguf_q4_1_offsets", q41_offset_kernel, dim3(grid_for(w->n_out, 256 / Q41_NQ), (unsigned)((rows + Q41_TT - 1) / Q41_TT)), dim3(256), lds,
                     (const uint16_t *)w->d, (const uint16_t *)w->m, (int)w->n_out, nb, xsum, nbp, (int)rows, part, ks, stride, y);
}

// Digits of `act_rows` activation rows that no XCD's L2 (4 MiB) can keep while every workgroup
// of a token tile reads them: then K is split so that a chunk's share does fit, and the chunks
// are dealt to XCDs (see the kernel).  Without the split a K = 32768 product over 128 rows
// fetches its 8 MiB of digits once per 128-row group: 1.2x the weight bytes in total.
static bool digits_exceed_l2(size_t act_rows, size_t nb) { return act_rows * pg_mm_row_bytes(nb) > (2u << 20); }

int pg_gguf_mm_splitk(const pg_ctx *ctx, size_t n_out, size_t k_in, size_t groups, size_t act_rows, bool grouped,
                      int *chunk_out, bool *xcd_chunks) {
    const size_t nb = k_in / 32;
    const size_t wgs = ((n_out + 127) / 128) * (groups ? groups : 1);
    // A short K is split only as far as every workgroup is still resident at once: a second round of
    // workgroups would pay the start-up latency again.  (Three workgroups fit on a CU; splitting for
    // three a CU instead of two measured the same on the 16-row product, with more partial planes to sum.)
    const size_t slots = 2 * (size_t)ctx->num_cu;
    size_t ks = slots / wgs;
    if (ks > 8) ks = 8;
    if (ks < 1) ks = 1;
    bool by_xcd = false;
    // (Plain products over 16 token tiles and more are not split: they run as super-tiles.)
    if ((grouped || groups < 16) && digits_exceed_l2(act_rows, nb)) {
        size_t c = 2;
        while (c < 8 && act_rows * pg_mm_row_bytes(nb) > c * (size_t)(2u << 20)) c *= 2;
        // worth it while the partial sums (written and read back) stay under a tenth of the weights
        const bool cheap = c * act_rows * 8 * 10 <= nb * 34 * (grouped ? groups : 1);  // per weight row
        if (c >= ks && nb / c >= 8 * NBU && cheap) {
            ks = c;
            by_xcd = true;
        }
    }
    size_t chunk = pg_round_up((nb + ks - 1) / ks, NBU);
    if (chunk < 2 * NBU) chunk = 2 * NBU;
    const size_t ks_real = (nb + chunk - 1) / chunk;
    if (ks_real != ks) by_xcd = false;  // the deal needs 2, 4 or 8 chunks exactly
    if (chunk_out) *chunk_out = (int)chunk;
    if (xcd_chunks) *xcd_chunks = by_xcd;
    return (int)ks_real;
}

// Rows up to which a product leaves its tensor without a tile-major copy.
static size_t few_rows_of(const pg_ctx *ctx, size_t n_out) { return n_out < 32 * (size_t)ctx->num_cu ? 16 : 8; }

// Up to 8 rows over a Q4_0 or Q8_0 tensor whose K is a multiple of 256: gguf_skinny_kernel, bound by how many bytes its rings keep
// in flight (4 x 4096 -> 14336 takes 9.0 us; with its arithmetic switched off 8.6 - 9.1).  From five rows on it is the better one
// only where a long K meets few columns (us, this one : gguf_ktile_kernel: 7 x 11776 -> 1804 12.7 : 14.8, 8 x 8704 -> 406 10.7 :
// 12.3; but 6 x 6144 -> 4297 14.1 : 10.5, 8 x 1536 -> 12190 11.5 : 8.1, 7 x 3584 -> 870 10.1 : 8.5), and of Q8_0 over a vocabulary
// (6 x 8192 -> 32768 54.5 : 72.4 from the planes as uploaded, 49.2 : 59.7 from the copy; 5 x 4096 -> 128256 104 : 116 and 99.6 : 98.9).
static bool skinny_takes(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_out, size_t k_in) {
    const size_t cus = (size_t)ctx->num_cu;
    const bool few_columns = k_in >= 6400 && n_out < 16 * cus, vocabulary = ggml_type == PG_GGML_Q8_0 && n_out > 64 * cus && m * n_out * k_in > 1400000000;
    return (ggml_type == PG_GGML_Q4_0 || ggml_type == PG_GGML_Q8_0) && m >= 2 && (m <= 4 || (m <= 8 && (few_columns || vocabulary))) &&
           k_in % 256 == 0 && k_in >= 1024 && n_out >= 1 && n_out < (1u << 30) && k_in < (1u << 24);
}

// Products small enough that digits, K chunks and their sum are three latencies: gguf_ktile_kernel.  Against that route (m 2 .. 400,
// K 256 .. 14336, N 256 .. 14336, 1450 products) it takes 0.6 to 0.8 of the time up to half a G multiply-adds, is level at 1.5 (more than
// 64 rows: 1; Q4_1 1.8 to 700 rows and 1 beyond, from 245 products of 66 to 1800 rows: 0.5 % over the better route on average, 18 % at most) and slower beyond, where a tile of 128 weight rows shares a token's digits; so it is with a long K, or a short one
// under many columns, over more than two row tiles (71 x 4896 -> 2614 24 : 31, 67 x 512 -> 13720 11.5 : 17).  Q4_1 up to 64 rows: the offsets' launch goes too (0.6 to 0.9 up to 5 G).  us, before : now:
// 35 x 1088 -> 465 (Q8_0) 12.4 : 7.6, 12 x 4096 -> 4096 (Q4_1) 9.9 : 8.0, 11 x 1056 -> 2116 (Q8_0) 11.5 : 7.6, 32 x 4096 -> 1024
// (Q4_0) 13.7 : 9.2, 64 x 4096 -> 4096 (Q4_1) 28.5 : 22.
// What the f16 matrix cores hold stays there, and Q4_1 below eight rows with the streaming kernel: both have finer digits.  (What they would take by their time
// alone does not: of 101 products within these lines none is faster there by more than 3 %.)
static bool ktile_takes(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_out, size_t k_in, bool planes) {
    const bool q41 = ggml_type == PG_GGML_Q4_1;
    if (!(ggml_type == PG_GGML_Q4_0 || ggml_type == PG_GGML_Q8_0 || q41) || m < (q41 ? 8 : 2) || k_in % 32 != 0 || k_in > 32768 || n_out < 1 || n_out >= (1u << 24))
        return false;
    // Up to eight rows, up to sixteen of fewer than 8192 columns: always, so that no product of so few rows needs the tile-major copy
    // (launch_ktile).  us over weights with a copy, gguf_mm_kernel : this: Q4_0 8 x 4096 -> 50257 36.7 : 32.9, 16 x 14336 -> 8000
    // 27.8 : 25.2, Q8_0 7 x 14336 -> 14336 45.1 : 45.1, 16 x 14336 -> 8000 32.2 : 32.6, the worst 8 x 14336 -> 12600 42.8 : 45.0.
    if (m <= few_rows_of(ctx, n_out) && k_in % 256 == 0 && k_in >= 1024) return true;
    const double g = 1e-9 * (double)m * (double)n_out * (double)k_in * (planes ? 1.5 : 1.0);
    if (k_in < 512 && n_out > 8192) return false;                                        // (all columns, hardly any K to split)
    if (m > 64 && (k_in >= (q41 ? 8192 : 6144) || (k_in < 1024 && m * n_out > 500000))) return false;
    if (g > (q41 ? (m <= 64 ? 5.0 : m <= 700 ? 1.8 : 1.0) : m <= 64 ? 1.4 : m <= 128 ? 0.9 : 0.7)) return false;
    return m <= 16 || !pg_gguf_hmm_holds(ctx, q41 ? PG_GGML_Q4_0 : ggml_type, m, n_out, k_in);
}

// Whether a product runs as one launch after the digits.  `planes`: the caller takes the K chunks of the other route unsummed, so that
// there is no launch for their sum to be saved and the lines lie at two thirds (the Llama block's steps of 10 to 180 tokens over four
// models: at 1 / 1.5 / 3 of the lines 0 to 1 % slower / best / 1 to 3 % slower; without this kernel 3 to 15 %.  us, before : now:
// 7 tokens of 1024 47 : 41, 30 of 2048 77 : 69, 45 of 2048 / 5632 93 : 76, 20 of 4096 115 : 102, 180 of 4096 322 : 301).
bool pg_gguf_one_launch_takes(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_out, size_t k_in, bool planes) {
    return skinny_takes(ctx, ggml_type, m, n_out, k_in) || ktile_takes(ctx, ggml_type, m, n_out, k_in, planes);
}

static pg_status launch_skinny(pg_ctx *ctx, size_t k_in, bool q8, const pg_skinny_group &grp, int wgs, int tiles, size_t m, const pg_mmdigits &md) {
    const int nb = (int)(k_in / 32), nbp = (int)pg_round_up(nb, 4);
    // Wavefronts (runs of K) per workgroup: as many as keep every workgroup resident at once, up to 16 a CU (4 a SIMD).  The rings: units
    // of 4.75 / 6.75 KiB for 4 / 8 token rows (Q8_0: 2 KiB more), two stages (three on fewer wavefronts: 10.7 - 10.9 against 9.0 us on
    // 4 x 4096 -> 14336).
    const size_t unit_bytes = (size_t)tiles * ((q8 ? 4096 : 2048) + 256) + (m <= 4 ? 4 : 8) * 512 + 512, units = (size_t)nb / 8;
    auto fits = [&](int nw_) {  // LDS is handed out per workgroup: nw wavefronts' rings each
        const size_t per_cu = std::min<size_t>((160u << 10) / ((size_t)nw_ * 2 * unit_bytes), 16 / nw_);
        return (size_t)wgs <= (size_t)ctx->num_cu * per_cu;
    };
    int nw = 8;
    while (nw > 1 && (!fits(nw) || units / nw < 4)) nw >>= 1;
#define PG_GSK(QTT, NBB, MTT, NWW)                                                                                             \
    if (q8 == (QTT == 8) && tiles == NBB && (m <= 4) == (MTT == 4) && nw == NWW) {                                             \
        auto kern = gguf_skinny_kernel<QTT, NBB, MTT, NWW, 2>;                                                                 \
        const size_t lds = (size_t)NWW * 2 * (NBB * ((QTT == 8 ? 4096 : 2048) + 256) + MTT * 512 + 512);                       \
        PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));                                                            \
        return pg_launch(ctx, QTT == 8 ? "gguf_q8_0_few_rows_mm" : "gguf_q4_0_few_rows_mm", kern, dim3((unsigned)wgs), dim3(64 * NWW), lds, \
                         (const int8_t *)md.digits, (const float *)md.xs, grp, nb, nbp, (int)m);                               \
    }
#define PG_GSK_NW(QTT, NBB, MTT) PG_GSK(QTT, NBB, MTT, 8) PG_GSK(QTT, NBB, MTT, 4) PG_GSK(QTT, NBB, MTT, 2) PG_GSK(QTT, NBB, MTT, 1)
    PG_GSK_NW(8, 1, 4) PG_GSK_NW(8, 2, 4) PG_GSK_NW(8, 1, 8) PG_GSK_NW(8, 2, 8)
    PG_GSK_NW(4, 1, 4) PG_GSK_NW(4, 2, 4) PG_GSK_NW(4, 1, 8) PG_GSK_NW(4, 2, 8)
#undef PG_GSK_NW
#undef PG_GSK
    return pg_fail(PG_EUNSUPPORTED, "gguf (few rows in one launch): no kernel of %d tiles, %d wavefronts", tiles, nw);
}

// The shape of a ktile launch: of the tokens a workgroup takes (MT) and its wavefronts (NW) the pair of least estimated time.  Rounds of
// workgroups (a CU's LDS over their rings), a wavefront's run of units, and what the fullest CU loads; Q4_1's further FMAs a unit.  Fitted
// to 1341 products within the lines above: 1 to 2 % over the best of the shapes on average.  (Tokens in groups of 8 or 16 while
// there are few: the digits of 32 are most of a ring and leave six wavefronts a CU.)
struct ktile_shape { int mt, nw; double factor; };
static constexpr ktile_shape KTILE_SHAPES[] = {{32, 2, 1.26}, {32, 3, 1.2}, {32, 6, 1.14}, {16, 4, 1.06}, {16, 8, 1.03}, {8, 4, 1.014}, {8, 8, 1.0}};
static size_t ktile_unit(int ggml_type, int mt) {
    return ggml_type == PG_GGML_Q8_0 ? (mt == 32 ? KTCfg<8, 32, false>::UNIT : mt == 16 ? KTCfg<8, 16, false>::UNIT : KTCfg<8, 8, false>::UNIT)
         : ggml_type == PG_GGML_Q4_1 ? (mt == 32 ? KTCfg<4, 32, true>::UNIT : mt == 16 ? KTCfg<4, 16, true>::UNIT : KTCfg<4, 8, true>::UNIT)
                                     : (mt == 32 ? KTCfg<4, 32, false>::UNIT : mt == 16 ? KTCfg<4, 16, false>::UNIT : KTCfg<4, 8, false>::UNIT);
}
static pg_status launch_ktile(pg_ctx *ctx, int ggml_type, size_t k_in, const pg_gguf_tensor *const *w, int count, const pg_skinny_group &grp, int wgs1,
                              size_t m, const pg_mmdigits &md, bool uploaded) {
    const int nb = (int)(k_in / 32), nbp = (int)pg_round_up(nb, 4);
    const bool q8 = ggml_type == PG_GGML_Q8_0, q41 = ggml_type == PG_GGML_Q4_1;
    const size_t units = ((size_t)nb + 3) / 4, cus = (size_t)ctx->num_cu;
    ktile_shape sh = KTILE_SHAPES[0];
    double best = 1e30;
    for (const ktile_shape &s : KTILE_SHAPES) {
        if ((s.mt == 8 && m > 32) || (s.mt == 16 && m > 64)) continue;
        const size_t unit = ktile_unit(ggml_type, s.mt), wgs = (size_t)wgs1 * ((m + s.mt - 1) / s.mt);
        const size_t per_cu = std::max<size_t>(1, std::min<size_t>((160u << 10) / ((size_t)s.nw * 2 * unit), (s.mt == 32 ? 8 : 16) / s.nw));
        const double rounds = (double)((wgs + cus * per_cu - 1) / (cus * per_cu)), run = (double)((units + s.nw - 1) / s.nw);
        const double cu_units = (double)((wgs + cus - 1) / cus * units);
        const double us = s.factor * (4.58 + 7.06e-6 * (double)(m * k_in) + rounds * (1.51 + 0.325 * run) + cu_units * (10.1e-6 * (double)unit + (q41 ? 0.042 : 0.0)));
        if (us < best) {
            best = us;
            sh = s;
        }
    }
    const int groups = (int)((m + sh.mt - 1) / sh.mt);
    const dim3 grid(groups == 1 ? (unsigned)wgs1 : (unsigned)((wgs1 + 7) / 8 * 8 * groups));
#define PG_KT(QTT, MTT, NWW)                                                                                                   \
    if ((QTT == 8 ? q8 : QTT == 5 ? q41 : !q8 && !q41) && sh.mt == MTT && sh.nw == NWW) {  /* (5 names Q4_1 here) */           \
        auto kern = uploaded ? gguf_ktile_kernel<QTT == 8 ? 8 : 4, MTT, NWW, QTT == 5, ktile_args<QTT == 5>, true>              \
                             : gguf_ktile_kernel<QTT == 8 ? 8 : 4, MTT, NWW, QTT == 5>;                                        \
        ktile_args<QTT == 5> args;                                                                                             \
        static_cast<pg_skinny_group &>(args) = grp;                                                                            \
        args.set(w, count, md);                                                                                                \
        const size_t lds = (size_t)NWW * 2 * KTCfg<QTT == 8 ? 8 : 4, MTT, QTT == 5>::UNIT;                                     \
        PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));                                                            \
        return pg_launch(ctx, QTT == 8 ? "gguf_q8_0_rows_tile" : QTT == 5 ? "gguf_q4_1_rows_tile" : "gguf_q4_0_rows_tile", kern, grid, \
                         dim3(64 * NWW), lds, (const int8_t *)md.digits, (const float *)md.xs, args, nb, nbp, (int)m, groups, wgs1); \
    }
#define PG_KTS(QTT) PG_KT(QTT, 32, 2) PG_KT(QTT, 32, 3) PG_KT(QTT, 32, 6) PG_KT(QTT, 16, 4) PG_KT(QTT, 16, 8) PG_KT(QTT, 8, 4) PG_KT(QTT, 8, 8)
    PG_KTS(8) PG_KTS(4) PG_KTS(5)
#undef PG_KTS
#undef PG_KT
    return pg_fail(PG_EUNSUPPORTED, "gguf (rows in tiles, one launch): no kernel of %d tokens, %d wavefronts", sh.mt, sh.nw);
}

// The experts' products of a MoE layer as tiles of 8 or 16 tokens of gguf_ktile_kernel (*mt tokens, *nw wavefronts a workgroup) where the two
// together are estimated below 0.93 of gguf_mm_kernel's: little work, whose K chunks, tail tiles and planes to be added are what costs
// there.  Both estimates count the expected tiles and the weights read; terms: rounds of workgroups, a wavefront's (here) or workgroup's
// (there) walk of K, what the fullest CU loads, its tokens' share of the arithmetic, and there the planes.  Fitted to 890 layers (2 to
// 256 tokens, 4 to 16 experts, 512 to 3072 x 1024 to 16384): 6 % mean error of each.  8.5 % less time over all of them (the best choice
// each time: 10 %), 13 to 20 % up to 16 tokens; the worst picks 3 to 4 % over.  us, before : now: 4 tokens, 2 of 8 experts of 2048 x 4096
// (Q8_0) 44.3 : 35.4, 26, 2 of 4 of 1568 x 1696 34.7 : 31.9.
bool pg_gguf_experts_tiles(const pg_ctx *ctx, int ggml_type, size_t T, size_t E, size_t top_k, size_t d, size_t ffn, int *mt, int *nw) {
    const size_t P = T * top_k, n_of[2] = {2 * ffn, d}, k_of[2] = {d, ffn};
    if (d > 32768 || ffn > 32768 || P > 65535) return false;
    const bool q8 = ggml_type == PG_GGML_Q8_0;
    const double cus = (double)ctx->num_cu, per_expert = (double)P / (double)E;
    const double weights = pg_moe_expected_tiles(T, E, top_k, (int)T) * 3.0 * (double)(d * ffn) * (q8 ? 34.0 / 32 : 18.0 / 32);
    const double common = 17.2 + 13.2e-6 * (double)P * (double)(d + ffn) + 0.066e-6 * weights;
    auto half = [](double v) { return v < 1.0 ? 1.0 : 0.5 * (v + ceil(v)); };  // (the last round is rarely full)
    const double heavy = per_expert > 16.0 ? 2.0 : 1.0 + 0.5 * (1.0 + erf((per_expert - 14.0) / 5.0));
    double there = common;
    for (int i = 0; i < 2; ++i) {
        int chunk = 0;
        const int ks = pg_gguf_mm_splitk(ctx, i ? d : pg_mm_pair_rows(ffn), k_of[i], E, i ? P : T, true, &chunk);
        const double wgs = pg_moe_expected_tiles(T, E, top_k, 32) * (double)((n_of[i] + 127) / 128 * ks), cu = std::max(1.0, wgs / cus);
        const double stages = (double)((std::min<size_t>(chunk, k_of[i] / 32) + 3) / 4);
        there += half(wgs / (3.0 * cus)) * (3.29 + 0.502 * stages) + cu * stages * ((q8 ? 0.0927 : 0.0463) + 0.0587 * heavy);
        if (ks > 1) there += 0.78e-6 * (double)ks * (double)P * (double)n_of[i];
    }
    static constexpr ktile_shape SHAPES[] = {{8, 4, 1.32}, {16, 4, 1.27}};
    double best = 1e300;
    for (const ktile_shape &s : SHAPES) {
        const size_t unit = ktile_unit(ggml_type, s.mt);
        const double per_cu = (double)std::max<size_t>(1, std::min<size_t>((160u << 10) / ((size_t)s.nw * 2 * unit), 16 / s.nw));
        double us = common + 0.005e-6 * weights;
        for (int i = 0; i < 2; ++i) {
            const size_t units = (k_of[i] / 32 + 3) / 4;
            const double wgs = pg_moe_expected_tiles(T, E, top_k, s.mt) * (double)((n_of[i] + 31) / 32);
            us += s.factor * (half(wgs / (cus * per_cu)) * (0.7 + 0.302 * (double)((units + s.nw - 1) / s.nw)) +
                              half(wgs / cus) * (double)units * (3.53e-6 * (double)unit + 0.00187 * s.mt));
        }
        if (us < best) {
            best = us;
            *mt = s.mt;
            *nw = s.nw;
        }
    }
    return best < 0.93 * there;
}

pg_status pg_launch_gguf_experts_tiles(pg_ctx *ctx, int ggml_type, size_t n_out, size_t k_in, const pg_mm_group &grp, size_t P, int mt, int nw,
                                       const pg_mmdigits &md, float *y) {
    const int nb = (int)(k_in / 32), nbp = (int)pg_round_up(nb, 4), tensors = grp.nseg < 0 ? 2 : 1;
    const bool q8 = ggml_type == PG_GGML_Q8_0, two = tensors == 2;
    const ktile_experts ex = {{grp.qs_table, two ? grp.qs_table2 : nullptr}, {grp.d_table, two ? grp.d_table2 : nullptr}, {y, two ? grp.out2 : nullptr},
                              grp.lists, grp.counts, grp.list_stride, grp.x_row_div, grp.num_experts, (int)n_out, (int)((n_out + 31) / 32)};
    const size_t gy = expert_tiles_bound(grp.num_experts, grp.list_stride, P, mt);
    if (!grp.counts || !grp.tiled || gy > 65535) return pg_fail(PG_EINVAL, "gguf experts (tiles): %zu token tiles", gy);
    const dim3 grid((unsigned)(ex.wgs1 * tensors), (unsigned)gy);
#define PG_KE(QTT, MTT, NWW)                                                                                                   \
    if (q8 == (QTT == 8) && mt == MTT && nw == NWW) {                                                                          \
        auto kern = gguf_ktile_kernel<QTT, MTT, NWW, false, ktile_experts>;                                                    \
        const size_t lds = (size_t)NWW * 2 * KTCfg<QTT, MTT, false>::UNIT;                                                     \
        PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));                                                            \
        return pg_launch(ctx, QTT == 8 ? "gguf_q8_0_experts_tile" : "gguf_q4_0_experts_tile", kern, grid, dim3(64 * NWW), lds, \
                         (const int8_t *)md.digits, (const float *)md.xs, ex, nb, nbp, 0, 1, 0);                               \
    }
#define PG_KES(QTT) PG_KE(QTT, 8, 4) PG_KE(QTT, 16, 4)
    PG_KES(8) PG_KES(4)
#undef PG_KES
#undef PG_KE
    return pg_fail(PG_EUNSUPPORTED, "gguf experts (tiles): no kernel of %d tokens, %d wavefronts", mt, nw);
}

pg_status pg_launch_gguf_one_launch(pg_ctx *ctx, int ggml_type, size_t k_in, const pg_gguf_tensor *const *w, float *const *y, int count,
                                    size_t m, const pg_mmdigits &md, const float *residual) {
    if (count < 1 || count > 3) return pg_fail(PG_EINVAL, "gguf (few rows in one launch): %d tensors (1 .. 3)", count);
    size_t n_total = 0;
    for (int i = 0; i < count; ++i) {
        if (w[i]->k_in != k_in || w[i]->ggml_type != ggml_type) return pg_fail(PG_EINVAL, "gguf (few rows in one launch): the tensors differ in K or type");
        n_total += w[i]->n_out;
    }
    const bool skinny = skinny_takes(ctx, ggml_type, m, n_total, k_in);
    if (!skinny && !ktile_takes(ctx, ggml_type, m, n_total, k_in, false)) return pg_fail(PG_EINVAL, "gguf (few rows in one launch): [%zu x %zu] x %zu", m, k_in, n_total);
    // Two 16-row weight tiles a workgroup of the skinny kernel where that still leaves a workgroup for every CU: the digits, which
    // every workgroup fetches for all of K, then cost half as much per weight byte.
    const int tiles = n_total / 32 >= (size_t)ctx->num_cu ? 2 : 1, rows = skinny ? 16 * tiles : 32;
    // The planes as uploaded, or everybody's tile-major copy where all have one: the same values in the same order, so the same bits.
    // Up to eight rows, up to sixteen of fewer than 8192 columns, do not make the copy (as many bytes as the tensor again, a wait, and a
    // refusal under a capture; without it 180 products took 2 % longer on average, the worst a third: Q8_0 13 x 11168 -> 3856 19.8 : 26.4).
    bool uploaded = skinny;
    for (int i = 0; i < count && !skinny; ++i) {
        if (m > few_rows_of(ctx, n_total)) PG_TRY(pg_gguf_ensure_tiled(ctx, w[i]));
        uploaded = uploaded || !pg_gguf_tiled(w[i]);
    }
    pg_skinny_group grp;
    int wgs = 0;
    for (int i = 0; i < 3; ++i) {
        const bool used = i < count;
        grp.qs[i] = !used ? nullptr : uploaded ? w[i]->qs : w[i]->qs_tiled;
        grp.d[i] = used ? w[i]->d : nullptr;
        grp.y[i] = used ? y[i] : nullptr;
        grp.res[i] = i == 0 ? residual : nullptr;
        grp.n[i] = used ? (int)w[i]->n_out : 0;
        grp.wg0[i] = used ? wgs : INT_MAX;
        if (used) wgs += (int)((w[i]->n_out + rows - 1) / rows);
    }
    return skinny ? launch_skinny(ctx, k_in, ggml_type == PG_GGML_Q8_0, grp, wgs, tiles, m, md) : launch_ktile(ctx, ggml_type, k_in, w, count, grp, wgs, m, md, uploaded);
}

pg_status pg_launch_gguf_mm(pg_ctx *ctx, int ggml_type, size_t n_out, size_t k_in, const uint8_t *qs,
                            const uint16_t *d, const pg_mm_group &grp, size_t total_pairs, const pg_mmdigits &md,
                            float *y, float *part, bool keep_parts) {
    if (total_pairs == 0) return PG_OK;
    const int nb = (int)(k_in / 32), nbp = (int)pg_round_up(nb, 4);
    const size_t experts = grp.counts ? (size_t)grp.num_experts : 1;
    int chunk = 0;
    size_t gy = experts * (size_t)grp.tiles_per_expert;
    // token tiles that certainly hold work: all of them without expert lists, one per expert with
    bool by_xcd = false;
    const bool second = grp.nseg < 0;
    if (second && (!grp.counts || !keep_parts)) return pg_fail(PG_EINVAL, "gguf_mm: a second tensor per expert needs expert lists and leaves its K chunks unsummed");
    const int ks = pg_gguf_mm_splitk(ctx, second ? pg_mm_pair_rows(n_out) : n_out, k_in, grp.counts ? experts : gy, md.rows, grp.counts != nullptr, &chunk, &by_xcd);
    if (ks > 1 && !part) return pg_fail(PG_EINVAL, "gguf_mm: split-K needs a partial-sum buffer");
    if (grp.nseg > 0 && ((ks > 1 && !keep_parts) || grp.counts || !grp.tiled))
        return pg_fail(PG_EINVAL, "gguf_mm: several tensors in one launch leave their K chunks unsummed, take no expert lists and read tile-major copies");
    if (gy > 65535) return pg_fail(PG_EUNSUPPORTED, "gguf_mm: too many token tiles");
    if (grp.counts) gy = expert_tiles_bound(experts, grp.list_stride, total_pairs, 32);
    dim3 grid(grid_for(n_out, 128) * (second ? 2 : 1), (unsigned)gy, (unsigned)ks);
    pg_mm_group g2 = grp;
    g2.remap_rg = g2.remap_tiles = 0;
    if (!grp.counts && ks == 1 && gy >= 16) {  // a plain product over many token tiles: see the kernel
        g2.remap_rg = (int)grid.x;
        g2.remap_tiles = (int)gy;
        const size_t supertiles = (size_t)((grid.x + 3) / 4) * ((gy + 7) / 8);
        grid = dim3((unsigned)((supertiles + 7) / 8 * 8 * 32), 1, 1);
    }
    g2.xcd_ks = 0;
    if (by_xcd) {
        g2.xcd_ks = ks;
        g2.remap_rg = (int)grid.x;
        g2.remap_tiles = (int)gy;
        const size_t per = 8 / (size_t)ks, tiles = (size_t)grid.x * gy;
        grid = dim3((unsigned)((tiles + per - 1) / per * 8), 1, 1);
    }
    float *dst = ks > 1 ? part : y;
    const size_t stride = total_pairs * n_out;
    const size_t lds = ggml_type == PG_GGML_Q4_0 ? (size_t)MMCfg<4>::RING * MMCfg<4>::STAGE : (size_t)MMCfg<8>::RING * MMCfg<8>::STAGE;
    auto launch = [&](auto kern, const char *name) -> pg_status {
        PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));
        return pg_launch(ctx, name, kern, grid, dim3(256), lds, qs, d, g2, (int)n_out, nb, nbp, chunk, md.digits, md.xs, dst,
                         stride);
    };
    const bool nt = grp.counts != nullptr;
    if (ggml_type == PG_GGML_Q4_0) PG_TRY(nt ? launch(gguf_mm_kernel<4, true>, "gguf_mm_q4_0") : launch(gguf_mm_kernel<4, false>, "gguf_mm_q4_0"));
    else PG_TRY(nt ? launch(gguf_mm_kernel<8, true>, "gguf_mm_q8_0") : launch(gguf_mm_kernel<8, false>, "gguf_mm_q8_0"));
    if (ks > 1 && !keep_parts)
        PG_TRY(pg_launch(ctx, "gguf_mm_sum_parts", sum_parts_kernel, dim3(grid_for(stride, 256)), dim3(256), 0, part, stride, ks,
                         stride, y));
    return PG_OK;
}
