// Many-row product over Q4_0 / Q8_0 block weights on the f16 matrix cores:
//   y[t, n] = sum_b d[n, b] * sum_{k in block b} q[n, k] * x[t, k]
// (the M >> 1 dequant-matmul of models::llama, src/models/llama/model.rs:243-257 +
// src/tensor.rs:1342-1353: dequantise the weight, then Tensor::matmul).
//
// The weights stay exact: a Q4_0 quant q - 8 in [-8, 7] (a Q8_0 quant in [-127, 127]) is an
// f16 value, made in registers from the packed bytes, and a GGUF block is 32 consecutive k,
// exactly the K of one v_mfma_f32_16x16x32_f16.  The activation rows are split once into two
// f16 planes, x * 2^e = hi + lo (e per row, so that the row's largest magnitude lands in
// [2^14, 2^15): hi carries 11 bits, lo the next 11, what is dropped is below 2^-22 of the
// row's maximum).  Per block and 16x16 tile two chained MFMAs give T = (hi + lo) . q, products
// of f16 values summed in f32, and the accumulator takes acc += d[n, b] * T in f32: one VALU
// FMA per output and block where the int8 block product (pg_gguf_mm.hip) needs four
// instructions, which is what bounds that kernel at many rows.
//
// Workgroup = 8 wavefronts over 16 MT rows x 512 weight rows side by side (64 each), MT = 4 .. 8, or (S = 2) four and four over
// 256.  K runs in stages of two blocks through LDS stages filled by direct global->LDS loads: the two activation planes
// [rows][128 B] (16-byte chunks XOR swizzled as in the W8A8 kernel), the weights' packed bytes [weight rows][2 blocks] and
// their f16 scales.  One barrier per stage.  Inside a stage the wavefront walks the row tiles of its blocks; at every
// step it issues loads of a stage to come, 8 MFMAs (4 weight tiles x hi, lo) into one of two sets of T registers,
// and between them the 16 FMAs that fold the previous step's T into the accumulators, so neither unit waits for the
// other.  The next block's weights are unpacked under a block's MFMAs.
//
// S = 1: a wavefront takes both blocks of a stage, and LDS holds two stages.  S = 2: a stage's first block is the first four
// wavefronts', its second the others', who add their sums up through LDS at the end; LDS holds three stages, so that the
// next block's weights have landed while this one multiplies.  A tile of half the width is half as long a walk, so where
// tiles are few K is cut into half as many chunks between workgroups, or none, and that many planes fewer go through
// memory; it brings the activations to LDS twice as often, which is why some wide launches keep S = 1.  us, S = 1 : S = 2,
// the kernel + the sum of its chunks: 100 x 4096 -> 28672 (Q4_0) 61.3 + 13.7 : 58.5 + 7.9, 250 x 2048 -> 16384 (Q8_0)
// 48.6 + 11.3 : 44.5, 500 x 2048 -> 11264 59.3 + 14.3 : 57.7, as long either way 777 x 14336 -> 4096 (Q8_0) 176 + 15.9 : 184 + 8.7 (S = 2 is
// taken); S = 1 is kept by 777 x 4096 -> 28672 (Q8_0) 367 : 401, 1024 x 4096 -> 28672 (Q4_0) 418 : 458, 300 x 4096 -> 28672 (Q4_0) 143 : 165.
//
// What bounds it: 1024 rows of 4096 -> 28672 (Q8_0) are 481 G f16 operations over the two planes and take 425 to 495 us
// (short and sustained runs), 0.97 to 1.13 PFLOP/s where a library's dense bf16 product holds 1.34: the chip's power limit
// first (1.85 to 2.1 of 2.4 GHz, either form, the matrix pipe busy 51 to 59 % of those cycles, 43 to 48 over short walks), the instruction mix of the step after it.  The tile's rows follow the launch (hmm_plan_for): 777 rows are 9 tiles
// of 96 (504 workgroups, two full rounds of the CUs: 366 us) and not 7 of 128 (392: 15 % of the rows padding, the second
// round half empty: 478 us).  Spreading the loads over the steps instead of issuing them together took 9 % (MT = 8) to
// 20 % (MT = 4) off a stage, asking for all rows' scales before the first store 8 to 25 us off every launch.
//
// A K too short to fill the part with tiles is cut into chunks; the chunks' planes are summed in a fixed order by
// pg_launch_sum_parts.
#include <limits.h>
#include <math.h>
#include <type_traits>
#include "pg_internal.h"
#include "pg_f16_planes.h"
#include "pg_quant_dev.h"
#include "pg_stream_addr.h"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef const void __attribute__((address_space(1))) *gptr_t;
typedef void __attribute__((address_space(3))) *lptr_t;

inline unsigned grid_for(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }

__device__ __forceinline__ int swz128(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }

// ---- activation rows -> two f16 planes and the rows' inverse scales (pg_f16_planes.h) ----
// A workgroup of T threads per row, which stays in registers (up to 4 * T * MAXV values) between its maximum and the split: every load
// is on its way before anything waits, vectors past the end are the last one again.  Read twice, 4 values a thread at a time, a row was as many
// memory latencies as it has 1024 values.  us, so : now: 100 x 14336 10.4 : 5.1, 300 x 14336 11.9 : 7.8, 777 x 14336 19.9 : 15.0, 400 x 8192
// 8.1 : 6.1, 1024 x 5632 9.5 : 7.7; rows of 4096 and fewer 0.92 to 1.02 of the time.
template <int MAXV, int T>
__global__ __launch_bounds__(T) void rows_to_f16_planes_vec_kernel(const float *__restrict__ x, int K, _Float16 *__restrict__ hi,
                                                                   _Float16 *__restrict__ lo, float *__restrict__ inv) {
    __shared__ float red[T / 64];
    const size_t row = blockIdx.x;
    const float4 *xr = reinterpret_cast<const float4 *>(x + row * K);
    const int nvec = K / 4;
    float4 v[MAXV];
#pragma unroll
    for (int i = 0; i < MAXV; ++i) v[i] = xr[min((int)threadIdx.x + i * T, nvec - 1)];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) amax = fmaxf(amax, fmaxf(fmaxf(pg_f16_mag(v[i].x), pg_f16_mag(v[i].y)), fmaxf(pg_f16_mag(v[i].z), pg_f16_mag(v[i].w))));
    amax = pg_wave_max_f32(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < T / 64; ++w) amax = fmaxf(amax, red[w]);
    const pg_f16_row_scale sc = pg_f16_row_scale_of(amax);
    if (threadIdx.x == 0) {
        inv[2 * row] = sc.i1;
        inv[2 * row + 1] = sc.i2;
    }
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
        const int at = threadIdx.x + i * T;
        const float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
        if (at < nvec) pg_f16_split4(f, sc, reinterpret_cast<uint2 *>(hi + row * K) + at, reinterpret_cast<uint2 *>(lo + row * K) + at);
    }
}

// Rows of any length (those above pass registers by 32768 values).
__global__ __launch_bounds__(256) void rows_to_f16_planes_kernel(const float *__restrict__ x, int K, _Float16 *__restrict__ hi,
                                                                 _Float16 *__restrict__ lo, float *__restrict__ inv) {
    const size_t row = blockIdx.x;
    const float *xr = x + row * K;
    __shared__ float red[4];
    float amax = 0.0f;
    for (int i = threadIdx.x * 4; i < K; i += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(xr + i);
        amax = fmaxf(amax, fmaxf(fmaxf(pg_f16_mag(v.x), pg_f16_mag(v.y)), fmaxf(pg_f16_mag(v.z), pg_f16_mag(v.w))));
    }
    amax = pg_wave_max_f32(amax);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const pg_f16_row_scale sc = pg_f16_row_scale_of(amax);
    if (threadIdx.x == 0) {
        inv[2 * row] = sc.i1;
        inv[2 * row + 1] = sc.i2;
    }
    for (int i = threadIdx.x * 4; i < K; i += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(xr + i);
        const float f[4] = {v.x, v.y, v.z, v.w};
        pg_f16_split4(f, sc, reinterpret_cast<uint2 *>(hi + row * K + i), reinterpret_cast<uint2 *>(lo + row * K + i));
    }
}

// 8 Q4_0 nibbles as stored at upload (two's complement of q - 8; nibble j = element j of the
// dword's 8) -> 8 f16 values q - 8.  0x6400 | q is the f16 1024 + q; minus 1032 it is q - 8.
__device__ __forceinline__ v8h nibbles_to_f16(uint32_t w) {
    w ^= 0x88888888u;
    const uint32_t a = w & 0x0F0F0F0Fu, b = (w >> 4) & 0x0F0F0F0Fu;
    const v2h bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    union { uint32_t u[4]; v2h h[4]; v8h v; } r;
    r.u[0] = __builtin_amdgcn_perm(b, a, 0x0c040c00u) | 0x64006400u;
    r.u[1] = __builtin_amdgcn_perm(b, a, 0x0c050c01u) | 0x64006400u;
    r.u[2] = __builtin_amdgcn_perm(b, a, 0x0c060c02u) | 0x64006400u;
    r.u[3] = __builtin_amdgcn_perm(b, a, 0x0c070c03u) | 0x64006400u;
#pragma unroll
    for (int p = 0; p < 4; ++p) r.h[p] = r.h[p] - bias;
    return r.v;
}

// 8 Q8_0 quants (two dwords of int8, element order) -> 8 f16 values.  A byte q as q + 128 under 0x64 is the f16
// 1152 + q; the bytes 0x64 come from the selector's second source.
__device__ __forceinline__ v8h bytes_to_f16(uint32_t w0, uint32_t w1) {
    w0 ^= 0x80808080u;
    w1 ^= 0x80808080u;
    const v2h bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    union { uint32_t u[4]; v2h h[4]; v8h v; } r;
    r.u[0] = __builtin_amdgcn_perm(w0, 0x64646464u, 0x00050004u);
    r.u[1] = __builtin_amdgcn_perm(w0, 0x64646464u, 0x00070006u);
    r.u[2] = __builtin_amdgcn_perm(w1, 0x64646464u, 0x00050004u);
    r.u[3] = __builtin_amdgcn_perm(w1, 0x64646464u, 0x00070006u);
#pragma unroll
    for (int p = 0; p < 4; ++p) r.h[p] = r.h[p] - bias;
    return r.v;
}

// The tensors of one launch: equal K, their panels of BN weight rows laid end to end in the launch's tile space.
struct hmm_group {
    const uint8_t *qs[PG_HMM_MAX_GROUP];
    const uint16_t *d[PG_HMM_MAX_GROUP];
    float *out[PG_HMM_MAX_GROUP];      // y, or the first K chunk's plane
    long long stride[PG_HMM_MAX_GROUP];  // floats from one K chunk's plane to the next
    int n[PG_HMM_MAX_GROUP];
    int panel0[PG_HMM_MAX_GROUP];      // first panel of tensor g (INT_MAX: unused)
};

constexpr int BKB = 2;       // blocks per stage
constexpr int HMM_BN = 512;  // weight rows per tile (S = 2: half as many): 64 per wavefront

// QT = 8 (Q8_0): a weight row is two streams of 16-byte half blocks (elements 0 .. 15 and 16 .. 31 of every block,
// as the upload splits them); a stage holds 64 bytes a row, chunk 2 block + half at position chunk ^ ((row >> 2) & 3),
// so that the 64-bit fragment reads of 16 rows spread over all banks.
template <int QT, int MT, int S>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gguf_hmm_kernel(const _Float16 *__restrict__ xh, const _Float16 *__restrict__ xl, const float *__restrict__ inv,
                        const hmm_group grp, int M, int nb, int tiles_m, int ntiles, int ksplit, int kt_per_split) {
    static_assert(MT >= 4 && MT <= 8, "4 to 8 row tiles a wavefront");
    static_assert(S == 1 || S == 2, "blocks of a stage shared between this many groups of wavefronts");
    constexpr int C = 8 / S;                                  // wavefronts side by side
    constexpr int BM = 16 * MT, BN = 64 * C;
    constexpr int WROW = QT == 8 ? 64 : 32;                   // bytes of packed weights per row and stage
    constexpr int LX = (BM / 8 + 7) / 8, LW = (BN * WROW / 1024 + 7) / 8;  // most wave-loads of a wavefront and stage: one plane, weights
    constexpr int XP = BM * 128;                              // one activation plane of a stage
    constexpr int OFF_XL = XP, OFF_W = 2 * XP, OFF_D = OFF_W + 8 * LW * 1024, STAGE = OFF_D + 8 * 256;
    constexpr int LPS = LW + 1 + 2 * LX, FULL = BM / 8 - 8 * (LX - 1);  // wavefronts from FULL on make one load of a plane less
    static_assert(S == 2 || LPS <= 2 * MT, "a load a step");
    extern __shared__ __attribute__((aligned(1024))) char lds[];

    // Workgroups are dealt round-robin to the 8 XCDs; each XCD gets a contiguous run of the launch's tiles (row tiles
    // fastest, K chunks slowest), so the tiles that share an L2 share weight panels; the runs differ by one at most.
    const int total = ntiles * ksplit, xcd = blockIdx.x % 8;
    const int tk = (int)((long long)total * xcd / 8) + blockIdx.x / 8;
    if (tk >= (int)((long long)total * (xcd + 1) / 8)) return;
    const int split = tk / ntiles, t = tk % ntiles;
    const int np = t / tiles_m;
    int g = 0;
#pragma unroll
    for (int i = 1; i < PG_HMM_MAX_GROUP; ++i) g = np >= grp.panel0[i] ? i : g;
    const uint8_t *__restrict__ qs = grp.qs[g];
    const uint16_t *__restrict__ d = grp.d[g];
    const int N = grp.n[g];
    const int m0 = (t % tiles_m) * BM, n0 = (np - grp.panel0[g]) * BN;
    const int K = nb * 32;
    const int kt0 = split * kt_per_split;
    const int KT = nb / BKB - kt0 < kt_per_split ? nb / BKB - kt0 : kt_per_split;
    float *__restrict__ y = grp.out[g] + (size_t)split * grp.stride[g];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, q4 = lane >> 4;
    const int cg = wave % C, sl = wave / C;  // the wavefront's 64 weight rows; S = 2: its block of a stage

    // ---- global -> LDS.  Activation planes: wave-load L covers rows 8L .. 8L+7 (lane -> row,
    // physical chunk; it fetches the logical chunk that belongs there).  Weights: wave-load L
    // covers rows 32L .. 32L+31, two 16-byte blocks a row, the block order flipped in every
    // second group of 8 rows (so that 16 rows' dword reads fall in 64 different banks).
    const char *xsrc[LX];
    {
        const int lr = lane >> 3, pc = lane & 7;
#pragma unroll
        for (int i = 0; i < LX; ++i) {
            const int row = 8 * (wave + 8 * i) + lr;  // (past the tile: never loaded)
            xsrc[i] = reinterpret_cast<const char *>(xh) + pg_hmm_plane_offset(pg_hmm_clamp_row(m0 + row, M), K, kt0, pc ^ swz128(row));
        }
    }
    const ptrdiff_t lo_minus_hi = reinterpret_cast<const char *>(xl) - reinterpret_cast<const char *>(xh);
    const char *wsrc[LW];
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        if constexpr (QT == 8) {
            const int row = 16 * (wave + 8 * i) + (lane >> 2);
            const int rc = row < BN ? row : BN - 1;
            const int c = (lane & 3) ^ ((row >> 2) & 3);  // logical chunk: 2 block + half
            wsrc[i] = reinterpret_cast<const char *>(qs) + pg_hmm_weight_offset_q8(pg_hmm_clamp_row(n0 + rc, N), c & 1, nb, kt0, c >> 1);
        } else {
            const int row = 32 * (wave + 8 * i) + (lane >> 1);
            const int rc = row < BN ? row : BN - 1;
            const int cb = (lane & 1) ^ ((row >> 3) & 1);
            wsrc[i] = reinterpret_cast<const char *>(qs) + pg_hmm_weight_offset(pg_hmm_clamp_row(n0 + rc, N), nb, kt0, cb);
        }
    }
    const char *dsrc;
    {
        const int row = cg * 64 + 2 * (lane & 31);   // this wavefront's own 64 weight rows, two per lane
        dsrc = reinterpret_cast<const char *>(d) + pg_hmm_scale_offset(pg_hmm_scale_row(n0 + row, N), nb, kt0, lane >> 5);
    }
    // Load L of a stage's LPS: the weights, the scales, the high plane, the low plane.  at: where the stage lies in LDS, kt: its index
    // within this workgroup's K chunk.
    auto issue = [&](int at, int kt, int L) {
        char *base = lds + at;
        if (L < LW) {
            __builtin_amdgcn_global_load_lds((gptr_t)(wsrc[L] + (size_t)kt * 32), (lptr_t)(base + OFF_W + (wave + 8 * L) * 1024), 16, 0, 0);
        } else if (L == LW) {
            __builtin_amdgcn_global_load_lds((gptr_t)(dsrc + (size_t)kt * 32), (lptr_t)(base + OFF_D + wave * 256), 4, 0, 0);
        } else {
            const int p = L - LW - 1, i = p % LX;
            if (i + 1 < LX || FULL == 8 || wave < FULL)
                __builtin_amdgcn_global_load_lds((gptr_t)(xsrc[i] + (p < LX ? 0 : lo_minus_hi) + (size_t)kt * 128),
                                                 (lptr_t)(base + (p < LX ? 0 : OFF_XL) + (wave + 8 * i) * 1024), 16, 0, 0);
        }
    };

    // ---- fragment offsets: lane = (row l15, k group q4 of 8 elements)
    int a_off[2 / S], w_off[2 / S], d_off[2 / S];
    {
        const int ra = l15, rb = cg * 64 + l15;
#pragma unroll
        for (int i = 0; i < 2 / S; ++i) {
            const int b = S == 1 ? i : sl;
            a_off[i] = ra * 128 + (((4 * b + q4) ^ swz128(ra)) * 16);                    // + 16 rows per row tile
            if constexpr (QT == 8) w_off[i] = OFF_W + rb * 64 + 16 * ((2 * b + (q4 >> 1)) ^ ((rb >> 2) & 3)) + 8 * (q4 & 1);
            else w_off[i] = OFF_W + rb * 32 + 16 * (b ^ ((rb >> 3) & 1)) + 4 * q4;       // + 16 rows per weight tile
            d_off[i] = OFF_D + wave * 256 + (b * 32 + (l15 >> 1)) * 4 + (l15 & 1) * 2;   // + 32 bytes per weight tile
        }
    }

    v4f acc[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0, 0, 0, 0};

    if constexpr (S == 2) {
        // What reads LDS in a step comes ahead of its loads: a read of f16 behind them waits for every load in flight, or so the compiler has it.
        constexpr int IPS = (LPS + 2) / 3;  // loads a step: all of them in the first three, so that most of the stage is theirs to land
        typedef int v2i __attribute__((ext_vector_type(2)));
        v8h fb[2][4], ah[2], al[2];  // by parity: of the stage (fb, df), of the step
        v4f T[2][4];
        float df[2][4];
        v2i wraw[4];
        _Float16 draw[4];
        int here = 0, next = STAGE, fill = 2 * STAGE;  // where the stage lies, the next one, and the one after that, whose loads are issued meanwhile
        auto read_w = [&](const char *base) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (QT == 8) wraw[j] = *reinterpret_cast<const v2i *>(base + w_off[0] + j * 16 * WROW);
                else wraw[j].x = *reinterpret_cast<const int *>(base + w_off[0] + j * 16 * WROW);
                draw[j] = *reinterpret_cast<const _Float16 *>(base + d_off[0] + j * 32);
            }
        };
        auto unpack = [&](int odd, int j) {
            if constexpr (QT == 8) fb[odd][j] = bytes_to_f16((unsigned)wraw[j].x, (unsigned)wraw[j].y);
            else fb[odd][j] = nibbles_to_f16((unsigned)wraw[j].x);
            df[odd][j] = (float)draw[j];
            asm volatile("" : "+v"(df[odd][j]));
        };
        auto stage = [&](auto parity, int kt) {
            constexpr int O = decltype(parity)::value;
            const char *base = lds + here, *ahead = lds + next;  // (behind the last stage: what lies there, read and not used)
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const int cur = (O * MT + q) & 1, nxt = cur ^ 1, ip = q > 0 ? q - 1 : MT - 1;
                const char *a = (q + 1 < MT ? base : ahead) + a_off[0] + (q + 1) % MT * 16 * 128;
                ah[nxt] = *reinterpret_cast<const v8h *>(a);
                al[nxt] = *reinterpret_cast<const v8h *>(a + OFF_XL);
                if (q == 0) read_w(ahead);
                if (kt + 2 < KT)
#pragma unroll
                    for (int L = q * IPS; L < (q + 1) * IPS; ++L)
                        if (L < LPS) issue(fill, kt + 2, L);
                constexpr int UPS = MT >= 6 ? 1 : 2, UP0 = MT >= 6 ? 2 : 1;
                if (q >= UP0 && q < UP0 + 4 / UPS)
#pragma unroll
                    for (int j = (q - UP0) * UPS; j < (q - UP0 + 1) * UPS; ++j) unpack(O ^ 1, j);
#pragma unroll
                for (int j = 0; j < 4; ++j) T[cur][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[cur], fb[O][j], (v4f){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) T[cur][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[cur], fb[O][j], T[cur][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // (a stage's last row tile: in the next stage)
                    const float scale = df[q > 0 ? O : O ^ 1][j];
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[ip][j][r] = __builtin_fmaf(T[nxt][j][r], scale, acc[ip][j][r]);
                    asm volatile("" : "+v"(acc[ip][j]));
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // The stage after next has landed, all wavefronts' shares of it, and this one is read to the end.
            if (kt + 1 < KT) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
        };
        auto turn = [&]() {
            const int free = here;
            here = next;
            next = fill;
            fill = free;
            asm volatile("" : "+s"(here), "+s"(next), "+s"(fill));  // (scalars to be added, not a vector register for every address)
        };
        using even = std::integral_constant<int, 0>;
        using odd = std::integral_constant<int, 1>;
#pragma unroll
        for (int L = 0; L < LPS; ++L) issue(here, 0, L);
#pragma unroll
        for (int L = 0; L < LPS; ++L) issue(next, 1, L);
        asm volatile("s_waitcnt vmcnt(0)\n s_barrier" ::: "memory");
        read_w(lds);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            unpack(0, j);
            T[1][j] = (v4f){0, 0, 0, 0};  // (of the stage before the first)
            df[1][j] = 0.0f;
        }
        ah[0] = *reinterpret_cast<const v8h *>(lds + a_off[0]);
        al[0] = *reinterpret_cast<const v8h *>(lds + OFF_XL + a_off[0]);
        for (int kt = 0; kt + 1 < KT; kt += 2) {
            stage(even{}, kt);
            turn();
            stage(odd{}, kt + 1);
            turn();
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[MT - 1][j][r] = __builtin_fmaf(T[1][j][r], df[1][j], acc[MT - 1][j][r]);
        if (KT & 1) {  // one more, plainly (as the loop's own way out it had the accumulators copied, and spilled)
            const char *base = lds + here;
            v8h f[4];
            float scale[4];
            read_w(base);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[j] = QT == 8 ? bytes_to_f16((unsigned)wraw[j].x, (unsigned)wraw[j].y) : nibbles_to_f16((unsigned)wraw[j].x);
                scale[j] = (float)draw[j];
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const v8h h = *reinterpret_cast<const v8h *>(base + a_off[0] + i * 16 * 128), l = *reinterpret_cast<const v8h *>(base + OFF_XL + a_off[0] + i * 16 * 128);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v4f t = __builtin_amdgcn_mfma_f32_16x16x32_f16(h, f[j], (v4f){0, 0, 0, 0}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_f16(l, f[j], t, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(t[r], scale[j], acc[i][j][r]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // Both groups' sums of a row tile meet in the group that stores it: even ones in the first, odd ones in the second.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
        int *sums = reinterpret_cast<int *>(lds);  // [side by side][row tile][weight tile][register][lane]
        auto at = [&](int i, int j, int r) { return (((cg * MT + i) * 4 + j) * 4 + r) * 64 + lane; };
#pragma unroll
        for (int i = 0; i < MT; ++i)
            if ((i & 1) != sl)
#pragma unroll
                for (int e = 0; e < 16; ++e) sums[at(i, e >> 2, e & 3)] = __float_as_int(acc[i][e >> 2][e & 3]);
        asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < MT; ++i)
            if ((i & 1) == sl)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][e >> 2][e & 3] += __int_as_float(sums[at(i, e >> 2, e & 3)]);
    } else {
#pragma unroll
        for (int L = 0; L < LPS; ++L) issue(0, 0, L);
        asm volatile("s_waitcnt vmcnt(0)\n s_barrier" ::: "memory");
        for (int kt = 0; kt < KT; ++kt) {
            const int s = kt & 1;
            const char *base = lds + s * STAGE;
            v8h fb[2][4];
            float df[2][4];
            uint32_t wraw[4][QT == 8 ? 2 : 1];
            _Float16 draw[4];
            auto read_w = [&](int b, int j, uint32_t (&raw)[QT == 8 ? 2 : 1]) {
                if constexpr (QT == 8) {
                    const uint2 t = *reinterpret_cast<const uint2 *>(base + w_off[b] + j * 16 * WROW);
                    raw[0] = t.x;
                    raw[1] = t.y;
                } else {
                    raw[0] = *reinterpret_cast<const uint32_t *>(base + w_off[b] + j * 16 * WROW);
                }
            };
            auto unpack = [&](const uint32_t (&raw)[QT == 8 ? 2 : 1]) -> v8h {
                if constexpr (QT == 8) return bytes_to_f16(raw[0], raw[1]);
                else return nibbles_to_f16(raw[0]);
            };
            v8h ah[2], al[2];
            v4f T[2][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                read_w(0, j, wraw[j]);
                fb[0][j] = unpack(wraw[j]);
                df[0][j] = (float)*reinterpret_cast<const _Float16 *>(base + d_off[0] + j * 32);
                asm volatile("" : "+v"(df[0][j]));   // a plain f32 register: the FMAs below are v_fma_f32, not mixed-precision ones
            }
            ah[0] = *reinterpret_cast<const v8h *>(base + a_off[0]);
            al[0] = *reinterpret_cast<const v8h *>(base + OFF_XL + a_off[0]);
#pragma unroll
            for (int q = 0; q < 2 * MT; ++q) {
                const int b = q / MT, cur = q & 1, nxt = cur ^ 1;
                // The next stage's loads, one a step: all at the stage's start, they held back the eight wavefronts' first
                // steps while the address unit took them in.
                if (q < LPS && kt + 1 < KT) issue((s ^ 1) * STAGE, kt + 1, q);
                if (q + 1 < 2 * MT) {
                    const int b1 = (q + 1) / MT, i1 = (q + 1) % MT;
                    ah[nxt] = *reinterpret_cast<const v8h *>(base + a_off[b1] + i1 * 16 * 128);
                    al[nxt] = *reinterpret_cast<const v8h *>(base + OFF_XL + a_off[b1] + i1 * 16 * 128);
                }
                if (q == 0) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        read_w(1, j, wraw[j]);
                        draw[j] = *reinterpret_cast<const _Float16 *>(base + d_off[1] + j * 32);
                    }
                }
                constexpr int UPS = MT >= 6 ? 1 : 2, UP0 = MT >= 6 ? 2 : 1;  // weight tiles of the second block unpacked a step, from step UP0 on
                if (q >= UP0 && q < UP0 + 4 / UPS) {
#pragma unroll
                    for (int u = (q - UP0) * UPS; u < (q - UP0 + 1) * UPS; ++u) {
                        fb[1][u] = unpack(wraw[u]);
                        df[1][u] = (float)draw[u];
                        asm volatile("" : "+v"(df[1][u]));
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) T[cur][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[cur], fb[b][j], (v4f){0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) T[cur][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[cur], fb[b][j], T[cur][j], 0, 0, 0);
                if (q > 0) {
                    const int bp = (q - 1) / MT, ip = (q - 1) % MT;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[ip][j][r] = __builtin_fmaf(T[nxt][j][r], df[bp][j], acc[ip][j][r]);
                        asm volatile("" : "+v"(acc[ip][j]));   // keeps the FMAs in this step (they would sink to the end of the stage)
                    }
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[MT - 1][j][r] = __builtin_fmaf(T[1][j][r], df[1][j], acc[MT - 1][j][r]);
                asm volatile("" : "+v"(acc[MT - 1][j]));
            }
            if (kt + 1 < KT) {
                // Only the next stage's fills are in flight: wait for mine and meet the others, who have then
                // also read this stage to the end; this stage takes the stage after next.
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
            }
        }
    }

    // ---- epilogue: register r of tile (i, j) is row 16 i + 4 q4 + r, weight row 16 j + l15.  All rows' scales are
    // asked for before the first store: one after the other their latencies were 20 to 30 us of every tile.
    float2 sc[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * q4 + r;
            sc[i][r] = reinterpret_cast<const float2 *>(inv)[m < M ? m : M - 1];
        }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(sc[i][r].x), "+v"(sc[i][r].y));
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * q4 + r;
            if (m >= M || (S == 2 && (i & 1) != sl)) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = n0 + cg * 64 + 16 * j + l15;
                if (n < N) __builtin_nontemporal_store(acc[i][j][r] * sc[i][r].x * sc[i][r].y, y + (size_t)m * N + n);
            }
        }
}

// The stages, or (S = 2) the sums that change hands.
template <int QT, int MT, int S> constexpr size_t hmm_lds_bytes() {
    constexpr size_t stages = (S + 1) * (size_t)(2 * 16 * MT * 128 + HMM_BN / S * (QT == 8 ? 64 : 32) + 8 * 256), sums = S == 2 ? MT * 16384 : 0;
    return stages > sums ? stages : sums;
}

}  // namespace

size_t pg_hmm_planes_bytes(size_t rows, size_t k) {
    return 2 * pg_round_up(rows * k * sizeof(_Float16), 256) + pg_round_up(2 * rows * sizeof(float), 256);
}

pg_hmm_planes pg_hmm_planes_carve(void *base, size_t rows, size_t k) {
    pg_hmm_planes p;
    char *c = static_cast<char *>(base);
    p.hi = c;
    c += pg_round_up(rows * k * sizeof(_Float16), 256);
    p.lo = c;
    c += pg_round_up(rows * k * sizeof(_Float16), 256);
    p.inv = reinterpret_cast<float *>(c);
    p.rows = rows;
    p.k = k;
    return p;
}

pg_status pg_launch_rows_to_f16_planes(pg_ctx *ctx, const float *x_dev, size_t rows, size_t k, const pg_hmm_planes &p) {
    if (rows == 0) return PG_OK;
    if (k % 4 != 0 || k > (size_t)INT_MAX) return pg_fail(PG_EINVAL, "rows_to_f16_planes: k = %zu", k);
    auto go = [&](auto kern, int threads) {
        return pg_launch(ctx, "rows_to_f16_planes", kern, dim3((unsigned)rows), dim3(threads), 0, x_dev, (int)k, (_Float16 *)p.hi, (_Float16 *)p.lo, p.inv);
    };
    if ((uintptr_t)x_dev % 16 == 0 && k <= 32768) {
        // (four times the threads where they are not many rows: the launch is then the latency of one)
        if (k <= 1024) return go(rows_to_f16_planes_vec_kernel<1, 256>, 256);
        if (k <= 2048) return go(rows_to_f16_planes_vec_kernel<2, 256>, 256);
        if (k <= 4096) return go(rows_to_f16_planes_vec_kernel<4, 256>, 256);
        if (k <= 8192) return go(rows_to_f16_planes_vec_kernel<2, 1024>, 1024);
        if (k <= 16384) return go(rows_to_f16_planes_vec_kernel<4, 1024>, 1024);
        return go(rows_to_f16_planes_vec_kernel<8, 1024>, 1024);
    }
    return go(rows_to_f16_planes_kernel, 256);
}

// The shape of a product of m rows with n_total weight rows (all the tensors of the launch): row tiles of a wavefront (mt), groups of
// wavefronts that share a stage's blocks (s) and K chunks (ks), those of least estimated time `us`; ks_fixed > 0: the best for that many
// chunks.  `keep`: the caller reads the chunks' planes itself.
// A launch takes as many rounds of the CUs as its fullest XCD has (one workgroup per CU), a round its stages and what its first loads and its
// results take, less of it where CUs are left idle (the others' clock makes that good); on top come the conversion of the rows, the output or the
// chunks' planes, and the pass over them.  All for a chip that has been busy for 0.1 s: these kernels are at its power limit, and in shorter runs they look 10 % better
// against the int8 ones.  Fitted to two thirds of 490 products (36 .. 1100 rows, K 1024 .. 14336, n 1000 .. 30000, up to 6e10 multiply-adds; the five
// best (mt, s, ks) of an earlier fit and four others timed on each): on the others 4.5 % mean error with s = 1 and 3.8 with s = 2, and what is picked
// takes 0.5 % longer than the best on average; the best with s = 1 alone takes 7 % more, with s = 2 alone 1.  (Q4_1's chunks are read by its offsets' launch.)
struct hmm_plan { int mt, s, ks; double us; };
static hmm_plan hmm_plan_for(const pg_ctx *ctx, bool q8, size_t m_, size_t n_total, size_t k_in, int ks_fixed, bool keep) {
    // (a call waits for this: 32-bit divisions, and no more chunks once there are three rounds)
    hmm_plan best = {8, 1, 1, 1e300};
    const unsigned m = (unsigned)m_, stages = (unsigned)(k_in / 64), cus_per_xcd = ctx->num_cu >= 8 ? (unsigned)ctx->num_cu / 8 : 1;
    const double out = 1e-6 * (double)m_ * (double)n_total, rows = 1.8 + 0.98e-6 * (double)m_ * (double)k_in, x = q8 ? 1.0 : 0.0;
    for (int s = 1; s <= 2; ++s) {
        const unsigned bn = HMM_BN / (unsigned)s, panels = ((unsigned)n_total + bn - 1) / bn;
        for (int mt = 8; mt >= 4; --mt) {
            const unsigned bm = 16 * (unsigned)mt, tiles = (m + bm - 1) / bm * panels;
            for (unsigned ks = ks_fixed > 0 ? (unsigned)ks_fixed : 1; ks <= (ks_fixed > 0 ? (unsigned)ks_fixed : 8u); ++ks) {
                const unsigned rounds = ((tiles * ks + 7) / 8 + cus_per_xcd - 1) / cus_per_xcd;
                if (ks_fixed <= 0 && ks > 1 && rounds > 3) break;
                const unsigned per = pg_hmm_chunk(stages, ks, s);
                if (!per || (ks_fixed <= 0 && ks > 1 && per < 8)) continue;
                const double idle = 1.0 - (double)(tiles * ks) / (double)(rounds * cus_per_xcd * 8);
                double us = s == 1 ? rounds * (per * (0.752 + 0.293 * mt + 0.241 * x) + 3.07 + 0.874 * mt) * (1.0 - 0.138 * idle)
                                   : rounds * (per * (0.521 + 0.133 * mt + 0.110 * x) + 2.55 + 0.686 * mt) * (1.0 - 0.078 * idle) + 2.0;
                us += 0.8 * out;
                if (ks > 1) us += keep ? (0.8 * ks + 0.6 * (ks - 1) - 0.8) * out : 2.5 + 1.53 * ks * out;
                if (us < best.us) best = {mt, s, (int)ks, us};
            }
        }
    }
    best.us += rows;
    return best;
}

// What gguf_mm_kernel takes with the rows' digits, us: rounds of workgroups of 128 weight rows x 32 tokens, three to a CU, by their stages of four
// blocks, what the fullest CU's stages take, the digits, the output, the K chunks' planes.  A last tile of up to 16 tokens is 0.7 of one and goes beside
// the others; from 16 token tiles on the fullest XCD's groups of 4 x 8 tiles count.  Fitted as above, 5.6 % mean error.
static double int8_us(const pg_ctx *ctx, bool q8, size_t m, size_t n_total, size_t k_in, bool keep) {
    const unsigned cus = (unsigned)ctx->num_cu, panels = (unsigned)((n_total + 127) / 128), tiles = (unsigned)((m + 31) / 32), k128 = (unsigned)(k_in / 128);
    const size_t groups = (size_t)panels * tiles, cut = std::min<size_t>(8, std::max<size_t>(1, 2 * (size_t)cus / groups));
    const unsigned stages = std::max(2u, (k128 + (unsigned)cut - 1) / (unsigned)cut), ks = std::max(1u, (k128 + stages - 1) / stages);
    const bool light = m - 32 * (size_t)(tiles - 1) <= 16;
    const double work = (double)panels * ks * (light ? tiles - 0.3 : (double)tiles) / cus, out = 1e-6 * (double)m * (double)n_total;
    double fullest = 0.195 * work + 0.805 * ceil((double)panels * ks * (light && tiles > 1 ? tiles - 1 : tiles) / cus), rounds = work < 3.0 ? 1.0 : 0.5 * (work / 3.0 + ceil(work / 3.0));
    if (tiles >= 16 && ks == 1) {
        fullest = std::min(ceil((double)((panels + 3) / 4) * ((tiles + 7) / 8) / 8.0), ceil((double)groups / cus) + 1.0);
        rounds = std::max(1.0, fullest / 3.0);
    }
    return 9.8 + stages * (rounds * 0.405 + fullest * (q8 ? 0.488 : 0.485)) + (ks > 1 ? (keep ? 1.5 : 2.55) * ks * out : 0.0) + 0.72e-6 * (double)m * (double)k_in + 0.93 * out;
}

static bool hmm_type_and_size(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_total, size_t k_in) {
    return ctx->hmm_mode != 2 && (ggml_type == PG_GGML_Q4_0 || ggml_type == PG_GGML_Q8_0) && k_in % 64 == 0 && k_in >= 256 && k_in <= ((size_t)1 << 24) && n_total >= 2 &&
           n_total <= ((size_t)1 << 24) && m >= 2 && m <= ((size_t)1 << 20);
}

// Products whose callers have this kernel's rounding (2^-22 of a row's largest value; the int8 block route's is 2^-16 of a block's), which no
// estimate takes from them: where it is asked for; all of 96 rows and 18 G (Q8_0: 24 G) multiply-adds; and from 65 rows on what two
// rough estimates, the one of the s = 1 tiles and the one of the int8 product, told apart by 7 %.
bool pg_gguf_hmm_holds(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_total, size_t k_in) {
    if (!hmm_type_and_size(ctx, ggml_type, m, n_total, k_in)) return false;
    const double g = 1e-9 * (double)m * (double)n_total * (double)k_in;
    if (ctx->hmm_mode == 1 || (m >= 96 && g >= (ggml_type == PG_GGML_Q8_0 ? 24.0 : 18.0))) return true;
    const double int8 = 12.0 + g * (5.0 + 1.5 * (k_in < 8192 ? (double)k_in : 8192.0) / 8192.0), rows = 4.9 + 1.2e-6 * (double)m * (double)k_in;
    if (m <= 64 || int8 < 30.0) return false;
    const size_t stages = k_in / 64, cus_per_xcd = ctx->num_cu >= 8 ? (size_t)ctx->num_cu / 8 : 1, panels = (n_total + HMM_BN - 1) / HMM_BN;
    for (size_t ks = 1; ks <= 8; ++ks) {
        const size_t per = (stages + ks - 1) / ks;
        if (ks > 1 && ((stages + per - 1) / per != ks || per < 8)) continue;  // an empty chunk, or one too short
        const double sum = ks > 1 ? 0.8 + 1.5e-6 * (double)(ks + 1) * (double)m * (double)n_total : 0.0;
        for (int mt = 8; mt >= 4; --mt) {
            const size_t bm = 16 * (size_t)mt, tiles = (m + bm - 1) / bm * panels * ks, rounds = ((tiles + 7) / 8 + cus_per_xcd - 1) / cus_per_xcd;
            if ((double)rounds * ((double)per * (0.86 + 0.25 * mt) + 3.0 + 0.48 * mt) + rows + sum < 0.93 * int8) return true;
        }
    }
    return false;
}

// Which products this kernel takes, and in how many K chunks: those above, and of the others, from 49 rows on, those that it is estimated to do in 0.9 of the
// int8 block product's time or less: 71 of the 490 products, none of which then takes more than 1 % longer than on the int8 route, on average 0.81 of
// it (at 0.94 it is 101, two of them 4 and 15 % longer).  us, int8 route : this: 635 x 6656 -> 2570 (Q4_0) 118 : 71, 179 x 7936 -> 5900 92 : 57,
// 1046 x 2688 -> 2167 70 : 49, 583 x 4736 -> 4313 (Q8_0) 105 : 78.
bool pg_gguf_hmm_takes(const pg_ctx *ctx, int ggml_type, size_t m, size_t n_total, size_t k_in, int *ks_out, bool keep, double extra_us) {
    if (!hmm_type_and_size(ctx, ggml_type, m, n_total, k_in) || (m <= 48 && ctx->hmm_mode != 1)) return false;
    const bool q8 = ggml_type == PG_GGML_Q8_0;
    const hmm_plan plan = hmm_plan_for(ctx, q8, m, n_total, k_in, 0, keep);
    if (ks_out) *ks_out = plan.ks;
    return plan.us + extra_us < 0.9 * int8_us(ctx, q8, m, n_total, k_in, keep) || pg_gguf_hmm_holds(ctx, ggml_type, m, n_total, k_in);
}

size_t pg_gguf_hmm_part_floats(size_t m, size_t n_total, int ks) { return ks > 1 ? (size_t)ks * m * n_total : 0; }

// ks > 1: the K chunks' planes go to `part` (tensor after tensor, ks planes of m x n_out each) and are summed into
// y[i]; with keep_parts they go to y[i] instead (ks planes, m * n_out floats apart) and stay unsummed.
pg_status pg_launch_gguf_hmm_group(pg_ctx *ctx, size_t k_in, const pg_gguf_tensor *const *w, float *const *y, int count, size_t m,
                                   const pg_hmm_planes &planes, int ks, float *part, bool keep_parts) {
    if (count < 1 || count > PG_HMM_MAX_GROUP) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): %d tensors (1 .. %d)", count, PG_HMM_MAX_GROUP);
    if (m == 0) return PG_OK;
    // (a Q4_1 tensor's nibbles and scales are laid out as a Q4_0 tensor's: its first term runs as the Q4_0 product)
    auto kind = [](int t) { return t == PG_GGML_Q4_1 ? PG_GGML_Q4_0 : t; };
    const int type = kind(w[0]->ggml_type);
    if (type != PG_GGML_Q4_0 && type != PG_GGML_Q8_0) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): ggml type %d", type);
    for (int i = 0; i < count; ++i)
        if (w[i]->k_in != k_in || kind(w[i]->ggml_type) != type) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): the tensors differ in K or type");
    if (k_in % 64 != 0 || planes.rows < m || planes.k != k_in) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): K = %zu, planes of %zu x %zu", k_in, planes.rows, planes.k);
    if (ks < 1 || (ks > 1 && !part && !keep_parts)) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): %d K chunks without a buffer for their planes", ks);
    const bool q8 = type == PG_GGML_Q8_0;
    size_t n_total = 0;
    for (int i = 0; i < count; ++i) n_total += w[i]->n_out;
    const hmm_plan plan = hmm_plan_for(ctx, q8, m, n_total, k_in, ks, keep_parts);
    const size_t bm = 16 * (size_t)plan.mt, bn = HMM_BN / (size_t)plan.s;
    hmm_group grp;
    int panels = 0;
    size_t part_off = 0;
    for (int i = 0; i < PG_HMM_MAX_GROUP; ++i) {
        const bool used = i < count;
        grp.qs[i] = used ? w[i]->qs : nullptr;
        grp.d[i] = used ? w[i]->d : nullptr;
        grp.n[i] = used ? (int)w[i]->n_out : 0;
        grp.panel0[i] = used ? panels : INT_MAX;
        grp.out[i] = used ? (ks > 1 && !keep_parts ? part + part_off : y[i]) : nullptr;
        grp.stride[i] = used && ks > 1 ? (long long)(m * w[i]->n_out) : 0;
        if (used) {
            panels += (int)((w[i]->n_out + bn - 1) / bn);
            part_off += (size_t)ks * m * w[i]->n_out;
        }
    }
    const int tiles_m = (int)((m + bm - 1) / bm), ntiles = tiles_m * panels;
    const int kt_per = (int)pg_hmm_chunk((unsigned)(k_in / 64), (unsigned)ks, plan.s);
    if (kt_per == 0) return pg_fail(PG_EINVAL, "gguf (f16 matrix cores): %d K chunks of %zu stages leave one empty", ks, k_in / 64);
    const dim3 grid((unsigned)(((size_t)ntiles * ks + 7) / 8 * 8));
    const int nb = (int)(k_in / 32);
#define PG_HMM_LAUNCH(QTT, MTT)                                                                                                 \
    case MTT: {                                                                                                                 \
        auto kern = plan.s == 2 ? gguf_hmm_kernel<QTT, MTT, 2> : gguf_hmm_kernel<QTT, MTT, 1>;                                  \
        const size_t lds = plan.s == 2 ? hmm_lds_bytes<QTT, MTT, 2>() : hmm_lds_bytes<QTT, MTT, 1>();                           \
        PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));                                                             \
        PG_TRY(pg_launch(ctx, QTT == 8 ? "gguf_hmm_q8_0" : "gguf_hmm_q4_0", kern, grid, dim3(512), lds, (const _Float16 *)planes.hi, \
                         (const _Float16 *)planes.lo, (const float *)planes.inv, grp, (int)m, nb, tiles_m, ntiles, ks, kt_per)); \
        break;                                                                                                                  \
    }
#define PG_HMM_TILES(QTT)                                                                                                       \
    switch (plan.mt) { PG_HMM_LAUNCH(QTT, 4) PG_HMM_LAUNCH(QTT, 5) PG_HMM_LAUNCH(QTT, 6) PG_HMM_LAUNCH(QTT, 7) PG_HMM_LAUNCH(QTT, 8) }
    if (q8) PG_HMM_TILES(8)
    else PG_HMM_TILES(4)
#undef PG_HMM_TILES
#undef PG_HMM_LAUNCH
    if (ks > 1 && !keep_parts) {
        size_t off = 0;
        for (int i = 0; i < count; ++i) {
            const size_t plane = m * w[i]->n_out;
            PG_TRY(pg_launch_sum_parts(ctx, part + off, plane, ks, plane, y[i]));
            off += (size_t)ks * plane;
        }
    }
    return PG_OK;
}
