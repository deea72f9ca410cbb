// MXFP4 weights (gpt_oss experts, examples/gpt_oss/moe.rs:5-117) on the scaled matrix-core
// instruction of gfx950, which takes FP4 (E2M1) codes and E8M0 block scales as they sit in the file.
//
// v_mfma_scale_f32_16x16x128_f8f6f4, D[16 x 16] += A[16 x 128] * B[128 x 16], with A in FP4 and B in
// FP8 (E4M3), every 32 consecutive k of a row of A / column of B scaled by 2^(byte - 127):
//   A  lane l holds row l % 16, k = 32 (l / 16) .. + 31: the 16 code bytes of one MXFP4 block, element e
//      in nibble e -- exactly the file's packing (byte i = elements 2i low, 2i + 1 high);
//   B  lane l holds column l % 16; its first 16 bytes are k = 16 (l / 16) .. + 15, its last 16 bytes
//      k = 64 + 16 (l / 16) .. + 15;
//   scale operands: one byte per lane (selected by op_sel), lane l = row or column l % 16, k block l / 16;
//   D  lane l holds column l % 16, rows 4 (l / 16) .. + 3.
// (Layouts read off the hardware with one-hot operands.)
//
// The weights are rows of A: 17 bytes per block are all the product reads.  An activation row is not
// representable in FP8, but a fixed-point rewriting of it is: per block x[k] = 2^se X[k], |X| < 2^23, and
// X = sum_j 32^j n_j with five balanced base-32 digits n_j in [-16, 16], each exact in E4M3.  Digit plane
// j of a row is one column of B with block scale byte 127 + se + 5 j, so the instruction itself applies
// both block scales and sums over K; the five columns of a row are added at the end.  Three activation
// rows (15 columns) share one pass over the weights.
//
// From some dozens of rows on the digits are FP6 (E2M3), which holds n / 8 for every integer to 16 as well: beside an FP4 operand
// the instruction then takes half the cycles (random operands, all CUs: 4.2 PFLOP/s in FP8, 6.6 in FP6).
//   B  lane l holds column l % 16, k = 32 (l / 16) .. + 31, element e in bits 6 e .. 6 e + 5 of its 24 bytes.
#include <math.h>
#include <type_traits>
#include "pg_internal.h"
#include "pg_stream_addr.h"
#include "pg_digits.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v3i __attribute__((ext_vector_type(3)));
typedef int v6i __attribute__((ext_vector_type(6)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef const v4i __attribute__((address_space(1))) *gv4i_ptr;
// (a pointer out of a table is not known to lead to global memory: the compiler reads through it by flat loads, which count as LDS
// reads too, and every wait for LDS then waits for memory)
typedef const uint32_t __attribute__((address_space(1))) *gu32_ptr;
typedef const float __attribute__((address_space(1))) *gf32_ptr;

constexpr int MX_PLANES = 5;  // digit planes per activation row
constexpr int MX_U = 8;       // chunks (of 4 blocks) per batch of weight loads in flight
constexpr int MX_MAX_T = 3;   // activation rows per pass over the weights

inline unsigned grid_for(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }
inline size_t mx_chunks(size_t nb) { return pg_mx_chunks(nb); }  // chunks of 4 blocks per row, whole scale dwords

// ---- device layout of a tensor ------------------------------------------------------
// Fragment-major: for every group of 16 rows and every chunk of 4 blocks (128 k), the 64 lanes' 16 code
// bytes in lane order (one fully coalesced 1 KiB load per instruction), and per 4 chunks one dword per
// lane with the 4 scale bytes.  Rows and blocks past the tensor's end hold zero codes; blocks whose
// scale byte is 0 (the reference's f32::from_bits(0) = 0.0, the hardware's 2^-127) also get zero codes.
__global__ void mxfp4_fragments_kernel(const uint8_t *__restrict__ blocks, const uint8_t *__restrict__ scales, int n_out,
                                       int nb, int ncp, uint4 *__restrict__ qs, uint8_t *__restrict__ sc) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // (row group, chunk, lane)
    const size_t nrg = ((size_t)n_out + 15) / 16;
    if (i >= nrg * ncp * 64) return;
    const int lane = (int)(i & 63), c = (int)((i >> 6) % ncp);
    const size_t rg = (i >> 6) / ncp;
    const size_t row = rg * 16 + (lane & 15);
    const int blk = 4 * c + (lane >> 4);
    uint4 v = {0, 0, 0, 0};
    unsigned e = 127;
    if (row < (size_t)n_out && blk < nb) {
        e = scales[row * nb + blk];
        if (e != 0) {
            const uint8_t *src = blocks + (row * nb + blk) * 16;  // any alignment
            unsigned wv[4];
            for (int t = 0; t < 4; ++t) wv[t] = src[4 * t] | (src[4 * t + 1] << 8) | (src[4 * t + 2] << 16) | ((unsigned)src[4 * t + 3] << 24);
            v = make_uint4(wv[0], wv[1], wv[2], wv[3]);
        }
    }
    qs[i] = v;
    sc[((rg * (ncp / 4) + c / 4) * 64 + lane) * 4 + (c & 3)] = (uint8_t)e;
}

// ---- one activation block -> five E4M3 digit planes in LDS ---------------------------
// Eight consecutive lanes hold one block (f = elements 4 sub .. 4 sub + 3); all eight call together.
// dig: the row's first plane, planes `stride` bytes apart, k-th element of plane j at dig[j * stride + k];
// sb:  scale bytes, plane j / block b at sb[(j * 4 + b % 4) * ncp + b / 4].
__device__ __forceinline__ void mx_emit_digits(const float (&f)[4], int b, int sub, char *dig, int stride, uint8_t *sb, int ncp) {
    float amax = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
    int bad = (f[0] != f[0]) | (f[1] != f[1]) | (f[2] != f[2]) | (f[3] != f[3]);
    amax = fmaxf(amax, __builtin_bit_cast(float, pg_dpp8<0xB1>(__builtin_bit_cast(int, amax))));
    bad |= pg_dpp8<0xB1>(bad);
    amax = fmaxf(amax, __builtin_bit_cast(float, pg_dpp8<0x4E>(__builtin_bit_cast(int, amax))));
    bad |= pg_dpp8<0x4E>(bad);
    amax = fmaxf(amax, __builtin_bit_cast(float, pg_dpp8<0x141>(__builtin_bit_cast(int, amax))));
    bad |= pg_dpp8<0x141>(bad);
    int se = 0;
    float inv = 1.0f;
    if (bad || !(amax <= 3.4028234663852886e38f)) {
        bad = 1;
        inv = 0.0f;
    } else if (amax > 0.0f) {
        int ex;
        (void)frexpf(amax, &ex);  // amax = f * 2^ex, f in [0.5, 1)
        se = ex - 23;             // |x| / 2^se < 2^23
        if (se < -126) se = -126;
        inv = ldexpf(1.0f, -se);
    }
    // Balanced base-32 digits, top down and all in f32 (every value is a small integer times a power of two,
    // so each step is exact): n_j = round(r / 32^j), r -= n_j 32^j; |n_j| <= 16.
    float r[4], d[MX_PLANES][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = f[e] * inv;
        r[e] = (t != t) ? 0.0f : rintf(t);
    }
#pragma unroll
    for (int j = MX_PLANES - 1; j >= 1; --j) {
        const float down = __builtin_bit_cast(float, (127 - 5 * j) << 23), up = -__builtin_bit_cast(float, (127 + 5 * j) << 23);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            d[j][e] = rintf(r[e] * down);
            r[e] = fmaf(d[j][e], up, r[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) d[0][e] = r[e];
#pragma unroll
    for (int j = 0; j < MX_PLANES; ++j) {  // integers in [-16, 16] are exact in E4M3: the conversion's rounding never acts
        int packed = __builtin_amdgcn_cvt_pk_fp8_f32(d[j][0], d[j][1], 0, false);
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(d[j][2], d[j][3], packed, true);
        *reinterpret_cast<int *>(dig + (size_t)j * stride + b * 32 + 4 * sub) = packed;
    }
    if (sub < MX_PLANES)  // a NaN / inf block poisons every product it enters: scale byte 255 is NaN
        sb[(sub * 4 + (b & 3)) * ncp + (b >> 2)] = (uint8_t)(bad ? 255 : 127 + se + 5 * sub);
}

// ---- the product ----------------------------------------------------------------------
// A workgroup of NW wavefronts = RG groups of 16 weight rows x KS = NW / RG slices of K, against T
// activation rows (blockIdx.y picks which); it first rewrites those rows (all of K) as digit planes in
// LDS while its first weight loads are in flight.  Each wavefront then walks its K slice in batches of
// MX_U chunks, the next batch requested before the current one is consumed, and the partial tiles of
// the KS slices and the 5 planes are added through LDS in a fixed order.
// PAIRS 1 and 2 (T = 1): blockIdx.z and y are a token and one of its gridDim.y entries in an MoE layer: the weights are that expert's
// entry of two pointer tables, the activation row is the token's (by_token) or the pair's, the output row the pair's.  2: mlp1, whose rows 2 i and 2 i + 1
// with their biases become value i of the output row, their swiglu (made where mlp2
// reads its rows it is made once for every 64 of mlp2's rows: 5 us more at 64 pairs of 2880 x 2880).  With the choice of the experts read
// as the caller made it, a layer of few pairs is three launches where it was five.  The expert and its tables are found by scalar loads
// behind the requests for the activation row: looked up ahead of them, by a lane an entry, that chain was in front of every one of up to
// eleven rounds of workgroups.  us, five launches : the look-up in front : now, 4 of 32 experts of 2880 x 2880: one token 24.5 : 20.5 : 19.6, two 33.5 :
// 32.0 : 28.5, 16 tokens 160.0 : 163.3 : 154.7; 16 tokens of 1440 x 2880 88.8 : 92.4 : 86.0; 4 of 16 of 1024 x 1024, two tokens 19.2 : 15.2 : 14.7.
struct mt_swiglu {
    const float *const *bias_tab;
    float alpha, clamp;
    // biased = h + bias; gate = biased[2i].min(clamp); linear = biased[2i+1].clamp(-clamp, clamp);
    // out[i] = gate * (1 / (1 + exp(-alpha * gate))) * (linear + 1)   examples/gpt_oss/moe.rs:155-166
    __device__ __forceinline__ static float of(float g0, float l0, float alpha, float clamp) {
        const float gate = fminf(g0, clamp);                                     // f32::min: a NaN operand loses
        const float linear = l0 != l0 ? l0 : fminf(fmaxf(l0, -clamp), clamp);    // f32::clamp keeps NaN
        const float activated = gate * (1.0f / (1.0f + expf(-alpha * gate)));
        return activated * (linear + 1.0f);
    }
};
struct mx_pairs {
    const uint8_t *const *qs_tab;
    const uint32_t *const *sc_tab;
    const int *idx;  // [tokens][top_k], the caller's
    int *chosen;     // [pairs], written by mlp1 (16 tokens, 4 of 32 experts: 1 us less than finding each again)
    int experts, by_token;
    mt_swiglu act;
};
// The experts of a token's entries 0 .. k, one after the other: an entry out of range, or one that an entry before it names, stands for
// the lowest expert not taken yet (copy_routing_kernel's rule).
struct mx_routed {
    unsigned long long taken[4] = {0, 0, 0, 0};
    __device__ __forceinline__ int next(int e, int experts, bool &named) {
        named = e >= 0 && e < experts;
        if (named) {
#pragma unroll
            for (int w = 0; w < 4; ++w)
                if (e >> 6 == w) named = !((taken[w] >> (e & 63)) & 1ull);
        }
        if (!named) {
#pragma unroll
            for (int w = 3; w >= 0; --w)
                if (~taken[w]) e = 64 * w + __builtin_ctzll(~taken[w]);
        }
#pragma unroll
        for (int w = 0; w < 4; ++w)
            if (e >> 6 == w) taken[w] |= 1ull << (e & 63);
        return e;
    }
};
static_assert(PG_MOE_MAX_EXPERTS <= 256, "mx_routed holds 256 experts");
// What the kernel does not write, at addresses that are the same for a wavefront: through the scalar cache.
template <typename T> __device__ __forceinline__ T mx_uniform(const T *p) {
    typedef const T __attribute__((address_space(4))) *ptr;
    return *(ptr)(uintptr_t)p;
}
// Entry k (up to 63) of a token, by a wavefront: the first four as scalars, later ones a lane an entry; only where one up to k is out
// of range or named twice they are walked.
__device__ __forceinline__ int mx_expert_of_entry(const int *__restrict__ idx, int k, int experts) {
    if (k < 4) {
        int a[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = mx_uniform(idx + (j < k ? j : k));
        bool fine = true;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            fine = fine && (unsigned)a[j] < (unsigned)experts;
#pragma unroll
            for (int l = j + 1; l < 4; ++l) fine = fine && (a[j] != a[l] || l > k);
        }
        if (fine) return a[3];  // (entry k, clamped)
    }
    const int lane = threadIdx.x & 63, e = idx[lane < k ? lane : k];
    bool odd = e < 0 || e >= experts;
    for (int j = 0; j < k; ++j) odd |= lane > j && lane <= k && e == __builtin_amdgcn_readlane(e, j);
    if (!__ballot(odd)) return __builtin_amdgcn_readlane(e, k);
    mx_routed taken;
    int expert = 0;
    bool named;
    for (int j = 0; j <= k; ++j) expert = taken.next(__builtin_amdgcn_readlane(e, j), experts, named);
    return __builtin_amdgcn_readfirstlane(expert);
}

template <int T, int RG, int NW, int PAIRS = 0>
__global__ __launch_bounds__(64 * NW) void mxfp4_rows_kernel(const uint8_t *__restrict__ qs_frag, const uint32_t *__restrict__ sc_frag,
                                                                  const float *__restrict__ x, float *__restrict__ y,
                                                                  int n_out, int nb, int ncp, int m, const mx_pairs pr) {
    static_assert(!PAIRS || T == 1, "a pair is one activation row");
    constexpr int KS = NW / RG, COLS = MX_PLANES * T;
    size_t x_row0 = (size_t)blockIdx.y * T;  // first activation row of this workgroup
    float bias = 0.0f;
    const size_t pair = (size_t)blockIdx.z * gridDim.y + blockIdx.y;
    if (PAIRS) x_row0 = pr.by_token ? blockIdx.z : pair;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int kp = ncp * 128, stride = kp + 16;  // plane stride = 16 (mod 256): the 16 columns of a 128-bit read fall into 16 different bank groups
    char *const dig = lds;
    uint8_t *const sb = reinterpret_cast<uint8_t *>(lds + (size_t)COLS * stride);
    float *const part = reinterpret_cast<float *>(lds + (size_t)COLS * stride + (((size_t)COLS * 4 * ncp + 15) & ~(size_t)15));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rgi = wave / KS, ksi = wave % KS;
    const int nrg = (n_out + 15) / 16;
    int rg = blockIdx.x * RG + rgi;
    rg = rg < nrg ? rg : nrg - 1;  // a spare wavefront repeats the last group; its result is not stored
    const int cps = ((ncp + KS - 1) / KS + 3) & ~3;  // chunks per K slice, whole scale dwords
    const int c0 = ksi * cps, c1 = (c0 + cps < ncp) ? c0 + cps : ncp;
    gv4i_ptr qa = nullptr;
    const uint32_t *__restrict__ sa = nullptr;

    v4i abuf[2][MX_U];
    uint32_t sabuf[2][MX_U / 4];
    auto load_batch = [&](v4i (&a)[MX_U], uint32_t (&s)[MX_U / 4], int cb) {
#pragma unroll
        for (int u = 0; u < MX_U; ++u) {
            const int c = cb + u;
            a[u] = __builtin_nontemporal_load(qa + (size_t)pg_mx_chunk(c, ncp) * 64);
        }
#pragma unroll
        for (int g = 0; g < MX_U / 4; ++g) {
            const int c = cb + 4 * g;
            s[g] = sa[(size_t)pg_mx_scale_word(c, ncp) * 64];
        }
    };
    // Loads return in issue order: the activation blocks of the first rounds (from L2) are requested
    // before the weights (from HBM), so that the digit arithmetic runs while the weights are in flight.
    const int sub = threadIdx.x & 7, nblk = 4 * ncp;
    // (No branch around a load: behind one the compiler waits for every load in flight, the weights too.
    // Block ids past the end load the last block again.)
    const int last = T * nblk - 1;
    auto row_of = [&](int id) { return T == 1 ? 0 : (id >= nblk) + (T > 2 && id >= 2 * nblk); };  // id / nblk
    auto x_valid = [&](int id) {
        const int t = row_of(id), b = id - t * nblk;
        return b < nb && x_row0 + t < (size_t)m;  // blocks nb .. 4 ncp - 1 and rows past m are zeros
    };
    auto load_x = [&](int id) {
        const int t = row_of(id), b = id - t * nblk;
        const size_t at = x_valid(id) ? ((x_row0 + t) * nb + b) * 8 + sub : 0;
        return reinterpret_cast<const float4 *>(x)[at];
    };
    auto emit = [&](int id, const float4 v) {
        const int t = row_of(id), b = id - t * nblk;
        const bool keep = x_valid(id);
        const float f[4] = {keep ? v.x : 0.0f, keep ? v.y : 0.0f, keep ? v.z : 0.0f, keep ? v.w : 0.0f};
        mx_emit_digits(f, b, sub, dig + (size_t)t * MX_PLANES * stride, stride, sb + (size_t)t * MX_PLANES * 4 * ncp, ncp);
    };
    constexpr int PER_ROUND = 8 * NW;  // blocks per round: 8 threads each
    constexpr int NPRE = 4;                  // rounds whose activation blocks are requested ahead of the weights
    const int g0 = threadIdx.x >> 3;
    float4 xv[NPRE];
#pragma unroll
    for (int r = 0; r < NPRE; ++r) {
        const int id = g0 + r * PER_ROUND;
        xv[r] = load_x(id < last ? id : last);
    }
    asm volatile("" ::: "memory");  // (keeps the compiler from moving these loads down to their uses)
    __builtin_amdgcn_sched_barrier(0);
    if (PAIRS) {  // (the pair's expert and its tables, scalar loads, while the activation blocks fly)
        const int expert = PAIRS == 2 ? mx_expert_of_entry(pr.idx + (size_t)blockIdx.z * gridDim.y, blockIdx.y, pr.experts) : mx_uniform(pr.chosen + pair);
        if (PAIRS == 2 && blockIdx.x == 0 && threadIdx.x == 0) pr.chosen[pair] = expert;
        qs_frag = mx_uniform(pr.qs_tab + expert);
        sc_frag = mx_uniform(pr.sc_tab + expert);
        if (PAIRS == 2) {  // (asked for now: one of the 16 RG rows a thread of the last step)
            const int row = (int)blockIdx.x * RG * 16 + (int)threadIdx.x % (RG * 16);
            bias = mx_uniform(pr.act.bias_tab + expert)[row < n_out ? row : n_out - 1];
        }
    }
    qa = (gv4i_ptr)(uintptr_t)qs_frag + (size_t)rg * ncp * 64 + lane;
    sa = sc_frag + (size_t)rg * (ncp / 4) * 64 + lane;
    load_batch(abuf[0], sabuf[0], c0 < ncp ? c0 : 0);  // (an empty slice consumes nothing)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < NPRE; ++r) {
        const int id = g0 + r * PER_ROUND;
        if (id <= last) emit(id, xv[r]);  // whole 8-thread groups together
    }
    for (int id = g0 + NPRE * PER_ROUND; id <= last; id += PER_ROUND) emit(id, load_x(id));
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");  // (not __syncthreads(): the weight loads stay in flight)

    // B side of this lane: column min(lane % 16, COLS - 1) (the spare columns repeat the last one and are dropped)
    const int col = (lane & 15) < COLS ? (lane & 15) : COLS - 1, q = lane >> 4;
    const char *const bcol = dig + (size_t)col * stride + 16 * q;
    const uint8_t *const sbl = sb + (size_t)(col * 4 + q) * ncp;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    auto consume = [&](const v4i (&a)[MX_U], const uint32_t (&s)[MX_U / 4], int cb) {
#pragma unroll
        for (int g = 0; g < MX_U / 4; ++g) {
            if (cb + 4 * g < c1) {  // the same for the whole wavefront
                const int sbv = *reinterpret_cast<const int *>(sbl + cb + 4 * g);
                const char *bp = bcol + (size_t)(cb + 4 * g) * 128;
                // (the byte selectors of the two scale operands are immediates)
#define PG_MX_STEP(U)                                                                                                   \
    do {                                                                                                                \
        const v4i b0 = *reinterpret_cast<const v4i *>(bp + (U) * 128), b1 = *reinterpret_cast<const v4i *>(bp + (U) * 128 + 64); \
        const v4i aw = a[4 * g + (U)];                                                                                  \
        const v8i A = {aw[0], aw[1], aw[2], aw[3], 0, 0, 0, 0};                                                         \
        const v8i B = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};                                         \
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, acc, 4, 0, (U), (int)s[g], (U), sbv);              \
    } while (0)
                PG_MX_STEP(0);
                PG_MX_STEP(1);
                PG_MX_STEP(2);
                PG_MX_STEP(3);
#undef PG_MX_STEP
            }
        }
    };
    for (int cb = c0; cb < c1; cb += 2 * MX_U) {
        if (cb + MX_U < c1) load_batch(abuf[1], sabuf[1], cb + MX_U);
        __builtin_amdgcn_sched_barrier(0);
        consume(abuf[0], sabuf[0], cb);
        if (cb + 2 * MX_U < c1) load_batch(abuf[0], sabuf[0], cb + 2 * MX_U);
        __builtin_amdgcn_sched_barrier(0);
        if (cb + MX_U < c1) consume(abuf[1], sabuf[1], cb + MX_U);
    }

    // part[wave][lane][r]: column lane % 16, row 4 (lane / 16) + r of this wavefront's tile
    *reinterpret_cast<v4f *>(part + ((size_t)wave * 64 + lane) * 4) = acc;
    __syncthreads();
    if (threadIdx.x < RG * 16 * T) {
        const int t = threadIdx.x / (RG * 16), rr = threadIdx.x % (RG * 16), g = rr / 16, i = rr % 16;
        float sum = 0.0f;
#pragma unroll
        for (int j = MX_PLANES - 1; j >= 0; --j)
#pragma unroll
            for (int k = 0; k < KS; ++k)
                sum += part[((size_t)(g * KS + k) * 64 + 16 * (i >> 2) + t * MX_PLANES + j) * 4 + (i & 3)];
        const size_t row = ((size_t)blockIdx.x * RG + g) * 16 + i, item = PAIRS ? pair : (size_t)blockIdx.y * T + t;
        if constexpr (PAIRS == 2) {
            const float v = sum + bias, linear = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false));
            if (!(row & 1) && row < (size_t)n_out) y[item * (n_out / 2) + row / 2] = mt_swiglu::of(v, linear, pr.act.alpha, pr.act.clamp);
        } else if (row < (size_t)n_out && (PAIRS || item < (size_t)m)) y[item * n_out + row] = sum;
    }
}

size_t mx_lds_bytes(int t, int ncp, int nw = 16) {
    const size_t cols = (size_t)MX_PLANES * t;
    return cols * ((size_t)ncp * 128 + 16) + ((cols * 4 * ncp + 15) & ~(size_t)15) + (size_t)nw * 64 * 4 * sizeof(float);
}

template <int T, int RG, int NW>
pg_status launch_rows(pg_ctx *ctx, const pg_gguf_tensor *w, const float *x, float *y, size_t m, int ncp) {
    const size_t lds = mx_lds_bytes(T, ncp, NW);
    auto kern = mxfp4_rows_kernel<T, RG, NW>;
    PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));
    const dim3 grid(grid_for((w->n_out + 15) / 16, RG), grid_for(m, T));
    return pg_launch(ctx, "mxfp4_rows", kern, grid, dim3(64 * NW), lds, (const uint8_t *)w->qs,
                     reinterpret_cast<const uint32_t *>(w->d), x, y, (int)w->n_out, (int)(w->k_in / 32), ncp, (int)m, mx_pairs{});
}

// One launch for `pairs` (token, expert) pairs, top_k a token; x has x_rows rows.
template <int RG, int NW, int PAIRS>
pg_status launch_rows_pairs(pg_ctx *ctx, size_t n_out, size_t k_in, const float *x, size_t x_rows, float *y, size_t pairs, size_t top_k, int ncp,
                            const mx_pairs &pr) {
    const size_t lds = mx_lds_bytes(1, ncp, NW);
    auto kern = mxfp4_rows_kernel<1, RG, NW, PAIRS>;
    PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));
    const dim3 grid(grid_for((n_out + 15) / 16, RG), (unsigned)top_k, (unsigned)(pairs / top_k));
    return pg_launch(ctx, "mxfp4_rows_pairs", kern, grid, dim3(64 * NW), lds, (const uint8_t *)nullptr, (const uint32_t *)nullptr, x, y,
                     (int)n_out, (int)(k_in / 32), ncp, (int)x_rows, pr);
}

}  // namespace

// y[m, n_out] = x[m, k_in] . W^T for an MXFP4 tensor; x 16-byte aligned.
pg_status pg_launch_mxfp4_rows(pg_ctx *ctx, const float *x_dev, size_t m, const pg_gguf_tensor *w, float *y_dev) {
    if (m == 0) return PG_OK;
    const int nb = (int)(w->k_in / 32), ncp = (int)mx_chunks((size_t)nb);
    int t = m < (size_t)MX_MAX_T ? (int)m : MX_MAX_T;
    while (t > 1 && mx_lds_bytes(t, ncp) > (96u << 10)) --t;  // room for a second workgroup per CU
    if (mx_lds_bytes(t, ncp) > (160u << 10))
        return pg_fail(PG_EUNSUPPORTED, "mxfp4: k_in %zu does not fit the digit planes in LDS (up to 28160)", w->k_in);
    if ((m + t - 1) / t > 65535) return pg_fail(PG_EUNSUPPORTED, "mxfp4: more than %d activation rows", 65535 * t);
    // Every workgroup rewrites the activation rows as digits, so the fewer workgroups the less of that work.
    // Up to one group of 16 weight rows per CU: 16 wavefronts on it, K in 16 slices.  Beyond: 8 wavefronts
    // with the fewest row groups per workgroup (1, 2 or 4; K in 8, 4 or 2 slices) with which all
    // workgroups are resident at once (two per CU), four past that.
    const size_t groups = (w->n_out + 15) / 16 * ((m + t - 1) / t), slots = (size_t)ctx->num_cu * 2;
    const int shape = groups <= (size_t)ctx->num_cu ? 0 : (groups <= slots ? 1 : ((groups + 1) / 2 <= slots ? 2 : 4));
#define PG_MX_LAUNCH(TT)                                                                                              \
    (shape == 0 ? launch_rows<TT, 1, 16>(ctx, w, x_dev, y_dev, m, ncp)                                                \
     : shape == 1 ? launch_rows<TT, 1, 8>(ctx, w, x_dev, y_dev, m, ncp)                                               \
     : shape == 2 ? launch_rows<TT, 2, 8>(ctx, w, x_dev, y_dev, m, ncp) : launch_rows<TT, 4, 8>(ctx, w, x_dev, y_dev, m, ncp))
    switch (t) {
        case 1: return PG_MX_LAUNCH(1);
        case 2: return PG_MX_LAUNCH(2);
        default: return PG_MX_LAUNCH(3);
    }
#undef PG_MX_LAUNCH
}

namespace {

// ---- many activation rows: tiles on the scaled matrix-core instruction ------------------------
// From a few dozen rows on the product is matrix-core work, and the instruction still does all of it: the block
// scales of both sides are applied inside, so there is no rescaling of accumulators and nothing to dequantise.
// An activation block becomes MT_PLANES balanced base-32 digits per value (20 bits under the block's largest
// magnitude, |error| <= 2^-20 of it), each plane a B operand whose block scale carries the digit's weight (FP6: against 64 bits the
// products' error is that of the same digits in FP8 to 1 %, 0.999 of it on average over 36 shapes); the
// planes accumulate into the same tile, so a row costs MT_PLANES instructions per 16 x 16 x 128 tile and no
// final sum.  A pre-pass writes the planes once, in the operand's own fragment order: per token group of 16
// and chunk of 128 k one record of MT_RECORD bytes,
//   [plane][64 lanes][16 B] [64 lanes][8 B]   lane = token % 16 + 16 (block of the chunk): the block's 32 digits of 6 bits
//   [64 lanes] scale dwords         lane = token % 16 + 16 (block of the chunk), byte j = plane j
constexpr int MT_PLANES = PG_MT_PLANES;
constexpr int MT_NW = PG_MT_NW;            // wavefronts per workgroup
constexpr int MT_FRAG = PG_MT_FRAG;        // bytes of one plane fragment
constexpr int MT_RECORD = PG_MT_RECORD;    // one token group's planes and scales of a chunk
constexpr int MT_UNITS = MT_RECORD / 16;   // in 16-byte units

// Experts' token lists, for the grouped products of an MoE layer: the token tiles (TB groups of 16 slots) of all
// experts follow one another, expert e's from tile goff[e]; slot i of an expert holds pair lists[e * stride + i].
struct mt_gather {
    const int *lists, *counts, *goff;  // [E][stride], [E], [E + 1]
    int stride, experts, tb, div;      // row of the source matrix = pair / div
};
// The expert whose tiles include token tile gt, its first tile and the slots it uses; expert -1 past the last tile.  Called by whole
// wavefronts with one gt: a lane reads the offset and the count of its expert and the ballot finds the place, so one round trip to
// memory stands before the lists' instead of one per halving and two more (every workgroup begins with it, none has anything else to
// do meanwhile).  Twenty tokens over 32 experts of 2880 x 2880, top 4: the four launches that look 97.1 -> 93.4 us together; 480 over 8 of
// 2048 x 2048 171 -> 165.
struct mt_place { int expert, first_tile, used; };
__device__ __forceinline__ mt_place mt_find(const mt_gather &g, int gt) {
    mt_place at = {-1, 0, 0};
    const int lane = threadIdx.x & 63;
    for (int base = 0;; base += 64) {
        const int e = base + lane;
        const int off = g.goff[e < g.experts ? e : g.experts], n = g.counts[e < g.experts ? e : g.experts - 1];
        const int here = __popcll(__ballot(e <= g.experts && off <= gt));  // (the offsets ascend)
        if (here > 0) {
            at.expert = base + here - 1;
            at.first_tile = __builtin_amdgcn_readlane(off, here - 1);
            at.used = __builtin_amdgcn_readlane(n, here - 1);
        }
        if (here < 64 || base + 64 > g.experts) break;
    }
    if (at.expert == g.experts) at.expert = -1;
    return at;
}

// The caller's routing on its way into the first product's planes, for calls of few pairs: every workgroup works out by itself what its slots
// hold (the pairs' entries in LDS, each expert's count, one ballot for the tile's expert), and one more writes what the later launches
// read -- what route_lists_kernel makes, entries that break the rules replaced as there.  A launch of its own was 4.9 us and the gap
// behind it.  us, with it : in the planes' launch: 20 tokens, top 4 of 32 experts of 2880 x 2880 97 : 94, 64 tokens 114 : 111; 19, top 4 of 8 of
// 544 x 864 29.0 : 26.5; 64, top 4 of 16 of 576 x 864 34.0 : 31.4; 200, top 1 of 4 of 704 x 512 28.9 : 27.3; 64, top 4 of 64 of 3808 x 3008
// 252 : 249; 70 drawn calls 0.936 of the time.  Beyond, a pair would no longer be a thread nor an expert a lane.
constexpr int MT_ROUTE_PAIRS = 256, MT_ROUTE_EXPERTS = 64;  // at most: a pair a thread, an expert a lane
struct mt_route {
    const int *idx;
    const float *w;
    int tokens, top_k, tile;  // tile: slots of a token tile
    int *topk_idx;
    float *topk_p;
    int *lists, *counts, *goff;
};
struct mt_route_lds {
    int pair[MT_ROUTE_PAIRS], count[MT_ROUTE_EXPERTS], broken;
    uint8_t zero[MT_ROUTE_PAIRS];     // pairs of weight 0
    uint16_t slots[4][16];            // by wavefront: the pairs of its 16 slots
};
// The pairs' experts and the experts' counts (256 threads).
__device__ __forceinline__ void mt_route_read(const mt_route &rt, int experts, mt_route_lds &l) {
    const int t = threadIdx.x, P = rt.tokens * rt.top_k;
    int e = t < P ? rt.idx[t] : 0;
    if (t < P) l.pair[t] = e;
    l.zero[t] = 0;
    if (t < MT_ROUTE_EXPERTS) l.count[t] = 0;
    if (t == 0) l.broken = 0;
    __syncthreads();
    if (t < P) {
        bool ok = (unsigned)e < (unsigned)experts;
        for (int j = t % rt.top_k; j > 0; --j) ok = ok && l.pair[t - j] != e;
        if (!ok) l.broken = 1;
    }
    __syncthreads();
    if (l.broken) {  // a token a thread, its entries in order
        if (t < rt.tokens) {
            int *mine = l.pair + t * rt.top_k;
            auto taken = [&](int x, int k) {
                bool is = false;
                for (int j = 0; j < k; ++j) is |= mine[j] == x;
                return is;
            };
            for (int k = 0; k < rt.top_k; ++k) {
                int x = mine[k];
                if ((unsigned)x < (unsigned)experts && !taken(x, k)) continue;
                x = 0;
                while (taken(x, k)) ++x;  // top_k <= experts: a free expert exists
                mine[k] = x;
                l.zero[t * rt.top_k + k] = 1;
            }
        }
        __syncthreads();
        e = l.pair[t < P ? t : 0];
    }
    if (t < P) atomicAdd(&l.count[e], 1);
    __syncthreads();
}
// Running sum over a wavefront's lanes.
__device__ __forceinline__ int mt_wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, true);  // row_bcast 15 into rows 1 and 3, then 31 into rows 2 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, true);
    return v;
}
// What the later launches read, by one workgroup.
__device__ __forceinline__ void mt_route_write(const mt_route &rt, int experts, const mt_route_lds &l) {
    const int t = threadIdx.x, lane = t & 63, P = rt.tokens * rt.top_k;
    if (t < P) {
        rt.topk_idx[t] = l.pair[t];
        rt.topk_p[t] = l.zero[t] ? 0.0f : rt.w[t];
    }
    if (t < 64) {
        const int c = lane < experts ? l.count[lane] : 0, tiles = (c + rt.tile - 1) / rt.tile, through = mt_wave_scan(tiles);
        if (lane < experts) {
            rt.counts[lane] = c;
            rt.goff[lane] = through - tiles;
        }
        if (lane == 63) rt.goff[experts] = through;
    }
    for (int e = t >> 6; e < experts; e += 4) {
        int base = 0;
        for (int p0 = 0; p0 < P; p0 += 64) {
            const int p = p0 + lane;
            const bool own = p < P && l.pair[p] == e;
            const unsigned long long mask = __ballot(own);
            if (own) rt.lists[(size_t)e * rt.tokens + base + __popcll(mask & ((1ull << lane) - 1ull))] = p;
            base += __popcll(mask);
        }
    }
}
// mt_find from the counts, and the pairs of 16 slots of the tile (slot `first` of its expert on) in l.slots.
__device__ __forceinline__ mt_place mt_route_find(const mt_route &rt, int experts, mt_route_lds &l, int gt, int sub) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, P = rt.tokens * rt.top_k;
    const int c = lane < experts ? l.count[lane] : 0, tiles = (c + rt.tile - 1) / rt.tile, through = mt_wave_scan(tiles);
    const unsigned long long here = __ballot(through - tiles <= gt && gt < through);
    mt_place at = {-1, 0, 0};
    if (!here) return at;
    at.expert = __ffsll((unsigned long long)here) - 1;
    at.first_tile = __builtin_amdgcn_readlane(through - tiles, at.expert);
    at.used = __builtin_amdgcn_readlane(c, at.expert);
    const int first = (gt - at.first_tile) * rt.tile + 16 * sub;
    int base = 0;
    for (int p0 = 0; p0 < P; p0 += 64) {
        const int p = p0 + lane;
        const bool own = p < P && l.pair[p] == at.expert;
        const unsigned long long mask = __ballot(own);
        const int slot = base + __popcll(mask & ((1ull << lane) - 1ull)) - first;
        if (own && (unsigned)slot < 16u) l.slots[wave][slot] = (uint16_t)p;
        base += __popcll(mask);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (its LDS accesses happen in order)
    return at;
}

// One thread = 16 consecutive k of one token (half a block).  A wavefront = the 16 tokens of a group x two blocks x
// their halves, tokens on consecutive lanes: what it writes are whole 256- and 128-byte runs of the records, and the
// 256 bytes it reads of every token row are two full lines.
// GATHER: the token groups are the experts' slots (mt_gather) instead of the rows in order.
// SWIGLU: x holds mlp1's outputs, [pairs][2 * 32 nb], and the values are their bias and swiglu, made on the way (a launch
// and a round trip of the pairs' rows less: 11.4 -> 8.1 us for 80 pairs of 2880).
// ROUTE: the routing too (mt_route), by workgroup 0 and, each for itself, the others.
template <bool GATHER, bool SWIGLU = false, bool ROUTE = false>
__global__ __launch_bounds__(256) void mxfp4_planes_kernel(const float *__restrict__ x, int m, int nb, int ncp, int token_groups,
                                                           char *__restrict__ bq, const mt_gather gat, const mt_swiglu act, const mt_route rt) {
    static_assert((GATHER || !SWIGLU) && (GATHER || !ROUTE) && !(SWIGLU && ROUTE), "pairs have experts, the first product's a routing to make");
    const float *bias = nullptr;
    __shared__ std::conditional_t<ROUTE, mt_route_lds, char> route;
    if constexpr (ROUTE) {
        mt_route_read(rt, gat.experts, route);
        if (blockIdx.x == 0) {
            mt_route_write(rt, gat.experts, route);
            return;
        }
    }
    const size_t wv = ((size_t)(blockIdx.x - (ROUTE ? 1 : 0)) * 256 + threadIdx.x) >> 6;  // (token group, pair of blocks)
    const int lane = threadIdx.x & 63, col = lane & 15, sub = (lane >> 4) & 1, npair = 2 * ncp;
    const size_t tg = wv / npair;
    if (tg >= (size_t)token_groups) return;  // (whole wavefronts)
    const int b = 2 * (int)(wv % npair) + (lane >> 5);
    size_t t = tg * 16 + col;
    bool valid = t < (size_t)m && b < nb;
    if (GATHER) {
        const int gt = (int)(tg / gat.tb);
        mt_place at;
        if constexpr (ROUTE) at = mt_route_find(rt, gat.experts, route, __builtin_amdgcn_readfirstlane(gt), __builtin_amdgcn_readfirstlane((int)(tg % gat.tb)));
        else at = mt_find(gat, __builtin_amdgcn_readfirstlane(gt));
        const int e = at.expert;
        if (e < 0) return;  // past the last expert's tiles (whole wavefronts)
        const int slot = ((gt - at.first_tile) * gat.tb + (int)(tg % gat.tb)) * 16 + col;
        valid = slot < at.used && b < nb;
        if constexpr (ROUTE) t = valid ? (size_t)(route.slots[threadIdx.x >> 6][col] / gat.div) : 0;
        else t = valid ? (size_t)(gat.lists[(size_t)e * gat.stride + slot] / gat.div) : 0;
        if (SWIGLU) bias = act.bias_tab[e];
    }
    float f[16];
    if constexpr (SWIGLU) {
#pragma unroll
        for (int e = 0; e < 16; ++e) f[e] = 0.0f;
        if (valid) {
            const int at = (b * 8 + sub * 4) * 2;  // in float4s: 16 pairs (gate, linear)
            float4 hv[8], bv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) hv[e] = reinterpret_cast<const float4 *>(x)[t * nb * 16 + at + e];
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[e] = reinterpret_cast<const float4 *>(bias)[at + e];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[2 * e] = mt_swiglu::of(hv[e].x + bv[e].x, hv[e].y + bv[e].y, act.alpha, act.clamp);
                f[2 * e + 1] = mt_swiglu::of(hv[e].z + bv[e].z, hv[e].w + bv[e].w, act.alpha, act.clamp);
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (valid) v = reinterpret_cast<const float4 *>(x)[(t * nb + b) * 8 + sub * 4 + e];
            f[4 * e] = v.x; f[4 * e + 1] = v.y; f[4 * e + 2] = v.z; f[4 * e + 3] = v.w;
        }
    }
    float amax = 0.0f;
    int bad = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        amax = fmaxf(amax, fabsf(f[e]));
        bad |= f[e] != f[e];
    }
    amax = fmaxf(amax, __shfl_xor(amax, 16, 64));  // the block's other half
    bad |= __shfl_xor(bad, 16, 64);
    int se = 0;
    float inv = 1.0f;
    if (bad || !(amax <= 3.4028234663852886e38f)) {
        bad = 1;
        inv = 0.0f;
    } else if (amax > 0.0f) {
        int ex;
        (void)frexpf(amax, &ex);          // amax = f * 2^ex, f in [0.5, 1)
        se = ex - (5 * MT_PLANES - 1);    // |x| / 2^se < 2^19 <= 16 (1 + 32 + 32^2 + 32^3)
        if (se < -126) se = -126;
        inv = ldexpf(1.0f, -se);
    }
    // Balanced base-32 digits, top down and all in f32 (every value is a small integer times a power of two, so
    // each step is exact): n_j = round(r / 32^j), r -= n_j 32^j; |n_j| <= 16.  Small integers keep the
    // instruction's own sum over k exact, which numbers spread over the format's exponent range do not (a split
    // into E4M3 values of decreasing size, four significant bits a plane, stopped at 2e-4 of the output's rms
    // however many planes it was given).
    float r[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const float tt = f[e] * inv;
        r[e] = (tt != tt) ? 0.0f : rintf(tt);
    }
    char *const head = bq + pg_mt_plane_store(tg, ncp, b, col, 0), *const tail = bq + pg_mt_plane_tail(tg, ncp, b, col, 0);
#pragma unroll
    for (int j = MT_PLANES - 1; j >= 0; --j) {
        // The conversion takes two runs of 16 and interleaves them: even elements, odd elements; this thread's sixteen are the first
        // 96 bits.  Integers in [-16, 16] over the scale of 8 are exact in E2M3.
        v16f even = {}, odd = {};
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            float d = r[e];
            if (j > 0) {
                const float down = __builtin_bit_cast(float, (127 - 5 * j) << 23), up = -__builtin_bit_cast(float, (127 + 5 * j) << 23);
                d = rintf(r[e] * down);
                r[e] = fmaf(d, up, r[e]);
            }
            if (e & 1) odd[e >> 1] = d;
            else even[e >> 1] = d;
        }
        const v6i pk = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, 8.0f);
        if (sub == 0) {
            *reinterpret_cast<v3i *>(head + j * MT_FRAG) = v3i{pk[0], pk[1], pk[2]};
        } else {
            *reinterpret_cast<int *>(head + j * MT_FRAG + 12) = pk[0];
            *reinterpret_cast<v2i *>(tail + j * MT_FRAG) = v2i{pk[1], pk[2]};
        }
    }
    if (sub == 0) {  // a NaN / inf block poisons every product it enters: scale byte 255 is NaN
        unsigned word = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) word |= (unsigned)(j >= MT_PLANES ? 127 : (bad ? 255 : 130 + se + 5 * j)) << (8 * j);
        *reinterpret_cast<unsigned *>(bq + pg_mt_scale_store(tg, ncp, b, col)) = word;
    }
}

// A workgroup = NW wavefronts x RA groups of 16 weight rows, against TB groups of 16 tokens, over one run of
// chunks (all of K, or one of `ks` runs whose partial tiles a later launch adds).  The weights go from memory
// straight into the A operand's registers, a ring of two chunks for the widest row tile and of four otherwise; the token records of
// a chunk are shared through LDS (staged through registers BD chunks ahead, two stages, one barrier per chunk).  Narrow tiles do
// little arithmetic per chunk, so what they need is requests in flight: the deeper staging is theirs.
// GROUPED: the token tiles are the experts' (mt_gather), the weights come from the expert's entry of two pointer
// tables, an output row is the pair the slot holds; one run of K.
// Weights that several tiles read are loaded plainly, the others with the hint that nothing reads them again: hinted, they left the
// L2 before the next tile came (480 tokens over 8 experts of 2048 x 2048, top 4: the two products 83 + 57 us, plain 78 + 54; but 90
// tokens over 32 of 2880 x 2880, one tile an expert, 67 + 36 hinted and 72 + 42 plain).
// What bounds a many-token product now is the matrix cores at about half their rate, the rest a chunk's barrier and LDS reads and
// the last, partly filled round.  421 tokens over 8 experts of 1280 x 1376, top 4, us: 42.4 + 29.8 in FP8 digits and batches
// of chunks under conditions; FP6 37.6 + 26.7; loads without conditions, plain and in XCD order, 25.8 + 19.4.  The 480 tokens above:
// 86 + 57, 74 + 47, 66 + 43, and on four wavefronts instead of eight 50 + 31.
struct mt_experts {
    const uint8_t *const *qs_tab;
    const uint32_t *const *sc_tab;
};

// A token tile with at most 16 / NPM slots in use: the spare columns of the B operand take NPM planes of each token (column
// = token * NPM + plane), so a chunk is 4 / NPM instructions instead of four, and only the operand bytes of those tokens
// pass through LDS, a batch of four chunks at a time (one barrier a batch).  The planes' sums are joined at the end.
// Bound by the weights' stream: twenty tokens over 32 experts of 2880 x 2880, top 4 (2.7 slots a tile), 250 and 125 MB in 49 and
// 27.6 us, 5.1 and 4.5 TB/s (as full tiles 71 + 40; with the next batch beside the current one in registers, copied, 51 + 30.5;
// scales by flat loads and the ring 51 + 28.8): a ring keeps four chunks under way at every moment and takes 95 registers
// where two batches took 128.
template <int RA, int NPM>
__device__ __forceinline__ void mxfp4_narrow_tile(char *lds, const gv4i_ptr qa, const gu32_ptr sa, const char *__restrict__ bq,
                                                  int ncp, int turn, v4f (&acc)[RA]) {
    constexpr int NI = MT_PLANES / NPM, CHUNK = NI * MT_FRAG + 256, STAGE = 4 * CHUNK;
    const int lane = threadIdx.x & 63, t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t a_stride = (size_t)ncp * 64;
    // this thread's units of a batch: operand unit (chunk t / 128, first 16 or last 8 bytes, lane) of every instruction, and a unit of
    // the scales; of the last 8 bytes it reads the 16 that they are a half of
    const int oc = t >> 7, ol = t & 63, ocol = ol & 15, from = ocol / NPM + 16 * (ol >> 4);
    const bool last8 = (wave & 1) != 0;
    const unsigned o_src = (unsigned)oc * MT_RECORD + (ocol % NPM) * MT_FRAG + (last8 ? 1024 + (from >> 1) * 16 : from * 16);
    const unsigned o_dst = (unsigned)oc * CHUNK + (last8 ? 1024 + ol * 8 : ol * 16);
    const unsigned s_src = (unsigned)(lane >> 4) * MT_RECORD + MT_PLANES * MT_FRAG + (lane & 15) * 16;
    const unsigned s_dst = (unsigned)(lane >> 4) * CHUNK + NI * MT_FRAG + (lane & 15) * 16;
    v4i so[NI], ss;
    auto fetch_b = [&](int c) {
        const char *at = bq + (size_t)c * MT_RECORD;
#pragma unroll
        for (int i = 0; i < NI; ++i) so[i] = *reinterpret_cast<const v4i *>(at + o_src + i * NPM * MT_FRAG);
        ss = *reinterpret_cast<const v4i *>(at + s_src);
    };
    auto put_b = [&](int stage) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            char *const at = lds + stage * STAGE + o_dst + i * MT_FRAG;
            if (last8) *reinterpret_cast<v2i *>(at) = from & 1 ? v2i{so[i][2], so[i][3]} : v2i{so[i][0], so[i][1]};
            else *reinterpret_cast<v4i *>(at) = so[i];
        }
        if (wave == 0) *reinterpret_cast<v4i *>(lds + stage * STAGE + s_dst) = ss;
    };
    auto chunk_at = [&](int i) { return i + turn < ncp ? i + turn : i + turn - ncp; };
    v4i a[4][RA];  // a ring: a chunk's weights are read as soon as the same place of the batch before is used
    uint32_t sca[RA], sca_next[RA];
    auto fetch_a = [&](int u, int c) {
#pragma unroll
        for (int r = 0; r < RA; ++r) a[u][r] = __builtin_nontemporal_load(qa + (size_t)r * a_stride + (size_t)(c + u) * 64 + lane);
    };
    auto fetch_s = [&](uint32_t (&sc)[RA], int c) {
#pragma unroll
        for (int r = 0; r < RA; ++r) sc[r] = sa[((size_t)r * (ncp / 4) + (c >> 2)) * 64 + lane];
    };
    const int col = lane & 15;
    const unsigned sc_at = NI * MT_FRAG + (col / NPM + 16 * (lane >> 4)) * 4, shift = 8 * (col % NPM);
#pragma unroll
    for (int r = 0; r < RA; ++r) acc[r] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    fetch_b(chunk_at(0));
    fetch_s(sca, chunk_at(0));
#pragma unroll
    for (int u = 0; u < 4; ++u) fetch_a(u, chunk_at(0));
    put_b(0);
    fetch_b(chunk_at(4 < ncp ? 4 : 0));
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
    auto batch = [&](int cb, int s, auto last_) {
        constexpr bool LAST = decltype(last_)::value;
        const int next = chunk_at(cb + 4 < ncp ? cb + 4 : 0);
        if (!LAST) fetch_s(sca_next, next);
        const char *st = lds + s * STAGE;
#define PG_MT_STEP(U, I)                                                                                                   \
    do {                                                                                                                   \
        const v4i b0 = *reinterpret_cast<const v4i *>(st + (U) * CHUNK + (I) * MT_FRAG + lane * 16);                       \
        const v2i b1 = *reinterpret_cast<const v2i *>(st + (U) * CHUNK + (I) * MT_FRAG + 1024 + lane * 8);                 \
        const int sb = (int)(*reinterpret_cast<const unsigned *>(st + (U) * CHUNK + sc_at) >> shift);                      \
        const v8i B = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], 0, 0};                                                    \
        _Pragma("unroll") for (int r = 0; r < RA; ++r) {                                                                   \
            const v4i aw = a[U][r];                                                                                        \
            const v8i A = {aw[0], aw[1], aw[2], aw[3], 0, 0, 0, 0};                                                        \
            acc[r] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, acc[r], 4, 2, (U), (int)sca[r], NPM * (I), sb); \
            asm volatile("" : "+v"(acc[r]) : : "memory");  /* (or every chunk's operands are read first: 32 to 64 registers) */ \
        }                                                                                                                  \
    } while (0)
#define PG_MT_STEPS(U)                      \
    do {                                    \
        PG_MT_STEP(U, 0);                   \
        if constexpr (NI == 2) PG_MT_STEP(U, 1); \
        if (!LAST) fetch_a(U, next);        \
        __builtin_amdgcn_sched_barrier(0);  \
    } while (0)
        static_assert(NI == 1 || NI == 2, "the instructions of a chunk are written out");
        PG_MT_STEPS(0);
        PG_MT_STEPS(1);
        PG_MT_STEPS(2);
        PG_MT_STEPS(3);
#undef PG_MT_STEPS
#undef PG_MT_STEP
        if (!LAST) {
            put_b(s ^ 1);
            fetch_b(chunk_at(cb + 8 < ncp ? cb + 8 : 0));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");  // (not __syncthreads(): the loads stay in flight)
        if (!LAST) {
#pragma unroll
            for (int r = 0; r < RA; ++r) sca[r] = sca_next[r];
        }
    };
    int s = 0;
#pragma unroll 1
    for (int cb = 0; cb + 4 < ncp; cb += 4, s ^= 1) batch(cb, s, std::false_type{});
    batch(ncp - 4, s, std::true_type{});
#pragma unroll
    for (int r = 0; r < RA; ++r)  // every lane of a token's columns: the sum over the planes
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = acc[r][i];
            v += __shfl_xor(v, 1, 64);
            if (NPM == 4) v += __shfl_xor(v, 2, 64);
            acc[r][i] = v;
        }
}

template <typename F, int... I>
__device__ __forceinline__ void mt_steps(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

template <int RA, int TB, int BD, bool GROUPED, int NW = MT_NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(GROUPED && TB == 1 && RA <= 2 ? 4 : 2))) void mxfp4_tiles_kernel(const uint8_t *__restrict__ qs_frag, const uint32_t *__restrict__ sc_frag,
                                                                 const char *__restrict__ bq, float *__restrict__ y, int n_out,
                                                                 int ncp, int m, int n_tt, int ks, int cps, size_t part_stride,
                                                                 int items, int per_xcd, const mt_gather gat, const mt_experts ex) {
    constexpr int STAGE = TB * MT_RECORD, UNITS = TB * MT_UNITS, ROUNDS = (UNITS + 64 * NW - 1) / (64 * NW);
    constexpr bool NT = TB == 1 || (!GROUPED && TB == 2);
    constexpr int DA = RA == 4 ? 2 : 4;  // weights read ahead, in chunks: a ring of registers
    constexpr int AHEAD = RA == 1 && TB > 1 ? 3 : 1;  // planes read ahead: the fewer products a plane feeds, the less of the LDS latency they cover
    static_assert(BD == 1 || BD == 2 || BD == 4, "the staging depth divides the unrolled batch");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // every XCD (workgroup id % 8) walks its own run of work items, token tiles of one row tile and K run first:
    // that run's weights stay in the XCD's L2 while its token tiles pass
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;
    int tt = item % n_tt, split = (item / n_tt) % ks, wt = item / (n_tt * ks), live = TB;
    mt_place at = {0, 0, 0};
    if (GROUPED) {  // n_tt = the row tiles here
        const int slot = (int)(blockIdx.x >> 3);
        split = 0;
        if (TB > 1) {  // every XCD walks its own run of tiles in order: an expert's weights are read by one or two of the eight
            const int all = gat.goff[gat.experts] * n_tt, mine = (all + 7) / 8, it = (int)(blockIdx.x & 7) * mine + slot;
            if (slot >= mine || it >= all) return;
            tt = it / n_tt;
            wt = it % n_tt;
        } else {  // hardly an expert has a second tile: token tile 8 i + x belongs to XCD x (the unused tail tiles spread evenly)
            tt = (slot / n_tt) * 8 + (int)(blockIdx.x & 7);
            wt = slot % n_tt;
        }
        at = mt_find(gat, tt);
        if (at.expert < 0) return;
        qs_frag = ex.qs_tab[at.expert];
        sc_frag = ex.sc_tab[at.expert];
        // an expert's last tile is rarely full: token groups without a slot in use are skipped (their records hold zeros)
        const int left = at.used - (tt - at.first_tile) * TB * 16;
        live = __builtin_amdgcn_readfirstlane(left >= TB * 16 ? TB : (left + 15) / 16);
    }
    const int kc0 = split * cps, run = pg_mt_run_end(split, cps, ncp) - kc0;  // whole batches of four chunks
    // Row groups lie a whole tensor row of chunks apart (24 KB for K = 2880): walked from the same end they would all be at the
    // same few memory channels at a time, so every row tile begins at a batch of its own and wraps round (71 -> 66 us for
    // the 250 MB of 30 experts' mlp1, before the narrow tiles).
    const int turn = 4 * (wt % (run >> 2));
    auto chunk_at = [&](int i) {  // the i-th chunk of the walk
        i += turn;
        return kc0 + (i < run ? i : i - run);
    };
    const int nrg = (n_out + 15) / 16;                       // >= RA (the launcher's choice of RA)
    const int rg_mine = (wt * NW + wave) * RA;            // the row groups whose tiles this wavefront stores
    const int rg0 = pg_mt_first_row_group(rg_mine, RA, nrg);  // the ones it reads: a spare wavefront repeats the last ones
    const size_t a_stride = (size_t)ncp * 64;                // v4i per row group
    const gv4i_ptr qa = (gv4i_ptr)(uintptr_t)qs_frag + (size_t)rg0 * a_stride;
    const gu32_ptr sa = (gu32_ptr)(uintptr_t)sc_frag + (size_t)rg0 * (ncp / 4) * 64;
    if constexpr (GROUPED && TB == 1) {
        const int first = (tt - at.first_tile) * 16, used = at.used - first;
        if (used <= 8) {
            v4f sum[RA];
            const char *const rec = bq + (size_t)tt * ncp * MT_RECORD;
            if (used <= 4) mxfp4_narrow_tile<RA, 4>(lds, qa, sa, rec, ncp, turn, sum);
            else mxfp4_narrow_tile<RA, 2>(lds, qa, sa, rec, ncp, turn, sum);
            const int npm = used <= 4 ? 4 : 2, slot = (lane & 15) / npm;
            if ((lane & 15) % npm != 0 || slot >= used || rg_mine >= nrg) return;
            const size_t token = (size_t)gat.lists[(size_t)at.expert * gat.stride + first + slot];
#pragma unroll
            for (int r = 0; r < RA; ++r) {
                if (rg0 + r < rg_mine) continue;  // rows a spare wavefront only repeated
                const size_t row = (size_t)(rg0 + r) * 16 + 4 * (lane >> 4);
                float *o = y + token * n_out + row;
                if (row + 3 < (size_t)n_out && (n_out & 3) == 0) {
                    *reinterpret_cast<v4f *>(o) = sum[r];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (row + i < (size_t)n_out) o[i] = sum[r][i];
                }
            }
            return;
        }
    }
    // this thread's share of a chunk's records: 16-byte unit u of the TB records, which lie ncp records apart
    const char *const b_base = bq + (size_t)tt * TB * ncp * MT_RECORD;
    unsigned b_off[ROUNDS];
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) b_off[i] = pg_mt_unit_offset((int)threadIdx.x + i * 64 * NW, UNITS, ncp);
    v4i sr[BD][ROUNDS];
#define PG_MT_FETCH_B(SLOT, C)                                                                                          \
    do {                                                                                                                \
        _Pragma("unroll") for (int i = 0; i < ROUNDS; ++i)                                                              \
            sr[SLOT][i] = *reinterpret_cast<const v4i *>(b_base + b_off[i] + (unsigned)(C) * MT_RECORD), __builtin_amdgcn_sched_barrier(0); \
    } while (0)
#define PG_MT_PUT_B(STG, SLOT)                                                                                          \
    do {                                                                                                                \
        _Pragma("unroll") for (int i = 0; i < ROUNDS; ++i) {                                                            \
            const int u = (int)threadIdx.x + i * 64 * NW;                                                            \
            if ((i + 1) * 64 * NW <= UNITS || u < UNITS) *reinterpret_cast<v4i *>(lds + (STG) * STAGE + u * 16) = sr[SLOT][i]; \
        }                                                                                                               \
    } while (0)
    v4i a[DA][RA];
    uint32_t sca[RA], sca_next[RA];
    auto fetch_a = [&](v4i (&dst)[RA], int c) {
#pragma unroll
        for (int r = 0; r < RA; ++r) dst[r] = NT ? __builtin_nontemporal_load(qa + (size_t)r * a_stride + (size_t)c * 64 + lane) : qa[(size_t)r * a_stride + (size_t)c * 64 + lane];
    };
    v4f acc[RA][TB];
#pragma unroll
    for (int r = 0; r < RA; ++r)
#pragma unroll
        for (int g = 0; g < TB; ++g) acc[r][g] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    const int c0 = chunk_at(0);
    PG_MT_FETCH_B(0, c0);
    if (BD > 1) PG_MT_FETCH_B(BD > 1 ? 1 : 0, c0 + 1);
    if (BD > 2) {
        PG_MT_FETCH_B(BD > 2 ? 2 : 0, c0 + 2);
        PG_MT_FETCH_B(BD > 2 ? 3 : 0, c0 + 3);
    }
#pragma unroll
    for (int u = 0; u < DA; ++u) fetch_a(a[u], c0 + u);
#pragma unroll
    for (int r = 0; r < RA; ++r) sca[r] = sa[((size_t)r * (ncp / 4) + (c0 >> 2)) * 64 + lane];
    PG_MT_PUT_B(0, 0);
    if (BD < run) PG_MT_FETCH_B(0, chunk_at(BD));
    __syncthreads();
    // Which loads a batch makes is known when it is compiled (the last batch is code of its own): with a condition around them the
    // compiler cannot count what is under way, and a chunk's weights waited for everything that was read after them as well.
    auto batch = [&](int cb, auto last_) {
        constexpr bool LAST = decltype(last_)::value;
        if (!LAST) {
            const int next = chunk_at(cb + 4);
#pragma unroll
            for (int r = 0; r < RA; ++r) sca_next[r] = sa[((size_t)r * (ncp / 4) + (next >> 2)) * 64 + lane];
        }
        // One step = one plane of one token group against the wavefront's RA row groups; the operand halves of the plane AHEAD steps on
        // are read meanwhile.  (The byte selectors of the two scale operands are immediates: chunk within the dword, plane within the dword.)
        auto chunk = [&](auto u_) {
            constexpr int U = decltype(u_)::value;
            const int c = cb + U;
            const char *st = lds + (U & 1) * STAGE;
            int sbv[TB];
#pragma unroll
            for (int g = 0; g < TB; ++g) sbv[g] = *reinterpret_cast<const int *>(st + g * MT_RECORD + MT_PLANES * MT_FRAG + lane * 4);
            v4i b[AHEAD + 1];
            v2i bt[AHEAD + 1];
            auto read = [&](int step) {
                const char *f = st + step / MT_PLANES * MT_RECORD + step % MT_PLANES * MT_FRAG;
                b[step % (AHEAD + 1)] = *reinterpret_cast<const v4i *>(f + lane * 16);
                bt[step % (AHEAD + 1)] = *reinterpret_cast<const v2i *>(f + 1024 + lane * 8);
            };
            auto step = [&](auto i_) {
                constexpr int I = decltype(i_)::value, G = I / MT_PLANES, J = I % MT_PLANES;
                if (GROUPED && G >= live) return;
                if (I + AHEAD < TB * MT_PLANES) read(I + AHEAD);
                const v4i b0 = b[I % (AHEAD + 1)];
                const v2i b1 = bt[I % (AHEAD + 1)];
                const v8i B = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], 0, 0};
#pragma unroll
                for (int r = 0; r < RA; ++r) {
                    const v4i aw = a[U % DA][r];
                    const v8i A = {aw[0], aw[1], aw[2], aw[3], 0, 0, 0, 0};
                    acc[r][G] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, acc[r][G], 4, 2, U, (int)sca[r], J, sbv[G]);
                    asm volatile("" : "+v"(acc[r][G]));  /* (or the compiler sinks every product to the end of the loop body) */
                }
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) read(i);
            __builtin_amdgcn_sched_barrier(0);
            mt_steps(step, std::make_integer_sequence<int, TB * MT_PLANES>{});
            if (!LAST || U < 3) {
                PG_MT_PUT_B((U + 1) & 1, (U + 1) % BD);
                __builtin_amdgcn_sched_barrier(0);
                if (!LAST || U + 1 + BD < 4) PG_MT_FETCH_B((U + 1) % BD, chunk_at(c + 1 + BD < run ? c + 1 + BD : run - 1));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!LAST || U + DA < 4) fetch_a(a[U % DA], chunk_at(c + DA));
            asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");  // (the loads stay in flight)
        };
        mt_steps(chunk, std::make_integer_sequence<int, 4>{});
        if (!LAST) {
#pragma unroll
            for (int r = 0; r < RA; ++r) sca[r] = sca_next[r];
        }
    };
#pragma unroll 1
    for (int cb = 0; cb + 4 < run; cb += 4) batch(cb, std::false_type{});
    batch(run - 4, std::true_type{});
#undef PG_MT_FETCH_B
#undef PG_MT_PUT_B
    // D: lane holds token lane % 16 of its group, weight rows 4 (lane / 16) .. + 3 of the row group
    float *const out = y + (size_t)split * part_stride;
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        if (rg_mine != rg0 && rg0 + r < rg_mine) continue;   // rows a spare wavefront only repeated
        if (rg_mine >= nrg) continue;
        const size_t row = (size_t)(rg0 + r) * 16 + 4 * (lane >> 4);
#pragma unroll
        for (int g = 0; g < TB; ++g) {
            size_t token = ((size_t)tt * TB + g) * 16 + (lane & 15);
            if (GROUPED) {
                const int slot = ((tt - at.first_tile) * TB + g) * 16 + (lane & 15);
                if (slot >= at.used) continue;
                token = (size_t)gat.lists[(size_t)at.expert * gat.stride + slot];
            } else if (token >= (size_t)m) {
                continue;
            }
            float *o = out + token * n_out + row;
            if (row + 3 < (size_t)n_out && (n_out & 3) == 0) {
                *reinterpret_cast<v4f *>(o) = acc[r][g];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row + i < (size_t)n_out) o[i] = acc[r][g][i];
            }
        }
    }
}

using mt_plan = pg_mxfp4_tiles_plan;

template <int RA, int TB, int BD>
pg_status launch_tiles(pg_ctx *ctx, const pg_gguf_tensor *w, const char *bq, float *y, size_t m, int ncp, const mt_plan &p) {
    const size_t lds = 2 * (size_t)TB * MT_RECORD;
    auto kern = mxfp4_tiles_kernel<RA, TB, BD, false>;
    PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));
    const size_t items = p.n_wt * p.n_tt * p.ks, per_xcd = (items + 7) / 8;
    return pg_launch(ctx, "mxfp4_tiles", kern, dim3((unsigned)(8 * per_xcd)), dim3(64 * MT_NW), lds, (const uint8_t *)w->qs,
                     reinterpret_cast<const uint32_t *>(w->d), bq, y, (int)w->n_out, ncp, (int)m, (int)p.n_tt, p.ks, p.cps,
                     m * w->n_out, (int)items, (int)per_xcd, mt_gather{}, mt_experts{});
}

// The grouped form: `max_tiles` token tiles at most (the launch covers them all; those past the experts' last exit).
template <int RA, int TB, int BD, int NW = MT_NW>
pg_status launch_tiles_grouped(pg_ctx *ctx, size_t n_out, int ncp, const char *bq, float *y, size_t n_wt, size_t max_tiles,
                               const mt_gather &gat, const mt_experts &ex) {
    const size_t lds = TB == 1 ? std::max<size_t>(2 * MT_RECORD, 2 * 4 * (2 * MT_FRAG + 256)) : 2 * (size_t)TB * MT_RECORD;  // (mxfp4_narrow_tile<RA, 2>)
    auto kern = mxfp4_tiles_kernel<RA, TB, BD, true, NW>;
    PG_TRY(pg_allow_dynamic_lds(ctx, (const void *)kern, lds));
    const size_t per_xcd = (max_tiles + 7) / 8 * n_wt, items = 8 * per_xcd;
    return pg_launch(ctx, "mxfp4_tiles_grouped", kern, dim3((unsigned)(8 * per_xcd)), dim3(64 * NW), lds, (const uint8_t *)nullptr,
                     (const uint32_t *)nullptr, bq, y, (int)n_out, ncp, 0, (int)n_wt, 1, ncp, (size_t)0, (int)items, (int)per_xcd, gat, ex);
}

}  // namespace

// The tile shape and K split for m rows of an [n_out, 32 nb] tensor: the widest row tile that still gives every CU a
// workgroup (and no wider than the tensor); with the narrowest still short of that, K in runs of at least 8 chunks.
pg_mxfp4_tiles_plan pg_mxfp4_tiles_plan_for(int num_cu, size_t n_out, size_t m, int ncp) {
    pg_mxfp4_tiles_plan p;
    p.tb = m <= 16 ? 1 : (m <= 32 ? 2 : 4);
    p.n_tt = (m + 16 * p.tb - 1) / (16 * p.tb);
    p.groups = p.n_tt * p.tb;
    const size_t nrg = (n_out + 15) / 16;
    p.ra = 4;
    while (p.ra > 1 && ((size_t)p.ra > nrg || (nrg + MT_NW * p.ra - 1) / (MT_NW * p.ra) * p.n_tt < (size_t)num_cu)) p.ra >>= 1;
    p.n_wt = (nrg + MT_NW * p.ra - 1) / (MT_NW * p.ra);
    const size_t tiles = p.n_wt * p.n_tt;
    p.ks = 1;
    if (tiles < (size_t)num_cu) p.ks = (int)std::min<size_t>(std::min<size_t>((size_t)num_cu / tiles, (size_t)ncp / 8), 16);
    if (p.ks < 1) p.ks = 1;
    p.cps = ((ncp / 4 + p.ks - 1) / p.ks) * 4;       // chunks per run: whole batches of four
    p.ks = (ncp + p.cps - 1) / p.cps;                // (no empty run)
    return p;
}

// Whether the tile kernel takes `m` activation rows of this tensor (otherwise the decode kernel's passes of three
// rows): from 16 rows, or 24 for a tensor under 2^25 weights, whose passes are short.
bool pg_mxfp4_tiles_takes(const pg_gguf_tensor *w, size_t m) {
    return w->ggml_type == PG_MXFP4 && m >= (w->n_out * w->k_in >= ((size_t)1 << 25) ? 16u : 24u) && m < ((size_t)1 << 27) &&
           w->n_out < ((size_t)1 << 27);
}

// y[m, n_out] = x[m, k_in] . W^T for an MXFP4 tensor over many rows; x 16-byte aligned.
pg_status pg_launch_mxfp4_tiles(pg_ctx *ctx, const float *x_dev, size_t m, const pg_gguf_tensor *w, float *y_dev) {
    const int nb = (int)(w->k_in / 32), ncp = (int)mx_chunks((size_t)nb);
    const mt_plan p = pg_mxfp4_tiles_plan_for(ctx->num_cu, w->n_out, m, ncp);
    PG_CHECK_ARG(p.n_wt * p.n_tt * p.ks < ((size_t)1 << 28), "mxfp4: %zu x %zu tiles", p.n_wt, p.n_tt);
    void *ws = nullptr;
    const size_t sz_b = pg_round_up(p.groups * ncp * (size_t)MT_RECORD, 256);
    const size_t sz_part = p.ks > 1 ? (size_t)p.ks * m * w->n_out * sizeof(float) : 0;
    PG_TRY(pg_workspace(ctx, sz_b + sz_part, &ws));
    char *bq = static_cast<char *>(ws);
    float *part = p.ks > 1 ? reinterpret_cast<float *>(bq + sz_b) : y_dev;
    const size_t threads = p.groups * 2 * (size_t)ncp * 64;  // a wavefront per token group and pair of blocks
    PG_CHECK_ARG((threads + 255) / 256 < ((size_t)1 << 31), "mxfp4: %zu rows x %zu is too much for one pre-pass", m, w->k_in);
    PG_TRY(pg_launch(ctx, "mxfp4_planes", mxfp4_planes_kernel<false>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, x_dev, (int)m, nb,
                     ncp, (int)p.groups, bq, mt_gather{}, mt_swiglu{}, mt_route{}));
    // the staging depth: the less arithmetic a chunk holds, the more chunks ahead
#define PG_MT_LAUNCH(RA_, BD1, BD2, BD4) \
    (p.tb == 1 ? launch_tiles<RA_, 1, BD1>(ctx, w, bq, part, m, ncp, p) \
     : p.tb == 2 ? launch_tiles<RA_, 2, BD2>(ctx, w, bq, part, m, ncp, p) \
                 : launch_tiles<RA_, 4, BD4>(ctx, w, bq, part, m, ncp, p))
    PG_TRY(p.ra == 4 ? PG_MT_LAUNCH(4, 4, 2, 1) : (p.ra == 2 ? PG_MT_LAUNCH(2, 4, 4, 2) : PG_MT_LAUNCH(1, 4, 4, 4)));
#undef PG_MT_LAUNCH
    if (p.ks > 1) PG_TRY(pg_launch_sum_parts(ctx, part, m * w->n_out, p.ks, m * w->n_out, y_dev));
    return PG_OK;
}

// ---- ABI --------------------------------------------------------------------------------
// A block is 16 bytes of FP4 (E2M1) codes, byte k = elements 2k (low nibble) and 2k+1, plus
// one E8M0 scale byte: value = LUT[code] * 2^(scale - 127)   (examples/gpt_oss/moe.rs:5-53).
PG_API pg_status pg_mxfp4_upload(pg_ctx *ctx, const uint8_t *blocks, const uint8_t *scales, size_t out_dim,
                                 size_t in_dim, pg_gguf_tensor **out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(out != nullptr, "pg_mxfp4_upload: out is null");
    *out = nullptr;
    PG_CHECK_ARG(out_dim > 0 && in_dim > 0 && blocks && scales, "pg_mxfp4_upload: empty tensor or null pointer");
    PG_CHECK_ARG(in_dim % 32 == 0, "pg_mxfp4_upload: in_dim %zu is not a multiple of 32", in_dim);
    PG_CHECK_ARG(out_dim < (1ull << 31) && in_dim < (1ull << 31) && out_dim * (in_dim / 32) < (1ull << 31),
                 "pg_mxfp4_upload: shape too large");
    const size_t nb = in_dim / 32, nblocks = out_dim * nb;
    const size_t ncp = mx_chunks(nb), nrg = (out_dim + 15) / 16;
    pg_gguf_tensor *t = new (std::nothrow) pg_gguf_tensor();
    if (!t) return pg_fail(PG_ENOMEM, "host allocation failed");
    t->qs = nullptr;
    t->d = nullptr;
    t->m = nullptr;
    t->qs_tiled = nullptr;
    t->ggml_type = PG_MXFP4;
    t->n_out = out_dim;
    t->k_in = in_dim;
    pg_tmp rb, rs;
    pg_status st = rb.alloc(ctx, nblocks * 16);
    if (st == PG_OK) st = rs.alloc(ctx, nblocks);
    hipError_t e = hipSuccess;
    if (st == PG_OK) {
        e = pg_dev_malloc(ctx, (void **)&t->qs, nrg * ncp * 64 * 16);
        if (e == hipSuccess) e = pg_dev_malloc(ctx, (void **)&t->d, nrg * (ncp / 4) * 64 * 4);
        if (e == hipSuccess) e = hipMemcpyAsync(rb.p, blocks, nblocks * 16, hipMemcpyHostToDevice, ctx->stream);
        if (e == hipSuccess) e = hipMemcpyAsync(rs.p, scales, nblocks, hipMemcpyHostToDevice, ctx->stream);
        if (e == hipSuccess) {
            mxfp4_fragments_kernel<<<grid_for(nrg * ncp * 64, 256), 256, 0, ctx->stream>>>(
                rb.as<uint8_t>(), rs.as<uint8_t>(), (int)out_dim, (int)nb, (int)ncp, reinterpret_cast<uint4 *>(t->qs),
                reinterpret_cast<uint8_t *>(t->d));
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess)
            st = pg_fail(e == hipErrorOutOfMemory ? PG_ENOMEM : PG_EDEVICE, "pg_mxfp4_upload: %s", hipGetErrorString(e));
    }
    if (st != PG_OK) { pg_gguf_free(ctx, t); return st; }
    *out = t;
    return PG_OK;
}

PG_API pg_status pg_mxfp4_matmul(pg_ctx *ctx, const float *input, const uint8_t *blocks, const uint8_t *scales,
                                 size_t out_dim, size_t in_dim, float *output) {
    pg_gguf_tensor *t = nullptr;
    PG_TRY(pg_mxfp4_upload(ctx, blocks, scales, out_dim, in_dim, &t));
    const pg_status st = pg_gguf_matmul(ctx, input, 1, t, output);
    pg_gguf_free(ctx, t);
    return st;
}

// Mxfp4Expert  examples/gpt_oss/moe.rs:55-117, swiglu :145-154.
struct pg_mxfp4_expert {
    pg_gguf_tensor *mlp1, *mlp2;  // [2 * intermediate, hidden], [hidden, intermediate]
    float *bias1, *bias2;         // [2 * intermediate], [hidden] (one allocation)
    size_t hidden, intermediate;
    float alpha, clamp;
};

namespace {
// biased = h + bias1, then the swiglu (mt_swiglu)
__global__ __launch_bounds__(256) void mxfp4_bias_swiglu_kernel(const float *__restrict__ h, const float *__restrict__ bias,
                                                                size_t rows, size_t inter, float alpha, float clamp,
                                                                float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * inter) return;
    const size_t r = i / inter, c = i - r * inter;
    out[i] = mt_swiglu::of(h[r * 2 * inter + 2 * c] + bias[2 * c], h[r * 2 * inter + 2 * c + 1] + bias[2 * c + 1], alpha, clamp);
}

__global__ __launch_bounds__(256) void bias_add_kernel(const float *__restrict__ a, const float *__restrict__ bias,
                                                       size_t rows, size_t cols, float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < rows * cols) out[i] = a[i] + bias[i % cols];
}
}  // namespace

PG_API void pg_mxfp4_expert_free(pg_ctx *ctx, pg_mxfp4_expert *e) {
    if (!e) return;
    if (ctx) {
        (void)pg_use(ctx);
        (void)hipStreamSynchronize(ctx->stream);
    }
    pg_gguf_free(ctx, e->mlp1);
    pg_gguf_free(ctx, e->mlp2);
    if (e->bias1) (void)hipFree(e->bias1);
    delete e;
}

PG_API pg_status pg_mxfp4_expert_create(pg_ctx *ctx, size_t hidden, size_t intermediate, float alpha, float clamp,
                                        const uint8_t *mlp1_blocks, const uint8_t *mlp1_scales,
                                        const uint8_t *mlp2_blocks, const uint8_t *mlp2_scales, const float *mlp1_bias,
                                        const float *mlp2_bias, pg_mxfp4_expert **out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(out != nullptr, "pg_mxfp4_expert_create: out is null");
    *out = nullptr;
    PG_CHECK_ARG(mlp1_bias && mlp2_bias, "pg_mxfp4_expert_create: null bias");
    pg_mxfp4_expert *e = new (std::nothrow) pg_mxfp4_expert{nullptr, nullptr, nullptr, nullptr, hidden, intermediate, alpha, clamp};
    if (!e) return pg_fail(PG_ENOMEM, "host allocation failed");
    pg_status st = pg_mxfp4_upload(ctx, mlp1_blocks, mlp1_scales, 2 * intermediate, hidden, &e->mlp1);
    if (st == PG_OK) st = pg_mxfp4_upload(ctx, mlp2_blocks, mlp2_scales, hidden, intermediate, &e->mlp2);
    if (st == PG_OK) {
        hipError_t he = pg_dev_malloc(ctx, (void **)&e->bias1, (2 * intermediate + hidden) * sizeof(float));
        if (he == hipSuccess) {
            e->bias2 = e->bias1 + 2 * intermediate;
            he = hipMemcpyAsync(e->bias1, mlp1_bias, 2 * intermediate * sizeof(float), hipMemcpyHostToDevice, ctx->stream);
        }
        if (he == hipSuccess) he = hipMemcpyAsync(e->bias2, mlp2_bias, hidden * sizeof(float), hipMemcpyHostToDevice, ctx->stream);
        if (he == hipSuccess) he = hipStreamSynchronize(ctx->stream);
        if (he != hipSuccess)
            st = pg_fail(he == hipErrorOutOfMemory ? PG_ENOMEM : PG_EDEVICE, "pg_mxfp4_expert_create: %s", hipGetErrorString(he));
    }
    if (st != PG_OK) { pg_mxfp4_expert_free(ctx, e); return st; }
    *out = e;
    return PG_OK;
}

// scratch_dev: [m, 3 * intermediate] floats (the mlp1 output, then the activated rows).
PG_API pg_status pg_mxfp4_expert_forward_dev(pg_ctx *ctx, const pg_mxfp4_expert *e, const float *x_dev, size_t m,
                                             float *scratch_dev, float *out_dev) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(e != nullptr, "pg_mxfp4_expert_forward: null expert");
    if (m == 0) return PG_OK;
    PG_CHECK_ARG(x_dev && scratch_dev && out_dev, "pg_mxfp4_expert_forward: null pointer");
    PG_CHECK_ARG((uintptr_t)x_dev % 16 == 0 && (uintptr_t)scratch_dev % 16 == 0,
                 "pg_mxfp4_expert_forward: x and scratch must be 16-byte aligned");
    PG_CHECK_ARG(m <= 65535, "pg_mxfp4_expert_forward: more than 65535 rows");
    const size_t inter = e->intermediate, hid = e->hidden;
    float *h = scratch_dev, *act = scratch_dev + m * 2 * inter;
    PG_TRY(pg_gguf_matmul_rows(ctx, x_dev, m, e->mlp1, h));
    PG_TRY(pg_launch(ctx, "mxfp4_bias_swiglu", mxfp4_bias_swiglu_kernel, dim3(grid_for(m * inter, 256)), dim3(256), 0,
                     (const float *)h, (const float *)e->bias1, m, inter, e->alpha, e->clamp, act));
    PG_TRY(pg_gguf_matmul_rows(ctx, act, m, e->mlp2, out_dev));
    return pg_launch(ctx, "bias_add", bias_add_kernel, dim3(grid_for(m * hid, 256)), dim3(256), 0, (const float *)out_dev,
                     (const float *)e->bias2, m, hid, out_dev);
}

PG_API pg_status pg_mxfp4_expert_forward(pg_ctx *ctx, const pg_mxfp4_expert *e, const float *x, size_t m, float *out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(e != nullptr, "pg_mxfp4_expert_forward: null expert");
    if (m == 0) return PG_OK;
    PG_CHECK_ARG(x && out, "pg_mxfp4_expert_forward: null pointer");
    pg_dev_block dx, ds, dout;
    PG_TRY(ds.alloc(ctx, m * 3 * e->intermediate * sizeof(float)));
    PG_TRY(dout.alloc(ctx, m * e->hidden * sizeof(float)));
    PG_TRY(pg_host_in(ctx, x, m * e->hidden * sizeof(float), dx));
    PG_TRY(pg_mxfp4_expert_forward_dev(ctx, e, dx.as<float>(), m, ds.as<float>(), dout.as<float>()));
    return pg_host_out(ctx, out, dout.p, m * e->hidden * sizeof(float));
}


// ---- the MoE layer over MXFP4 experts, grouped ------------------------------------------------
// MoELayer::forward after its router  examples/gpt_oss/moe.rs:286-352: the reference walks the tokens and calls
// Mxfp4Expert::forward once per (token, chosen expert).  Here every expert's tokens form token tiles of the tile
// kernel, all experts in one launch per product: routing lists, the pairs' activation rows gathered into digit
// records, mlp1 of all experts, bias + swiglu per pair, records again, mlp2, and out[t] = sum_k w[t,k] (y + bias2)
// in k order.
namespace {


// output[t] += weight * (out + mlp2_bias) over the token's experts in the order given  (examples/gpt_oss/moe.rs:104-108, 330-334)
// out[t] = sum_k weight (y + bias2), k ascending; idx and weight as the caller chose them or already put in order (mx_routed).  CH
// entries' loads are in flight together.  `per` workgroups a token, so its entries, their experts and the bias rows' addresses are
// the same for a workgroup and are scalars; a thread owns one V: four columns (hidden is a multiple of 32), of few outputs
// one (9 x 4 of 1088 columns 5.2 -> 4.0 us, by fours 5.5).  Bound by three dependent reads, entry, table and bias: 421 tokens x 4 of 1280 columns 7.7 -> 5.7 us (one column a thread), 20 x 4 of 2880 4.8 -> 4.7.
template <typename V, int CH>
__global__ __launch_bounds__(256) void mxfp4_moe_combine_kernel(const float *__restrict__ yb, const float *const *__restrict__ bias_tab,
                                                                const int *__restrict__ idx, const float *__restrict__ weight,
                                                                unsigned per, unsigned hidden, int top_k, int experts, float *__restrict__ out) {
    typedef const V __attribute__((address_space(1))) *gV_ptr;
    constexpr unsigned W = sizeof(V) / 4;
    const size_t t = blockIdx.x / per;
    const unsigned c = (blockIdx.x % per) * blockDim.x + threadIdx.x;
    if (c >= hidden / W) return;
    mx_routed taken;
    float acc[W] = {};
    for (int k0 = 0; k0 < top_k; k0 += CH) {
        int e[CH];
        float w[CH];
        V v[CH], b[CH];
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const size_t p = t * top_k + (k0 + j < top_k ? k0 + j : top_k - 1);
            v[j] = reinterpret_cast<const V *>(yb + p * hidden)[c];
            e[j] = __builtin_amdgcn_readfirstlane(idx[p]);
            w[j] = weight[p];
        }
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            bool named = true;
            if (k0 + j < top_k) e[j] = taken.next(e[j], experts, named);
            else e[j] = e[0];
            w[j] = named ? w[j] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < CH; ++j) b[j] = ((gV_ptr)(uintptr_t)mx_uniform(bias_tab + e[j]))[c];
#pragma unroll
        for (int j = 0; j < CH; ++j)
            if (k0 + j < top_k) {
#pragma unroll
                for (unsigned x = 0; x < W; ++x) {
                    const float result = reinterpret_cast<const float *>(&v[j])[x] + reinterpret_cast<const float *>(&b[j])[x], prod = w[j] * result;
                    acc[x] = acc[x] + prod;
                }
            }
    }
    float *const o = out + t * hidden + c * W;
    if (W == 4 && ((uintptr_t)out & 15) == 0) {
        *reinterpret_cast<v4f *>(o) = v4f{acc[0], acc[1 % W], acc[2 % W], acc[3 % W]};
    } else {  // (the caller's pointer may be any float's)
#pragma unroll
        for (unsigned x = 0; x < W; ++x) o[x] = acc[x];
    }
}

// One grouped product: rows `src` (pair / div) of the experts' slots -> records -> tiles against tensor table `which`.
// With `act`: the rows are the swiglu of src, mlp1's outputs.
// How the tiles of a grouped product are cut: TB groups of 16 slots, RA groups of 16 weight rows a wavefront, NW wavefronts.
struct mt_shape { int tb, ra, nw; };

// The tiling of least estimated time for both products together.  `load` workgroups stand on the fullest CU (the average and the part
// `whole` of what is missing to the number above it); a launch takes begin + load * each, a chunk of it `chunk` + load * wg, of which
// empty groups of tail tiles and empty slots of single-group tiles cost only the part `fixed`; the weights of the experts that are hit
// come at `rate` TB/s.  The two times are joined by a square for tiles of 16 slots and by a seventh power for 32, whose arithmetic
// hides the stream better.  The experts' slots are binomials.  Timed on 770 shapes (16 to 1700 tokens, 4 to 32 experts, 256 to 3800
// wide), every tiling of each product: the choice is 2 % over the best one on average; 64 slots, and 32 on eight wavefronts, would
// give another 0.4 %.
// Where hardly a tile is half full (six slots an expert on average, or twelve if the weights alone take 40 us), the estimates err by
// up to 40 % for 32 slots, which pay for 16: one group of slots, and the widest row tile that leaves every CU two workgroups.  (60
// tokens over 32 experts of 2144 x 1280, top 2: 58 us, as 32 slots 75; 90 over 32 of 2880 x 2880, top 4: 124, as 32 slots 143.)
struct mt_cost { mt_shape s; double begin, chunk, wg, fixed, each, rate, whole; };
constexpr mt_cost MT_COSTS[] = {{{1, 1, 8}, 0.97, 0.113, 0.387, 0.14, 0.95, 7.23, 0.65},
                                {{1, 2, 8}, 0.66, 0.010, 0.674, 0.24, 1.63, 7.18, 0.75},
                                {{1, 4, 8}, 0.00, 0.000, 1.014, 0.27, 3.22, 6.42, 1.00},
                                {{2, 1, 4}, 3.07, 0.105, 0.289, 0.40, 0.50, 3.54, 0.69},
                                {{2, 2, 4}, 3.21, 0.164, 0.314, 0.11, 0.86, 4.64, 0.71},
                                {{2, 4, 4}, 3.72, 0.148, 0.505, 0.00, 1.49, 5.03, 0.77}};
void choose_tiles(const pg_ctx *ctx, size_t T, size_t E, size_t top_k, const size_t (&n_out)[2], const int (&ncp)[2], mt_shape (&out)[2]) {
    const size_t P = T * top_k, cus = (size_t)ctx->num_cu;
    const double hit = (double)E * (1.0 - pow(1.0 - (double)top_k / (double)E, (double)T));
    auto bytes = [&](int i) { return hit * (double)n_out[i] * ncp[i] * 68.0; };
    if (P < 6 * E || (P < 12 * E && (bytes(0) + bytes(1)) / 5.6e6 > 40.0)) {
        const size_t max_tiles = P / 16 + E;
        for (int i = 0; i < 2; ++i) {
            const size_t nrg = (n_out[i] + 15) / 16;
            int ra = 4;
            while (ra > 1 && ((size_t)ra > nrg || (nrg + MT_NW * ra - 1) / (MT_NW * ra) * max_tiles < 2 * cus)) ra >>= 1;
            out[i] = {1, ra, MT_NW};
        }
        return;
    }
    double best = 1e300;
    for (int tb = 1; tb <= 2; ++tb) {
        const double tiles = pg_moe_expected_tiles(T, E, top_k, 16 * tb);
        const double live = tb == 1 ? (double)P / (16.0 * tiles) : std::min(1.0, ((double)P / 16.0 + 0.5 * hit) / (tiles * tb));
        const double joined = tb == 1 ? 2.0 : 7.0;
        mt_shape pick[2] = {};
        double sum = 0.0;
        for (int i = 0; i < 2; ++i) {
            const size_t nrg = (n_out[i] + 15) / 16;
            double least = 1e299;
            for (const mt_cost &c : MT_COSTS) {
                if (c.s.tb != tb || (size_t)c.s.ra > nrg) continue;
                const double w = std::max(1.0, tiles * (double)((nrg + c.s.nw * c.s.ra - 1) / (c.s.nw * c.s.ra)) / (double)cus);
                const double load = w + c.whole * (ceil(w) - w);
                const double work = c.begin + load * c.each + ncp[i] * (c.chunk + load * c.wg * (c.fixed + (1.0 - c.fixed) * live));
                const double us = pow(pow(work, joined) + pow(3.0 + bytes(i) / (c.rate * 1e6), joined), 1.0 / joined);
                if (us < least) {
                    least = us;
                    pick[i] = c.s;
                }
            }
            sum += least;
        }
        if (sum < best) {
            best = sum;
            out[0] = pick[0];
            out[1] = pick[1];
        }
    }
}

pg_status moe_product(pg_ctx *ctx, const float *src, size_t k_in, size_t n_out, const mt_shape &sh, size_t max_tiles, mt_gather gat, int div,
                      const void **tab, size_t experts, int which, char *bq, float *y, const mt_swiglu *act = nullptr, const mt_route *rt = nullptr) {
    const int nb = (int)(k_in / 32), ncp = (int)mx_chunks((size_t)nb);
    gat.div = div;
    const size_t groups = max_tiles * sh.tb, threads = groups * 2 * (size_t)ncp * 64;
    PG_CHECK_ARG((threads + 255) / 256 < ((size_t)1 << 31), "mxfp4 moe: too many pairs x %zu for one pre-pass", k_in);
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (act) PG_TRY(pg_launch(ctx, "mxfp4_planes_swiglu", mxfp4_planes_kernel<true, true>, grid, dim3(256), 0, src, 0, nb, ncp, (int)groups, bq, gat, *act, mt_route{}));
    else if (rt) PG_TRY(pg_launch(ctx, "mxfp4_planes_route", mxfp4_planes_kernel<true, false, true>, dim3(grid.x + 1), dim3(256), 0, src, 0, nb, ncp, (int)groups, bq, gat, mt_swiglu{}, *rt));
    else PG_TRY(pg_launch(ctx, "mxfp4_planes_gather", mxfp4_planes_kernel<true>, grid, dim3(256), 0, src, 0, nb, ncp, (int)groups, bq, gat, mt_swiglu{}, mt_route{}));
    const size_t nrg = (n_out + 15) / 16, n_wt = (nrg + sh.nw * sh.ra - 1) / (sh.nw * sh.ra);
    PG_CHECK_ARG(n_wt * max_tiles < ((size_t)1 << 28), "mxfp4 moe: %zu x %zu tiles", n_wt, max_tiles);
    const mt_experts ex = {reinterpret_cast<const uint8_t *const *>(tab + (size_t)(2 * which) * experts),
                           reinterpret_cast<const uint32_t *const *>(tab + (size_t)(2 * which + 1) * experts)};
#define PG_MTG(TB, RA, BD, NW) \
    if (sh.tb == TB && sh.ra == RA && sh.nw == NW) return launch_tiles_grouped<RA, TB, BD, NW>(ctx, n_out, ncp, bq, y, n_wt, max_tiles, gat, ex);
    PG_MTG(1, 1, 4, 8) PG_MTG(1, 2, 2, 8) PG_MTG(1, 4, 4, 8) PG_MTG(2, 1, 4, 4) PG_MTG(2, 2, 1, 4) PG_MTG(2, 4, 1, 4)
#undef PG_MTG
    return pg_fail(PG_EUNSUPPORTED, "mxfp4 moe: no kernel of %d x 16 slots, %d row groups, %d wavefronts", sh.tb, sh.ra, sh.nw);
}

// Whether up to 64 pairs are faster one by one than as tiles although pairs share experts (P > 2 E): the decode kernel streams an
// expert's 3 * hidden * inter FP4 weights per pair at 6.2 TB/s over 15 us of launches, the tiles stream those of the
// experts that T tokens are expected to hit at 5.2 over 27, but at least the walk of one row tile through both K.
// (us, pairs against tiles: 8 experts of 960, top 2, 16 tokens 22.0 / 28.2; of 1440, top 4, 6 tokens 28.8 / 34.3, 8 tokens
// 33.1 / 33.8, 10 tokens 37.3 / 32.2; of 2880, top 2, 10 tokens 60.1 / 47.3.  Both timed on 351 shapes, 4 to 30 experts,
// hidden and inter 256 to 5760: 0.6 % over the faster one on average.  Where it errs: few output columns under a long K, which
// the decode kernel streams at less than half that rate -- hidden 512, inter 3360 to 4096, 36 to 40 pairs 43-47 / 35 -- and
// narrow experts of 2048 x 512, which would gain 15 % as pairs.  Such calls keep the finer digits they have.  The tiles' 27 and 20 us
// hold a routing launch that up to 64 experts no longer have: 4 us less would move calls from the pairs' exact activations to the tiles'
// digits, so the line stays where it was.)
bool pairs_faster(size_t T, size_t E, size_t top_k, size_t hidden, size_t inter) {
    const double us_per_expert = 3.0 * (double)hidden * (double)inter * (17.0 / 32.0) / 1e6;  // at 1 TB/s
    const double hit = (double)E * (1.0 - pow(1.0 - (double)top_k / (double)E, (double)T));
    const double pairs = 15.0 + (double)(T * top_k) * us_per_expert / 6.2;
    const double tiles = std::max(20.0 + 0.00415 * (double)(hidden + inter), 27.0 + hit * us_per_expert / 5.2);
    return pairs < tiles;
}

// The same product pair by pair on the decode kernel (few pairs).
bool pairs_fit(int ncp) { return mx_lds_bytes(1, ncp) <= (160u << 10); }
template <int PAIRS>
pg_status moe_product_pairs(pg_ctx *ctx, const float *src, size_t src_rows, size_t k_in, size_t n_out, size_t pairs, int by_token,
                            const void **tab, size_t experts, int which, const int *idx, int *chosen, size_t top_k, float *y, const mt_swiglu &act) {
    const int ncp = (int)mx_chunks(k_in / 32);
    const mx_pairs pr = {reinterpret_cast<const uint8_t *const *>(tab + (size_t)(2 * which) * experts),
                         reinterpret_cast<const uint32_t *const *>(tab + (size_t)(2 * which + 1) * experts), idx, chosen, (int)experts, by_token, act};
    // as pg_launch_mxfp4_rows chooses: 16 wavefronts on a row group while there is at most one group per CU, else 8
    // on the fewest row groups that keep every workgroup resident at once
    const size_t groups = (n_out + 15) / 16 * pairs, slots = (size_t)ctx->num_cu * 2;
    if (groups <= (size_t)ctx->num_cu) return launch_rows_pairs<1, 16, PAIRS>(ctx, n_out, k_in, src, src_rows, y, pairs, top_k, ncp, pr);
    if (groups <= slots) return launch_rows_pairs<1, 8, PAIRS>(ctx, n_out, k_in, src, src_rows, y, pairs, top_k, ncp, pr);
    if ((groups + 1) / 2 <= slots) return launch_rows_pairs<2, 8, PAIRS>(ctx, n_out, k_in, src, src_rows, y, pairs, top_k, ncp, pr);
    return launch_rows_pairs<4, 8, PAIRS>(ctx, n_out, k_in, src, src_rows, y, pairs, top_k, ncp, pr);
}

}  // namespace

PG_API pg_status pg_mxfp4_moe_ffn_routed_dev(pg_ctx *ctx, const float *x_dev, size_t T, const int32_t *expert_idx_dev,
                                             const float *weight_dev, size_t top_k, const pg_mxfp4_expert *const *experts, size_t E,
                                             float *out_dev) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(E >= 1 && E <= (size_t)PG_MOE_MAX_EXPERTS, "pg_mxfp4_moe_ffn: %zu experts (1..%d supported)", E, PG_MOE_MAX_EXPERTS);
    PG_CHECK_ARG(top_k >= 1 && top_k <= E, "pg_mxfp4_moe_ffn: top_k %zu of %zu experts", top_k, E);
    PG_CHECK_ARG(experts && experts[0], "pg_mxfp4_moe_ffn: null expert table");
    const size_t hidden = experts[0]->hidden, inter = experts[0]->intermediate;
    const float alpha = experts[0]->alpha, clamp = experts[0]->clamp;
    for (size_t e = 0; e < E; ++e) {
        PG_CHECK_ARG(experts[e] != nullptr, "pg_mxfp4_moe_ffn: expert %zu is null", e);
        PG_CHECK_ARG(experts[e]->hidden == hidden && experts[e]->intermediate == inter && experts[e]->alpha == alpha &&
                         experts[e]->clamp == clamp, "pg_mxfp4_moe_ffn: expert %zu differs in shape, alpha or clamp", e);
    }
    if (T == 0) return PG_OK;
    PG_CHECK_ARG(x_dev && expert_idx_dev && weight_dev && out_dev, "pg_mxfp4_moe_ffn: null pointer");
    PG_CHECK_ARG((uintptr_t)x_dev % 16 == 0, "pg_mxfp4_moe_ffn: x must be 16-byte aligned");
    PG_CHECK_ARG(T * top_k < (1ull << 20), "pg_mxfp4_moe_ffn: too many (token, expert) pairs");
    const size_t P = T * top_k;
    const int ncp1 = (int)mx_chunks(hidden / 32), ncp2 = (int)mx_chunks(inter / 32);
    mt_shape shape[2];
    choose_tiles(ctx, T, E, top_k, {2 * inter, hidden}, {ncp1, ncp2}, shape);
    const int tb = shape[0].tb;
    const size_t max_tiles = P / (16 * (size_t)tb) + E;  // sum over experts of ceil(count / (16 tb)) stays below
    // With few pairs hardly two of them meet in an expert, and a pair is a one-row product: the decode kernel, one
    // workgroup column per pair (exact activations; no expert lists).  Otherwise the experts' token tiles on the tile kernel.
    const bool by_pairs = P <= 64 && (P <= 2 * E || pairs_faster(T, E, top_k, hidden, inter)) && pairs_fit(ncp1) && pairs_fit(ncp2);
    const size_t sz_idx = pg_round_up(P * sizeof(int), 256), sz_p = pg_round_up(P * sizeof(float), 256);
    const size_t sz_lists = pg_round_up(E * T * sizeof(int), 256), sz_counts = pg_round_up((2 * E + 1) * sizeof(int), 256);
    const size_t sz_rec = pg_round_up(max_tiles * tb * (size_t)std::max(ncp1, ncp2) * MT_RECORD, 256);
    const size_t sz_h = pg_round_up(P * 2 * inter * sizeof(float), 256);
    const size_t sz_y = pg_round_up(P * hidden * sizeof(float), 256);
    void *ws = nullptr;
    PG_TRY(pg_workspace(ctx, sz_idx + sz_p + sz_lists + sz_counts + sz_rec + sz_h + sz_y, &ws));
    char *p = static_cast<char *>(ws);
    int *topk_idx = reinterpret_cast<int *>(p); p += sz_idx;
    float *topk_p = reinterpret_cast<float *>(p); p += sz_p;
    int *lists = reinterpret_cast<int *>(p); p += sz_lists;
    int *counts = reinterpret_cast<int *>(p), *goff = counts + E; p += sz_counts;
    char *rec = p; p += sz_rec;
    float *h = reinterpret_cast<float *>(p); p += sz_h;
    float *yb = reinterpret_cast<float *>(p);
    // [mlp1 codes | mlp1 scales | mlp2 codes | mlp2 scales | bias1 | bias2], E each
    const void *host_tab[6 * PG_MOE_MAX_EXPERTS];
    for (size_t e = 0; e < E; ++e) {
        host_tab[0 * E + e] = experts[e]->mlp1->qs; host_tab[1 * E + e] = experts[e]->mlp1->d;
        host_tab[2 * E + e] = experts[e]->mlp2->qs; host_tab[3 * E + e] = experts[e]->mlp2->d;
        host_tab[4 * E + e] = experts[e]->bias1;    host_tab[5 * E + e] = experts[e]->bias2;
    }
    const void **tab = nullptr;
    PG_TRY(pg_moe_cached_table(ctx, host_tab, 6 * E, &tab));
    const mt_swiglu sw = {reinterpret_cast<const float *const *>(tab + 4 * E), alpha, clamp};
    if (by_pairs) {
        PG_TRY(moe_product_pairs<2>(ctx, x_dev, T, hidden, 2 * inter, P, 1, tab, E, 0, expert_idx_dev, topk_idx, top_k, h, sw));
        PG_TRY(moe_product_pairs<1>(ctx, h, P, inter, hidden, P, 0, tab, E, 1, nullptr, topk_idx, top_k, yb, mt_swiglu{}));
    } else {
        const bool route = P <= (size_t)MT_ROUTE_PAIRS && E <= (size_t)MT_ROUTE_EXPERTS;
        if (!route) PG_TRY(pg_launch_moe_routing(ctx, nullptr, expert_idx_dev, weight_dev, T, E, top_k, topk_idx, topk_p, lists, counts, goff, 16 * tb));
        const mt_route rt = {expert_idx_dev, weight_dev, (int)T, (int)top_k, 16 * tb, topk_idx, topk_p, lists, counts, goff};
        const mt_gather gat = {lists, counts, goff, (int)T, (int)E, tb, 1};
        PG_TRY(moe_product(ctx, x_dev, hidden, 2 * inter, shape[0], max_tiles, gat, (int)top_k, tab, E, 0, rec, h, nullptr, route ? &rt : nullptr));
        PG_TRY(moe_product(ctx, h, inter, hidden, shape[1], max_tiles, gat, 1, tab, E, 1, rec, yb, &sw));
    }
    const bool four = T * hidden >= 65536;
    const size_t columns = four ? hidden / 4 : hidden;
    const unsigned wg = (unsigned)std::min<size_t>(256, pg_round_up(columns, 64)), per = grid_for(columns, wg);
    PG_CHECK_ARG(T * per < ((size_t)1 << 31), "pg_mxfp4_moe_ffn: %zu tokens of %zu outputs in one launch", T, hidden);
    auto kern = four ? (top_k <= 2 ? mxfp4_moe_combine_kernel<v4f, 2> : mxfp4_moe_combine_kernel<v4f, 4>)
                     : (top_k <= 2 ? mxfp4_moe_combine_kernel<float, 2> : mxfp4_moe_combine_kernel<float, 4>);
    return pg_launch(ctx, "mxfp4_moe_combine", kern, dim3((unsigned)(T * per)), dim3(wg), 0,
                     (const float *)yb, reinterpret_cast<const float *const *>(tab + 5 * E), by_pairs ? expert_idx_dev : (const int *)topk_idx,
                     by_pairs ? weight_dev : (const float *)topk_p, per, (unsigned)hidden, (int)top_k, (int)E, out_dev);
}

PG_API pg_status pg_mxfp4_moe_ffn_routed(pg_ctx *ctx, const float *x, size_t T, const int32_t *expert_idx, const float *weight,
                                         size_t top_k, const pg_mxfp4_expert *const *experts, size_t E, float *out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(experts && experts[0], "pg_mxfp4_moe_ffn: null expert table");
    if (T == 0) return PG_OK;
    PG_CHECK_ARG(x && expert_idx && weight && out, "pg_mxfp4_moe_ffn: null pointer");
    PG_CHECK_ARG(E >= 1 && E <= (size_t)PG_MOE_MAX_EXPERTS && top_k >= 1 && top_k <= E, "pg_mxfp4_moe_ffn: top_k %zu of %zu experts", top_k, E);
    // the reference indexes self.experts[expert_idx] (examples/gpt_oss/moe.rs:104-108) and would panic on an index out
    // of range; its top-k never names an expert twice for a token, which the grouped products rely on
    for (size_t t = 0; t < T; ++t)
        for (size_t k = 0; k < top_k; ++k) {
            const int32_t e = expert_idx[t * top_k + k];
            PG_CHECK_ARG(e >= 0 && (size_t)e < E, "pg_mxfp4_moe_ffn: token %zu names expert %d of %zu", t, (int)e, E);
            for (size_t j = 0; j < k; ++j)
                PG_CHECK_ARG(expert_idx[t * top_k + j] != e, "pg_mxfp4_moe_ffn: token %zu names expert %d twice", t, (int)e);
        }
    const size_t hidden = experts[0]->hidden;
    pg_dev_block dx, di, dw, dout;
    PG_TRY(dout.alloc(ctx, T * hidden * sizeof(float)));
    PG_TRY(pg_host_in(ctx, x, T * hidden * sizeof(float), dx));
    PG_TRY(pg_host_in(ctx, expert_idx, T * top_k * sizeof(int32_t), di));
    PG_TRY(pg_host_in(ctx, weight, T * top_k * sizeof(float), dw));
    PG_TRY(pg_mxfp4_moe_ffn_routed_dev(ctx, dx.as<float>(), T, di.as<int32_t>(), dw.as<float>(), top_k, experts, E, dout.as<float>()));
    return pg_host_out(ctx, out, dout.p, T * hidden * sizeof(float));
}
