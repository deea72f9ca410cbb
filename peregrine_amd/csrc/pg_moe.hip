// Grouped MoE expert FFN over block-quantised (Q8_0 / Q4_0) experts, entirely
// stream-ordered on the device (no host round trip for the routing):
//   1. route: softmax over the E router logits of each token, top-k by stable
//      descending order (ties -> lower expert index)   examples/grok1/moe.rs:76-89
//   2. gate / up products of every (token, k) pair against its expert's weights
//   3. h = act(g) * u                                   grok1/moe.rs:27-34, deepseek/moe.rs:55-59
//   4. down product of every pair
//   5. out[t] = 0 + p_0 * y_0 + p_1 * y_1 ... in k order, multiply then add
//      (examples/grok1/moe.rs:99-104), raw softmax probabilities.
#include "pg_internal.h"
#include "pg_digits.h"
#include "pg_act_dev.h"
#include "pg_quant_dev.h"
#include <algorithm>

namespace {

inline unsigned grid_for(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }

constexpr int MAX_EXPERTS = PG_MOE_MAX_EXPERTS;

// One thread per token.
__global__ void route_topk_kernel(const float *__restrict__ logits, int T, int E, int top_k,
                                  int *__restrict__ topk_idx, float *__restrict__ topk_p) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) return;
    const float *x = logits + (size_t)t * E;
    float mx = -INFINITY;
    for (int e = 0; e < E; ++e)
        if (x[e] > mx) mx = x[e];
    float sum = 0.0f;
    for (int e = 0; e < E; ++e) sum += expf(x[e] - mx);
    // k passes of "largest remaining, lowest index on ties" == stable descending sort
    unsigned taken[MAX_EXPERTS / 32];
    for (int i = 0; i < MAX_EXPERTS / 32; ++i) taken[i] = 0u;
    for (int k = 0; k < top_k; ++k) {
        int best = -1;
        float bp = 0.0f;
        for (int e = 0; e < E; ++e) {
            if (taken[e >> 5] & (1u << (e & 31))) continue;
            const float p = expf(x[e] - mx) / sum;
            if (best < 0 || p > bp) { best = e; bp = p; }
        }
        taken[best >> 5] |= 1u << (best & 31);
        topk_idx[(size_t)t * top_k + k] = best;
        topk_p[(size_t)t * top_k + k] = bp;
    }
}

// The same, or a copy of the caller's routing (see below), and the experts' lists and first token tiles, in ONE launch of one
// workgroup while the routing is small: as launches of their own they are the launch and little else (copy, lists and
// offsets of 20 tokens over 32 experts 13.8 us, 4.8 here; softmax, top-k and lists of 64 over 8 11.0, 4.8 here).  The logits pass through
// LDS (a row per thread, an odd number of words apart) and hold the probabilities afterwards, -1 where taken; the chosen
// experts stay there as bytes for the lists.  MAX_ROUTE_LDS bytes at most.
// DIG: the further workgroups write the activation rows' digits for the first product, 1 / 2 = byte planes of Q4_0 / Q8_0
// (pg_emit_mm_digits), 3 / 4 = those of the streaming product (pg_emit_digits): neither waits for the other, and as a launch of its
// own the digits' took 4.6 us (a layer of 26 tokens, 2 of 4 experts of 1568 x 1696, Q8_0: 31.9 -> 29.5 us; 4, 2 of 8 of 2048 x 4096: 35.4 -> 33.3).
constexpr size_t MAX_ROUTE_LDS = 48u << 10;
__host__ __device__ inline size_t route_row(size_t E) { return E | 1; }
inline size_t route_lds(size_t T, size_t E, size_t top_k, bool logits) { return pg_round_up((logits ? T * route_row(E) * sizeof(float) : 0) + T * top_k, 4); }  // (read four bytes at a time)
// (The caller's own routing holds no logits.  Where a table of them would not fit it took the three launches as well, 18.5 us and two gaps for
// 422 tokens over 32 experts, top 4: layers of 422 tokens of 800 x 2752 117.0 : 108.5 us, 380 of 1024 x 1024 67.1 : 59.8, 512 of 2880 x 2880
// 259.7 : 250.4, 400 of 512 x 640, top 2 47.0 : 41.5.)
inline bool route_in_one(size_t T, size_t E, size_t top_k, bool logits) {
    // (Lists: a wavefront of the 16 takes every 16th expert and looks at 256 pairs at a time.  From 16 experts on that is 32 looks at the most; with fewer
    // some wavefronts stand idle and the tokens count instead, up to 48 K entries read by one workgroup.  The three launches read them by as many
    // wavefronts as tokens / 64, but their lists look at 64 pairs at a time, from memory.  us, three launches : one, over every T and k that the rule
    // takes: 1 expert 12442 tokens 59 : 18, 2 of 2 117 : 39, 2 of 4 119 : 40, 1 of 8 62 : 21, 4 of 8 of 3687 74 : 30, 2 of 16 40 : 18, few tokens 8.9 : 6.5;
    // past it 32 experts 0.7 to 1.0 of their time, 64 0.95 to 1.7, more 0.86 to 4.9.)
    return T * top_k * E <= (1u << 17) && route_lds(T, E, top_k, logits) <= MAX_ROUTE_LDS;
}
// A token's softmax and top-k on one wavefront, a lane an expert (up to 64): the steps of the thread's loops in route_lists_kernel, whose every look at an
// expert waits for LDS -- E (3 + k) of them one behind the other, some 130 cycles each, are 6 us for 16 experts and 4 choices.  The sum
// of the exponentials is added up in the same order; a NaN anywhere makes the sum and with it every probability NaN, and the lowest experts
// not taken are the choice.
__device__ __forceinline__ void route_token(const float *x, int E, int top_k, uint8_t *mine, int *idx, float *p_out) {
    const int lane = threadIdx.x & 63;
    const bool in = lane < E;
    const float v = in ? x[lane] : -INFINITY, mx = pg_wave_max_f32(v);
    const float ex = expf(v - mx);
    float sum = 0.0f;
    for (int e = 0; e < E; ++e) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ex), e));
    const float p = ex / sum;
    bool free = in;
    for (int k = 0; k < top_k; ++k) {
        const float best = pg_wave_max_f32(free ? p : -1.0f);
        const unsigned long long at = __ballot(free && (p == best || p != p));
        const int e = __ffsll(at) - 1;
        if (lane == e) {
            free = false;
            mine[k] = (uint8_t)e;
            idx[k] = e;
            p_out[k] = p;
        }
    }
}
// Up to 16 tokens, a wavefront each; a second round of them is as long as the first (1.3 us, 16 experts and 4 choices), where all threads' walks are one.  us, a
// layer, a thread a token : a wavefront: one token, 4 of 16 experts of 2400 x 2080 (Q4_0) 26.6 : 22.4, 8 of 32 of 2048 x 768 35.1 : 18.9, 2 of 8 of 1024 x 2816 (Q8_0)
// 16.1 : 14.9, 10 tokens, 4 of 8 of 896 x 7936 55.4 : 54.1; but 45, 2 of 16 of 608 x 2656 36.9 : 37.8, 64, 4 of 16 of 2048 x 2048 61.9 : 64.3.
__device__ __forceinline__ bool route_by_wave(int T, int E) { return T <= 16 && E <= 64; }

struct route_digits {
    const float *x;
    int nb, nbp, blocks;  // blocks of 32 a row, the same rounded up to 4, blocks of all rows
    int8_t *digits;
    float *xs;
};
template <bool LOGITS, int DIG>
__global__ __launch_bounds__(1024) void route_lists_kernel(const float *__restrict__ logits, const int *__restrict__ idx_in,
                                                           const float *__restrict__ w_in, int T, int E, int top_k,
                                                           int *__restrict__ topk_idx, float *__restrict__ topk_p,
                                                           int *__restrict__ lists, int *__restrict__ counts, int *__restrict__ goff, int tile,
                                                           const route_digits rd) {
    if (DIG && blockIdx.x > 0) {
        const int i = ((int)blockIdx.x - 1) * 128 + (int)(threadIdx.x >> 3), sub = threadIdx.x & 7;
        if (i >= rd.blocks) return;  // whole 8-thread groups leave together
        const int row = i / rd.nb, b = i - row * rd.nb;
        const float4 v = reinterpret_cast<const float4 *>(rd.x + (size_t)i * 32)[sub];
        const float f[4] = {v.x, v.y, v.z, v.w};
        if constexpr (DIG == 1 || DIG == 2) pg_emit_mm_digits<DIG == 1>(f, row, b, sub, rd.nb, rd.nbp, rd.digits, rd.xs);
        else if constexpr (DIG != 0) pg_emit_digits<DIG == 3>(f, row, b, sub, rd.nb, rd.digits, rd.xs);
        return;
    }
    extern __shared__ __attribute__((aligned(16))) float prob[];  // [T][route_row(E)] (LOGITS), then the pairs' experts as bytes
    __shared__ int cnt[MAX_EXPERTS];
    const int row = (int)route_row(E), P = T * top_k;
    uint8_t *const chosen = reinterpret_cast<uint8_t *>(prob + (LOGITS ? T * row : 0));
    if (LOGITS) {
        for (int i = threadIdx.x; i < T * E; i += 1024) prob[i / E * row + i % E] = logits[i];
        __syncthreads();
    }
    const bool by_wave = LOGITS && route_by_wave(T, E);
    if (by_wave) {
        const int t = threadIdx.x >> 6;
        if (t < T) route_token(prob + t * row, E, top_k, chosen + t * top_k, topk_idx + t * top_k, topk_p + t * top_k);
    }
    for (int t = threadIdx.x; !by_wave && t < T; t += 1024) {
        uint8_t *mine = chosen + t * top_k;
        if (LOGITS) {
            float *x = prob + t * row;
            float mx = -INFINITY;
            for (int e = 0; e < E; ++e)
                if (x[e] > mx) mx = x[e];
            float sum = 0.0f;
            for (int e = 0; e < E; ++e) {
                x[e] = expf(x[e] - mx);
                sum += x[e];
            }
            for (int e = 0; e < E; ++e) x[e] = x[e] / sum;
            for (int k = 0; k < top_k; ++k) {
                int best = -1;
                float bp = 0.0f;
                for (int e = 0; e < E; ++e) {
                    const float p = x[e];
                    if (p == -1.0f) continue;
                    if (best < 0 || p > bp) { best = e; bp = p; }
                }
                x[best] = -1.0f;
                mine[k] = (uint8_t)best;
                topk_idx[t * top_k + k] = best;
                topk_p[t * top_k + k] = bp;
            }
        } else {
            auto taken = [&](int e, int k) {
                bool is = false;
                for (int j = 0; j < k; ++j) is |= mine[j] == (uint8_t)e;
                return is;
            };
            for (int k = 0; k < top_k; ++k) {
                int e = idx_in[t * top_k + k];
                float w = w_in[t * top_k + k];
                if (e < 0 || e >= E || taken(e, k)) {
                    e = 0;
                    while (taken(e, k)) ++e;  // top_k <= E: a free expert exists
                    w = 0.0f;
                }
                mine[k] = (uint8_t)e;
                topk_idx[t * top_k + k] = e;
                topk_p[t * top_k + k] = w;
            }
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int e = threadIdx.x >> 6; e < E; e += 16) {
        int base = 0;
        // Past two looks of a pair a lane, four pairs a lane: a look waits for LDS once (1684 pairs 7.5 -> 6.2 us, 480 6.4 -> 5.6; 20 pairs
        // 5.3, by fours 5.6).
        if (P <= 128) {
            for (int p0 = 0; p0 < P; p0 += 64) {
                const int p = p0 + lane;
                const bool own = p < P && chosen[p] == e;
                const unsigned long long mask = __ballot(own);
                if (own) lists[(size_t)e * T + base + __popcll(mask & ((1ull << lane) - 1ull))] = p;
                base += __popcll(mask);
            }
        } else {
            for (int p0 = 0; p0 < P; p0 += 256) {
                const int p = p0 + 4 * lane;
                const unsigned four = p < P ? *reinterpret_cast<const unsigned *>(chosen + p) : 0u;
                int before = base;
                bool own[4];
    #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    own[i] = p + i < P && (int)(four >> (8 * i) & 255u) == e;
                    const unsigned long long mask = __ballot(own[i]);
                    before += __popcll(mask & ((1ull << lane) - 1ull));
                    base += __popcll(mask);
                }
    #pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (own[i]) lists[(size_t)e * T + before++] = p + i;
            }
        }
        if (lane == 0) {
            counts[e] = base;
            cnt[e] = (base + tile - 1) / tile;
        }
    }
    if (!goff) return;
    __syncthreads();
    if ((int)threadIdx.x <= E) {  // first token tile of every expert, and their number
        int run = 0;
        for (int e = 0; e < (int)threadIdx.x; ++e) run += cnt[e];
        goff[threadIdx.x] = run;
    }
}

// A routing that the caller made (another gate: examples/deepseek/moe.rs:111-215, examples/gpt_oss/moe.rs:298-330)
// is copied into the same arrays.  The grouped products assume what every top-k gate delivers: a token's experts are
// distinct and inside 0 .. E - 1.  An entry that breaks this is replaced by the lowest expert the token does not use
// yet, with weight 0, so that nothing downstream can index outside a table whatever the buffers hold (the entry's
// own contribution is then 0 times a finite product).  One thread per token.
__global__ void copy_routing_kernel(const int *__restrict__ idx_in, const float *__restrict__ w_in, int T, int E, int top_k,
                                    int *__restrict__ topk_idx, float *__restrict__ topk_p) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) return;
    unsigned taken[MAX_EXPERTS / 32];
    for (int i = 0; i < MAX_EXPERTS / 32; ++i) taken[i] = 0u;
    for (int k = 0; k < top_k; ++k) {
        int e = idx_in[(size_t)t * top_k + k];
        float w = w_in[(size_t)t * top_k + k];
        if (e < 0 || e >= E || (taken[e >> 5] & (1u << (e & 31)))) {
            e = 0;
            while (taken[e >> 5] & (1u << (e & 31))) ++e;  // top_k <= E: a free expert exists
            w = 0.0f;
        }
        taken[e >> 5] |= 1u << (e & 31);
        topk_idx[(size_t)t * top_k + k] = e;
        topk_p[(size_t)t * top_k + k] = w;
    }
}

// Per expert, the (token, k) pairs routed to it, in ascending pair order.  One wavefront per
// expert: ballot + prefix count over 64 pairs at a time.
__global__ __launch_bounds__(64) void expert_lists_kernel(const int *__restrict__ topk_idx, int P, int stride,
                                                          int *__restrict__ lists, int *__restrict__ counts) {
    const int e = blockIdx.x, lane = threadIdx.x;
    int base = 0;
    for (int p0 = 0; p0 < P; p0 += 64) {
        const int p = p0 + lane;
        const bool mine = p < P && topk_idx[p] == e;
        const unsigned long long mask = __ballot(mine);
        if (mine) lists[(size_t)e * stride + base + __popcll(mask & ((1ull << lane) - 1ull))] = p;
        base += __popcll(mask);
    }
    if (lane == 0) counts[e] = base;
}

// First tile of `tile` pairs of every expert: goff[e] = sum over e' < e of ceil(counts[e'] / tile); goff[experts] = all.
__global__ __launch_bounds__(64) void tile_offsets_kernel(const int *__restrict__ counts, int experts, int tile, int *__restrict__ goff) {
    if (threadIdx.x != 0) return;
    int run = 0;
    for (int e = 0; e < experts; ++e) {
        goff[e] = run;
        run += (counts[e] + tile - 1) / tile;
    }
    goff[experts] = run;
}

// act(g) * u of every pair as the digit planes of the matrix-core product; g and u as the sums of `planes` planes, `stride`
// floats apart, in ascending order.  (As two launches, with the products through memory: 10.5 us for 128 pairs of 8192, 5.6 here.)
template <bool NIB>
__global__ __launch_bounds__(256) void act_mm_digits_kernel(const float *__restrict__ g, const float *__restrict__ u, int planes, size_t stride,
                                                            int act, int nb, int nbp, int8_t *__restrict__ digits, float *__restrict__ xs) {
    const size_t row = blockIdx.y;
    const int b = blockIdx.x * 32 + (threadIdx.x >> 3), sub = threadIdx.x & 7;
    if (b >= nb) return;  // whole 8-thread groups leave together
    const size_t at = ((row * nb + b) * 8 + sub) * 4;
    float4 gp[8], up[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
        if (s < planes) {
            gp[s] = *reinterpret_cast<const float4 *>(g + s * stride + at);
            up[s] = *reinterpret_cast<const float4 *>(u + s * stride + at);
        }
    float4 gv = gp[0], uv = up[0];
#pragma unroll
    for (int s = 1; s < 8; ++s)
        if (s < planes) {
            gv.x += gp[s].x; gv.y += gp[s].y; gv.z += gp[s].z; gv.w += gp[s].w;
            uv.x += up[s].x; uv.y += up[s].y; uv.z += up[s].z; uv.w += up[s].w;
        }
    const float gf[4] = {gv.x, gv.y, gv.z, gv.w}, uf[4] = {uv.x, uv.y, uv.z, uv.w};
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = pg_act(act, gf[i]) * uf[i];
    pg_emit_mm_digits<NIB>(o, row, b, sub, nb, nbp, digits, xs);
}

// The same as rows of the streaming kernel's digits.
template <bool NIB>
__global__ __launch_bounds__(256) void act_digits_kernel(const float *__restrict__ g, const float *__restrict__ u, int act, int nb, int8_t *__restrict__ digits,
                                                         float *__restrict__ xs) {
    const size_t row = blockIdx.y;
    const int b = blockIdx.x * 32 + (threadIdx.x >> 3), sub = threadIdx.x & 7;
    if (b >= nb) return;  // whole 8-thread groups leave together
    const size_t at = ((row * nb + b) * 8 + sub) * 4;
    const float4 gv = *reinterpret_cast<const float4 *>(g + at), uv = *reinterpret_cast<const float4 *>(u + at);
    const float o[4] = {pg_act(act, gv.x) * uv.x, pg_act(act, gv.y) * uv.y, pg_act(act, gv.z) * uv.z, pg_act(act, gv.w) * uv.w};
    pg_emit_digits<NIB>(o, row, b, sub, nb, digits, xs);
}

// yb: the down product's outputs, the sums of `planes` planes (its K chunks) in ascending order.
// `shared` (optional): the shared experts' output, added last (y.add(&z), examples/deepseek/moe.rs:298-300).
// `per` workgroups a token, so the token and its weights are the same for a workgroup (no division by d in every thread); a thread
// owns one V (four columns where rows are whole float4s), and the planes of two entries, PL at a time, are asked for together.
// What it takes is that round trip: 194 tokens x 4 entries x 4 planes of 832 columns 6.3 -> 4.6 us (one column a thread, an entry's
// planes one after the other); small ones stay at a launch's 4 to 5.
template <typename V, int PL>
__global__ __launch_bounds__(256) void combine_kernel(const float *__restrict__ yb, int planes, size_t stride, const float *__restrict__ topk_p,
                                                      unsigned per, int d, int top_k, const float *__restrict__ shared, float *__restrict__ out) {
    constexpr int W = sizeof(V) / 4;
    const size_t t = blockIdx.x / per;
    const unsigned c = (blockIdx.x % per) * blockDim.x + threadIdx.x;
    if (c >= (unsigned)(d / W)) return;
    float acc[W] = {};
    for (int k0 = 0; k0 < top_k; k0 += 2) {
        const int k1 = k0 + 1 < top_k ? k0 + 1 : k0;
        const float *const y[2] = {yb + (t * top_k + k0) * d, yb + (t * top_k + k1) * d};
        const float w[2] = {topk_p[t * top_k + k0], topk_p[t * top_k + k1]};
        float v[2][W];
        for (int s0 = 0; s0 < planes; s0 += PL) {
            V in[2][PL];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int s = 0; s < PL; ++s) in[q][s] = reinterpret_cast<const V *>(y[q] + (size_t)(s0 + s < planes ? s0 + s : s0) * stride)[c];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int s = 0; s < PL; ++s)
                    if (s0 + s < planes) {
                        const float *f = reinterpret_cast<const float *>(&in[q][s]);
#pragma unroll
                        for (int x = 0; x < W; ++x) v[q][x] = s0 + s == 0 ? f[x] : v[q][x] + f[x];
                    }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (k0 + q < top_k) {
#pragma unroll
                for (int x = 0; x < W; ++x) {
                    const float prod = w[q] * v[q][x];
                    acc[x] = acc[x] + prod;
                }
            }
    }
    V r;
    float *o = reinterpret_cast<float *>(&r);
#pragma unroll
    for (int x = 0; x < W; ++x) o[x] = shared ? acc[x] + shared[t * d + c * W + x] : acc[x];
    reinterpret_cast<V *>(out + t * d)[c] = r;
}

}  // namespace

double pg_moe_expected_tiles(size_t T, size_t E, size_t top_k, int slots) {
    const double p = (double)top_k / (double)E, mu = (double)T * p, sd = sqrt(std::max(mu * (1.0 - p), 1e-9));
    double tiles = 1.0 - pow(1.0 - p, (double)T);
    for (size_t j = 1; j * slots < T; ++j) {
        const double more = 0.5 * erfc(((double)(j * slots) + 0.5 - mu) / (sd * 1.41421356));
        if (more < 1e-4) break;
        tiles += more;
    }
    return tiles * (double)E;
}

// A table of device pointers (an expert set's planes) in a device buffer kept with the context, one per distinct
// table; uploaded (blocking: the source is the caller's stack frame) only on a table's first use.
pg_status pg_moe_cached_table(pg_ctx *ctx, const void *const *host_tab, size_t n, const void ***dev_tab) {
    for (size_t i = 0; i < ctx->moe_tabs.size(); ++i) {
        auto &t = ctx->moe_tabs[i];
        if (t.host.size() == n && memcmp(t.host.data(), host_tab, n * sizeof(void *)) == 0) {
            *dev_tab = static_cast<const void **>(t.dev);
            if (i + 1 != ctx->moe_tabs.size()) std::rotate(ctx->moe_tabs.begin() + i, ctx->moe_tabs.begin() + i + 1, ctx->moe_tabs.end());  // most recent last
            return PG_OK;
        }
    }
    // Least recently used out first.  A layer has two sets (row-major planes for one token, tile-major ones for
    // more), and a model alternates its layers: 512 sets hold both for 256 layers (the reference's Grok-1 has 64,
    // examples/grok1/model.rs:35), so a decode loop after a prefill misses on no layer.
    if (ctx->moe_tabs.size() >= 512) {  // a bounded cache: drop a set once nothing can still read it
        PG_HIP(hipStreamSynchronize(ctx->stream));
        (void)hipFree(ctx->moe_tabs.front().dev);
        ctx->moe_tabs.erase(ctx->moe_tabs.begin());
    }
    void *dev = nullptr;
    PG_HIP(pg_dev_malloc(ctx, &dev, n * sizeof(void *)));
    const hipError_t ce = hipMemcpy(dev, host_tab, n * sizeof(void *), hipMemcpyHostToDevice);
    if (ce != hipSuccess) {
        (void)hipFree(dev);
        return pg_fail(PG_EDEVICE, "uploading an expert table: %s", hipGetErrorString(ce));
    }
    ctx->moe_tabs.push_back({std::vector<const void *>(host_tab, host_tab + n), dev});
    *dev_tab = static_cast<const void **>(dev);
    return PG_OK;
}

// The routing of T tokens as the expert products want it: topk_idx / topk_p [T * top_k] (from the router's logits,
// grok1's softmax -> top-k, or a copy of the caller's own choice with out-of-range and repeated experts made
// harmless), and per expert the (token, k) pairs routed to it in ascending order (lists [E][T], counts [E]).
// With `goff` also the first of each expert's tiles of `tile` pairs, and their number in goff[E]; with `dig` the activation rows' digits too.
pg_status pg_launch_moe_routing(pg_ctx *ctx, const float *router_logits_dev, const int *idx_dev, const float *weight_dev, size_t T,
                                size_t E, size_t top_k, int *topk_idx, float *topk_p, int *lists, int *counts, int *goff, int tile,
                                const pg_moe_digits *dig) {
    if (route_in_one(T, E, top_k, router_logits_dev != nullptr)) {
        const size_t lds = route_lds(T, E, top_k, router_logits_dev != nullptr);
        route_digits rd = {};
        if (dig) {
            const int nb = (int)(dig->k / 32);
            rd = {dig->x, nb, (int)pg_round_up(nb, 4), (int)T * nb, dig->mm ? dig->mm->digits : dig->stream->digits, dig->mm ? dig->mm->xs : dig->stream->xs};
        }
        const dim3 grid(1 + (unsigned)((rd.blocks + 127) / 128));
        auto go = [&](auto *kern) {
            return pg_launch(ctx, dig ? "moe_route_lists_digits" : "moe_route_lists", kern, grid, dim3(1024), lds, router_logits_dev, idx_dev, weight_dev,
                             (int)T, (int)E, (int)top_k, topk_idx, topk_p, lists, counts, goff, tile, rd);
        };
        const bool nib = dig && dig->ggml_type == PG_GGML_Q4_0, by_logits = router_logits_dev != nullptr;
        switch (!dig ? 0 : (dig->mm ? 1 : 3) + !nib) {
            case 0: return by_logits ? go(route_lists_kernel<true, 0>) : go(route_lists_kernel<false, 0>);
            case 1: return by_logits ? go(route_lists_kernel<true, 1>) : go(route_lists_kernel<false, 1>);
            case 2: return by_logits ? go(route_lists_kernel<true, 2>) : go(route_lists_kernel<false, 2>);
            case 3: return by_logits ? go(route_lists_kernel<true, 3>) : go(route_lists_kernel<false, 3>);
            default: return by_logits ? go(route_lists_kernel<true, 4>) : go(route_lists_kernel<false, 4>);
        }
    }
    if (dig) PG_TRY(dig->mm ? pg_launch_x_to_mm_digits(ctx, dig->x, T, dig->k, dig->ggml_type, *dig->mm) : pg_launch_x_to_digits(ctx, dig->x, T, dig->k, dig->ggml_type, *dig->stream));
    if (router_logits_dev)
        PG_TRY(pg_launch(ctx, "moe_route_topk", route_topk_kernel, dim3(grid_for(T, 64)), dim3(64), 0,
                         router_logits_dev, (int)T, (int)E, (int)top_k, topk_idx, topk_p));
    else
        PG_TRY(pg_launch(ctx, "moe_copy_routing", copy_routing_kernel, dim3(grid_for(T, 64)), dim3(64), 0,
                         idx_dev, weight_dev, (int)T, (int)E, (int)top_k, topk_idx, topk_p));
    PG_TRY(pg_launch(ctx, "moe_expert_lists", expert_lists_kernel, dim3((unsigned)E), dim3(64), 0, (const int *)topk_idx,
                     (int)(T * top_k), (int)T, lists, counts));
    if (!goff) return PG_OK;
    return pg_launch(ctx, "moe_tile_offsets", tile_offsets_kernel, dim3(1), dim3(64), 0, (const int *)counts, (int)E, tile, goff);
}

// The expert FFN behind both entry points: the routing comes from `router_logits_dev` (grok1's softmax -> top-k) or,
// when that is null, from `idx_dev` / `weight_dev` as the caller's gate made them.
static pg_status moe_ffn_core(pg_ctx *ctx, const float *x_dev, size_t T, const float *router_logits_dev,
                              const int *idx_dev, const float *weight_dev, size_t E, size_t top_k,
                              const pg_gguf_tensor *const *gate, const pg_gguf_tensor *const *up,
                              const pg_gguf_tensor *const *down, int act, const float *shared_dev, float *out_dev) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(E >= 1 && E <= MAX_EXPERTS, "pg_moe_ffn: %zu experts (1..%d supported)", E, MAX_EXPERTS);
    PG_CHECK_ARG(top_k >= 1 && top_k <= E, "pg_moe_ffn: top_k %zu of %zu experts", top_k, E);
    PG_CHECK_ARG(act == PG_ACT_SILU || act == PG_ACT_GELU_TANH, "pg_moe_ffn: unknown activation %d", act);
    PG_CHECK_ARG(gate && up && down && gate[0] && up[0] && down[0], "pg_moe_ffn: null expert table");
    const size_t d = gate[0]->k_in, ffn = gate[0]->n_out;
    const int type = gate[0]->ggml_type;
    PG_CHECK_ARG(type == PG_GGML_Q4_0 || type == PG_GGML_Q8_0, "pg_moe_ffn: experts must be Q4_0 or Q8_0 block tensors");
    for (size_t e = 0; e < E; ++e) {
        PG_CHECK_ARG(gate[e] && up[e] && down[e], "pg_moe_ffn: expert %zu has a null tensor", e);
        PG_CHECK_ARG(gate[e]->k_in == d && gate[e]->n_out == ffn && up[e]->k_in == d &&
                         up[e]->n_out == ffn && down[e]->k_in == ffn && down[e]->n_out == d,
                     "pg_moe_ffn: expert %zu shapes do not match [ffn=%zu, d=%zu]", e, ffn, d);
        PG_CHECK_ARG(gate[e]->ggml_type == type && up[e]->ggml_type == type && down[e]->ggml_type == type,
                     "pg_moe_ffn: expert %zu mixes block types", e);
    }
    if (T == 0) return PG_OK;
    PG_CHECK_ARG(x_dev && (router_logits_dev || (idx_dev && weight_dev)) && out_dev, "pg_moe_ffn: null pointer");
    PG_CHECK_ARG((uintptr_t)x_dev % 16 == 0, "pg_moe_ffn: x must be 16-byte aligned");
    PG_CHECK_ARG(T * top_k < (1ull << 20), "pg_moe_ffn: too many (token, expert) pairs");
    const size_t P = T * top_k;

    // Which products take the streaming kernel (18 / 22-bit activations, one item per pair) instead
    // of the matrix-core one (16-bit activations per block):
    //  * a product whose own K spans only a few blocks (as everywhere);
    //  * all three when the experts are narrow (ffn < 512).  An error of 2^-16 of a block's
    //    absmax in g or u is multiplied by the partner factor in h = act(g) * u; where that factor
    //    is an outlier (|g| of 10 and more happens) the one h element carries an absolute error far
    //    above the others', and the down product only averages it away over many terms: its share
    //    of an output's error falls as 1 / sqrt(ffn) (measured 1.4e-3 of the row rms at ffn 64,
    //    below 2e-4 from ffn 2048 up).  Narrow experts are tiny products; the price is nil.
    const bool narrow = ffn < 512 && P <= 65535;
    // 3. one token: its top_k pairs meet top_k different experts with one activation row each, which is the
    //    streaming kernel's case (Grok-1-sized experts, Q8_0, top 2: 315 -> 227 us, the three products at 6.3 TB/s;
    //    from two tokens on pairs share experts and the matrix-core kernel, which reads an expert once, wins)
    const bool one_token = T == 1;
    const bool down_stream = narrow || one_token || ffn / 32 < PG_MM_MIN_BLOCKS, up_stream = down_stream || d / 32 < PG_MM_MIN_BLOCKS;
    // Their gate, up and act(gate) * up are then one launch, up to 150 MB of gate weights; beyond, three: workgroups of one wavefront stream more
    // evenly than the four whose block of 32 outputs becomes digits.  us, four launches : one, the layer: one token, 16 experts of 2304 x
    // 1376 (Q8_0) 26.2 : 18.0, 8 of 1024 x 2816, top 2 29.0 : 15.8, 8 of 4096 x 14336 (Q4_0) 52.9 : 47.1, Q8_0 (125 MB) 79.1 : 77.7; but 800 pairs
    // of 1024 x 256 (223 MB) 163 : 166, one token through 2 of 6144 x 32768 (428 MB) 211 : 218, 400 pairs of 2048 x 480 (418 MB) 198 : 225.
    const bool one_launch = down_stream && (double)P * (double)ffn * (double)d * (type == PG_GGML_Q4_0 ? 0.5625 : 1.0625) <= 1.5e8;
    PG_CHECK_ARG(!(up_stream || down_stream) || P <= 65535, "pg_moe_ffn: too many pairs for experts this small");

    // Arena layout.
    // (K chunks' planes stay apart: the launch that reads a product adds them.)
    const size_t pair_rows = pg_mm_pair_rows(ffn);
    int mt = 0, nw = 0;
    const bool as_tiles = !up_stream && !down_stream && pg_gguf_experts_tiles(ctx, type, T, E, top_k, d, ffn, &mt, &nw);
    const int ks_up = up_stream || as_tiles ? 1 : pg_gguf_mm_splitk(ctx, pair_rows, d, E, T, true, nullptr);
    const int ks_down = down_stream || as_tiles ? 1 : pg_gguf_mm_splitk(ctx, d, ffn, E, P, true, nullptr);
    const size_t sz_idx = pg_round_up(P * sizeof(int), 256);
    const size_t sz_p = pg_round_up(P * sizeof(float), 256);
    const size_t sz_lists = pg_round_up(E * T * sizeof(int), 256), sz_counts = pg_round_up(E * sizeof(int), 256);
    const size_t sz_gu = one_launch ? 0 : pg_round_up((size_t)ks_up * P * ffn * sizeof(float), 256), sz_y = pg_round_up((size_t)ks_down * P * d * sizeof(float), 256);
    const size_t sz_xd = up_stream ? pg_xdigits_bytes(T, d) : pg_mmdigits_bytes(T, d);
    const size_t sz_hd = down_stream ? pg_xdigits_bytes(P, ffn) : pg_mmdigits_bytes(P, ffn);
    void *ws = nullptr;
    PG_TRY(pg_workspace(ctx, sz_idx + sz_p + sz_lists + sz_counts + 2 * sz_gu + sz_y + sz_xd + sz_hd, &ws));
    char *p = static_cast<char *>(ws);
    int *topk_idx = reinterpret_cast<int *>(p); p += sz_idx;
    float *topk_p = reinterpret_cast<float *>(p); p += sz_p;
    int *lists = reinterpret_cast<int *>(p); p += sz_lists;
    int *counts = reinterpret_cast<int *>(p); p += sz_counts;
    float *g = reinterpret_cast<float *>(p); p += sz_gu;
    float *u = reinterpret_cast<float *>(p); p += sz_gu;
    float *yb = reinterpret_cast<float *>(p); p += sz_y;
    char *xd_base = p; p += sz_xd;
    char *hd_base = p;

    // Expert pointer tables: [gate qs | gate d | up qs | up d | down qs | down d], E each, in a
    // device buffer kept with the context, one per distinct set of experts (a model's layers
    // alternate); uploaded (blocking: the source is this stack frame) only on a set's first use.
    // The quant planes are the tile-major copies (made on an expert's first use) for the
    // matrix-core kernel, the row-major planes for the streaming one.
    const void *host_tab[6 * MAX_EXPERTS];
    for (size_t e = 0; e < E; ++e) {
        if (!up_stream) {
            PG_TRY(pg_gguf_ensure_tiled(ctx, gate[e]));
            PG_TRY(pg_gguf_ensure_tiled(ctx, up[e]));
        }
        if (!down_stream) PG_TRY(pg_gguf_ensure_tiled(ctx, down[e]));
        host_tab[0 * E + e] = up_stream ? gate[e]->qs : gate[e]->qs_tiled; host_tab[1 * E + e] = gate[e]->d;
        host_tab[2 * E + e] = up_stream ? up[e]->qs : up[e]->qs_tiled;     host_tab[3 * E + e] = up[e]->d;
        host_tab[4 * E + e] = down_stream ? down[e]->qs : down[e]->qs_tiled; host_tab[5 * E + e] = down[e]->d;
    }
    const void **tab = nullptr;
    PG_TRY(pg_moe_cached_table(ctx, host_tab, 6 * E, &tab));

    const pg_xdigits xd = pg_xdigits_carve(xd_base, T, d);
    const pg_mmdigits xm = pg_mmdigits_carve(xd_base, T, d);  // (the one or the other is used)
    const pg_moe_digits dig = {x_dev, d, type, up_stream ? nullptr : &xm, up_stream ? &xd : nullptr};
    PG_TRY(pg_launch_moe_routing(ctx, router_logits_dev, idx_dev, weight_dev, T, E, top_k, topk_idx, topk_p, lists, counts, nullptr, 1, &dig));
    auto table = [&](int which) { return reinterpret_cast<const uint8_t *const *>(tab + which * E); };
    auto dtable = [&](int which) { return reinterpret_cast<const uint16_t *const *>(tab + which * E); };
    // Each token reaches an expert at most once, so an expert owns at most T pairs.
    const int tiles = (int)((T + 31) / 32);
    const pg_gemv_batch bg = {(int)P, table(0), dtable(1), topk_idx, (int)top_k};  // pair p: activation row p / top_k against expert topk_idx[p]
    if (one_launch) {
        PG_TRY(pg_launch_gguf_gemv_act_digits(ctx, type, ffn, d, bg, table(2), dtable(3), act, xd, pg_xdigits_carve(hd_base, P, ffn)));
    } else if (up_stream) {
        PG_TRY(pg_launch_gguf_gemv(ctx, type, ffn, d, nullptr, nullptr, bg, xd, g));
        const pg_gemv_batch bu = {(int)P, table(2), dtable(3), topk_idx, (int)top_k};
        PG_TRY(pg_launch_gguf_gemv(ctx, type, ffn, d, nullptr, nullptr, bu, xd, u));
    } else {
        pg_mm_group gg = {(int)E, table(0), dtable(1), lists, counts, (int)T, tiles, (int)T, (int)top_k, 0, 0, 1};
        gg.nseg = -1;  // gate and up in one launch
        gg.qs_table2 = table(2);
        gg.d_table2 = dtable(3);
        gg.out2 = u;
        PG_TRY(as_tiles ? pg_launch_gguf_experts_tiles(ctx, type, ffn, d, gg, P, mt, nw, xm, g)
                        : pg_launch_gguf_mm(ctx, type, ffn, d, nullptr, nullptr, gg, P, xm, g, g, true));
    }
    const int nb = (int)(ffn / 32);
    const dim3 blocks(grid_for(nb, 32), (unsigned)P);
    const bool nib = type == PG_GGML_Q4_0;
    if (down_stream) {
        const pg_xdigits hd = pg_xdigits_carve(hd_base, P, ffn);
        if (!one_launch)
            PG_TRY(pg_launch(ctx, "moe_act_digits", nib ? act_digits_kernel<true> : act_digits_kernel<false>, blocks, dim3(256), 0, (const float *)g,
                             (const float *)u, act, nb, hd.digits, hd.xs));
        const pg_gemv_batch bd = {(int)P, table(4), dtable(5), topk_idx, 1};
        PG_TRY(pg_launch_gguf_gemv(ctx, type, d, ffn, nullptr, nullptr, bd, hd, yb));
    } else {
        const pg_mmdigits hd = pg_mmdigits_carve(hd_base, P, ffn);
        auto *kern = nib ? act_mm_digits_kernel<true> : act_mm_digits_kernel<false>;
        if (P > 65535) return pg_fail(PG_EUNSUPPORTED, "pg_moe_ffn: more than 65535 pairs");
        PG_TRY(pg_launch(ctx, "moe_act_mm_digits", kern, blocks, dim3(256), 0, (const float *)g, (const float *)u,
                         ks_up, P * ffn, act, nb, (int)pg_round_up(nb, 4), hd.digits, hd.xs));
        const pg_mm_group gd = {(int)E, table(4), dtable(5), lists, counts, (int)T, tiles, (int)T, 1, 0, 0, 1};
        PG_TRY(as_tiles ? pg_launch_gguf_experts_tiles(ctx, type, d, ffn, gd, P, mt, nw, hd, yb)
                        : pg_launch_gguf_mm(ctx, type, d, ffn, nullptr, nullptr, gd, P, hd, yb, yb, true));
    }
    // (below, four columns a thread leave too few wavefronts: 2 tokens of 1248 23.5 us against 22.9)
    const bool vec = T * d >= 65536 && d % 4 == 0 && (((uintptr_t)yb | (uintptr_t)out_dev | (uintptr_t)shared_dev) & 15) == 0;
    const size_t columns = vec ? d / 4 : d;
    const unsigned wg = (unsigned)std::min<size_t>(256, pg_round_up(columns, 64)), per = grid_for(columns, wg);
    PG_CHECK_ARG(T * per < ((size_t)1 << 31), "pg_moe_ffn: %zu tokens of %zu outputs in one launch", T, d);
    return pg_launch(ctx, "moe_combine", ks_down > 1 ? (vec ? combine_kernel<float4, 4> : combine_kernel<float, 4>) : (vec ? combine_kernel<float4, 1> : combine_kernel<float, 1>), dim3((unsigned)(T * per)), dim3(wg), 0,
                     (const float *)yb, ks_down, P * d, (const float *)topk_p, per, (int)d, (int)top_k, shared_dev, out_dev);
}

PG_API pg_status pg_moe_ffn_dev(pg_ctx *ctx, const float *x_dev, size_t T,
                                const float *router_logits_dev, size_t E, size_t top_k,
                                const pg_gguf_tensor *const *gate, const pg_gguf_tensor *const *up,
                                const pg_gguf_tensor *const *down, int act, float *out_dev) {
    PG_CHECK_ARG(T == 0 || router_logits_dev, "pg_moe_ffn: null router logits");
    return moe_ffn_core(ctx, x_dev, T, router_logits_dev, nullptr, nullptr, E, top_k, gate, up, down, act, nullptr, out_dev);
}

PG_API pg_status pg_moe_ffn_routed_dev(pg_ctx *ctx, const float *x_dev, size_t T, const int32_t *expert_idx_dev,
                                       const float *weight_dev, size_t E, size_t top_k,
                                       const pg_gguf_tensor *const *gate, const pg_gguf_tensor *const *up,
                                       const pg_gguf_tensor *const *down, int act, const float *shared_dev, float *out_dev) {
    PG_CHECK_ARG(T == 0 || (expert_idx_dev && weight_dev), "pg_moe_ffn_routed: null routing");
    return moe_ffn_core(ctx, x_dev, T, nullptr, expert_idx_dev, weight_dev, E, top_k, gate, up, down, act, shared_dev, out_dev);
}

PG_API pg_status pg_moe_ffn_routed(pg_ctx *ctx, const float *x, size_t T, const int32_t *expert_idx, const float *weight,
                                   size_t E, size_t top_k, const pg_gguf_tensor *const *gate,
                                   const pg_gguf_tensor *const *up, const pg_gguf_tensor *const *down, int act,
                                   const float *shared, float *out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(gate && gate[0], "pg_moe_ffn_routed: null expert table");
    if (T == 0) return PG_OK;
    PG_CHECK_ARG(x && expert_idx && weight && out, "pg_moe_ffn_routed: null pointer");
    PG_CHECK_ARG(E >= 1 && E <= MAX_EXPERTS && top_k >= 1 && top_k <= E, "pg_moe_ffn_routed: top_k %zu of %zu experts", top_k, E);
    // the reference indexes self.experts[expert_idx] and would panic on an index out of range; a token's experts are
    // distinct in every gate on this path (the grouped products rely on it)
    for (size_t t = 0; t < T; ++t)
        for (size_t k = 0; k < top_k; ++k) {
            const int32_t e = expert_idx[t * top_k + k];
            PG_CHECK_ARG(e >= 0 && (size_t)e < E, "pg_moe_ffn_routed: token %zu names expert %d of %zu", t, (int)e, E);
            for (size_t j = 0; j < k; ++j)
                PG_CHECK_ARG(expert_idx[t * top_k + j] != e, "pg_moe_ffn_routed: token %zu names expert %d twice", t, (int)e);
        }
    const size_t d = gate[0]->k_in, P = T * top_k;
    pg_dev_block dx, di, dw, dsh, dout;
    PG_TRY(dout.alloc(ctx, T * d * sizeof(float)));
    PG_TRY(pg_host_in(ctx, x, T * d * sizeof(float), dx));
    PG_TRY(pg_host_in(ctx, expert_idx, P * sizeof(int32_t), di));
    PG_TRY(pg_host_in(ctx, weight, P * sizeof(float), dw));
    if (shared) PG_TRY(pg_host_in(ctx, shared, T * d * sizeof(float), dsh));
    PG_TRY(pg_moe_ffn_routed_dev(ctx, dx.as<float>(), T, di.as<int32_t>(), dw.as<float>(), E, top_k, gate, up, down, act,
                                 shared ? dsh.as<float>() : nullptr, dout.as<float>()));
    return pg_host_out(ctx, out, dout.p, T * d * sizeof(float));
}

PG_API pg_status pg_moe_ffn(pg_ctx *ctx, const float *x, size_t T, const float *router_logits,
                            size_t E, size_t top_k, const pg_gguf_tensor *const *gate,
                            const pg_gguf_tensor *const *up, const pg_gguf_tensor *const *down,
                            int act, float *out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(gate && gate[0], "pg_moe_ffn: null expert table");
    if (T == 0) return PG_OK;
    PG_CHECK_ARG(x && router_logits && out, "pg_moe_ffn: null pointer");
    const size_t d = gate[0]->k_in;
    pg_dev_block dx, dl, dout;
    PG_TRY(dout.alloc(ctx, T * d * sizeof(float)));
    PG_TRY(pg_host_in(ctx, x, T * d * sizeof(float), dx));
    PG_TRY(pg_host_in(ctx, router_logits, T * E * sizeof(float), dl));
    PG_TRY(pg_moe_ffn_dev(ctx, dx.as<float>(), T, dl.as<float>(), E, top_k, gate, up, down, act, dout.as<float>()));
    return pg_host_out(ctx, out, dout.p, T * d * sizeof(float));
}
