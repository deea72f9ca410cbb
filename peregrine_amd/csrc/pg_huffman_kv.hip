// peregrine's HuffmanKVCache: a key/value cache whose older tokens are quantised to int8 with
// one scale per head and Huffman-coded in chunks, with a window of recent tokens kept as f32.
//
//   HuffmanKVCache::new / append / compress_oldest_chunk / remove_oldest_tokens   reference: src/huffman.rs:517-610
//   HuffmanKVCache::compress_chunk / decompress_chunk                             reference: src/huffman.rs:612-680
//   HuffmanKVCache::len / get_kv                                                  reference: src/huffman.rs:683-724
//
// Everything is device work here, and all the chunks that one append cuts (both sides) are one batch of three or four
// launches: the heads' absolute maxima and the int8 values with a histogram per 4096 of them (one launch, or for large batches two); the code table, one
// workgroup a chunk, which also turns the small histograms into the bit at which each 4096 values start; and the
// encoder.  The host takes part once per batch: it learns the coded sizes (words that the table kernel stores in
// pinned memory) and allocates exactly that much, or, from a cache's second batch on, has launched the encoder into what the
// batch before took and 1 / 64 where that suits (at most 1 / 32 too much; compress_batch).  A batch was 10 launches, 12 copies and 8
// waits per pair of chunks before, and the tables were built on the host from copied histograms: 3000 tokens of
// 8 x 128, appended 512 at a time in chunks of 256 and read back, took 3.9-4.5 ms, of which 0.8 ms of kernels; now 0.16.
//
// The encoder knows where every code starts, so it leaves an index beside the stream (a 16-bit offset per 64 values,
// 0.25 bit a value): the decoder of such a chunk is one launch that starts a thread per 64 values, with no search for
// code boundaries, and writes the scaled f32 values into the caller's layout.  A chunk made from stored parts has no
// index and goes through the self-synchronising decoder of the Huffman-coded weights and a scaling launch.
#include <atomic>
#include <chrono>
#include <memory>
#include <new>
#include <vector>
#include "pg_internal.h"
#include "pg_quant_dev.h"

namespace {

constexpr int NUM_SYMBOLS = 256;
constexpr int KV_MAX_BITS = 12;                // longest code (src/huffman.rs:30)
constexpr int KV_LUT = 1 << KV_MAX_BITS;
constexpr int KV_LEVELS = 96;                  // words: by length, the first 12 bits beyond its codes, then where its symbols start less its first code; the symbols by code
constexpr int KV_WG = 256;
constexpr int ENC_SPT = 16;                    // symbols per thread of the encoder
constexpr int ENC_PER_WG = KV_WG * ENC_SPT;    // symbols per workgroup: one histogram and one start bit each
constexpr int SUB_SYMS = 64;                   // symbols per entry of the index, and per thread of the decoder
constexpr int DEC_PER_WG = KV_WG * SUB_SYMS;   // symbols per workgroup of the decoder
constexpr unsigned KV_MAX_SPLITS = 64;         // workgroups per head of the maximum and scaling kernels
constexpr size_t KV_BATCH_SYMBOLS = 64u << 20; // symbols of one batch: bounds what a batch takes of the scratch arena
constexpr unsigned KV_BATCH_CHUNKS = 2048;     // and its chunks

// Device layout of a coded chunk: [scales][code lengths][decode table]{[start bit per 4096][offset per 64]}[stream, padded].
struct kv_layout {
    size_t o_book, o_lut, o_wg, o_sub, o_bits;
    __host__ __device__ kv_layout(size_t heads, size_t total, bool indexed) {
        const size_t nwg = (total + ENC_PER_WG - 1) / ENC_PER_WG, nsub = (total + SUB_SYMS - 1) / SUB_SYMS;
        o_book = (heads * sizeof(float) + 255) / 256 * 256;
        o_lut = o_book + NUM_SYMBOLS;
        o_wg = o_lut + KV_LUT * sizeof(uint16_t);
        o_sub = o_wg + (indexed ? (nwg + 1) * sizeof(unsigned long long) : 0);
        o_bits = (o_sub + (indexed ? nsub * sizeof(uint16_t) : 0) + 255) / 256 * 256;
    }
    // with the stream's last word whole and 16 bytes of zeros behind it
    __host__ __device__ size_t size(unsigned long long bytes) const { return (o_bits + (bytes + 3) / 4 * 4 + 16 + 255) / 256 * 256; }
};

// One batch: chunk c of `count` is side c % sides, number c / sides of that side; its head h starts at
// data[side] + number * chunk_step + h * head_stride, head_elems values.  Scratch is per chunk, back to back.
struct kv_batch {
    const float *data[2];
    size_t chunk_step, head_stride;
    unsigned sides, count, heads, head_elems, total, nwg, splits;
    float *amax;                  // [count][heads][splits]
    float *scales;                // [count][heads]
    int8_t *q;                    // [count][q_stride]
    size_t q_stride;
    uint16_t *hist;               // [count][nwg][256]
    unsigned long long *wg_bit;   // [count][nwg + 1] start bits, then the total
    unsigned *codes;              // [count][256] length << 16 | code
    unsigned *levels;             // [count][KV_LEVELS] what the decode table is made of
    __device__ const float *head(unsigned c, unsigned h) const { return data[c % sides] + (size_t)(c / sides) * chunk_step + (size_t)h * head_stride; }
};

// New rows on their way into the window, for the batch's first launch to write while it reads them: a head's values from `from`
// on are `elems` values at src[side] + h * src_stride.  No rows: from is beyond every chunk and parts is 0.
struct kv_incoming {
    const float *src[2];
    float *dst[2];  // where they go, heads `dst_stride` apart
    size_t src_stride, dst_stride, from, elems;
    unsigned parts;  // times as many workgroups per (side, head) as a chunk's head has
};

// Lane exchange by DPP: the value of lane ^ D.
template <int D> __device__ __forceinline__ unsigned lane_xor(unsigned v) {
    if constexpr (D == 1) return __builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);        // quad_perm 1 0 3 2
    else if constexpr (D == 2) return __builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);   // quad_perm 2 3 0 1
    else if constexpr (D == 3) return __builtin_amdgcn_mov_dpp((int)v, 0x1B, 0xF, 0xF, true);   // quad_perm 3 2 1 0
    else if constexpr (D == 7) return __builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    else if constexpr (D == 15) return __builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, true); // row_mirror
    else if constexpr (D == 4) return lane_xor<3>(lane_xor<7>(v));
    else if constexpr (D == 8) return __builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);  // row_ror 8
    else if constexpr (D == 31) return lane_xor<16>(lane_xor<15>(v));
    else if constexpr (D == 63) return lane_xor<32>(lane_xor<31>(v));
    else {
        const auto two = D == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false) : __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return threadIdx.x & D ? two[0] : two[1];
    }
}
template <int D> __device__ __forceinline__ unsigned long long lane_xor(unsigned long long v) {
    return (unsigned long long)lane_xor<D>((unsigned)(v >> 32)) << 32 | lane_xor<D>((unsigned)v);
}
// Largest |v| of every head (NaN ignored, as f32::max does), one value per split; and the incoming rows' copy.  Grid
// (heads * splits, chunks + sides * parts).  As two launches the copy took 4 us of an append's 43.
template <class V>
__global__ __launch_bounds__(KV_WG) void kv_absmax_kernel(const kv_batch b, const kv_incoming in) {
    constexpr unsigned VN = sizeof(V) / 4;
    __shared__ float red[4];
    const unsigned split = blockIdx.x % b.splits, h = blockIdx.x / b.splits, c = blockIdx.y;
    if (c >= b.count) {
        const unsigned side = (c - b.count) / in.parts, part = (c - b.count) % in.parts * b.splits + split;
        const V *src = reinterpret_cast<const V *>(in.src[side] + (size_t)h * in.src_stride);
        V *dst = reinterpret_cast<V *>(in.dst[side] + (size_t)h * in.dst_stride);
        for (size_t i = (size_t)part * KV_WG + threadIdx.x; i < in.elems / VN; i += (size_t)in.parts * b.splits * KV_WG) dst[i] = src[i];
        return;
    }
    const size_t at = (size_t)(c / b.sides) * b.chunk_step;  // of the head's first value in the window
    const V *p = reinterpret_cast<const V *>(b.head(c, h));
    const V *q = reinterpret_cast<const V *>(in.src[c % b.sides] + (size_t)h * in.src_stride);
    const unsigned n = b.head_elems / VN, old = (unsigned)min((size_t)n, (in.from > at ? in.from - at : 0) / VN);
    const size_t skip = at / VN - in.from / VN;  // of q's values, from window to incoming (wraps where the chunk starts in the window)
    float m = 0.0f;
    for (unsigned i = split * KV_WG + threadIdx.x; i < n; i += b.splits * KV_WG) {
        const V v = i < old ? p[i] : q[skip + i];
        const float *x = reinterpret_cast<const float *>(&v);
#pragma unroll
        for (unsigned k = 0; k < VN; ++k) m = fmaxf(m, fabsf(x[k]));
    }
    m = pg_block_max_256(m, red);
    if (threadIdx.x == 0) b.amax[((size_t)c * b.heads + h) * b.splits + split] = m;
}

// q = round(v / scale) clamped to +-127 with scale = amax / 127 (1 for an all-zero head), the scales, and the
// histogram of each workgroup's ENC_PER_WG values (a table per wavefront: fewer lanes meet on a common value).
// src/huffman.rs:624-646.  Grid (nwg, chunks).
__global__ __launch_bounds__(KV_WG) void kv_quant_hist_kernel(const kv_batch b, int vec) {
    __shared__ unsigned lh[4][NUM_SYMBOLS];
    __shared__ float sc[ENC_PER_WG];  // scales of the heads the workgroup meets (every value its own head at the most)
    const unsigned c = blockIdx.y, t = threadIdx.x, base = blockIdx.x * ENC_PER_WG;
    const unsigned last = min(base + ENC_PER_WG, b.total) - 1;
    const unsigned h0 = base / b.head_elems, h1 = last / b.head_elems;
    float4 v[ENC_SPT / 4];
    if (vec)  // four values of one head each
#pragma unroll
        for (int j = 0; j < ENC_SPT / 4; ++j) {
            const unsigned i = base + (j * KV_WG + t) * 4, h = i / b.head_elems;
            if (i < b.total) v[j] = *reinterpret_cast<const float4 *>(b.head(c, h) + (i - h * b.head_elems));
        }
    for (unsigned h = h0 + t; h <= h1; h += KV_WG) {
        const float *a = b.amax + ((size_t)c * b.heads + h) * b.splits;
        float m = 0.0f;
#pragma unroll 8
        for (unsigned s = 0; s < b.splits; ++s) m = fmaxf(m, a[s]);
        const float scale = (m == 0.0f) ? 1.0f : m / 127.0f;
        sc[h - h0] = scale;
        if (base <= h * b.head_elems) b.scales[(size_t)c * b.heads + h] = scale;  // the workgroup of the head's first value
    }
    for (int i = 0; i < 4; ++i) lh[i][t] = 0;
    __syncthreads();
    unsigned *mine = lh[t >> 6];
    int8_t *q = b.q + (size_t)c * b.q_stride;
#pragma unroll
    for (int j = 0; j < ENC_SPT / 4; ++j) {
        const unsigned i = base + (j * KV_WG + t) * 4;
        if (vec) {
            if (i >= b.total) continue;
            const float inv = 1.0f / sc[i / b.head_elems - h0];
            const int x0 = pg_quant_to_i8(v[j].x * inv), x1 = pg_quant_to_i8(v[j].y * inv), x2 = pg_quant_to_i8(v[j].z * inv), x3 = pg_quant_to_i8(v[j].w * inv);
            *reinterpret_cast<unsigned *>(q + i) = (x0 & 255) | (x1 & 255) << 8 | (x2 & 255) << 16 | (unsigned)x3 << 24;
            atomicAdd(mine + x0 + 128, 1u);
            atomicAdd(mine + x1 + 128, 1u);
            atomicAdd(mine + x2 + 128, 1u);
            atomicAdd(mine + x3 + 128, 1u);
        } else {
            for (unsigned k = i; k < i + 4 && k < b.total; ++k) {
                const unsigned h = k / b.head_elems;
                const int x = pg_quant_to_i8(b.head(c, h)[k - h * b.head_elems] * (1.0f / sc[h - h0]));
                q[k] = (int8_t)x;
                atomicAdd(mine + x + 128, 1u);
            }
        }
    }
    __syncthreads();
    b.hist[((size_t)c * b.nwg + blockIdx.x) * NUM_SYMBOLS + t] = (uint16_t)(lh[0][t] + lh[1][t] + lh[2][t] + lh[3][t]);
}

// Both of the above in one launch, for heads of which every workgroup can afford to look at the whole: a workgroup takes
// 4096 values, finds the maximum of each head that they meet by itself (what the workgroups of a head read in common
// comes out of the L2), quantises its values and counts them.  New rows are read where the caller has them; workgroups behind
// the chunks' write them to the window.  Grid 8 * ceil(nwg / 8) * chunks + sides * heads * parts.
//
// Taken while the repeated reads cost less than a launch: us, both launches : this, by chunks of heads x values: 2 x 4 x 4096
// 7.0 : 4.0; 4 x 8 x 32768 7.2 : 5.6; 2 x 8 x 49152 7.4 : 6.2; 2 x 8 x 65536 7.3 : 7.0; but 8 x 8 x 32768 7.8 : 8.0, 8 x 32 x 16384 9.7 : 11.4,
// 2 x 2 x 262144 7.7 : 15.8.  (Runs dealt to the XCDs one by one: 8 x 8 x 32768 13.1.)
constexpr unsigned WHOLE_WG = 1024;
constexpr size_t WHOLE_HEAD = 65536, WHOLE_READS = 12u << 20;  // values of a head, and that all workgroups read together, at the most
template <class V>
__global__ __launch_bounds__(WHOLE_WG) __attribute__((amdgpu_waves_per_eu(8, 8))) void kv_whole_kernel(const kv_batch b, const kv_incoming in) {
    constexpr unsigned VN = sizeof(V) / 4, PER = ENC_PER_WG / WHOLE_WG / VN;
    __shared__ unsigned lh[4][NUM_SYMBOLS];
    __shared__ float sc[ENC_PER_WG];  // scales of the heads the workgroup meets (every value its own head at the most)
    __shared__ unsigned red[2][WHOLE_WG / 64];
    const unsigned t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const unsigned per_xcd = (b.nwg + 7) / 8;  // workgroup id % 8 = XCD: each takes consecutive runs, so that few of them read a head
    if (blockIdx.x >= 8 * per_xcd * b.count) {
        const unsigned g = blockIdx.x - 8 * per_xcd * b.count, row = g / in.parts, side = row / b.heads, h = row % b.heads;
        const V *src = reinterpret_cast<const V *>(in.src[side] + (size_t)h * in.src_stride);
        V *dst = reinterpret_cast<V *>(in.dst[side] + (size_t)h * in.dst_stride);
        for (size_t i = (size_t)(g % in.parts) * WHOLE_WG + t; i < in.elems / VN; i += (size_t)in.parts * WHOLE_WG) dst[i] = src[i];
        return;
    }
    const unsigned c = blockIdx.x / (8 * per_xcd), run = (blockIdx.x & 7) * per_xcd + blockIdx.x / 8 % per_xcd, base = run * ENC_PER_WG;
    if (run >= b.nwg) return;
    const unsigned last = min(base + ENC_PER_WG, b.total) - 1, h0 = base / b.head_elems, h1 = last / b.head_elems;
    const size_t at = (size_t)(c / b.sides) * b.chunk_step;  // of the head's first value in the window
    const unsigned n = b.head_elems / VN, old = (unsigned)min((size_t)n, (in.from > at ? in.from - at : 0) / VN);
    const size_t skip = at / VN - in.from / VN;  // of the incoming values, from window to incoming (wraps where the chunk starts in the window)
    const float *src = in.src[c % b.sides];
    auto load = [&](unsigned h, unsigned i) {
        return i < old ? reinterpret_cast<const V *>(b.head(c, h))[i] : reinterpret_cast<const V *>(src + (size_t)h * in.src_stride)[skip + i];
    };
    V v[PER];
#pragma unroll
    for (unsigned j = 0; j < PER; ++j) {
        const unsigned i = base + (j * WHOLE_WG + t) * VN, h = i / b.head_elems;
        if (i < b.total) v[j] = load(h, (i - h * b.head_elems) / VN);
    }
    if (t < 4 * NUM_SYMBOLS) (&lh[0][0])[t] = 0;
    // |v| of all but NaN is in order as bits
    auto max_of = [&](unsigned h, unsigned from, unsigned step) {
        float m = 0.0f;
#pragma unroll 8
        for (unsigned i = from; i < n; i += step) {
            const V x = load(h, i);
            const float *f = reinterpret_cast<const float *>(&x);
#pragma unroll
            for (unsigned k = 0; k < VN; ++k) m = fmaxf(m, fabsf(f[k]));
        }
        unsigned r = __float_as_uint(m);
        r = max(r, lane_xor<1>(r));
        r = max(r, lane_xor<2>(r));
        r = max(r, lane_xor<4>(r));
        r = max(r, lane_xor<8>(r));
        r = max(r, lane_xor<16>(r));
        return max(r, lane_xor<32>(r));
    };
    auto scale_is = [&](unsigned h, unsigned bits) {
        const float m = __uint_as_float(bits), scale = (m == 0.0f) ? 1.0f : m / 127.0f;
        sc[h - h0] = scale;
        if (base <= h * b.head_elems) b.scales[(size_t)c * b.heads + h] = scale;  // the workgroup of the head's first value
    };
    if (b.head_elems >= 2048) {  // three heads at the most
        for (unsigned h = h0; h <= h1; ++h) {
            const unsigned r = max_of(h, t, WHOLE_WG);
            if (lane == 0) red[(h - h0) & 1][wave] = r;
            __syncthreads();
            if (wave == 0) {
                unsigned m = red[(h - h0) & 1][lane & 15];
                m = max(m, lane_xor<1>(m));
                m = max(m, lane_xor<2>(m));
                m = max(m, lane_xor<4>(m));
                m = max(m, lane_xor<8>(m));
                if (lane == 0) scale_is(h, m);
            }
        }
    } else {
        for (unsigned h = h0 + wave; h <= h1; h += WHOLE_WG / 64) {
            const unsigned r = max_of(h, lane, 64);
            if (lane == 0) scale_is(h, r);
        }
    }
    __syncthreads();
    unsigned *mine = lh[wave & 3];
    int8_t *q = b.q + (size_t)c * b.q_stride;
#pragma unroll
    for (unsigned j = 0; j < PER; ++j) {
        const unsigned i = base + (j * WHOLE_WG + t) * VN;
        if (i >= b.total) continue;
        const float inv = 1.0f / sc[i / b.head_elems - h0];
        const float *f = reinterpret_cast<const float *>(&v[j]);
        unsigned four = 0;
#pragma unroll
        for (unsigned k = 0; k < VN; ++k) {
            const int x = pg_quant_to_i8(f[k] * inv);
            four |= (x & 255u) << (8 * k);
            atomicAdd(mine + x + 128, 1u);
        }
        if (VN == 4) *reinterpret_cast<unsigned *>(q + i) = four;
        else q[i] = (int8_t)four;
    }
    __syncthreads();
    if (t < NUM_SYMBOLS) b.hist[((size_t)c * b.nwg + run) * NUM_SYMBOLS + t] = (uint16_t)(lh[0][t] + lh[1][t] + lh[2][t] + lh[3][t]);
}

// The smaller of both for end = 0, the larger for end = ~0: one instruction, their median with `end`.
__device__ __forceinline__ unsigned end_of(unsigned x, unsigned o, unsigned end) { return max(min(x, o), min(max(x, o), end)); }
__device__ __forceinline__ unsigned long long end_of(unsigned long long x, unsigned long long o, unsigned end) { return (end != 0) == (o > x) ? o : x; }
// The smaller of a lane and lane ^ D stays where bit B of the lane is clear, the larger where it is set.
template <int D, int B, class K> __device__ __forceinline__ void order_pair(K &x) {
    const unsigned end = threadIdx.x & B ? ~0u : 0u;
    if constexpr (sizeof(K) == 4 && (D == 16 || D == 32)) {  // the swap leaves both in every lane
        const auto two = D == 16 ? __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false) : __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
        x = end_of(two[0], two[1], end);
    } else x = end_of(x, lane_xor<D>(x), end);
}
// A bitonic sequence of 64 lanes into ascending order.
template <class K> __device__ __forceinline__ void order_bitonic(K &x) {
    order_pair<32, 32>(x);
    order_pair<16, 16>(x);
    order_pair<8, 8>(x);
    order_pair<4, 4>(x);
    order_pair<2, 2>(x);
    order_pair<1, 1>(x);
}
// Any 64 into ascending order: runs of 2, 4, .. 64 by meeting their mirror image.
template <class K> __device__ __forceinline__ void order_wave(K &x) {
    order_pair<1, 1>(x);
    order_pair<3, 2>(x); order_pair<1, 1>(x);
    order_pair<7, 4>(x); order_pair<2, 2>(x); order_pair<1, 1>(x);
    order_pair<15, 8>(x); order_pair<4, 4>(x); order_pair<2, 2>(x); order_pair<1, 1>(x);
    order_pair<31, 16>(x); order_pair<8, 8>(x); order_pair<4, 4>(x); order_pair<2, 2>(x); order_pair<1, 1>(x);
    order_pair<63, 32>(x); order_pair<16, 16>(x); order_pair<8, 8>(x); order_pair<4, 4>(x); order_pair<2, 2>(x); order_pair<1, 1>(x);
}

// Running sum over the lanes of a row of 16.
__device__ __forceinline__ unsigned row_scan(unsigned v) {
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);
    return v;
}

// And over a wavefront's.
__device__ __forceinline__ unsigned wave_scan(unsigned v) {
    v = row_scan(v);
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, true);  // row_bcast 15 into rows 1 and 3, then 31 into rows 2 and 3
    v += __builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, true);
    return v;
}

// LDS that one wavefront writes and reads: its accesses happen in program order, so only the compiler has to keep it.
__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// The Huffman merges of n leaves on one wavefront; returns the number of rounds.  Two queues, leaves and the nodes made of
// them, both ascending, of keys weight << 9 | id (ids of nodes from NUM_SYMBOLS on), with NONE behind their ends.  The sum m of
// the two lightest trees is the smallest weight that a new node can have, so all trees of weight <= m are taken, two
// by two, before any node that the round makes (a tie goes to the one that was there first: a leaf before a node).  A
// round puts the 64 lightest of both queues' heads in order across the lanes -- min of the one ascending and the other
// descending is bitonic, six exchanges of two instructions -- and pairs neighbours, up to 32 at a time.
constexpr unsigned TREE_PAD = NUM_SYMBOLS + 64;  // (a round reads 64 from a queue's head on; what is not taken is written behind)
template <class K>
__device__ __forceinline__ unsigned merge_trees(unsigned n, const K *leaf_key, K *node_key, unsigned *parent) {
    const unsigned lane = threadIdx.x & 63;
    unsigned lh = 0, qh = 0, made = 0, rounds = 0;
    for (unsigned alive = n; alive > 1; ++rounds) {
        K x = min(leaf_key[lh + lane], node_key[qh + 63 - lane]);
        order_bitonic(x);
        const unsigned id = (unsigned)x & 511u, w = (unsigned)(x >> 9), sum = w + lane_xor<1>(w);
        const unsigned m = __builtin_amdgcn_readlane(sum, 0);
        const unsigned taken = min((unsigned)__popcll(__ballot(w <= m)), alive) & ~1u, node = made + lane / 2;  // (two at least)
        const bool in = lane < taken;
        node_key[in ? node : TREE_PAD] = (K)sum << 9 | (NUM_SYMBOLS + node);
        const unsigned leaves = __popcll(__ballot(id < NUM_SYMBOLS) & ~0ull >> (64 - taken));
        parent[in ? id : 2 * NUM_SYMBOLS - 1] = node;
        lh += leaves;
        qh += taken - leaves;
        made += taken / 2;
        alive -= taken / 2;
        wave_lds_fence();  // the nodes are read by other lanes
    }
    return rounds;
}

// The chunk's code table and where its 4096-value runs start: one workgroup of 1024 a chunk.  K holds weight << 9 | id: 32
// bits for chunks below 2^23 values, else 64.
//
// Lengths as HuffmanTable::from_frequencies gives them (src/huffman.rs:35-150: two queues over the symbols sorted by
// frequency, a leaf wins a tie; depths clamped to 12), and where the clamp over-subscribes the code the same repair
// as table_that_decodes in pg_huffman.hip.
//
// One workgroup on its CU, so what counts is the chain of dependent steps.  What one wavefront can do alone it does
// without a barrier (merges, depths, counts, repair), exchanges are DPP moves with one instruction each to order a pair, and
// the histograms stay in registers until the runs' bits are known.  A chunk of 262144 normally distributed values, cycles
// (with every symbol compared with every other, exchanges by compare and select, queues that a round pads itself, and
// branches around its stores): histograms 2.5 k, order 1.8 k (4.5 k), merges 7.4 k for 18 rounds (13.9 k), depths and counts 2 k, repair 1.5 k
// (3.2 k), codes and runs 2 k (6 k): 9.3 us where it was 15.9; 16384 values 8.1 (13.0).  The decode table is left to the encoder's launch,
// which the host does not wait for, and the host hears of the stream's bits before codes and runs: an append's next one is
// on its way 1.3 us earlier.
constexpr unsigned KEPT_ROWS = 4;  // histograms a wavefront keeps: 16 wavefronts, so all of a chunk of up to 64 of them
template <class K>
__global__ __launch_bounds__(1024) void kv_table_kernel(const kv_batch b, unsigned long long *host_bits) {
    constexpr K NONE = ~(K)0;
    __shared__ __attribute__((aligned(16))) unsigned freq[NUM_SYMBOLS];
    __shared__ K order[2][NUM_SYMBOLS];
    __shared__ unsigned rank_down[NUM_SYMBOLS];  // by place in the ascending order
    __shared__ K leaf_key[TREE_PAD], node_key[TREE_PAD + 1];
    __shared__ unsigned leaf_w[NUM_SYMBOLS];
    __shared__ uint8_t leaf_sym[NUM_SYMBOLS], leaf_len[NUM_SYMBOLS];
    __shared__ unsigned parent[2 * NUM_SYMBOLS];  // of the leaves (by ascending frequency), then of the nodes
    __shared__ unsigned up_tree[NUM_SYMBOLS];     // of the nodes: levels << 16 | ancestor
    __shared__ __attribute__((aligned(16))) unsigned cnt[16], first_code[16], limit[16], offset[16];
    __shared__ unsigned lane_cnt[4][16];
    __shared__ __attribute__((aligned(16))) uint8_t bl[NUM_SYMBOLS];
    __shared__ __attribute__((aligned(16))) uint8_t by_len[NUM_SYMBOLS];
    __shared__ unsigned over, wsum[16], stream_sum[4][2];
    __shared__ unsigned run_bits[1024];
    const unsigned c = blockIdx.x, t = threadIdx.x, s = t & 255, p = t >> 8;
    const unsigned lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint2 *rows = reinterpret_cast<const uint2 *>(b.hist + (size_t)c * b.nwg * NUM_SYMBOLS);  // four counts of 16 bits
    const bool kept = b.nwg <= 16 * KEPT_ROWS;

    // a wavefront adds up every sixteenth row, four rows in flight
    uint2 h[KEPT_ROWS];
#pragma unroll
    for (unsigned k = 0; k < KEPT_ROWS; ++k) h[k] = wave + 16 * k < b.nwg ? rows[(size_t)(wave + 16 * k) * 64 + lane] : uint2{0, 0};
    if (t < 16) {
        cnt[t] = 0;
        limit[t] = ~0u;
    }
    if (p == 0) {
        freq[s] = ~0u;  // (kept less one: what is not in use then comes behind all others)
        bl[s] = 0;
    }
    if (t < TREE_PAD) leaf_key[t] = node_key[t] = NONE;
    __syncthreads();
    {
        unsigned sum[4] = {0, 0, 0, 0};
        for (unsigned i = wave;;) {
#pragma unroll
            for (unsigned k = 0; k < KEPT_ROWS; ++k) { sum[0] += h[k].x & 0xFFFFu; sum[1] += h[k].x >> 16; sum[2] += h[k].y & 0xFFFFu; sum[3] += h[k].y >> 16; }
            i += 16 * KEPT_ROWS;
            if (i >= b.nwg) break;
#pragma unroll
            for (unsigned k = 0; k < KEPT_ROWS; ++k) h[k] = i + 16 * k < b.nwg ? rows[(size_t)(i + 16 * k) * 64 + lane] : uint2{0, 0};
        }
        if (wave < b.nwg)
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) atomicAdd(&freq[4 * lane + k], sum[k]);
    }
    __syncthreads();
    // Symbols in order of frequency, ties by symbol: four wavefronts put 64 each in order, then runs of 128 and 256 meet their
    // mirror image through LDS.  Place t of the ascending order ends up with thread t.
    unsigned n = 0;  // symbols in use
#pragma unroll
    for (unsigned k = 0; k < 4; ++k) n += __popcll(__ballot(freq[64 * k + lane] != ~0u));
    {
        const unsigned f = freq[s] + 1;
        K x = f ? (K)f << 8 | s : NONE;
        if (p == 0) {
            order_wave(x);
            order[0][t] = x;
        }
        __syncthreads();
        if (p == 0) {
            x = end_of(x, order[0][t ^ 127], t & 64 ? ~0u : 0u);
            order_bitonic(x);
            order[1][t] = x;
        }
        __syncthreads();
        if (p == 0) {
            x = end_of(x, order[1][t ^ 255], t & 128 ? ~0u : 0u);
            order[0][t] = x;
        }
        __syncthreads();
        if (p == 0) {
            x = end_of(x, order[0][t ^ 64], t & 64 ? ~0u : 0u);
            order_bitonic(x);
            if (t < n) {
                leaf_w[t] = (unsigned)(x >> 8);
                leaf_key[t] = x >> 8 << 9 | t;
                leaf_sym[t] = (uint8_t)x;
            }
        }
    }
    __syncthreads();
    if (wave == 0) {
        const unsigned rounds = merge_trees<K>(n, leaf_key, node_key, parent);
        // the nodes' levels below the root: everyone takes over its ancestor's way up (a round adds at most one level)
        unsigned up[4];
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
            const unsigned node = 64 * k + lane, of = parent[NUM_SYMBOLS + node];
            up[k] = node + 2 < n ? 1u << 16 | of : node;
            up_tree[node] = up[k];
        }
        for (unsigned reach = 1; reach < rounds; reach *= 2) {
            wave_lds_fence();
            unsigned a[4];
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) a[k] = up_tree[up[k] & 0xFFFFu];
            wave_lds_fence();
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) up_tree[64 * k + lane] = up[k] = (up[k] & ~0xFFFFu) + a[k];
        }
        wave_lds_fence();
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
            const unsigned leaf = 64 * k + lane, of = parent[leaf], levels = up_tree[leaf < n && n > 1 ? of : 0] >> 16;
            const unsigned len = leaf >= n ? 0u : n < 2 ? 1u : min(levels + 1u, (unsigned)KV_MAX_BITS);
            leaf_len[leaf] = (uint8_t)len;
            atomicAdd(&cnt[len], 1u);
        }
        wave_lds_fence();
        unsigned cn = lane >= 1 && lane <= KV_MAX_BITS ? cnt[lane] : 0u;  // lane l holds the number of codes of length l
        auto get = [&](int l) { return (unsigned)__builtin_amdgcn_readlane(cn, l); };
        auto add = [&](int l, unsigned x) { cn += lane == (unsigned)l ? x : 0u; };
        int excess = pg_wave_sum_i32((int)(cn * (lane <= KV_MAX_BITS ? KV_LUT >> lane : 0))) - KV_LUT;  // of the Kraft sum, in 1 / 4096
        const bool too_many = excess > 0;
        if (too_many) {
            // While there is too much, lengthen by a bit the least frequent symbol of the deepest level below the limit:
            // it stays the deepest until it gets there, so whole symbols go to the limit level by level, as many as the
            // excess holds, and the last one part of the way.
            int l = KV_MAX_BITS - 1;
#pragma unroll 1
            for (; l >= 1 && excess > 0; --l) {
                const int gain = (KV_LUT >> l) - 1;
                const unsigned had = get(l);
                unsigned x = (unsigned)((float)excess / (float)gain);  // (both below 2^21: off by one at the most)
                if ((int)x * gain > excess) --x;
                else if ((int)(x + 1) * gain <= excess) ++x;
                x = min(x, had);
                add(l, 0u - x);
                add(KV_MAX_BITS, x);
                excess -= (int)x * gain;
                if (excess > 0 && had > x) break;
            }
#pragma unroll 1
            for (; l >= 1 && l < KV_MAX_BITS && excess > 0; ++l) {
                add(l, ~0u);
                add(l + 1, 1u);
                excess -= KV_LUT >> (l + 1);
            }
            unsigned slack = (unsigned)-excess;  // and what is left goes to the most frequent symbols
            const unsigned all = cn;
            unsigned from = 1;
#pragma unroll 1
            for (;;) {  // the next length with symbols that the slack can shorten
                const unsigned long long can = __ballot(lane > from && lane <= KV_MAX_BITS && all > 0 && (unsigned)(KV_LUT >> (lane & 15)) <= slack);
                if (!can) break;
                from = (unsigned)__ffsll((unsigned long long)can) - 1;
                unsigned had = (unsigned)__builtin_amdgcn_readlane(all, from);
#pragma unroll 1
                for (; had > 0 && (unsigned)(KV_LUT >> from) <= slack; --had) {
                    unsigned to = from;
#pragma unroll 1
                    for (; to > 1 && (unsigned)(KV_LUT >> to) <= slack; --to) slack -= KV_LUT >> to;
                    add(from, ~0u);
                    add(to, 1u);
                }
            }
        }
        // src/huffman.rs:152-186: the codes of a length follow those of the shorter ones
        unsigned kraft = lane <= KV_MAX_BITS ? cn << (KV_MAX_BITS - lane) : 0u, off = cn;
        const unsigned own = kraft;
        kraft = row_scan(kraft);
        off = row_scan(off);
        if (lane >= 1 && lane <= KV_MAX_BITS + 1) {
            offset[lane] = off - cn;
            if (lane <= KV_MAX_BITS) {
                first_code[lane] = (kraft - own) >> (KV_MAX_BITS - lane);
                limit[lane] = kraft;
            }
        }
        if (lane == 0) over = too_many;
    } else if (wave >= 4 && wave < 8) {  // meanwhile the descending order, ties by symbol
        const unsigned i = t - 256;
        if (i < n) {
            const unsigned w = leaf_w[i];
            unsigned lo = 0, hi = 0;  // leaves below w, and of at most w
#pragma unroll 1
            for (unsigned step = 256; step > 0; step >>= 1) {
                if (lo + step <= n && leaf_w[lo + step - 1] < w) lo += step;
                if (hi + step <= n && leaf_w[hi + step - 1] <= w) hi += step;
            }
            rank_down[i] = n - hi + i - lo;
        }
    }
    __syncthreads();
    unsigned out_len = 0;
    if (t < n) {
        unsigned len = leaf_len[t];
        if (over) {  // the repaired lengths go out again, shortest to most frequent (ties: lower symbol first)
            const unsigned down = rank_down[t];
            len = 1;
#pragma unroll
            for (int l = 2; l <= KV_MAX_BITS; ++l) len += offset[l] <= down ? 1 : 0;
        }
        out_len = len;
        bl[leaf_sym[t]] = (uint8_t)len;
    }
    // The stream's bits go to the host as soon as they are known: it makes room and launches the encoder meanwhile, and the caller has its
    // next append on the way (microseconds that the device otherwise waits out behind the encoder).
    if (p == 0) {
        const unsigned long long bits = t < n ? (unsigned long long)leaf_w[t] * out_len : 0ull;  // (below 2^35)
        const unsigned lo = (unsigned)pg_wave_sum_i32((int)(bits & 0xFFFFFu)), hi = (unsigned)pg_wave_sum_i32((int)(bits >> 20));
        if (lane == 0) {
            stream_sum[wave][0] = lo;
            stream_sum[wave][1] = hi;
        }
    }
    __syncthreads();
    if (t == 1023) {
        unsigned long long bits = 1;  // (0 = not there yet)
        for (unsigned w = 0; w < 4; ++w) bits += stream_sum[w][0] + ((unsigned long long)stream_sum[w][1] << 20);
        __hip_atomic_store(host_bits + c, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // the symbol's place among those of its length
    unsigned before = 0, len = 0;
    if (p == 0) {
        len = bl[s];
        unsigned of_len = 0;  // lane l: symbols of length l
#pragma unroll
        for (unsigned l = 1; l <= KV_MAX_BITS; ++l) {
            const unsigned long long m = __ballot(len == l);
            if (len == l) before = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            if (lane == l) of_len = __popcll(m);
        }
        if (lane < 16) lane_cnt[wave][lane] = of_len;
    }
    const unsigned lens = reinterpret_cast<const unsigned *>(bl)[lane];
    const unsigned lens_lo = (lens & 255u) | (lens & 0xFF00u) << 8, lens_hi = (lens >> 16 & 255u) | (lens & 0xFF000000u) >> 8;
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    auto u2 = [](unsigned v) { return __builtin_bit_cast(u16x2, v); };
    auto bits_of = [&](uint2 v) {
        return (unsigned)pg_wave_sum_i32((int)__builtin_amdgcn_udot2(u2(v.x), u2(lens_lo), __builtin_amdgcn_udot2(u2(v.y), u2(lens_hi), 0u, false), false));
    };
    unsigned long long *wg_bit = b.wg_bit + (size_t)c * (b.nwg + 1);
    if (kept) {
#pragma unroll
        for (unsigned k = 0; k < KEPT_ROWS; ++k)
            if (wave + 16 * k < b.nwg) {
                const unsigned bits = bits_of(h[k]);
                if (lane == 0) run_bits[wave + 16 * k] = bits;
            }
    }
    __syncthreads();
    if (p == 0) {
        unsigned e = 0;
        if (len) {
#pragma unroll
            for (unsigned w = 0; w < 3; ++w) before += w < wave ? lane_cnt[w][len] : 0u;
            e = len << 16 | (first_code[len] + before);
            by_len[offset[len] + before] = (uint8_t)s;
        }
        b.codes[(size_t)c * NUM_SYMBOLS + s] = e;
    }
    // where the runs start, and the stream's bits
    unsigned long long run = 0;
    if (kept) {
        if (wave == 4) {
            const unsigned v = lane < b.nwg ? run_bits[lane] : 0u, incl = wave_scan(v);
            if (lane < b.nwg) wg_bit[lane] = incl - v;
            run = (unsigned)__builtin_amdgcn_readlane(incl, 63);
            if (lane == 0) wg_bit[b.nwg] = run;
        }
    } else {
        for (unsigned at = 0; at < b.nwg; at += 1024) {
            for (unsigned i = at + wave; i < min(at + 1024u, b.nwg); i += 16) {
                const unsigned bits = bits_of(rows[(size_t)i * 64 + lane]);
                if (lane == 0) run_bits[i - at] = bits;
            }
            __syncthreads();
            const unsigned v = at + t < b.nwg ? run_bits[t] : 0u;
            const unsigned incl = wave_scan(v);
            if (lane == 63) wsum[wave] = incl;
            __syncthreads();
            unsigned long long pre = run;
            for (unsigned w = 0; w < wave; ++w) pre += wsum[w];
            if (at + t < b.nwg) wg_bit[at + t] = pre + incl - v;
            for (unsigned w = 0; w < 16; ++w) run += wsum[w];
            __syncthreads();
        }
        if (t == 256) wg_bit[b.nwg] = run;
    }
    __syncthreads();
    if (t < KV_LEVELS) b.levels[(size_t)c * KV_LEVELS + t] = t < 16 ? limit[t] : t < 32 ? offset[t - 16] - first_code[t - 16] : reinterpret_cast<const unsigned *>(by_len)[t - 32];
}

// Four entries of the decode table, length << 8 | symbol; codes nobody has decode as (length 0, value 0).
__device__ __forceinline__ ushort4 lut_entries(const unsigned *levels, unsigned x) {
    const unsigned *limit = levels, *start = levels + 16;
    const uint8_t *by_len = reinterpret_cast<const uint8_t *>(levels + 32);
    unsigned l = 1;  // (the limits ascend)
#pragma unroll
    for (int i = 1; i <= KV_MAX_BITS; ++i) l += x >= limit[i] ? 1 : 0;
    ushort4 e;
    uint16_t *ev = reinterpret_cast<uint16_t *>(&e);
    auto entry = [&](unsigned x, unsigned l) { return l > KV_MAX_BITS ? (uint16_t)128 : (uint16_t)(l << 8 | by_len[start[l] + (x >> (KV_MAX_BITS - l))]); };
    if (l <= KV_MAX_BITS - 2 || l > KV_MAX_BITS) {  // one code for the four, or none
        ev[0] = ev[1] = ev[2] = ev[3] = entry(x, l);
    } else {
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
            while (l <= KV_MAX_BITS && x + k >= limit[l]) ++l;
            ev[k] = entry(x + k, l);
        }
    }
    return e;
}

__host__ __device__ inline unsigned long long kv_stream_bytes(unsigned long long bits) { return (bits + 7) / 8; }

// Where up to KV_PLACES chunks of a batch, from number `first` on, are written to.
constexpr unsigned KV_PLACES = 32;
struct kv_places {
    unsigned first;
    char *at[KV_PLACES];
    // GUESSED: bytes that every chunk of a side has for its stream; what all chunks have to need, in units of 256 bytes
    unsigned long long room[2];
    unsigned least;
    // the window's rows that move to the front in the same launch (workgroups behind the chunks', which read the int8
    // values only): heads of both sides, `rest` values each, from `from` values on
    float *hot[2];
    size_t hot_stride, from, rest;
    bool vec;  // in steps of 16 bytes
};

// p[i] = p[from + i] for i < rest, where rest may be the longer: a thread takes whole chains i, i + from, i + 2 from, .. , so that what it
// overwrites only it reads, and it has read it before.  (A launch per `from` values moved took 3.2 us each.)
template <class V> __device__ __forceinline__ void move_to_front(V *p, size_t from, size_t rest, size_t first, size_t step) {
    for (size_t i = first; i < min(from, rest); i += step) {
        size_t j = i;
        for (; j + 3 * from < rest; j += 4 * from) {
            const V v0 = p[j + from], v1 = p[j + 2 * from], v2 = p[j + 3 * from], v3 = p[j + 4 * from];
            p[j] = v0;
            p[j + from] = v1;
            p[j + 2 * from] = v2;
            p[j + 3 * from] = v3;
        }
        for (; j < rest; j += from) p[j] = p[j + from];
    }
}

// Appends the code `e` (length << 16 | code) to a right-aligned window; returns the next whole word if one is full.
__device__ __forceinline__ bool push_code(unsigned e, unsigned long long &acc, unsigned &nacc, unsigned &word) {
    const unsigned l = e >> 16;
    acc = (acc << l) | (e & 0xFFFFu);
    nacc += l;
    if (nacc < 32) return false;
    nacc -= 32;
    word = (unsigned)(acc >> nacc);
    acc &= (1ull << nacc) - 1ull;
    return true;
}

// HuffmanTable::encode (src/huffman.rs:216-251) in parallel: grid (nwg + 1, chunks).  A workgroup's bit range is
// known; its threads put their codes together in LDS and the workgroup stores the words that START in its
// range, whole: the bits that the last of them takes from the next run it encodes itself (up to 31 values), so no word
// has two writers and nothing is zeroed first.  The last workgroup of a chunk writes its head and the decode table.  What bounds it is
// latency: with all loads ahead of the first wait and the head beside the runs, 20 chunks of 262144 values take 5.7 us (one
// after another 6.7).
// GUESSED: launched before the host knows the sizes.  Unless every stream of the batch fits its room, and the rooms are not much too
// large, the launch does nothing at all -- no stream is written and the window does not move -- and the host, which decides by
// the same sizes, takes over.
template <bool GUESSED>
__global__ __launch_bounds__(KV_WG) void kv_encode_kernel(const kv_batch b, const kv_places places, char **__restrict__ table) {
    __shared__ unsigned lc[NUM_SYMBOLS], wsum[4];
    __shared__ unsigned words[ENC_PER_WG * KV_MAX_BITS / 32 + 2], follow[32];
    const unsigned c = places.first + blockIdx.y, g = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const kv_layout lay(b.heads, b.total, true);
    // all that a run needs is requested at once, ahead of the first use of any of it
    const unsigned cc = min(c, b.count - 1);
    const unsigned long long stream_bits = b.wg_bit[(size_t)min(lane, b.count - 1) * (b.nwg + 1) + b.nwg];
    const unsigned long long *wg_bit = b.wg_bit + (size_t)cc * (b.nwg + 1);
    const unsigned long long first = wg_bit[g], last = wg_bit[min(g + 1, b.nwg)];
    const unsigned code = b.codes[(size_t)cc * NUM_SYMBOLS + t];
    const int8_t *q = b.q + (size_t)cc * b.q_stride;
    const unsigned base = g * ENC_PER_WG + t * ENC_SPT;
    const unsigned count = base >= b.total ? 0u : min(b.total - base, (unsigned)ENC_SPT);
    const uint4 v = *reinterpret_cast<const uint4 *>(q + (count ? base : 0));  // (q is padded to a multiple of 16)
    const unsigned beyond = (g + 1) * ENC_PER_WG + (t & 31);
    const uint8_t after = (uint8_t)q[min(beyond, b.total - 1)];
    if constexpr (GUESSED) {
        const bool second = b.sides == 2 && (lane & 1);  // (of the sides, also 64 chunks on)
        const unsigned long long room0 = places.room[0], room1 = places.room[1], room = second ? room1 : room0;
        const unsigned long long bytes = kv_stream_bytes(stream_bits);
        bool fits = lane >= b.count || bytes <= room;
        unsigned need = lane >= b.count ? 0u : (unsigned)(lay.size(bytes) / 256);
        for (unsigned i = lane + 64; i < b.count; i += 64) {
            const unsigned long long more = kv_stream_bytes(b.wg_bit[(size_t)i * (b.nwg + 1) + b.nwg]);
            fits = fits && more <= room;
            need += (unsigned)(lay.size(more) / 256);
        }
        if (__ballot(!fits) || (unsigned)pg_wave_sum_i32((int)need) < places.least) return;  // (the same for all workgroups)
    }
    if (c >= b.count) {
        const unsigned row = c - b.count;
        float *p = (row < b.heads ? places.hot[0] : places.hot[1]) + (size_t)(row % b.heads) * places.hot_stride;
        if (places.vec) move_to_front(reinterpret_cast<float4 *>(p), places.from / 4, places.rest / 4, (size_t)g * KV_WG + t, (size_t)gridDim.x * KV_WG);
        else move_to_front(p, places.from, places.rest, (size_t)g * KV_WG + t, (size_t)gridDim.x * KV_WG);
        return;
    }
    char *dst = places.at[blockIdx.y];
    if (g == b.nwg) {  // the chunk's head, with the decode table
        if (t < KV_LEVELS) words[t] = b.levels[(size_t)c * KV_LEVELS + t];
        for (unsigned h = t; h < b.heads; h += KV_WG) reinterpret_cast<float *>(dst)[h] = b.scales[(size_t)c * b.heads + h];
        dst[lay.o_book + t] = (char)(code >> 16);
        if (t == 0) {
            reinterpret_cast<unsigned long long *>(dst + lay.o_wg)[b.nwg] = first;
            if (table) table[c] = dst;
        }
        if (t < 4) reinterpret_cast<unsigned *>(dst + lay.o_bits)[(size_t)((first + 31) >> 5) + t] = 0;  // the padding
        __syncthreads();
        for (unsigned i = t; i < KV_LUT / 4; i += KV_WG) reinterpret_cast<ushort4 *>(dst + lay.o_lut)[i] = lut_entries(words, 4 * i);
        return;
    }
    lc[t] = code;
    for (unsigned i = t; i < sizeof(words) / 4; i += KV_WG) words[i] = 0;
    // the values that may fill this run's last word up: 31 bits, a value takes at least one
    if (t < 32) follow[t] = beyond < b.total ? after ^ 128u : NUM_SYMBOLS;
    __syncthreads();
    const unsigned sw[4] = {v.x, v.y, v.z, v.w};
    unsigned e[ENC_SPT], bits = 0;
#pragma unroll
    for (unsigned j = 0; j < ENC_SPT; ++j) {
        e[j] = j < count ? lc[((sw[j >> 2] >> (8 * (j & 3))) & 255u) ^ 128u] : 0u;
        bits += e[j] >> 16;
    }
    const unsigned incl = wave_scan(bits);
    if (lane == 63) wsum[t >> 6] = incl;
    __syncthreads();
    unsigned start = incl - bits;  // within the run
    for (unsigned w = 0; w < (t >> 6); ++w) start += wsum[w];
    if (count && (t & (SUB_SYMS / ENC_SPT - 1)) == 0)
        reinterpret_cast<uint16_t *>(dst + lay.o_sub)[base / SUB_SYMS] = (uint16_t)start;  // below 4096 * 12
    const unsigned r = (unsigned)(first & 31);  // bits of the first word that belong to the run before
    {
        unsigned k = (r + start) >> 5, nacc = (r + start) & 31, word;
        unsigned long long acc = 0;
#pragma unroll
        for (unsigned j = 0; j < ENC_SPT; ++j)
            if (push_code(e[j], acc, nacc, word)) atomicOr(&words[k++], word);
        if (nacc && count) atomicOr(&words[k], (unsigned)(acc << (32 - nacc)));
    }
    __syncthreads();
    if (t == 0 && ((unsigned)last & 31)) {  // fill the last word up from the next run
        unsigned nacc = (unsigned)last & 31, k = (unsigned)((last >> 5) - (first >> 5)), word;
        unsigned long long acc = words[k] >> (32 - nacc);
        bool full = false;
        for (unsigned i = 0; !full && i < 32 && follow[i] < NUM_SYMBOLS; ++i) full = push_code(lc[follow[i]], acc, nacc, word);
        words[k] = full ? word : (unsigned)(acc << (32 - nacc));
    }
    __syncthreads();
    unsigned *out = reinterpret_cast<unsigned *>(dst + lay.o_bits) + (size_t)(first >> 5);
    const unsigned nwords = (unsigned)(((last + 31) >> 5) - (first >> 5));
    for (unsigned i = t + (r ? 1 : 0); i < nwords; i += KV_WG) out[i] = __builtin_bswap32(words[i]);
    if (t == 0) reinterpret_cast<unsigned long long *>(dst + lay.o_wg)[g] = first;
}

// Chunks with an index, decoded, scaled and laid out, and the window copied behind them.  Chunk c (address table[c], or
// `single`) is side c % sides, number c / sides: its head h goes to out[side] + number * chunk_step + h * out_stride.
struct kv_decode_args {
    char *const *table;
    const char *single;
    float *out[2];
    size_t chunk_step, out_stride;
    unsigned sides, count, heads, head_elems, total, wgs;  // wgs = workgroups per chunk
    const float *hot[2];       // window rows: head h at hot[side] + h * hot_stride, hot_elems values to out[side] + hot_at + h * out_stride
    size_t hot_stride, hot_at;
    unsigned hot_elems, hot_wgs;  // hot_wgs = workgroups per (side, head)
};

// A thread decodes SUB_SYMS values from the bit the index names: table and stream in LDS (the workgroup's part of the
// stream is contiguous), a 64-bit window in registers with the next word already read; the values go through LDS so
// that the f32 stores are whole lines.  What it takes is the chain of 64 table look-ups, about 100 ns each:
// 20 chunks of 262144 values in 14.3 us, 8 of 16384 in 10.8 (16.8 and 13.5 with the window filled up under a branch after every value;
// the search for code boundaries, the scans, the write pass and the scaling launch took 170).  Loads marked as global memory instead
// of flat ones are 0.4 us slower here.
template <bool VEC>
__global__ __launch_bounds__(KV_WG) void kv_decode_kernel(const kv_decode_args a) {
    constexpr unsigned MAX_WORDS = DEC_PER_WG * KV_MAX_BITS / 32 + 4;
    __shared__ __attribute__((aligned(16))) uint16_t lut[KV_LUT];
    __shared__ unsigned words[MAX_WORDS];
    constexpr unsigned DEC_SCALES = 64;
    __shared__ float sc[DEC_SCALES];  // of the first heads that the workgroup meets
    __shared__ unsigned sym[KV_WG * (SUB_SYMS / 4 + 1)];  // four values a word; a thread's words start an odd number apart
    const unsigned t = threadIdx.x, nchunk = a.count * a.wgs;
    if (blockIdx.x >= nchunk) {  // the window
        const unsigned g = blockIdx.x - nchunk, row = g / a.hot_wgs, part = g % a.hot_wgs, side = row / a.heads, h = row % a.heads;
        const float *src = a.hot[side] + (size_t)h * a.hot_stride;
        float *dst = a.out[side] + a.hot_at + (size_t)h * a.out_stride;
        const unsigned end = min(a.hot_elems, (part + 1) * DEC_PER_WG);
        if (VEC)
            for (unsigned i = part * DEC_PER_WG + t * 4; i < end; i += KV_WG * 4) *reinterpret_cast<float4 *>(dst + i) = *reinterpret_cast<const float4 *>(src + i);
        else
            for (unsigned i = part * DEC_PER_WG + t; i < end; i += KV_WG) dst[i] = src[i];
        return;
    }
    const unsigned c = blockIdx.x / a.wgs, g = blockIdx.x % a.wgs;
    const char *chunk = a.table ? a.table[c] : a.single;
    const kv_layout lay(a.heads, a.total, true);
    const uint4 *lut_g = reinterpret_cast<const uint4 *>(chunk + lay.o_lut);
    uint4 lut_v[KV_LUT * 2 / 16 / KV_WG];
#pragma unroll
    for (unsigned i = 0; i < KV_LUT * 2 / 16 / KV_WG; ++i) lut_v[i] = lut_g[i * KV_WG + t];
    constexpr unsigned RUNS = DEC_PER_WG / ENC_PER_WG;
    const unsigned long long *wg_bit = reinterpret_cast<const unsigned long long *>(chunk + lay.o_wg);
    const unsigned nwg = (a.total + ENC_PER_WG - 1) / ENC_PER_WG, r0 = g * RUNS, r1 = min(r0 + RUNS, nwg);
    const unsigned long long w0 = wg_bit[r0] >> 5, w1 = (wg_bit[r1] + 31) >> 5;
    const unsigned *stream = reinterpret_cast<const unsigned *>(chunk + lay.o_bits) + w0;
    const unsigned nwords = min((unsigned)(w1 - w0) + 3, MAX_WORDS);  // (up to 16 bytes of padding follow a stream)
    const float *scales = reinterpret_cast<const float *>(chunk);
    const unsigned h0 = g * DEC_PER_WG / a.head_elems;
    const float scale_t = scales[min(h0 + (t & (DEC_SCALES - 1)), a.heads - 1)];
    const unsigned base = g * DEC_PER_WG, sub = g * KV_WG + t;
    const unsigned count = base + t * SUB_SYMS >= a.total ? 0u : min(a.total - (base + t * SUB_SYMS), (unsigned)SUB_SYMS), from = count ? sub : 0;
    const unsigned pos = (unsigned)(wg_bit[from / (ENC_PER_WG / SUB_SYMS)] - (w0 << 5)) + reinterpret_cast<const uint16_t *>(chunk + lay.o_sub)[from];
    for (unsigned at = 0; at < nwords; at += 8 * KV_WG) {  // eight loads in flight
        unsigned w[8];
#pragma unroll
        for (unsigned j = 0; j < 8; ++j) w[j] = stream[min(at + j * KV_WG + t, nwords - 1)];
#pragma unroll
        for (unsigned j = 0; j < 8; ++j)
            if (at + j * KV_WG + t < nwords) words[at + j * KV_WG + t] = __builtin_bswap32(w[j]);
    }
#pragma unroll
    for (unsigned i = 0; i < KV_LUT * 2 / 16 / KV_WG; ++i) reinterpret_cast<uint4 *>(lut)[i * KV_WG + t] = lut_v[i];
    if (t < DEC_SCALES) sc[t] = scale_t;
    __syncthreads();
    if (count) {
        unsigned k = pos >> 5;
        unsigned long long buf = ((unsigned long long)words[k] << 32 | words[k + 1]) << (pos & 31);
        unsigned avail = 64 - (pos & 31);
        k += 2;
        unsigned next = words[k];
        unsigned *o = sym + t * (SUB_SYMS / 4 + 1);
        for (unsigned j = 0; j < count; j += 4) {
            unsigned four = 0;
#pragma unroll
            for (unsigned i = 0; i < 4; i += 2) {
                // more than 32 bits hold two codes: the window is filled up once for both, and without a branch
                const bool low = avail <= 32;
                buf |= (unsigned long long)(low ? next : 0u) << ((32 - avail) & 63);
                avail += low ? 32 : 0;
                k = min(k + (low ? 1u : 0u), MAX_WORDS - 1);
                next = words[k];
#pragma unroll
                for (unsigned x = 0; x < 2; ++x) {
                    const unsigned e = lut[buf >> (64 - KV_MAX_BITS)], l = e >> 8;
                    four |= (e & 255u) << (8 * (i + x));
                    buf <<= l;
                    avail -= l;
                }
            }
            o[j / 4] = four;
        }
    }
    __syncthreads();
    float *out = a.out[c % a.sides] + (size_t)(c / a.sides) * a.chunk_step;
#pragma unroll 4
    for (unsigned j = 0; j < DEC_PER_WG / (4 * KV_WG); ++j) {
        const unsigned local = (j * KV_WG + t) * 4, i = base + local;
        if (i >= a.total) break;
        const unsigned four = sym[local / SUB_SYMS * (SUB_SYMS / 4 + 1) + local % SUB_SYMS / 4];
        if (VEC) {
            const unsigned h = i / a.head_elems;
            const float scale = h - h0 < DEC_SCALES ? sc[h - h0] : scales[h];
            float4 v;
            v.x = (float)((int)(four & 255u) - 128) * scale;
            v.y = (float)((int)(four >> 8 & 255u) - 128) * scale;
            v.z = (float)((int)(four >> 16 & 255u) - 128) * scale;
            v.w = (float)((int)(four >> 24) - 128) * scale;
            *reinterpret_cast<float4 *>(out + (size_t)h * a.out_stride + (i - h * a.head_elems)) = v;
        } else {
            for (unsigned k = 0; k < 4 && i + k < a.total; ++k) {
                const unsigned h = (i + k) / a.head_elems;
                out[(size_t)h * a.out_stride + (i + k - h * a.head_elems)] = (float)((int)(four >> (8 * k) & 255u) - 128) * scales[h];
            }
        }
    }
}

// decoded_i8 as f32 * scale[head]   src/huffman.rs:669-677 for several chunks in one launch: grid
// (splits, heads, chunks); chunk c's values start at q + q_off and go to rows of out_stride floats per head.
struct dequant_item {
    const float *scales;
    float *out;
    size_t q_off, head_elems, out_stride;
};

__global__ __launch_bounds__(KV_WG) void kv_dequant_kernel(const int8_t *__restrict__ q, const dequant_item *__restrict__ items) {
    const dequant_item it = items[blockIdx.z];
    const float scale = it.scales[blockIdx.y];
    const int8_t *p = q + it.q_off + (size_t)blockIdx.y * it.head_elems;
    float *o = it.out + (size_t)blockIdx.y * it.out_stride;
    for (size_t i = (size_t)blockIdx.x * KV_WG + threadIdx.x; i < it.head_elems; i += (size_t)gridDim.x * KV_WG)
        o[i] = (float)p[i] * scale;
}

unsigned splits_for(size_t head_elems) {
    const size_t s = (head_elems + 4 * KV_WG - 1) / (4 * KV_WG);
    return (unsigned)std::min<size_t>(std::max<size_t>(s, 1), KV_MAX_SPLITS);
}

}  // namespace

// CompressedChunk  src/huffman.rs:500-513 in device memory (kv_layout).
struct pg_huffman_kv_chunk {
    mutable uint8_t codebook[NUM_SYMBOLS];  // copies of what the device holds, once `on_host`
    mutable std::vector<float> scales;
    mutable bool on_host = false;
    std::shared_ptr<pg_dev_block> block;  // shared by the chunks of a batch
    char *dev = nullptr;
    size_t bytes = 0;  // of the bitstream
    size_t num_tokens = 0, num_heads = 0, head_dim = 0;
    bool decodable = false;  // the codebook fits the decode table (always, for chunks made here)
    bool indexed = false;    // made here: with the index the one-launch decoder reads
    size_t symbols() const { return num_heads * num_tokens * head_dim; }
    kv_layout layout() const { return kv_layout(num_heads, symbols(), indexed); }
    const float *scales_dev() const { return reinterpret_cast<const float *>(dev); }
    const uint16_t *lut_dev() const { return reinterpret_cast<const uint16_t *>(dev + layout().o_lut); }
    const uint8_t *bits_dev() const { return reinterpret_cast<const uint8_t *>(dev + layout().o_bits); }
};

// HuffmanKVCache  src/huffman.rs:484-497
struct pg_huffman_kv_cache {
    pg_kv_cache *hot = nullptr;
    std::vector<pg_huffman_kv_chunk *> k_chunks, v_chunks;
    size_t compressed_len = 0, compress_threshold = 0, chunk_size = 0;
    size_t expect[2] = {0, 0};  // bytes that a chunk's stream is expected to take, by side (compress_batch)
    // The chunks' addresses on the device, key and value side in turn (written by the encoder).  An outgrown table
    // may still be read by work in flight and stays until the cache goes.
    pg_dev_block table_mem;
    char **table = nullptr;
    size_t table_cap = 0;
    std::vector<pg_dev_block> old_tables;
    // Before ctx's stream uses any of it.  `user` = the pool of the context that used the cache last: what its stream has made
    // since is its own, everything else was marked then, so only another context has anything to mark.  (An address that
    // a later context's pool takes over belongs to no block any more: the same holds.  Reads may come from several threads.)
    std::atomic<const pg_dev_pool *> user{nullptr};
    void touch(const pg_ctx *ctx) {
        hot->touch(ctx);
        if (user.load() == ctx->pool.get()) return;
        table_mem.touch(ctx);
        for (auto &t : old_tables) t.touch(ctx);
        for (auto *v : {&k_chunks, &v_chunks})
            for (auto *p : *v) p->block->touch(ctx);
        user.store(ctx->pool.get());
    }
    bool foreign() const {
        bool any = hot->k_mem.foreign || hot->v_mem.foreign || table_mem.foreign;
        for (auto &t : old_tables) any = any || t.foreign;
        for (auto *v : {&k_chunks, &v_chunks})
            for (auto *p : *v) any = any || p->block->foreign;
        return any;
    }
};

static pg_status chunk_shape_ok(const char *who, size_t num_tokens, size_t num_heads, size_t head_dim) {
    PG_CHECK_ARG(num_heads < 65536, "%s: %zu heads (at most 65535)", who, num_heads);
    PG_CHECK_ARG(num_tokens < (1ull << 31) && head_dim < (1ull << 31) &&
                     (num_tokens == 0 || head_dim == 0 || num_heads == 0 ||
                      num_tokens * head_dim < (1ull << 31) / (num_heads ? num_heads : 1)),
                 "%s: %zu heads x %zu tokens x %zu values is beyond 2^31 symbols", who, num_heads, num_tokens, head_dim);
    return PG_OK;
}

// Allocates the device memory of a chunk without an index, zeroes it (stream ordered) and puts scales and the decode
// table of c->codebook in place.
static pg_status chunk_alloc(pg_ctx *ctx, pg_huffman_kv_chunk *c, size_t bytes) {
    c->bytes = bytes;
    c->on_host = true;
    const kv_layout lay = c->layout();
    c->block = std::make_shared<pg_dev_block>();
    PG_TRY(c->block->alloc(ctx, lay.size(bytes)));
    c->dev = static_cast<char *>(c->block->p);
    PG_HIP(hipMemsetAsync(c->dev, 0, lay.size(bytes), ctx->stream));
    std::vector<uint16_t> lut(KV_LUT);
    c->decodable = pg_huffman_host_lut(c->codebook, lut.data()) == PG_OK;  // else: reported when the chunk is decoded
    if (c->num_heads) PG_HIP(hipMemcpyAsync(c->dev, c->scales.data(), c->num_heads * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    if (c->decodable)
        PG_HIP(hipMemcpyAsync(c->dev + lay.o_lut, lut.data(), lut.size() * sizeof(uint16_t), hipMemcpyHostToDevice, ctx->stream));
    PG_HIP(hipStreamSynchronize(ctx->stream));  // lut is a local
    return PG_OK;
}

// Waits until the `n` words at `words` (pinned, zeroed before the launch that stores them) are there.  The kernel that
// stores them is usually a few tens of microseconds away and waking from a stream wait costs ten: so this looks for a
// while first.
static pg_status wait_for_words(pg_ctx *ctx, const uint64_t *words, size_t n) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    size_t have = 0;
    for (;;) {
        while (have < n && __atomic_load_n(words + have, __ATOMIC_ACQUIRE)) ++have;
        if (have == n) return PG_OK;
        if (std::chrono::steady_clock::now() > until) break;
    }
    PG_HIP(hipStreamSynchronize(ctx->stream));
    for (; have < n; ++have)
        if (!__atomic_load_n(words + have, __ATOMIC_ACQUIRE)) return pg_fail(PG_EDEVICE, "huffman kv: the table kernel left no size");
    return PG_OK;
}

// The window's move to the front, for compress_batch to fold into its last launch where it can (done = true once it is certain).
struct kv_shift {
    float *hot[2];
    size_t stride, from, rest;
    bool done = false;
};

// New rows behind the window, for compress_batch's first launch to write (written = true).
struct kv_rows {
    kv_incoming in;
    bool written = false;
};

// compress_chunk of `count` chunks of one shape (none of them empty), chunk c being number c / sides of side c % sides:
// head h of it starts at data[side] + number * chunk_step + h * head_stride.  Their addresses go to table_dev[0 ..) if given.
// `rows` (if given) are still to be written to the window behind data[]: the first launch does.
// `expect` (if given): room for streams of that many bytes, by side, is made and the encoder launched before their sizes are known, so
// that it follows the table at once instead of 8 us later.  Where a stream is longer, or the rooms take more than 1 / 32 over what
// the chunks need, that launch does nothing (GUESSED), and the batch is encoded into exactly what it needs once the sizes
// are known, as where there was no memory for the guess.  0 = wait for the sizes first.  Set to what a batch like the last
// one needs and 1 / 64 more: of normally distributed rows, in appends of 1 to 4 chunks of 16384 to 262144 values, one batch in
// 16 does not suit its guess.
// Whatever fails -- memory on the device or on the host -- fails before the window moves: the cache is then as it was.
static pg_status compress_batch(pg_ctx *ctx, const float *const *data, size_t sides, size_t count, size_t chunk_step, size_t head_stride,
                                size_t num_tokens, size_t num_heads, size_t head_dim, char **table_dev, kv_shift *shift, kv_rows *rows, size_t *expect,
                                std::vector<std::unique_ptr<pg_huffman_kv_chunk>> &out) {
    const size_t head_elems = num_tokens * head_dim, total = num_heads * head_elems;
    const size_t nwg = (total + ENC_PER_WG - 1) / ENC_PER_WG;
    const size_t most = std::max<size_t>(1, std::min<size_t>(KV_BATCH_SYMBOLS / total, KV_BATCH_CHUNKS) / sides) * sides;
    out.reserve(count);
    for (size_t first = 0; first < count; first += most) {
        kv_batch b;
        const size_t n = std::min(most, count - first);
        bool vec = head_elems % 4 == 0 && head_stride % 4 == 0 && chunk_step % 4 == 0;
        for (size_t s = 0; s < 2; ++s) {
            b.data[s] = data[s < sides ? s : 0] + first / sides * chunk_step;
            vec = vec && (uintptr_t)b.data[s] % 16 == 0;
        }
        b.chunk_step = chunk_step; b.head_stride = head_stride;
        b.sides = (unsigned)sides; b.count = (unsigned)n; b.heads = (unsigned)num_heads; b.head_elems = (unsigned)head_elems;
        b.total = (unsigned)total; b.nwg = (unsigned)nwg;
        b.splits = (unsigned)std::min<size_t>(std::max<size_t>((head_elems + ENC_PER_WG - 1) / ENC_PER_WG, 1), KV_MAX_SPLITS);
        b.q_stride = pg_round_up(total, 16);
        size_t off = 0;
        auto take = [&](size_t bytes) { const size_t at = off; off += pg_round_up(bytes, 256); return at; };
        const size_t o_amax = take(n * num_heads * b.splits * 4), o_scales = take(n * num_heads * 4), o_q = take(n * b.q_stride);
        const size_t o_hist = take(n * nwg * NUM_SYMBOLS * 2), o_bit = take(n * (nwg + 1) * 8), o_codes = take(n * NUM_SYMBOLS * 4);
        const size_t o_levels = take(n * KV_LEVELS * 4);
        void *ws = nullptr, *pin = nullptr;
        PG_TRY(pg_workspace(ctx, off, &ws));
        char *base = static_cast<char *>(ws);
        b.amax = reinterpret_cast<float *>(base + o_amax);
        b.scales = reinterpret_cast<float *>(base + o_scales);
        b.q = reinterpret_cast<int8_t *>(base + o_q);
        b.hist = reinterpret_cast<uint16_t *>(base + o_hist);
        b.wg_bit = reinterpret_cast<unsigned long long *>(base + o_bit);
        b.codes = reinterpret_cast<unsigned *>(base + o_codes);
        b.levels = reinterpret_cast<unsigned *>(base + o_levels);
        kv_incoming in = {{b.data[0], b.data[1]}, {nullptr, nullptr}, 0, 0, ~(size_t)0, 0, 0};
        bool vec_in = vec;
        if (rows && first == 0) {
            in = rows->in;
            vec_in = vec && in.from % 4 == 0 && in.elems % 4 == 0 && in.src_stride % 4 == 0 && in.dst_stride % 4 == 0;
            for (size_t s = 0; s < 2; ++s) vec_in = vec_in && ((uintptr_t)in.src[s] | (uintptr_t)in.dst[s]) % 16 == 0;
        }
        if (head_elems <= WHOLE_HEAD && n * nwg <= 2 * (size_t)ctx->num_cu && n * nwg * head_elems <= WHOLE_READS) {
            in.parts = (unsigned)((in.elems + 4 * ENC_PER_WG - 1) / (4 * ENC_PER_WG));
            PG_TRY(pg_launch(ctx, "huffman_kv_quant", vec_in ? kv_whole_kernel<float4> : kv_whole_kernel<float>,
                             dim3((b.nwg + 7) / 8 * 8 * b.count + (unsigned)(sides * num_heads) * in.parts), dim3(WHOLE_WG), 0, b, in));
        } else {
            in.parts = (unsigned)std::min<size_t>((in.elems + b.splits * ENC_PER_WG - 1) / (b.splits * ENC_PER_WG), KV_MAX_SPLITS);
            PG_TRY(pg_launch(ctx, "huffman_kv_absmax", vec_in ? kv_absmax_kernel<float4> : kv_absmax_kernel<float>,
                             dim3(b.splits * b.heads, b.count + (unsigned)sides * in.parts), dim3(KV_WG), 0, b, in));
            PG_TRY(pg_launch(ctx, "huffman_kv_quant", kv_quant_hist_kernel, dim3(b.nwg, b.count), dim3(KV_WG), 0, b, (int)vec));
        }
        if (rows) rows->written = true;
        // (while the device is at it)
        PG_TRY(pg_pinned(ctx, n * sizeof(uint64_t), &pin));
        std::vector<std::unique_ptr<pg_huffman_kv_chunk>> made(n);
        for (auto &ch : made) {
            ch.reset(new (std::nothrow) pg_huffman_kv_chunk());
            if (!ch) return pg_fail(PG_ENOMEM, "host allocation failed");
        }
        auto block = std::make_shared<pg_dev_block>();
        std::vector<char *> at(n);
        bool moves = false;  // the encoder's launch moves the window
        uint64_t *sizes = static_cast<uint64_t *>(pin);
        std::fill(sizes, sizes + n, (uint64_t)0);
        PG_TRY(pg_launch(ctx, "huffman_kv_table", b.total < (1u << 23) ? kv_table_kernel<unsigned> : kv_table_kernel<unsigned long long>, dim3(b.count), dim3(1024), 0, b, (unsigned long long *)sizes));
        const kv_layout lay(num_heads, total, true);
        // the encoder and the window's move: chunk c has room for bytes_of(c) of stream
        unsigned least = 0;
        auto encode = [&](auto bytes_of, bool guess) -> pg_status {
            size_t bytes = 0;
            for (size_t c = 0; c < n; ++c) bytes += lay.size(bytes_of(c));
            PG_TRY(block->alloc(ctx, bytes));
            least = (unsigned)((bytes / 256 * 32 + 32) / 33);
            bytes = 0;
            for (size_t c = 0; c < n; ++c) {
                at[c] = static_cast<char *>(block->p) + bytes;
                bytes += lay.size(bytes_of(c));
            }
            moves = false;
            for (size_t c0 = 0; c0 < n; c0 += KV_PLACES) {
                kv_places places;
                places.first = (unsigned)c0;
                places.room[0] = expect ? expect[0] : 0;
                places.room[1] = expect ? expect[1] : 0;
                places.least = least;
                const size_t here = std::min<size_t>(KV_PLACES, n - c0);
                std::copy(at.begin() + c0, at.begin() + c0 + here, places.at);
                size_t rows = 0;
                if (shift && first + c0 + here == count && here + sides * num_heads <= 65535) {
                    places.hot[0] = shift->hot[0];
                    places.hot[1] = shift->hot[1];
                    places.hot_stride = shift->stride;
                    places.from = shift->from;
                    places.rest = shift->rest;
                    places.vec = shift->from % 4 == 0 && shift->rest % 4 == 0 && shift->stride % 4 == 0 && ((uintptr_t)shift->hot[0] | (uintptr_t)shift->hot[1]) % 16 == 0;
                    rows = sides * num_heads;
                    moves = true;
                }
                PG_TRY(pg_launch(ctx, "huffman_kv_encode", guess ? kv_encode_kernel<true> : kv_encode_kernel<false>, dim3(b.nwg + 1, (unsigned)(here + rows)),
                                 dim3(KV_WG), 0, b, places, table_dev ? table_dev + first : nullptr));
            }
            return PG_OK;
        };
        const bool guesses = expect && expect[0] && expect[sides - 1];
        pg_status guessed = PG_ENOMEM;
        if (guesses) guessed = encode([&](size_t c) { return expect[c % sides]; }, true);
        PG_TRY(wait_for_words(ctx, sizes, n));  // (also after a failure: the table kernel writes them until then)
        if (guessed != PG_ENOMEM) PG_TRY(guessed);
        auto stream_bytes = [&](size_t c) { return (size_t)kv_stream_bytes(sizes[c] - 1); };
        size_t longest[2] = {0, 0}, need = 0;
        for (size_t c = 0; c < n; ++c) {
            longest[c % sides] = std::max(longest[c % sides], stream_bytes(c));
            need += lay.size(stream_bytes(c)) / 256;
        }
        bool suits = guessed == PG_OK && need >= least;
        for (size_t s = 0; s < sides; ++s) suits = suits && longest[s] <= expect[s];
        if (!suits) PG_TRY(encode(stream_bytes, false));
        if (shift && moves) shift->done = true;
        for (size_t s = 0; expect && s < sides; ++s) expect[s] = longest[s] + longest[s] / 64;
        for (size_t c = 0; c < n; ++c) {
            pg_huffman_kv_chunk *ch = made[c].get();
            ch->num_tokens = num_tokens; ch->num_heads = num_heads; ch->head_dim = head_dim;
            ch->block = block;
            ch->dev = at[c];
            ch->bytes = stream_bytes(c);
            ch->decodable = ch->indexed = true;
            out.push_back(std::move(made[c]));
        }
    }
    return PG_OK;
}

// compress_chunk on device data: head h's num_tokens * head_dim values start at data + h * head_stride.
static pg_status compress_dev(pg_ctx *ctx, const float *data, size_t head_stride, size_t num_tokens, size_t num_heads,
                              size_t head_dim, pg_huffman_kv_chunk **out) {
    *out = nullptr;
    PG_TRY(chunk_shape_ok("huffman kv compress_chunk", num_tokens, num_heads, head_dim));
    if (num_tokens * num_heads * head_dim == 0) {  // an empty table, an empty stream; absmax == 0.0 -> scale 1.0
        std::unique_ptr<pg_huffman_kv_chunk> c(new (std::nothrow) pg_huffman_kv_chunk());
        if (!c) return pg_fail(PG_ENOMEM, "host allocation failed");
        c->num_tokens = num_tokens; c->num_heads = num_heads; c->head_dim = head_dim;
        std::fill(c->codebook, c->codebook + NUM_SYMBOLS, (uint8_t)0);
        c->scales.assign(num_heads, 1.0f);
        PG_TRY(chunk_alloc(ctx, c.get(), 0));
        *out = c.release();
        return PG_OK;
    }
    std::vector<std::unique_ptr<pg_huffman_kv_chunk>> made;
    PG_TRY(compress_batch(ctx, &data, 1, 1, 0, head_stride, num_tokens, num_heads, head_dim, nullptr, nullptr, nullptr, nullptr, made));
    *out = made[0].release();
    return PG_OK;
}

// The one-launch decoder over chunks of one shape with an index (args.table or args.single), and the window's rows.
static pg_status launch_decode(pg_ctx *ctx, kv_decode_args a) {
    bool vec = a.head_elems % 4 == 0 && a.out_stride % 4 == 0 && a.chunk_step % 4 == 0 && a.hot_elems % 4 == 0 && a.hot_stride % 4 == 0 && a.hot_at % 4 == 0;
    for (unsigned s = 0; s < a.sides; ++s) vec = vec && (uintptr_t)a.out[s] % 16 == 0 && (uintptr_t)a.hot[s] % 16 == 0;
    a.wgs = (a.total + DEC_PER_WG - 1) / DEC_PER_WG;
    a.hot_wgs = (a.hot_elems + DEC_PER_WG - 1) / DEC_PER_WG;
    const size_t grid = (size_t)a.count * a.wgs + (size_t)a.hot_wgs * a.sides * a.heads;
    if (grid == 0) return PG_OK;
    return pg_launch(ctx, "huffman_kv_decode", vec ? kv_decode_kernel<true> : kv_decode_kernel<false>, dim3((unsigned)grid), dim3(KV_WG), 0, a);
}

// decompress_chunk of chunks made from stored parts, several in one pass: chunk i's head h goes to out[i] + h * out_stride[i].
static pg_status decompress_many(pg_ctx *ctx, const pg_huffman_kv_chunk *const *chunks, float *const *out, const size_t *out_stride,
                                 size_t count) {
    std::vector<pg_huffman_dev_stream> streams;
    std::vector<dequant_item> items;
    size_t total = 0, max_head_elems = 0, heads = 0;
    for (size_t i = 0; i < count; ++i) {
        const pg_huffman_kv_chunk *c = chunks[i];
        if (c->symbols() == 0) continue;
        if (!c->decodable) {  // sets the message
            std::vector<uint16_t> lut(pg_huffman_lut_entries());
            PG_TRY(pg_huffman_host_lut(c->codebook, lut.data()));
        }
        PG_CHECK_ARG(heads == 0 || heads == c->num_heads, "huffman kv: chunks of %zu and %zu heads in one pass", heads, c->num_heads);
        heads = c->num_heads;
        streams.push_back({c->bits_dev(), c->bytes, c->symbols(), c->lut_dev(), total});
        items.push_back({c->scales_dev(), out[i], total, c->num_tokens * c->head_dim, out_stride[i]});
        max_head_elems = std::max(max_head_elems, c->num_tokens * c->head_dim);
        total += pg_round_up(c->symbols(), 16);
    }
    if (items.empty()) return PG_OK;
    PG_CHECK_ARG(items.size() < 65536, "huffman kv: %zu chunks in one pass", items.size());
    const size_t o_items = pg_round_up(total, 256);
    pg_tmp buf;
    PG_TRY(buf.alloc(ctx, o_items + items.size() * sizeof(dequant_item)));
    PG_HIP(hipMemcpyAsync(buf.as<char>() + o_items, items.data(), items.size() * sizeof(dequant_item), hipMemcpyHostToDevice, ctx->stream));
    PG_TRY(pg_huffman_decode_device_streams(ctx, streams.data(), streams.size(), buf.as<int8_t>()));
    PG_TRY(pg_launch(ctx, "huffman_kv_dequant", kv_dequant_kernel, dim3(splits_for(max_head_elems), (unsigned)heads, (unsigned)items.size()),
                     dim3(KV_WG), 0, (const int8_t *)buf.as<int8_t>(), reinterpret_cast<const dequant_item *>(buf.as<char>() + o_items)));
    PG_HIP(hipStreamSynchronize(ctx->stream));  // buf is freed on return
    return PG_OK;
}

static pg_status decompress_dev(pg_ctx *ctx, const pg_huffman_kv_chunk *c, float *out, size_t out_stride) {
    c->block->touch(ctx);
    if (!c->indexed) return decompress_many(ctx, &c, &out, &out_stride, 1);
    kv_decode_args a = {};
    a.single = c->dev;
    a.out[0] = out;
    a.out_stride = out_stride;
    a.sides = a.count = 1;
    a.heads = (unsigned)c->num_heads; a.head_elems = (unsigned)(c->num_tokens * c->head_dim); a.total = (unsigned)c->symbols();
    return launch_decode(ctx, a);
}

PG_API pg_status pg_huffman_kv_compress_chunk_dev(pg_ctx *ctx, const float *data_dev, size_t head_stride, size_t num_tokens,
                                                  size_t num_heads, size_t head_dim, pg_huffman_kv_chunk **out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(out != nullptr, "pg_huffman_kv_compress_chunk_dev: out is null");
    *out = nullptr;
    PG_CHECK_ARG(data_dev || num_tokens * num_heads * head_dim == 0, "pg_huffman_kv_compress_chunk_dev: null data");
    PG_CHECK_ARG(head_stride >= num_tokens * head_dim, "pg_huffman_kv_compress_chunk_dev: head_stride %zu < %zu values per head",
                 head_stride, num_tokens * head_dim);
    return compress_dev(ctx, data_dev, head_stride, num_tokens, num_heads, head_dim, out);
}

PG_API pg_status pg_huffman_kv_compress_chunk(pg_ctx *ctx, const float *data, size_t num_tokens, size_t num_heads,
                                              size_t head_dim, pg_huffman_kv_chunk **out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(out != nullptr, "pg_huffman_kv_compress_chunk: out is null");
    *out = nullptr;
    PG_TRY(chunk_shape_ok("pg_huffman_kv_compress_chunk", num_tokens, num_heads, head_dim));
    const size_t total = num_tokens * num_heads * head_dim;
    PG_CHECK_ARG(data || total == 0, "pg_huffman_kv_compress_chunk: null data");
    pg_tmp d;
    PG_TRY(d.alloc(ctx, total * sizeof(float)));
    if (total) PG_HIP(hipMemcpyAsync(d.p, data, total * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    PG_TRY(compress_dev(ctx, d.as<float>(), num_tokens * head_dim, num_tokens, num_heads, head_dim, out));
    const hipError_t e = hipStreamSynchronize(ctx->stream);  // d is freed on return
    if (e == hipSuccess) return PG_OK;
    delete *out;
    *out = nullptr;
    return pg_fail(PG_EDEVICE, "huffman kv compress_chunk: %s", hipGetErrorString(e));
}

PG_API pg_status pg_huffman_kv_chunk_from_parts(pg_ctx *ctx, const uint8_t *bitstream, size_t bytes, const float *scales,
                                                const uint8_t *codebook, size_t num_tokens, size_t num_heads, size_t head_dim,
                                                pg_huffman_kv_chunk **out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(out != nullptr, "pg_huffman_kv_chunk_from_parts: out is null");
    *out = nullptr;
    PG_TRY(chunk_shape_ok("pg_huffman_kv_chunk_from_parts", num_tokens, num_heads, head_dim));
    PG_CHECK_ARG(codebook && (scales || num_heads == 0) && (bitstream || bytes == 0), "pg_huffman_kv_chunk_from_parts: null pointer");
    std::unique_ptr<pg_huffman_kv_chunk> c(new (std::nothrow) pg_huffman_kv_chunk());
    if (!c) return pg_fail(PG_ENOMEM, "host allocation failed");
    c->num_tokens = num_tokens; c->num_heads = num_heads; c->head_dim = head_dim;
    std::copy(codebook, codebook + NUM_SYMBOLS, c->codebook);
    c->scales.assign(scales, scales + num_heads);
    PG_TRY(chunk_alloc(ctx, c.get(), bytes));
    if (bytes) PG_HIP(hipMemcpyAsync(c->dev + c->layout().o_bits, bitstream, bytes, hipMemcpyHostToDevice, ctx->stream));
    PG_HIP(hipStreamSynchronize(ctx->stream));
    *out = c.release();
    return PG_OK;
}

PG_API void pg_huffman_kv_chunk_free(pg_ctx *ctx, pg_huffman_kv_chunk *c) {
    if (!c) return;
    if (ctx) {
        (void)pg_use(ctx);
        if (c->block) c->block->touch(ctx);
        if (!c->block || c->block->foreign) (void)hipStreamSynchronize(ctx->stream);
    }
    delete c;
}

PG_API pg_status pg_huffman_kv_chunk_info(const pg_huffman_kv_chunk *c, size_t *num_tokens, size_t *num_heads, size_t *head_dim,
                                          size_t *bitstream_bytes) {
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_chunk_info: null chunk");
    if (num_tokens) *num_tokens = c->num_tokens;
    if (num_heads) *num_heads = c->num_heads;
    if (head_dim) *head_dim = c->head_dim;
    if (bitstream_bytes) *bitstream_bytes = c->bytes;
    return PG_OK;
}

PG_API pg_status pg_huffman_kv_chunk_parts(pg_ctx *ctx, const pg_huffman_kv_chunk *c, uint8_t *bitstream, float *scales,
                                           uint8_t *codebook) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_chunk_parts: null chunk");
    c->block->touch(ctx);
    if ((codebook || scales) && !c->on_host) {
        c->scales.resize(c->num_heads);
        PG_HIP(hipMemcpyAsync(c->codebook, c->dev + c->layout().o_book, NUM_SYMBOLS, hipMemcpyDeviceToHost, ctx->stream));
        PG_HIP(hipMemcpyAsync(c->scales.data(), c->dev, c->num_heads * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
        PG_HIP(hipStreamSynchronize(ctx->stream));
        c->on_host = true;
    }
    if (codebook) std::copy(c->codebook, c->codebook + NUM_SYMBOLS, codebook);
    if (scales) std::copy(c->scales.begin(), c->scales.end(), scales);
    if (bitstream && c->bytes) {
        PG_HIP(hipMemcpyAsync(bitstream, c->bits_dev(), c->bytes, hipMemcpyDeviceToHost, ctx->stream));
        PG_HIP(hipStreamSynchronize(ctx->stream));
    }
    return PG_OK;
}

PG_API pg_status pg_huffman_kv_decompress_chunk_dev(pg_ctx *ctx, const pg_huffman_kv_chunk *c, float *out_dev, size_t head_stride) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_decompress_chunk_dev: null chunk");
    PG_CHECK_ARG(out_dev || c->symbols() == 0, "pg_huffman_kv_decompress_chunk_dev: null output");
    PG_CHECK_ARG(head_stride >= c->num_tokens * c->head_dim, "pg_huffman_kv_decompress_chunk_dev: head_stride %zu < %zu values per head",
                 head_stride, c->num_tokens * c->head_dim);
    return decompress_dev(ctx, c, out_dev, head_stride);
}

PG_API pg_status pg_huffman_kv_decompress_chunk(pg_ctx *ctx, const pg_huffman_kv_chunk *c, float *out) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_decompress_chunk: null chunk");
    const size_t total = c->symbols();
    if (total == 0) return PG_OK;
    PG_CHECK_ARG(out != nullptr, "pg_huffman_kv_decompress_chunk: null output");
    pg_tmp d;
    PG_TRY(d.alloc(ctx, total * sizeof(float)));
    PG_TRY(decompress_dev(ctx, c, d.as<float>(), c->num_tokens * c->head_dim));
    PG_HIP(hipMemcpyAsync(out, d.p, total * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    PG_HIP(hipStreamSynchronize(ctx->stream));
    return PG_OK;
}

// ---- the cache ---------------------------------------------------------------------------

PG_API pg_status pg_huffman_kv_cache_create(pg_ctx *ctx, size_t num_kv_heads, size_t head_dim, size_t compress_threshold,
                                            size_t chunk_size, pg_huffman_kv_cache **out) {
    PG_CHECK_ARG(out != nullptr, "pg_huffman_kv_cache_create: out is null");
    *out = nullptr;
    // with chunk_size 0 the reference's append loops forever once the threshold is reached (src/huffman.rs:545-556)
    PG_CHECK_ARG(chunk_size > 0, "pg_huffman_kv_cache_create: chunk_size is 0");
    pg_huffman_kv_cache *c = new (std::nothrow) pg_huffman_kv_cache();
    if (!c) return pg_fail(PG_ENOMEM, "host allocation failed");
    const pg_status st = pg_kv_cache_create(ctx, num_kv_heads, head_dim, &c->hot);
    if (st != PG_OK) {
        delete c;
        return st;
    }
    c->compress_threshold = std::max(compress_threshold, chunk_size);  // src/huffman.rs:535
    c->chunk_size = chunk_size;
    *out = c;
    return PG_OK;
}

PG_API void pg_huffman_kv_cache_free(pg_ctx *ctx, pg_huffman_kv_cache *c) {
    if (!c) return;
    if (ctx) {
        (void)pg_use(ctx);
        c->touch(ctx);
        if (c->foreign()) (void)hipStreamSynchronize(ctx->stream);
    }
    pg_kv_cache_free(ctx, c->hot);
    for (auto *p : c->k_chunks) delete p;
    for (auto *p : c->v_chunks) delete p;
    delete c;
}

PG_API size_t pg_huffman_kv_cache_len(const pg_huffman_kv_cache *c) { return c ? c->compressed_len + c->hot->len : 0; }
PG_API size_t pg_huffman_kv_cache_compressed_len(const pg_huffman_kv_cache *c) { return c ? c->compressed_len : 0; }
PG_API size_t pg_huffman_kv_cache_num_chunks(const pg_huffman_kv_cache *c) { return c ? c->k_chunks.size() : 0; }
PG_API size_t pg_huffman_kv_cache_compress_threshold(const pg_huffman_kv_cache *c) { return c ? c->compress_threshold : 0; }
PG_API pg_status pg_huffman_kv_cache_hot(pg_huffman_kv_cache *c, pg_kv_cache **out) {
    PG_CHECK_ARG(c && out, "pg_huffman_kv_cache_hot: null pointer");
    *out = c->hot;
    return PG_OK;
}

PG_API pg_status pg_huffman_kv_cache_chunk(const pg_huffman_kv_cache *c, int value_side, size_t index,
                                           const pg_huffman_kv_chunk **out) {
    PG_CHECK_ARG(c && out, "pg_huffman_kv_cache_chunk: null pointer");
    const auto &v = value_side ? c->v_chunks : c->k_chunks;
    PG_CHECK_ARG(index < v.size(), "pg_huffman_kv_cache_chunk: chunk %zu of %zu", index, v.size());
    *out = v[index];
    return PG_OK;
}

// Room for `chunks` addresses in the cache's table.
static pg_status table_reserve(pg_ctx *ctx, pg_huffman_kv_cache *c, size_t chunks) {
    if (chunks <= c->table_cap) return PG_OK;
    const size_t cap = std::max<size_t>(std::max<size_t>(chunks, 2 * c->table_cap), 64);
    pg_dev_block grown;
    PG_TRY(grown.alloc(ctx, cap * sizeof(char *)));
    if (c->table) {
        PG_HIP(hipMemcpyAsync(grown.p, c->table, c->table_cap * sizeof(char *), hipMemcpyDeviceToDevice, ctx->stream));
        c->old_tables.push_back(std::move(c->table_mem));
    }
    c->table_mem = std::move(grown);
    c->table = static_cast<char **>(c->table_mem.p);
    c->table_cap = cap;
    return PG_OK;
}

// The reference compresses the oldest chunk_size tokens and shifts the rest to the front, once per
// chunk; here every chunk that an append cuts, of both sides, is one batch and the window is shifted once.
// `rows`: the window's last ones, still to be written.
static pg_status compress_hot(pg_ctx *ctx, pg_huffman_kv_cache *c, kv_rows *rows) {
    pg_kv_cache *hot = c->hot;
    if (hot->len < c->compress_threshold) return PG_OK;
    const size_t hd = hot->head_dim, stride = hot->capacity * hd, heads = hot->num_kv_heads, tokens = c->chunk_size;
    const size_t chunks = (hot->len - c->compress_threshold) / tokens + 1;  // compress_threshold >= chunk_size: every chunk is whole
    PG_TRY(chunk_shape_ok("huffman kv append", tokens, heads, hd));
    PG_TRY(table_reserve(ctx, c, c->k_chunks.size() * 2 + 2 * chunks));
    for (auto *v : {&c->k_chunks, &c->v_chunks})
        if (v->size() + chunks > v->capacity()) v->reserve(std::max(v->size() + chunks, 2 * v->capacity()));
    const float *data[2] = {hot->k, hot->v};
    std::vector<std::unique_ptr<pg_huffman_kv_chunk>> made;
    kv_shift shift{{hot->k, hot->v}, stride, chunks * tokens * hd, (hot->len - chunks * tokens) * hd};
    const pg_status st = compress_batch(ctx, data, 2, 2 * chunks, tokens * hd, stride, tokens, heads, hd, c->table + c->k_chunks.size() * 2, &shift, rows, c->expect, made);
    size_t done = 0;
    for (size_t i = 0; i + 1 < made.size(); i += 2) {
        c->k_chunks.push_back(made[i].release());
        c->v_chunks.push_back(made[i + 1].release());
        done += tokens;
    }
    if (done == 0) return st;
    c->compressed_len += done;
    const size_t rest = hot->len - done;
    // Where the encoder has not done it: the rest moves to the front in slices no longer than the distance it moves, oldest first on
    // the one stream, so that no copy reads what it writes; nothing is allocated and nothing waited for.
    for (size_t at = shift.done ? rest : 0; at < rest; at += done)
        PG_TRY(pg_launch_kv_rows(ctx, hot->k + at * hd, hot->v + at * hd, stride, hot->k + (done + at) * hd, hot->v + (done + at) * hd, stride,
                                 std::min(done, rest - at) * hd, heads));
    hot->len = rest;
    return st;
}

// Whether an append of seq_len tokens cuts a chunk: the host reads its size, which a capturing stream refuses -- ahead of the
// append to the window, so that nothing has changed then.
static pg_status append_ok(pg_ctx *ctx, const pg_huffman_kv_cache *c, size_t seq_len) {
    return c->hot->len + seq_len < c->compress_threshold ? PG_OK : pg_refuse_capture(ctx, "pg_huffman_kv_cache_append: a chunk");
}

PG_API pg_status pg_huffman_kv_cache_append_dev(pg_ctx *ctx, pg_huffman_kv_cache *c, const float *new_k_dev,
                                                const float *new_v_dev, size_t seq_len) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_cache_append: null cache");
    PG_TRY(append_ok(ctx, c, seq_len));
    c->touch(ctx);
    pg_kv_cache *hot = c->hot;
    const size_t hd = hot->head_dim, had = hot->len;
    if (seq_len == 0 || had + seq_len < c->compress_threshold) {
        PG_TRY(pg_kv_cache_append_dev(ctx, hot, new_k_dev, new_v_dev, seq_len));
        return compress_hot(ctx, c, nullptr);
    }
    PG_TRY(pg_kv_cache_append_room(ctx, hot, new_k_dev, new_v_dev, seq_len));
    const size_t from = had * hd, stride = hot->capacity * hd;
    float *k = hot->k + from, *v = hot->v + from;
    kv_rows rows{{{new_k_dev, new_v_dev}, {k, v}, seq_len * hd, stride, from, seq_len * hd, 0}};
    hot->len += seq_len;
    const pg_status st = compress_hot(ctx, c, &rows);
    if (!rows.written) PG_TRY(pg_launch_kv_rows(ctx, k, v, stride, new_k_dev, new_v_dev, seq_len * hd, seq_len * hd, hot->num_kv_heads));
    return st;
}

PG_API pg_status pg_huffman_kv_cache_append(pg_ctx *ctx, pg_huffman_kv_cache *c, const float *new_k, const float *new_v,
                                            size_t seq_len) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_cache_append: null cache");
    PG_TRY(append_ok(ctx, c, seq_len));
    c->touch(ctx);
    PG_TRY(pg_kv_cache_append(ctx, c->hot, new_k, new_v, seq_len));
    return compress_hot(ctx, c, nullptr);
}

PG_API pg_status pg_huffman_kv_cache_get_kv_dev(pg_ctx *ctx, const pg_huffman_kv_cache *c, float *k_dev, float *v_dev) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_cache_get_kv: null cache");
    const pg_kv_cache *hot = c->hot;
    const size_t total_len = c->compressed_len + hot->len, hd = hot->head_dim, heads = hot->num_kv_heads;
    if (total_len * hd * heads == 0) return PG_OK;
    PG_CHECK_ARG(k_dev && v_dev, "pg_huffman_kv_cache_get_kv: null output");
    const_cast<pg_huffman_kv_cache *>(c)->touch(ctx);
    kv_decode_args a = {};
    a.out[0] = k_dev;
    a.out[1] = v_dev;
    a.out_stride = total_len * hd;
    a.chunk_step = c->chunk_size * hd;
    a.sides = 2;
    a.heads = (unsigned)heads; a.head_elems = (unsigned)(c->chunk_size * hd); a.total = (unsigned)(heads * c->chunk_size * hd);
    // every chunk of both sides in one launch, the window's rows with them (a launch takes up to 2^30 workgroups of 16384 values)
    const size_t chunks = 2 * c->k_chunks.size(), most = std::max<size_t>(1, (1u << 30) / (a.total / DEC_PER_WG + 1)) * 2;
    for (size_t first = 0; first < chunks; first += most) {
        a.table = c->table + first;
        a.count = (unsigned)std::min(most, chunks - first);
        for (int s = 0; s < 2; ++s) a.out[s] = (s ? v_dev : k_dev) + first / 2 * a.chunk_step;
        if (first + most >= chunks && hot->len > 0 && hot->len * hd < (1ull << 31)) {
            a.hot[0] = hot->k;
            a.hot[1] = hot->v;
            a.hot_stride = hot->capacity * hd;
            a.hot_at = c->compressed_len * hd - first / 2 * a.chunk_step;
            a.hot_elems = (unsigned)(hot->len * hd);
        }
        PG_TRY(launch_decode(ctx, a));
    }
    if (hot->len > 0 && a.hot_elems == 0)
        PG_TRY(pg_launch_kv_rows(ctx, k_dev + c->compressed_len * hd, v_dev + c->compressed_len * hd, total_len * hd, hot->k, hot->v,
                                 hot->capacity * hd, hot->len * hd, heads));
    return PG_OK;
}

PG_API pg_status pg_huffman_kv_cache_get_kv(pg_ctx *ctx, const pg_huffman_kv_cache *c, float *k, float *v) {
    PG_TRY(pg_use(ctx));
    PG_CHECK_ARG(c != nullptr, "pg_huffman_kv_cache_get_kv: null cache");
    const size_t n = (c->compressed_len + c->hot->len) * c->hot->head_dim * c->hot->num_kv_heads;
    if (n == 0) return PG_OK;
    PG_CHECK_ARG(k && v, "pg_huffman_kv_cache_get_kv: null output");
    pg_tmp d;
    PG_TRY(d.alloc(ctx, 2 * n * sizeof(float)));
    PG_TRY(pg_huffman_kv_cache_get_kv_dev(ctx, c, d.as<float>(), d.as<float>() + n));
    PG_HIP(hipMemcpyAsync(k, d.p, n * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    PG_HIP(hipMemcpyAsync(v, d.as<float>() + n, n * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    PG_HIP(hipStreamSynchronize(ctx->stream));
    return PG_OK;
}
