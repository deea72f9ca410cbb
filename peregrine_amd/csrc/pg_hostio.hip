// Arrays of the host-pointer entry points, on their way to the device and back.
//
// A caller's array is pageable, so it crosses in two steps: the host's copy to or from pinned memory, and the transfer.
// Left to hipMemcpyAsync a 196 x 768 product with 3072 columns (0.6 MB in, 2.4 MB out) spent 195 us of its 224 there: the
// two steps one after the other, each transfer with the 10 us that a copy engine takes to begin and the stream wait takes
// to end.  Here the transfers are launches -- a wavefront reads and writes pinned memory over PCIe like any other -- that
// follow the products on the stream in 4 us, and the way out is a pipeline: the launch stores a word per 16 KB that has
// arrived and the host copies each piece while the next ones are on the wire.  That product now takes 115 us: 0.6 MB in
// and 2.4 MB out are 54 on the wire, the host's copies 65.
#include <immintrin.h>
#include <chrono>
#include "pg_internal.h"

namespace {

constexpr size_t STAGE_BYTES = 16u << 20;   // the most that a context's pinned block grows to
constexpr size_t PIECE = 16u << 10;         // bytes of one word on the way out
constexpr unsigned PUSH_WGS = 8;            // workgroups on the way out: fewer do not fill the wire, more end together
constexpr size_t IN_PIECE = 1u << 20;       // bytes that the host copies before it launches their transfer

// dst[0 .. n) = src[0 .. n), 16 bytes a lane, eight in flight (the reads are a PCIe round trip away).
__global__ __launch_bounds__(256) void host_pull_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, unsigned n) {
    const unsigned base = blockIdx.x * 2048 + threadIdx.x;
    uint4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (base + i * 256 < n) v[i] = src[base + i * 256];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (base + i * 256 < n) dst[base + i * 256] = v[i];
}

// The way out: workgroup w moves pieces w, w + grid, .. of `bytes` and says so in seen[piece] after each.  Few workgroups
// (PUSH_WGS), so that the pieces arrive one after the other: with one workgroup a piece all of them arrived at the end
// and the host copied afterwards (149 us for the call above; 8 workgroups 115, 4 139).
__global__ __launch_bounds__(256) void host_push_kernel(const char *__restrict__ src, char *__restrict__ dst, size_t bytes, unsigned *seen,
                                                        unsigned epoch) {
    unsigned p = blockIdx.x;
    for (size_t at = (size_t)p * PIECE; at < bytes; at += (size_t)gridDim.x * PIECE, p += gridDim.x) {
        const unsigned n = (unsigned)((bytes - at < PIECE ? bytes - at : PIECE) / 4), n4 = n / 4;
        const unsigned *s = reinterpret_cast<const unsigned *>(src + at);
        unsigned *d = reinterpret_cast<unsigned *>(dst + at);
#pragma unroll 8
        for (unsigned i = threadIdx.x; i < n4; i += 256) reinterpret_cast<uint4 *>(d)[i] = reinterpret_cast<const uint4 *>(s)[i];
        if (threadIdx.x < n - 4 * n4) d[4 * n4 + threadIdx.x] = s[4 * n4 + threadIdx.x];
        __syncthreads();  // every wavefront's stores are acknowledged
        if (threadIdx.x == 0) __hip_atomic_store(seen + p, epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace

// A region of the context's pinned block: regions are taken one behind the other; when they are used up the stream is
// waited for (nothing on it refers to the block then) and they start over.
static pg_status stage_take(pg_ctx *ctx, size_t bytes, void **out) {
    const size_t want = pg_round_up(bytes, 256);
    if (ctx->stage_used + want > ctx->stage_bytes) {
        PG_HIP(hipStreamSynchronize(ctx->stream));
        ctx->stage_used = 0;
        if (want > ctx->stage_bytes) {
            if (ctx->stage) PG_HIP(hipHostFree(ctx->stage));
            ctx->stage = nullptr;
            ctx->stage_bytes = 0;
            size_t grown = 1u << 20;
            while (grown < 2 * want && grown < STAGE_BYTES) grown *= 2;
            if (grown < want) grown = want;
            PG_HIP(hipHostMalloc(&ctx->stage, grown, hipHostMallocDefault));
            ctx->stage_bytes = grown;
        }
    }
    *out = static_cast<char *>(ctx->stage) + ctx->stage_used;
    ctx->stage_used += want;
    return PG_OK;
}

pg_status pg_host_pinned(pg_ctx *ctx, const void *host, size_t bytes, void **pinned) {
    PG_TRY(stage_take(ctx, bytes, pinned));
    memcpy(*pinned, host, bytes);
    return PG_OK;
}

pg_status pg_host_in(pg_ctx *ctx, const void *host, size_t bytes, pg_dev_block &dev) {
    PG_TRY(dev.alloc(ctx, pg_round_up(bytes, 16)));
    for (size_t at = 0; at < bytes; at += IN_PIECE) {
        const size_t n = std::min(IN_PIECE, bytes - at);
        void *pin = nullptr;
        PG_TRY(pg_host_pinned(ctx, static_cast<const char *>(host) + at, n, &pin));
        const unsigned n16 = (unsigned)((n + 15) / 16);  // (regions and blocks are whole sixteens)
        PG_TRY(pg_launch(ctx, "host_pull", host_pull_kernel, dim3((n16 + 2047) / 2048), dim3(256), 0, static_cast<const uint4 *>(pin),
                         reinterpret_cast<uint4 *>(static_cast<char *>(dev.p) + at), n16));
    }
    return PG_OK;
}

// The host's copy out of pinned memory that the device has just written, so that every line comes from memory.  Four
// 256-bit loads ahead of their stores keep more lines on their way than memcpy's string move: 2.4 MB in 55 us against
// 78, close to what the wire takes (43).
__attribute__((target("avx2"))) static void copy_out_avx2(char *to, const char *from, size_t n) {
    size_t i = 0;
    for (; i + 128 <= n; i += 128) {
        const __m256i a = _mm256_loadu_si256(reinterpret_cast<const __m256i *>(from + i));
        const __m256i b = _mm256_loadu_si256(reinterpret_cast<const __m256i *>(from + i + 32));
        const __m256i c = _mm256_loadu_si256(reinterpret_cast<const __m256i *>(from + i + 64));
        const __m256i d = _mm256_loadu_si256(reinterpret_cast<const __m256i *>(from + i + 96));
        _mm256_storeu_si256(reinterpret_cast<__m256i *>(to + i), a);
        _mm256_storeu_si256(reinterpret_cast<__m256i *>(to + i + 32), b);
        _mm256_storeu_si256(reinterpret_cast<__m256i *>(to + i + 64), c);
        _mm256_storeu_si256(reinterpret_cast<__m256i *>(to + i + 96), d);
    }
    memcpy(to + i, from + i, n - i);
}
static void copy_out(char *to, const char *from, size_t n) {
    static const bool avx2 = __builtin_cpu_supports("avx2");
    if (avx2) copy_out_avx2(to, from, n);
    else memcpy(to, from, n);
}

// Looks for *word == epoch for a while (a transfer is tens of microseconds away, and a stream wait costs ten by itself),
// then waits for the stream.
static pg_status await_word(pg_ctx *ctx, const unsigned *word, unsigned epoch) {
    if (__atomic_load_n(word, __ATOMIC_ACQUIRE) == epoch) return PG_OK;
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    for (unsigned i = 1;; ++i) {
        if (__atomic_load_n(word, __ATOMIC_ACQUIRE) == epoch) return PG_OK;
        if (i % 64 == 0 && std::chrono::steady_clock::now() > until) break;
    }
    PG_HIP(hipStreamSynchronize(ctx->stream));
    if (__atomic_load_n(word, __ATOMIC_ACQUIRE) != epoch) return pg_fail(PG_EDEVICE, "a transfer to the host did not complete");
    return PG_OK;
}

pg_status pg_host_out(pg_ctx *ctx, void *host, const void *dev, size_t bytes) {
    if (bytes == 0) return PG_OK;
    // two windows in turn: while the host empties one, the other fills
    const size_t window = std::min(pg_round_up(bytes, PIECE), STAGE_BYTES / 4), windows = (bytes + window - 1) / window;
    struct side { char *data; unsigned *seen; unsigned epoch; } s[2];
    const size_t pieces = window / PIECE;
    for (size_t i = 0; i < std::min<size_t>(windows, 2); ++i) {
        void *p = nullptr;
        // both windows in one region, or the second taking could start the block over while the first is in use
        if (i == 0) PG_TRY(stage_take(ctx, (window + pg_round_up(pieces * 4, 256)) * std::min<size_t>(windows, 2), &p));
        else p = reinterpret_cast<char *>(s[0].seen) + pg_round_up(pieces * 4, 256);
        s[i].data = static_cast<char *>(p);
        s[i].seen = reinterpret_cast<unsigned *>(s[i].data + window);
        s[i].epoch = 0;
    }
    auto launch = [&](size_t w) {
        side &x = s[w & 1];
        const size_t n = std::min(window, bytes - w * window);
        x.epoch = ++ctx->stage_epoch ? ctx->stage_epoch : ++ctx->stage_epoch;
        for (size_t p = 0; p < pieces; ++p) __atomic_store_n(x.seen + p, x.epoch - 1, __ATOMIC_RELAXED);  // whatever lay there
        return pg_launch(ctx, "host_push", host_push_kernel, dim3((unsigned)std::min<size_t>((n + PIECE - 1) / PIECE, PUSH_WGS)), dim3(256), 0,
                         static_cast<const char *>(dev) + w * window, x.data, n, x.seen, x.epoch);
    };
    PG_TRY(launch(0));
    for (size_t w = 0; w < windows; ++w) {
        if (w + 1 < windows) PG_TRY(launch(w + 1));
        const side &x = s[w & 1];
        const size_t n = std::min(window, bytes - w * window);
        char *to = static_cast<char *>(host) + w * window;
        for (size_t at = 0; at < n; at += PIECE) {
            PG_TRY(await_word(ctx, x.seen + at / PIECE, x.epoch));
            copy_out(to + at, x.data + at, std::min(PIECE, n - at));
        }
    }
    return PG_OK;
}
