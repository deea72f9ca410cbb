// Many query rows of grouped-query attention on the f16 matrix cores, every f32 operand as the sum of two halves
// (included by pg_llama.hip behind attn_args).
//
// x * 2^e = hi + lo: hi is x * 2^e rounded to f16, lo the remainder rounded to f16, 22 to 24 significant bits for what is not
// far below the scale.  e brings the largest magnitude of a query row, or of a tile of 32 keys or values, to [2^14, 2^15);
// halves are 2^-39 of that apart: a key or value that is 2^-s of its tile's largest, s > 15, keeps 39 - s bits where f32 keeps 24.
// Probabilities are taken times 2^7 and end at 2^-32 of the row's largest (2^-30 where a tile's values are up to 4 times smaller than the
// sums' unit).  hi hi + hi lo + lo hi leaves out lo lo, below 2^-24 of the product.  The matrix
// instruction sums 16 products a step in f32: a score of 128 terms takes 24 roundings of a running sum where the f32 instruction,
// two products a step, takes 64, which is what either's error comes from (the launcher's rule has the measured ones).  Three of these take
// 3/16 of the f32 instructions' time.
//
// The keys' and values' halves are made once for all rows (kv_halves_kernel), in the order in which the product's lanes
// read them: a workgroup's four wavefronts then share a tile of 32 keys through LDS, filled by direct loads of whole KiB
// and read without bank conflicts.
#pragma once

typedef const void __attribute__((address_space(1))) *gptr_t;
typedef void __attribute__((address_space(3))) *lptr_t;
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// The power of two that brings `amax` (finite) to [2^14, 2^15).  (Denormals stay where 2^126 takes them.)
__device__ __forceinline__ float half_scale(float amax) {
    const int ex = (int)(__float_as_uint(amax) >> 23 & 255u);  // amax in 2^(ex - 127) * [1, 2)
    return amax > 0.0f ? __uint_as_float((unsigned)min(max(127 + 141 - ex, 1), 253) << 23) : 1.0f;
}
__device__ __forceinline__ float finite_mag(float x) {
    const float a = fabsf(x);
    return a < INFINITY ? a : 0.0f;  // (NaN: 0)
}
// The halves of x * s.  A value that is not finite is `lo` alone: it meets only the other side's hi, so a product is
// infinite or NaN where f32's is.
__device__ __forceinline__ void halves(float x, float s, _Float16 &hi, _Float16 &lo) {
    const bool finite = fabsf(x) < INFINITY;
    const float v = finite ? x * s : 0.0f;
    hi = (_Float16)v;
    lo = (_Float16)(finite ? v - (float)hi : x);
}

// Planes of one (kv head, tile of 32 keys): keys, then values, each [hi, lo][HD / 16 steps][64 lanes][8 values]:
//   keys    step i: lane = 32 h + key, values d = 16 i + 8 h ..
//   values  step j * (HD / 32) + dt: lane = 32 h + d % 32 of d-tile dt, keys 16 j + 8 (e / 4) + 4 h + e % 4, e = 0 .. 7
// (the order in which a lane holds its probabilities); the inverse scales (keys, values) behind all planes: [kv heads][tiles][2].
// Keys past `len` are zero.  Grid (tiles, kv heads).
constexpr float HALVES_NO_VALUES = 0x1p-126f;  // the inverse scale of a tile of zeros, the least there is
template <int HD> constexpr int half_unit_bytes() { return 2 * 32 * HD * 2; }
__host__ __device__ constexpr int halves_lds_bytes(int unit) { return 4 * unit > 4 * 32 * 68 * 4 ? 4 * unit : 4 * 32 * 68 * 4; }
__host__ __device__ inline size_t half_scales_offset(int unit, size_t nkv, size_t tiles) { return nkv * tiles * 2 * unit; }
template <int HD>
__global__ __launch_bounds__(256) void kv_halves_kernel(const float *__restrict__ k, const float *__restrict__ v, size_t k_stride, size_t v_stride, int len,
                                                        char *__restrict__ planes) {
    constexpr int PLANE = HD * 64, UB = half_unit_bytes<HD>(), FR = HD * 4 / 256;  // bytes of a half; fragments a thread
    __shared__ float kmax[4], vmax[4];
    const int tile = blockIdx.x, kvh = blockIdx.y, tiles = gridDim.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, l = lane & 31;
    const float *kp = k + (size_t)kvh * k_stride, *vp = v + (size_t)kvh * v_stride;
    char *out = planes + ((size_t)kvh * tiles + tile) * 2 * UB;
    float x[FR][8], y[FR][8], xm = 0.0f, ym = 0.0f;
    const int key = 32 * tile + l;
#pragma unroll
    for (int f = 0; f < FR; ++f) {
        const int step = wave + 4 * f, j = step / (HD / 32), dt = step % (HD / 32);
        float4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
        if (key < len) {
            a = *reinterpret_cast<const float4 *>(kp + (size_t)key * HD + 16 * step + 8 * h);
            b = *reinterpret_cast<const float4 *>(kp + (size_t)key * HD + 16 * step + 8 * h + 4);
        }
        x[f][0] = a.x; x[f][1] = a.y; x[f][2] = a.z; x[f][3] = a.w; x[f][4] = b.x; x[f][5] = b.y; x[f][6] = b.z; x[f][7] = b.w;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int vk = 32 * tile + 16 * j + 8 * (e >> 2) + 4 * h + (e & 3);
            const float t = vp[(size_t)min(vk, len - 1) * HD + 32 * dt + l];
            y[f][e] = vk < len ? t : 0.0f;
        }
    }
#pragma unroll
    for (int f = 0; f < FR; ++f)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            xm = fmaxf(xm, finite_mag(x[f][e]));
            ym = fmaxf(ym, finite_mag(y[f][e]));
        }
    xm = pg_block_max_256(xm, kmax);
    ym = pg_block_max_256(ym, vmax);
    const float ks = half_scale(xm), vs = half_scale(ym);
    if (threadIdx.x == 0)  // (no values: no say in the sums' unit)
        reinterpret_cast<float2 *>(planes + half_scales_offset(UB, gridDim.y, tiles))[(size_t)kvh * tiles + tile] = float2{1.0f / ks, ym > 0.0f ? 1.0f / vs : HALVES_NO_VALUES};
#pragma unroll
    for (int f = 0; f < FR; ++f) {
        v8h kh, kl, vh, vl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            _Float16 a, b;
            halves(x[f][e], ks, a, b);
            kh[e] = a; kl[e] = b;
            halves(y[f][e], vs, a, b);
            vh[e] = a; vl[e] = b;
        }
        char *at = out + ((wave + 4 * f) * 64 + lane) * 16;
        *reinterpret_cast<v8h *>(at) = kh;
        *reinterpret_cast<v8h *>(at + PLANE) = kl;
        *reinterpret_cast<v8h *>(at + UB) = vh;
        *reinterpret_cast<v8h *>(at + UB + PLANE) = vl;
    }
}

// A workgroup takes 128 rows of a kv head (row index = token * group + head in group), 32 to a wavefront, and a run of aa.chunk
// of the key tiles that they see.  Per tile S^T = K Q^T and O^T += V^T P^T with the columns = rows of the query, as in the f32
// kernel above: the tile of S^T that a lane holds is, register by register, the operand of the second product.  The ring
// holds four units (a tile's keys or its values): one consumed, two landed or landing, one asked for when everybody has left its
// place; 64 KiB for HD = 128: two workgroups a CU (by their registers), not in step with each other, so that the softmax of one runs beside the
// matrix instructions of the other.  Rows that one run covers are finished here, others leave (maximum, exp-sum, unnormalised
// row) in aa.part for attn_halves_combine_kernel.
constexpr int HALVES_ROWS = 128, HALVES_CHUNK_MAX = 512, HALVES_RING = 4;  // (CHUNK_MAX: the tiles of a run, by the array of their scales)
constexpr float HALVES_SLACK = 5.0f, LOG2E = 1.44269504f;
__device__ __forceinline__ int halves_tiles(const attn_args &aa, int blk, int nrows) {  // key tiles that a block of rows sees
    const int last_qt = min(blk * HALVES_ROWS + HALVES_ROWS - 1, nrows - 1) / aa.group;
    return ((aa.mask_kind != 0 ? min(aa.len, aa.offset + last_qt + 1) : aa.len) + 31) / 32;
}
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gqa_attention_halves_kernel(const char *__restrict__ planes, int n_blocks, attn_args aa, int nkvh, int tiles_all) {
    constexpr int NDT = HD / 32, NQ = HD / 16, PLANE = HD * 64, UB = half_unit_bytes<HD>(), LPU = UB / 4096, NS = HALVES_RING;
    extern __shared__ __attribute__((aligned(1024))) char half_lds[];  // [NS][UB]; afterwards the wavefronts' tiles of 32 rows x 64 + 4 values
    __shared__ float2 inv[HALVES_CHUNK_MAX];  // the tiles' inverse scales
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, h = lane >> 5;
    const int kvh = blockIdx.x % nkvh, blk = n_blocks - 1 - (int)(blockIdx.x / nkvh) % n_blocks, run = (int)(blockIdx.x / nkvh) / n_blocks;
    const int G = aa.group, nrows = G * aa.seq_q;
    const int tiles = halves_tiles(aa, blk, nrows), t0 = run * aa.chunk, cnt = min(tiles - t0, aa.chunk);
    if (cnt <= 0) return;
    const int last_qt = min(blk * HALVES_ROWS + HALVES_ROWS - 1, nrows - 1) / G;
    const int kend = aa.mask_kind != 0 ? min(aa.len, aa.offset + last_qt + 1) : aa.len;
    const char *src = planes + ((size_t)kvh * tiles_all + t0) * 2 * UB + wave * (UB / 4) + lane * 16;
    char *own = half_lds + wave * (UB / 4);
    auto issue = [&](int u, int slot) {
        if (u < 2 * cnt)
#pragma unroll
            for (int j = 0; j < LPU; ++j)
                __builtin_amdgcn_global_load_lds((gptr_t)(src + (size_t)u * UB + j * 1024), (lptr_t)(own + slot * UB + j * 1024), 16, 0, 0);
    };
    issue(0, 0);
    issue(1, 1);
    static_assert(NS == 4, "the last two places take the queries on their way in");
    const unsigned g_inv = (unsigned)((0x100000000ull + G - 1) / G), g_one = G == 1 ? ~0u : 0u;  // R / G = mulhi(R, g_inv) for R G < 2^32, G > 1
    auto row_of = [&](int r, int &t, int &head) {                     // of the block's head group: token and query head
        const int rc = min(r, nrows - 1);
        t = (int)(__umulhi((unsigned)rc, g_inv) | ((unsigned)rc & g_one));  // (2^32 / 1 is 0 in 32 bits)
        head = kvh * G + rc - t * G;
        return r < nrows;
    };
    const int row0 = blk * HALVES_ROWS + wave * 32, row = row0 + col, qt_min = min(row0, nrows - 1) / G;
    int qt, qh;
    row_of(row, qt, qh);
    v8h q[2][NQ];
    float s_unit;  // of a raw score, times the softmax scale
    {
        // The rows come in through LDS, half of them at a time: whole 128-byte lines an instruction, read back as 16-byte chunks
        // placed by chunk ^ row.  (Loaded as the lanes hold them, 16 bytes of 64 places an instruction: 6 k cycles.)
        constexpr int CH = HD / 8, RI = 64 / CH;  // chunks of a half row, rows an instruction
        char *stage = half_lds + 2 * UB + wave * (UB / 2);
        typedef float v4f __attribute__((ext_vector_type(4)));
        v4f in0[CH / 2], in1[CH / 2], x[NQ][2];
#pragma unroll
        for (int i = 0; i < CH / 2; ++i) {
            int t, head;
            row_of(row0 + RI * i + lane / CH, t, head);
            const float *qp = aa.q + ((size_t)head * aa.seq_q + t) * HD + 4 * (lane % CH);
            in0[i] = *reinterpret_cast<const v4f *>(qp);
            in1[i] = *reinterpret_cast<const v4f *>(qp + HD / 2);
        }
        auto through = [&](const v4f (&in)[CH / 2], auto part) {
#pragma unroll
            for (int i = 0; i < CH / 2; ++i) {
                const int r = RI * i + lane / CH;
                *reinterpret_cast<v4f *>(stage + r * CH * 16 + ((lane ^ r) % CH) * 16) = in[i];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // (its own wavefront's part)
#pragma unroll
            for (int i = 0; i < NQ / 2; ++i)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    x[decltype(part)::value * (NQ / 2) + i][e] = *reinterpret_cast<const v4f *>(stage + col * CH * 16 + ((4 * i + 2 * h + e) ^ (col % CH)) * 16);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        };
        through(in0, std::integral_constant<int, 0>{});
        through(in1, std::integral_constant<int, 1>{});
        float qm = 0.0f;  // the largest magnitude; NaN if there is one
#pragma unroll
        for (int i = 0; i < NQ; ++i)
#pragma unroll
            for (int e = 0; e < 8; e += 2) qm = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(x[i][e / 4][e % 4]), fabsf(x[i][e / 4][e % 4 + 1])), qm);
        qm = __builtin_elementwise_maximum(qm, __shfl_xor(qm, 32));
        const bool odd = __builtin_expect(__any(!(qm < INFINITY)), 0);
        if (odd) {
            qm = 0.0f;
#pragma unroll
            for (int i = 0; i < NQ; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) qm = fmaxf(qm, finite_mag(x[i][e / 4][e % 4]));
            qm = fmaxf(qm, __shfl_xor(qm, 32));
        }
        const float qs = half_scale(qm);
        s_unit = aa.scale / qs;
        if (odd) {
#pragma unroll
            for (int i = 0; i < NQ; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    _Float16 a, b;
                    halves(x[i][e / 4][e % 4], qs, a, b);
                    q[0][i][e] = a; q[1][i][e] = b;
                }
        } else {
#pragma unroll
            for (int i = 0; i < NQ; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const _Float16 a = (_Float16)(x[i][e / 4][e % 4] * qs);
                    q[0][i][e] = a; q[1][i][e] = (_Float16)fmaf(x[i][e / 4][e % 4], qs, -(float)a);
                }
        }
    }
    for (int i = threadIdx.x; i < cnt; i += 256) inv[i] = reinterpret_cast<const float2 *>(planes + half_scales_offset(UB, nkvh, tiles_all))[(size_t)kvh * tiles_all + t0 + i];
    __syncthreads();
    // Of the sums in o.  It follows the tiles' own, up at once and down in steps of more than 4, to 2^-64 of the largest at the lowest (o
    // then stays inside f32): the probabilities, times a tile's unit over this one, keep their halves' bits also behind a tile of
    // far larger values that a row may not see at all.
    float unit = inv[0].y, top = unit;
    float m = -INFINITY, l = 0.f;
    v16f o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
    issue(2, 2);
    int slot = 0;
    // unit u has landed for everybody, and everybody has left the place of unit u - 1, which u + NS - 1 gets
    auto next_unit = [&](int u) {
        if (u + NS - 2 < 2 * cnt) asm volatile("s_waitcnt vmcnt(%0)\n s_barrier" ::"n"((NS - 2) * LPU) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n s_barrier" ::: "memory");
        const char *base = half_lds + slot * UB + lane * 16;
        issue(u + NS - 1, slot == 0 ? NS - 1 : slot - 1);
        slot = slot == NS - 1 ? 0 : slot + 1;
        return base;
    };
    for (int it = 0; it < cnt; ++it) {
        const char *kb = next_unit(2 * it);
        const float k_unit = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(inv[it].x)));
        const float v_unit = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(inv[it].y)));
        v16f s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const v8h k0 = *reinterpret_cast<const v8h *>(kb + i * 1024), k1 = *reinterpret_cast<const v8h *>(kb + PLANE + i * 1024);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k1, q[0][i], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k0, q[1][i], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k0, q[0][i], s, 0, 0, 0);
        }
        const int t = t0 + it, k0 = 32 * t;
        // The raw scores' unit, kept off the ends of f32's range: a hidden score's -inf times 0, or a zero times inf, is NaN.  (Raw scores
        // are below 2^38: with the smallest unit all that is seen weighs the same, as it does with a smaller one.)
        float u = k_unit * s_unit;
        u = aa.scale > 0.f ? __builtin_amdgcn_fmed3f(u, 0x1p-126f, 0x1p126f) : aa.scale < 0.f ? __builtin_amdgcn_fmed3f(u, -0x1p126f, -0x1p-126f) : u;
        if (aa.logit_cap > 0.f || !(aa.scale > 0.f)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = aa.logit_cap > 0.f ? aa.logit_cap * tanhf(s[r] * u / aa.logit_cap) : s[r] * u;
            u = 1.0f;
        }
        if (!(k0 + 31 < kend && (aa.mask_kind == 0 || (aa.mask_kind == 1 && k0 + 31 <= aa.offset + qt_min)))) {
            const int mk = aa.mask_kind, qp = aa.offset + qt;  // attn_masked() as in the f32 kernel
            const uint32_t gw = mk == 3 ? aa.gbits[t] : 0u;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int kin = 8 * (r >> 2) + 4 * h + (r & 3), key = k0 + kin;
                const bool far = qp - key > aa.window;
                const bool hide = (key >= kend) | ((mk != 0) & (key > qp)) | ((mk == 2) & (key >= aa.sink) & far) | ((mk == 3) & far & !((gw >> kin) & 1u));
                s[r] = hide ? -INFINITY : s[r];
            }
        }
        float mt = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        mt *= u;
        // The probabilities' reference m follows the maximum in steps of more than HALVES_SLACK only (most tiles raise some row's
        // maximum a little): up to e^5 times 2^7 a probability is a half all the same.
        const float want = fmaxf(v_unit, top * 0x1p-64f);
        const bool new_unit = v_unit > unit || (want < 0.25f * unit && v_unit > HALVES_NO_VALUES);
        if (__any(mt > m + HALVES_SLACK || m == -INFINITY) || new_unit) {
            const float m_new = mt > m + HALVES_SLACK || m == -INFINITY ? fmaxf(m, mt) : m;
            float alpha = m == -INFINITY ? 1.0f : exp2f((m - m_new) * LOG2E);
            l *= alpha;
            m = m_new;
            if (new_unit) {  // (uniform, powers of two)
                alpha *= unit / want;
                unit = want;
                top = fmaxf(top, want);
            }
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        }
        const float to = 7.0f - (m == -INFINITY ? 0.0f : m * LOG2E), ul = u * LOG2E;  // (nothing visible yet: -inf stays below)
        const float p_scale = v_unit / unit;
        v8h p[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = __builtin_amdgcn_exp2f(fmaf(s[8 * j + e], ul, to));
                l += x;
                const _Float16 hi = (_Float16)(x * p_scale);
                p[0][j][e] = hi;
                p[1][j][e] = (_Float16)fmaf(x, p_scale, -(float)hi);
            }
        const char *vb = next_unit(2 * it + 1);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const char *at = vb + (j * NDT + dt) * 1024;
                const v8h v0 = *reinterpret_cast<const v8h *>(at), v1 = *reinterpret_cast<const v8h *>(at + PLANE);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v1, p[0][j], o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, p[1][j], o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v0, p[0][j], o[dt], 0, 0, 0);
            }
    }
    const float lt = l + __shfl_xor(l, 32);
    const bool whole = tiles <= aa.chunk;
    const float w = unit * (!whole ? 1.0f : lt > 0.f ? 1.0f / lt : 0.f);
    const size_t rec = HD + 4;
    if (!whole && h == 0 && row < nrows) *reinterpret_cast<float2 *>(aa.part + (((size_t)qt * aa.nqh + qh) * aa.splits + run) * rec) = float2{m, lt};
    // The rows leave through LDS, two d-tiles at a time: sixteen lanes to 256 bytes of a row.  (Stored as the lanes hold them, 16 bytes of
    // 64 places an instruction, they took 6 k cycles.)
    __syncthreads();
    float *tile = reinterpret_cast<float *>(half_lds) + wave * 32 * 68;
    float *dst[8];
    bool live[8];
    int first = row0;  // (worked out again: kept from the prologue, these places would cost the loop its registers)
    asm volatile("" : "+s"(first));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        int t, head;
        live[i] = row_of(first + 4 * i + (lane >> 4), t, head);
        const size_t r_out = (size_t)t * aa.nqh + head;
        dst[i] = (whole ? aa.out + r_out * HD : aa.part + (r_out * aa.splits + run) * rec + 4) + 4 * (lane & 15);
    }
#pragma unroll
    for (int d2 = 0; d2 < NDT; d2 += 2) {
#pragma unroll
        for (int dt = d2; dt < d2 + 2; ++dt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<float4 *>(tile + col * 68 + 32 * (dt - d2) + 8 * r4 + 4 * h) =
                    float4{o[dt][4 * r4] * w, o[dt][4 * r4 + 1] * w, o[dt][4 * r4 + 2] * w, o[dt][4 * r4 + 3] * w};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // (its own wavefront's tile)
        float4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const float4 *>(tile + (4 * i + (lane >> 4)) * 68 + 4 * (lane & 15));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (live[i]) {
                float4 *at = reinterpret_cast<float4 *>(dst[i] + 32 * d2);
                if (whole && aa.accumulate) {
                    const float4 old = *at;
                    v[i].x += old.x; v[i].y += old.y; v[i].z += old.z; v[i].w += old.w;
                }
                *at = v[i];
            }
    }
}

// The runs' records of every row that has more than one, HD / 4 lanes to a row; and what the next product reads instead of f32:
// AS = 3 / 4 byte digits for Q4_0 / Q8_0 (pg_emit_mm_digits), 5 f16 planes, a token to a workgroup of 1024 (nqh * HD <= 4096).  Rows of one run
// are then read from where the kernel above left them.  As a launch of its own behind this one the next product's input took 4 to 7 us: blocks of 711 tokens of
// d 1024 (Q8_0) 126 : 121.5 us, 679 of 2048 256.5 : 251, 602 behind 1841 270 : 264.5, Q4_0 450 of 2048 214 : 208.5, 350 164.5 : 160.5; as f16 planes
// 777 behind 100 of 4096 859 : 848 (the merge 9.8 + 6.2 : 10.9).
// MOST: runs at the most; four take a third of the registers of sixteen (34 : 106), so that twice the wavefronts wait for memory at a time (the f16 planes 15 : 10.9).
constexpr int HALVES_RUNS_MAX = 16, HALVES_RUNS_FEW = 4;
struct halves_next {
    int8_t *digits;
    float *xs;
    _Float16 *hi, *lo;
    float *inv;
};
template <int HD, int AS, int MOST>
__global__ __launch_bounds__(AS == 5 ? 1024 : 256) void attn_halves_combine_kernel(attn_args aa, halves_next next) {
    constexpr int LPR = HD / 4;
    const int G = aa.group, nrows = G * aa.seq_q, rows = aa.nqh * aa.seq_q;
    const int r_out = AS == 5 ? (int)blockIdx.x * aa.nqh + (int)threadIdx.x / LPR : (int)blockIdx.x * (256 / LPR) + (int)threadIdx.x / LPR;
    const int d = (threadIdx.x % LPR) * 4;
    const bool live = AS == 5 ? (int)threadIdx.x < aa.nqh * LPR : r_out < rows;
    if (AS != 5 && !live) return;
    const int qt = AS == 5 ? (int)blockIdx.x : r_out / aa.nqh, head = r_out - qt * aa.nqh, row = qt * G + head % G;
    const int tiles = halves_tiles(aa, row / HALVES_ROWS, nrows), runs = live ? (tiles + aa.chunk - 1) / aa.chunk : 0;
    if (AS == 0 && runs < 2) return;
    float4 *at = reinterpret_cast<float4 *>(aa.out + (size_t)r_out * HD + d);
    float4 w = {0.f, 0.f, 0.f, 0.f};
    if (runs >= 2) {
        const float *rec = aa.part + (size_t)r_out * aa.splits * (HD + 4);
        float2 ml[MOST];
        float4 v[MOST];
#pragma unroll
        for (int i = 0; i < MOST; ++i)
            if (i < aa.splits) {
                const float *p = rec + (size_t)min(i, runs - 1) * (HD + 4);
                ml[i] = *reinterpret_cast<const float2 *>(p);
                v[i] = *reinterpret_cast<const float4 *>(p + 4 + d);
            }
        float m = -INFINITY;
#pragma unroll
        for (int i = 0; i < MOST; ++i)
            if (i < runs) m = fmaxf(m, ml[i].x);
        float l = 0.f;
        float4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < MOST; ++i)
            if (i < runs) {
                const float e = ml[i].x == -INFINITY ? 0.f : expf(ml[i].x - m);
                l = fmaf(ml[i].y, e, l);
                o.x = fmaf(v[i].x, e, o.x); o.y = fmaf(v[i].y, e, o.y); o.z = fmaf(v[i].z, e, o.z); o.w = fmaf(v[i].w, e, o.w);
            }
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        w = float4{o.x * inv, o.y * inv, o.z * inv, o.w * inv};
    } else if (runs == 1) {
        w = *at;
    }
    if constexpr (AS == 0) {
        if (aa.accumulate) {
            const float4 old = *at;
            w.x += old.x; w.y += old.y; w.z += old.z; w.w += old.w;
        }
        *at = w;
    } else {
        const float f[4] = {w.x, w.y, w.z, w.w};
        if constexpr (AS == 5) {
            __shared__ float red[16];
            float amax = fmaxf(fmaxf(pg_f16_mag(f[0]), pg_f16_mag(f[1])), fmaxf(pg_f16_mag(f[2]), pg_f16_mag(f[3])));
            for (int o = 32; o; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
            if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
            __syncthreads();
            for (int i = 0; i < 16; ++i) amax = fmaxf(amax, red[i]);
            const pg_f16_row_scale sc = pg_f16_row_scale_of(amax);
            if (threadIdx.x == 0) {
                next.inv[2 * qt] = sc.i1;
                next.inv[2 * qt + 1] = sc.i2;
            }
            const size_t k = (size_t)r_out * HD + d;
            if (live) pg_f16_split4(f, sc, reinterpret_cast<uint2 *>(next.hi + k), reinterpret_cast<uint2 *>(next.lo + k));
        } else {
            const int nb = aa.nqh * (HD / 32);
            pg_emit_mm_digits<AS == 3>(f, (size_t)qt, head * (HD / 32) + d / 32, threadIdx.x & 7, nb, (nb + 3) / 4 * 4, next.digits, next.xs);
        }
    }
}
