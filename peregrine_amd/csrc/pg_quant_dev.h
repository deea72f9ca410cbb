// Device helpers of the activation quantisation, shared by the row kernels (pg_quant.hip) and the
// one-row product that quantises its own activations (pg_gemv_w8a8.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

// round -> clamp(-127,127) -> `as i8` (NaN -> 0), returned as int.   src/quant.rs:101-106
// Half away from zero is truncation after adding the float just under a half with the value's sign: with a half itself 0.49999997 would
// reach 1, and every k + 0.5 still does (the exact sum lies a quarter of an ulp or less below k + 1 and rounds up to it; from 0.5 it lies half an ulp below 1, a
// tie, which goes to the even 1).  Checked against roundf for every
// float to 144.  The conversion truncates, takes NaN to 0 and saturates (asm: in C++ that would be undefined).  Five vector instructions with
// the caller's product, where roundf, two clamps and two tests for NaN were fourteen.  With the maximum below, us, before : now: the
// products of a layer for one row 42.7 : 41.4, 27 rows of a smaller one 34.4 : 33.5; a single small product and layers of
// 2048 rows (468 : 464) within what runs differ.
__device__ __forceinline__ int pg_quant_to_i8(float v) {
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(v + copysignf(0x1.fffffep-2f, v)));
    return min(max(i, -127), 127);
}

// Four of them as the bytes of a dword.
__device__ __forceinline__ int pg_quant4_to_i8(float x, float y, float z, float w) {
    const unsigned lo = __builtin_amdgcn_perm((unsigned)pg_quant_to_i8(y), (unsigned)pg_quant_to_i8(x), 0x0C0C0400u);
    const unsigned hi = __builtin_amdgcn_perm((unsigned)pg_quant_to_i8(w), (unsigned)pg_quant_to_i8(z), 0x04000C0Cu);
    return (int)(lo | hi);
}

// Maximum over the 64 lanes of a wavefront, all of them active, in every lane; values of either sign and -inf (scores, logits), NaN passed over as by fmaxf: DPP moves within rows of 16 lanes, then the four rows' through scalar
// registers (six exchanges through LDS were a chain of 0.2 us).
__device__ __forceinline__ float pg_wave_max_f32(float v) {
    auto step = [](float x, auto ctrl) {
        const int y = __builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, false);
        return fmaxf(x, __int_as_float(y));
    };
    v = step(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    v = step(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    v = step(v, std::integral_constant<int, 0x141>{});  // row_half_mirror
    v = step(v, std::integral_constant<int, 0x140>{});  // row_mirror
    const int b = __float_as_int(v);
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(b, 0)), __int_as_float(__builtin_amdgcn_readlane(b, 16))),
                 fmaxf(__int_as_float(__builtin_amdgcn_readlane(b, 32)), __int_as_float(__builtin_amdgcn_readlane(b, 48))));
}

// Sum over aligned groups of `lanes` (1, 2, 4 .. 64), in every lane of the group; every step adds what lane ^ 1, 2, 4 .. holds (a
// mirror image does where the lanes it differs in hold the same).  A shuffle through LDS at every step was most of the scores' latency in the short attention
// kernels: a block of 1024 (Q4_0), 2 tokens behind 154 42.7 -> 41.3 us, of 2048, 4 behind 100 46.4 -> 45.0.
__device__ __forceinline__ float pg_group_sum_f32(float v, int lanes) {
    auto step = [](float x, auto ctrl) { return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, false)); };
    if (lanes > 1) v = step(v, std::integral_constant<int, 0xB1>{});
    if (lanes > 2) v = step(v, std::integral_constant<int, 0x4E>{});
    if (lanes > 4) v = step(v, std::integral_constant<int, 0x141>{});
    if (lanes > 8) v = step(v, std::integral_constant<int, 0x140>{});
    if (lanes > 16) {
        const unsigned b = __float_as_uint(v);
        const auto two = __builtin_amdgcn_permlane16_swap(b, b, false, false);
        v = __uint_as_float(two[0]) + __uint_as_float(two[1]);
    }
    if (lanes > 32) {
        const unsigned b = __float_as_uint(v);
        const auto two = __builtin_amdgcn_permlane32_swap(b, b, false, false);
        v = __uint_as_float(two[0]) + __uint_as_float(two[1]);
    }
    return v;
}

// Maximum over a 256-thread workgroup; `red` = 4 floats of LDS.  Ends with every thread past a barrier.
__device__ __forceinline__ float pg_block_max_256(float v, float *red) {
    v = pg_wave_max_f32(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    return v;
}

// The same without draining the wavefront's outstanding global loads (__syncthreads() waits for
// vmcnt(0) as well): for kernels that keep weight rows in flight across the reduction.
__device__ __forceinline__ float pg_block_max_256_keep_loads(float v, float *red) {
    v = pg_wave_max_f32(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
    v = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    return v;
}
