// Wave-wide helpers of the kernels that keep their tables in LDS.
#pragma once
#include <hip/hip_runtime.h>

namespace gs {

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double swap32_add(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(int(h[0]), int(l[0])) + __hiloint2double(int(h[1]), int(l[1]));
}
__device__ __forceinline__ double swap16_add(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(int(h[0]), int(l[0])) + __hiloint2double(int(h[1]), int(l[1]));
}
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_move<0x128>(v);
    v += dpp_move<0x124>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0xB1>(v);
    return v;
}
// Sum over the 64 lanes, the same in every lane, in the order of the sweeps' sums (xor 32, 16, .. 1), so that a step gives
// the same norms to the last bit whichever kernel runs it: swaps of half waves and of rows, rotations in the row of 16
// (by 8, and by 4 once the row repeats after 8), quad permutations.
__device__ __forceinline__ double wave_sum(double v) {
    v = swap32_add(v, v);
    return row_sum(swap16_add(v, v));
}

// The same sums of two and of four values at once: half waves, then rows, take one value each, so that only the first
// levels work on more than one register.  sum2: v[0], v[1] in the lower and upper half; sum4: v[0], v[2], v[1], v[3] in
// rows 0 .. 3.
__device__ __forceinline__ double sum2(const double (&v)[4]) {
    const double x = swap32_add(v[0], v[1]);
    return row_sum(swap16_add(x, x));
}
__device__ __forceinline__ double sum4(const double (&v)[4]) {
    return row_sum(swap16_add(swap32_add(v[0], v[1]), swap32_add(v[2], v[3])));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Has the value in a register here, so that what made it is not moved behind the branches that follow.
__device__ __forceinline__ void here(double& v) { asm volatile("" : "+v"(v)); }

// Orders the wave's own LDS accesses (the compiler's; a wave's LDS instructions execute in order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace gs
