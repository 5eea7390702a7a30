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
// Sum over the 64 lanes, the same in every lane, in the order of the sweeps' sums (xor 32, 16, .. 1), so that a step gives
// the same norms to the last bit whichever kernel runs it: swaps of half waves and of rows, rotations in the row of 16
// (by 8, and by 4 once the row repeats after 8), quad permutations.
__device__ __forceinline__ double wave_sum(double v) {
    const auto l5 = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    const auto h5 = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(int(h5[0]), int(l5[0])) + __hiloint2double(int(h5[1]), int(l5[1]));
    const auto l4 = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto h4 = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(int(h4[0]), int(l4[0])) + __hiloint2double(int(h4[1]), int(l4[1]));
    v += dpp_move<0x128>(v);
    v += dpp_move<0x124>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0xB1>(v);
    return v;
}

// Orders the wave's own LDS accesses (the compiler's; a wave's LDS instructions execute in order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace gs
