// Wave-level moves and sums of doubles (gfx950, 64 lanes).
#pragma once

#include <hip/hip_runtime.h>

namespace stm {

// One DPP move of a double (both halves); lanes of rows outside ROWS keep
// `old`'s value.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_move(double v, double old) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL,
                                               ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL,
                                               ROWS, 0xf, false);
    return __hiloint2double(hi, lo);
}

// The sum of v over the wave, in VALU (DPP) steps rather than LDS round
// trips, in a fixed order: pairs, quads, the quads of a row, then rows
// (r0 + r1) and (r2 + r3), then (r2 + r3) + (r0 + r1).  Uniform result.
__device__ __forceinline__ double wave_sum(double v) {
    v = v + dpp_move<0xb1>(v, 0.0);          // quad_perm [1, 0, 3, 2]
    v = v + dpp_move<0x4e>(v, 0.0);          // quad_perm [2, 3, 0, 1]
    v = v + dpp_move<0x124>(v, 0.0);         // row_ror 4
    v = v + dpp_move<0x128>(v, 0.0);         // row_ror 8
    v = v + dpp_move<0x142, 0xa>(v, 0.0);    // row_bcast 15 into rows 1, 3
    v = v + dpp_move<0x143, 0xc>(v, 0.0);    // row_bcast 31 into rows 2, 3
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
    return __hiloint2double(hi, lo);
}

}  // namespace stm
