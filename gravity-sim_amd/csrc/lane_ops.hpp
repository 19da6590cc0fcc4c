// Exchanges between the lanes of a wave that need no LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace gsim {

// v of the lane named by a DPP control; the kDppXor* controls name lane ^ n
// within each row of 16 lanes (^ 7 and ^ 15 mirror 8 and 16 lanes).
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xF, 0xF, true));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppXor7 = 0x141, kDppXor15 = 0x140;

}  // namespace gsim
