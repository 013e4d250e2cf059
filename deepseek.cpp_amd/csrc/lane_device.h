// lane_device.h -- a value from the lane at xor distance 1, 2, 4, .. 32, for waves with all lanes on (what __shfl_xor gives).
//
// __shfl_xor is an LDS instruction (ds_bpermute: an address, a round trip of some 100 cycles, six of them in a row for a wave's sum, eighteen for
// a block's largest value and its place).  Inside a row of 16 lanes the exchange is a modifier of a vector instruction, across rows one of
// gfx950's two lane swaps.  Both in turn on one card, us a token: DeepSeek-V2-Lite's shapes, Q2_K 1459 -> 1431, F8E5M2 1608 -> 1589; 27 small layers with
// recurrences 2098 -> 2064; V3's shapes and wide layers the same.  `off` is a constant behind unrolling.  Still by LDS: attention in
// kernels_mix_few.hip, mla_flash_kernel, sampling, and shifts (__shfl_up: the mLSTM's gates).
#pragma once
#include <hip/hip_runtime.h>
template <typename T>
__device__ __forceinline__ T lane_xor(T v, int off) {
  static_assert(sizeof(T) == 4, "32-bit values");
  const unsigned u = __builtin_bit_cast(unsigned, v);
  unsigned r;
  if (off == 32 || off == 16) {
    const unsigned lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    if (off == 32) {
      const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);  // the lower half's values twice, the upper half's twice
      r = lane & 32 ? s[0] : s[1];
    } else {
      const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);  // rows 0 0 2 2, rows 1 1 3 3
      r = lane & 16 ? s[0] : s[1];
    }
  } else if (off == 8) {
    r = __builtin_amdgcn_update_dpp(u, u, 0x128, 0xf, 0xf, true);  // rotate the row by 8
  } else if (off == 4) {
    r = __builtin_amdgcn_update_dpp(u, u, 0x104, 0xf, 0x5, false);  // quads 0 and 2 of a row from 4 lanes above,
    r = __builtin_amdgcn_update_dpp(r, u, 0x114, 0xf, 0xa, false);  // quads 1 and 3 from 4 lanes below
  } else if (off == 2) {
    r = __builtin_amdgcn_update_dpp(u, u, 0x4e, 0xf, 0xf, true);
  } else {
    r = __builtin_amdgcn_update_dpp(u, u, 0xb1, 0xf, 0xf, true);
  }
  return __builtin_bit_cast(T, r);
}
