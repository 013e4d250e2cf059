// route_device.h -- the router's choice of experts on the device: per row, and for up to 16 rows as one workgroup's work.
#pragma once
#include "lane_device.h"
#include "layered_kernels.h"
#include "seq_device.h"

#include <math.h>

enum { ROUTE_EPL = 8, ROUTE_MAX_EXPERTS = 64 * ROUTE_EPL };
// floats in an order that whole numbers have (0: none; no number and both zeros as one float each), and back
DEV unsigned order_of(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v + 0.f);
  return v != v ? 1u : u >> 31 ? ~u : u | 0x80000000u;
}
DEV float of_order(unsigned o) { return __builtin_bit_cast(float, o >> 31 ? o ^ 0x80000000u : ~o); }
DEV unsigned wave_max(unsigned v) {
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));   // quad_perm [1, 0, 3, 2]
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));   // quad_perm [2, 3, 0, 1]
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));  // row_half_mirror
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));  // row_mirror
  v = max(v, lane_xor(v, 16));
  v = max(v, lane_xor(v, 32));
  return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}
// One wave chooses the `top` largest of a row's logits (lowest index first among equals) and the softmax over them; lane k holds
// choice k for k < top (top <= 64).  All lanes are on.  A choice is the largest value of the wave and the first lane that has it: with value and index
// exchanged together, six rounds of a dozen instructions each, the chain was four times as long (route_count_kernel).
DEV void choose(const float* z, int experts, int top, int lane, int* e_out, float* w_out) {
  unsigned v[ROUTE_EPL];
#pragma unroll
  for (int i = 0; i < ROUTE_EPL; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < experts ? order_of(z[e]) : 0u;
  }
  int mine = 0;
  float zm = -INFINITY, first = 0.f;
  for (int k = 0; k < top; ++k) {
    unsigned best = v[0];
#pragma unroll
    for (int i = 1; i < ROUTE_EPL; ++i) best = max(best, v[i]);
    best = wave_max(best);
    int be = -1;
#pragma unroll
    for (int i = 0; i < ROUTE_EPL; ++i) {
      const unsigned long long has = __ballot(v[i] == best);
      if (be < 0 && has) {
        be = 64 * i + __ffsll(has) - 1;
        if (be == 64 * i + lane) v[i] = 0u;
      }
    }
    const float value = of_order(best);
    if (k == 0) first = value;
    if (lane == k) {
      mine = be;
      zm = value;
    }
  }
  const float ex = lane < top ? expf(zm - first) : 0.f;
  *w_out = ex / wave_sum(ex);
  *e_out = mine;
}
// Up to 16 rows, by one workgroup of 1024 threads: a wave per row chooses, then the list of chosen experts.  lds: route_few_lds() bytes
DEV void route_few_body(const MoeArgs& a, char* lds) {
  typedef unsigned char row16[16];
  row16* slot_of = reinterpret_cast<row16*>(lds);
  int* wave_n = reinterpret_cast<int*>(lds + ROUTE_MAX_EXPERTS * 16);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < ROUTE_MAX_EXPERTS * 4; i += 1024) reinterpret_cast<unsigned*>(slot_of)[i] = 0xffffffffu;
  __syncthreads();
  const int ns = a.top + a.shared;
  if (wave < a.rows) {
    int e;
    float w;
    choose(a.logits + (size_t)wave * a.ld_logits, a.experts, a.top, lane, &e, &w);
    if (lane < ns) {
      a.weight[wave * ns + lane] = lane < a.top ? w : 1.f;
      a.slot_pos[wave * ns + lane] = wave * ns + lane;
    }
    if (lane < a.top) {
      a.chosen[wave * a.top + lane] = e;
      slot_of[e][wave] = (unsigned char)lane;
    }
  }
  __syncthreads();
  bool used = false;
  if (tid < a.experts) {
    const unsigned* s = reinterpret_cast<const unsigned*>(slot_of[tid]);
    used = (s[0] & s[1] & s[2] & s[3]) != 0xffffffffu;
  }
  const unsigned long long mask = __ballot(used);
  if (lane == 0) wave_n[wave] = __popcll(mask);
  __syncthreads();
  int base = 0, total = 0;
  for (int i = 0; i < 16; ++i) {
    if (i < wave) base += wave_n[i];
    total += wave_n[i];
  }
  if (used) {
    const int p = base + __popcll(mask & ((1ull << lane) - 1));
    a.active[p] = tid;
    for (int r = 0; r < 16; ++r) a.active_slot[p * 16 + r] = slot_of[tid][r] == 0xff ? -1 : slot_of[tid][r];
  }
  if (a.shared && tid < 16) {
    a.active_slot[total * 16 + tid] = tid < a.rows ? a.top : -1;
    if (tid == 0) a.active[total] = a.experts;
  }
  if (tid == 0) *a.n_active = total + a.shared;
}
enum { ROUTE_FEW_LDS = ROUTE_MAX_EXPERTS * 16 + 64 };
