// route_device.h -- the router's choice of experts on the device: per row, and for up to 16 rows as one workgroup's work.
#pragma once
#include "lane_device.h"
#include "layered_kernels.h"
#include "seq_device.h"

#include <math.h>

enum { ROUTE_EPL = 8, ROUTE_MAX_EXPERTS = 64 * ROUTE_EPL };
// one wave chooses the `top` largest of a row's logits (lowest index first among equals) and the softmax over them; lane k holds
// choice k for k < top (top <= 64)
DEV void choose(const float* z, int experts, int top, int lane, int* e_out, float* w_out) {
  float v[ROUTE_EPL];
#pragma unroll
  for (int i = 0; i < ROUTE_EPL; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < experts ? z[e] : -INFINITY;
  }
  int mine = 0;
  float zm = -INFINITY, first = 0.f;
  unsigned taken = 0;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int be = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < ROUTE_EPL; ++i) {
      const int e = lane + 64 * i;
      if (e < experts && !((taken >> i) & 1) && (v[i] > best || be == 0x7fffffff)) {
        best = v[i];
        be = e;
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float ob = lane_xor(best, off);
      const int oe = lane_xor(be, off);
      if (oe != 0x7fffffff && (be == 0x7fffffff || ob > best || (ob == best && oe < be))) {
        best = ob;
        be = oe;
      }
    }
    if ((be & 63) == lane) taken |= 1u << (be >> 6);
    if (k == 0) first = best;
    if (lane == k) {
      mine = be;
      zm = best;
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
