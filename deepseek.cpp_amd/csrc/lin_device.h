// lin_device.h -- what the matrix products of layered models share: epilogues out of one lane's accumulator, parts of k, operands.
#pragma once
#include "seq_device.h"

// ---- epilogues: four consecutive features of one row, out of one lane's accumulator ----------------
DEV float glu(float g, float u, float limit, float alpha, float offset) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoid_f(alpha * g) * (u + offset);
}
// EPI: a.epi, or -1: whatever it is.  (A tile's kernel holds its epilogue once per accumulator, and every copy of what it could be as well is read into the
// instruction cache, 64 KiB, for one pass: 12 us of a 256 x 256 tile's 70, with 163 KiB of code.)
template <int EPI>
DEV f32x4 activated(const LinArgs& a, int feature, f32x4 v) {
  const int epi = EPI < 0 ? a.epi : EPI;
  if (epi == LIN_SOFTCAP) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a.p0 * tanhf(v[i] / a.p0);
  } else if (epi == LIN_SCALE) {
    v *= a.p0;
  } else if (epi == LIN_XIELU) {
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (exp(z) - 1 - z: its absolute error is a rounding of 1, and z / 2 is beside it)
      v[i] = 0.5f * v[i] + (v[i] > 0.f ? a.p0 * v[i] * v[i] : a.p1 * (__expf(fminf(v[i], 0.f)) - 1.f - v[i]));
  } else if (epi == LIN_TANH_F && feature >= a.n_wide) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = tanhf(v[i]);
  }
  return v;
}
template <typename T, int EPI = -1>
DEV void store_plain(const LinArgs& a, int row, int feature, f32x4 v) {
  typedef typename Frag<T>::four four;
  v = activated<EPI>(a, feature, v);
  if (feature < a.n_wide) *reinterpret_cast<four*>(reinterpret_cast<T*>(a.out_t) + (size_t)row * a.ld_t + feature) = to_four<T>(v);
  else *reinterpret_cast<f32x4*>(a.out_f + (size_t)row * a.ld_f + feature - a.n_wide) = v;
}
// Feature tiles rt and rt + 1 of a row in bfloat16, 16 bytes a lane instead of twice 8: lane rows 0 and 2 keep tile rt and take its other halves from rows 1
// and 3, which take tile rt + 1's.  All lanes are on; `in`: there is such a row.  (Rows of whole 16 bytes: wide_pairs.)
__host__ DEV bool wide_pairs(const LinArgs& a) { return (a.ld_t & 7) == 0 && ((unsigned long long)a.out_t & 15) == 0; }
template <int EPI>
DEV void store_wide_pair(const LinArgs& a, bool in, int row, int rt, const f32x4& u, const f32x4& v) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const u32x2 p = __builtin_bit_cast(u32x2, to_four<bf16>(activated<EPI>(a, rt * 16, u))), q = __builtin_bit_cast(u32x2, to_four<bf16>(activated<EPI>(a, rt * 16 + 16, v)));
  const auto s = __builtin_amdgcn_permlane16_swap(p.x, q.x, false, false), t = __builtin_amdgcn_permlane16_swap(p.y, q.y, false, false);
  if (in) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(a.out_t) + (size_t)row * a.ld_t + (rt + (lane >> 4 & 1)) * 16 + (lane >> 5) * 8) = u32x4{s[0], t[0], s[1], t[1]};
}
template <typename T>
DEV void store_glu(const LinArgs& a, int row, int feature, const f32x4& g, const f32x4& u) {
  typedef typename Frag<T>::four four;
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = glu(g[i], u[i], a.p0, a.p1, a.p2);
  *reinterpret_cast<four*>(reinterpret_cast<T*>(a.out_t) + (size_t)row * a.ld_t + feature) = to_four<T>(v);
}

// k tiles per part: even, so that a part is whole steps of the prompt kernels
__host__ DEV int part_tiles(int kt, int parts) { return parts > 1 ? ((kt / 2 + parts - 1) / parts) * 2 : kt; }
__host__ DEV int part_tiles(const LinArgs& a) { return part_tiles(a.kt, a.parts); }
// the operand a product's features from `feature` on read
template <typename T>
DEV const T* operand(const LinArgs& a, int feature) {
  const T* p = reinterpret_cast<const T*>(a.a_t);
  return a.a_seg ? p + (size_t)min(feature / a.a_seg, a.a_ops - 1) * a.a_stride : p;
}
