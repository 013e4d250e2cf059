// lin_device.h -- what the matrix products of layered models share: epilogues out of one lane's accumulator, parts of k, operands.
#pragma once
#include "seq_device.h"

// ---- epilogues: four consecutive features of one row, out of one lane's accumulator ----------------
DEV float glu(float g, float u, float limit, float alpha, float offset) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoid_f(alpha * g) * (u + offset);
}
template <typename T>
DEV void store_plain(const LinArgs& a, int row, int feature, f32x4 v) {
  typedef typename Frag<T>::four four;
  if (a.epi == LIN_SOFTCAP) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a.p0 * tanhf(v[i] / a.p0);
  } else if (a.epi == LIN_SCALE) {
    v *= a.p0;
  } else if (a.epi == LIN_XIELU) {
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (exp(z) - 1 - z: its absolute error is a rounding of 1, and z / 2 is beside it)
      v[i] = 0.5f * v[i] + (v[i] > 0.f ? a.p0 * v[i] * v[i] : a.p1 * (__expf(fminf(v[i], 0.f)) - 1.f - v[i]));
  } else if (a.epi == LIN_TANH_F && feature >= a.n_wide) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = tanhf(v[i]);
  }
  if (feature < a.n_wide) *reinterpret_cast<four*>(reinterpret_cast<T*>(a.out_t) + (size_t)row * a.ld_t + feature) = to_four<T>(v);
  else *reinterpret_cast<f32x4*>(a.out_f + (size_t)row * a.ld_f + feature - a.n_wide) = v;
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
