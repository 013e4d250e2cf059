// join_device.h -- one row of the residual sum between the products of layered models, the norm behind it, and the convolution and blends that may
// follow for a sequence's only token: by itself (kernels_join.hip), or in front of the product that reads it (kernels_enter.hip).
#pragma once
#include "seq_device.h"

// A workgroup takes a row; a thread keeps VPT groups of V consecutive elements in registers (V = 4, or 1 for widths that 4 does not divide).
template <typename S, int V>
DEV void load_v(const S* p, bool in, float (&v)[V]) {
  if constexpr (V == 4) {
    typedef S s4 __attribute__((ext_vector_type(4)));
    const s4 q = in ? *reinterpret_cast<const s4*>(p) : s4{};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (float)q[e];
  } else {
    v[0] = in ? (float)p[0] : 0.f;
  }
}
template <typename S, int V>
DEV void store_v(S* p, const float (&v)[V]) {
  if constexpr (V == 4) {
    typedef S s4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<s4*>(p) = s4{(S)v[0], (S)v[1], (S)v[2], (S)v[3]};
  } else {
    p[0] = (S)v[0];
  }
}
// PUB: for readers on other compute units of the same launch - written through, past this unit's caches
template <typename S, int V, bool PUB>
DEV void store_h(S* p, const float (&v)[V]) {
  if constexpr (PUB) {
    typedef S s4 __attribute__((ext_vector_type(4)));
    static_assert(sizeof(S) == 2 && V == 4, "8 bytes a store");
    const s4 s = {(S)v[0], (S)v[1], (S)v[2], (S)v[3]};
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    store_v<S, V>(p, v);
  }
}
// A sequence's only token of the pass: V channels of h through the convolution.  TAPS = 4: what that needs from memory is requested at
// once, early enough to be there when h is (the blends' weights: up to MAX_MIX); TAPS = 1: any number of taps, one after the other.
template <int V, int TAPS>
struct ConvOne {
  enum { MAX_MIX = 5, KEPT = TAPS > 1 ? TAPS - 1 : 1, MIX = TAPS > 1 ? (int)MAX_MIX : 1 };
  float old[KEPT][V], w[V * TAPS], mu[MIX][V], prev[V];
  const float* hist;
  float *next, *p_next;
  DEV void load(const JoinArgs& j, const SeqDesc& s, int c) {
    const ConvArgs& a = j.conv;
    const int D = j.width, taps = TAPS > 1 ? TAPS : a.taps;
    hist = reinterpret_cast<const float*>(s.state + a.off_in) + (size_t)s.flip * (taps - 1) * D + c;
    next = reinterpret_cast<float*>(s.state + a.off_in) + (size_t)(s.flip ^ 1) * (taps - 1) * D + c;
    p_next = reinterpret_cast<float*>(s.state + a.off_prev) + c + (size_t)(s.flip ^ 1) * D;
    if (c >= D) return;
    if constexpr (TAPS > 1) {  // (what the descriptor has no part in first)
#pragma unroll
      for (int e = 0; e < TAPS; ++e) load_v<float, V>(a.w + (size_t)c * taps + e * V, true, *reinterpret_cast<float(*)[V]>(w + e * V));
      if (a.mu) {
#pragma unroll
        for (int i = 0; i < MIX; ++i) load_v<float, V>(a.mu + (size_t)min(i, a.n_mix - 1) * D + c, true, mu[i]);
      }
#pragma unroll
      for (int t = 0; t < KEPT; ++t) load_v<float, V>(hist + (size_t)t * D, s.pos0 - (taps - 1) + t >= 0, old[t]);
    }
    if (a.mu) load_v<float, V>(reinterpret_cast<const float*>(s.state + a.off_prev) + c + (size_t)s.flip * D, s.pos0 > 0, prev);
  }
  template <typename T, bool PUB>
  DEV void run(const JoinArgs& j, int row, int pos0, int c, const float (&h)[V]) {
    const ConvArgs& a = j.conv;
    const int D = j.width, taps = TAPS > 1 ? TAPS : a.taps;
    T* out = reinterpret_cast<T*>(a.out_t) + (size_t)row * a.ld + c;
    float y[V];
#pragma unroll
    for (int e = 0; e < V; ++e) y[e] = 0.f;
    if constexpr (TAPS > 1) {
#pragma unroll
      for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] += (t == TAPS - 1 ? h[e] : old[t < KEPT ? t : 0][e]) * w[e * TAPS + t];
#pragma unroll
      for (int t = 1; t < KEPT; ++t) store_v<float, V>(next + (size_t)(t - 1) * D, old[t]);
    } else {
      for (int t = 0; t < taps - 1; ++t) {
        float o[V];
        load_v<float, V>(hist + (size_t)t * D, pos0 - (taps - 1) + t >= 0, o);
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] += o[e] * a.w[(size_t)(c + e) * taps + t];
        if (t > 0) store_v<float, V>(next + (size_t)(t - 1) * D, o);
      }
#pragma unroll
      for (int e = 0; e < V; ++e) y[e] += h[e] * a.w[(size_t)(c + e) * taps + taps - 1];
    }
    if (taps > 1) store_v<float, V>(next + (size_t)(taps - 2) * D, h);
#pragma unroll
    for (int e = 0; e < V; ++e) y[e] += h[e];
    if (!a.mu) {
      store_h<T, V, PUB>(out, y);
      return;
    }
    store_v<float, V>(p_next, y);
    auto blend = [&](int i, const float (&m)[V]) {
      float v[V];
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = y[e] + (prev[e] - y[e]) * m[e];
      store_h<T, V, PUB>(out + i * a.mix_stride, v);
    };
    if constexpr (TAPS > 1) {
#pragma unroll
      for (int i = 0; i < MIX; ++i)
        if (i < a.n_mix) blend(i, mu[i]);
    } else {
      for (int i = 0; i < a.n_mix; ++i) {
        float m[V];
        load_v<float, V>(a.mu + (size_t)i * D + c, true, m);
        blend(i, m);
      }
    }
  }
};
// the sum of up to 8 rows, all requested at once (threads with many groups of elements: one row after the other)
template <int V, bool MANY>
struct LoadSum {
  float q[MANY ? 1 : 8][V];
  DEV void load(const float* p, bool in, int parts, size_t stride) {
    if constexpr (MANY) {
      load_v<float, V>(p, in, q[0]);
#pragma unroll 1
      for (int u = 1; u < parts; ++u) {
        float w[V];
        load_v<float, V>(p + u * stride, in, w);
#pragma unroll
        for (int e = 0; e < V; ++e) q[0][e] += w[e];
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) load_v<float, V>(p + u * stride, in && u < max(parts, 1), q[u]);
    }
  }
  DEV void sum(float (&v)[V]) const {
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = MANY ? q[0][e] : ((q[0][e] + q[1][e]) + (q[2][e] + q[3][e])) + ((q[4][e] + q[5][e]) + (q[6][e] + q[7][e]));
  }
};
template <int NT>
struct JoinLds {
  float red[NT / 64], w[64];
  int pos[64];
};
// CONV: taps of the convolution behind the norm (single tokens; ConvOne), 0: none
template <typename T, int NT, int VPT, int V, int CONV, bool PUB>
DEV void join_row(const JoinArgs& a, int block, JoinLds<NT>& lds) {
  float(&red)[NT / 64] = lds.red;
  float(&s_w)[64] = lds.w;
  int(&s_pos)[64] = lds.pos;
  const int tid = threadIdx.x, D = a.width;
  const int row = a.only_want ? a.p.want[block] : block;
  const int hrow = block;
  float x[VPT][V], add[VPT][V];
  auto at = [&](int i) { return V * (tid + i * NT); };
  // with a convolution behind the norm (single tokens: row = sequence): everything it reads and the norms' weights, requested behind the
  // sum's operands (one group per thread) or together with its use (more)
  ConvOne<V, (CONV > 1 ? CONV : 1)> cv;
  SeqDesc sq{};
  float nw[V], pw[V];
  if constexpr (CONV > 0) sq = seq_at(a.p.seqs + row);
  if (a.y_t && tid < a.n_slots) {
    s_w[tid] = a.weight[(size_t)row * a.n_slots + tid];
    s_pos[tid] = a.slot_pos[(size_t)row * a.n_slots + tid];
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if (a.embed) load_v<bf16, V>(reinterpret_cast<const bf16*>(a.embed) + (size_t)a.p.tokens[row] * D + at(i), at(i) < D, x[i]);
    else load_v<float, V>(a.x + (size_t)row * D + at(i), at(i) < D, x[i]);
#pragma unroll
    for (int e = 0; e < V; ++e) add[i][e] = 0.f;
  }
  if constexpr (CONV > 0 && VPT == 1) {
    if (!a.mix_a) {
      load_v<float, V>(a.norm_w + at(0), at(0) < D, nw);
      cv.load(a, sq, at(0));
    }
  }
  if (a.mix_a) {
    const float* ma = a.mix_a + (size_t)row * a.mix_ld;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      LoadSum<V, (VPT > 2)> q;
      q.load(ma + at(i), at(i) < D, a.parts_a, a.mix_stride);
      if constexpr (CONV > 0 && VPT == 1) {
        if (a.post_w) load_v<float, V>(a.post_w + at(0), at(0) < D, pw);
        load_v<float, V>(a.norm_w + at(0), at(0) < D, nw);
        cv.load(a, sq, at(0));
      }
      q.sum(add[i]);
    }
    if (a.mix_b) {
      const float* mb = a.mix_b + (size_t)row * a.mix_ld;
      float vb[VPT][V];
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        LoadSum<V, (VPT > 2)> q;
        q.load(mb + at(i), at(i) < D, a.parts_b, a.mix_stride);
        q.sum(vb[i]);
      }
      const float sa = block_sum<NT>(squares<VPT, V, V == 1 ? 0 : 1>(add), red), sb = block_sum<NT>(squares<VPT, V, V == 1 ? 0 : 1>(vb), red);
      const float ra = 1.f / sqrtf(sa / D + a.eps), rb = 1.f / sqrtf(sb / D + a.eps);
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        float wa[V], wb[V];
        load_v<float, V>(a.pair_wa + at(i), at(i) < D, wa);
        load_v<float, V>(a.pair_wb + at(i), at(i) < D, wb);
#pragma unroll
        for (int e = 0; e < V; ++e) {  // (of the two products one is rounded, in rows of up to 1024 that four does not divide the first: see squares)
          const float u = add[i][e] * ra, v = vb[i][e] * rb;
          add[i][e] = 0.5f * (NT == 256 && V == 1 ? fmaf(v, wb[e], product(u, wa[e])) : fmaf(u, wa[e], product(v, wb[e])));
        }
      }
    } else if (a.post_w) {
      const float sa = block_sum<NT>(squares<VPT, V, V == 1 ? 0 : 1>(add), red);
      const float ra = 1.f / sqrtf(sa / D + a.eps);
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        float w[V];
        if constexpr (CONV > 0 && VPT == 1) {
#pragma unroll
          for (int e = 0; e < V; ++e) w[e] = pw[e];
        } else {
          load_v<float, V>(a.post_w + at(i), at(i) < D, w);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) add[i][e] *= ra * (w[e] + a.norm_offset);
      }
    }
  }
  if (a.y_t) {
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < a.n_slots; ++k) {
      const float w = s_w[k];
      const T* y = reinterpret_cast<const T*>(a.y_t) + (size_t)s_pos[k] * a.y_ld;
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        float v[V];
        load_v<T, V>(y + at(i), at(i) < D, v);
#pragma unroll
        for (int e = 0; e < V; ++e) add[i][e] += w * v[e];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
#pragma unroll
    for (int e = 0; e < V; ++e) x[i][e] += add[i][e];
    if (!a.only_want && at(i) < D) store_v<float, V>(a.x + (size_t)row * D + at(i), x[i]);
  }
  if (!a.norm_w) return;
  const float ss = block_sum<NT>(squares<VPT, V>(x), red);
  const float r = 1.f / sqrtf(ss / D + a.eps);
  T* h = reinterpret_cast<T*>(a.h_t) + (size_t)hrow * a.h_ld;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if (at(i) >= D) continue;
    float w[V];
    if constexpr (CONV > 0 && VPT == 1) {
#pragma unroll
      for (int e = 0; e < V; ++e) w[e] = nw[e];
    } else {
      if constexpr (CONV > 0) cv.load(a, sq, at(i));
      load_v<float, V>(a.norm_w + at(i), true, w);
    }
#pragma unroll
    for (int e = 0; e < V; ++e) w[e] = x[i][e] * r * (w[e] + a.norm_offset);
    if constexpr (CONV > 0) cv.template run<T, PUB>(a, row, sq.pos0, at(i), w);
    else if (a.h_f) store_v<float, V>(a.h_f + (size_t)row * D + at(i), w);
    else store_h<T, V, PUB>(h + at(i), w);
  }
}

// The same for a sequence's only token in front of a sandwich layer's sublayer, four taps: no branch between the loads, which are buffer loads of ranges that are
// empty where there is nothing to read, so that all of them are on their way at once (behind a branch the compiler waits for each).  What one compute
// unit takes in bounds it then (a row of 2048: 144 - 184 KiB, of 7168: 350), so SPLIT workgroups share a row: each adds up all of it, for the
// norms, and makes a part of what follows.  (The new residual goes to x_next: the others still read the old one.)  A launch for one row of 2048 without /
// with blends 5.8 / about 8 us as before -> 4.8 / 6.3 without branches -> 4.6 / 5.4 by two workgroups (by four 4.6 / 5.3); four rows of 7168 11.0 / 12.0 ->
// 10.4 / 15 -> 9.0 / 12 by two, 8.3 / 11.0 by four, 8.1 / 10.8 by eight.  PARTS: the most parts of the sum; MIX: blends.
static inline bool sandwich_fits(const JoinArgs& a) {
  return a.conv.w && a.conv.taps == 4 && (!a.conv.mu || a.conv.n_mix <= 5) && !(a.width & 3) && a.width <= 8192 && a.parts_a <= (a.width > 4096 ? 4 : 8) && !a.mix_b && !a.y_t &&
         a.norm_w && !a.only_want && a.x_next;
}
DEV __amdgpu_buffer_rsrc_t range(const void* p, bool there, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, there ? bytes : 0, 0x00020000);
}
DEV f32x4 load4(const __amdgpu_buffer_rsrc_t& r, int at) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
}
DEV void store4(const __amdgpu_buffer_rsrc_t& r, int at, const f32x4& v) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, at, 0, 0);
}
template <bool PUB>
DEV void store_out(const __amdgpu_buffer_rsrc_t& r, int at, const f32x4& v, bf16) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, to_four<bf16>(v)), r, at * 2, 0, PUB ? 16 /* sc1 */ : 0);
}
template <bool PUB>
DEV void store_out(const __amdgpu_buffer_rsrc_t& r, int at, const f32x4& v, float) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, at * 4, 0, PUB ? 16 : 0);
}
template <typename T, int NT, int VPT, int PARTS, int SPLIT, bool MIX, bool PUB>
DEV void sandwich_row(const JoinArgs& a, const SeqDesc* seqs, int block, float (&red)[NT / 64]) {
  enum { TAPS = 4, KEPT = 3, MAX_MIX = 5 };
  const ConvArgs& cv = a.conv;
  const int tid = threadIdx.x, D = a.width, bytes = D * 4, row = block / SPLIT, per = (D / 4 + SPLIT - 1) / SPLIT, first = block % SPLIT * per;
  auto at = [&](int i) { return 4 * (tid + i * NT); };
  auto own = [&](int i) { return (unsigned)(tid + i * NT - first) < (unsigned)per ? at(i) : 1 << 20; };  // behind every range: not this workgroup's
  const SeqDesc sq = seq_late(seqs + row);
  f32x4 x[VPT], q[VPT][PARTS], pw[VPT], nw[VPT], w[VPT][TAPS], mu[VPT][MAX_MIX], old[VPT][KEPT], prev[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (a.embed) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      float e[4];
      load_v<bf16, 4>(reinterpret_cast<const bf16*>(a.embed) + (size_t)a.p.tokens[row] * D + at(i), at(i) < D, e);
      x[i] = f32x4{e[0], e[1], e[2], e[3]};
    }
  }
  const auto rx = range(a.x_next + (size_t)row * D, true, bytes);
  const auto rx_in = range(a.x + (size_t)row * D, !a.embed, bytes), rp = range(a.post_w, a.post_w, bytes), rn = range(a.norm_w, true, bytes), rw = range(cv.w, true, bytes * TAPS);
  f32x4 xs[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    xs[i] = load4(rx_in, at(i) * 4);
#pragma unroll
    for (int u = 0; u < PARTS; ++u) q[i][u] = load4(range(a.mix_a + (size_t)row * a.mix_ld + u * a.mix_stride, a.mix_a && u < max(a.parts_a, 1), bytes), at(i) * 4);
    pw[i] = load4(rp, at(i) * 4);
    nw[i] = load4(rn, own(i) * 4);
#pragma unroll
    for (int e = 0; e < TAPS; ++e) w[i][e] = load4(rw, own(i) * 4 * TAPS + e * 16);
  }
  auto load_mu = [&]() {
    if constexpr (MIX) {
#pragma unroll
      for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int k = 0; k < MAX_MIX; ++k) mu[i][k] = load4(range(cv.mu + (size_t)k * D, k < cv.n_mix, bytes), own(i) * 4);
    }
  };
  if constexpr (VPT == 1) load_mu();
  // (the descriptor came first)
  char* state = reinterpret_cast<char*>(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned long long)sq.state >> 32)) << 32) |
                                        (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned long long)sq.state));
  const int pos0 = __builtin_amdgcn_readfirstlane(sq.pos0), flip = __builtin_amdgcn_readfirstlane(sq.flip);
  char* in = state + cv.off_in;
  const size_t half = (size_t)KEPT * bytes;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
#pragma unroll
    for (int t = 0; t < KEPT; ++t) old[i][t] = load4(range(in + flip * half + (size_t)t * bytes, pos0 - KEPT + t >= 0, bytes), own(i) * 4);
    if constexpr (MIX) prev[i] = load4(range(state + cv.off_prev + (size_t)flip * bytes, pos0 > 0, bytes), own(i) * 4);
  }
  f32x4 sum[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
#pragma unroll
    for (int n = 1; n < PARTS; n *= 2)
#pragma unroll
      for (int u = 0; u + n < PARTS; u += 2 * n) q[i][u] += q[i][u + n];
    sum[i] = q[i][0];
  }
  const float sa = block_sum<NT>(squares<VPT, 4>(sum), red);
  const float ra = 1.f / sqrtf(sa / D + a.eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float add = a.post_w ? sum[i][e] * (ra * (pw[i][e] + a.norm_offset)) : sum[i][e];
      x[i][e] = (a.embed ? x[i][e] : xs[i][e]) + add;
    }
    store4(rx, own(i) * 4, x[i]);
  }
  const float ss = block_sum<NT>(squares<VPT, 4>(x), red);
  if constexpr (VPT > 1) load_mu();  // (for the registers)
  const float r = 1.f / sqrtf(ss / D + a.eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    f32x4 h, y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = x[i][e] * r * (nw[i][e] + a.norm_offset);
      float z = 0.f;
#pragma unroll
      for (int t = 0; t < TAPS; ++t) z += (t == KEPT ? h[e] : old[i][t < KEPT ? t : 0][e]) * w[i][e][t];
      y[e] = z + h[e];
    }
    const size_t other = (flip ^ 1) * half;
#pragma unroll
    for (int t = 1; t < KEPT; ++t) store4(range(in + other + (size_t)(t - 1) * bytes, true, bytes), own(i) * 4, old[i][t]);
    store4(range(in + other + (size_t)(KEPT - 1) * bytes, true, bytes), own(i) * 4, h);
    auto out = [&](int k) { return range(reinterpret_cast<T*>(cv.out_t) + (size_t)row * cv.ld + (size_t)k * cv.mix_stride, !MIX || k < cv.n_mix, D * (int)sizeof(T)); };
    if constexpr (MIX) {
      store4(range(state + cv.off_prev + (size_t)(flip ^ 1) * bytes, true, bytes), own(i) * 4, y);
#pragma unroll
      for (int k = 0; k < MAX_MIX; ++k) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = y[e] + (prev[i][e] - y[e]) * mu[i][k][e];
        store_out<PUB>(out(k), own(i), v, T{});
      }
    } else {
      store_out<PUB>(out(0), own(i), y, T{});
    }
  }
}
