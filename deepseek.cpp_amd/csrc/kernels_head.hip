// kernels_head.hip -- MHA of one token (src/infer.cpp:943-1049, 728-762): per head, the rows of wkv_b (and of wq_b: head_attn_latent_kernel), RoPE, the cache
// entries and attention in one launch, with everything that does not depend on anything requested at once.
//
// head_attn_kernel (kernels_gemv.hip) does the same as a chain: latents, rows, query, rope's inputs, cache write, keys, each a trip of 0.7 - 1 us behind a
// barrier that waits for stores.  Of those only the latents -> rows -> current key and value depend on each other.  So: the latents, the query, the
// rope's inputs and the head's rows are requested at entry, keys and values (of up to 256 positions) behind the first barrier; the current position's
// key and value go from LDS into the scores and the mix, rounded as the cache rounds them, and to the cache at the very end; barriers are for LDS
// only.  Values, sums and their orders are head_attn_kernel's: the same bits.  Without a query latent the output leaves in 32 bits and wo quantises it (8 blocks for
// V2-Lite: cheaper in each of its workgroups than a hand-over between heads here).
// Bound by latency: 16 workgroups.  V2-Lite, medians over a token's launches, us: Q2_K at 62 positions 13.4 -> 7.4, F8E5M2 at 25 12.6 -> 9.3 (its 131 KB of rows are 2.7 us for the one compute unit); a token 1130 -> 985, 1602 -> 1505.
#include "dsk_internal.h"
#include "gemv_device.h"
#include "head_rows.h"

namespace {

// what attention needs of a head's shape, and where
struct HeadShape { int H, h, hd, vd, nope, rope, is_v3; uint16_t *kcache, *vcache; int kv_pos, kv_len; };

// Keys and values on their way: 16 lanes a position, positions 4 wave .. + 3 of every 64; thread (g, i4) the values of positions g, g + TG, ...  Buffer loads: one
// lane offset each for keys and values, a step's distance added to it, and zeros without traffic behind the context's end (head_rows.h).
template <int VN>
struct HeadKV {
  rsrc_t KB, VB;
  u32 krow, vrow, koff, voff;
  int grp, sl, TG, g, i4;
  ad::f16x4 k[4][3], v[VN];
};
template <int VN>
DEV void head_keys(const HeadShape& S, HeadKV<VN>& R, int t0) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (!head_step_there(t0 + u * HEAD_KEY_STEP, S.kv_len)) break;
    const u32 at = R.koff + (u32)(t0 + u * HEAD_KEY_STEP) * R.krow;
#pragma unroll
    for (int j = 0; j < 3; ++j) R.k[u][j] = __builtin_bit_cast(ad::f16x4, __builtin_amdgcn_raw_buffer_load_b64(R.KB, (int)(at + 128 * j), 0, 0));
  }
}
template <int VN>
DEV void head_places(const HeadShape& S, HeadKV<VN>& R, int tid, int wave, int lane) {
  const int tpp = S.vd >> 2;
  R.grp = lane >> 4; R.sl = lane & 15;
  R.TG = 1024 / tpp; R.g = tid / tpp; R.i4 = tid - R.g * tpp;
  R.krow = head_row_bytes(S.H, S.hd); R.vrow = head_row_bytes(S.H, S.vd);
  R.KB = __builtin_amdgcn_make_buffer_rsrc(S.kcache, 0, (int)(S.kv_len * R.krow), 0x00020000);
  R.VB = __builtin_amdgcn_make_buffer_rsrc(S.vcache, 0, (int)(S.kv_len * R.vrow), 0x00020000);
  R.koff = head_key_at(wave * 4 + R.grp, R.sl, S.H, S.h, S.hd);
  R.voff = head_value_at(R.g, R.i4, R.TG, S.H, S.h, S.vd);
}
// values of the group's position g + first, where any group has one
template <int VN>
DEV void head_value(const HeadShape& S, const HeadKV<VN>& R, int first, ad::f16x4& v) {
  if (head_step_there(first, S.kv_len)) v = __builtin_bit_cast(ad::f16x4, __builtin_amdgcn_raw_buffer_load_b64(R.VB, (int)(R.voff + (u32)first * R.vrow), 0, 0));
}
template <int VN>
DEV void head_values(const HeadShape& S, HeadKV<VN>& R) {
#pragma unroll
  for (int j = 0; j < VN; ++j) head_value(S, R, j * R.TG, R.v[j]);
}
// rotation of the sink keys by one position, in f16 (src/infer.cpp:1008-1020), in front of the keys' requests
DEV void head_sinks(const HeadShape& S, const StepParams* sp, int kv_sink, int tid) {
  const int half = S.rope >> 1;
  for (int r = 0; r < kv_sink; ++r) {
    uint16_t* kh = S.kcache + ((size_t)r * S.H + S.h) * S.hd + S.nope;
    float re = 0.f, im = 0.f;
    if (tid < half) ad::rope_rot(ad::h2f(kh[2 * tid]), ad::h2f(kh[2 * tid + 1]), sp->rope_cs1[2 * tid], sp->rope_cs1[2 * tid + 1], re, im);
    __syncthreads();
    if (tid < half) {
      kh[S.is_v3 ? 2 * tid : tid] = ad::f2h(re);
      kh[S.is_v3 ? 2 * tid + 1 : tid + half] = ad::f2h(im);
    }
    __syncthreads();
  }
}
// Scores, softmax and mix (src/infer.cpp:1022-1045) in attn_mha_body's order; returns output tid of the head (tid < vd).  qv: the lane's 12 values of the rotated query;
// kvb_s: the head's rows of wkv_b; kr_s: this position's rotated key part, as the cache will hold it.  part: 4096 floats, att: kv_len.
template <int VN>
DEV float head_attend(const HeadShape& S, HeadKV<VN>& R, const float (&qv)[3][4], const float* kvb_s, const uint16_t* kr_s, float* att, float* part, int tid, int wave, int lane,
                      bool timed, unsigned long long (&stamps)[2]) {
  constexpr int NW = 16, NT = 1024;
  const int hd = S.hd, vd = S.vd, nope = S.nope, kv_len = S.kv_len, kv_pos = S.kv_pos, grp = R.grp, sl = R.sl, TG = R.TG, g = R.g, i4 = R.i4;
  {
    const bool in2 = 128 + sl * 4 < hd, in1 = 64 + sl * 4 < hd, in0 = sl * 4 < hd;
    const float inv = sqrtf((float)hd);
    const int pw = wave * 4 + grp;
    for (int t0 = 0; t0 < kv_len; t0 += 256) {
      if ((kv_pos & 63) == pw && kv_pos >= t0 && kv_pos < t0 + 256) {  // this position's key is not in the cache yet
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int d0 = min(64 * j + sl * 4, hd - 4);
          const f32x4 x = *reinterpret_cast<const f32x4*>(kvb_s + min(d0, nope - 4));
          const ad::f16x4 y = *reinterpret_cast<const ad::f16x4*>(kr_s + max(d0 - nope, 0));
          const ad::f16x4 c = d0 < nope ? ad::f16x4{(_Float16)x.x, (_Float16)x.y, (_Float16)x.z, (_Float16)x.w} : y;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (u == (kv_pos - t0) >> 6) R.k[u][j] = c;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * 64 + pw;
        if (t0 + u * 64 >= kv_len) break;
        float p = 0.f;
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (j == 0 ? in0 : j == 1 ? in1 : in2) {
            p = fmaf(qv[j][0], (float)R.k[u][j].x, p);
            p = fmaf(qv[j][1], (float)R.k[u][j].y, p);
            p = fmaf(qv[j][2], (float)R.k[u][j].z, p);
            p = fmaf(qv[j][3], (float)R.k[u][j].w, p);
          }
        p = ad::row16_sum(p);
        if (sl == 0 && t < kv_len) att[t] = p / inv;
      }
      if (t0 + 256 < kv_len) head_keys(S, R, t0 + 256);
    }
  }
  lds_barrier();
  if (timed) stamps[0] = wall_clock64();
  // ---- softmax (src/infer.cpp:472-487): a wave's trees over 64 positions, the waves' sums in order ----
  if (kv_len <= 64) {
    if (wave == 0) {
      const float a0 = lane < kv_len ? att[lane] : -INFINITY;
      const float mx = ad::wave_max_dpp(a0);
      const float e = lane < kv_len ? expf(a0 - mx) : 0.f;
      const float sum = ad::wave_sum_dpp(e);
      if (lane < kv_len) att[lane] = e / sum;
    }
  } else {
    float mx = -INFINITY;
    for (int t = tid; t < kv_len; t += NT) mx = fmaxf(mx, att[t]);
    mx = ad::wave_max_dpp(mx);
    if (lane == 0) part[wave] = mx;
    lds_barrier();
    mx = part[0];
    for (int i = 1; i < NW; ++i) mx = fmaxf(mx, part[i]);
    float sum = 0.f;
    for (int t = tid; t < kv_len; t += NT) {
      const float e = expf(att[t] - mx);
      att[t] = e;
      sum += e;
    }
    sum = ad::wave_sum_dpp(sum);
    if (lane == 0) part[NW + wave] = sum;
    lds_barrier();
    float total = 0.f;
    for (int i = 0; i < NW; ++i) total += part[NW + i];
    for (int t = tid; t < kv_len; t += NT) att[t] = att[t] / total;
  }
  lds_barrier();
  // ---- values: every thread its positions in order, then the groups in order ----
  auto value_here = [&]() {  // this position's, as the cache will hold it
    const f32x4 x = *reinterpret_cast<const f32x4*>(kvb_s + nope + i4 * 4);
    return ad::f16x4{(_Float16)x.x, (_Float16)x.y, (_Float16)x.z, (_Float16)x.w};
  };
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  auto mix = [&](int t, ad::f16x4 y) {
    if (t == kv_pos) y = value_here();
    const float w = att[t];
    acc[0] = fmaf(w, (float)y.x, acc[0]);
    acc[1] = fmaf(w, (float)y.y, acc[1]);
    acc[2] = fmaf(w, (float)y.z, acc[2]);
    acc[3] = fmaf(w, (float)y.w, acc[3]);
  };
  if (g < TG) {
#pragma unroll
    for (int j = 0; j < VN; ++j)
      if (g + j * TG < kv_len) mix(g + j * TG, R.v[j]);
    for (int first = VN * TG; first < kv_len; first += 4 * TG) {  // (uniform)
      ad::f16x4 y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) head_value(S, R, first + j * TG, y[j]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (g + first + j * TG < kv_len) mix(g + first + j * TG, y[j]);
    }
    *reinterpret_cast<f32x4*>(part + (size_t)g * vd + i4 * 4) = f32x4{acc[0], acc[1], acc[2], acc[3]};
  }
  lds_barrier();
  if (timed) stamps[1] = wall_clock64();
  float o = 0.f;
  if (tid < vd) {
    const int ng = min(TG, kv_len);  // (the others' sums are zeros)
    for (int g0 = 0; g0 < ng; g0 += 8) {
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = part[min(g0 + i, ng - 1) * vd + tid];
#pragma unroll
      for (int i = 0; i < 8; ++i) o += g0 + i < ng ? y[i] : 0.f;
    }
  }
  return o;
}
// the cache entries (src/infer.cpp:985-1005), by the upper half of the workgroup
DEV void head_cache(const HeadShape& S, const float* kvb_s, const uint16_t* kr_s, int tid) {
  uint16_t* kc = S.kcache + ((size_t)S.kv_pos * S.H + S.h) * S.hd;
  uint16_t* vc = S.vcache + ((size_t)S.kv_pos * S.H + S.h) * S.vd;
  const int i = tid - 512;
  if (i < 0) return;
  if (i < S.nope) kc[i] = ad::f2h(kvb_s[i]);
  if (i < S.rope) kc[S.nope + i] = kr_s[i];
  if (i < S.vd) vc[i] = ad::f2h(kvb_s[S.nope + i]);
}

}  // namespace

// RS x ROUNDS row sets of a wave, two rounds on their way
template <int QT, int RS, int ROUNDS>
__global__ __launch_bounds__(1024) void head_attn_short_kernel(const StepParams* __restrict__ sp, const float* __restrict__ kv_a, const float* __restrict__ norm_w,
                                                              const float* __restrict__ q, uint16_t* kcache, uint16_t* vcache, int H, int hv, const HeadShortArgs A) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float scratch[16];
  __shared__ __attribute__((aligned(16))) float q_s[256];
  __shared__ __attribute__((aligned(16))) float kvb_s[512];
  __shared__ __attribute__((aligned(16))) uint16_t kr_s[128];  // this position's rotated key part, as the cache holds it
  __shared__ __attribute__((aligned(16))) float part[4096];
  constexpr bool KQ = QT == DSK_QUANT_Q2_K || QT == DSK_QUANT_Q3_K;
  constexpr int NW = 16, NT = 1024, VN = RS == 4 ? 2 : QT == DSK_QUANT_Q3_K ? 4 : 8;  // (VN: values of a thread requested early; as many as the registers hold)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, h = blockIdx.x;
  if (h >= H) {  // prefetch workgroups (HeadAttnArgs::pf_wgs)
    tail_prefetch(A.pf_p, A.pf_n, tid, NT);
    return;
  }
  const unsigned long long t_entry = A.timeline ? wall_clock64() : 0ull;
  unsigned long long t_staged = 0, t_rows = 0, stamps[2] = {0, 0};
  const int hd = hv & 0xffff, vd = hv >> 16, nope = A.nope, rope = A.rope, n = A.lora, nrows = nope + vd, half = rope >> 1;
  uint8_t* act = smem;
  float* att = reinterpret_cast<float*>(smem + A.lds_kv);
  // ---- requests.  What few waves need comes first: an older load in a branch does not blur what the compiler knows of the ones behind it ----
  f32x4 lt, lw;
  float2 qp, kp, cs;
  float qn;
  const bool latent_wave = wave < (n + 255) >> 8, rope_wave = wave == NW - 1, q_wave = wave >= 8 && wave < 8 + ((nope + 63) >> 6);
  const bool latent = tid * 4 < n;  // (n is a multiple of 256 for K-quants; float rows may end inside a wave)
  if (rope_wave) {
    const int i = min(lane, half - 1);
    qp = *reinterpret_cast<const float2*>(q + (size_t)h * hd + nope + 2 * i);
    kp = *reinterpret_cast<const float2*>(kv_a + n + 2 * i);
    cs = *reinterpret_cast<const float2*>(sp->rope_cs + 2 * i);
  }
  if (q_wave) qn = q[(size_t)h * hd + min(tid - 512, nope - 1)];
  if (latent_wave) {
    const int i = latent ? tid * 4 : n - 4;
    lt = *reinterpret_cast<const f32x4*>(kv_a + i);
    lw = *reinterpret_cast<const f32x4*>(norm_w + i);
  }
  const int lpr_log2 = A.lkv_log2, RPW = 64 >> lpr_log2, rloc = lane >> lpr_log2, sub = lane & ((1 << lpr_log2) - 1);
  const int base = wave * RPW + rloc, sets_stride = NW * RPW;
  WPtr P;
  P.present = true; P.qs = A.qs; P.sc = A.sc; P.hm = A.hm; P.dm = A.dm; P.scale = A.scale; P.qs2 = P.sc2 = P.hm2 = P.dm2 = nullptr; P.scale2 = nullptr;
  struct Rows {
    ChunkKQ<KQ ? QT : DSK_QUANT_Q2_K, RS, 1, false> k;
    u32x4 w[RS];
    float sv[RS];
  };
  auto request_rows = [&](Rows& R, int set0) {
    int row[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) row[r] = h * nrows + min(base + (set0 + r) * sets_stride, nrows - 1);
    if constexpr (KQ) {
      int rowblk[RS];
#pragma unroll
      for (int r = 0; r < RS; ++r) rowblk[r] = row[r] * (n >> 8) + (sub >> 2);
      load_chunk_kq<QT, RS, 1, false>(R.k, kq_rsrc<QT, false>(P), 1, 1 << lpr_log2, sub, lpr_log2, sub & 3, rowblk, 0);
    } else {  // (one exact column step: the item of a lane is its place in the row)
      constexpr int EPI = FTraits<KQ ? DSK_QUANT_F16 : QT>::EPI, ESZ = 16 / EPI;
      const int sc_col = A.sh1 >= 0 ? sub * EPI >> A.sh1 : sub * EPI / A.b1;
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        R.w[r] = ldg_nt(reinterpret_cast<const u32x4*>(P.qs + (size_t)row[r] * n * ESZ + sub * 16));
        R.sv[r] = QT == DSK_QUANT_F8E5M2 && P.scale ? P.scale[(A.sh0 >= 0 ? row[r] >> A.sh0 : row[r] / A.b0) * A.sc_cols + sc_col] : 1.0f;
      }
    }
  };
  Rows ra, rb;
  request_rows(ra, 0);
  request_rows(rb, RS);
  const int kv_pos = sp->kv_pos, kv_len = sp->kv_len, kv_sink = sp->kv_sink;
  // ---- rmsnorm of the latent (src/infer.cpp:950, 601-611): the sum of squares in the order of the two forms of head_attn_kernel ----
  if (latent_wave) {
    float ss = 0.f;
    if constexpr (KQ) ss = fmaf(lt.x, lt.x, fmaf(lt.y, lt.y, fmaf(lt.z, lt.z, lt.w * lt.w)));
    else if (latent) {
      ss = fmaf(lt.x, lt.x, ss);
      ss = fmaf(lt.y, lt.y, ss);
      ss = fmaf(lt.z, lt.z, ss);
      ss = fmaf(lt.w, lt.w, ss);
    }
    ss = wave_sum(ss);
    if (lane == 0) scratch[wave] = ss;
  } else if (lane == 0) {
    scratch[wave] = 0.f;
  }
  lds_barrier();
  const HeadShape S{H, h, hd, vd, nope, rope, A.is_v3, kcache, vcache, kv_pos, kv_len};
  HeadKV<VN> R;
  if (kv_sink > 0) head_sinks(S, sp, kv_sink, tid);
  head_places(S, R, tid, wave, lane);
  head_keys(S, R, 0);
  head_values(S, R);
  // ---- the latent staged; the query and this position's key part rotated ----
  if (latent_wave) {
    if constexpr (KQ) {
      float total = 0.f;
      for (int i = 0; i < n >> 8; ++i) total += scratch[i];
      const float scale = 1.0f / sqrtf(total / (float)n + A.eps);
      const float y[4] = {lt.x * scale * lw.x, lt.y * scale * lw.y, lt.z * scale * lw.z, lt.w * scale * lw.w};
      q8k_block_lds<QT == DSK_QUANT_Q2_K>(y, lane, act + (size_t)wave * 4 * ITEM_LDS);
    } else {
      const float scale = 1.0f / sqrtf(scratch_total<NW>(scratch) / (float)n + A.eps);
      constexpr int EPI = FTraits<KQ ? DSK_QUANT_F16 : QT>::EPI;
      if (latent) reinterpret_cast<f32x4*>(act)[quad_place<EPI>(tid, n / EPI)] = lt * scale * lw;
    }
  }
  if (rope_wave) {
    if (lane < half) {
      float re, im;
      const int a = A.is_v3 ? 2 * lane : lane, b = A.is_v3 ? 2 * lane + 1 : lane + half;
      ad::rope_rot(qp.x, qp.y, cs.x, cs.y, re, im);
      q_s[nope + a] = re;
      q_s[nope + b] = im;
      ad::rope_rot(kp.x, kp.y, cs.x, cs.y, re, im);
      kr_s[a] = ad::f2h(re);
      kr_s[b] = ad::f2h(im);
    }
  }
  if (q_wave && tid - 512 < nope) q_s[tid - 512] = qn;
  lds_barrier();
  if (A.timeline) t_staged = wall_clock64();
  if constexpr (KQ) {
    if (A.tap_qs && h == 0) dump_staged_q8_inline<QT == DSK_QUANT_Q2_K>(act, n, A.tap_qs, A.tap_d, tid, NT);
  }
  // ---- the head's rows of wkv_b ----
  f32x4 xa4[KQ ? 1 : FTraits<KQ ? DSK_QUANT_F16 : QT>::EPI / 4];
  if constexpr (!KQ) {
    constexpr int EPI = FTraits<KQ ? DSK_QUANT_F16 : QT>::EPI;
#pragma unroll
    for (int i = 0; i < EPI / 4; ++i) xa4[i] = reinterpret_cast<const f32x4*>(act)[i * (n / EPI) + sub];  // (quad_place)
  }
  auto finish_rows = [&](const Rows& R, int set0) {
    float acc[RS], dummy[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) acc[r] = 0.f;
    if constexpr (KQ) compute_chunk_kq<QT, RS, 1, false>(R.k, 1, 1 << lpr_log2, sub, lpr_log2, sub & 3, 0, act + sub * ITEM_LDS, acc, dummy);
    else {
#pragma unroll
      for (int r = 0; r < RS; ++r) acc[r] = fmaf(fitem<QT>(R.w[r], reinterpret_cast<const float*>(xa4), 0.f), R.sv[r], 0.f);
    }
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      const float o = lanes_sum(acc[r], lpr_log2);
      if (sub == 0 && base + (set0 + r) * sets_stride < nrows) kvb_s[base + (set0 + r) * sets_stride] = o;
    }
  };
#pragma unroll
  for (int r = 0; r < ROUNDS; r += 2) {
    finish_rows(ra, r * RS);
    if (r + 2 < ROUNDS) request_rows(ra, (r + 2) * RS);
    finish_rows(rb, (r + 1) * RS);
    if (r + 2 < ROUNDS) request_rows(rb, (r + 3) * RS);
  }
  lds_barrier();
  if (A.timeline) t_rows = wall_clock64();
  float qv[3][4];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(q_s + min(64 * j + R.sl * 4, hd - 4));
    const bool in = 64 * j + R.sl * 4 < hd;
    qv[j][0] = in ? t.x : 0.f; qv[j][1] = in ? t.y : 0.f; qv[j][2] = in ? t.z : 0.f; qv[j][3] = in ? t.w : 0.f;
  }
  const float o = head_attend(S, R, qv, kvb_s, kr_s, att, part, tid, wave, lane, A.timeline != nullptr, stamps);
  if (tid < vd) A.out[(size_t)h * vd + tid] = o;
  head_cache(S, kvb_s, kr_s, tid);
  if (A.timeline && tid == 0 && blockIdx.x < DSK_TL_WGS) {
    unsigned long long* tl = A.timeline + (size_t)blockIdx.x * 8;
    tl[0] = t_entry; tl[1] = t_staged; tl[2] = t_rows; tl[3] = stamps[0]; tl[4] = stamps[1]; tl[5] = wall_clock64();
  }
}

// ------------------------------------------------------------------------------------------------------------
// The same behind a query latent, for DeepSeek-V3's heads in Q2_K (192 rows of 1536, 256 of 512, 8 lanes a row): the two latents normed and quantised in one pass, then
// wkv_b's and wq_b's rows as in head_attn_kernel, whose order and bits these are.  A compute unit returns loads in order and holds ~50 KB of them: the first rows
// are requested at entry, the next behind the latents, keys and values behind those and under the multiplies.  The output is quantised here, by the last of
// a block's heads (64 blocks: dearer in each of wo's workgroups).  128 heads, us a launch: at 20 positions 16.5 -> 12.3, at 200 20.2 -> 14.8; five of V3's blocks 487 -> 465 a
// token.
// ------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void head_attn_latent_kernel(const StepParams* __restrict__ sp, const float* __restrict__ q_a, const float* __restrict__ kv_a,
                                                               const float* __restrict__ q_norm, const float* __restrict__ kv_norm, uint16_t* kcache, uint16_t* vcache,
                                                               const HeadAttnArgs A) {
  constexpr int QT = DSK_QUANT_Q2_K, NQ = 1536, NKV = 512, NBQ = NQ / 256, NBKV = NKV / 256, HD = 192, NOPE = 128, VN = 8;
  __shared__ __attribute__((aligned(16))) uint8_t act[(NQ + NKV) / 64 * ITEM_LDS];
  __shared__ float scratch[16];
  __shared__ __attribute__((aligned(16))) float q_s[HD];
  __shared__ __attribute__((aligned(16))) float kvb_s[256];
  __shared__ __attribute__((aligned(16))) float cs_s[64];
  __shared__ __attribute__((aligned(16))) uint16_t kr_s[64];
  __shared__ __attribute__((aligned(16))) float part[4096];
  __shared__ int last_flag;
  extern __shared__ __attribute__((aligned(16))) float att[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, h = blockIdx.x;
  const int H = A.a.n_heads;
  if (h >= H) {  // prefetch workgroups (HeadAttnArgs::pf_wgs)
    tail_prefetch(A.pf_p, A.pf_n, tid, 1024);
    return;
  }
  unsigned long long* const tl = A.timeline && h < DSK_TL_WGS ? A.timeline + (size_t)h * 8 : nullptr;
  const unsigned long long t_entry = tl ? wall_clock64() : 0ull;
  unsigned long long t_staged = 0, t_rows = 0, stamps[2] = {0, 0};
  uint8_t *act_q = act, *act_kv = act + NQ / 64 * ITEM_LDS;
  // ---- requests at entry: the rope's inputs (one wave), the latents (a block each of eight waves), the head's rows of wkv_b ----
  float2 kp, cs;
  f32x4 lt, lw;
  if (wave == 15) {
    kp = *reinterpret_cast<const float2*>(kv_a + NKV + 2 * (lane & 31));
    cs = *reinterpret_cast<const float2*>(sp->rope_cs + 2 * (lane & 31));
  }
  const bool is_q = wave < NBQ, mine = wave < NBQ + NBKV;
  if (mine) {
    lt = *reinterpret_cast<const f32x4*>((is_q ? q_a + wave * 256 : kv_a + (wave - NBQ) * 256) + lane * 4);
    lw = *reinterpret_cast<const f32x4*>((is_q ? q_norm + wave * 256 : kv_norm + (wave - NBQ) * 256) + lane * 4);
  }
  const int rloc = lane >> 3, sub = lane & 7, q = sub & 3, lr0 = wave * 8 + rloc, lr1 = 128 + lr0;
  WPtr P;
  P.present = true; P.hm = nullptr; P.scale = P.scale2 = nullptr; P.qs2 = P.sc2 = P.hm2 = P.dm2 = nullptr;
  P.qs = A.tkv.qs; P.sc = A.tkv.sc; P.dm = A.tkv.dm;
  const KQRsrc Bk = kq_rsrc<QT, false>(P);
  P.qs = A.tq.qs; P.sc = A.tq.sc; P.dm = A.tq.dm;
  const KQRsrc Bq = kq_rsrc<QT, false>(P);
  const int rbq0[1] = {(h * HD + lr0) * NBQ + (sub >> 2)}, rbq1[1] = {(h * HD + (lr1 < HD ? lr1 : HD - 1)) * NBQ + (sub >> 2)};
  const int rbk0[1] = {(h * 256 + lr0) * NBKV + (sub >> 2)}, rbk1[1] = {(h * 256 + lr1) * NBKV + (sub >> 2)};
  ChunkKQ<QT, 1, 3, false> cq0, cq1;
  ChunkKQ<QT, 1, 1, false> ck0, ck1;
  load_chunk_kq<QT, 1, 1, false>(ck0, Bk, 1, 8, sub, 3, q, rbk0, 0);
  load_chunk_kq<QT, 1, 1, false>(ck1, Bk, 1, 8, sub, 3, q, rbk1, 0);
  const int kv_pos = sp->kv_pos, kv_len = sp->kv_len, kv_sink = sp->kv_sink;
  // ---- both latents normed and quantised (src/infer.cpp:946-974, quant.cpp:616-653); this position's key part rotated ----
  if (mine) {
    float ss = fmaf(lt.x, lt.x, fmaf(lt.y, lt.y, fmaf(lt.z, lt.z, lt.w * lt.w)));
    ss = wave_sum(ss);
    if (lane == 0) scratch[wave] = ss;
  }
  lds_barrier();
  if (mine) {
    float total = 0.f;
    if (is_q) for (int i = 0; i < NBQ; ++i) total += scratch[i];
    else for (int i = NBQ; i < NBQ + NBKV; ++i) total += scratch[i];
    const float scale = 1.0f / sqrtf(total / (float)(is_q ? NQ : NKV) + (is_q ? A.tq.eps : A.tkv.eps));
    const float y[4] = {lt.x * scale * lw.x, lt.y * scale * lw.y, lt.z * scale * lw.z, lt.w * scale * lw.w};
    q8k_block_lds<LAY_Q2>(y, lane, act + (size_t)wave * 4 * ITEM_LDS);
  }
  const int is_v3 = A.a.is_v3;
  if (wave == 15 && lane < 32) {
    float re, im;
    ad::rope_rot(kp.x, kp.y, cs.x, cs.y, re, im);
    kr_s[is_v3 ? 2 * lane : lane] = ad::f2h(re);
    kr_s[is_v3 ? 2 * lane + 1 : lane + 32] = ad::f2h(im);
    cs_s[2 * lane] = cs.x;
    cs_s[2 * lane + 1] = cs.y;
  }
  lds_barrier();
  if (tl) t_staged = wall_clock64();
  if (A.tap_qs && h == 0) {  // parity tap
    dump_staged_q8_inline<LAY_Q2>(act_q, NQ, A.tap_qs, A.tap_d, tid, 1024);
    dump_staged_q8_inline<LAY_Q2>(act_kv, NKV, A.tap_qs + A.tap_stride, A.tap_d + (A.tap_stride >> 8), tid, 1024);
  }
  // ---- the rows, in the order of their arrival ----
  const HeadShape S{H, h, HD, 128, NOPE, 64, is_v3, kcache, vcache, kv_pos, kv_len};
  HeadKV<VN> R;
  load_chunk_kq<QT, 1, 3, false>(cq0, Bq, 3, 24, sub, 3, q, rbq0, 0);
  if (wave < 8) load_chunk_kq<QT, 1, 3, false>(cq1, Bq, 3, 24, sub, 3, q, rbq1, 0);
  if (kv_sink > 0) head_sinks(S, sp, kv_sink, tid);
  float acc[1] = {0.f}, dummy[1] = {0.f};
  compute_chunk_kq<QT, 1, 1, false>(ck0, 1, 8, sub, 3, q, 0, act_kv + sub * ITEM_LDS, acc, dummy);
  float v = lanes_sum(acc[0], 3);
  if (sub == 0) kvb_s[lr0] = v;
  acc[0] = 0.f;
  compute_chunk_kq<QT, 1, 1, false>(ck1, 1, 8, sub, 3, q, 0, act_kv + sub * ITEM_LDS, acc, dummy);
  v = lanes_sum(acc[0], 3);
  if (sub == 0) kvb_s[lr1] = v;
  acc[0] = 0.f;
  compute_chunk_kq<QT, 1, 3, false>(cq0, 3, 24, sub, 3, q, 0, act_q + sub * ITEM_LDS, acc, dummy);
  v = lanes_sum(acc[0], 3);
  if (sub == 0) q_s[lr0] = v;
  head_places(S, R, tid, wave, lane);  // (in the registers of the rows that are done)
  head_keys(S, R, 0);
  if (wave < 8) {
    acc[0] = 0.f;
    compute_chunk_kq<QT, 1, 3, false>(cq1, 3, 24, sub, 3, q, 0, act_q + sub * ITEM_LDS, acc, dummy);
    v = lanes_sum(acc[0], 3);
    if (sub == 0) q_s[lr1] = v;
  }
  head_values(S, R);
  lds_barrier();
  if (tl) t_rows = wall_clock64();
  // ---- the query's part of this lane, rotated where it is read (src/infer.cpp:648-685) ----
  float qv[3][4];
  const int sl = lane & 15;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(q_s + 64 * j + sl * 4);
    qv[j][0] = t.x; qv[j][1] = t.y; qv[j][2] = t.z; qv[j][3] = t.w;
  }
  if (is_v3) {  // pairs (2 p, 2 p + 1) stay where they are
    const f32x4 t = *reinterpret_cast<const f32x4*>(q_s + NOPE + sl * 4), c = *reinterpret_cast<const f32x4*>(cs_s + sl * 4);
    ad::rope_rot(t.x, t.y, c.x, c.y, qv[2][0], qv[2][1]);
    ad::rope_rot(t.z, t.w, c.z, c.w, qv[2][2], qv[2][3]);
  } else {  // real parts in front of imaginary ones
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int o = sl * 4 + i, p = o & 31;
      float re, im;
      ad::rope_rot(q_s[NOPE + 2 * p], q_s[NOPE + 2 * p + 1], cs_s[2 * p], cs_s[2 * p + 1], re, im);
      qv[2][i] = o < 32 ? re : im;
    }
  }
  const float o = head_attend(S, R, qv, kvb_s, kr_s, att, part, tid, wave, lane, tl != nullptr, stamps);
  ad::attn_out_q8(A.a, h, tid, o, &last_flag);
  head_cache(S, kvb_s, kr_s, tid);
  if (tl && tid == 0) { tl[0] = t_entry; tl[1] = t_staged; tl[2] = t_rows; tl[3] = stamps[0]; tl[4] = stamps[1]; tl[5] = wall_clock64(); }
}
// (the launches head_attn_latent_kernel is for: everything about the heads is compiled in)
bool head_latent_supported(const HeadAttnArgs& A, int max_kv) {
  return A.quant == DSK_QUANT_Q2_K && A.has_q && !A.tiled && A.lq_log2 == 3 && A.lkv_log2 == 3 && A.tq.n == 1536 && A.tkv.n == 512 && A.a.head_dim == 192 && A.a.nope == 128 &&
         A.a.rope == 64 && A.a.v_dim == 128 && A.a.lora == 512 && A.tq.act_mode == ACT_F32_NORM && A.tkv.act_mode == ACT_F32_NORM &&
         head_rows_fit(max_kv, A.a.n_heads, 192, 128);
}
int launch_head_latent(hipStream_t st, const HeadAttnArgs& A, const StepParams* sp, int max_kv) {
  const size_t lds = (size_t)max_kv * 4;
  if (lds > 120 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn: kv_len %d does not fit LDS", max_kv);
  auto k = head_attn_latent_kernel;
  if (lds > 40 * 1024) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(k, dim3(A.a.n_heads + (A.pf_wgs > 0 ? A.pf_wgs : 0)), dim3(1024), lds, st, sp, A.tq.a_f32, A.tkv.a_f32, A.tq.norm_w, A.tkv.norm_w, A.a.key_cache, A.a.value_cache, A);
  return DSK_OK;
}

// ---- host side ------------------------------------------------------------------------------------------
int head_short_plan(HeadShortArgs& S, const HeadAttnArgs& A, int max_kv) {
  const bool kq = A.quant == DSK_QUANT_Q2_K || A.quant == DSK_QUANT_Q3_K;
  const int epi = kq ? 64 : A.quant == DSK_QUANT_F16 ? 8 : 16, n = A.tkv.n, nope = A.a.nope, vd = A.a.v_dim, rope = A.a.rope, hd = A.a.head_dim;
  S.grid = 0;
  if (!head_rows_fit(max_kv, A.a.n_heads, hd, vd)) return DSK_OK;
  if (A.has_q || A.tiled || A.quant == DSK_QUANT_F32 || A.tkv.act_mode != ACT_F32_NORM) return DSK_OK;
  // rows of one column step, at most 16 row sets of the workgroup (floats: two rounds of 8; K-quants: one of 2); the norm one piece a thread, in the first 8 waves
  const int lpr = 1 << A.lkv_log2, sets = (nope + vd + 16 * (64 / lpr) - 1) / (16 * (64 / lpr));
  if (n % (kq ? 256 : epi) || n % 4 || n / epi != lpr || n > 2048 || sets > (kq ? 2 : 16)) return DSK_OK;
  if (hd != nope + rope || hd > 192 || hd % 4 || nope % 4 || nope < 4 || nope > 448 || rope < 2 || rope > 128 || rope % 2 || vd % 4 || vd < 4 || vd > 256 || nope + vd > 512 ||
      1024 / (vd / 4) * vd > 4096 || A.a.n_heads < 1) return DSK_OK;
  S.qs = A.tkv.qs; S.sc = A.tkv.sc; S.hm = A.tkv.hm; S.dm = A.tkv.dm; S.scale = A.tkv.scale;
  S.quant = A.quant; S.nope = nope; S.rope = rope; S.lora = n; S.is_v3 = A.a.is_v3; S.eps = A.tkv.eps; S.out = A.a.out; S.lkv_log2 = A.lkv_log2; S.lds_kv = A.lds_kv;
  S.b0 = A.b0 < 1 ? 1 : A.b0; S.b1 = A.b1 < 1 ? 1 : A.b1; S.H = A.a.n_heads; S.hd = hd; S.vd = vd; S.kv_a = A.a.kv_a; S.norm_w = A.tkv.norm_w; S.q = A.a.q;
  S.key_cache = A.a.key_cache; S.value_cache = A.a.value_cache; S.timeline = A.timeline;
  S.sets = sets;
  S.sh0 = (S.b0 & (S.b0 - 1)) ? -1 : __builtin_ctz(S.b0); S.sh1 = (S.b1 & (S.b1 - 1)) ? -1 : __builtin_ctz(S.b1); S.sc_cols = (n + S.b1 - 1) / S.b1;
  S.grid = A.a.n_heads;
  return DSK_OK;
}
int launch_head_short(hipStream_t st, const HeadShortArgs& S, const StepParams* sp, int max_kv) {
  const size_t lds = (size_t)S.lds_kv + (size_t)max_kv * 4;
  if (lds > 120 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn: kv_len %d does not fit LDS", max_kv);
  auto go = [&](auto k) {
    if (lds > 40 * 1024) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k, dim3(S.grid + (S.pf_wgs > 0 ? S.pf_wgs : 0)), dim3(1024), lds, st, sp, S.kv_a, S.norm_w, S.q, S.key_cache, S.value_cache, S.H, S.hd | S.vd << 16, S);
  };
  // (a set past the head's end costs what a real one does)
  auto floats = [&](auto qt) {
    constexpr int QT = decltype(qt)::value;
    if (S.sets > 8) go(head_attn_short_kernel<QT, 4, 4>);
    else if (S.sets > 4) go(head_attn_short_kernel<QT, 4, 2>);
    else if (S.sets > 2) go(head_attn_short_kernel<QT, 2, 2>);
    else go(head_attn_short_kernel<QT, 1, 2>);
  };
  switch (S.quant) {
    case DSK_QUANT_F16: floats(std::integral_constant<int, DSK_QUANT_F16>{}); break;
    case DSK_QUANT_F8E5M2: floats(std::integral_constant<int, DSK_QUANT_F8E5M2>{}); break;
    case DSK_QUANT_Q2_K: go(head_attn_short_kernel<DSK_QUANT_Q2_K, 1, 2>); break;
    default: go(head_attn_short_kernel<DSK_QUANT_Q3_K, 1, 2>); break;
  }
  return DSK_OK;
}
