// kernels_experts.hip -- the routed experts of one token in launches of their own, for models whose launches are bound by latency and not by
// bytes (one GPU, K-quant planes, F8E5M2 and F16; V2-Lite's shapes): the gate inside the first half, rows of x owned by workgroups in the second.
//
// Replaces, for the selected experts e_0..e_{K-1} of a token (src/infer.cpp:853-878, 899-903), the launches of the generic multi-task GEMV:
//     router rows' scores, rmsnorm(x) left behind                             router_scores_kernel
//     moe_gate, h_k = act(W1[e_k] xb) * (W3[e_k] xb), the shared expert's too  experts_up_kernel
//     o_k  = W2[e_k] h_k,  x += w_k * o_k  (k order),  x += shared_out        experts_down_kernel
// Nothing is handed over inside a launch.  Lanes per row, column steps, trees of lanes and the order of the combine are the generic launches', with
// float weights the one launch's (kernels_moe.hip moe_ffn_f_kernel): the same bits.
#include "dsk_internal.h"
#include "gemv_device.h"

namespace {

// Q8_K of FOUR 256-blocks by one wave, 16 lanes each, into item records (quantize_row_q8_K_ref, src/quant.cpp:616-653; the codes, scale and sums of
// q8k_block_lds).  Lane j of a block holds quads j, 16 + j, 32 + j, 48 + j of its 64.  What a wave spends on one block's maximum, division and
// exchanges serves four here: ~45 vector instructions a block instead of ~100.
template <int LAY>
DEV void q8k_four_blocks_lds(const f32x4 (&t)[4], int lane, uint8_t* blk) {
  const int j = lane & 15;
  float v[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { v[i][0] = t[i].x; v[i][1] = t[i].y; v[i][2] = t[i].z; v[i][3] = t[i].w; }
  float hi = 0.f, lo = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) { hi = fmaxf(hi, v[i][c]); lo = fminf(lo, v[i][c]); }
  hi = fmaxf(hi, dpp_f32<DPP_XOR1>(hi)); lo = fminf(lo, dpp_f32<DPP_XOR1>(lo));
  hi = fmaxf(hi, dpp_f32<DPP_XOR2>(hi)); lo = fminf(lo, dpp_f32<DPP_XOR2>(lo));
  hi = fmaxf(hi, dpp_f32<DPP_HALF_MIRROR>(hi)); lo = fminf(lo, dpp_f32<DPP_HALF_MIRROR>(lo));
  hi = fmaxf(hi, dpp_f32<DPP_MIRROR>(hi)); lo = fminf(lo, dpp_f32<DPP_MIRROR>(lo));
  // the signed value of the FIRST element of largest magnitude: the larger side's, and if both sides are as large the one of the lower index
  // (rare: looked for only then)
  float vmax = hi > -lo ? hi : lo;
  if (__any(hi == -lo && hi > 0.f)) {
    u32 key = 0xffffffffu;
#pragma unroll
    for (int i = 3; i >= 0; --i)
#pragma unroll
      for (int c = 3; c >= 0; --c)
        if (fabsf(v[i][c]) == hi) key = (u32)((64 * i + 4 * j + c) * 2 + (v[i][c] < 0.f ? 1 : 0));
    key = min(key, dpp_u32<DPP_XOR1>(key));
    key = min(key, dpp_u32<DPP_XOR2>(key));
    key = min(key, dpp_u32<DPP_HALF_MIRROR>(key));
    key = min(key, dpp_u32<DPP_MIRROR>(key));
    if (hi == -lo && hi > 0.f) vmax = key & 1u ? lo : hi;
  }
  // (a block of zeros: codes 0 * v = 0 and scale 0)
  const float iscale = vmax != 0.f ? __fdiv_rn(-127.f, vmax) : 0.f;
  const float d = vmax != 0.f ? __fmul_rn(vmax, 1.0f / -127.f) : 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u32 q[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) q[c] = (u32)min((int)rintf(__fmul_rn(iscale, v[i][c])), 127);
    const u32 packed = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u) | __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
    int sum = sdot4(packed, 0x01010101u, 0);
    sum += (int)dpp_u32<DPP_XOR1>((u32)sum);
    sum += (int)dpp_u32<DPP_XOR2>((u32)sum);
    const int sb = 4 * i + (j >> 2), h = sb >> 3, sidx = (sb >> 1) & 3, lh = sb & 1;  // sub-block of the quad (gemv_device.h: item records)
    uint8_t* rec = blk + (2 * h + lh) * ITEM_LDS;
    *reinterpret_cast<u32*>(rec + sidx * 16 + (j & 3) * 4) = packed;
    if ((j & 3) == 0) {
      if (LAY == LAY_Q2) {
        rec[64 + sidx] = (uint8_t)(sum >> 8);
        rec[68 + sidx] = (uint8_t)(sum & 0xff);
      } else {
        reinterpret_cast<short*>(rec + 64)[sidx] = (short)sum;
      }
    }
  }
  if (j < 4) {
    float* m = reinterpret_cast<float*>(blk + j * ITEM_LDS + 72);
    if (LAY == LAY_Q2) { m[0] = d * 0.0625f; m[1] = d; }
    else m[0] = d;
  }
}

// moe_gate for up to 64 experts without groups (src/infer.cpp:493-599) by ONE wave, lane e = expert e: the softmax's trees and the order of the sum of the
// weights are gate_body's (router_device.h), whose other 15 waves only add zeros here; the k rounds of "largest unmasked, first among equals" are k
// rounds of a wave maximum.  Returns in lane k < K the k-th expert, w its weight; sc: the lane's expert's score.
DEV int gate_wave(float v, float bias, bool has_bias, int lane, int E, int K, int scoring, int norm_topk_prob, float scaling, float& sc, float& w) {
  if (scoring == DSK_SCORE_SOFTMAX) {  // src/infer.cpp:472-487
    float mx = v;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, lane_xor(mx, off));
    const float ex = lane < E ? expf(v - mx) : 0.f;
    float sum = ex;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += lane_xor(sum, off);
    v = ex / sum;
  } else {
    v = 1.0f / (1.0f + expf(-v));  // sigmoid, src/infer.cpp:489-491
  }
  if (has_bias) v += bias;
  if (lane >= E) v = -INFINITY;
  sc = v;
  float left = v;
  unsigned long long taken = 0;
  int sel = 0;
  float sk = 0.f, wsum = 0.f;
  for (int k = 0; k < K; ++k) {
    const float m = ad::wave_max_dpp(left);
    unsigned long long at = __ballot(left == m && lane < E) & ~taken;
    if (at == 0) at = ~taken;  // (scores that are no numbers: the first ones left; K <= E)
    const int e = __builtin_ctzll(at);
    taken |= 1ull << e;
    const float s = u2f(__builtin_amdgcn_readlane(__builtin_bit_cast(u32, v), e));
    wsum += s;
    if (lane == k) { sel = e; sk = s; }
    if (lane == e) left = -INFINITY;
  }
  if (!norm_topk_prob) wsum = 1.0f;
  w = sk / wsum * scaling;
  return sel;
}

// An argument read at entry, with the others, in one trip.  The compiler reads a kernel's arguments where they are used, a trip each, and turns
// `cond ? a.p : a.q` into a choice between their two places and a read behind it.
template <typename T>
DEV T arg(T v) {
  asm volatile("" : "+s"(v));
  return v;
}
// v / d for 0 <= v < 2^16 / d (moe_down_plan looks at the range): m = ceil(2^16 / d)
DEV int div_small(int v, int m) { return (v * m) >> 16; }

}  // namespace

// ------------------------------------------------------------------------------------------------------------
// The router's rows (src/infer.cpp:839, 847): workgroup = 2 rows x 8 column slices, slices added in order like router_gate_kernel's.  The gate is the next
// launch's, so nothing is published, counted or waited for here; and a wave's weights do not wait for the norm's scale: everything is requested at
// entry.  Workgroup b leaves block b of rmsnorm(x) behind, as Q8_K or in 32 bits.  64 experts of 2048 columns: 7.5 us with the gate in the last workgroup to
// arrive, 3.9 here; in F8E5M2 models, whose x is left in 32 bits, 7.2 and 4.8 (medians over a token's launches, here and below).
// ------------------------------------------------------------------------------------------------------------
template <int NL>  // 256-column pieces of a slice
__global__ __launch_bounds__(1024) void router_scores_kernel(const float* __restrict__ x, const float* __restrict__ norm_w, const float* __restrict__ w, float* __restrict__ scores,
                                                            int dim, int E, float eps, int8_t* q_qs, float* q_d, int16_t* q_bsums, float* xn) {
  constexpr int SL = 8;
  __shared__ float scratch[16], part[16];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x;
  const int r = wave & 1, sl = wave >> 1, row = min(bid * 2 + r, E - 1);
  const int k0 = sl * NL * 256;
  f32x4 xs, xv[NL], nw[NL], wv[NL];
  xs = *reinterpret_cast<const f32x4*>(x + min(tid * 4, dim - 4));
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int i = min(k0 + k * 256, dim - 256) + lane * 4;
    xv[k] = *reinterpret_cast<const f32x4*>(x + i);
    nw[k] = *reinterpret_cast<const f32x4*>(norm_w + i);
    wv[k] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + (size_t)row * dim + i));
  }
  // the sum of squares and its trees as in router_norm_scale (dim <= 4096: a thread has one piece)
  float ss = 0.f;
  if (tid * 4 < dim) {
    ss = fmaf(xs.x, xs.x, ss);
    ss = fmaf(xs.y, xs.y, ss);
    ss = fmaf(xs.z, xs.z, ss);
    ss = fmaf(xs.w, xs.w, ss);
  }
  ss = wave_sum(ss);
  if (lane == 0) scratch[wave] = ss;
  lds_barrier();
  const float scale = 1.0f / sqrtf(scratch_total<16>(scratch) / (float)dim + eps);
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    if (k0 + k * 256 >= dim) continue;  // wave-uniform
    const float y[4] = {xv[k].x * scale * nw[k].x, xv[k].y * scale * nw[k].y, xv[k].z * scale * nw[k].z, xv[k].w * scale * nw[k].w};
    acc = fmaf(wv[k].x, y[0], acc);
    acc = fmaf(wv[k].y, y[1], acc);
    acc = fmaf(wv[k].z, y[2], acc);
    acc = fmaf(wv[k].w, y[3], acc);
    const int b = (k0 >> 8) + k;
    if (r == 0 && b % (int)gridDim.x == bid) {
      if (q_qs) ad::q8k_block(y, lane, q_qs + (size_t)b * 256, q_d + b, q_bsums + (size_t)b * 16);
      else *reinterpret_cast<f32x4*>(xn + b * 256 + lane * 4) = f32x4{y[0], y[1], y[2], y[3]};
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) part[wave] = acc;
  lds_barrier();
  if (tid < 2 && bid * 2 + tid < E) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < SL; ++k) v += part[k * 2 + tid];
    scores[bid * 2 + tid] = v;
  }
}

// one wave's gate over the router's scores: the chosen experts to the workgroup's LDS, and by workgroup 0 to memory
DEV void decide(const float* scores, const float* bias_p, int lane, int bid, int E, int K, int scoring, int norm_topk, float scaling, int* sel_s, const MoeUpArgs& a) {
  const int e = lane < E ? lane : E - 1;
  const float v = scores[e], bias = bias_p ? bias_p[e] : 0.f;
  float sc, w;
  const int sel = gate_wave(lane < E ? v : -INFINITY, bias, bias_p != nullptr, lane, E, K, scoring, norm_topk, scaling, sc, w);
  sel_s[lane] = sel;
  if (bid == 0) {
    if (lane < E) a.scores_out[lane] = sc;
    if (lane < K) { a.route_e[lane] = sel; a.route_w[lane] = w; }
  }
}

// ------------------------------------------------------------------------------------------------------------
// First half: every workgroup decides the gate for itself out of the scores (one wave, ~0.5 us: less than handing a decision over), while other waves stage the
// normed vector; then its share of the shared expert's and of the chosen experts' rows, all of a wave's requested at once.  Bound by latency (16.5 MB: 2.5
// us): V2-Lite's shapes in Q2_K 9.4 us by the generic launch, whose waves took two rounds, 8.1 - 8.4 here; with the router's launch a token 1303 -> 1130 us.
// ------------------------------------------------------------------------------------------------------------
template <int QT>
__global__ __launch_bounds__(1024) void experts_up_kernel(const float* __restrict__ scores, const int8_t* __restrict__ a_qs, const float* __restrict__ a_d,
                                                         const int16_t* __restrict__ a_bsums, int E, int K, const MoeUpArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int sel_s[64];
  constexpr int CW = 12;  // waves that multiply; three stage, one decides
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x, G = gridDim.x;
  const int lpr_log2 = arg(a.lpr_log2), RPW = 64 >> lpr_log2;
  const uint8_t *w1_qs = arg(a.w1_qs), *w1_sc = arg(a.w1_sc), *w1_dm = arg(a.w1_dm), *w3_qs = arg(a.w3_qs), *w3_sc = arg(a.w3_sc), *w3_dm = arg(a.w3_dm);
  const uint8_t *sw1_qs = arg(a.sw1_qs), *sw1_sc = arg(a.sw1_sc), *sw1_dm = arg(a.sw1_dm), *sw3_qs = arg(a.sw3_qs), *sw3_sc = arg(a.sw3_sc), *sw3_dm = arg(a.sw3_dm);
  const uint8_t *w1_hm = nullptr, *w3_hm = nullptr, *sw1_hm = nullptr, *sw3_hm = nullptr;
  if (QT == DSK_QUANT_Q3_K) { w1_hm = arg(a.w1_hm); w3_hm = arg(a.w3_hm); sw1_hm = arg(a.sw1_hm); sw3_hm = arg(a.sw3_hm); }
  float* const hb = glob(arg(a.hb));
  const float* const bias_p = glob(arg(a.bias));
  const int mi = arg(a.mi), shared_n = arg(a.shared_n), dim = arg(a.dim), act = arg(a.act), hb_stride = arg(a.hb_stride), scoring = arg(a.scoring), norm_topk = arg(a.norm_topk_prob);
  const float scaling = arg(a.scaling);
  const u32 div_mi = arg(a.div_mi);
  int8_t* const tap_qs = glob(arg(a.tap_qs));
  if (wave == 15) {
    decide(scores, bias_p, lane, bid, E, K, scoring, norm_topk, scaling, sel_s, a);
  } else if (wave >= CW) {
    for (int i = tid - CW * 64; i < dim >> 4; i += 192) {  // runs of 16 codes, their sums and their block's scale into item records (stage_q8)
      const u32x4 run = reinterpret_cast<const u32x4*>(a_qs)[i];
      const int bs = a_bsums[i];
      const float d = a_d[i >> 4];
      const int b = i >> 4, j = i & 15, h = j >> 3, sidx = (j >> 1) & 3, lh = j & 1;
      uint8_t* rec = smem + (size_t)(b * 4 + 2 * h + lh) * ITEM_LDS;
      *reinterpret_cast<u32x4*>(rec + sidx * 16) = run;
      float* m = reinterpret_cast<float*>(rec + 72);
      if (QT == DSK_QUANT_Q2_K) {
        rec[64 + sidx] = (uint8_t)(bs >> 8);
        rec[68 + sidx] = (uint8_t)(bs & 0xff);
        m[0] = d * 0.0625f;
        m[1] = d;
      } else {
        reinterpret_cast<short*>(rec + 64)[sidx] = (short)bs;
        m[0] = d;
      }
    }
  }
  lds_barrier();
  if (tap_qs && bid == 0) dump_staged_q8_inline<QT == DSK_QUANT_Q2_K>(smem, dim, tap_qs, a.tap_d, tid, 1024);
  if (wave >= CW) return;
  const int rloc = lane >> lpr_log2, sub = lane & ((1 << lpr_log2) - 1), q = sub & 3, nb = dim >> 8, items = 1 << lpr_log2;
  // this workgroup's rows of the shared expert and of the chosen ones (slot-major), each an even share, in steps of RPW rows
  const int s_lo = (int)((unsigned)(shared_n * bid) / (unsigned)G), s_hi = (int)((unsigned)(shared_n * (bid + 1)) / (unsigned)G);
  const int v_lo = (int)((unsigned)(K * mi * bid) / (unsigned)G), v_hi = (int)((unsigned)(K * mi * (bid + 1)) / (unsigned)G);
  const int JS = (s_hi - s_lo + RPW - 1) >> (6 - lpr_log2), J = JS + ((v_hi - v_lo + RPW - 1) >> (6 - lpr_log2));
  const uint8_t* lds_lane = smem + sub * ITEM_LDS;
  struct Step { ChunkKQ<QT, 1, 1, true> c; int out; };
  auto request = [&](int j, Step& S) {
    const bool sh = j < JS;  // wave-uniform
    const int v = (sh ? s_lo + j * RPW : v_lo + (j - JS) * RPW) + rloc, end = sh ? s_hi : v_hi;
    const bool valid = j < J && v < end;
    const int vv = min(v, max(end - 1, 0)), slot = sh ? K : min((int)__umulhi((u32)vv, div_mi), K - 1), rr = sh ? vv : vv - slot * mi;
    S.out = valid ? slot * hb_stride + rr : -1;
    const int rowblk[1] = {((sh ? 0 : sel_s[slot] * mi) + rr) * nb + (sub >> 2)};
    KQRsrc B;
    B.qs = make_rsrc_n(sh ? sw1_qs : w1_qs, j < J); B.sc = make_rsrc_n(sh ? sw1_sc : w1_sc, j < J);
    B.dm = make_rsrc_n(sh ? sw1_dm : w1_dm, j < J); B.hm = make_rsrc_n(sh ? sw1_hm : w1_hm, j < J);
    B.qs2 = make_rsrc_n(sh ? sw3_qs : w3_qs, j < J); B.sc2 = make_rsrc_n(sh ? sw3_sc : w3_sc, j < J);
    B.dm2 = make_rsrc_n(sh ? sw3_dm : w3_dm, j < J); B.hm2 = make_rsrc_n(sh ? sw3_hm : w3_hm, j < J);
    load_chunk_kq<QT, 1, 1, true>(S.c, B, 1, items, sub, lpr_log2, q, rowblk, 0);
  };
  auto finish = [&](const Step& S) {
    float acc[1] = {0.f}, acc2[1] = {0.f};
    compute_chunk_kq<QT, 1, 1, true>(S.c, 1, items, sub, lpr_log2, q, 0, lds_lane, acc, acc2);
    const float g = lanes_sum(acc[0], lpr_log2), u = lanes_sum(acc2[0], lpr_log2);
    if (sub == 0 && S.out >= 0) hb[S.out] = act_fn(g, act) * u;  // src/infer.cpp:859-872
  };
  for (int j = wave; j < J; j += 2 * CW) {
    Step S0, S1;
    request(j, S0);
    request(j + CW, S1);  // (a step that is not there reads through an empty descriptor: no branch around its loads)
    finish(S0);
    finish(S1);
  }
}

// ------------------------------------------------------------------------------------------------------------
// The same for F8E5M2 and F16 weights: a row is ITS steps of a whole wave (moe_ffn_f_kernel's lanes and order), its values' factors stay in registers for all rows of
// a wave, and the next two rows are on their way while one is multiplied.  V2-Lite's shapes in F8E5M2: 46 MB in 12.4 - 13.2 us, a pure stream of that size taking 9.6 (16
// waves that multiply instead of 12, or the shared expert's rows requested before the gate: the same).
// ------------------------------------------------------------------------------------------------------------
template <int QT, int ITS>
__global__ __launch_bounds__(1024) void experts_up_f_kernel(const float* __restrict__ scores, const float* __restrict__ xn, int E, int K, const MoeUpArgs a) {
  constexpr int EPI = FTraits<QT>::EPI, CW = 12, ITEMS = ITS * 64, DIM = ITEMS * EPI;
  constexpr bool F8 = QT == DSK_QUANT_F8E5M2;
  __shared__ __attribute__((aligned(16))) float x_s[DIM];
  __shared__ int sel_s[64];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x, G = gridDim.x;
  const uint8_t *w1 = arg(a.w1_qs), *w3 = arg(a.w3_qs), *sw1 = arg(a.sw1_qs), *sw3 = arg(a.sw3_qs);
  const float *w1_scale = nullptr, *w3_scale = nullptr, *sw1_scale = nullptr, *sw3_scale = nullptr;
  if (F8) { w1_scale = arg(a.w1_scale); w3_scale = arg(a.w3_scale); sw1_scale = arg(a.sw1_scale); sw3_scale = arg(a.sw3_scale); }
  const size_t e_qs = arg(a.e13_qs), e_scale = arg(a.e13_scale);
  float* const hb = glob(arg(a.hb));
  const float* const bias_p = glob(arg(a.bias));
  const int mi = arg(a.mi), shared_n = arg(a.shared_n), act = arg(a.act), hb_stride = arg(a.hb_stride), scoring = arg(a.scoring), norm_topk = arg(a.norm_topk_prob);
  const int b0 = arg(a.b0), sh0 = arg(a.sh0), sc_cols = arg(a.sc_cols);
  const float scaling = arg(a.scaling);
  const u32 div_mi = arg(a.div_mi);
  int sc_off[ITS];  // (the scale's column of an item)
#pragma unroll
  for (int u = 0; u < ITS; ++u) sc_off[u] = (a.sh1 >= 0 ? (u * 64 + lane) * EPI >> a.sh1 : (u * 64 + lane) * EPI / a.b1) * 4;
  const int s_lo = (int)((unsigned)(shared_n * bid) / (unsigned)G), s_hi = (int)((unsigned)(shared_n * (bid + 1)) / (unsigned)G);
  const int v_lo = (int)((unsigned)(K * mi * bid) / (unsigned)G), v_hi = (int)((unsigned)(K * mi * (bid + 1)) / (unsigned)G);
  const int JS = s_hi - s_lo, J = JS + v_hi - v_lo;
  struct Row { u32x4 w[ITS], u[ITS]; float sw[ITS], su[ITS]; int out; };
  auto request = [&](int j, Row& R) {  // (a row that is not there reads through an empty descriptor)
    const bool live = j < J, sh = j < JS;
    const int v = sh ? s_lo + j : min(v_lo + j - JS, v_hi - 1), slot = sh ? K : (int)__umulhi((u32)max(v, 0), div_mi), rr = sh ? v : v - slot * mi;
    const int e = sh ? 0 : __builtin_amdgcn_readfirstlane(sel_s[min(slot, K - 1)]);
    R.out = live ? slot * hb_stride + rr : -1;
    const size_t at = (sh ? 0 : e * e_qs) + (size_t)rr * (DIM * FTraits<QT>::ESZ);
    const rsrc_t B1 = make_rsrc_n((sh ? sw1 : w1) + at, live), B3 = make_rsrc_n((sh ? sw3 : w3) + at, live);
#pragma unroll
    for (int u = 0; u < ITS; ++u) {
      R.w[u] = __builtin_amdgcn_raw_buffer_load_b128(B1, lane * 16, u * 1024, BUF_NT);
      R.u[u] = __builtin_amdgcn_raw_buffer_load_b128(B3, lane * 16, u * 1024, BUF_NT);
    }
    if constexpr (F8) {
      const size_t sat = (sh ? 0 : e * e_scale) + (size_t)(sh0 >= 0 ? rr >> sh0 : rr / b0) * sc_cols;
      const rsrc_t S1 = make_rsrc_n((sh ? sw1_scale : w1_scale) + sat, live), S3 = make_rsrc_n((sh ? sw3_scale : w3_scale) + sat, live);
#pragma unroll
      for (int u = 0; u < ITS; ++u) {
        R.sw[u] = u2f(__builtin_amdgcn_raw_buffer_load_b32(S1, sc_off[u], 0, 0));
        R.su[u] = u2f(__builtin_amdgcn_raw_buffer_load_b32(S3, sc_off[u], 0, 0));
      }
    }
  };
  float xa[ITS][EPI];
  auto finish = [&](const Row& R) {
    float g = 0.f, up = 0.f;
#pragma unroll
    for (int u = 0; u < ITS; ++u) {
      g = fmaf(fitem<QT>(R.w[u], xa[u], 0.f), F8 ? R.sw[u] : 1.0f, g);
      up = fmaf(fitem<QT>(R.u[u], xa[u], 0.f), F8 ? R.su[u] : 1.0f, up);
    }
    g = lanes_sum(g, 6);
    up = lanes_sum(up, 6);
    if (lane == 0 && R.out >= 0) hb[R.out] = act_fn(g, act) * up;  // src/infer.cpp:859-872
  };
  if (wave == 15) {
    decide(scores, bias_p, lane, bid, E, K, scoring, norm_topk, scaling, sel_s, a);
  } else if (wave >= CW) {
    for (int i = tid - CW * 64; i < DIM / 4; i += 192)
      reinterpret_cast<f32x4*>(x_s)[quad_place<EPI>(i, ITEMS)] = reinterpret_cast<const f32x4*>(xn)[i];
  }
  lds_barrier();
  if (wave >= CW) return;
#pragma unroll
  for (int u = 0; u < ITS; ++u)
#pragma unroll
    for (int k = 0; k < EPI / 4; ++k) {
      const f32x4 t = reinterpret_cast<const f32x4*>(x_s)[k * ITEMS + u * 64 + lane];
      xa[u][4 * k] = t.x; xa[u][4 * k + 1] = t.y; xa[u][4 * k + 2] = t.z; xa[u][4 * k + 3] = t.w;
    }
  Row A, B;
  request(wave, A);
  request(wave + CW, B);
  for (int j = wave; j < J; j += 2 * CW) {
    finish(A);
    request(j + 2 * CW, A);
    finish(B);
    request(j + 3 * CW, B);
  }
}

// ------------------------------------------------------------------------------------------------------------
// Second half: workgroup b owns rows [b * rows_wg, +rows_wg) of x for ALL slots, so that nothing has to be handed over between workgroups (the
// generic launch deals (slot, rows) to its workgroups and needs a publish, an arrival, an acquire and a read before the last one can add up).  What a
// workgroup needs of it is a chain: the experts' ids, the weights, the multiplies.  Its first waves do that; the others meanwhile read and
// quantise the slots' hidden vectors (12288 values for V2-Lite), so that neither waits for the other's loads.  Bound by latency: 8.3 MB of weights
// are 1.2 us.  V2-Lite (6 of 64 experts of 1536, shared 3072, Q2_K), us a launch: generic 13.0 (224 workgroups of 4 waves, two rows per lane and the
// hand-over), here 7.5; with the arguments read where they are used, two copies of the quantisation and a stack of descriptors 9.6.  A token
// 1460 -> 1303 us.
// ------------------------------------------------------------------------------------------------------------
template <int QT>
__global__ __launch_bounds__(1024) void experts_down_kernel(const float* __restrict__ hb, const int* __restrict__ route_e, const float* __restrict__ route_w,
                                                           float* x, int hb_stride, int K, int cw, const MoeDownArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NW = 16, U = QT == DSK_QUANT_Q2_K ? 6 : 4;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x;
  const uint8_t *w2_qs = arg(a.w2_qs), *w2_sc = arg(a.w2_sc), *w2_dm = arg(a.w2_dm), *sw2_qs = arg(a.sw2_qs), *sw2_sc = arg(a.sw2_sc), *sw2_dm = arg(a.sw2_dm);
  const uint8_t *w2_hm = nullptr, *sw2_hm = nullptr;
  if (QT == DSK_QUANT_Q3_K) { w2_hm = arg(a.w2_hm); sw2_hm = arg(a.sw2_hm); }
  float* const eout = glob(arg(a.eout));
  const int mi = arg(a.mi), shared_n = arg(a.shared_n), dim = arg(a.dim), rows_wg = arg(a.rows_wg), lpr_log2 = arg(a.lpr_log2), lds_b = arg(a.lds_b), div_nb = arg(a.div_nb),
            div_rows = arg(a.div_rows);
  int8_t* const tap_qs = glob(arg(a.tap_qs));
  uint8_t* act = smem;                                                   // [slot][lds_b] item records
  float* o_s = reinterpret_cast<float*>(smem + (size_t)lds_b * (K + 1));  // [slot][rows_wg]
  const int nbR = mi >> 8, nbS = shared_n >> 8, slots = K + (nbS > 0 ? 1 : 0);
  const int r_lo = bid * rows_wg, nrows = min(rows_wg, dim - r_lo);
  float xv = 0.f, rw = 0.f;  // the rows' old values, the slots' weights (the last wave adds up)
  if (wave < cw) {
    const int e_all = route_e[lane < K ? lane : K - 1];
    const int RPW = 64 >> lpr_log2;
    const int rloc = lane >> lpr_log2, sub = lane & ((1 << lpr_log2) - 1), q = sub & 3;
    // steps of RPW rows: the shared expert's first (its rows are the longest), then the routed slots' (slot, row) slot-major
    const int WS = nbS > 0 ? (rows_wg + RPW - 1) >> (6 - lpr_log2) : 0, WR = (rows_wg * K + RPW - 1) >> (6 - lpr_log2);
    ChunkKQ<QT, 1, U, false> c;
    bool wait = true;
    for (int st = wave; st < WS + WR; st += cw) {
      const bool sh = st < WS;  // wave-uniform
      const int v = (sh ? st : st - WS) * RPW + rloc;
      const int slot = sh ? K : min(div_small(v, div_rows), K - 1), rr0 = sh ? v : v - slot * rows_wg;
      const bool valid = rr0 < nrows;
      const int rr = valid ? rr0 : nrows - 1, nb = sh ? nbS : nbR, items = nb * 4, its = (items + (1 << lpr_log2) - 1) >> lpr_log2;
      const int e = sh ? 0 : __shfl(e_all, slot);
      const int rowblk[1] = {(e * dim + r_lo + rr) * nb + (sub >> 2)};
      WPtr P;
      P.present = true; P.qs2 = P.sc2 = P.hm2 = P.dm2 = nullptr; P.scale = P.scale2 = nullptr;
      P.qs = sh ? sw2_qs : w2_qs; P.sc = sh ? sw2_sc : w2_sc; P.hm = sh ? sw2_hm : w2_hm; P.dm = sh ? sw2_dm : w2_dm;
      const KQRsrc B = kq_rsrc<QT, false>(P);
      const uint8_t* lds_lane = act + (size_t)slot * lds_b + sub * ITEM_LDS;
      float acc[1] = {0.f}, dummy[1] = {0.f};
      for (int it0 = 0; it0 < its; it0 += U) {
        load_chunk_kq<QT, 1, U, false>(c, B, its, items, sub, lpr_log2, q, rowblk, it0);
        if (wait) lds_barrier();  // the hidden vectors are staged; this wave's first weights stay on their way
        wait = false;
        compute_chunk_kq<QT, 1, U, false>(c, its, items, sub, lpr_log2, q, it0, lds_lane, acc, dummy);
      }
      const float o = lanes_sum(acc[0], lpr_log2);
      if (sub == 0 && valid) o_s[slot * rows_wg + rr] = o;
    }
    if (wait) lds_barrier();
  } else {
    const int sw = NW - cw, nblk = K * nbR + nbS, r16 = lane >> 4, j = lane & 15;
    for (int b0 = (wave - cw) * 4; b0 < nblk; b0 += sw * 8) {  // two groups of four blocks at once
      f32x4 t0[4], t1[4];
      auto request = [&](int bb0, f32x4 (&t)[4]) {
        const int b = min(bb0 + r16, nblk - 1);  // (lanes past the end: the last block again, the same values to the same place)
        const int s = b < K * nbR ? div_small(b, div_nb) : K, bb = b - s * nbR;
        const float* src = hb + (size_t)s * hb_stride + bb * 256 + j * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = *reinterpret_cast<const f32x4*>(src + 64 * i);
        return act + (size_t)s * lds_b + (size_t)bb * 4 * ITEM_LDS;
      };
      uint8_t* dst = request(b0, t0);
      uint8_t* const dst1 = request(b0 + sw * 4, t1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
      for (int p = 0; p < 2; ++p) {  // (one copy of the code)
        q8k_four_blocks_lds<QT == DSK_QUANT_Q2_K>(t0, lane, dst);
#pragma unroll
        for (int i = 0; i < 4; ++i) t0[i] = t1[i];
        dst = dst1;
        if (b0 + sw * 4 >= nblk) break;
      }
    }
    xv = x[r_lo + (lane < nrows ? lane : nrows - 1)];
    rw = route_w[lane < K ? lane : K - 1];
    lds_barrier();
  }
  if (tap_qs && bid == 0)  // parity tap: what the slots staged
    for (int s = 0; s < slots; ++s)
      dump_staged_q8_inline<QT == DSK_QUANT_Q2_K>(act + (size_t)s * lds_b, s < K ? mi : shared_n, tap_qs + (size_t)s * a.tap_stride,
                                                 a.tap_d + (size_t)s * (a.tap_stride >> 8), tid, 1024);
  lds_barrier();
  if (wave == NW - 1 && lane < nrows) {  // x += w_k * o_k in k order (src/infer.cpp:874-877), then the shared expert (:900-903)
    for (int k = 0; k < slots; ++k) {
      const float o = o_s[k * rows_wg + lane];
      eout[(size_t)k * dim + r_lo + lane] = o;
      if (k < K) xv = fmaf(o, u2f(__builtin_amdgcn_readlane(__builtin_bit_cast(u32, rw), k)), xv);
      else xv += o;
    }
    x[r_lo + lane] = xv;
  }
}

// ------------------------------------------------------------------------------------------------------------
// The same for F8E5M2 and F16 weights (lanes, order and combine of moe_ffn_f_kernel): nothing to quantise, so all waves copy the hidden vectors, between the
// request of their first weights and their use.  V2-Lite's shapes in F8E5M2: 23 MB in 8.5 us.  Router, first and second half were 7.2 + 23.6 us with both halves in one
// launch, 4.8 + 12.4 + 8.5 here: the hand-over inside it cost more than a launch; a token 1505 -> 1341 us.
// ------------------------------------------------------------------------------------------------------------
template <int QT>
__global__ __launch_bounds__(1024) void experts_down_f_kernel(const float* __restrict__ hb, const int* __restrict__ route_e, const float* __restrict__ route_w, float* x,
                                                             int hb_stride, int K, const MoeDownArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NW = 16, EPI = FTraits<QT>::EPI, ESZ = FTraits<QT>::ESZ, U = 6, HQ = 4;
  constexpr bool F8 = QT == DSK_QUANT_F8E5M2;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x;
  const uint8_t *w2 = arg(a.w2_qs), *sw2 = arg(a.sw2_qs);
  const float *w2_scale = nullptr, *sw2_scale = nullptr;
  if (F8) { w2_scale = arg(a.w2_scale); sw2_scale = arg(a.sw2_scale); }
  const size_t e_qs = arg(a.e2_qs), e_scale = arg(a.e2_scale);
  float* const eout = glob(arg(a.eout));
  const int mi = arg(a.mi), shared_n = arg(a.shared_n), dim = arg(a.dim), rows_wg = arg(a.rows_wg), lpr_log2 = arg(a.lpr_log2), lds_b = arg(a.lds_b), div_q = arg(a.div_nb),
            div_rows = arg(a.div_rows), b0 = arg(a.b0), b1 = arg(a.b1), sh0 = arg(a.sh0), sh1 = arg(a.sh1);
  float* o_s = reinterpret_cast<float*>(smem + (size_t)lds_b * (K + 1));  // [slot][rows_wg]
  const int slots = K + (shared_n > 0 ? 1 : 0), r_lo = bid * rows_wg, nrows = min(rows_wg, dim - r_lo);
  float xv = 0.f, rw = 0.f;
  if (wave == NW - 1) {
    xv = x[r_lo + (lane < nrows ? lane : nrows - 1)];
    rw = route_w[lane < K ? lane : K - 1];
  }
  const int e_all = route_e[lane < K ? lane : K - 1];
  // 1. the hidden vectors' pieces of 16 bytes, the first HQ of a thread: piece i of the slots behind each other
  const int pR = mi >> 2, pieces = K * pR + (shared_n >> 2);
  auto piece = [&](int i, const float*& src, uint8_t*& dst) {
    const int ii = min(i, pieces - 1), s = ii < K * pR ? (int)__umulhi((u32)ii, (u32)div_q) : K, j = ii - s * pR, n = s < K ? mi : shared_n;
    src = hb + (size_t)s * hb_stride + j * 4;
    dst = smem + (size_t)s * lds_b + (size_t)quad_place<EPI>(j, n / EPI) * 16;
  };
  f32x4 hv[HQ];
  uint8_t* hd[HQ];
#pragma unroll
  for (int k = 0; k < HQ; ++k) {
    const float* src;
    piece(tid + k * 1024, src, hd[k]);
    hv[k] = *reinterpret_cast<const f32x4*>(src);
  }
  // 2. this wave's steps of RPW rows: the shared expert's first (the longest), then the routed slots'; the first two chunks of U column steps
  const int RPW = 64 >> lpr_log2, rloc = lane >> lpr_log2, sub = lane & ((1 << lpr_log2) - 1);
  const int WS = shared_n > 0 ? (rows_wg + RPW - 1) >> (6 - lpr_log2) : 0, WR = (rows_wg * K + RPW - 1) >> (6 - lpr_log2);
  struct Chunk { u32x4 w[U]; float sv[U]; };
  struct Step { const uint8_t* row; const float* sc; int items, its, slot, rr; bool valid; };
  auto step_of = [&](int st) {
    Step S;
    const bool sh = st < WS;
    const int v = (sh ? st : st - WS) * RPW + rloc, n = sh ? shared_n : mi;
    S.slot = sh ? K : min(div_small(v, div_rows), K - 1);
    const int rr0 = sh ? v : v - S.slot * rows_wg;
    S.valid = st < WS + WR && rr0 < nrows;
    S.rr = min(rr0, nrows - 1);
    S.items = n / EPI;
    S.its = (S.items + (1 << lpr_log2) - 1) >> lpr_log2;
    const int e = sh ? 0 : __shfl(e_all, S.slot), r = r_lo + S.rr;
    S.row = (sh ? sw2 : w2 + e * e_qs) + (size_t)r * n * ESZ;
    if (F8) S.sc = (sh ? sw2_scale : w2_scale + e * e_scale) + (size_t)(sh0 >= 0 ? r >> sh0 : r / b0) * (sh1 >= 0 ? (n + b1 - 1) >> sh1 : (n + b1 - 1) / b1);
    return S;
  };
  auto request = [&](const Step& S, int it0, Chunk& C) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int item = min(sub + ((it0 + u) << lpr_log2), S.items - 1);
      C.w[u] = ldg_nt(reinterpret_cast<const u32x4*>(S.row + (size_t)item * 16));
      if (F8) C.sv[u] = S.sc[sh1 >= 0 ? item * EPI >> sh1 : item * EPI / b1];
    }
  };
  auto multiply = [&](const Step& S, int it0, const Chunk& C, float acc) {
    const f32x4* l = reinterpret_cast<const f32x4*>(smem + (size_t)S.slot * lds_b);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (it0 + u >= S.its) break;
      const int it = sub + ((it0 + u) << lpr_log2), item = min(it, S.items - 1);
      float xa[EPI];
#pragma unroll
      for (int k = 0; k < EPI / 4; ++k) {
        const f32x4 t = l[k * S.items + item];  // (quad_place)
        xa[4 * k] = t.x; xa[4 * k + 1] = t.y; xa[4 * k + 2] = t.z; xa[4 * k + 3] = t.w;
      }
      const float sv = it < S.items ? (F8 ? C.sv[u] : 1.0f) : 0.f;
      acc = fmaf(fitem<QT>(C.w[u], xa, 0.f), sv, acc);
    }
    return acc;
  };
  Chunk A, B;
  Step S = step_of(wave);
  if (wave < WS + WR) {
    request(S, 0, A);
    if (U < S.its) request(S, U, B);
  }
  // 3. the hidden vectors into LDS
#pragma unroll
  for (int k = 0; k < HQ; ++k) *reinterpret_cast<f32x4*>(hd[k]) = hv[k];  // (pieces past the end: the last one again)
  for (int i = tid + HQ * 1024; i < pieces; i += 1024) {
    const float* src;
    uint8_t* dst;
    piece(i, src, dst);
    *reinterpret_cast<f32x4*>(dst) = *reinterpret_cast<const f32x4*>(src);
  }
  lds_barrier();
  // 4. column steps in order
  for (int st = wave; st < WS + WR; st += NW) {
    if (st != wave) {
      S = step_of(st);
      request(S, 0, A);
      if (U < S.its) request(S, U, B);
    }
    float acc = 0.f;
    for (int it0 = 0; it0 < S.its; it0 += 2 * U) {
      acc = multiply(S, it0, A, acc);
      if (it0 + 2 * U < S.its) request(S, it0 + 2 * U, A);
      if (it0 + U < S.its) acc = multiply(S, it0 + U, B, acc);
      if (it0 + 3 * U < S.its) request(S, it0 + 3 * U, B);
    }
    const float o = lanes_sum(acc, lpr_log2);
    if (sub == 0 && S.valid) o_s[S.slot * rows_wg + S.rr] = o;
  }
  lds_barrier();
  if (wave == NW - 1 && lane < nrows) {  // x += w_k * o_k in k order (src/infer.cpp:874-877), then the shared expert (:900-903)
    for (int k = 0; k < slots; ++k) {
      const float o = o_s[k * rows_wg + lane];
      eout[(size_t)k * dim + r_lo + lane] = o;
      if (k < K) xv = fmaf(o, u2f(__builtin_amdgcn_readlane(__builtin_bit_cast(u32, rw), k)), xv);
      else xv += o;
    }
    x[r_lo + lane] = xv;
  }
}

// ---- host side ------------------------------------------------------------------------------------------
int moe_up_plan(MoeUpArgs& a, int n_cus) {
  const bool kq = a.quant == DSK_QUANT_Q2_K || a.quant == DSK_QUANT_Q3_K, f8 = a.quant == DSK_QUANT_F8E5M2;
  if (!kq && !f8 && a.quant != DSK_QUANT_F16) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: weights");
  if (a.E < 1 || a.E > 64 || a.K < 1 || a.K > a.E || a.K > 15 || a.mi < 1 || a.shared_n < 0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: shapes");
  // router slices of one or two pieces, the norm of one piece a thread; K-quants: rows of one column step; floats: of 1, 2 or (F16) 4 steps of a whole wave
  if (a.dim % 256 || a.dim > 4096) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: rows of %d", a.dim);
  if (kq && a.dim / 64 != 1 << a.lpr_log2) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: rows of %d", a.dim);
  if (!kq) {
    a.its = a.dim / (f8 ? 16 : 8) / 64;
    if (a.lpr_log2 != 6 || a.its * 64 * (f8 ? 16 : 8) != a.dim || !(a.its == 1 || a.its == 2 || (a.its == 4 && !f8))) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: rows of %d", a.dim);
    if (a.b0 < 1) a.b0 = 1;
    if (a.b1 < 1) a.b1 = 1;
    a.sh0 = (a.b0 & (a.b0 - 1)) ? -1 : __builtin_ctz(a.b0); a.sh1 = (a.b1 & (a.b1 - 1)) ? -1 : __builtin_ctz(a.b1); a.sc_cols = (a.dim + a.b1 - 1) / a.b1;
  }
  if (kq && ((double)a.E * a.mi * (a.dim / 256) * 64.0 >= 2147483648.0 || (double)a.shared_n * (a.dim / 256) * 64.0 >= 2147483648.0))
    DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: a stack exceeds the 31-bit offset of a buffer load");
  // (v * ceil(2^32 / d) >> 32 == v / d while v * (d - 1) < 2^32)
  if (a.mi < 2 || (double)a.K * a.mi * a.mi >= 4294967296.0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: too many rows");
  a.div_mi = (unsigned)((4294967296ull + a.mi - 1) / a.mi);
  if ((double)(a.K * a.mi > a.shared_n ? a.K * a.mi : a.shared_n) * n_cus >= 4294967296.0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_up: too many rows");
  const int rows = a.K * a.mi + a.shared_n, RPW = 64 >> a.lpr_log2;
  a.grid = n_cus < (rows + RPW - 1) / RPW ? n_cus : (rows + RPW - 1) / RPW;
  a.lds = a.dim / 64 * ITEM_LDS;
  return DSK_OK;
}

int launch_router_scores(hipStream_t st, const RouterArgs& r, float* xn) {
  auto go = [&](auto k) {
    const dim3 grid((r.n_routed + 1) / 2), block(1024);
    if (g_prof_start && g_prof_stop)
      hipExtLaunchKernelGGL(k, grid, block, 0u, st, g_prof_start, g_prof_stop, 0u, r.x, r.norm_w, r.w, r.partial, r.dim, r.n_routed, r.eps, r.q_qs, r.q_d, r.q_bsums, xn);
    else hipLaunchKernelGGL(k, grid, block, 0u, st, r.x, r.norm_w, r.w, r.partial, r.dim, r.n_routed, r.eps, r.q_qs, r.q_d, r.q_bsums, xn);
  };
  if (r.dim > 2048) go(router_scores_kernel<2>);  // (pieces of a slice as in router_body: ceil(dim / 2048))
  else go(router_scores_kernel<1>);
  return DSK_OK;
}

int launch_moe_up(hipStream_t st, const MoeUpArgs& a) {
  auto go = [&](auto k) {
    if (g_prof_start && g_prof_stop)
      hipExtLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, g_prof_start, g_prof_stop, 0u, a.scores, a.a_qs, a.a_d, a.a_bsums, a.E, a.K, a);
    else hipLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, a.scores, a.a_qs, a.a_d, a.a_bsums, a.E, a.K, a);
  };
  auto floats = [&](auto k) {
    if (g_prof_start && g_prof_stop) hipExtLaunchKernelGGL(k, dim3(a.grid), dim3(1024), 0u, st, g_prof_start, g_prof_stop, 0u, a.scores, a.xn, a.E, a.K, a);
    else hipLaunchKernelGGL(k, dim3(a.grid), dim3(1024), 0u, st, a.scores, a.xn, a.E, a.K, a);
  };
  switch (a.quant) {
    case DSK_QUANT_Q2_K: go(experts_up_kernel<DSK_QUANT_Q2_K>); break;
    case DSK_QUANT_Q3_K: go(experts_up_kernel<DSK_QUANT_Q3_K>); break;
    case DSK_QUANT_F8E5M2: a.its == 1 ? floats(experts_up_f_kernel<DSK_QUANT_F8E5M2, 1>) : floats(experts_up_f_kernel<DSK_QUANT_F8E5M2, 2>); break;
    default: a.its == 1 ? floats(experts_up_f_kernel<DSK_QUANT_F16, 1>) : a.its == 2 ? floats(experts_up_f_kernel<DSK_QUANT_F16, 2>) : floats(experts_up_f_kernel<DSK_QUANT_F16, 4>);
  }
  return DSK_OK;
}

int moe_down_plan(MoeDownArgs& a, int n_cus) {
  const bool kq = a.quant == DSK_QUANT_Q2_K || a.quant == DSK_QUANT_Q3_K, f8 = a.quant == DSK_QUANT_F8E5M2;
  const int unit = kq ? 256 : f8 ? 16 : 8;
  if (!kq && !f8 && a.quant != DSK_QUANT_F16) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: weights");
  if (a.K < 1 || a.K > 15 || a.dim < 1 || a.mi < unit || a.mi % unit || a.shared_n % unit || a.shared_n < 0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: shapes");
  const int lpr = 1 << a.lpr_log2, RPW = 64 / lpr, nbR = a.mi >> 8, nbS = a.shared_n >> 8;
  if (lpr > 64 || (kq && (lpr < 4 || (nbR * 4) % lpr || (nbS * 4) % lpr))) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: %d lanes do not divide the rows", lpr);
  a.rows_wg = (a.dim + n_cus - 1) / n_cus;
  a.grid = (a.dim + a.rows_wg - 1) / a.rows_wg;
  if (a.rows_wg > 64) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: %d rows per workgroup", a.rows_wg);
  // K-quants: one descriptor spans the stack: a lane's byte offset (expert, row, block) must fit its 32-bit offset field
  if (kq && ((double)a.n_experts * a.dim * nbR * 64.0 >= 2147483648.0 || (double)a.dim * nbS * 64.0 >= 2147483648.0))
    DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: a stack exceeds the 31-bit offset of a buffer load");
  // (v * ceil(2^16 / d) >> 16 == v / d while v * (d - 1) < 2^16; with 2^32 likewise)
  const long nblk = (long)a.K * nbR + nbS, nv = (long)a.K * a.rows_wg + RPW;
  a.div_rows = (65536 + a.rows_wg - 1) / a.rows_wg;
  if (nv * (a.rows_wg - 1) >= 65536) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: too many rows");
  if (kq) {
    a.div_nb = (65536 + nbR - 1) / nbR;
    if (nblk * (nbR - 1) >= 65536 || nblk >= 32768) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: too many blocks");
  } else {
    if (a.mi < 8 || (double)(a.K * (a.mi / 4) + a.shared_n / 4) * (a.mi / 4) >= 4294967296.0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: too many values");
    a.div_nb = (unsigned)((4294967296ull + a.mi / 4 - 1) / (a.mi / 4));
    if (a.b0 < 1) a.b0 = 1;
    if (a.b1 < 1) a.b1 = 1;
    a.sh0 = (a.b0 & (a.b0 - 1)) ? -1 : __builtin_ctz(a.b0); a.sh1 = (a.b1 & (a.b1 - 1)) ? -1 : __builtin_ctz(a.b1);
  }
  const int nB = a.mi > a.shared_n ? a.mi : a.shared_n;
  a.lds_b = kq ? nB / 64 * ITEM_LDS : nB * 4;
  const size_t lds = (size_t)a.lds_b * (a.K + 1) + (size_t)(a.K + 1) * a.rows_wg * 4;
  if (lds > 150 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: activations do not fit LDS");
  a.lds = (int)lds;
  const int steps = (nbS > 0 ? (a.rows_wg + RPW - 1) / RPW : 0) + (a.rows_wg * a.K + RPW - 1) / RPW;
  a.cw = steps < 8 ? steps : 8;
  return DSK_OK;
}

int launch_moe_down(hipStream_t st, const MoeDownArgs& a) {
  auto go = [&](auto k) {
    if (a.lds > 48 * 1024) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, a.lds);
    if (g_prof_start && g_prof_stop)
      hipExtLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, g_prof_start, g_prof_stop, 0u, a.hb, a.route_e, a.route_w, a.x, a.hb_stride, a.K, a.cw, a);
    else hipLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, a.hb, a.route_e, a.route_w, a.x, a.hb_stride, a.K, a.cw, a);
  };
  auto floats = [&](auto k) {
    if (a.lds > 48 * 1024) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, a.lds);
    if (g_prof_start && g_prof_stop)
      hipExtLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, g_prof_start, g_prof_stop, 0u, a.hb, a.route_e, a.route_w, a.x, a.hb_stride, a.K, a);
    else hipLaunchKernelGGL(k, dim3(a.grid), dim3(1024), (uint32_t)a.lds, st, a.hb, a.route_e, a.route_w, a.x, a.hb_stride, a.K, a);
  };
  switch (a.quant) {
    case DSK_QUANT_Q2_K: go(experts_down_kernel<DSK_QUANT_Q2_K>); break;
    case DSK_QUANT_Q3_K: go(experts_down_kernel<DSK_QUANT_Q3_K>); break;
    case DSK_QUANT_F8E5M2: floats(experts_down_f_kernel<DSK_QUANT_F8E5M2>); break;
    default: floats(experts_down_f_kernel<DSK_QUANT_F16>);
  }
  return DSK_OK;
}
