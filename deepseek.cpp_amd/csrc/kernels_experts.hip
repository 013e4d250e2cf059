// kernels_experts.hip -- the routed experts of one token in launches of their own, for models whose launches are bound by latency and not by
// bytes (one GPU, K-quant planes; V2-Lite's shapes): rows of x owned by workgroups in the second half.
//
// Replaces, for the selected experts e_0..e_{K-1} of a token (src/infer.cpp:853-878, 899-903), the launches of the generic multi-task GEMV:
//     o_k  = W2[e_k] h_k,  x += w_k * o_k  (k order),  x += shared_out        experts_down_kernel
// Lanes per row, column steps, trees of lanes and the order of the combine are the generic launches': the same bits.
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

// v / d for 0 <= v < 2^16 / d (moe_down_plan looks at the range): m = ceil(2^16 / d)
DEV int div_small(int v, int m) { return (v * m) >> 16; }

}  // namespace

// ------------------------------------------------------------------------------------------------------------
// Second half: workgroup b owns rows [b * rows_wg, +rows_wg) of x for ALL slots, so that nothing has to be handed over between workgroups (the
// generic launch deals (slot, rows) to its workgroups and needs a publish, an arrival, an acquire and a read before the last one can add up).  What a
// workgroup needs of it is a chain: the experts' ids, the weights, the multiplies.  Its first waves do that; the others meanwhile read and
// quantise the slots' hidden vectors (12288 values for V2-Lite), so that neither waits for the other's loads.  Bound by latency: 8.3 MB of weights
// are 1.2 us.  V2-Lite (6 of 64 experts of 1536, shared 3072, Q2_K), us a launch: generic 13.2 (224 workgroups of 4 waves, two rows per lane and the
// hand-over), here 7.4; with the arguments read where they are used, two copies of the quantisation and a stack of descriptors 9.6.  A token
// 1460 -> 1303 us.
// ------------------------------------------------------------------------------------------------------------
template <int QT>
__global__ __launch_bounds__(1024) void experts_down_kernel(const float* __restrict__ hb, const int* __restrict__ route_e, const float* __restrict__ route_w,
                                                           float* x, int hb_stride, int K, int cw, const MoeDownArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NW = 16, U = QT == DSK_QUANT_Q2_K ? 6 : 4;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, bid = blockIdx.x;
  uint8_t* act = smem;                                                   // [slot][lds_b] item records
  float* o_s = reinterpret_cast<float*>(smem + (size_t)a.lds_b * (K + 1));  // [slot][rows_wg]
  const int nbR = a.mi >> 8, nbS = a.shared_n >> 8, slots = K + (nbS > 0 ? 1 : 0);
  const int r_lo = bid * a.rows_wg, nrows = min(a.rows_wg, a.dim - r_lo);
  // (everything of the arguments that is needed later is read now, in one trip: where it is used it would be one of its own)
  asm volatile("" ::"s"(a.w2_qs), "s"(a.w2_sc), "s"(a.w2_dm), "s"(a.sw2_qs), "s"(a.sw2_sc), "s"(a.sw2_dm), "s"(a.eout), "s"(a.dim), "s"(a.rows_wg), "s"(a.lpr_log2),
               "s"(a.lds_b), "s"(a.tap_qs));
  float xv = 0.f, rw = 0.f;  // the rows' old values, the slots' weights (the last wave adds up)
  if (wave < cw) {
    const int e_all = route_e[lane < K ? lane : K - 1];
    const int lpr_log2 = a.lpr_log2, RPW = 64 >> lpr_log2;
    const int rloc = lane >> lpr_log2, sub = lane & ((1 << lpr_log2) - 1), q = sub & 3;
    // steps of RPW rows: the shared expert's first (its rows are the longest), then the routed slots' (slot, row) slot-major
    const int WS = nbS > 0 ? (a.rows_wg + RPW - 1) >> (6 - lpr_log2) : 0, WR = (a.rows_wg * K + RPW - 1) >> (6 - lpr_log2);
    ChunkKQ<QT, 1, U, false> c;
    bool wait = true;
    for (int st = wave; st < WS + WR; st += cw) {
      const bool sh = st < WS;  // wave-uniform
      const int v = (sh ? st : st - WS) * RPW + rloc;
      const int slot = sh ? K : min(div_small(v, a.div_rows), K - 1), rr0 = sh ? v : v - slot * a.rows_wg;
      const bool valid = rr0 < nrows;
      const int rr = valid ? rr0 : nrows - 1, nb = sh ? nbS : nbR, items = nb * 4, its = (items + (1 << lpr_log2) - 1) >> lpr_log2;
      const int e = sh ? 0 : __shfl(e_all, slot);
      const int rowblk[1] = {(e * a.dim + r_lo + rr) * nb + (sub >> 2)};
      WPtr P;
      P.present = true; P.qs2 = P.sc2 = P.hm2 = P.dm2 = nullptr; P.scale = P.scale2 = nullptr;
      P.qs = sh ? a.sw2_qs : a.w2_qs; P.sc = sh ? a.sw2_sc : a.w2_sc; P.hm = sh ? a.sw2_hm : a.w2_hm; P.dm = sh ? a.sw2_dm : a.w2_dm;
      const KQRsrc B = kq_rsrc<QT, false>(P);
      const uint8_t* lds_lane = act + (size_t)slot * a.lds_b + sub * ITEM_LDS;
      float acc[1] = {0.f}, dummy[1] = {0.f};
      for (int it0 = 0; it0 < its; it0 += U) {
        load_chunk_kq<QT, 1, U, false>(c, B, its, items, sub, lpr_log2, q, rowblk, it0);
        if (wait) lds_barrier();  // the hidden vectors are staged; this wave's first weights stay on their way
        wait = false;
        compute_chunk_kq<QT, 1, U, false>(c, its, items, sub, lpr_log2, q, it0, lds_lane, acc, dummy);
      }
      const float o = lanes_sum(acc[0], lpr_log2);
      if (sub == 0 && valid) o_s[slot * a.rows_wg + rr] = o;
    }
    if (wait) lds_barrier();
  } else {
    const int sw = NW - cw, nblk = K * nbR + nbS, r16 = lane >> 4, j = lane & 15;
    for (int b0 = (wave - cw) * 4; b0 < nblk; b0 += sw * 8) {  // two groups of four blocks at once
      f32x4 t0[4], t1[4];
      auto request = [&](int bb0, f32x4 (&t)[4]) {
        const int b = min(bb0 + r16, nblk - 1);  // (lanes past the end: the last block again, the same values to the same place)
        const int s = b < K * nbR ? div_small(b, a.div_nb) : K, bb = b - s * nbR;
        const float* src = hb + (size_t)s * hb_stride + bb * 256 + j * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) t[i] = *reinterpret_cast<const f32x4*>(src + 64 * i);
        return act + (size_t)s * a.lds_b + (size_t)bb * 4 * ITEM_LDS;
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
  if (a.tap_qs && bid == 0)  // parity tap: what the slots staged
    for (int s = 0; s < slots; ++s)
      dump_staged_q8_inline<QT == DSK_QUANT_Q2_K>(act + (size_t)s * a.lds_b, s < K ? a.mi : a.shared_n, a.tap_qs + (size_t)s * a.tap_stride,
                                                 a.tap_d + (size_t)s * (a.tap_stride >> 8), tid, 1024);
  lds_barrier();
  if (wave == NW - 1 && lane < nrows) {  // x += w_k * o_k in k order (src/infer.cpp:874-877), then the shared expert (:900-903)
    for (int k = 0; k < slots; ++k) {
      const float o = o_s[k * a.rows_wg + lane];
      a.eout[(size_t)k * a.dim + r_lo + lane] = o;
      if (k < K) xv = fmaf(o, u2f(__builtin_amdgcn_readlane(__builtin_bit_cast(u32, rw), k)), xv);
      else xv += o;
    }
    x[r_lo + lane] = xv;
  }
}

// ---- host side ------------------------------------------------------------------------------------------
int moe_down_plan(MoeDownArgs& a, int n_cus) {
  const bool q2 = a.quant == DSK_QUANT_Q2_K, q3 = a.quant == DSK_QUANT_Q3_K;
  if (!q2 && !q3) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: K-quant planes only");
  if (a.K < 1 || a.K > 15 || a.dim < 1 || a.mi < 256 || a.mi % 256 || a.shared_n % 256 || a.shared_n < 0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: shapes");
  const int lpr = 1 << a.lpr_log2, RPW = 64 / lpr, nbR = a.mi >> 8, nbS = a.shared_n >> 8;
  if (lpr < 4 || lpr > 64 || (nbR * 4) % lpr || (nbS * 4) % lpr) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: %d lanes do not divide the rows", lpr);
  a.rows_wg = (a.dim + n_cus - 1) / n_cus;
  a.grid = (a.dim + a.rows_wg - 1) / a.rows_wg;
  if (a.rows_wg > 64) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: %d rows per workgroup", a.rows_wg);
  // one descriptor spans the stack: a lane's byte offset (expert, row, block) must fit its 32-bit offset field
  if ((double)a.n_experts * a.dim * nbR * 64.0 >= 2147483648.0 || (double)a.dim * nbS * 64.0 >= 2147483648.0)
    DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: a stack exceeds the 31-bit offset of a buffer load");
  a.div_nb = (65536 + nbR - 1) / nbR;
  a.div_rows = (65536 + a.rows_wg - 1) / a.rows_wg;
  // (v * ceil(2^16 / d) >> 16 == v / d while v * (d - 1) < 2^16)
  const long nblk = (long)a.K * nbR + nbS, nv = (long)a.K * a.rows_wg + RPW;
  if (nblk * (nbR - 1) >= 65536 || nv * (a.rows_wg - 1) >= 65536 || nblk >= 32768) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_down: too many blocks");
  const int nB = nbR > nbS ? nbR : nbS;
  a.lds_b = nB * 4 * ITEM_LDS;
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
  if (a.quant == DSK_QUANT_Q2_K) go(experts_down_kernel<DSK_QUANT_Q2_K>);
  else go(experts_down_kernel<DSK_QUANT_Q3_K>);
  return DSK_OK;
}
