// kernels_chunk_scan.hip -- the recurrences of layered models over chunks of 16 tokens, as 32-bit matrix products.
//
// Inside a chunk that starts from the state S0 [dim][vdim], with G_t the product of the decays of its tokens up to t (per key channel)
// and all ratios of such products taken as products of the decays in between (they are at most 1: nothing overflows):
//   delta rule   u_t = beta_t (v_t - (k_t G_t)^T S0 - sum_{s<t} A_ts u_s),    A_ts = sum_d k_t k_s G_t / G_s
//                o_t = (q_t G_t)^T S0 + sum_{s<=t} B_ts u_s,                  B_ts = sum_d q_t k_s G_t / G_s
//                S  <- G_16 S0 + sum_s (k_s G_16 / G_s) u_s^T
//   mLSTM        the same without A (u = v); the decay is one number per token, exp(f + m_before - m), and k_s carries exp(i_s - m_s).
//                A column of ones behind v makes the normaliser n one more column of S.
//   wkv          the same without A, read before the write: o_t = (q_t G_(t-1))^T S0 + sum_{s<=t} B_ts v_s with B_ts = sum_d q_t k_s
//                G_(t-1) / G_s below the diagonal, and the bonus on it: B_tt = sum_d q_t u k_t
// *_prepare: everything that does not depend on S0, for all chunks at once - the operands with decays multiplied in, B, and
// T = (I + diag(beta) A)^-1 diag(beta), so that U = T (V - Kg S0).  chunk_scan: one workgroup per (16 columns, head, sequence)
// goes through the chunks; 4 waves share the key channels, a fifth forms the outputs.  S stays in MFMA accumulators: their layout (column = lane % 16, rows
// 4 (lane / 16) + i) is an operand layout of v_mfma_f32_16x16x4_f32 when step i stands for the k values {4 g + i}.
#include "layered_kernels.h"
#include "seq_device.h"

#include <math.h>

static int cdiv(int a, int b) { return (a + b - 1) / b; }
enum { CH = RECUR_CHUNK };

struct Ops {  // one chunk's operands of one head
  float *kg, *qg, *ke, *gend, *t, *b;
};
DEV Ops ops_at(float* base, size_t chunk, int heads, int h, int dim) {
  const int dp = (dim + 15) / 16 * 16;
  Ops o;
  o.kg = base + (chunk * heads + h) * (49 * (size_t)dp + 512);
  o.qg = o.kg + 16 * dp;
  o.ke = o.qg + 16 * dp;
  o.gend = o.ke + 16 * dp;
  o.t = o.gend + dp;
  o.b = o.t + 256;
  return o;
}

// Operands of a chunk come in by whole rows: wave w takes tokens w, w + 4, ... and 64 channels at a time, two times that at once.  load(t, d) reads one
// that is there (behind a branch the compiler waits for each load), keep(place, there, values) puts it into LDS.  The same holds for what is read from LDS
// behind: all decays of a channel first, then the sums over them.  2048 tokens, 16 heads of 128 (delta rule) 52 us with a branch at each, 37.5 so, 301 tokens
// 20.7 and 13.0; 1996 tokens, 32 heads of 64 (wkv) 37 and 30; 2048 tokens of mLSTM 18 and 13.9.
template <typename V, typename L, typename K>
DEV void by_rows(int n, int dim, int dp, L load, K keep) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  for (int d0 = lane; d0 < dp; d0 += 128) {
    V v[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[i][u] = load(min(wave + 4 * u, n - 1), min(d0 + 64 * i, dim - 1));
    __builtin_amdgcn_sched_barrier(0);  // (all on their way first)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (d0 + 64 * i < dp) keep((wave + 4 * u) * dp + d0 + 64 * i, wave + 4 * u < n && d0 + 64 * i < dim, v[i][u]);
  }
}

// ---- delta rule: operands -----------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void delta_prepare_kernel(const DeltaArgs a, float* __restrict__ base) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x, h = blockIdx.y, dim = a.dim, dp = (dim + 15) / 16 * 16;
  float *sk = lds, *sq = sk + 16 * dp, *sg = sq + 16 * dp, *sA = sg + 16 * dp, *sb = sA + 16 * 17;
  const SeqDesc s = seq_at(a.p.seqs + a.p.chunk[2 * blockIdx.x]);
  const int t0 = a.p.chunk[2 * blockIdx.x + 1], n = min((int)CH, s.len - t0);
  const int kv = h / (a.heads / a.kv_heads), nq = a.kv_heads * dim;
  const size_t row0 = (size_t)s.row0 + t0;
  struct In {
    float k, q, g;
  };
  const float *K = a.k + row0 * nq + (size_t)kv * dim, *Q = a.q + row0 * nq + (size_t)kv * dim, *G = a.head_decay ? a.g + row0 * a.heads + h : a.g + row0 * a.heads * dim + (size_t)h * dim;
  const int ld_g = a.head_decay ? a.heads : a.heads * dim, one = a.head_decay ? 0 : 1;
  by_rows<In>(n, dim, dp, [&](int t, int d) { return In{K[(size_t)t * nq + d], Q[(size_t)t * nq + d], G[(size_t)t * ld_g + d * one]}; },
              [&](int i, bool in, const In& v) {  // rows past the end: no key, no query, no decay
                sk[i] = in ? v.k : 0.f;
                sq[i] = in ? v.q : 0.f;
                sg[i] = in ? v.g : 1.f;
              });
  if (tid < 16) sb[tid] = tid < n ? a.beta[(row0 + tid) * a.heads + h] : 0.f;
  __syncthreads();
  const Ops o = ops_at(base, blockIdx.x, a.heads, h, dim);
  for (int d = tid & 127; d < dp; d += 128) {  // (half of the waves go forwards, half backwards)
    if (tid < 128) {
      float G = 1.f;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        G *= sg[t * dp + d];
        o.kg[t * dp + d] = sk[t * dp + d] * G;
        o.qg[t * dp + d] = sq[t * dp + d] * G;
      }
      o.gend[d] = G;
      continue;
    }
    float E = 1.f, e[16];
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      e[t] = sk[t * dp + d] * E;
      E *= sg[t * dp + d];
    }
#pragma unroll
    for (int t = 0; t < 16; t += 4) *reinterpret_cast<f32x4*>(o.ke + (size_t)d * 16 + t) = f32x4{e[t], e[t + 1], e[t + 2], e[t + 3]};
  }
  // A and B: thread -> (token s, every 16th channel), all later tokens t in registers
  const int sx = tid >> 4, dg = tid & 15;
  float aA[16], aB[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) aA[t] = aB[t] = 0.f;
  for (int d = dg; d < dp; d += 16) {
    float w = 0.f, k[16], q[16], g[16];
    const float ks = sk[sx * dp + d];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      k[t] = sk[t * dp + d];
      q[t] = sq[t * dp + d];
      g[t] = sg[t * dp + d];
    }
    __builtin_amdgcn_sched_barrier(0);  // (else the compiler reads a decay behind a branch, and waits for each)
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      w *= g[t];
      w = t == sx ? ks : w;
      aA[t] += k[t] * w;
      aB[t] += q[t] * w;
    }
  }
  float A = 0.f, B = 0.f;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const float At = row_sum(aA[t]), Bt = row_sum(aB[t]);
    A = dg == t ? At : A;
    B = dg == t ? Bt : B;
  }
  sA[dg * 17 + sx] = A;
  o.b[dg * 16 + sx] = sx <= dg ? B : 0.f;
  __syncthreads();
  if (tid < 16) {  // column tid of T, by forward substitution: x[t], then its part of every later row
    float r[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) r[t] = 0.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const float x = sb[t] * ((t == tid ? 1.f : 0.f) - r[t]);
      o.t[t * 16 + tid] = x;
#pragma unroll
      for (int u = t + 1; u < 16; ++u) r[u] += sA[u * 17 + t] * x;
    }
  }
}

// ---- mLSTM: running maximum, operands --------------------------------------------------------------------------
// m_t = max(f_t + m_(t-1), i_t) composes: (F, I) then (f, i) = (F + f, max(I + f, i)); one workgroup per (head, sequence), a wave per 64 tokens.
// What bounds it is the chain of a wave's turn (gates, six exchanges that depend on each other, exponentials), not bytes, and only its last sum and
// maximum depend on the tokens before: the waves make their turns side by side and hand the two numbers on through LDS.  2048 tokens, 16 heads, a
// wave taking all turns one after the other: 43 us (37 with its loads requested two turns ahead), so 13; the sums are formed in the same order.
enum { GATE_WAVES = 16 };
__global__ __launch_bounds__(64 * GATE_WAVES) void mlstm_gates_kernel(const MlstmArgs a, const ChunkScan c) {
  __shared__ float tot[2][GATE_WAVES][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.x;
  const SeqDesc s = seq_at(a.p.seqs + blockIdx.y);
  float* M = reinterpret_cast<float*>(s.state + a.off_m) + h;
  float m = s.pos0 > 0 ? M[s.flip * a.heads] : 0.f;
  for (int t0 = 0, buf = 0; t0 < s.len; t0 += 64 * GATE_WAVES, buf ^= 1) {
    const int t = t0 + tid;
    const bool in = t < s.len;
    const size_t row = (size_t)s.row0 + (in ? t : 0);
    const float* G = a.gate_f + row * a.ld_gate;
    const float i = in ? a.gate_cap * tanhf((G[a.col_i + h] + a.b_i[h]) / a.gate_cap) : -INFINITY;
    const float f = in ? logsigmoid_f(a.gate_cap * tanhf((G[a.col_f + h] + a.b_f[h]) / a.gate_cap)) : 0.f;
    float F = f, I = i;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float pF = __shfl_up(F, off), pI = __shfl_up(I, off);
      if (lane >= off) {
        I = fmaxf(pI + F, I);
        F += pF;
      }
    }
    if (lane == 63) {
      tot[buf][wave][0] = F;
      tot[buf][wave][1] = I;
    }
    __syncthreads();  // (two buffers: the next turn's numbers go beside these)
    const int turns = min((int)GATE_WAVES, (s.len - t0 + 63) >> 6);
    float mine = m;  // in front of this wave's turn
    for (int w = 0; w < turns; ++w) {
      if (w == wave) mine = m;
      m = fmaxf(tot[buf][w][0] + m, tot[buf][w][1]);  // (lanes past the end carry it on)
    }
    const float mt = fmaxf(F + mine, I);
    float before = __shfl_up(mt, 1);
    if (lane == 0) before = mine;
    if (in) {
      c.keep[row * a.heads + h] = expf(fminf(f + before - mt, 0.f));
      c.add[row * a.heads + h] = expf(fminf(i - mt, 0.f));
      c.floor[row * a.heads + h] = expf(-mt);
    }
  }
  if (tid == 0) M[(s.flip ^ 1) * a.heads] = m;
}
template <typename T>
__global__ __launch_bounds__(256) void mlstm_prepare_kernel(const MlstmArgs a, const ChunkScan c) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x, h = blockIdx.y, dim = a.dim, dp = (dim + 15) / 16 * 16;
  float *sk = lds, *sq = sk + 16 * dp, *keep = sq + 16 * dp, *add = keep + 16;
  const SeqDesc s = seq_at(a.p.seqs + a.p.chunk[2 * blockIdx.x]);
  const int t0 = a.p.chunk[2 * blockIdx.x + 1], n = min((int)CH, s.len - t0);
  const size_t row0 = (size_t)s.row0 + t0;
  struct In {
    T k, q;
  };
  const T* P = reinterpret_cast<const T*>(a.proj_t) + row0 * a.ld + h * dim;
  by_rows<In>(n, dim, dp, [&](int t, int d) { return In{P[(size_t)t * a.ld + a.col_k + d], P[(size_t)t * a.ld + a.col_q + d]}; },
              [&](int i, bool in, const In& v) {
                sk[i] = in ? (float)v.k : 0.f;
                sq[i] = in ? (float)v.q * a.q_scale : 0.f;
              });
  if (tid < 16) {
    keep[tid] = tid < n ? c.keep[(row0 + tid) * a.heads + h] : 1.f;
    add[tid] = tid < n ? c.add[(row0 + tid) * a.heads + h] : 0.f;
  }
  __syncthreads();
  const Ops o = ops_at(c.ops, blockIdx.x, a.heads, h, dim);
  for (int d = tid & 127; d < dp; d += 128) {
    if (tid < 128) {
      float G = 1.f;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        G *= keep[t];
        o.qg[t * dp + d] = sq[t * dp + d] * G;
      }
      o.gend[d] = G;
      continue;
    }
    float E = 1.f, e[16];
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      e[t] = sk[t * dp + d] * add[t] * E;
      E *= keep[t];
    }
#pragma unroll
    for (int t = 0; t < 16; t += 4) *reinterpret_cast<f32x4*>(o.ke + (size_t)d * 16 + t) = f32x4{e[t], e[t + 1], e[t + 2], e[t + 3]};
  }
  const int sx = tid >> 4, dg = tid & 15;
  float acc[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) acc[t] = 0.f;
  for (int d = dg; d < dp; d += 16) {
    const float ks = sk[sx * dp + d];
#pragma unroll
    for (int t = 0; t < 16; ++t) acc[t] += sq[t * dp + d] * ks;
  }
  float w = 0.f, B = 0.f;
  const float own = add[sx];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    w *= keep[t];
    w = t == sx ? own : w;
    const float Bt = row_sum(acc[t]) * w;
    B = dg == t ? Bt : B;
  }
  o.b[dg * 16 + sx] = sx <= dg ? B : 0.f;
}

// ---- wkv: operands ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void wkv_prepare_kernel(const WkvArgs a, float* __restrict__ base) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x, h = blockIdx.y, dim = a.dim, dp = (dim + 15) / 16 * 16;
  float *sk = lds, *sq = sk + 16 * dp, *sg = sq + 16 * dp, *su = sg + 16 * dp;
  const SeqDesc s = seq_at(a.p.seqs + a.p.chunk[2 * blockIdx.x]);
  const int t0 = a.p.chunk[2 * blockIdx.x + 1], n = min((int)CH, s.len - t0);
  const size_t row0 = (size_t)s.row0 + t0;
  struct In {
    T k, r;
    float low, w0;
  };
  const T* P = reinterpret_cast<const T*>(a.proj_t) + row0 * a.ld + h * dim;
  const float *low = a.low_f + row0 * a.ld_low + h * dim, *w0 = a.w0 + h * dim;
  by_rows<In>(n, dim, dp, [&](int t, int d) { return In{P[(size_t)t * a.ld + a.col_k + d], P[(size_t)t * a.ld + a.col_r + d], low[(size_t)t * a.ld_low + d], w0[d]}; },
              [&](int i, bool in, const In& v) {  // rows past the end: no key, no query, no decay
                sk[i] = in ? (float)v.k : 0.f;
                sq[i] = in ? (float)v.r : 0.f;
                sg[i] = in ? expf(-expf(v.low + v.w0)) : 1.f;
              });
  for (int d = tid; d < dp; d += 256) su[d] = d < dim ? a.u[h * dim + d] : 0.f;
  __syncthreads();
  const Ops o = ops_at(base, blockIdx.x, a.heads, h, dim);
  for (int d = tid & 127; d < dp; d += 128) {
    if (tid < 128) {
      float G = 1.f;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        o.qg[t * dp + d] = sq[t * dp + d] * G;
        G *= sg[t * dp + d];
      }
      o.gend[d] = G;
      continue;
    }
    float E = 1.f, e[16];
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      e[t] = sk[t * dp + d] * E;
      E *= sg[t * dp + d];
    }
#pragma unroll
    for (int t = 0; t < 16; t += 4) *reinterpret_cast<f32x4*>(o.ke + (size_t)d * 16 + t) = f32x4{e[t], e[t + 1], e[t + 2], e[t + 3]};
  }
  const int sx = tid >> 4, dg = tid & 15;
  float acc[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) acc[t] = 0.f;
  for (int d = dg; d < dp; d += 16) {
    float w = 0.f, q[16], g[16];
    const float ks = sk[sx * dp + d], bonus = ks * su[d];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      q[t] = sq[t * dp + d];
      g[t] = sg[t * dp + d];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const float p = t == sx ? bonus : w;
      acc[t] = t < 15 ? fmaf(q[t], p, acc[t]) : acc[t] + product(q[t], p);  // (the last row's have always been rounded: results stay what they are)
      w *= g[t];
      w = t == sx ? ks : w;
    }
  }
  float B = 0.f;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const float Bt = row_sum(acc[t]);
    B = dg == t ? Bt : B;
  }
  o.b[dg * 16 + sx] = sx <= dg ? B : 0.f;
}

// ---- the chunks of a sequence, one after the other -------------------------------------------------------------
struct ScanArgs {
  PassDesc p;
  int heads, dim, vdim;
  float* ops;
  const void* v;       // delta: floats [rows][heads * vdim]; mLSTM: proj_t + col_v
  int ld_v;
  float* o;            // [rows][heads][cols]
  size_t off_s, off_n;
};
enum { SCAN_DELTA, SCAN_MLSTM, SCAN_WKV };
enum { SCAN_WAVES = 5 };  // four that share the key channels, one for the outputs
typedef __amdgpu_buffer_rsrc_t rsrc_t;
DEV const char* uniform_ptr(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  return (const char*)(((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(v >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((unsigned)v));
}
DEV rsrc_t buffer_of(const char* p, int bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, bytes, 0x00020000); }
DEV f32x4 load4(rsrc_t r, int off, int base) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, base, 0)); }
template <typename T>
DEV float load1(rsrc_t r, int off) {
  if constexpr (sizeof(T) == 2) return __builtin_bit_cast(float, (unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0) << 16);
  else return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
// One chunk after the other: what bounds it is a chunk's chain - W over a wave's key channels, the exchange of its four parts through LDS, U, the update
// of S - so everything else is taken off it.  The outputs are a fifth wave's work, a chunk behind and out of LDS alone: a wave that stores and
// loads waits for its stores (mLSTM: 77 us with its loads in that wave, 47 without).  Their half of S0's products is issued in the shadow of the
// exchange.  Operands come as buffer loads whose offsets stay in registers (a chunk costs scalar additions), a chunk or two ahead
// (NB; more gained nothing), and the waits count: no step of the loop may be skipped behind another, and a wave's tiles are all there
// (FULL) or tested.  All columns of a head read the same operands: an XCD takes a range of (head, sequence, columns) in this order, so
// that its L2 gets them once and every XCD has a share of each sequence.  (With the sequence in front a long one had two XCDs to itself, two
// workgroups to a compute unit, and the others waited: 900, 300 and 100 tokens, delta rule of 16 heads 115 us, 63 in this order; 331, 700, 64 and 901
// tokens 129, now 102.)  Three waves a SIMD: two workgroups share a compute unit.
// In prompts' passes, with the outputs in turn by the four waves -> now: 2048 tokens, 16 heads: delta rule of 128 x 128 190 -> 133 us, mLSTM of
// 64 x 129 110 -> 52; those four sequences: delta rule 126 -> 102, wkv of 32 heads of 64 x 64 63 -> 42; 64 heads, 400, 333, 400 and 350 tokens: delta
// rule 283 -> 290 (the card is full either way), wkv of 112 heads 84 -> 72.
template <typename T, int KIND, int NTL, bool FULL>
__global__ __launch_bounds__(64 * SCAN_WAVES) __attribute__((amdgpu_waves_per_eu(NTL > 2 ? 2 : 3))) void chunk_scan_kernel(const ScanArgs a) {
  constexpr bool DELTA = KIND == SCAN_DELTA, NORM = KIND == SCAN_MLSTM;
  constexpr int NB = NTL > 1 ? 2 : 3;
  __shared__ __attribute__((aligned(16))) f32x4 ex_w[DELTA ? 2 : 1][4][64], ex_x[2][4][64], ex_u[2][64], ex_b[2][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c16 = lane & 15;
  const int dp = (a.dim + 15) / 16 * 16, tiles = dp >> 4;
  const int cols = NORM ? a.vdim + 1 : a.vdim, col_tiles = (cols + 15) >> 4;
  const int place = xcd_range(blockIdx.x, gridDim.x), hs = place / col_tiles, h = hs / a.p.n_seqs;
  const int col = (place - hs * col_tiles) * 16 + c16;
  const bool live = col < cols, norm = NORM && col == a.vdim;
  const SeqDesc s = seq_at(a.p.seqs + (hs - h * a.p.n_seqs));
  const int nc = (s.len + CH - 1) / CH;
  // this sequence's and head's operands and values, chunk by chunk (chunks behind the last: the last again)
  const int ops_bytes = (49 * dp + 512) * 4, ld = a.ld_v * (int)sizeof(T);
  const char* ops0 = uniform_ptr(a.ops) + ((size_t)__builtin_amdgcn_readfirstlane(s.chunk0) * a.heads + h) * ops_bytes;
  const char* v0 = uniform_ptr(a.v) + (size_t)__builtin_amdgcn_readfirstlane(s.row0) * ld + (size_t)h * a.vdim * sizeof(T);
  auto ops_of = [&](int c) { return buffer_of(ops0 + (size_t)min(c, nc - 1) * a.heads * ops_bytes, ops_bytes); };
  auto v_of = [&](int c) {  // (rows past the sequence's end read zero, and columns behind the last one's values compute something nobody stores)
    c = min(c, nc - 1);
    return buffer_of(v0 + (size_t)c * CH * ld, (min((int)CH, s.len - c * CH) - 1) * ld + a.vdim * (int)sizeof(T));
  };
  const int vcol = min(col, a.vdim - 1), v_off = g * 4 * ld + vcol * (int)sizeof(T), small_off = (c16 * 16 + g * 4) * 4;
  const int at_q = 64 * dp, at_ke = 128 * dp, at_g = 192 * dp, at_t = 196 * dp, at_b = 196 * dp + 1024;

  if (wave == 4) {  // the outputs of a chunk: O = the parts of (q G)^T S0 + B U, everything out of LDS: behind its stores this wave waits for no load
    const int row_bytes = a.heads * cols * 4;
    const char* o0 = uniform_ptr(a.o) + (size_t)__builtin_amdgcn_readfirstlane(s.row0) * row_bytes + (size_t)h * cols * 4;
    const int o_off = live ? g * 4 * row_bytes + col * 4 : 0x7ff00000;  // (out of every range: not stored, like the rows past the end)
    lds_barrier();
    for (int c = 0; c < nc; ++c) {
      lds_barrier();  // that of chunk c + 1: what chunk c's waves wrote behind theirs is here
      const f32x4 U = ex_u[c & 1][lane], B = ex_b[c & 1][lane];
      f32x4 O = (ex_x[c & 1][0][lane] + ex_x[c & 1][1][lane]) + (ex_x[c & 1][2][lane] + ex_x[c & 1][3][lane]);
#pragma unroll
      for (int e = 0; e < 4; ++e) O = __builtin_amdgcn_mfma_f32_16x16x4f32(B[e], U[e], O, 0, 0, 0);
      const rsrc_t r = buffer_of(o0 + (size_t)c * CH * row_bytes, (min((int)CH, s.len - c * CH) - 1) * row_bytes + cols * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = O[e];  // (a bit cast of an element of a vector in place takes the first one)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, o_off + e * row_bytes, 0, 0);
      }
    }
    return;
  }

  float* S0 = reinterpret_cast<float*>(s.state + a.off_s) + (size_t)h * a.dim * a.vdim;
  float* N0 = !NORM ? nullptr : reinterpret_cast<float*>(s.state + a.off_n) + (size_t)h * a.dim;
  const size_t nn = (size_t)a.heads * a.dim;
  f32x4 S[NTL];
  int k_off[NTL], ke_off[NTL], g_off[NTL];
#pragma unroll
  for (int i = 0; i < NTL; ++i) {
    const int tile = FULL ? wave + 4 * i : min(wave + 4 * i, tiles - 1);
    k_off[i] = (c16 * dp + tile * 16 + g * 4) * 4;
    ke_off[i] = ((tile * 16 + c16) * 16 + g * 4) * 4;
    g_off[i] = (tile * 16 + g * 4) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = (wave + 4 * i) * 16 + g * 4 + e;
      S[i][e] = s.pos0 > 0 && live && k < a.dim ? (norm ? N0[s.flip * nn + k] : S0[(size_t)k * a.vdim + col]) : 0.f;
    }
  }
  struct Operands {
    f32x4 kg[NTL], qg[NTL], ke[NTL], ge[NTL], t, b;
    float v[4];
  };
  auto load = [&](int c, Operands& x) {
    const rsrc_t o = ops_of(c), r = v_of(c);
#pragma unroll
    for (int i = 0; i < NTL; ++i)
      if (DELTA) x.kg[i] = load4(o, k_off[i], 0);
#pragma unroll
    for (int i = 0; i < NTL; ++i) x.qg[i] = load4(o, k_off[i], at_q);
#pragma unroll
    for (int e = 0; e < 4; ++e) x.v[e] = load1<T>(r, v_off + e * ld);
    if (DELTA) x.t = load4(o, small_off, at_t);
    x.b = load4(o, small_off, at_b);
#pragma unroll
    for (int i = 0; i < NTL; ++i) {
      x.ke[i] = load4(o, ke_off[i], at_ke);
      x.ge[i] = load4(o, g_off[i], at_g);
    }
  };
  auto step = [&](int c, Operands& x) {  // ... and requests the operands of chunk c + NB into x
    f32x4 W = {0.f, 0.f, 0.f, 0.f}, X = {0.f, 0.f, 0.f, 0.f};
    if (DELTA) {
#pragma unroll
      for (int i = 0; i < NTL; ++i)
        if (FULL || wave + 4 * i < tiles)
#pragma unroll
          for (int e = 0; e < 4; ++e) W = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kg[i][e], S[i][e], W, 0, 0, 0);
      ex_w[c & 1][wave][lane] = W;
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < NTL; ++i)
      if (FULL || wave + 4 * i < tiles)
#pragma unroll
        for (int e = 0; e < 4; ++e) X = __builtin_amdgcn_mfma_f32_16x16x4f32(x.qg[i][e], S[i][e], X, 0, 0, 0);
    lds_barrier();  // (the operands of the next chunks stay in flight)
    f32x4 U;
#pragma unroll
    for (int e = 0; e < 4; ++e) U[e] = norm ? 1.f : x.v[e];
    if (DELTA) {
      W = (ex_w[c & 1][0][lane] + ex_w[c & 1][1][lane]) + (ex_w[c & 1][2][lane] + ex_w[c & 1][3][lane]);
      const f32x4 r = U - W;
      U = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) U = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t[e], r[e], U, 0, 0, 0);
    }
    ex_x[c & 1][wave][lane] = X;
#pragma unroll
    for (int i = 0; i < NTL; ++i)
      if (FULL || wave + 4 * i < tiles) S[i] *= x.ge[i];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
      if (FULL || wave + 4 * i < tiles)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.ke[i][e], U[e], S[i], 0, 0, 0);
    if (wave == (c & 3)) {
      ex_u[c & 1][lane] = U;
      ex_b[c & 1][lane] = x.b;
    }
    load(c + NB, x);
  };
  Operands x[NB];
#pragma unroll
  for (int u = 0; u < NB; ++u) load(u, x[u]);
  int c = 0;
  for (; c + NB <= nc; c += NB)
#pragma unroll
    for (int u = 0; u < NB; ++u) step(c + u, x[u]);
#pragma unroll
  for (int u = 0; u + 1 < NB; ++u)
    if (c + u < nc) step(c + u, x[u]);
  lds_barrier();  // (the last chunk's outputs)
#pragma unroll
  for (int i = 0; i < NTL; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = (wave + 4 * i) * 16 + g * 4 + e;
      if (!live || k >= a.dim) continue;
      if (norm) N0[(s.flip ^ 1) * nn + k] = S[i][e];
      else S0[(size_t)k * a.vdim + col] = S[i][e];
    }
}

// ---- launches ------------------------------------------------------------------------------------------------------
template <typename T, int KIND>
static int scan_t(hipStream_t st, const ScanArgs& a) {
  if (a.dim < 1 || a.dim > RECUR_MAX_DIM) DSK_FAIL(DSK_ERR_UNSUPPORTED, "recurrence: key size %d (max %d)", a.dim, (int)RECUR_MAX_DIM);
  const dim3 grid((unsigned)cdiv(KIND == SCAN_MLSTM ? a.vdim + 1 : a.vdim, 16) * a.heads * a.p.n_seqs);
  const int tiles = cdiv(a.dim, 16);
  if (tiles == 4) hipLaunchKernelGGL((chunk_scan_kernel<T, KIND, 1, true>), grid, dim3(64 * SCAN_WAVES), 0, st, a);
  else if (tiles < 4) hipLaunchKernelGGL((chunk_scan_kernel<T, KIND, 1, false>), grid, dim3(64 * SCAN_WAVES), 0, st, a);
  else if (tiles == 8) hipLaunchKernelGGL((chunk_scan_kernel<T, KIND, 2, true>), grid, dim3(64 * SCAN_WAVES), 0, st, a);
  else if (tiles < 8) hipLaunchKernelGGL((chunk_scan_kernel<T, KIND, 2, false>), grid, dim3(64 * SCAN_WAVES), 0, st, a);
  else hipLaunchKernelGGL((chunk_scan_kernel<T, KIND, 4, false>), grid, dim3(64 * SCAN_WAVES), 0, st, a);
  return DSK_OK;
}
int launch_delta_chunks(hipStream_t st, const DeltaArgs& a, const ChunkScan& c) {
  const int dp = (a.dim + 15) / 16 * 16;
  const size_t lds = ((size_t)48 * dp + 16 * 17 + 16) * 4;
  HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(delta_prepare_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(delta_prepare_kernel, dim3(a.p.n_chunks, a.heads), dim3(256), lds, st, a, c.ops);
  return scan_t<float, SCAN_DELTA>(st, ScanArgs{a.p, a.heads, a.dim, a.vdim, c.ops, a.v, a.heads * a.vdim, a.o, a.off_s, 0});
}
template <typename T>
static int mlstm_t(hipStream_t st, const MlstmArgs& a, const ChunkScan& c) {
  const int dp = (a.dim + 15) / 16 * 16;
  hipLaunchKernelGGL(mlstm_gates_kernel, dim3(a.heads, a.p.n_seqs), dim3(64 * GATE_WAVES), 0, st, a, c);
  hipLaunchKernelGGL(mlstm_prepare_kernel<T>, dim3(a.p.n_chunks, a.heads), dim3(256), ((size_t)32 * dp + 32) * 4, st, a, c);
  return scan_t<T, SCAN_MLSTM>(st, ScanArgs{a.p, a.heads, a.dim, a.vdim, c.ops, reinterpret_cast<const T*>(a.proj_t) + a.col_v, a.ld, a.o, a.off_s, a.off_n});
}
int launch_mlstm_chunks(hipStream_t st, const MlstmArgs& a, const ChunkScan& c, bool f32) { return f32 ? mlstm_t<float>(st, a, c) : mlstm_t<bf16>(st, a, c); }
template <typename T>
static int wkv_t(hipStream_t st, const WkvArgs& a, const ChunkScan& c) {
  if (a.dim > RECUR_MAX_DIM) DSK_FAIL(DSK_ERR_UNSUPPORTED, "wkv: key size %d (max %d)", a.dim, (int)RECUR_MAX_DIM);
  const int dp = (a.dim + 15) / 16 * 16;
  hipLaunchKernelGGL(wkv_prepare_kernel<T>, dim3(a.p.n_chunks, a.heads), dim3(256), (size_t)49 * dp * 4, st, a, c.ops);
  return scan_t<T, SCAN_WKV>(st, ScanArgs{a.p, a.heads, a.dim, a.dim, c.ops, reinterpret_cast<const T*>(a.proj_t) + a.col_v, a.ld, a.o, a.off_s, 0});
}
int launch_wkv_chunks(hipStream_t st, const WkvArgs& a, const ChunkScan& c, bool f32) { return f32 ? wkv_t<float>(st, a, c) : wkv_t<bf16>(st, a, c); }
