// kernels_misc.hip -- everything on the decode path that is not a weight-streaming GEMV:
// Q8_K activation quantisation, RMSNorm (+ residual / MoE combine), RoPE + KV-cache writes,
// decode attention (MHA and latent MLA), the MoE router + top-k gate, embedding-row dequant,
// upload-time re-layout of K-quant blocks, synthetic-weight fills and the bandwidth probe.
#include "dsk_internal.h"
#include "router_device.h"
#include <math.h>

typedef unsigned int u32;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
#define DEV __device__ __forceinline__

DEV float h2f(unsigned short b) { return (float)__builtin_bit_cast(_Float16, b); }
DEV unsigned short f2h(float f) { return __builtin_bit_cast(unsigned short, (_Float16)f); }  // RNE like _cvtss_sh(x,0), src/codec.h:26-27

DEV float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += lane_xor(v, off);
  return v;
}
DEV float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, lane_xor(v, off));
  return v;
}
// block-wide reductions through a small LDS scratch (deterministic order); all threads get the result
DEV float block_sum(float v, float* scratch, int tid, int nthreads) {
  v = wave_sum(v);
  const int nw = nthreads >> 6;
  __syncthreads();
  if ((tid & 63) == 0) scratch[tid >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += scratch[i];
  return t;
}
DEV float block_max(float v, float* scratch, int tid, int nthreads) {
  v = wave_max(v);
  const int nw = nthreads >> 6;
  __syncthreads();
  if ((tid & 63) == 0) scratch[tid >> 6] = v;
  __syncthreads();
  float t = scratch[0];
  for (int i = 1; i < nw; ++i) t = fmaxf(t, scratch[i]);
  return t;
}

// ------------------------------------------------------------------------------------
// Q8_K quantisation of one 256-block by one wave (lane holds elements 4*lane..4*lane+3).
// quantize_row_q8_K_ref, src/quant.cpp:616-653: max = signed value of the FIRST element
// with the largest |x|; iscale = -127/max (IEEE divide); q = min(127, rne(iscale*x));
// bsums over 16; d = 1/iscale, which the reference's -ffast-math build evaluates as
// max * (1/-127) (see oracle/dsk_oracle.c).
// ------------------------------------------------------------------------------------
DEV void q8k_block(const float (&v)[4], int lane, int8_t* qs_blk, float* d_out, int16_t* bsums_blk) {
  float amax = 0.f, vmax = 0.f;
  int imax = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float ax = fabsf(v[i]);
    if (ax > amax) { amax = ax; vmax = v[i]; imax = lane * 4 + i; }
  }
  if (amax == 0.f) imax = lane * 4;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float oa = lane_xor(amax, off), ov = lane_xor(vmax, off);
    const int oi = lane_xor(imax, off);
    if (oa > amax || (oa == amax && oi < imax)) { amax = oa; vmax = ov; imax = oi; }
  }
  int q[4] = {0, 0, 0, 0};
  float d = 0.f;
  if (amax != 0.f) {
    const float iscale = __fdiv_rn(-127.f, vmax);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = (int)rintf(__fmul_rn(iscale, v[i]));
      q[i] = r < 127 ? r : 127;
    }
    d = __fmul_rn(vmax, 1.0f / -127.f);
  }
  const u32 packed = (u32)(q[0] & 0xff) | ((u32)(q[1] & 0xff) << 8) | ((u32)(q[2] & 0xff) << 16) | ((u32)(q[3] & 0xff) << 24);
  reinterpret_cast<u32*>(qs_blk)[lane] = packed;
  int s = q[0] + q[1] + q[2] + q[3];
  s += lane_xor(s, 1);
  s += lane_xor(s, 2);
  if ((lane & 3) == 0) bsums_blk[lane >> 2] = (int16_t)s;
  if (lane == 0) *d_out = d;
}

__global__ __launch_bounds__(256) void quantize_q8k_kernel(const float* __restrict__ x, int nb, int8_t* qs, float* d, int16_t* bsums) {
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= nb) return;
  const f32x4 t = *reinterpret_cast<const f32x4*>(x + (size_t)b * 256 + lane * 4);
  const float v[4] = {t.x, t.y, t.z, t.w};
  q8k_block(v, lane, qs + (size_t)b * 256, d + b, bsums + (size_t)b * 16);
}

// stand-alone MoE combine of the expert-sharded path (after the all-reduce of the slot outputs)
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ x, const float* __restrict__ eout, const float* __restrict__ w,
                                                          int n_slots, int add_shared, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float xv = x[i];
  for (int k = 0; k < n_slots; ++k) xv = fmaf(eout[(size_t)k * n + i], w[k], xv);
  if (add_shared) xv += eout[(size_t)n_slots * n + i];
  x[i] = xv;
}
int launch_moe_combine(hipStream_t st, float* x, const float* eout, const float* weights, int n_slots, int add_shared, int n) {
  hipLaunchKernelGGL(moe_combine_kernel, dim3((n + 255) / 256), dim3(256), 0, st, x, eout, weights, n_slots, add_shared, n);
  return DSK_OK;
}

// ... after the ALL-GATHER form of the exchange (option "exchange_allgather"): gathered[r] holds rank r's n_slots slot rows, of
// which only the rows of the experts r owns mean anything; slot k is read from the rank that owns expert experts[k]
// (dsk_expert_owner: e / per, per = ceil(E / world)), the shared expert's row from this rank's own buffer.  Same k-ordered
// multiply-adds on the same values as moe_combine_kernel after the sum all-reduce.
__global__ __launch_bounds__(256) void moe_combine_gathered_kernel(float* __restrict__ x, const float* __restrict__ gathered,
                                                                   const float* __restrict__ eout, const int* __restrict__ experts,
                                                                   const float* __restrict__ w, int n_slots, int add_shared, int n, int per) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float xv = x[i];
  for (int k = 0; k < n_slots; ++k) {
    const int owner = experts[k] / per;
    xv = fmaf(gathered[((size_t)owner * n_slots + k) * n + i], w[k], xv);
  }
  if (add_shared) xv += eout[(size_t)n_slots * n + i];
  x[i] = xv;
}
int launch_moe_combine_gathered(hipStream_t st, float* x, const float* gathered, const float* eout, const int* experts,
                                const float* weights, int n_slots, int add_shared, int n, int per) {
  hipLaunchKernelGGL(moe_combine_gathered_kernel, dim3((n + 255) / 256), dim3(256), 0, st, x, gathered, eout, experts, weights,
                     n_slots, add_shared, n, per);
  return DSK_OK;
}

int launch_quantize_q8k(hipStream_t st, const float* x, int n, int8_t* qs, float* d, int16_t* bsums) {
  if (n <= 0 || n % 256) DSK_FAIL(DSK_ERR_INVALID, "q8k: n=%d must be a positive multiple of 256", n);
  const int nb = n / 256;
  hipLaunchKernelGGL(quantize_q8k_kernel, dim3((nb + 3) / 4), dim3(256), 0, st, x, nb, qs, d, bsums);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// norm jobs: [MoE combine ->] rmsnorm -> [f32 out] -> [Q8_K out] -> [rope on a tail vector]
// rmsnorm: src/infer.cpp:601-611; combine: src/infer.cpp:874-877, 900-903.
// One workgroup (1024 threads) per job.
// ------------------------------------------------------------------------------------
struct NormJobs2 {
  NormJob j[2];
};

DEV void rope_pairs(float* vec, int d, const float* cs, int is_v3, int tid, int nthreads) {
  // rope (V2: de-interleaving) src/infer.cpp:648-668; rope_v3 (in place) src/infer.cpp:670-685.
  // cs[2*j], cs[2*j+1] = cos, sin of pos * theta^(-2j/d), computed on the host with libm.
  float re = 0.f, im = 0.f;
  const int p = tid;
  if (p < d / 2) {
    const float v0 = vec[2 * p], v1 = vec[2 * p + 1];
    const float c = cs[2 * p], s = cs[2 * p + 1];
    ad::rope_rot(v0, v1, c, s, re, im);
  }
  __syncthreads();
  if (p < d / 2) {
    if (is_v3) {
      vec[2 * p] = re;
      vec[2 * p + 1] = im;
    } else {
      vec[p] = re;
      vec[p + d / 2] = im;
    }
  }
}

__global__ __launch_bounds__(1024) void norm_jobs_kernel(NormJobs2 jobs, const StepParams* __restrict__ sp) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float scratch[16];
  const NormJob& J = jobs.j[blockIdx.x];
  float* l_y = reinterpret_cast<float*>(smem);
  const int tid = threadIdx.x, n = J.n;

  float ss = 0.f;
  for (int i = tid; i < n; i += 1024) {
    float xv = J.x[i];
    if (J.eout) {
      for (int k = 0; k < J.n_routed_slots; ++k) xv = fmaf(J.eout[(size_t)k * n + i], J.eweights[k], xv);
      if (J.add_shared) xv += J.eout[(size_t)J.n_routed_slots * n + i];
      if (J.x_store) J.x_store[i] = xv;
    }
    l_y[i] = xv;
    ss = fmaf(xv, xv, ss);
  }
  if (J.weight) {
    const float total = block_sum(ss, scratch, tid, 1024);
    const float scale = 1.0f / sqrtf(total / (float)n + J.eps);
    for (int i = tid; i < n; i += 1024) {
      const float y = l_y[i] * scale * J.weight[i];
      l_y[i] = y;
      if (J.y_f32) J.y_f32[i] = y;
    }
  } else if (J.y_f32) {
    for (int i = tid; i < n; i += 1024) J.y_f32[i] = l_y[i];
  }
  __syncthreads();
  if (J.q_qs) {
    const int wave = tid >> 6, lane = tid & 63;
    for (int b = wave; b < (n >> 8); b += 16) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(l_y + b * 256 + lane * 4);
      const float v[4] = {t.x, t.y, t.z, t.w};
      q8k_block(v, lane, J.q_qs + (size_t)b * 256, J.q_d + b, J.q_bsums + (size_t)b * 16);
    }
  }
  if (J.rope_vec) rope_pairs(J.rope_vec, J.rope_d, sp->rope_cs, J.rope_v3, tid, 1024);
}

int launch_norm_jobs(hipStream_t st, const NormJob* jobs, int n_jobs, const StepParams* sp) {
  if (n_jobs < 1 || n_jobs > 2) DSK_FAIL(DSK_ERR_INVALID, "norm jobs: 1..2 jobs");
  NormJobs2 a;
  int nmax = 0;
  for (int i = 0; i < n_jobs; ++i) {
    a.j[i] = jobs[i];
    if (jobs[i].q_qs && jobs[i].n % 256) DSK_FAIL(DSK_ERR_INVALID, "norm job: q8 output needs n %% 256 == 0 (n=%d)", jobs[i].n);
    if (jobs[i].n > nmax) nmax = jobs[i].n;
  }
  if (n_jobs == 1) a.j[1] = jobs[0];
  const size_t lds = (size_t)nmax * 4;
  if (lds > 150 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "norm job: n=%d too large", nmax);
  if (lds > 64 * 1024) hipFuncSetAttribute((const void*)norm_jobs_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(norm_jobs_kernel, dim3(n_jobs), dim3(1024), lds, st, a, sp);
  return DSK_OK;
}

// rope only (op-level API): n_heads vectors of length d, one workgroup each
__global__ void rope_only_kernel(float* vec, int d, const float* cs, int is_v3) {
  rope_pairs(vec + (size_t)blockIdx.x * d, d, cs, is_v3, threadIdx.x, blockDim.x);
}
int launch_rope_only(hipStream_t st, float* vec, int n_heads, int d, const float* cs, int is_v3) {
  hipLaunchKernelGGL(rope_only_kernel, dim3(n_heads), dim3(64 * ((d / 2 + 63) / 64)), 0, st, vec, d, cs, is_v3);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// upload-time re-layout of K-quant blocks into planes (see dsk_internal.h)
// ------------------------------------------------------------------------------------
__global__ void repack_q2k_kernel(const u32* __restrict__ aos, size_t n_blocks, uint8_t* qs, uint8_t* sc, uint8_t* dm) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t b = gid / 21;
  const int j = (int)(gid % 21);
  if (b >= n_blocks) return;
  const u32 w = aos[b * 21 + j];  // 84-byte blocks: scales[16] | qs[64] | d | dmin (src/quant.h:41-52)
  if (j < 4) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int jj = 4 * j + t;  // sub-block index 8h + 2s + lh
      const int h = jj >> 3, s = (jj >> 1) & 3, lh = jj & 1;
      sc[b * 16 + (2 * h + lh) * 4 + s] = (uint8_t)(w >> (8 * t));
    }
  } else if (j < 20) {
    reinterpret_cast<u32*>(qs)[b * 16 + (j - 4)] = w;
  } else {
    reinterpret_cast<u32*>(dm)[b] = w;
  }
}
int launch_repack_q2k(hipStream_t st, const uint8_t* aos, size_t n_blocks, uint8_t* qs, uint8_t* sc, uint8_t* dm) {
  const size_t total = n_blocks * 21;
  hipLaunchKernelGGL(repack_q2k_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<const u32*>(aos), n_blocks, qs, sc, dm);
  return DSK_OK;
}

// Q2_K into the TILED layout (tile_device.h): block gb0 + i of the reference's [matrix][row][block] order -> its place in the
// tile records (16-row x 256-column tiles of 1344 bytes, strips of a matrix contiguous, rows padded to 16 per matrix)
DEV size_t tile_block_base(size_t gb, int rows, int nb, size_t e_bytes, int* r16) {
  const size_t per = (size_t)rows * nb;
  const size_t mat = gb / per, rem = gb - mat * per;
  const int r = (int)(rem / nb), b = (int)(rem - (size_t)r * nb);
  *r16 = r & 15;
  return mat * e_bytes + ((size_t)(r >> 4) * nb + b) * 1344;
}
__global__ void repack_q2k_tiles_kernel(const u32* __restrict__ aos, size_t gb0, size_t n_blocks, int rows, int nb, size_t e_bytes, uint8_t* tiles) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t i = gid / 21;
  const int j = (int)(gid % 21);
  if (i >= n_blocks) return;
  const u32 w = aos[i * 21 + j];  // 84-byte blocks: scales[16] | qs[64] | d | dmin (src/quant.h:41-52)
  int n;
  uint8_t* T = tiles + tile_block_base(gb0 + i, rows, nb, e_bytes, &n);
  if (j < 4) *reinterpret_cast<u32*>(T + 1024 + 4 * (n + 16 * j)) = w;                                 // scales[4j .. 4j + 3]
  else if (j < 20) *reinterpret_cast<u32*>(T + 16 * (n + 16 * ((j - 4) >> 2)) + 4 * ((j - 4) & 3)) = w;  // qs bytes [4 (j - 4), + 4)
  else *reinterpret_cast<u32*>(T + 1280 + 4 * n) = w;
}
int launch_repack_q2k_tiles(hipStream_t st, const uint8_t* aos, size_t gb0, size_t n_blocks, int rows, int nb, size_t e_bytes, uint8_t* tiles) {
  const size_t total = n_blocks * 21;
  hipLaunchKernelGGL(repack_q2k_tiles_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, reinterpret_cast<const u32*>(aos), gb0,
                     n_blocks, rows, nb, e_bytes, tiles);
  return DSK_OK;
}
// the same from the PLANE layout (a checkpoint repacked offline as planes-v1): qs[blk][64], sc[blk][16] in quarter order
// sc'[4 (2h + lh) + s] = scales[8h + 2s + lh], dm[blk]
__global__ void planes_to_tiles_q2k_kernel(const u32* __restrict__ qs, const uint8_t* __restrict__ sc, const u32* __restrict__ dm, size_t gb0,
                                           size_t n_blocks, int rows, int nb, size_t e_bytes, uint8_t* tiles) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t i = gid / 21;
  const int j = (int)(gid % 21);
  if (i >= n_blocks) return;
  int n;
  uint8_t* T = tiles + tile_block_base(gb0 + i, rows, nb, e_bytes, &n);
  if (j < 4) {
    u32 w = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int jj = 4 * j + t, h = jj >> 3, s = (jj >> 1) & 3, lh = jj & 1;
      w |= (u32)sc[i * 16 + (2 * h + lh) * 4 + s] << (8 * t);
    }
    *reinterpret_cast<u32*>(T + 1024 + 4 * (n + 16 * j)) = w;
  } else if (j < 20) {
    *reinterpret_cast<u32*>(T + 16 * (n + 16 * ((j - 4) >> 2)) + 4 * ((j - 4) & 3)) = qs[i * 16 + (j - 4)];
  } else {
    *reinterpret_cast<u32*>(T + 1280 + 4 * n) = dm[i];
  }
}
int launch_planes_to_tiles_q2k(hipStream_t st, const uint8_t* qs, const uint8_t* sc, const uint8_t* dm, size_t gb0, size_t n_blocks, int rows, int nb,
                               size_t e_bytes, uint8_t* tiles) {
  const size_t total = n_blocks * 21;
  hipLaunchKernelGGL(planes_to_tiles_q2k_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, reinterpret_cast<const u32*>(qs), sc,
                     reinterpret_cast<const u32*>(dm), gb0, n_blocks, rows, nb, e_bytes, tiles);
  return DSK_OK;
}

__global__ void repack_q3k_kernel(const unsigned short* __restrict__ aos, size_t n_blocks, unsigned short* qs,
                                  unsigned short* hm, unsigned short* sc, unsigned short* dm) {
  const size_t gid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t b = gid / 55;
  const int j = (int)(gid % 55);
  if (b >= n_blocks) return;
  const unsigned short w = aos[b * 55 + j];  // 110-byte blocks: hmask[32] | qs[64] | scales[12] | d (src/quant.h:70-76)
  if (j < 16) hm[b * 16 + j] = w;
  else if (j < 48) qs[b * 32 + (j - 16)] = w;
  else if (j < 54) sc[b * 6 + (j - 48)] = w;
  else dm[b] = w;
}
int launch_repack_q3k(hipStream_t st, const uint8_t* aos, size_t n_blocks, uint8_t* qs, uint8_t* hm, uint8_t* sc, uint8_t* dm) {
  const size_t total = n_blocks * 55;
  hipLaunchKernelGGL(repack_q3k_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<const unsigned short*>(aos), n_blocks, reinterpret_cast<unsigned short*>(qs),
                     reinterpret_cast<unsigned short*>(hm), reinterpret_cast<unsigned short*>(sc),
                     reinterpret_cast<unsigned short*>(dm));
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// embedding row: Model::_copy_embedding, src/infer.cpp:1217-1263 (one thread per element)
// ------------------------------------------------------------------------------------
DEV int q3k_scale_b(const uint8_t* S, int j) {  // src/quant.cpp:402-407
  const int low4 = j < 8 ? (S[j] & 0xF) : (S[j - 8] >> 4);
  const int hi2 = (S[8 + (j & 3)] >> (2 * (j >> 2))) & 3;
  return (low4 | (hi2 << 4)) - 32;
}

// blockIdx.y = the row of a batch (dsk_hydrate: the tokens of a chunk come from its step rows, x holds gridDim.y rows of dim floats).
// sp_dev: sp lies in host memory, and the first workgroup leaves a copy there for the token's other launches: one round trip to the host in the token's
// first launch instead of a copy of 4.2 us in front of it.
__global__ void embed_kernel(DTensor t, const StepParams* __restrict__ sp, StepParams* __restrict__ sp_dev, int token_override, int b0, int b1, float* __restrict__ x) {
  if (sp_dev && blockIdx.x == 0)
    for (int k = threadIdx.x; k < (int)(sizeof(StepParams) / 4); k += blockDim.x) reinterpret_cast<int*>(sp_dev)[k] = reinterpret_cast<const int*>(sp)[k];
  const int token = token_override >= 0 ? token_override : sp[blockIdx.y].token;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int dim = t.n;
  if (i >= dim) return;
  x += (size_t)blockIdx.y * dim;
  const size_t nb = dim >> 8;
  float y;
  switch (t.quant) {
    case DSK_QUANT_F32: y = reinterpret_cast<const float*>(t.qs)[(size_t)token * dim + i]; break;
    case DSK_QUANT_F16: y = h2f(reinterpret_cast<const unsigned short*>(t.qs)[(size_t)token * dim + i]); break;
    case DSK_QUANT_F8E5M2: {
      const int ncols = (dim + b1 - 1) / b1;
      const float s = t.scale[(size_t)(token / b0) * ncols + i / b1];
      y = h2f((unsigned short)((unsigned short)t.qs[(size_t)token * dim + i] << 8)) * s;
      break;
    }
    case DSK_QUANT_Q2_K: {  // dequantize_row_q2_K, src/quant.cpp:217-247
      if (t.tiled) {  // tile records (tile_device.h): 16-row x 256-column tiles of 1344 bytes
        const uint8_t* T = t.qs + ((size_t)(token >> 4) * nb + (i >> 8)) * 1344;
        const int n = token & 15, e = i & 255, h = e >> 7, s = (e >> 5) & 3, l = e & 31, jj = e >> 4;
        const int byte = 32 * h + l;
        const int q = (T[16 * (n + 16 * (byte >> 4)) + (byte & 15)] >> (2 * s)) & 3;
        const int scb = T[1024 + 4 * (n + 16 * (jj >> 2)) + (jj & 3)];
        const u32 dmw = *reinterpret_cast<const u32*>(T + 1280 + 4 * n);
        const float dl = h2f(dmw & 0xffff) * (scb & 0xF), ml = h2f(dmw >> 16) * (scb >> 4);
        y = dl * q - ml;
        break;
      }
      const size_t b = (size_t)token * nb + (i >> 8);
      const int e = i & 255, h = e >> 7, s = (e >> 5) & 3, l = e & 31, lh = l >> 4;
      const int q = (t.qs[b * 64 + 32 * h + l] >> (2 * s)) & 3;
      const int scb = t.sc[b * 16 + (2 * h + lh) * 4 + s];
      const u32 dmw = reinterpret_cast<const u32*>(t.dm)[b];
      const float dl = h2f(dmw & 0xffff) * (scb & 0xF), ml = h2f(dmw >> 16) * (scb >> 4);
      y = dl * q - ml;
      break;
    }
    default: {  // dequantize_row_q3_K, src/quant.cpp:384-432
      const size_t b = (size_t)token * nb + (i >> 8);
      const int e = i & 255, h = e >> 7, s = (e >> 5) & 3, l = e & 31, lh = l >> 4;
      const int ql = (t.qs[b * 64 + 32 * h + l] >> (2 * s)) & 3;
      const int hb = (t.hm[b * 32 + l] >> (4 * h + s)) & 1;
      const int sc = q3k_scale_b(t.sc + b * 12, 8 * h + 2 * s + lh);
      const float dl = h2f(reinterpret_cast<const unsigned short*>(t.dm)[b]) * sc;
      y = dl * (ql - (hb ? 0 : 4));
      break;
    }
  }
  x[i] = y;
}
int launch_embed(hipStream_t st, const DTensor& t, const StepParams* sp, StepParams* sp_dev, int token_override, int b0, int b1, float* x) {
  hipLaunchKernelGGL(embed_kernel, dim3((t.n + 255) / 256), dim3(256), 0, st, t, sp, sp_dev, token_override, b0, b1, x);
  return DSK_OK;
}
int launch_embed_rows(hipStream_t st, const DTensor& t, const StepParams* sps, int P, int b0, int b1, float* x) {
  hipLaunchKernelGGL(embed_kernel, dim3((t.n + 255) / 256, P), dim3(256), 0, st, t, sps, nullptr, -1, b0, b1, x);
  return DSK_OK;
}

// gate_body / router_body live in router_device.h (shared with kernels_gemv.hip)
// (1024 threads like the router launch's last workgroup, so that the op-level entry point runs - and its tests with exact ties
// cover - the same four-lanes-per-candidate rank loops)
__global__ __launch_bounds__(1024) void gate_kernel(const float* __restrict__ partial, int ksplit, const float* __restrict__ bias,
                                                   int E, int K, int norm_topk_prob, float scaling, int scoring, int topk_method,
                                                   int n_group, int topk_group, int* __restrict__ active_experts,
                                                   float* __restrict__ active_weights, float* __restrict__ scores_out) {
  __shared__ __attribute__((aligned(16))) float s[512];
  __shared__ __attribute__((aligned(16))) int surv[256];
  __shared__ float scratch[16];
  __shared__ int sel[256];
  const int e = threadIdx.x;
  float v = 0.f;
  if (e < E)
    for (int c = 0; c < ksplit; ++c) v += partial[(size_t)c * E + e];
  rd::gate_body(e, v, bias, E, K, norm_topk_prob, scaling, scoring, topk_method, n_group, topk_group, active_experts, active_weights,
            scores_out, s, surv, sel, scratch, 1024);
}
int launch_gate(hipStream_t st, const float* partial, int ksplit, const float* bias, int n_routed, int n_active,
                int norm_topk_prob, float scaling, int scoring, int topk_method, int n_group, int topk_group,
                int* active_experts, float* active_weights, float* scores_out) {
  if (n_routed > 256) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_gate: more than 256 routed experts (src/infer.cpp:527)");
  if (n_active > n_routed) DSK_FAIL(DSK_ERR_INVALID, "moe_gate: n_active > n_routed");
  if (topk_method == DSK_TOPK_GROUP_LIMITED_GREEDY && (n_group <= 0 || n_routed % n_group || topk_group * n_group < n_active))
    DSK_FAIL(DSK_ERR_INVALID, "moe_gate: bad group config (E=%d, n_group=%d, topk_group=%d, k=%d)", n_routed, n_group, topk_group, n_active);
  hipLaunchKernelGGL(gate_kernel, dim3(1), dim3(1024), 0, st, partial, ksplit, bias, n_routed, n_active, norm_topk_prob, scaling,
                     scoring, topk_method, n_group, topk_group, active_experts, active_weights, scores_out);
  return DSK_OK;
}

// sum over the 16 lanes of a DPP row (every lane gets the total; VALU speed, no ds_bpermute)
DEV float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));  // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true));  // row_mirror
  return v;
}

// full-wave sum, fixed order: DPP inside the 16-lane rows, then the four rows
DEV float wave_sum_dpp(float v) {
  v = row16_sum(v);
  const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
  const float b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
  const float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
  const float d = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
  return (a + b) + (c + d);
}

template <int RW>
__global__ __launch_bounds__(1024) void router_gate_kernel(RouterArgs a) {
  rd::router_body<RW>(a, blockIdx.x, gridDim.x);
}
int launch_router_gate(hipStream_t st, const RouterArgs& a) {
  if (a.dim % 4) DSK_FAIL(DSK_ERR_INVALID, "router: dim %% 4 != 0");
  if (a.n_routed > 256) DSK_FAIL(DSK_ERR_UNSUPPORTED, "moe_gate: more than 256 routed experts (src/infer.cpp:527)");
  if (a.n_active > a.n_routed) DSK_FAIL(DSK_ERR_INVALID, "moe_gate: n_active > n_routed");
  if (a.topk_method == DSK_TOPK_GROUP_LIMITED_GREEDY && (a.n_group <= 0 || a.n_routed % a.n_group || a.topk_group * a.n_group < a.n_active))
    DSK_FAIL(DSK_ERR_INVALID, "moe_gate: bad group config (E=%d, n_group=%d, topk_group=%d, k=%d)", a.n_routed, a.n_group, a.topk_group, a.n_active);
  // ksplit = column slices per row: 4 -> 4 rows per workgroup, 8 -> 2 rows per workgroup
  if (a.ksplit >= 8) hipLaunchKernelGGL(router_gate_kernel<2>, dim3((a.n_routed + 1) / 2), dim3(1024), 0, st, a);
  else hipLaunchKernelGGL(router_gate_kernel<4>, dim3((a.n_routed + 3) / 4), dim3(1024), 0, st, a);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// MHA path: RoPE on q, assemble k/v, f16 cache write, attention-sink rotation.
// BlockMHA::_attention_impl, src/infer.cpp:956-1020.  One workgroup per head.
// ------------------------------------------------------------------------------------
// q_lds != null: the rotated query goes to LDS only (the fused kernel is its single consumer)
template <int NT>
DEV void rope_kv_mha_body(const AttnMhaArgs& a, const StepParams* __restrict__ sp, int h, int tid, float* q_lds = nullptr) {
  const int hd = a.head_dim, nope = a.nope, rope = a.rope, vd = a.v_dim;
  const int kv_pos = sp->kv_pos, kv_sink = sp->kv_sink;
  if (q_lds) {
    const float* qg = a.q + (size_t)h * hd;
    if (tid < nope) q_lds[tid] = qg[tid];
    if (tid < rope / 2) {  // rope (V2: de-interleaving) src/infer.cpp:648-668; rope_v3 :670-685
      const float v0 = qg[nope + 2 * tid], v1 = qg[nope + 2 * tid + 1];
      const float c = sp->rope_cs[2 * tid], s = sp->rope_cs[2 * tid + 1];
      float re, im;
      ad::rope_rot(v0, v1, c, s, re, im);
      if (a.is_v3) {
        q_lds[nope + 2 * tid] = re;
        q_lds[nope + 2 * tid + 1] = im;
      } else {
        q_lds[nope + tid] = re;
        q_lds[nope + tid + rope / 2] = im;
      }
    }
  } else {
    rope_pairs(a.q + (size_t)h * hd + nope, rope, sp->rope_cs, a.is_v3, tid, NT);  // q rope, in place
  }
  // key = [k_nope | rope(k_rope)], value  -> f16 caches at kv_pos
  uint16_t* kc = a.key_cache + ((size_t)kv_pos * a.n_heads + h) * hd;
  uint16_t* vc = a.value_cache + ((size_t)kv_pos * a.n_heads + h) * vd;
  const float* kvb = a.kv_b + (size_t)h * (nope + vd);
  for (int i = tid; i < nope; i += NT) kc[i] = f2h(kvb[i]);
  for (int i = tid; i < vd; i += NT) vc[i] = f2h(kvb[nope + i]);
  if (tid < rope / 2) {
    const float* kr = a.kv_a + a.lora;
    const float v0 = kr[2 * tid], v1 = kr[2 * tid + 1];
    const float c = sp->rope_cs[2 * tid], s = sp->rope_cs[2 * tid + 1];
    float re, im;
    ad::rope_rot(v0, v1, c, s, re, im);
    if (a.is_v3) {
      kc[nope + 2 * tid] = f2h(re);
      kc[nope + 2 * tid + 1] = f2h(im);
    } else {
      kc[nope + tid] = f2h(re);
      kc[nope + tid + rope / 2] = f2h(im);
    }
  }
  // sinks: rotate the rope part of cached keys 0..kv_sink-1 by one position, in f16
  // (src/infer.cpp:1008-1020, rope f16 variants :687-724)
  for (int r = 0; r < kv_sink; ++r) {
    uint16_t* kh = a.key_cache + ((size_t)r * a.n_heads + h) * hd + nope;
    float re = 0.f, im = 0.f;
    if (tid < rope / 2) {
      const float v0 = h2f(kh[2 * tid]), v1 = h2f(kh[2 * tid + 1]);
      const float c = sp->rope_cs1[2 * tid], s = sp->rope_cs1[2 * tid + 1];
      ad::rope_rot(v0, v1, c, s, re, im);
    }
    __syncthreads();
    if (tid < rope / 2) {
      if (a.is_v3) {
        kh[2 * tid] = f2h(re);
        kh[2 * tid + 1] = f2h(im);
      } else {
        kh[tid] = f2h(re);
        kh[tid + rope / 2] = f2h(im);
      }
    }
    __syncthreads();
  }
}
__global__ __launch_bounds__(256) void rope_kv_mha_kernel(AttnMhaArgs a, const StepParams* __restrict__ sp) {
  rope_kv_mha_body<256>(a, sp, blockIdx.x, threadIdx.x);
}
int launch_rope_kv_mha(hipStream_t st, const AttnMhaArgs& a, const StepParams* sp) {
  if (a.rope > 128 || (a.rope & 1)) DSK_FAIL(DSK_ERR_UNSUPPORTED, "rope dim %d (max 128, even)", a.rope);
  hipLaunchKernelGGL(rope_kv_mha_kernel, dim3(a.n_heads), dim3(256), 0, st, a, sp);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// attn (per head), src/infer.cpp:728-762: scores = q.k / sqrt(head_dim), softmax, sum att*v.
// One workgroup per head; scores live in LDS (kv_len floats).
// ------------------------------------------------------------------------------------
// returns this thread's output element (valid for tid < v_dim).  part: 256 / (v_dim / 4) * v_dim floats.
// Scores: 16 lanes per cached position (4 positions per wave step, 128-byte coalesced f16 reads);
// values: 4 output dims per thread, v_dim / 4 threads per position.
// q: the head's query (global, or the LDS copy the fused kernel rotated in place).  NT threads; part: NT / (v_dim / 4) * v_dim floats.
template <int NT>
DEV float attn_mha_body(const AttnMhaArgs& a, const float* q, int kv_len, int h, int tid, float* att, float* scratch, float* part) {
  const int wave = tid >> 6, lane = tid & 63, grp = lane >> 4, sl = lane & 15;
  const int hd = a.head_dim, vd = a.v_dim, H = a.n_heads;
  float qv[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d0 = 64 * j + sl * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) qv[j][i] = d0 < hd ? q[d0 + i] : 0.f;
  }
  const float inv = sqrtf((float)hd);
  // 4 positions per 16-lane group and step (16 per wave, 64 per workgroup): up to 16 eight-byte loads in
  // flight per lane, so a long context streams the cache instead of paying one latency per position
  for (int t0 = wave * 16; t0 < kv_len; t0 += NT / 4) {
    f16x4 k[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + u * 4 + grp;
      if (t < kv_len) {
        const uint16_t* kr = a.key_cache + ((size_t)t * H + h) * hd;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (64 * j + sl * 4 < hd) k[u][j] = *reinterpret_cast<const f16x4*>(kr + 64 * j + sl * 4);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + u * 4 + grp;
      float p = 0.f;
      if (t < kv_len) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (64 * j + sl * 4 < hd) {
            p = fmaf(qv[j][0], (float)k[u][j].x, p);
            p = fmaf(qv[j][1], (float)k[u][j].y, p);
            p = fmaf(qv[j][2], (float)k[u][j].z, p);
            p = fmaf(qv[j][3], (float)k[u][j].w, p);
          }
      }
      p = row16_sum(p);
      if (sl == 0 && t < kv_len) att[t] = p / inv;
    }
  }
  // the first two value rows of this thread are requested now: their latency hides behind the softmax
  const int tpp = vd >> 2;        // threads per position
  const int TG = NT / tpp;        // positions in flight
  const int g = tid / tpp, i4 = tid - g * tpp;
  f16x4 vpre[2] = {};
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (g < TG && g + k * TG < kv_len)
      vpre[k] = *reinterpret_cast<const f16x4*>(a.value_cache + ((size_t)(g + k * TG) * H + h) * vd + i4 * 4);
  __syncthreads();
  // softmax, src/infer.cpp:472-487
  float mx = -INFINITY;
  for (int t = tid; t < kv_len; t += NT) mx = fmaxf(mx, att[t]);
  mx = block_max(mx, scratch, tid, NT);
  float sum = 0.f;
  for (int t = tid; t < kv_len; t += NT) {
    const float e = expf(att[t] - mx);
    att[t] = e;
    sum += e;
  }
  sum = block_sum(sum, scratch, tid, NT);
  for (int t = tid; t < kv_len; t += NT) att[t] = att[t] / sum;
  __syncthreads();
  // mix values: thread (g, i4) sums positions g, g+TG, ... for outputs 4*i4..4*i4+3; groups are added in order
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (g < TG) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int t = g + k * TG;
      if (t < kv_len) {
        const float w = att[t];
        acc[0] = fmaf(w, (float)vpre[k].x, acc[0]);
        acc[1] = fmaf(w, (float)vpre[k].y, acc[1]);
        acc[2] = fmaf(w, (float)vpre[k].z, acc[2]);
        acc[3] = fmaf(w, (float)vpre[k].w, acc[3]);
      }
    }
    for (int t0 = g + 2 * TG; t0 < kv_len; t0 += 4 * TG) {  // 4 rows in flight per thread
      f16x4 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (t0 + k * TG < kv_len) v[k] = *reinterpret_cast<const f16x4*>(a.value_cache + ((size_t)(t0 + k * TG) * H + h) * vd + i4 * 4);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (t0 + k * TG < kv_len) {
          const float w = att[t0 + k * TG];
          acc[0] = fmaf(w, (float)v[k].x, acc[0]);
          acc[1] = fmaf(w, (float)v[k].y, acc[1]);
          acc[2] = fmaf(w, (float)v[k].z, acc[2]);
          acc[3] = fmaf(w, (float)v[k].w, acc[3]);
        }
    }
    *reinterpret_cast<f32x4*>(part + (size_t)g * vd + i4 * 4) = f32x4{acc[0], acc[1], acc[2], acc[3]};
  }
  __syncthreads();
  float o = 0.f;
  if (tid < vd)
    for (int gg = 0; gg < TG; ++gg) o += part[gg * vd + tid];
  return o;
}
__global__ __launch_bounds__(256) void attn_mha_kernel(AttnMhaArgs a, const StepParams* __restrict__ sp, int kv_len_override) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float scratch[4];
  __shared__ __attribute__((aligned(16))) float part[1024];
  const int h = blockIdx.x, tid = threadIdx.x;
  const float o = attn_mha_body<256>(a, a.q + (size_t)h * a.head_dim, kv_len_override > 0 ? kv_len_override : sp->kv_len, h, tid,
                                reinterpret_cast<float*>(smem), scratch, part);
  if (tid < a.v_dim) a.out[(size_t)h * a.v_dim + tid] = o;
}

int launch_attn_mha(hipStream_t st, const AttnMhaArgs& a, const StepParams* sp, int kv_len_override, int max_kv) {
  if (a.head_dim > 256 || a.head_dim % 4 || a.v_dim > 256 || a.v_dim % 4) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn: head_dim %d / v_head_dim %d", a.head_dim, a.v_dim);
  const size_t lds = (size_t)max_kv * 4;
  if (lds > 150 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn: kv_len %d does not fit LDS", max_kv);
  if (lds > 64 * 1024) hipFuncSetAttribute((const void*)attn_mha_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(attn_mha_kernel, dim3(a.n_heads), dim3(256), lds, st, a, sp, kv_len_override);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// MLA path: BlockMLA::_attention_impl, src/infer.cpp:1072-1130.
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void rope_kv_mla_kernel(AttnMlaArgs a, const StepParams* __restrict__ sp) {
  const int h = blockIdx.x, tid = threadIdx.x;
  const int rope = a.rope, lora = a.lora;
  rope_pairs(a.q_rope + (size_t)h * rope, rope, sp->rope_cs, a.is_v3, tid, 256);
  if (h != 0) return;
  const int kv_pos = sp->kv_pos, kv_sink = sp->kv_sink;
  uint16_t* nc = a.nope_cache + (size_t)kv_pos * lora;
  uint16_t* rc = a.rope_cache + (size_t)kv_pos * rope;
  for (int i = tid; i < lora; i += 256) nc[i] = f2h(a.kv_a[i]);
  if (tid < rope / 2) {
    const float* kr = a.kv_a + lora;
    const float v0 = kr[2 * tid], v1 = kr[2 * tid + 1];
    const float c = sp->rope_cs[2 * tid], s = sp->rope_cs[2 * tid + 1];
    float re, im;
    ad::rope_rot(v0, v1, c, s, re, im);
    if (a.is_v3) {
      rc[2 * tid] = f2h(re);
      rc[2 * tid + 1] = f2h(im);
    } else {
      rc[tid] = f2h(re);
      rc[tid + rope / 2] = f2h(im);
    }
  }
  for (int r = 0; r < kv_sink; ++r) {  // src/infer.cpp:1103-1110
    uint16_t* kh = a.rope_cache + (size_t)r * rope;
    float re = 0.f, im = 0.f;
    if (tid < rope / 2) {
      const float v0 = h2f(kh[2 * tid]), v1 = h2f(kh[2 * tid + 1]);
      const float c = sp->rope_cs1[2 * tid], s = sp->rope_cs1[2 * tid + 1];
      ad::rope_rot(v0, v1, c, s, re, im);
    }
    __syncthreads();
    if (tid < rope / 2) {
      if (a.is_v3) {
        kh[2 * tid] = f2h(re);
        kh[2 * tid + 1] = f2h(im);
      } else {
        kh[tid] = f2h(re);
        kh[tid + rope / 2] = f2h(im);
      }
    }
    __syncthreads();
  }
}
// MLA model path, one workgroup: rmsnorm of the latent (src/infer.cpp:1089), f16 cache entries of this position
// (:1092-1097), rotation of the sink keys (:1103-1110).
__global__ __launch_bounds__(256) void mla_kv_write_kernel(MlaKvArgs a, const StepParams* __restrict__ sp) {
  rd::mla_kv_write_body(a, sp, threadIdx.x, 256);
}
int launch_mla_kv_write(hipStream_t st, const MlaKvArgs& a, const StepParams* sp) {
  if (a.rope > 128 || (a.rope & 1)) DSK_FAIL(DSK_ERR_UNSUPPORTED, "rope dim %d (max 128, even)", a.rope);
  hipLaunchKernelGGL(mla_kv_write_kernel, dim3(1), dim3(256), 0, st, a, sp);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// MLA attention on the matrix cores (long contexts).  See MlaFlashArgs in dsk_internal.h.
// v_mfma_f32_32x32x8_f16: A four f16 per lane A[i = l&31][k = 4*(l>>5) ..+3], B four f16 per lane B[k = 4*(l>>5) ..+3][j = l&31],
// C/D 16 f32 per lane: col = l&31, row = (reg&3) + 8*(reg>>2) + 4*(l>>5).  The cache entries ARE f16; the f32 operand of
// each product (q, the softmax weights) goes in as hi + lo f16 halves, two MFMAs: exact products, f32 accumulation
// (round 1 used v_mfma_f32_32x32x2_f32: twice the instructions for the same bits to ~1e-7).
// ------------------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
#define FL_KSTRIDE 580   // halfs per staged cache row (576 + 4): 290 dwords, odd multiple of 2 -> conflict-free column reads
#define FL_PSTRIDE 33

// 8 waves per workgroup: the K range of the score GEMM and the latent columns of the value GEMM are split 8 ways, so a
// wave issues 18 + 16 MFMAs per 32-position block and two waves share a SIMD.  All B operands of a block are read
// from LDS into registers BEFORE the MFMA chain (a dependent ds_read -> cvt -> mfma per step tripled the time).
#define FL_NWV 8
__global__ __launch_bounds__(FL_NWV * 64) void mla_flash_kernel(MlaFlashArgs a, const StepParams* __restrict__ sp, int kv_len_override) {
  extern __shared__ __attribute__((aligned(16))) uint8_t fl_smem[];
  {  // the batched prompt path: token blockIdx.z of the chunk (decode: z = 0, nothing moves)
    const size_t z = blockIdx.z;
    sp += z;
    a.q_c += z * a.tok_qc_stride;
    a.q_rope += z * a.tok_qr_stride;
    a.part_o += z * a.n_chunks * a.n_heads * a.lora;
    a.part_ml += z * a.n_chunks * a.n_heads * 2;
  }
  unsigned short* Ks = reinterpret_cast<unsigned short*>(fl_smem);                                   // [32][FL_KSTRIDE]
  float (*Sp)[32][FL_PSTRIDE] = reinterpret_cast<float (*)[32][FL_PSTRIDE]>(fl_smem + 32 * FL_KSTRIDE * 2);  // [FL_NWV][32][33]
  float (*Pm)[FL_PSTRIDE] = reinterpret_cast<float (*)[FL_PSTRIDE]>(fl_smem + 32 * FL_KSTRIDE * 2 + FL_NWV * 32 * FL_PSTRIDE * 4);
  __shared__ float m_s[32], l_s[32], al_s[32];
  const int hg = blockIdx.y, tid = threadIdx.x, w = tid >> 6, l = tid & 63, i = l & 31, kh = l >> 5;
  unsigned long long* tl = a.timeline && blockIdx.x * gridDim.y + blockIdx.y < DSK_TL_WGS ? a.timeline + (size_t)(blockIdx.x * gridDim.y + blockIdx.y) * 8 : nullptr;
  if (tl && tid == 0) tl[0] = wall_clock64();
  constexpr int lora = 512, rope = 64, KT = lora + rope;  // 576: launch_mla_flash admits only these (compile-time: the staging loops unroll)
  const int head = hg * 32 + i;
  const bool hv = head < a.n_heads;
  // ---- this wave's eighth of the K range of Q, one value per (MFMA step, lane): k = 2*(ks0 + s) + kh ----
  constexpr int steps = 288 / FL_NWV;  // k-pairs per wave: (512 + 64) / 2 / 8 (launch_mla_flash admits only these dims)
  const int ks0 = w * steps;
  // ---- requests first.  The Q tile of this head group (written a launch ago by other CUs: L2 misses) depends on nothing,
  // not even on the context length: its 9 float4 per thread leave before kv_len has been read; then the first 32 cache
  // rows of this chunk (HBM; they do not depend on q) ----
  constexpr int NQ = 32 * 144 / (FL_NWV * 64);
  f32x4 qv[NQ], cs[NQ];
#pragma unroll
  for (int j = 0; j < NQ; ++j) {
    const int c = tid + j * (FL_NWV * 64);
    const int r = c / 144, k = (c - r * 144) * 4;
    const int hh = hg * 32 + r;
    qv[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    cs[j] = f32x4{1.f, 0.f, 1.f, 0.f};
    if (hh < a.n_heads) {
      if (k < lora) qv[j] = *reinterpret_cast<const f32x4*>(a.q_c + (size_t)hh * lora + k);
      else {
        qv[j] = *reinterpret_cast<const f32x4*>(a.q_rope + (size_t)hh * rope + (k - lora));
        if (a.rotate_q) cs[j] = *reinterpret_cast<const f32x4*>(sp->rope_cs + (k - lora));  // (cos, sin) of pairs (k - lora) / 2, + 1
      }
    }
  }
  const int kv_len = kv_len_override > 0 ? kv_len_override : sp->kv_len;
  const int chunk_len = a.chunk_len > 0 ? a.chunk_len : MLA_FL_CHUNK(kv_len, a.n_chunks);
  const int p0 = blockIdx.x * chunk_len;
  if (p0 >= kv_len || kv_len < a.min_kv) return;  // (uniform; a workgroup past the context drops its Q requests)
  const int p1 = min(kv_len, p0 + chunk_len);
  // 32 rows x 72 sixteen-byte pieces over 512 threads: 4.5 per thread, all in flight at once; rows past the chunk are zero
  constexpr int per_row = KT / 8, NK = (32 * per_row + FL_NWV * 64 - 1) / (FL_NWV * 64);
  u32x4 kv4[NK];
  auto request_rows = [&](int b0) {
    const int nvalid = min(32, p1 - b0);
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + j * (FL_NWV * 64);
      const int r = c / per_row, k = (c - r * per_row) * 8;
      kv4[j] = u32x4{0u, 0u, 0u, 0u};
      if (c < 32 * per_row && r < nvalid) {
        if (k < lora) kv4[j] = *reinterpret_cast<const u32x4*>(a.nope_cache + (size_t)(b0 + r) * lora + k);
        else kv4[j] = *reinterpret_cast<const u32x4*>(a.rope_cache + (size_t)(b0 + r) * rope + (k - lora));
      }
    }
  };
  auto store_rows = [&]() {
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int c = tid + j * (FL_NWV * 64);
      const int r = c / per_row, k = (c - r * per_row) * 8;
      if (c < 32 * per_row) {  // the staged row stride is 8-byte aligned only: two 8-byte stores
        *reinterpret_cast<uint2*>(Ks + r * FL_KSTRIDE + k) = uint2{kv4[j].x, kv4[j].y};
        *reinterpret_cast<uint2*>(Ks + r * FL_KSTRIDE + k + 4) = uint2{kv4[j].z, kv4[j].w};
      }
    }
  };
  request_rows(p0);
  // Q tile of this head group through LDS (coalesced row reads; per-lane strided global reads cost 12 us).  The whole
  // [32][576] tile fits the dynamic LDS of the main loop (not yet in use).  32 x 144 float4 over 512 threads = 9 per
  // thread, ALL requested before the first is stored (the tile was written by other CUs a launch ago: every load is an L2
  // miss; one round trip, not nine).  The rope pairs are rotated by the thread that loaded them (src/infer.cpp:648-685),
  // so that a lane then only picks its strided elements: 8-byte LDS reads, row stride 578 floats.
  // A operands of the score MFMAs (v_mfma_f32_32x32x8_f16: lane (i, kh) holds 4 consecutive k of row i): this wave's 72
  // k-values of Q as nine (hi, lo) f16 quadruples, q = hi + lo to 22 bits; the products with the f16 cache entries are
  // exact in f32 and accumulate in f32, so the scores keep f32 accuracy at half the f32 MFMA's instruction count
  half4 qh[steps / 4], ql[steps / 4];
  {
    constexpr int QST = 578;
    float* Qs = reinterpret_cast<float*>(fl_smem);
#pragma unroll
    for (int j = 0; j < NQ; ++j) {
      const int c = tid + j * (FL_NWV * 64);
      const int r = c / 144, k = (c - r * 144) * 4;
      float* row = Qs + r * QST;
      if (k < lora || !a.rotate_q) {
        *reinterpret_cast<float2*>(row + k) = float2{qv[j].x, qv[j].y};
        *reinterpret_cast<float2*>(row + k + 2) = float2{qv[j].z, qv[j].w};
      } else {
        const float re0 = qv[j].x * cs[j].x - qv[j].y * cs[j].y, im0 = qv[j].x * cs[j].y + qv[j].y * cs[j].x;
        const float re1 = qv[j].z * cs[j].z - qv[j].w * cs[j].w, im1 = qv[j].z * cs[j].w + qv[j].w * cs[j].z;
        if (a.is_v3) {  // rotated in place, interleaved (rope_v3)
          *reinterpret_cast<float2*>(row + k) = float2{re0, im0};
          *reinterpret_cast<float2*>(row + k + 2) = float2{re1, im1};
        } else {        // V2: real parts to [j], imaginary parts to [j + rope / 2]
          const int j0 = (k - lora) >> 1;
          *reinterpret_cast<float2*>(row + lora + j0) = float2{re0, re1};
          *reinterpret_cast<float2*>(row + lora + rope / 2 + j0) = float2{im0, im1};
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < steps / 4; ++m) {
      const float* src = Qs + i * QST + 2 * ks0 + 8 * m + 4 * kh;
      const float2 t0 = *reinterpret_cast<const float2*>(src), t1 = *reinterpret_cast<const float2*>(src + 2);
      const float f[4] = {t0.x, t0.y, t1.x, t1.y};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = hv ? f[e] : 0.f;
        const _Float16 hi = (_Float16)v;
        qh[m][e] = hi;
        ql[m][e] = (_Float16)(v - (float)hi);
      }
    }
    __syncthreads();
  }
  if (tl && tid == 0) tl[1] = wall_clock64();
  constexpr int NTO = 2;  // 32-column output tiles per wave: 512 / 8 / 32
  f32x16 oacc[NTO];
#pragma unroll
  for (int t = 0; t < NTO; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[t][r] = 0.f;
  if (tid < 32) { m_s[tid] = -INFINITY; l_s[tid] = 0.f; }
  const float inv = sqrtf((float)a.head_dim);
  store_rows();  // the chunk's first 32 cache rows (latent | rope) as f16
  for (int b0 = p0; b0 < p1; b0 += 32) {
    const int nvalid = min(32, p1 - b0);
    const bool more = b0 + 32 < p1;
    __syncthreads();
    if (tl && tid == 0 && b0 == p0) tl[2] = wall_clock64();
    if (more) request_rows(b0 + 32);  // the next 32 rows travel while this block is multiplied
    // ---- partial scores of this wave's K range: S[head][pos] ----
    half4 kb[steps / 4];  // B operands: 4 consecutive k of cache row i, as stored (f16): one 8-byte LDS read each
    const unsigned short* krow = Ks + i * FL_KSTRIDE + 2 * ks0 + 4 * kh;
#pragma unroll
    for (int m = 0; m < steps / 4; ++m) kb[m] = __builtin_bit_cast(half4, *reinterpret_cast<const uint2*>(krow + 8 * m));
    f32x16 sacc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
#pragma unroll
    for (int m = 0; m < steps / 4; ++m) {
      sacc = __builtin_amdgcn_mfma_f32_32x32x8f16(qh[m], kb[m], sacc, 0, 0, 0);
      sacc = __builtin_amdgcn_mfma_f32_32x32x8f16(ql[m], kb[m], sacc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) Sp[w][(r & 3) + 8 * (r >> 2) + 4 * kh][i] = sacc[r];
    // value operands of this wave for the whole block (B of v_mfma_f32_32x32x8_f16: 4 consecutive positions of one latent
    // column): requested now, consumed after the softmax
    half4 vb[4][NTO];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int t = 0; t < NTO; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          vb[m][t][e] = __builtin_bit_cast(_Float16, Ks[(8 * m + 4 * kh + e) * FL_KSTRIDE + w * (NTO * 32) + t * 32 + i]);
    __syncthreads();
    if (tl && tid == 0 && b0 == p0) tl[3] = wall_clock64();
    // ---- sum the partial tiles in wave order, online softmax per head row: threads 0..255 -> (row, 4 columns) ----
    if (tid < 256) {
      const int r = tid >> 3, c4 = (tid & 7) * 4;
      float sv[4], mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float acc = 0.f;
#pragma unroll
        for (int ww = 0; ww < FL_NWV; ++ww) acc += Sp[ww][r][c4 + j];
        sv[j] = acc / inv;
        if (c4 + j >= nvalid) sv[j] = -INFINITY;
        mx = fmaxf(mx, sv[j]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 1));
      mx = fmaxf(mx, __shfl_xor(mx, 2));
      mx = fmaxf(mx, __shfl_xor(mx, 4));
      const float m_old = m_s[r], m_new = fmaxf(m_old, mx);
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float pv = c4 + j < nvalid ? expf(sv[j] - m_new) : 0.f;
        Pm[r][c4 + j] = pv;
        ps += pv;
      }
      ps += __shfl_xor(ps, 1);
      ps += __shfl_xor(ps, 2);
      ps += __shfl_xor(ps, 4);
      // the 8 threads of a row are lanes of ONE wave: every read of m_s[r] / l_s[r] above precedes this write
      if ((tid & 7) == 0) {
        al_s[r] = m_old == -INFINITY ? 0.f : expf(m_old - m_new);
        l_s[r] = l_s[r] * al_s[r] + ps;
        m_s[r] = m_new;
      }
    }
    __syncthreads();
    if (tl && tid == 0 && b0 == p0) tl[4] = wall_clock64();
    // ---- O = O * alpha + P . V for this wave's 64 latent columns ----
    half4 ph[4], pl[4];  // P[i][8m + 4kh ..+3] as (hi, lo) f16 quadruples
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = Pm[i][8 * m + 4 * kh + e];
        const _Float16 hi = (_Float16)v;
        ph[m][e] = hi;
        pl[m][e] = (_Float16)(v - (float)hi);
      }
#pragma unroll
    for (int t = 0; t < NTO; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[t][r] *= al_s[(r & 3) + 8 * (r >> 2) + 4 * kh];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int t = 0; t < NTO; ++t) {
        oacc[t] = __builtin_amdgcn_mfma_f32_32x32x8f16(ph[m], vb[m][t], oacc[t], 0, 0, 0);
        oacc[t] = __builtin_amdgcn_mfma_f32_32x32x8f16(pl[m], vb[m][t], oacc[t], 0, 0, 0);
      }
    __syncthreads();  // Ks / Pm are rewritten by the next block
    if (more) store_rows();
    if (tl && tid == 0 && b0 == p0) tl[5] = wall_clock64();
  }
  if (tl && tid == 0) tl[6] = wall_clock64();
  // ---- partials: O (un-normalised), running max and sum ----
  const int chunk = blockIdx.x;
#pragma unroll
  for (int t = 0; t < NTO; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int hrow = hg * 32 + (r & 3) + 8 * (r >> 2) + 4 * kh;
      if (hrow < a.n_heads) a.part_o[((size_t)chunk * a.n_heads + hrow) * lora + w * (NTO * 32) + t * 32 + i] = oacc[t][r];
    }
  }
  if (tid < 32 && hg * 32 + tid < a.n_heads) {
    a.part_ml[((size_t)chunk * a.n_heads + hg * 32 + tid) * 2] = m_s[tid];
    a.part_ml[((size_t)chunk * a.n_heads + hg * 32 + tid) * 2 + 1] = l_s[tid];
  }
  if (tl && tid == 0) tl[7] = wall_clock64();
}
int launch_mla_flash(hipStream_t st, const MlaFlashArgs& a, const StepParams* sp, int kv_len_override, int n_tokens) {
  if (a.lora != 512 || a.rope != 64) DSK_FAIL(DSK_ERR_UNSUPPORTED, "mla flash attention: kv_lora_rank %d / rope %d (512 / 64 only)", a.lora, a.rope);
  if (a.chunk_len < 0 || a.chunk_len % 32 || a.n_chunks < 1) DSK_FAIL(DSK_ERR_INVALID, "mla flash attention: chunk_len %d", a.chunk_len);
  const size_t lds = 32 * FL_KSTRIDE * 2 + FL_NWV * 32 * FL_PSTRIDE * 4 + 32 * FL_PSTRIDE * 4;
  static bool attr_set = false;
  if (!attr_set) { hipFuncSetAttribute((const void*)mla_flash_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); attr_set = true; }
  hipLaunchKernelGGL(mla_flash_kernel, dim3(a.n_chunks, (a.n_heads + 31) / 32, n_tokens), dim3(FL_NWV * 64), lds, st, a, sp, kv_len_override);
  return DSK_OK;
}

// merge the chunk partials of one head: out = sum_c e^(m_c - M) O_c / sum_c e^(m_c - M) l_c
__global__ __launch_bounds__(512) void mla_merge_kernel(MlaFlashArgs a, const StepParams* __restrict__ sp, int kv_len_override, float* __restrict__ out) {
  const int h = blockIdx.x, tid = threadIdx.x;
  const int kv_len = kv_len_override > 0 ? kv_len_override : sp->kv_len;
  const int chunk_len = a.chunk_len > 0 ? a.chunk_len : MLA_FL_CHUNK(kv_len, a.n_chunks);
  const int nc = min(a.n_chunks, (kv_len + chunk_len - 1) / chunk_len);
  float M = -INFINITY;
  for (int c = 0; c < nc; ++c) M = fmaxf(M, a.part_ml[((size_t)c * a.n_heads + h) * 2]);
  float L = 0.f;
  for (int c = 0; c < nc; ++c) L += expf(a.part_ml[((size_t)c * a.n_heads + h) * 2] - M) * a.part_ml[((size_t)c * a.n_heads + h) * 2 + 1];
  for (int i = tid; i < a.lora; i += 512) {
    float o = 0.f;
    for (int c = 0; c < nc; ++c) o = fmaf(expf(a.part_ml[((size_t)c * a.n_heads + h) * 2] - M), a.part_o[((size_t)c * a.n_heads + h) * a.lora + i], o);
    out[(size_t)h * a.lora + i] = o / L;
  }
}
int launch_mla_merge(hipStream_t st, const MlaFlashArgs& a, const StepParams* sp, int kv_len_override, float* out) {
  hipLaunchKernelGGL(mla_merge_kernel, dim3(a.n_heads), dim3(512), 0, st, a, sp, kv_len_override, out);
  return DSK_OK;
}

int launch_rope_kv_mla(hipStream_t st, const AttnMlaArgs& a, const StepParams* sp) {
  if (a.rope > 128 || (a.rope & 1)) DSK_FAIL(DSK_ERR_UNSUPPORTED, "rope dim %d (max 128, even)", a.rope);
  hipLaunchKernelGGL(rope_kv_mla_kernel, dim3(a.n_heads), dim3(256), 0, st, a, sp);
  return DSK_OK;
}

// attn_mla (per head), src/infer.cpp:766-804.  All heads read the same latent cache (L2-resident).
__global__ __launch_bounds__(256) void attn_mla_kernel(AttnMlaArgs a, const StepParams* __restrict__ sp, int kv_len_override) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float scratch[4];
  float* att = reinterpret_cast<float*>(smem);
  const int h = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lora = a.lora, rope = a.rope;
  const int kv_len = kv_len_override > 0 ? kv_len_override : sp->kv_len;
  const float* qc = a.q_c + (size_t)h * lora;
  const float* qr = a.q_rope + (size_t)h * rope;
  const float inv = sqrtf((float)a.head_dim);
  for (int t = wave; t < kv_len; t += 4) {
    float p = 0.f;
    const uint16_t* c = a.nope_cache + (size_t)t * lora;
    for (int i = lane * 4; i < lora; i += 256) {
      const f16x4 k = *reinterpret_cast<const f16x4*>(c + i);
      const f32x4 qq = *reinterpret_cast<const f32x4*>(qc + i);
      p = fmaf(qq.x, (float)k.x, p);
      p = fmaf(qq.y, (float)k.y, p);
      p = fmaf(qq.z, (float)k.z, p);
      p = fmaf(qq.w, (float)k.w, p);
    }
    const uint16_t* r = a.rope_cache + (size_t)t * rope;
    for (int i = lane; i < rope; i += 64) p = fmaf(qr[i], h2f(r[i]), p);
    p = wave_sum(p);
    if (lane == 0) att[t] = p / inv;
  }
  __syncthreads();
  float mx = -INFINITY;
  for (int t = tid; t < kv_len; t += 256) mx = fmaxf(mx, att[t]);
  mx = block_max(mx, scratch, tid, 256);
  float sum = 0.f;
  for (int t = tid; t < kv_len; t += 256) {
    const float e = expf(att[t] - mx);
    att[t] = e;
    sum += e;
  }
  sum = block_sum(sum, scratch, tid, 256);
  for (int t = tid; t < kv_len; t += 256) att[t] = att[t] / sum;
  __syncthreads();
  for (int i = tid; i < lora; i += 256) {
    float acc = 0.f;
    for (int t = 0; t < kv_len; ++t) acc = fmaf(att[t], h2f(a.nope_cache[(size_t)t * lora + i]), acc);
    a.out[(size_t)h * lora + i] = acc;
  }
}
int launch_attn_mla(hipStream_t st, const AttnMlaArgs& a, const StepParams* sp, int kv_len_override, int max_kv) {
  if (a.lora % 4) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn_mla: kv_lora_rank %d", a.lora);
  const size_t lds = (size_t)max_kv * 4;
  if (lds > 150 * 1024) DSK_FAIL(DSK_ERR_UNSUPPORTED, "attn_mla: kv_len %d does not fit LDS", max_kv);
  if (lds > 64 * 1024) hipFuncSetAttribute((const void*)attn_mla_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(attn_mla_kernel, dim3(a.n_heads), dim3(256), lds, st, a, sp, kv_len_override);
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// synthetic weights generated directly in HBM (220 GB does not fit host storage).
// Counter-based hash RNG => deterministic in (seed, index), independent of launch geometry.
// ------------------------------------------------------------------------------------
DEV uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
DEV float u01(uint64_t r) { return (float)((r >> 40) + 1) * (1.0f / 16777217.0f); }
DEV float gauss(uint64_t seed, uint64_t i) {
  const uint64_t r = mix64(seed ^ (i * 0xD1342543DE82EF95ull));
  const float u1 = u01(r), u2 = u01(mix64(r));
  return sqrtf(-2.0f * logf(u1)) * cosf(6.28318530718f * u2);
}

__global__ void fill_u32_kernel(u32* p, size_t n, uint64_t seed) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = (u32)mix64(seed ^ (i * 0x9E3779B97F4A7C15ull));
}
// Q2_K d/dmin: w = d*sc*q - dmin*m with uniform nibbles has std ~13.9 d and zero mean for dmin = 1.5 d
__global__ void fill_dm_q2k_kernel(u32* dm, size_t n_blocks, uint64_t seed, float wscale) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_blocks; i += (size_t)gridDim.x * blockDim.x) {
    const uint64_t r = mix64(seed ^ (i * 0xA24BAED4963EE407ull));
    const float d = (0.5f + u01(r)) * wscale / 13.9f;
    dm[i] = (u32)f2h(d) | ((u32)f2h(1.5f * d) << 16);
  }
}
// tiled Q2_K (tile_device.h): the d | dmin words of every tile (16 words at byte 1280 of each 1344-byte record); rows past
// `rows` of a matrix are padding: d = dmin = 0
__global__ void fill_dm_tiles_kernel(uint8_t* tiles, size_t n_tiles, int rows, int nb, uint64_t seed, float wscale) {
  const size_t strips_per_mat = (size_t)((rows + 15) >> 4);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_tiles * 16; i += (size_t)gridDim.x * blockDim.x) {
    const size_t tile = i >> 4;
    const int n = (int)(i & 15);
    const size_t strip = tile / nb;
    const int row = (int)(strip % strips_per_mat) * 16 + n;
    const uint64_t r = mix64(seed ^ (i * 0xA24BAED4963EE407ull));
    const float d = (0.5f + u01(r)) * wscale / 13.9f;
    *reinterpret_cast<u32*>(tiles + tile * 1344 + 1280 + 4 * n) = row < rows ? ((u32)f2h(d) | ((u32)f2h(1.5f * d) << 16)) : 0u;
  }
}
// Q3_K: (sc-32)*q has std ~43 for uniform fields
__global__ void fill_d_q3k_kernel(unsigned short* dm, size_t n_blocks, uint64_t seed, float wscale) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_blocks; i += (size_t)gridDim.x * blockDim.x) {
    const uint64_t r = mix64(seed ^ (i * 0xA24BAED4963EE407ull));
    dm[i] = f2h((0.5f + u01(r)) * wscale / 43.3f);
  }
}
__global__ void fill_f32_kernel(float* p, size_t n, uint64_t seed, float mean, float std) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = mean + std * gauss(seed, i);
}
__global__ void fill_f16_kernel(unsigned short* p, size_t n, uint64_t seed, float std) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = f2h(std * gauss(seed, i));
}
__global__ void fill_f8_kernel(uint8_t* p, size_t n, uint64_t seed) {  // N(0,1) truncated to e5m2 (src/codec.h:49-57)
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = (uint8_t)(f2h(gauss(seed, i)) >> 8);
}
__global__ void fill_uniform_f32_kernel(float* p, size_t n, uint64_t seed, float lo, float hi) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = lo + (hi - lo) * u01(mix64(seed ^ (i * 0x9E3779B97F4A7C15ull)));
}

static unsigned fill_grid(size_t n) {
  size_t g = (n + 255) / 256;
  return (unsigned)(g > 8192 ? 8192 : (g ? g : 1));
}

int launch_fill_f32(hipStream_t st, float* p, size_t n, uint64_t seed, float mean, float std) {
  hipLaunchKernelGGL(fill_f32_kernel, dim3(fill_grid(n)), dim3(256), 0, st, p, n, seed, mean, std);
  return DSK_OK;
}

// Fill every plane of a (possibly expert-stacked) weight tensor.  wscale = target std of a weight.
int launch_fill_tensor(hipStream_t st, const DTensor& t, uint64_t seed, float wscale) {
  const size_t mats = t.n_experts > 0 ? (size_t)t.local_experts : 1;
  const size_t numel = mats * (size_t)t.rows * t.n;
  switch (t.quant) {
    case DSK_QUANT_F32:
      hipLaunchKernelGGL(fill_f32_kernel, dim3(fill_grid(numel)), dim3(256), 0, st, reinterpret_cast<float*>(t.qs), numel, seed, 0.f, wscale);
      break;
    case DSK_QUANT_F16:
      hipLaunchKernelGGL(fill_f16_kernel, dim3(fill_grid(numel)), dim3(256), 0, st, reinterpret_cast<unsigned short*>(t.qs), numel, seed, wscale);
      break;
    case DSK_QUANT_F8E5M2: {
      hipLaunchKernelGGL(fill_f8_kernel, dim3(fill_grid(numel)), dim3(256), 0, st, t.qs, numel, seed);
      const size_t ns = mats * t.e_scale;
      hipLaunchKernelGGL(fill_uniform_f32_kernel, dim3(fill_grid(ns)), dim3(256), 0, st, t.scale, ns, seed ^ 0x5ca1e, 0.5f * wscale, 1.5f * wscale);
      break;
    }
    case DSK_QUANT_Q2_K: {
      if (t.tiled) {
        const size_t n_tiles = mats * (size_t)((t.rows + 15) >> 4) * (t.n >> 8);
        hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(n_tiles * 336)), dim3(256), 0, st, reinterpret_cast<u32*>(t.qs), n_tiles * 336, seed);
        hipLaunchKernelGGL(fill_dm_tiles_kernel, dim3(fill_grid(n_tiles * 16)), dim3(256), 0, st, t.qs, n_tiles, t.rows, t.n >> 8, seed ^ 0xd3, wscale);
        break;
      }
      const size_t nblk = numel / 256;
      hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(nblk * 16)), dim3(256), 0, st, reinterpret_cast<u32*>(t.qs), nblk * 16, seed);
      hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(nblk * 4)), dim3(256), 0, st, reinterpret_cast<u32*>(t.sc), nblk * 4, seed ^ 0x51);
      hipLaunchKernelGGL(fill_dm_q2k_kernel, dim3(fill_grid(nblk)), dim3(256), 0, st, reinterpret_cast<u32*>(t.dm), nblk, seed ^ 0xd3, wscale);
      break;
    }
    case DSK_QUANT_Q3_K: {
      const size_t nblk = numel / 256;
      hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(nblk * 16)), dim3(256), 0, st, reinterpret_cast<u32*>(t.qs), nblk * 16, seed);
      hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(nblk * 8)), dim3(256), 0, st, reinterpret_cast<u32*>(t.hm), nblk * 8, seed ^ 0x77);
      hipLaunchKernelGGL(fill_u32_kernel, dim3(fill_grid(nblk * 3)), dim3(256), 0, st, reinterpret_cast<u32*>(t.sc), nblk * 3, seed ^ 0x51);
      hipLaunchKernelGGL(fill_d_q3k_kernel, dim3(fill_grid(nblk)), dim3(256), 0, st, reinterpret_cast<unsigned short*>(t.dm), nblk, seed ^ 0xd3, wscale);
      break;
    }
    default: DSK_FAIL(DSK_ERR_INVALID, "fill: bad quant");
  }
  return DSK_OK;
}

// ------------------------------------------------------------------------------------
// streaming-read probe: the "measured roofline" denominator
// ------------------------------------------------------------------------------------
// Every wave streams its own contiguous share with 8 sixteen-byte loads per lane in flight, re-issued as they are consumed
// (tools/ldsdma_probe.hip, mode 0: 6.7-6.8 TB/s on MI355X, 26.5 GB/s per CU at 256 workgroups and 43 GB/s per CU at 128 - the
// grid-stride form with 4 loads per lane that rounds 1-3 used measured 6.05-6.26 TB/s: the denominator of every
// "fraction of measured" was 8-10 % too low).
__global__ __launch_bounds__(1024) void read_bw_kernel(const uint8_t* __restrict__ p, size_t bytes_per_wave, float* sink) {
  constexpr int D = 8;
  constexpr int BUF_NT = 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t wid = (size_t)blockIdx.x * 16 + wave;
  const unsigned long long base = (unsigned long long)(p + wid * bytes_per_wave);
  const u32 blo = __builtin_amdgcn_readfirstlane((u32)base), bhi = __builtin_amdgcn_readfirstlane((u32)(base >> 32));
  const __amdgpu_buffer_rsrc_t R = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((unsigned long long)bhi << 32) | blo), 0, -1, 0x00020000);
  const int steps = (int)(bytes_per_wave >> 10);  // 1 KiB per wave and step
  u32x4 v[D];
  u32 acc = 0;
#pragma unroll
  for (int d = 0; d < D; ++d) v[d] = __builtin_amdgcn_raw_buffer_load_b128(R, lane * 16, d << 10, BUF_NT);
  for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const u32x4 w = v[d];
      acc += w.x + w.y + w.z + w.w;
      if (s0 + D + d < steps) v[d] = __builtin_amdgcn_raw_buffer_load_b128(R, lane * 16, (s0 + D + d) << 10, BUF_NT);
    }
  }
  if (acc == 0x12345678u) *sink = 1.f;  // keep the loads alive
}
int launch_read_bw(hipStream_t st, const void* p, size_t bytes, float* sink) {
  // 256 sixteen-wave workgroups; the share of a wave is a whole number of 8 KiB (steps in multiples of the depth)
  const size_t per_wave = bytes / (256 * 16) / 8192 * 8192;
  if (per_wave == 0 || per_wave > (1u << 30)) DSK_FAIL(DSK_ERR_INVALID, "read_bw: %zu bytes", bytes);
  hipLaunchKernelGGL(read_bw_kernel, dim3(256), dim3(1024), 0, st, static_cast<const uint8_t*>(p), per_wave, sink);
  return DSK_OK;
}
