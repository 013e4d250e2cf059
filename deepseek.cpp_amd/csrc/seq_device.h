// seq_device.h -- device pieces shared by the kernels of layered models: activation types, matrix fragments, reductions.
//
// Activations are T = bf16 or float; weights are always bf16 in HBM (a 32-bit run multiplies their exact values).  Every matrix
// lives as FRAGMENTS of 16 rows x 32 columns: 64 lanes x 8 consecutive k, lane = (k / 8) * 16 + row, 1 KiB contiguous - the
// operand order of v_mfma_f32_16x16x32_bf16.  A wave reads a fragment with one 16-byte load per lane from consecutive
// addresses, in HBM and in LDS alike.  A 32-bit run multiplies the same fragments with eight v_mfma_f32_16x16x4_f32: step j
// takes element j of every lane, so lane groups stand for the k values {8 g + j}.  Its prompt products take each activation apart
// into three bf16 numbers instead (Split).
#pragma once
#include "dsk_internal.h"
#include "glob_device.h"
#include "lane_device.h"
#include "layered_kernels.h"

typedef __bf16 bf16;
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
#define DEV __device__ __forceinline__
DEV SeqDesc seq_at(const SeqDesc* p) {
  SeqDesc s = *p;
  s.state = glob(s.state);
  return s;
}
// the same by vector loads: scalar loads come back in any order, so that the first use of any value out of the kernel's arguments waits for all of them
DEV SeqDesc seq_late(const SeqDesc* p) {
  int zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  return seq_at(glob(p) + zero);
}

template <typename T>
struct Frag;
template <>
struct Frag<bf16> {
  typedef bf16x8 type;
  typedef bf16x4 four;
};
template <>
struct Frag<float> {
  typedef f32x8 type;
  typedef f32x4 four;
};

DEV f32x4 mma(const bf16x8& w, const bf16x8& a, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, c, 0, 0, 0); }
DEV f32x4 mma(const bf16x8& w, const f32x8& a, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 8; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32((float)w[j], a[j], c, 0, 0, 0);
  return c;
}
DEV f32x4 mma(const f32x8& w, const f32x8& a, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 8; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], a[j], c, 0, 0, 0);
  return c;
}

// A finite 32-bit activation as the exact sum of three bf16 numbers: its top 8 significant bits, the next 8, the last 8 (cut off, not rounded, so
// that each rest is exact; b2 alone can fall under the smallest bf16, below 2^-110).  A product with a finite bf16 weight is then three bf16
// products, each exact in 32 bits and summed in 32 bits: the precision of v_mfma_f32_16x16x4_f32 at a fifth of its cycles (three
// 16x16x32 of 16 cycles for eight of 32).  Where an activation or a weight is not finite the sum of the three is no finite number either,
// but not always the right one: such sums are added up again by that instruction (rows_body).
typedef unsigned u32x4v __attribute__((ext_vector_type(4)));
struct Split {
  u32x4v b[3];  // eight bf16 each
};
DEV void split_pair(const f32x8& x, int i, Split& o) {  // elements 2 i and 2 i + 1
  unsigned p[3][2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float v = x[2 * i + e];  // (a bit cast of an element of a vector reads element 0)
    const unsigned bits = __builtin_bit_cast(unsigned, v);
    const float r = v - __builtin_bit_cast(float, bits & 0xffff0000u);  // (of an infinity or no number: no number)
    const unsigned rest = __builtin_bit_cast(unsigned, r);
    p[0][e] = bits;
    p[1][e] = rest;
    p[2][e] = __builtin_bit_cast(unsigned, r - __builtin_bit_cast(float, rest & 0xffff0000u));
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) o.b[k][i] = __builtin_amdgcn_perm(p[k][1], p[k][0], 0x07060302);  // the high halves of two words
}

// A block of 16 rows x 32 columns on its way from row-major memory to operands: loaded row by row, four lanes to a row, lane l's 8 columns
// at place l of the block in LDS.  Inside a row the groups are exchanged by the row's place, so that the lanes that read one group of 16 rows
// meet every LDS bank once.
DEV int block_row(int lane) { return lane >> 2; }                                              // what lane l loads ...
DEV int block_group(int lane) { return (lane & 3) ^ (lane >> 4); }
DEV int block_place(int lane) { return (lane & 15) * 4 + ((lane >> 4) ^ ((lane >> 2) & 3)); }  // ... and the place that lane l of an operand reads

template <typename T>
DEV typename Frag<T>::four to_four(const f32x4& v) {
  return __builtin_convertvector(v, typename Frag<T>::four);
}

// a barrier for LDS traffic only: global loads and stores stay in flight across it (__syncthreads drains them)
// The wait is stated twice: the compiler does not know of the one inside the assembly, and without the first it makes the first instruction that uses
// what was read in front of the barrier wait for everything that is read behind it.
DEV void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

DEV float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
DEV float silu_f(float x) { return x * sigmoid_f(x); }
DEV float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
DEV float logsigmoid_f(float x) { return -softplus_f(-x); }

DEV float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += lane_xor(v, off);
  return v;
}
// sum over a row of 16 lanes, result in all of them: four DPP adds
template <int CTRL>
DEV float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
DEV float row_sum(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_f<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_f<0x141>(v);  // row_half_mirror
  v += dpp_f<0x140>(v);  // row_mirror
  return v;
}
// a product that is rounded: not to be fused with a sum
DEV float product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
// The sum of a thread's N x V squares in one order of roundings: the square at `rounded` is, all others go into the sum as they are, in order.  (Left to
// itself the compiler rounds the first or the second, by what stands around it.  A norm's last bit moves the bfloat16 roundings behind it, and a router's
// close calls follow those: results would change with the neighbourhood of this sum.)
template <int N, int V, int ROUNDED = 1, typename R>
DEV float squares(const R (&x)[N]) {
  constexpr int F = ROUNDED < N * V ? ROUNDED : 0;
  float s = product(x[F / V][F % V], x[F / V][F % V]);
#pragma unroll
  for (int i = 0; i < N * V; ++i)
    if (i != F) s = fmaf(x[i / V][i % V], x[i / V][i % V], s);
  return s;
}
// sum over a workgroup of NT threads, result in every thread; scratch: NT / 64 floats of LDS
template <int NT>
DEV float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) s += scratch[i];
  return s;
}

// Workgroups go round robin over the 8 XCDs, each with an L2 of its own: XCD x takes the x-th eighth of the work, in order, so that neighbours, which
// read the same weights or operands, meet in one L2.
DEV int xcd_range(int b, int n) {
  const int x = b & 7, base = n >> 3, extra = n & 7;
  return x * base + min(x, extra) + (b >> 3);
}
