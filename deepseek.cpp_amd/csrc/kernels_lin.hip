// kernels_lin.hip -- matrix products of layered models on fragment-packed bf16 weights (seq_device.h), and the packing itself.
//
//   lin_kernel      prompts: 128 features x 128 rows per workgroup, 4 waves of 64 x 64, both operands through LDS in fragment
//                   order (global_load_lds, 16 bytes per lane: LDS reads are lane-linear, no bank conflicts), two buffers
//   rows_kernel     the same in 32 bits, 128 features x 128 or 64 rows, each wave with rows of its own
//   lin_big_kernel  lin_kernel's with 256 x 256 and a ring of four stages, where there are enough of such tiles (bf16)
//   lin_direct_kernel  32-bit activations times a few k tiles, operands straight from memory
//   few_kernel      up to 16 rows (decoding): 4 waves share 16 or 64 features and split k; weights stream from HBM straight into the
//                   MFMA operand registers, 1 KiB contiguous per wave and load
//   expert_kernel   the experts' products of prompts, rows gathered per expert: 256 features x 128 (64, 32) rows, weights straight
//                   into registers (32 bits: rows_kernel's tiles)
// few_kernel takes plain products and the experts', several of them in one launch.
#include "layered_kernels.h"
#include "lin_device.h"

#include <math.h>

#include <algorithm>

typedef const __attribute__((address_space(1))) void* gptr;
typedef __attribute__((address_space(3))) void* lptr;

static int cdiv(int a, int b) { return (a + b - 1) / b; }

// ---- packing -----------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pack_kernel(const uint16_t* __restrict__ src, int rows, int k, uint16_t* __restrict__ dst, int kt, int row0, int col0,
                                                   int interleave, int transpose) {
  const size_t n = (size_t)rows * k;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const int r = (int)(transpose ? i % k : i / k), c = (int)(transpose ? i / k : i % k) + col0;
    const int tile = interleave >= 0 ? 2 * (r >> 4) + interleave : (r + row0) >> 4;
    const int rr = interleave >= 0 ? r & 15 : (r + row0) & 15;
    dst[((size_t)tile * kt + (c >> 5)) * 512 + (((c & 31) >> 3) * 16 + rr) * 8 + (c & 7)] = src[i];
  }
}
int launch_pack(hipStream_t st, const uint16_t* src, int rows, int k, uint16_t* dst, int kt, int row0, int col0, int interleave, bool transpose) {
  const size_t n = (size_t)rows * k;
  hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, st, src, rows, k, dst, kt, row0, col0, interleave, (int)transpose);
  return DSK_OK;
}
__global__ __launch_bounds__(256) void widen_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    dst[i] = __builtin_bit_cast(float, (unsigned)src[i] << 16);
}
int launch_widen(hipStream_t st, const uint16_t* src, float* dst, size_t n) {
  hipLaunchKernelGGL(widen_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, src, dst, n);
  return DSK_OK;
}
__global__ __launch_bounds__(256) void exp_kernel(float* __restrict__ x, int n) {
  for (int i = threadIdx.x; i < n; i += 256) x[i] = expf(x[i]);
}
int launch_exp(hipStream_t st, float* x, int n) {
  hipLaunchKernelGGL(exp_kernel, dim3(1), dim3(256), 0, st, x, n);
  return DSK_OK;
}
DEV float random_pm1(uint64_t seed, size_t i) {  // splitmix64 of the index
  uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(int)(z >> 40) * (2.f / 16777216.f) - 1.f;
}
template <typename D>
__global__ __launch_bounds__(256) void random_kernel(D* __restrict__ dst, size_t n, float scale, uint64_t seed) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = (D)(scale * random_pm1(seed, i));
}
int launch_fill_random(hipStream_t st, uint16_t* dst, size_t n, float scale, uint64_t seed) {
  if (n) hipLaunchKernelGGL(random_kernel<bf16>, dim3(4096), dim3(256), 0, st, reinterpret_cast<bf16*>(dst), n, scale, seed);
  return DSK_OK;
}
int launch_fill_random_f32(hipStream_t st, float* dst, size_t n, float scale, uint64_t seed) {
  if (n) hipLaunchKernelGGL(random_kernel<float>, dim3(256), dim3(256), 0, st, dst, n, scale, seed);
  return DSK_OK;
}

// ---- prompts -------------------------------------------------------------------------------------
// What a workgroup keeps in LDS.  bf16: two stages of two k tiles (8 weight tiles and 8 row groups each), 64 KiB; deeper rings with a barrier
// per k tile were no faster (two workgroups on a compute unit hide each other's waits).
enum { LIN_STEP = 2, LIN_STAGE = LIN_STEP * 16 * 1024, LIN_LDS = 2 * LIN_STAGE };
enum { LONE_RING = 4 };  // stages of one k tile, 64 KiB as well
static_assert(LONE_RING * 16 * 1024 == LIN_LDS, "one size for both");
// 32 bits, 64 J rows: a ring of three stages of one k tile (8 weight tiles, 4 J row groups of two KiB), 72 or 48 KiB.
enum { ROWS_RING = 3 };
template <int J>
__host__ DEV constexpr int rows_stage() { return 8 * 1024 * (1 + J); }
// 32 features (tiles rt, rt + 1) x 32 rows (from `first` on) of a wave by itself on v_mfma_f32_16x16x4_f32, operands straight from memory: one chain of
// the instruction per sum.  f0: a feature whose operand it is.
template <int EPI>
DEV void direct_tile(const LinArgs& a, const int* gather, int row0, int n_rows, int f0, int rt, int first, int k0, int k1) {
  const int lane = threadIdx.x & 63;
  const bf16x8* w[2];
  const float* x[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    w[i] = reinterpret_cast<const bf16x8*>(a.w) + (size_t)min(rt + i, a.rt - 1) * a.kt * 64 + lane;
    int r = min(first + i * 16 + (lane & 15), n_rows - 1);
    r = gather ? gather[row0 + r] : row0 + r;
    x[i] = operand<float>(a, f0) + (size_t)r * a.lda + (lane >> 4) * 8;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int kt = k0; kt < k1; kt += 2) {  // (k1 - k0 is even)
    bf16x8 wk[2][2];
    f32x8 xk[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        wk[u][i] = w[i][(size_t)(kt + u) * 64];
        xk[u][i] = *reinterpret_cast<const f32x8*>(x[i] + (size_t)(kt + u) * 32);
      }
    __builtin_amdgcn_sched_barrier(0);  // (all on their way first)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mma(wk[u][i], xk[u][j], acc[i][j]);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = first + j * 16 + (lane & 15);
    if (r >= n_rows || rt >= a.rt) continue;
    if constexpr (EPI == LIN_GLU) {
      store_glu<float>(a, row0 + r, (rt >> 1) * 16 + (lane >> 4) * 4, acc[0][j], acc[1][j]);
    } else {
      store_plain<float, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[0][j]);
      if (rt + 1 < a.rt) store_plain<float, EPI>(a, row0 + r, rt * 16 + 16 + (lane >> 4) * 4, acc[1][j]);
    }
  }
}
// 128 features from f0 on x n_rows <= 128 rows, k tiles [k0, k1), bf16: 4 waves of 64 x 64.
template <int EPI>
DEV void lin_body(const LinArgs& a, int row0, int n_rows, int f0, int k0, int k1, char* lds) {
  constexpr int KS = LIN_STEP, WB = 8 * KS * 1024;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1, n = k1 - k0;
  const int rt0 = f0 >> 4;
  // this wave's share of the staging: two weight tiles and two row groups, the k tiles of a stage
  const char *src_w[2], *src_a[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)  // (tiles past the end: any valid one, never stored)
    src_w[i] = reinterpret_cast<const char*>(a.w) + ((size_t)min(rt0 + 2 * wave + i, a.rt - 1) * a.kt + k0) * 1024 + lane * 16;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = row0 + min((2 * wave + i) * 16 + block_row(lane), n_rows - 1);
    src_a[i] = reinterpret_cast<const char*>(operand<bf16>(a, f0) + (size_t)r * a.lda + (size_t)k0 * 32) + block_group(lane) * 16;
  }
  auto stage = [&](int kt, char* buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        __builtin_amdgcn_global_load_lds((gptr)(src_w[i] + (size_t)(kt + kk) * 1024), (lptr)(buf + ((2 * wave + i) * KS + kk) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        __builtin_amdgcn_global_load_lds((gptr)(src_a[i] + (size_t)(kt + kk) * 64), (lptr)(buf + WB + ((2 * wave + i) * KS + kk) * 1024), 16, 0, 0);
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  stage(0, lds);
  for (int kt = 0; kt < n; kt += KS) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads into LDS; the barrier makes it everybody's
    __syncthreads();
    char* cur = lds + ((kt / KS) & 1) * LIN_STAGE;
    if (kt + KS < n) stage(kt + KS, lds + (((kt / KS) & 1) ^ 1) * LIN_STAGE);
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      bf16x8 w[4], x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const bf16x8*>(cur + ((wm * 4 + i) * KS + kk) * 1024 + lane * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = *reinterpret_cast<const bf16x8*>(cur + WB + ((wn * 4 + j) * KS + kk) * 1024 + block_place(lane) * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mma(w[i], x[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = wn * 64 + j * 16 + (lane & 15);
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rt = rt0 + wm * 4 + i;
      if (rt < a.rt) store_plain<bf16, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[i][j]);
    }
  }
}
// The same where workgroups have a compute unit each: nobody else hides their waits.  While a k tile is multiplied the next one's operands are read into the
// other set of registers and the loads of LONE_RING - 1 more are on their way.  k = 2048, up to 256 workgroups: 20.4 - 24 us -> 15.5 - 18, with weights
// out of HBM (2048 x 27648, 216 workgroups of 40 rows, k = 7168) 107 -> 77; but of two on a compute unit each (300 rows x 16896, k = 2048) 33.6 -> 34.4, and
// 1100 rows x 27648, k = 7168 462 -> 550.  A ring of three: as fast, 93 us out of HBM.
template <int EPI>
DEV void lone_body(const LinArgs& a, int row0, int n_rows, int f0, int k0, int k1, char* lds) {
  constexpr int R = LONE_RING, STAGE = 16 * 1024, WB = 8 * 1024;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1, n = k1 - k0;
  const int rt0 = f0 >> 4;
  // this wave's share of the staging: two weight tiles and two row groups
  const char *src_w[2], *src_a[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)  // (tiles past the end: any valid one, never stored)
    src_w[i] = reinterpret_cast<const char*>(a.w) + ((size_t)min(rt0 + 2 * wave + i, a.rt - 1) * a.kt + k0) * 1024 + lane * 16;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = row0 + min((2 * wave + i) * 16 + block_row(lane), n_rows - 1);
    src_a[i] = reinterpret_cast<const char*>(operand<bf16>(a, f0) + (size_t)r * a.lda + (size_t)k0 * 32) + block_group(lane) * 16;
  }
  auto stage = [&](int kt, char* buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_amdgcn_global_load_lds((gptr)(src_w[i] + (size_t)kt * 1024), (lptr)(buf + (2 * wave + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_amdgcn_global_load_lds((gptr)(src_a[i] + (size_t)kt * 64), (lptr)(buf + WB + (2 * wave + i) * 1024), 16, 0, 0);
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Operands {
    bf16x8 w[4], x[4];
  };
  auto read = [&](const char* buf, int i, Operands& o) {
    o.w[i] = *reinterpret_cast<const bf16x8*>(buf + (wm * 4 + i) * 1024 + lane * 16);
    o.x[i] = *reinterpret_cast<const bf16x8*>(buf + WB + (wn * 4 + i) * 1024 + block_place(lane) * 16);
  };
  int cur = 0;
  auto step = [&](int kt, const Operands& now, Operands& next) {
    // tile kt + 1 is here when at most the loads of R - 2 tiles are outstanding; behind the barrier everybody's are, and everybody holds
    // tile kt in registers, so that its buffer takes tile kt + R (past the end: the last one again, never read)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (R - 2)) : "memory");
    lds_barrier();
    stage(min(kt + R, n - 1), lds + cur * STAGE);
    cur = cur + 1 == R ? 0 : cur + 1;
    const char* buf = lds + cur * STAGE;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // two reads beside four matrix instructions
      read(buf, i, next);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mma(now.w[i], now.x[j], acc[i][j]);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  Operands p, q;
#pragma unroll
  for (int i = 0; i < R; ++i) stage(min(i, n - 1), lds + i * STAGE);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (R - 1)) : "memory");
  lds_barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i) read(lds, i, p);
  for (int kt = 0; kt < n; kt += 2) {  // (n is even)
    step(kt, p, q);
    step(kt + 1, q, p);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = wn * 64 + j * 16 + (lane & 15);
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rt = rt0 + wm * 4 + i;
      if (rt < a.rt) store_plain<bf16, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[i][j]);
    }
  }
}
// 128 features from f0 on x n_rows <= 64 J rows, k tiles [k0, k1), 32 bits: 4 waves of 128 features x 16 J rows.  gather: a table (slot -> row) or
// nullptr; out rows are row0 + local row.
// Activations are taken apart into three bf16 numbers (split_pair, 44 vector instructions for 16 rows of a k tile, 176 cycles); a wave has rows of its own, so
// that no two of them take the same ones apart: per wave and k tile 24 J matrix instructions (384 J cycles) and 44 J vector instructions beside them.
// While a k tile is multiplied the next one's operands are read and taken apart, and the loads of ROWS_RING - 1 more are on their way (rings of four and
// five were not faster, and leave room for a workgroup less).  The matrix instructions bound it where compute units are full (128 rows: 1.23 us for two
// workgroups' steps of 64 columns, of 1.28), what a wave does alone where they are not.  4 waves of 64 x 64, each row taken apart by two of them and that
// work behind the matrix work, took 99 us for 301 x 2048 x 16896, 100 for 301 x 16896 x 2048 and 42 - 65 for 301 x 2048 x 2176 - 8320; this 62, 62 and
// 25 - 39, with v_mfma_f32_16x16x4_f32 the first was 303.
template <int J, int EPI>
DEV void rows_body(const LinArgs& a, const int* gather, int row0, int n_rows, int f0, int k0, int k1, char* lds) {
  constexpr int R = ROWS_RING, STAGE = rows_stage<J>(), WB = 8 * 1024, LOADS = 2 + 2 * J;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = k1 - k0;
  const int rt0 = f0 >> 4, own = wave * 16 * J;
  // this wave's share of the staging: two weight tiles and its own rows (a block of 16 x 32 floats is two loads of 8 rows)
  const char *src_w[2], *src_a[2 * J];
#pragma unroll
  for (int i = 0; i < 2; ++i)  // (tiles past the end: any valid one, never stored)
    src_w[i] = reinterpret_cast<const char*>(a.w) + ((size_t)min(rt0 + 2 * wave + i, a.rt - 1) * a.kt + k0) * 1024 + lane * 16;
#pragma unroll
  for (int h = 0; h < 2 * J; ++h) {
    int r = min(own + h * 8 + (lane >> 3), n_rows - 1);
    r = gather ? gather[row0 + r] : row0 + r;
    src_a[h] = reinterpret_cast<const char*>(operand<float>(a, f0) + (size_t)r * a.lda + (size_t)k0 * 32) + ((lane & 7) ^ (lane >> 3)) * 16;
  }
  auto stage = [&](int kt, char* buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_amdgcn_global_load_lds((gptr)(src_w[i] + (size_t)kt * 1024), (lptr)(buf + (2 * wave + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int h = 0; h < 2 * J; ++h) __builtin_amdgcn_global_load_lds((gptr)(src_a[h] + (size_t)kt * 128), (lptr)(buf + WB + (wave * 2 * J + h) * 1024), 16, 0, 0);
  };
  f32x4 acc[8][J];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Operands {
    bf16x8 w[8];
    Split x[J];
  };
  // eight lanes to the 128 bytes of a row, its pieces of 16 bytes exchanged by the row's place as in block_place
  const int at = (lane & 15) * 128 + (((lane >> 4) * 2) ^ (lane & 7)) * 16;
  auto read_x = [&](const char* buf, f32x8 (&x)[J]) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const char* s = buf + WB + (wave * J + j) * 2048;
      x[j] = __builtin_shufflevector(*reinterpret_cast<const f32x4*>(s + at), *reinterpret_cast<const f32x4*>(s + (at ^ 16)), 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto read_w = [&](const char* buf, int i, Operands& o) { o.w[i] = *reinterpret_cast<const bf16x8*>(buf + i * 1024 + lane * 16); };
  int cur = 0;
  auto step = [&](int kt, const Operands& now, Operands& next) {
    // tile kt + 1 is here when at most the loads of R - 2 tiles are outstanding; behind the barrier everybody's are, and everybody holds
    // tile kt in registers, so that its buffer takes tile kt + R (past the end: the last one again, never read)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS * (R - 2)) : "memory");
    lds_barrier();
    stage(min(kt + R, n - 1), lds + cur * STAGE);
    cur = cur + 1 == R ? 0 : cur + 1;
    const char* buf = lds + cur * STAGE;
    f32x8 x[J];
    read_x(buf, x);
    __builtin_amdgcn_sched_barrier(0);
    // Four matrix instructions at a time: beside the first eight the weights are read, beside the last 16 J the next rows are taken apart, a pair of
    // columns (11 vector instructions) by four of them.  (One piece after the other: no instruction waits for the last.)
#pragma unroll
    for (int g = 0; g < 6 * J; ++g) {
      const int j = g / 6, piece = 2 - g % 6 / 2, half = g % 2 * 4, pair = g - 2 * J;
#pragma unroll
      for (int i = half; i < half + 4; ++i) acc[i][j] = mma(now.w[i], __builtin_bit_cast(bf16x8, now.x[j].b[piece]), acc[i][j]);
      if (g < 2)
#pragma unroll
        for (int i = half; i < half + 4; ++i) read_w(buf, i, next);
      if (pair >= 0) split_pair(x[pair / 4], pair % 4, next.x[pair / 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (g < 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (pair >= 0) __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  Operands p, q;
#pragma unroll
  for (int i = 0; i < R; ++i) stage(min(i, n - 1), lds + i * STAGE);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS * (R - 1)) : "memory");
  lds_barrier();
  {
    f32x8 x[J];
    read_x(lds, x);
#pragma unroll
    for (int i = 0; i < 8; ++i) read_w(lds, i, p);
#pragma unroll
    for (int i = 0; i < 4 * J; ++i) split_pair(x[i / 4], i % 4, p.x[i / 4]);
  }
  for (int kt = 0; kt < n; kt += 2) {  // (n is even)
    step(kt, p, q);
    step(kt + 1, q, p);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (own >= n_rows) return;
  // Three pieces stand for the activation while everything is finite: an infinity's rest is no number, and neither is a zero rest times an
  // infinite weight.  A wave with a sum that is not finite adds its tiles up again.
  float bad = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad = fmaf(acc[i][j][e], 0.f, bad);
  if (__any(bad != bad)) {
#pragma unroll 1
    for (int i = 0; i < 8; i += 2) direct_tile<EPI>(a, gather, row0, min(n_rows, own + 16 * J), f0, rt0 + i, own, k0, k1);
    return;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r = own + j * 16 + (lane & 15);
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int rt = rt0 + i;
      if (rt >= a.rt) continue;
      if constexpr (EPI == LIN_GLU) {
        if (!(i & 1)) store_glu<float>(a, row0 + r, (rt >> 1) * 16 + (lane >> 4) * 4, acc[i][j], acc[i | 1][j]);
      } else {
        store_plain<float, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[i][j]);
      }
    }
  }
}

// bf16, 256 features x up to 16 NJ rows: 4 waves of 64 features each, all of them on every row.  A weight tile is one wave's own, so weights go
// straight into its registers a step (two k tiles) ahead - 1 KiB of consecutive bytes a load -, and LDS holds the rows alone: 8 + NJ operand
// reads out of it feed 4 NJ matrix instructions where lin_body needs 16 for 16.  What bounds it is what compute units take out of L2 (the gate /
// up launch below about 2.5 GB: 10 TB/s over the card) and, with the last tiles of experts seldom full, work on rows that are not there: hence
// NJ = 8, 4 and 2.  64 experts of 1408 over 2048 rows, top 6, width 2048: gate / up 337 -> 254 us, down 201 -> 164 us (lin_body with a grid of
// row tiles x feature tiles before).
// For plain products, whose row tiles are full, it is within 3 % of lin_kernel either way, and lin_big_kernel has more work per byte.
template <int NJ>
__host__ DEV constexpr int wide_stage() { return 2 * NJ * 1024; }
template <int NJ, int EPI>
DEV void wide_body(const LinArgs& a, const int* gather, int row0, int n_rows, int f0, int k0, int k1, char* lds) {
  constexpr int STAGE = wide_stage<NJ>(), AL = NJ / 2;  // AL: this wave's loads of rows in a step
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = k1 - k0;
  const int rt0 = (f0 >> 4) + 4 * wave;
  const char *src_w[4], *src_a[AL];
#pragma unroll
  for (int i = 0; i < 4; ++i) src_w[i] = reinterpret_cast<const char*>(a.w) + ((size_t)min(rt0 + i, a.rt - 1) * a.kt + k0) * 1024;  // (past the end: never stored)
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int id = wave * AL + i;  // row group id / 2, k tile id % 2
    int r = min((id >> 1) * 16 + block_row(lane), n_rows - 1);
    r = gather ? gather[row0 + r] : row0 + r;
    src_a[i] = reinterpret_cast<const char*>(operand<bf16>(a, f0) + (size_t)r * a.lda + (size_t)(k0 + (id & 1)) * 32 + block_group(lane) * 8);
  }
  struct Weights {
    bf16x8 w[2][4];
  };
  auto load = [&](int kt, char* buf, Weights& o) {
#pragma unroll
    for (int i = 0; i < AL; ++i)
      __builtin_amdgcn_global_load_lds((gptr)(src_a[i] + (size_t)kt * 64), (lptr)(buf + (wave * AL + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i) o.w[kk][i] = *reinterpret_cast<const bf16x8*>(src_w[i] + (size_t)(kt + kk) * 1024 + lane * 16);
  };
  f32x4 acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int kt, const char* cur, char* other, const Weights& now, Weights& next) {
    // what was requested a step ago is here, the barrier makes it everybody's (the builtin: the compiler counts the weights' loads itself)
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    lds_barrier();
    load(min(kt + 2, n - 2), other, next);  // (past the end: the last step's again, not used)
    bf16x8 x[2][NJ];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < NJ; ++j) x[kk][j] = *reinterpret_cast<const bf16x8*>(cur + (2 * j + kk) * 1024 + block_place(lane) * 16);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][j] = mma(now.w[kk][i], x[kk][j], acc[i][j]);
    // requests first, then an operand is read four groups of matrix instructions ahead of its own
    __builtin_amdgcn_sched_group_barrier(0x020, 8 + AL, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < 2 * NJ; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      if (i < 2 * NJ - 4) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };
  Weights p, q;
  load(0, lds, p);
  for (int kt = 0; kt < n; kt += 4) {  // (n is even)
    step(kt, lds, lds + STAGE, p, q);
    if (kt + 2 < n) step(kt + 2, lds + STAGE, lds, q, p);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int r = j * 16 + (lane & 15);
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rt = rt0 + i;
      if (rt >= a.rt) continue;
      if constexpr (EPI == LIN_GLU) {
        if (!(i & 1)) store_glu<bf16>(a, row0 + r, (rt >> 1) * 16 + (lane >> 4) * 4, acc[i][j], acc[i | 1][j]);
      } else {
        store_plain<bf16, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[i][j]);
      }
    }
  }
}
// The same for few rows, which are bound by the weights' way out of HBM: a ring of four k tiles, the weights' in registers, the rows' in LDS (NJ KiB each),
// where wide_body has two steps of two.  64 experts of 1408, 60 prompt rows: gate / up 136 -> 125 us (5.9 TB/s), down 92.7 -> 89; 300 rows: down 101 -> 92, but gate / up
// of 33 to 64 rows are left to wide_body (151, 155 so).  Rings of six and eight are no faster; 128 rows by a ring of three 268 -> 271 us.
template <int NJ, int EPI>
DEV void thin_body(const LinArgs& a, const int* gather, int row0, int n_rows, int f0, char* lds) {
  constexpr int RING = 4, STAGE = NJ * 1024;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = a.kt;
  const int rt0 = (f0 >> 4) + 4 * wave, own = min(wave, NJ - 1);  // (with fewer row groups than waves some load the same one)
  const char* src_w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) src_w[i] = reinterpret_cast<const char*>(a.w) + (size_t)min(rt0 + i, a.rt - 1) * a.kt * 1024 + lane * 16;  // (past the end: never stored)
  int r = min(own * 16 + block_row(lane), n_rows - 1);
  r = gather ? gather[row0 + r] : row0 + r;
  const char* src_a = reinterpret_cast<const char*>(operand<bf16>(a, f0) + (size_t)r * a.lda + block_group(lane) * 8);
  bf16x8 w[RING][4];
  auto load = [&](int kt, int slot) {
    __builtin_amdgcn_global_load_lds((gptr)(src_a + (size_t)kt * 64), (lptr)(lds + slot * STAGE + own * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[slot][i] = *reinterpret_cast<const bf16x8*>(src_w[i] + (size_t)kt * 1024);
  };
  f32x4 acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto use = [&](int slot) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(lds + slot * STAGE + j * 1024 + block_place(lane) * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][j] = mma(w[slot][i], x, acc[i][j]);
    }
  };
  // Loads are counted: every one of a k tile's five is used, so that none can go, and groups do not mix.
  auto step = [&](int kt, int slot) {
    // this k tile is here when at most the loads of the RING - 2 behind it are outstanding; the barrier makes it everybody's, and everybody has read
    // the one before it, whose place the one RING - 1 tiles on takes
    __builtin_amdgcn_s_waitcnt(0x0f70 | (RING - 2) * 5);  // vmcnt (the builtin: the compiler counts the weights' loads itself)
    lds_barrier();
    load(kt + RING - 1, (slot + RING - 1) % RING);
    use(slot);
  };
#pragma unroll
  for (int i = 0; i < RING - 1; ++i) {
    load(min(i, n - 1), i);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  }
  static_assert(RING == 4, "what is left below");
  int kt = 0;
  for (; kt + 2 * RING - 2 < n; kt += RING)
#pragma unroll
    for (int i = 0; i < RING; ++i) step(kt + i, i);
  const int left = n - kt;  // 4 or 6, or n = 2; steps while there is a k tile to request, and then all that is on its way at once
  if (left > 2) step(kt, 0);
  if (left > 4) {
    step(kt + 1, 1);
    step(kt + 2, 2);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  lds_barrier();
  if (left == 6) {
    use(3);
    use(0);
    use(1);
  } else if (left == 4) {
    use(1);
    use(2);
    use(3);
  } else {
    use(0);
    use(1);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int r = j * 16 + (lane & 15);
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rt = rt0 + i;
      if (rt >= a.rt) continue;
      if constexpr (EPI == LIN_GLU) {
        if (!(i & 1)) store_glu<bf16>(a, row0 + r, (rt >> 1) * 16 + (lane >> 4) * 4, acc[i][j], acc[i | 1][j]);
      } else {
        store_plain<bf16, EPI>(a, row0 + r, rt * 16 + (lane >> 4) * 4, acc[i][j]);
      }
    }
  }
}
template <bool LONE, int EPI>
__global__ __launch_bounds__(256, 2) void lin_kernel(LinArgs a, const int row_tiles, const int tiles) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int b = xcd_range(blockIdx.x, tiles), row0 = b % row_tiles * 128, per = part_tiles(a), k0 = blockIdx.y * per;
  a.out_f += blockIdx.y * a.part_stride;
  if constexpr (LONE) lone_body<EPI>(a, row0, min(128, a.rows - row0), b / row_tiles * 128, k0, min(a.kt, k0 + per), lds);
  else lin_body<EPI>(a, row0, min(128, a.rows - row0), b / row_tiles * 128, k0, min(a.kt, k0 + per), lds);
}
template <int J, int EPI>
__global__ __launch_bounds__(256, 4 - J) void rows_kernel(LinArgs a, const int row_tiles, const int tiles) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int b = xcd_range(blockIdx.x, tiles), row0 = b % row_tiles * 64 * J, per = part_tiles(a), k0 = blockIdx.y * per;
  a.out_f += blockIdx.y * a.part_stride;
  rows_body<J, EPI>(a, nullptr, row0, min(64 * J, a.rows - row0), b / row_tiles * 128, k0, min(a.kt, k0 + per), lds);
}

// LinArgs.direct: products of a few k tiles (the decay of time mixing: two), 64 features x 64 rows per workgroup.  Three pieces have nothing to save
// there, latency and the output bound it: 2048 features of 1996 rows 12.4 us, of 301 rows 8.0 (in three pieces by tiles of 128 x 128 21.6 and 9.6, by
// its tiles with this instruction 24.8 and 11.6; waves of 64 x 64 with the whole k in one straight line 24.5 and 21.7).  And a sum is one chain, as in
// few_body: in bfloat16 runs another rounding of the decay turns roundings behind it.
__global__ __launch_bounds__(256) void lin_direct_kernel(const LinArgs a, const int row_tiles, const int tiles) {
  const int b = xcd_range(blockIdx.x, tiles), row0 = b % row_tiles * 64, f0 = b / row_tiles * 64, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  direct_tile<LIN_STORE>(a, nullptr, row0, min(64, a.rows - row0), f0, (f0 >> 4) + (wave & 1) * 2, (wave >> 1) * 32, 0, a.kt);
}

// 256 features x 256 rows per workgroup: 8 waves of 128 x 64; twice the matrix work per byte staged.  A ring of RING stages of one k tile
// (32 KiB): while a tile is multiplied the next one's operands are read into the other set of registers, and RING - 1 more are on their way.
//
// streams = 0: a workgroup per tile (and part of k).  Else the tiles of a row of them, k step by k step behind each other, are dealt out evenly to that
// many workgroups, each of which works off one stretch without a stop between tiles: a product whose tiles do not fill the last round of compute units loses
// none of them.  A tile that a stretch's end cuts (never in more than two pieces: streams <= feature tiles) is still added up in one order, as everywhere
// else: a workgroup takes the tiles of its stretch from the last one down, so that the front of the tile at its end, whose sums it leaves for the next
// stretch, is its first work, and going on from the sums of the tile at its start its last.  Should those not be there after `looks` looks, it works off
// the front itself.  The row tiles of one stretch are neighbours on one XCD and run in step, so that weights and rows meet in its L2.
enum { RING = 4 };
struct LinStream {
  int streams;
  float* sums;        // [streams][row tiles][256 x 256]: of the front of the tile that the stretch's start cuts
  unsigned* pieces;   // [streams][row tiles]: CUT_STORED and CUT_TAKEN as they come, zero between launches; behind them (LIN_SLOTS) `looks`
};
enum { CUT_STORED = 1, CUT_TAKEN = 2 };
template <int EPI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void lin_big_kernel(LinArgs a, const int row_tiles, const int tiles, const LinStream ls) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ unsigned s_there;
  constexpr int STAGE = 32 * 1024;
  const int b = xcd_range(blockIdx.x, ls.streams ? ls.streams * row_tiles : tiles), row_tile = b % row_tiles, row0 = row_tile * 256, stream = b / row_tiles;
  // this workgroup's k tiles, counted through the feature tiles
  int first, last;
  if (ls.streams) {
    const long long pairs = (long long)(tiles / row_tiles) * (a.kt >> 1);
    first = (int)(pairs * stream / ls.streams) * 2;
    last = (int)(pairs * (stream + 1) / ls.streams) * 2;
  } else {
    const int per = part_tiles(a);
    first = stream * a.kt + blockIdx.y * per;
    last = min(first + per, (stream + 1) * a.kt);
    a.out_f += blockIdx.y * a.part_stride;
  }
  const int f_first = first / a.kt, f_last = (last - 1) / a.kt;
  const int k_first = first - f_first * a.kt, k_last = last - f_last * a.kt;  // of the first tile from, of the last one up to
  const int n_rows = min(256, a.rows - row0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  int at_a[2];  // this wave's share of a stage: weight tiles and row groups 2 * wave + {0, 1}
#pragma unroll
  for (int i = 0; i < 2; ++i) at_a[i] = (row0 + min((2 * wave + i) * 16 + block_row(lane), n_rows - 1)) * a.lda + block_group(lane) * 8;
  int f_in = f_last, k_in = f_last == f_first ? k_first : 0, to_in = k_last;  // what is requested next
  auto stage = [&](char* buf) {  // (past the end: the last tile again, never read)
    const bf16* x = operand<bf16>(a, f_in * 256) + (size_t)k_in * 32;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int slot = 2 * wave + i;
      const uint16_t* w = a.w + ((size_t)min(f_in * 16 + slot, a.rt - 1) * a.kt + k_in) * 512;
      __builtin_amdgcn_global_load_lds((gptr)(w + lane * 8), (lptr)(buf + slot * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gptr)(x + at_a[i]), (lptr)(buf + 16 * 1024 + slot * 1024), 16, 0, 0);
    }
    const bool end = k_in + 1 == to_in, down = end && f_in > f_first;
    f_in -= down;
    k_in = down ? (f_in == f_first ? k_first : 0) : k_in + !end;
    to_in = down ? a.kt : to_in;
  };
  f32x4 acc[8][4];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  struct Operands {
    bf16x8 w[8], x[4];
  };
  auto read = [&](const char* buf, Operands& o) {
#pragma unroll
    for (int j = 0; j < 4; ++j) o.x[j] = *reinterpret_cast<const bf16x8*>(buf + 16 * 1024 + (wn * 4 + j) * 1024 + block_place(lane) * 16);
#pragma unroll
    for (int i = 0; i < 8; ++i) o.w[i] = *reinterpret_cast<const bf16x8*>(buf + (wm * 8 + i) * 1024 + lane * 16);
  };
  int cur = 0;
  auto step = [&](const Operands& now, Operands& next) {
    // the next k tile is here when at most the loads of RING - 2 tiles are outstanding; behind the barrier everybody's are, and everybody holds
    // this one in registers, so that its buffer takes the one RING tiles on
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (RING - 2)) : "memory");
    lds_barrier();
    stage(lds + cur * STAGE);
    cur = cur + 1 == RING ? 0 : cur + 1;
    read(lds + cur * STAGE, next);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mma(now.w[i], now.x[j], acc[i][j]);
#pragma unroll
    for (int i = 0; i < 12; ++i) {  // one LDS read, then matrix work that does not wait for it
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
  };
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  // the front of the tile at the stretch's end: its sums for the next stretch
  auto leave = [&]() {
    const int at = (stream + 1) * row_tiles + row_tile;
    const auto r = __builtin_amdgcn_make_buffer_rsrc(ls.sums + (size_t)at * 65536, 0, 65536 * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), r, tid * 16, (i * 4 + j) * 8192, 16 /* sc1 */);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0 && __hip_atomic_fetch_add(ls.pieces + at, (unsigned)CUT_STORED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      __hip_atomic_store(ls.pieces + at, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // (not waited for)
  };
  // the sums of the tile that the stretch's start cuts: true if they are there
  auto take = [&]() {
    const int at = stream * row_tiles + row_tile;
    __syncthreads();
    if (tid == 0) {
      unsigned* word = ls.pieces + at;
      const int looks = (int)ls.pieces[LIN_SLOTS];
      for (int i = 0; i < looks && !__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); ++i) __builtin_amdgcn_s_sleep(8);
      const unsigned there = __hip_atomic_fetch_add(word, (unsigned)CUT_TAKEN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (there) __hip_atomic_store(word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_there = looks < 0 ? 0 : there;
    }
    __syncthreads();
    if (!s_there) return false;
    const auto r = __builtin_amdgcn_make_buffer_rsrc(ls.sums + (size_t)at * 65536, 0, 65536 * 4, 0x00020000);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, tid * 16, (i * 4 + j) * 8192, 16));
    return true;
  };
  Operands p, q;
  bool empty = true;  // the ring
  for (int f = f_last; f >= f_first; --f) {
    int at = f == f_first ? k_first : 0;
    const int end = f == f_last ? k_last : a.kt;
    clear();
    if (ls.streams && at > 0) {
      empty = !take();
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): a step counts loads into LDS alone (the builtin: the compiler knows that the sums are here)
      if (empty) {
        lds_barrier();
        at = k_in = cur = 0;
        to_in = end;
      }
    }
    if (empty) {
#pragma unroll
      for (int i = 0; i < RING; ++i) stage(lds + i * STAGE);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (RING - 1)) : "memory");
      lds_barrier();
      read(lds, p);
      empty = false;
    }
    for (; at < end; at += 2) {  // (stretches and parts are even)
      step(p, q);
      step(q, p);
    }
    if (ls.streams && end < a.kt) {
      leave();
      continue;
    }
    const int rt0 = f * 16 + wm * 8;
    const bool pairs = wide_pairs(a) && (rt0 + 8) * 16 <= a.n_wide && rt0 + 8 <= a.rt;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = wn * 64 + j * 16 + (lane & 15);
      if (pairs) {
#pragma unroll
        for (int i = 0; i < 8; i += 2) store_wide_pair<EPI == LIN_TANH_F ? LIN_STORE : EPI>(a, r < n_rows, row0 + r, rt0 + i, acc[i][j], acc[i + 1][j]);
      } else if (r < n_rows) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (rt0 + i < a.rt) store_plain<bf16, EPI>(a, row0 + r, (rt0 + i) * 16 + (lane >> 4) * 4, acc[i][j]);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (a step counts loads alone)
  }
}

static LinArgs expert_lin(const MoeArgs& m, bool down) {  // the parts of an expert product that do not depend on the expert
  LinArgs a{};
  a.a_t = down ? m.hidden_t : m.h_t;
  a.lda = down ? m.hidden_ld : m.width_ld;
  a.epi = down ? LIN_STORE : LIN_GLU;
  a.out_t = down ? m.y_t : m.hidden_t;
  a.ld_t = down ? m.y_ld : m.hidden_ld;
  a.n_wide = 0x7fffffff;
  a.p1 = m.alpha;
  a.p2 = m.offset;
  return a;
}
DEV void set_expert(LinArgs& a, const MoeArgs& m, const ExpertMat& e, int expert) {
  const bool sh = expert == m.experts;
  a.w = sh ? e.shared : e.w + (size_t)expert * e.stride;
  a.kt = sh ? e.shared_kt : e.kt;
  a.rt = sh ? e.shared_rt : e.rt;
  a.p0 = sh ? m.shared_limit : m.limit;
}
// grid.x: an upper bound of the tiles.  The routed experts' come first, in groups of four row tiles (mostly one expert's, they are sorted) and in a
// group feature tile by feature tile, and an XCD takes a contiguous range: the workgroups that read one weight tile meet in one L2, and
// the rows of a group stay in it.  The shared expert's tiles, the longest, start first.
template <typename T, bool down>
__global__ __launch_bounds__(256, 2) void expert_kernel(LinArgs a, const MoeArgs m, const int shared_tiles) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int FT = sizeof(T) == 2 ? 16 : 8, EPI = down ? LIN_STORE : LIN_GLU;
  const ExpertMat& e = down ? m.down : m.up;
  const int row_tiles = *m.n_tiles - shared_tiles, ft = (e.rt + FT - 1) / FT, sft = (e.shared_rt + FT - 1) / FT;
  int b = blockIdx.x, tile, f;
  const int first = (shared_tiles * sft + 7) & ~7;
  if (b < first) {
    if (b >= shared_tiles * sft) return;
    b = xcd_range(b, shared_tiles * sft);
    f = b / shared_tiles;
    tile = row_tiles + b % shared_tiles;
  } else {
    b -= first;
    if (b >= row_tiles * ft) return;
    b = xcd_range(b, row_tiles * ft);
    const int group = b / (4 * ft), n = min(4, row_tiles - 4 * group);
    b -= group * 4 * ft;
    f = b / n;
    tile = 4 * group + b % n;
  }
  set_expert(a, m, e, m.tiles[4 * tile]);
  const int* gather = down ? nullptr : m.slot_row;
  const int row0 = m.tiles[4 * tile + 1], rows = m.tiles[4 * tile + 2];
  if constexpr (sizeof(T) == 2) {
    if (rows > 64) wide_body<8, EPI>(a, gather, row0, rows, f * 256, 0, a.kt, lds);
    else if (rows > 32 && down) thin_body<4, EPI>(a, gather, row0, rows, f * 256, lds);
    else if (rows > 32) wide_body<4, EPI>(a, gather, row0, rows, f * 256, 0, a.kt, lds);
    else thin_body<2, EPI>(a, gather, row0, rows, f * 256, lds);
  } else {
    if (rows > 64) rows_body<2, EPI>(a, gather, row0, rows, f * 128, 0, a.kt, lds);
    else rows_body<1, EPI>(a, gather, row0, rows, f * 128, 0, a.kt, lds);
  }
}

// ---- up to 16 rows -------------------------------------------------------------------------------
// One workgroup = NR feature tiles of 16 (GLU: NR / 2 gate / up pairs): wave w takes k tiles w, w + 4, ...; partial sums meet in LDS.
// a_row: A row of this lane's column; out_row: out row or -1.
template <typename T, int NR, bool GLU>
DEV void few_body(const LinArgs& a, int rt0, int k_first, int k_end, int a_row, int out_row, float* lds) {
  typedef typename Frag<T>::type frag;
  constexpr int U = NR == 1 && sizeof(T) == 2 ? 8 : 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bf16x8* w0 = reinterpret_cast<const bf16x8*>(a.w) + lane;
  size_t tile[NR];  // (a group's tiles past the last are its last, and not stored)
#pragma unroll
  for (int i = 0; i < NR; ++i) tile[i] = (size_t)min(rt0 + i, a.rt - 1) * a.kt;
  const T* x0 = operand<T>(a, rt0 * 16) + (size_t)a_row * a.lda + (lane >> 4) * 8;
  f32x4 acc[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 w[U][NR];
  frag x[U];
  auto load = [&](int u, int k) {
#pragma unroll
    for (int i = 0; i < NR; ++i) w[u][i] = w0[(tile[i] + k) * 64];
    x[u] = *reinterpret_cast<const frag*>(x0 + (size_t)k * 32);
  };
  int k0 = k_first + wave;
  if (k0 + 4 * (U - 1) < k_end) {  // a whole round of U k tiles
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, k0 + 4 * u);
    __builtin_amdgcn_sched_barrier(0);  // (all on their way first)
    // While another whole round follows, a tile is requested as soon as its registers are free: the stream does not stop between rounds.  (No
    // condition inside: a load is moved behind it, and then waited for alone.)  All of a step's products against rounds that wait: 27 lite layers, one
    // row 1772 -> 1743 us, four in 32 bits 2241 -> 2106; three wide ones, four rows 1184 -> 1170, 16 rows 5795 -> 5773.
    for (; k0 + 4 * (2 * U - 1) < k_end; k0 += 4 * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int i = 0; i < NR; ++i) acc[i] = mma(w[u][i], x[u], acc[i]);
        load(u, k0 + 4 * (U + u));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < NR; ++i) acc[i] = mma(w[u][i], x[u], acc[i]);
    k0 += 4 * U;
  }
  if (k0 < k_end) {  // the last, short one: zeros behind the end
#pragma unroll
    for (int u = 0; u < U - 1; ++u) load(u, min(k0 + 4 * u, k_end - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U - 1; ++u) {
      const bool in = k0 + 4 * u < k_end;
      const frag xu = in ? x[u] : frag{};
#pragma unroll
      for (int i = 0; i < NR; ++i) acc[i] = mma(in ? w[u][i] : bf16x8{}, xu, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) *reinterpret_cast<f32x4*>(lds + ((wave * NR + i) * 64 + lane) * 4) = acc[i];
  __syncthreads();
  constexpr int PER = GLU ? 2 : 1;  // wave v adds up the v-th tile or pair
  if (wave >= NR / PER || rt0 + wave * PER >= a.rt) return;
  f32x4 sum[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    sum[i] = *reinterpret_cast<const f32x4*>(lds + ((wave * PER + i) * 64 + lane) * 4);
#pragma unroll
    for (int v = 1; v < 4; ++v) sum[i] += *reinterpret_cast<const f32x4*>(lds + ((v * NR + wave * PER + i) * 64 + lane) * 4);
  }
  if (out_row < 0) return;
  if constexpr (GLU) store_glu<T>(a, out_row, ((rt0 >> 1) + wave) * 16 + (lane >> 4) * 4, sum[0], sum[1]);
  else store_plain<T>(a, out_row, (rt0 + wave) * 16 + (lane >> 4) * 4, sum[0]);
}

struct FewArgs {
  LinArgs t[4];
  int wg_end[4];   // workgroups of products 0 .. i
  int groups[4];   // ... of one part of product i
  int n;
  int expert_wgs;  // in front of them: expert blocks
  int tiles_per_expert;
  int down;
  LinArgs e;
  MoeArgs m;
};
// A load of the operand is `rows` segments of 64 bytes in as many lines, at 16 rows twice the lines of a weight tile's load: where enough
// workgroups are left (launch_few) one takes NT tiles (of gate and up: two pairs) per load of the operand.
template <typename T, int NT>
__global__ __launch_bounds__(256) void few_kernel(const FewArgs f) {
  constexpr int GT = NT > 1 ? 4 : 2;  // tiles of a gate / up group
  __shared__ __attribute__((aligned(16))) float lds[4 * (NT > GT ? NT : GT) * 64 * 4];
  const int c = threadIdx.x & 15;
  int b = blockIdx.x;
  if (b < f.expert_wgs) {
    const int i = b / f.tiles_per_expert, tile = b % f.tiles_per_expert;
    if (i >= *f.m.n_active) return;
    const int expert = f.m.active[i];
    LinArgs a = f.e;
    set_expert(a, f.m, f.down ? f.m.down : f.m.up, expert);
    const int nr = f.down ? NT : GT;
    if (tile * nr >= a.rt) return;
    // a lane whose row did not choose the expert reads the first row that did: a load of the operand then touches as many lines as the expert has
    // rows, not 16.  (A scalar read of that lane: a lane exchange in a branch reads nothing of lanes that are not in it.)
    const int slot = c < f.m.rows ? f.m.active_slot[i * 16 + c] : -1;
    const int own = min(c, f.m.rows - 1) * (f.m.top + f.m.shared) + max(slot, 0);
    const int one = max(__ffsll(__ballot(slot >= 0)) - 1, 0), first = __builtin_amdgcn_readlane(own, one);
    const int row = slot >= 0 ? c : one, pos = slot >= 0 ? own : first;
    const int out = slot >= 0 ? own : -1;
    if (f.down) few_body<T, NT, false>(a, tile * NT, 0, a.kt, pos, out, lds);
    else few_body<T, GT, true>(a, tile * GT, 0, a.kt, row, out, lds);
    return;
  }
  b -= f.expert_wgs;
  int i = 0;
  while (i + 1 < f.n && b >= f.wg_end[i]) ++i;
  LinArgs a = f.t[i];
  if (i > 0) b -= f.wg_end[i - 1];
  const int row = min(c, a.rows - 1), part = b / f.groups[i], per = part_tiles(a);
  if (a.out_at) a.out_f = glob(*glob(a.out_at));
  a.out_f += part * a.part_stride;
  few_body<T, NT, false>(a, b % f.groups[i] * NT, part * per, min(a.kt, part * per + per), a.row_seq ? a.seqs[a.row_seq[row]].row0 : row, c < a.rows ? c : -1, lds);
}

// ---- launches ------------------------------------------------------------------------------------
static int check_lin(const LinArgs& a, const char* what) {
  if (!a.w || !a.a_t || a.rows < 1 || a.kt < 2 || (a.kt & 1) || a.rt < 1 || a.lda < a.kt * 32) DSK_FAIL(DSK_ERR_INVALID, "%s: rows %d kt %d rt %d lda %d", what, a.rows, a.kt, a.rt, a.lda);
  if (a.parts > 1 && (a.n_wide || a.epi != LIN_STORE || part_tiles(a) * (a.parts - 1) >= a.kt)) DSK_FAIL(DSK_ERR_INVALID, "%s: %d parts of %d", what, a.parts, a.kt);
  if (a.out_at && a.parts > 1) DSK_FAIL(DSK_ERR_INVALID, "%s: %d parts of an output that moves", what, a.parts);
  if (a.a_seg < 0 || (a.a_seg & 15) || (a.a_seg && a.a_ops < 1)) DSK_FAIL(DSK_ERR_INVALID, "%s: %d features per operand", what, a.a_seg);
  return DSK_OK;
}
template <typename K>
static int allow_lds(K k, int bytes) {
  HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  return DSK_OK;
}
// Microseconds a prompt product takes on 256 compute units, by measurement of 20 shapes of 100 - 2000 rows and k of 2048 - 27648 (within a tenth of most): a
// step of 64 columns takes a workgroup of 128 x 128 alone on its compute unit 0.4 us (0.6 with weights out of HBM), two of them 1.0 - 1.08; one of 256 x 256
// takes 1.17 us, and 1.55 when all of them run (the card's clock).  Both start and end in 3 and 8 us; a part more writes and reads its sums.
// Stretches (LinStream) leave no compute unit empty, but their rows and weights meet in L2 less often (1.72 us), and tiles that they cut are stored and read:
// 2000 rows and 2048 x 16896 132 us, by 128 x 128 163, by 256 x 256 163; 7168 x 32896 762, 1066, 868; 1500 rows and 7168 x 27648 518, 658, 526.
// In 32 bits a step of 64 columns takes a workgroup of 128 rows alone 1.08 us (1.5 with weights out of HBM), two of them 2.45, and one of 64 rows 0.64, three of them 1.96 (us by 128 and
// by 64 rows: 301 rows and 2048 x 16896 78 and 62, 2000 rows 347 and 365; 301 rows and 2048 x 2176 40 and 25).
enum { LIN_SMALL, LIN_HALF, LIN_BIG, LIN_STREAM };  // (the second: 64 rows instead of 128, 32 bits)
static int lin_streams(int rows, int rt) {  // stretches of a row of 256 x 256 tiles; 0: they would cut a tile more than once
  const int n = LIN_SLOTS / cdiv(rows, 256);  // (a workgroup for each compute unit)
  return n >= 2 && n <= cdiv(rt, 16) ? n : 0;
}
static double lin_cost(int rows, int rt, int kt, int parts, int kind, bool f32) {
  const double k = part_tiles(kt, parts) / 2, sums = (parts - 1) * 3.2e-5 * rows * rt;
  if (f32 ? kind > LIN_HALF : kind == LIN_HALF) return 1e9;
  if (kind == LIN_STREAM) {
    const int n = lin_streams(rows, rt);
    return n && parts == 1 ? 32 + 1.72 * k * cdiv(rt, 16) / n : 1e9;
  }
  if (f32) {  // rounds of as many workgroups as compute units have room for, and what the last one leaves empty
    const bool half = kind == LIN_HALF;
    const int n = cdiv(rows, half ? 64 : 128) * cdiv(rt, 8) * parts, at_once = half ? 768 : 512;
    const double r = n % at_once / 256.;
    const double rest = r == 0 ? 0 : half ? (r <= 1 ? 0.64 : (r <= 2 ? 0.72 : 1.) + 0.32 * r) : r <= 1 ? 1.3 : 1.75 + 0.35 * r;
    return 3 + (n / at_once * (half ? 1.96 : 2.45) + rest) * k + sums;
  }
  if (kind == LIN_BIG) {
    const int n = cdiv(rows, 256) * cdiv(rt, 16) * parts, rest = n % 256;
    return n / 256 * (8 + 1.55 * k) + (rest ? 8 + (1.17 + 0.38 / 256 * rest) * k : 0) + sums;
  }
  const int n = cdiv(rows, 128) * cdiv(rt, 8) * parts, rest = n % 512;
  return 3 + (n / 512 * 1.08 + (rest == 0 ? 0 : n <= 256 ? 0.6 : rest <= 256 ? 0.85 : 1.0)) * k + sums;
}
static int lin_kind(int rows, int rt, int kt, int parts, bool f32) {
  int best = LIN_SMALL;
  for (int kind : {LIN_HALF, LIN_BIG, LIN_STREAM})
    if (lin_cost(rows, rt, kt, parts, kind, f32) < lin_cost(rows, rt, kt, parts, best, f32)) best = kind;
  return best;
}
static int lin_kind(const LinArgs& a, int parts, bool f32, const LinSpace& space) {
  if (!f32 && (a.a_seg & 255)) return LIN_SMALL;
  int kind = lin_kind(a.rows, a.rt, a.kt, parts, f32);
  if (f32) return kind;
  if (a.tile) kind = a.tile == 128 ? LIN_SMALL : parts == 1 && lin_streams(a.rows, a.rt) ? LIN_STREAM : LIN_BIG;
  return kind == LIN_STREAM && space.slots < LIN_SLOTS ? LIN_BIG : kind;
}
template <typename C>
static int cheapest_parts(int kt, int most, C cost) {
  int best = 1;
  double least = 0;
  for (int n = 1; n <= most && (n == 1 || kt / n >= 16); ++n) {
    const double c = cost(n);
    if (n == 1 || c < least) {
      least = c;
      best = n;
    }
  }
  return cdiv(kt, part_tiles(kt, best));  // (no part may be empty)
}
int lin_parts(int rows, int rt, int kt, bool f32, int most) {
  return cheapest_parts(kt, most, [&](int n) { return lin_cost(rows, rt, kt, n, lin_kind(rows, rt, kt, n, f32), f32); });
}
// Where a router reads what comes of a product the number of parts is no matter of tuning: it decides the order in which a sum is added up, with that the
// roundings behind it, and a router decides close calls by those.  A step of 27 such layers behind a prompt of 300 tokens came out 0.13 apart, relative,
// from a change of a sum's last bit in one row.  So these costs stay as they are, whatever the kernels take (tiles and stretches alike add a part up in the order of k):
// the mixers' products of a width of 2048 take 15.0 us for 700 rows (lin_cost's parts: 13.2), 17.7 for 1200 (18.3), 22.4 for 2048 (20.9).
int lin_parts_fixed(int rows, int rt, int kt, bool f32, int most) {
  return cheapest_parts(kt, most, [&](int parts) {
    const double k = part_tiles(kt, parts) / 2, sums = (parts - 1) * 3.2e-5 * rows * rt;
    const int n = cdiv(rows, 128) * cdiv(rt, 8) * parts;
    const double small = (n <= 256 ? (f32 ? 1.75 : 1.05) * k : cdiv(n, 512) * (f32 ? 3.2 : 1.3) * k) + 5 + sums;
    return f32 ? small : std::min(small, cdiv(cdiv(rows, 256) * cdiv(rt, 16) * parts, 256) * (15 + 1.84 * k) + sums);
  });
}
bool lin_streams_some(int rows, int rt, int kt, int tile) {
  bool some = false;
  for (int r = rows; r > 0; r -= 256)  // (row tiles decide)
    some = some || (tile ? tile == 256 && lin_streams(r, rt) : lin_kind(r, rt, kt, 1, false) == LIN_STREAM);
  return some;
}
int lin_parts_few(int rt, int kt, int most) {
  const int n = std::max(std::min({1024 / rt, kt / 16, most}), 1);
  return cdiv(kt, part_tiles(kt, n));
}
#define LIN_EPI(K, T) (a.epi == LIN_STORE ? K<T LIN_STORE> : a.epi == LIN_XIELU ? K<T LIN_XIELU> : a.epi == LIN_TANH_F ? K<T LIN_TANH_F> : K<T - 1>)
int launch_lin(hipStream_t st, const LinArgs& a, bool f32, const LinSpace& space) {
  DSK_TRY(check_lin(a, "lin"));
  if ((a.a_seg & 127) || a.row_seq || a.out_at) DSK_FAIL(DSK_ERR_INVALID, "lin: %d features per operand", a.a_seg);
  const int kind = lin_kind(a, std::max(a.parts, 1), f32, space);
  if (kind > LIN_HALF) {
    const int row_tiles = cdiv(a.rows, 256), tiles = row_tiles * cdiv(a.rt, 16);
    const LinStream ls{kind == LIN_STREAM ? lin_streams(a.rows, a.rt) : 0, space.sums, space.pieces};
    auto k = LIN_EPI(lin_big_kernel, );
    DSK_TRY(allow_lds(k, RING * 32 * 1024));
    hipLaunchKernelGGL(k, dim3(ls.streams ? ls.streams * row_tiles : tiles, std::max(a.parts, 1)), dim3(512), RING * 32 * 1024, st, a, row_tiles, tiles, ls);
    return DSK_OK;
  }
  if (a.direct) {
    if (!f32 || a.parts > 1 || a.epi != LIN_STORE) DSK_FAIL(DSK_ERR_INVALID, "lin: direct products are 32-bit ones in one part, stored as they are");
    const int row_tiles = cdiv(a.rows, 64), tiles = row_tiles * cdiv(a.rt, 4);
    hipLaunchKernelGGL(lin_direct_kernel, dim3(tiles), dim3(256), 0, st, a, row_tiles, tiles);
    return DSK_OK;
  }
  const int high = kind == LIN_HALF ? 64 : 128, row_tiles = cdiv(a.rows, high), tiles = row_tiles * cdiv(a.rt, 8);
  const int lds = !f32 ? (int)LIN_LDS : ROWS_RING * (kind == LIN_HALF ? rows_stage<1>() : rows_stage<2>());
  const dim3 grid(tiles, std::max(a.parts, 1));
#define LIN_J1 1,
#define LIN_J2 2,
#define LIN_LONE true,
#define LIN_SHARED false,
  const bool lone = tiles * std::max(a.parts, 1) <= LIN_SLOTS;  // (lin_cost: compute units)
  auto k = !f32 ? (lone ? LIN_EPI(lin_kernel, LIN_LONE) : LIN_EPI(lin_kernel, LIN_SHARED)) : kind == LIN_HALF ? LIN_EPI(rows_kernel, LIN_J1) : LIN_EPI(rows_kernel, LIN_J2);
  DSK_TRY(allow_lds(k, lds));
  hipLaunchKernelGGL(k, grid, dim3(256), lds, st, a, row_tiles, tiles);
  return DSK_OK;
}
int launch_experts(hipStream_t st, const MoeArgs& m, bool down, bool f32) {
  const LinArgs a = expert_lin(m, down);
  const ExpertMat& e = down ? m.down : m.up;
  const int shared_tiles = m.shared ? cdiv(m.rows, MOE_TILE) : 0, ft = f32 ? 8 : 16;
  const dim3 grid((m.max_tiles - shared_tiles) * cdiv(e.rt, ft) + ((shared_tiles * cdiv(e.shared_rt, ft) + 7) & ~7));
  const int lds = f32 ? ROWS_RING * rows_stage<2>() : 2 * wide_stage<8>();
  auto k = f32 ? (down ? expert_kernel<float, true> : expert_kernel<float, false>) : (down ? expert_kernel<bf16, true> : expert_kernel<bf16, false>);
  DSK_TRY(allow_lds(k, lds));
  hipLaunchKernelGGL(k, grid, dim3(256), lds, st, a, m, shared_tiles);
  return DSK_OK;
}
// Four tiles per workgroup from 9 rows and 1536 tiles on, in bf16: a step of 16 sequences, us with one tile -> four, 8080 tiles 450 -> 320, 2328
// tiles 136 -> 106, 1572 94 -> 71, the experts' down 8832 88 -> 66; below, the card is left empty: 1056 tiles 16.4 -> 21, 582 13 -> 15.5.  Up to
// 8 rows the operand is the smaller part (6400 tiles of 8 rows 84 -> 82), and in 32 bits 5 rows of 896 tiles were slower (105 -> 133).
constexpr int FEW_TILES = 4;
static int launch_few(hipStream_t st, FewArgs& f, const LinArgs* a, int n, int experts, int expert_tiles, int rows, bool f32) {
  int tiles = experts * expert_tiles;
  bool whole = true;  // (a workgroup's tiles read one operand)
  for (int i = 0; i < n; ++i) {
    rows = std::max(rows, a[i].rows);
    tiles += a[i].rt * std::max(a[i].parts, 1);
    whole = whole && a[i].a_seg % (16 * FEW_TILES) == 0;
  }
  const int nt = !f32 && rows > 8 && tiles >= 1536 && whole ? FEW_TILES : 1;
  if (n > 4) DSK_FAIL(DSK_ERR_INVALID, "lin_few: %d products", n);
  f.n = n;
  int wgs = 0;
  for (int i = 0; i < n; ++i) {
    DSK_TRY(check_lin(a[i], "lin_few"));
    if (a[i].rows > 16) DSK_FAIL(DSK_ERR_INVALID, "lin_few: %d rows", a[i].rows);
    f.t[i] = a[i];
    f.groups[i] = cdiv(a[i].rt, nt);
    f.wg_end[i] = wgs += f.groups[i] * std::max(a[i].parts, 1);
  }
  f.tiles_per_expert = cdiv(expert_tiles, f.down ? nt : nt > 1 ? 4 : 2);
  f.expert_wgs = experts * f.tiles_per_expert;
  auto k = f32 ? few_kernel<float, 1> : nt > 1 ? few_kernel<bf16, FEW_TILES> : few_kernel<bf16, 1>;
  hipLaunchKernelGGL(k, dim3(f.expert_wgs + wgs), dim3(256), 0, st, f);
  return DSK_OK;
}
int launch_lin_few(hipStream_t st, const LinArgs* a, int n, bool f32) {
  FewArgs f{};
  return launch_few(st, f, a, n, 0, 0, 0, f32);
}
int launch_experts_few(hipStream_t st, const MoeArgs& m, bool down, const LinArgs* also, int n_also, bool f32) {
  if (m.rows > 16) DSK_FAIL(DSK_ERR_INVALID, "experts_few: %d rows", m.rows);
  FewArgs f{};
  f.m = m;
  f.down = down;
  f.e = expert_lin(m, down);
  const ExpertMat& e = down ? m.down : m.up;
  const int rt = m.shared ? (e.rt > e.shared_rt ? e.rt : e.shared_rt) : e.rt;
  return launch_few(st, f, also, n_also, m.max_active, rt, m.rows, f32);
}
