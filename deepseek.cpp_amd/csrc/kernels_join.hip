// kernels_join.hip -- between the matrix products of layered models: the 32-bit residual sum with the norm behind it, the causal
// convolution and the blends with the previous token that may follow the norm, and the router's choice of experts.
#include "join_device.h"
#include "layered_kernels.h"
#include "route_device.h"

#include <math.h>

// ---- residual + norm -----------------------------------------------------------------------------
template <typename T, int NT, int VPT, int V, int CONV>
__global__ __launch_bounds__(NT) void join_kernel(const JoinArgs a) {
  __shared__ JoinLds<NT> lds;
  join_row<T, NT, VPT, V, CONV, false>(a, blockIdx.x, lds);
}
template <typename T, int NT, int VPT, int PARTS, int SPLIT, bool MIX>
__global__ __launch_bounds__(NT) void sandwich_kernel(const SeqDesc* __restrict__ seqs, const JoinArgs a) {
  __shared__ float red[NT / 64];
  sandwich_row<T, NT, VPT, PARTS, SPLIT, MIX, false>(a, seqs, blockIdx.x, red);
}
template <typename T>
static int sandwich_t(hipStream_t st, const JoinArgs& a, int n) {
  const int D = a.width;
#define ROW(NT, VPT, PARTS, SPLIT) \
  hipLaunchKernelGGL((a.conv.mu ? sandwich_kernel<T, NT, VPT, PARTS, SPLIT, true> : sandwich_kernel<T, NT, VPT, PARTS, SPLIT, false>), dim3(n * SPLIT), dim3(NT), 0, st, a.p.seqs, a)
  if (D <= 1024) ROW(256, 1, 8, 1);
  else if (D <= 2048) ROW(512, 1, 8, 2);
  else if (D <= 4096) ROW(512, 2, 8, 4);
  else ROW(1024, 2, 4, 4);
#undef ROW
  return DSK_OK;
}
template <typename T, int CONV>
static int join_t(hipStream_t st, const JoinArgs& a, int n) {
  const int D = a.width;
#define JOIN(NT, VPT, V) hipLaunchKernelGGL((join_kernel<T, NT, VPT, V, CONV>), dim3(n), dim3(NT), 0, st, a)
  if (D > 16384) DSK_FAIL(DSK_ERR_UNSUPPORTED, "join: width %d (max 16384)", D);
  if (D & 3) {
    if (D <= 1024) JOIN(256, 4, 1);
    else JOIN(1024, 16, 1);
  } else if (D <= 256) JOIN(64, 1, 4);
  else if (D <= 1024) JOIN(256, 1, 4);
  else if (D <= 2048) JOIN(512, 1, 4);
  else if (D <= 4096) JOIN(512, 2, 4);
  else if (D <= 8192) JOIN(1024, 2, 4);
  else JOIN(1024, 4, 4);
#undef JOIN
  return DSK_OK;
}
bool join_moves(const JoinArgs& a) { return sandwich_fits(a); }
int launch_join(hipStream_t st, const JoinArgs& a, bool f32) {
  const int n = a.only_want ? a.p.n_want : a.p.rows;
  if (n < 1) DSK_FAIL(DSK_ERR_INVALID, "join: no rows");
  if (sandwich_fits(a)) return f32 ? sandwich_t<float>(st, a, n) : sandwich_t<bf16>(st, a, n);
  if (!a.conv.w) return f32 ? join_t<float, 0>(st, a, n) : join_t<bf16, 0>(st, a, n);
  if (a.conv.taps == 4 && a.conv.n_mix <= ConvOne<1, 4>::MAX_MIX) return f32 ? join_t<float, 4>(st, a, n) : join_t<bf16, 4>(st, a, n);
  return f32 ? join_t<float, 1>(st, a, n) : join_t<bf16, 1>(st, a, n);
}

// ---- convolution in front of a sublayer, portions --------------------------------------------------------
// A thread takes one channel of the (up to 16) rows of a chunk; TAPS = 0: any number of taps, read from memory again and again.
// Its rows are requested at once, from places that are always there, and what doesn't belong is dropped behind (behind a branch the compiler waits for
// each row); the kept inputs of the next portion come out of the registers.  What bounds it is that chain of loads, sums and stores, so a thread has one
// channel, not four, and a compute unit four times the waves: 2048 channels of 1996 rows 11.2 -> 10.5 us, of 301 rows in 32 bits 7.8 -> 6.2 (two channels: 11.7
// and 7.0).  With work for all of them either way the width of a load counts (conv_wide).
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void conv_kernel(const PassDesc p, int D, const float* __restrict__ h_f, const ConvArgs a) {
  constexpr int R = RECUR_CHUNK, K = TAPS ? TAPS : 1;
  const int c = blockIdx.y * 256 + threadIdx.x, taps = TAPS ? TAPS : a.taps;
  if (c >= D) return;
  const SeqDesc s = seq_at(p.seqs + p.chunk[2 * blockIdx.x]);
  const int t0 = p.chunk[2 * blockIdx.x + 1], n_rows = min(R, s.len - t0);
  const float* H = h_f + (size_t)s.row0 * D + c;
  const float* hist = reinterpret_cast<const float*>(s.state + a.off_in) + (size_t)s.flip * (taps - 1) * D + c;
  float* next = reinterpret_cast<float*>(s.state + a.off_in) + (size_t)(s.flip ^ 1) * (taps - 1) * D + c;
  float* P = a.mu ? reinterpret_cast<float*>(s.state + a.off_prev) + c : nullptr;
  T* out = reinterpret_cast<T*>(a.out_t) + (size_t)(s.row0 + t0) * a.ld + c;
  const bool has_prev = a.mu != nullptr;
  if constexpr (TAPS > 1) {
    float w[K], x[R + K], old[K], first = 0.f;  // inputs t0 - taps .. t0 + 15 (the first one only for the previous token's y)
#pragma unroll
    for (int r = 0; r < R + K; ++r) x[r] = H[(size_t)min(max(t0 - K + r, 0), s.len - 1) * D];
#pragma unroll
    for (int r = 1; r < K; ++r) old[r] = hist[(size_t)(r - 1) * D];
#pragma unroll
    for (int j = 0; j < K; ++j) w[j] = a.w[(size_t)c * K + j];
    if (has_prev) first = P[(size_t)s.flip * D];
#pragma unroll
    for (int r = 0; r < K; ++r) x[r] = t0 - K + r >= 0 ? x[r] : r > 0 && t0 == 0 && s.pos0 - K + r >= 0 ? old[r] : 0.f;
    float y[R + 1];  // behind the previous token's
#pragma unroll
    for (int t = 0; t <= R; ++t) {  // of input x[t + K - 1]
      float z = 0.f;
#pragma unroll
      for (int j = 0; j < K; ++j) z += x[t + j] * w[j];
      y[t] = x[t + K - 1] + z;
    }
    if (has_prev) y[0] = t0 > 0 ? y[0] : s.pos0 > 0 ? first : 0.f;
    for (int i = 0; i < (has_prev ? a.n_mix : 1); ++i) {
      const float mu = has_prev ? a.mu[(size_t)i * D + c] : 0.f;
#pragma unroll
      for (int t = 0; t < R; ++t)
        if (t < n_rows) out[i * a.mix_stride + (size_t)t * a.ld] = (T)(y[t + 1] + (y[t] - y[t + 1]) * mu);
    }
    if (t0 + n_rows < s.len) return;
    float last[K - 1], end = 0.f;  // the portion's end: what the next one needs, in the other copy
#pragma unroll
    for (int t = 0; t < R; ++t) {
      end = t < n_rows ? y[t + 1] : end;
#pragma unroll
      for (int j = 0; j < K - 1; ++j) last[j] = t == 0 || t < n_rows ? x[t + 2 + j] : last[j];
    }
#pragma unroll
    for (int j = 0; j < K - 1; ++j) next[(size_t)j * D] = last[j];
    if (has_prev) P[(size_t)(s.flip ^ 1) * D] = end;
  } else {
    auto input = [&](int u) {  // row u of the portion; before it: the kept inputs, zero before the sequence's start
      if (u >= 0) return H[(size_t)u * D];
      return u >= 1 - taps && s.pos0 + u >= 0 ? hist[(size_t)(u + taps - 1) * D] : 0.f;
    };
    auto conv = [&](int u) {
      float z = 0.f;
      for (int j = 0; j < taps; ++j) z += input(u - (taps - 1) + j) * a.w[(size_t)c * taps + j];
      return z + input(u);
    };
    float y = 0.f, prev = 0.f;
    if (has_prev) prev = t0 > 0 ? conv(t0 - 1) : s.pos0 > 0 ? P[(size_t)s.flip * D] : 0.f;
    for (int t = 0; t < n_rows; ++t) {
      y = conv(t0 + t);
      for (int i = 0; i < (has_prev ? a.n_mix : 1); ++i) out[i * a.mix_stride + (size_t)t * a.ld] = (T)(has_prev ? y + (prev - y) * a.mu[(size_t)i * D + c] : y);
      prev = y;
    }
    if (t0 + n_rows < s.len) return;
    for (int j = 0; j < taps - 1; ++j) next[(size_t)j * D] = input(s.len - (taps - 1) + j);
    if (has_prev) P[(size_t)(s.flip ^ 1) * D] = y;
  }
}
// The same with four channels a thread, by loads and stores of 16 bytes a lane: rows are requested as their places come, and the sums of a row are the same, in
// the same order.  Beyond 4 M elements (us with one channel / with four, without blends and with): 2048 channels of 700 rows 5.8 / 7.3 and 15.2 / 16.9, of 2000 8.6 / 8.7
// and 19.3 / 19.9, of 4000 15.1 / 13.1 and 32.9 / 25.3; 7168 channels of 300 rows 6.4 / 7.1 and 16.0 / 17.1, of 500 7.5 / 7.5 and 20.0 / 19.2, of 2000 20.3 / 17.8 and
// 40.9 / 31.1; in 32 bits, 2000 rows, 22.1 / 18.8.  (Slower in a few places where rows are a power of two apart: 4096 channels of 1600 rows 10.8 / 14.8.)
static bool conv_wide(const PassDesc& p, int D, const ConvArgs& a) {
  return a.taps >= 2 && a.taps <= 4 && !(D & 3) && !(a.ld & 3) && (size_t)p.n_chunks * D > 1 << 18;
}
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void conv_wide_kernel(const PassDesc p, int D, const float* __restrict__ h_f, const ConvArgs a) {
  constexpr int R = RECUR_CHUNK, K = TAPS;
  const int c = 4 * (blockIdx.y * 256 + threadIdx.x);
  if (c >= D) return;
  const SeqDesc s = seq_at(p.seqs + p.chunk[2 * blockIdx.x]);
  const int t0 = p.chunk[2 * blockIdx.x + 1], n_rows = min(R, s.len - t0);
  const float* H = h_f + (size_t)s.row0 * D + c;
  const float* hist = reinterpret_cast<const float*>(s.state + a.off_in) + (size_t)s.flip * (K - 1) * D + c;
  float* next = reinterpret_cast<float*>(s.state + a.off_in) + (size_t)(s.flip ^ 1) * (K - 1) * D + c;
  float* P = a.mu ? reinterpret_cast<float*>(s.state + a.off_prev) + c : nullptr;
  T* out = reinterpret_cast<T*>(a.out_t) + (size_t)(s.row0 + t0) * a.ld + c;
  const bool has_prev = a.mu != nullptr;
  auto input = [&](int u, float (&v)[4]) {  // row u of the portion; before it: the kept inputs, zero before the sequence's start
    if (u >= 0) load_v<float, 4>(H + (size_t)u * D, true, v);
    else load_v<float, 4>(hist + (size_t)(max(u, 1 - K) + K - 1) * D, u >= 1 - K && s.pos0 + u >= 0, v);
  };
  float w[4][K], x[R + K][4], y[R + 1][4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int j = 0; j < K; ++j) w[e][j] = a.w[(size_t)(c + e) * K + j];
#pragma unroll
  for (int r = 0; r < R + K; ++r) input(min(t0 - K + r, s.len - 1), x[r]);
#pragma unroll
  for (int t = 0; t <= R; ++t)  // of input x[t + K - 1]
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float z = 0.f;
#pragma unroll
      for (int j = 0; j < K; ++j) z += x[t + j][e] * w[e][j];
      y[t][e] = x[t + K - 1][e] + z;
    }
  if (has_prev && t0 == 0) load_v<float, 4>(P + (size_t)s.flip * D, s.pos0 > 0, y[0]);
  for (int i = 0; i < (has_prev ? a.n_mix : 1); ++i) {
    float mu[4];
    load_v<float, 4>(has_prev ? a.mu + (size_t)i * D + c : a.w, has_prev, mu);
#pragma unroll
    for (int t = 0; t < R; ++t) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = y[t + 1][e] + (y[t][e] - y[t + 1][e]) * mu[e];
      if (t < n_rows) store_v<T, 4>(out + i * a.mix_stride + (size_t)t * a.ld, v);
    }
  }
  if (t0 + n_rows < s.len) return;
  for (int j = 0; j < K - 1; ++j) {  // the portion's end: what the next one needs, in the other copy
    float v[4];
    input(s.len - (K - 1) + j, v);
    store_v<float, 4>(next + (size_t)j * D, v);
  }
  if (!has_prev) return;
#pragma unroll
  for (int t = 1; t < R; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) y[t + 1][e] = t < n_rows ? y[t + 1][e] : y[t][e];
  store_v<float, 4>(P + (size_t)(s.flip ^ 1) * D, y[R]);
}
template <typename T>
static void conv_t(hipStream_t st, const PassDesc& p, int D, const float* h_f, const ConvArgs& a) {
  if (conv_wide(p, D, a)) {
    const dim3 grid(p.n_chunks, (D / 4 + 255) / 256);
    if (a.taps == 2) hipLaunchKernelGGL((conv_wide_kernel<T, 2>), grid, dim3(256), 0, st, p, D, h_f, a);
    else if (a.taps == 3) hipLaunchKernelGGL((conv_wide_kernel<T, 3>), grid, dim3(256), 0, st, p, D, h_f, a);
    else hipLaunchKernelGGL((conv_wide_kernel<T, 4>), grid, dim3(256), 0, st, p, D, h_f, a);
    return;
  }
  const dim3 grid(p.n_chunks, (D + 255) / 256);
  switch (a.taps) {
    case 2: hipLaunchKernelGGL((conv_kernel<T, 2>), grid, dim3(256), 0, st, p, D, h_f, a); break;
    case 3: hipLaunchKernelGGL((conv_kernel<T, 3>), grid, dim3(256), 0, st, p, D, h_f, a); break;
    case 4: hipLaunchKernelGGL((conv_kernel<T, 4>), grid, dim3(256), 0, st, p, D, h_f, a); break;
    default: hipLaunchKernelGGL((conv_kernel<T, 0>), grid, dim3(256), 0, st, p, D, h_f, a);
  }
}
int launch_conv(hipStream_t st, const PassDesc& p, int width, const float* h_f, const ConvArgs& a, bool f32) {
  if (a.taps < 1 || width < 1 || p.n_chunks < 1) DSK_FAIL(DSK_ERR_INVALID, "conv: width %d, %d taps", width, a.taps);
  if (f32) conv_t<float>(st, p, width, h_f, a);
  else conv_t<bf16>(st, p, width, h_f, a);
  return DSK_OK;
}

// ---- router ----------------------------------------------------------------------------------------
// Many rows: two launches, ROUTE_ROWS rows to a workgroup in both.  The first chooses and leaves how often each expert was chosen by its rows; in the second every
// workgroup adds those up (offsets of the experts' ranges, and where its own rows' slots lie in them) and places its slots, and the tiles' table is made by all
// of them.  With counters in memory (a workgroup's counts added to them, a launch of one workgroup for the offsets, ranges taken from cursors) it was three
// launches, 11.0 + 4.7 + 4.8 us for 2048 rows and 64 experts, 8.7 + 4.6 + 4.6 for 40; two: 6.6 + 5.0 and 6.1 + 4.8.
// Every workgroup adding up all the others' counts is work by the square of the rows, so past ROUTE_SQUARE numbers read a launch between the two makes running sums of
// the counts and the second reads two of them an expert (route_sums_kernel).  Second launch alone, us: 4096 rows and 256 experts, at the line, 8.2; 8192 rows
// 19.0, with the sums 5.0 + 5.0; 16384 rows 61.7 and 5.5 + 6.3, of 64 experts 20.0 and 5.1 + 6.1.
enum { ROUTE_SQUARE = 1 << 24 };
static_assert(ROUTE_ROWS * 64 == 1024, "a wave a row, and a thread for each of its slots (check_route: at most 64)");
__global__ __launch_bounds__(1024) void route_count_kernel(const MoeArgs a) {  // a wave per row, one histogram
  __shared__ int hist[ROUTE_MAX_EXPERTS];
  const int tid = threadIdx.x, lane = tid & 63, ns = a.top + a.shared;
  for (int i = tid; i < a.experts; i += 1024) hist[i] = 0;
  const int row = blockIdx.x * ROUTE_ROWS + (tid >> 6);
  int e = 0;
  float w = 1.f;
  if (row < a.rows) choose(a.logits + (size_t)row * a.ld_logits, a.experts, a.top, lane, &e, &w);
  __syncthreads();
  if (row < a.rows) {
    if (lane < a.top) {
      atomicAdd(&hist[e], 1);
      a.chosen[(size_t)row * a.top + lane] = e;
    }
    if (lane < ns) a.weight[(size_t)row * ns + lane] = lane < a.top ? w : 1.f;
  }
  lds_barrier();
  for (int i = tid; i < a.experts; i += 1024) a.count[(size_t)blockIdx.x * a.experts + i] = hist[i];
}
// Running sums over the workgroups' counts, in place, the sums over all in a row behind them: 16 experts to a workgroup, 64 runs of its rows.
__global__ __launch_bounds__(1024) void route_sums_kernel(int* count, int experts, int groups) {
  __shared__ int part[16][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = tid & 15, run = tid >> 4, e = blockIdx.x * 16 + col;
  const int per = (groups + 63) / 64, g0 = min(run * per, groups), g1 = e < experts ? min(g0 + per, groups) : g0;
  int* const c = count + min(e, experts - 1);
  int sum = 0;
#pragma unroll 8
  for (int g = g0; g < g1; ++g) sum += c[(size_t)g * experts];
  int before = sum;  // inclusive over the wave's four runs, then over the waves
  for (int d = 16; d < 64; d <<= 1) {
    const int o = __shfl_up(before, d);
    before += lane >= d ? o : 0;
  }
  if (lane >= 48) part[wave][col] = before;
  before -= sum;
  __syncthreads();
  for (int w = 0; w < wave; ++w) before += part[w][col];
  if (run == 63 && e < experts) c[(size_t)groups * experts] = before + sum;
  for (int at = g0; at < g1; at += 8) {
    int v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c[(size_t)min(at + i, g1 - 1) * experts];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (at + i < g1) c[(size_t)(at + i) * experts] = before;
      before += v[i];
    }
  }
}
template <bool SUMMED>
__global__ __launch_bounds__(1024) void route_sort_kernel(const MoeArgs a) {
  __shared__ int total[1024], before[1024], base[ROUTE_MAX_EXPERTS], n[ROUTE_MAX_EXPERTS], wave_off[ROUTE_MAX_EXPERTS / 64], wave_til[ROUTE_MAX_EXPERTS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ns = a.top + a.shared, me = blockIdx.x, groups = gridDim.x;
  const int row = me * ROUTE_ROWS + tid / ns, k = tid % ns;  // this thread's slot (ns <= 64)
  const bool in = tid < ROUTE_ROWS * ns && row < a.rows;
  const int mine = in && k < a.top ? a.chosen[(size_t)row * a.top + k] : -1;
  const int shift = a.experts <= 64 ? 6 : a.experts <= 128 ? 7 : a.experts <= 256 ? 8 : 9, per = 1024 >> shift, e = tid & ((1 << shift) - 1);
  int sum = 0, sum_before = 0;
  if (!SUMMED && e < a.experts) {
    const int* c = a.count + e;
#pragma unroll 8
    for (int g = tid >> shift; g < groups; g += per) {
      const int v = c[(size_t)g * a.experts];
      sum += v;
      sum_before += g < me ? v : 0;
    }
  }
  if (!SUMMED) {
    total[tid] = sum;
    before[tid] = sum_before;
  }
  if (tid < ROUTE_MAX_EXPERTS) n[tid] = 0;
  __syncthreads();
  // experts' counts, and inclusive sums of counts and tiles: a thread an expert, within a wave and over the waves
  int count = 0, off = 0, til = 0;
  if (tid < ROUTE_MAX_EXPERTS) {
    int own_before = 0;
    if (SUMMED && tid < a.experts) {
      count = a.count[(size_t)groups * a.experts + tid];
      own_before = a.count[(size_t)me * a.experts + tid];
    } else if (tid < a.experts) {
      for (int g = 0; g < per; ++g) {
        count += total[(g << shift) + tid];
        own_before += before[(g << shift) + tid];
      }
    }
    off = count;
    til = (count + MOE_TILE - 1) / MOE_TILE;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(off, d), t = __shfl_up(til, d);
      off += lane >= d ? o : 0;
      til += lane >= d ? t : 0;
    }
    if (lane == 63) {
      wave_off[wave] = off;
      wave_til[wave] = til;
    }
    base[tid] = own_before;
  }
  __syncthreads();
  int slots = 0, t0 = 0;
#pragma unroll
  for (int w = 0; w < ROUTE_MAX_EXPERTS / 64; ++w) {
    if (w < wave) {
      off += wave_off[w];
      til += wave_til[w];
    }
    slots += wave_off[w];
    t0 += wave_til[w];
  }
  if (tid < a.experts) {
    base[tid] += off - count;
    if (tid % groups == me)
      for (int i = 0, t = til - (count + MOE_TILE - 1) / MOE_TILE; i < count; i += MOE_TILE, ++t) {
        a.tiles[4 * t] = tid;
        a.tiles[4 * t + 1] = off - count + i;
        a.tiles[4 * t + 2] = min(MOE_TILE, count - i);
      }
  }
  if (me == 0) {
    const int st = a.shared ? (a.rows + MOE_TILE - 1) / MOE_TILE : 0;
    for (int i = tid; i < st; i += 1024) {
      a.tiles[4 * (t0 + i)] = a.experts;
      a.tiles[4 * (t0 + i) + 1] = slots + i * MOE_TILE;
      a.tiles[4 * (t0 + i) + 2] = min(MOE_TILE, a.rows - i * MOE_TILE);
    }
    if (tid == 0) *a.n_tiles = t0 + st;
  }
  lds_barrier();
  if (!in) return;
  const int pos = mine >= 0 ? base[mine] + atomicAdd(&n[mine], 1) : a.rows * a.top + row;
  a.slot_pos[(size_t)row * ns + k] = pos;
  a.slot_row[pos] = row;
}
__global__ __launch_bounds__(1024) void route_few_kernel(const MoeArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[ROUTE_FEW_LDS];
  route_few_body(a, lds);
}
static int check_route(const MoeArgs& a) {
  if (a.experts < 1 || a.experts > ROUTE_MAX_EXPERTS || a.top < 1 || a.top > a.experts || a.top + a.shared > 64 || a.rows < 1)
    DSK_FAIL(DSK_ERR_UNSUPPORTED, "router: top %d of %d experts (at most 63 of %d)", a.top, a.experts, (int)ROUTE_MAX_EXPERTS);
  return DSK_OK;
}
int launch_route(hipStream_t st, const MoeArgs& a) {
  DSK_TRY(check_route(a));
  const dim3 grid((a.rows + ROUTE_ROWS - 1) / ROUTE_ROWS);
  hipLaunchKernelGGL(route_count_kernel, grid, dim3(1024), 0, st, a);
  if ((long long)grid.x * grid.x * a.experts > ROUTE_SQUARE) {
    hipLaunchKernelGGL(route_sums_kernel, dim3((a.experts + 15) / 16), dim3(1024), 0, st, a.count, a.experts, (int)grid.x);
    hipLaunchKernelGGL(route_sort_kernel<true>, grid, dim3(1024), 0, st, a);
  } else {
    hipLaunchKernelGGL(route_sort_kernel<false>, grid, dim3(1024), 0, st, a);
  }
  return DSK_OK;
}
int launch_route_few(hipStream_t st, const MoeArgs& a) {
  DSK_TRY(check_route(a));
  if (a.rows > 16) DSK_FAIL(DSK_ERR_INVALID, "route_few: %d rows", a.rows);
  hipLaunchKernelGGL(route_few_kernel, dim3(1), dim3(1024), 0, st, a);
  return DSK_OK;
}
