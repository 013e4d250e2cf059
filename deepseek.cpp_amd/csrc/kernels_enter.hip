// kernels_enter.hip -- steps of a few single tokens: the residual sum with its norm (and convolution) and the product that reads it, in one launch.
//
// By itself the sum is a chain of round trips that keeps memory idle for 4.5 us, and the product behind it starts with a round trip for its first
// weights.  Here the first workgroups make the rows, and the others - a feature tile to four waves that share k - request up to 16 KiB of weights a wave
// before anything else and wait for the rows with the weights on their way.  The product is few_body's, with the same sums in the same order.
//
// The hand-over: rows are stored past the caches, every storing wave waits until its stores have arrived, then one lane sets the workgroup's word; a reader
// polls the words and loads the rows with loads that its own caches do not serve.  The workgroups of the rows (ENTER_SPLIT for one of a sandwich layer) are the first
// of the grid and wait for nothing, so they are running before any reader looks; one that has looked `spins` times all the same reports it and goes on.
//
// What bounds it is that chain, slower among the weights' requests: a sum ready 4.3 us after the start of a launch of 8.7 MB is ready after 9 us in one
// of 69 MB, whose weights take 10.5.  Both launches / this one, us, one row of 2048: 33 MB behind blends 14.4 / 12.6, 33 MB 14.2 / 11.0, 8.7 MB 9.4 / 7.1, 69 MB
// 19.2 / 16.0, the logits' 419 MB 76.7 / 70.  16 tiles a wave ahead: with 12 the 69 MB take 18.0, with 8 18.6 (a second round waits for the rows), and 80 registers let
// three workgroups share a compute unit, all of a launch at once (84: 18.5).  (That is the sum alone and with the convolution; with blends behind it, 92 registers,
// two share one, and launches of more than 512 workgroups - more than 16 K features - come in two rounds.)  Readers that poll the rows themselves, a tag in every 8 bytes, took
// 19.2: their loads are in the sum's way.
//
// Up to 8 rows and a width of 2048 (launch_enter): a step of 27 lite layers, us of kernels, apart / together, one row 1914 / 1766, two 1926 / 1798, four 1997 / 1898, eight
// 2194 / 2144, but sixteen 2667 / 2740, as each reader takes all rows past its caches; four rows of 7168 by 1024 threads: 69 MB 21 / 26 us, 396 MB 80 / 80.
#include "join_device.h"
#include "layered_kernels.h"
#include "lin_device.h"

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
enum { ENTER_NT = 512, ENTER_TILES = ENTER_NT / 256, ENTER_AHEAD = 16, ENTER_LDS = 96 * 1024 };
// rounds of ENTER_AHEAD tiles in which a wave works off its k tiles, and LDS bytes of a row of them: zeros behind the last tile, rows start 4 banks apart
__host__ DEV int enter_rounds(int kt) { return (kt + 4 * ENTER_AHEAD - 1) / (4 * ENTER_AHEAD); }
__host__ DEV int enter_stride(int kt) { return enter_rounds(kt) * 4 * ENTER_AHEAD * 64 + 16; }

struct EnterArgs {
  JoinArgs j;
  LinArgs a;
  EnterSync s;
};
// KIND: 0 the sum and norm alone, 1 convolution behind them, 2 convolution and blends.  (What the first loads need stands alone in front of the arguments:
// that much of them is in registers when a wave starts.)
template <int KIND>
__global__ __launch_bounds__(ENTER_NT) void enter_kernel(const uint16_t* __restrict__ weights, const int kt, const int tiles, const int rows, const SeqDesc* __restrict__ seqs,
                                                   const unsigned* __restrict__ tag_at, const EnterArgs e) {
  constexpr int NT = ENTER_NT, U = ENTER_AHEAD;
  extern __shared__ __attribute__((aligned(16))) char xs[];
  __shared__ union {
    JoinLds<NT> join;
    float sums[NT * 4];
  } lds;
  LinArgs a = e.a;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int makers = KIND ? rows * ENTER_SPLIT : rows;
  if ((int)blockIdx.x < makers) {
    const unsigned tag = *tag_at + e.s.launch;
    if constexpr (KIND) sandwich_row<bf16, NT, 1, 8, ENTER_SPLIT, KIND == 2, true>(e.j, seqs, blockIdx.x, lds.join.red);
    else join_row<bf16, NT, 1, 4, 0, true>(e.j, blockIdx.x, lds.join);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) __hip_atomic_store(e.s.ready + blockIdx.x, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const int part = wave & 3, rt0 = ((int)blockIdx.x - makers) * ENTER_TILES, rt = rt0 + (wave >> 2);  // k tiles part, part + 4, ...
  const auto wr = range(weights + (size_t)min(rt, tiles - 1) * kt * 512, true, kt * 1024);
  const int at = part * 1024 + lane * 16;
  auto load = [&](int i) { return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, at + i * 4096, 0, 0)); };  // (zeros behind the last one)
  bf16x8 w[U];
#pragma unroll
  for (int u = 0; u < U; ++u) w[u] = load(u);
  __builtin_amdgcn_sched_barrier(0);
  if (a.out_at) a.out_f = glob(*glob(a.out_at));
  if (wave == 0) {
    const unsigned tag = *tag_at + e.s.launch;
    unsigned spins = 0;
    while (!__all(lane >= makers || __hip_atomic_load(e.s.ready + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == tag)) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins > e.s.spins) {
        if (lane == 0) __hip_atomic_store(e.s.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        break;
      }
    }
  }
  lds_barrier();
  // the rows into LDS, 16 bytes a thread
  const int stride = enter_stride(kt), rounds = enter_rounds(kt), per = rounds * U * 16;
  const bf16* h = operand<bf16>(a, rt0 * 16);
  for (int r = 0; r < rows; ++r) {
    const auto hr = range(h + (size_t)r * a.lda, true, kt * 64);
    for (int c = tid; c < per; c += NT) *reinterpret_cast<u32x4*>(xs + r * stride + c * 16) = __builtin_amdgcn_raw_buffer_load_b128(hr, c * 16, 0, 16 /* sc1 */);
  }
  lds_barrier();
  const char* x0 = xs + min(lane & 15, rows - 1) * stride + part * 64 + (lane >> 4) * 16;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto round = [&](int i, bool more) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc = mma(w[u], *reinterpret_cast<const bf16x8*>(x0 + (i + u) * 256), acc);
      if (more) w[u] = load(i + U + u);  // as soon as its registers are free
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int i = 0;
  for (; i < (rounds - 1) * U; i += U) round(i, true);
  round(i, false);
  *reinterpret_cast<f32x4*>(lds.sums + tid * 4) = acc;
  lds_barrier();
  if (part || rt >= tiles || (lane & 15) >= rows) return;
#pragma unroll
  for (int v = 1; v < 4; ++v) acc += *reinterpret_cast<const f32x4*>(lds.sums + (tid + v * 64) * 4);
  store_plain<bf16>(a, lane & 15, rt * 16 + (lane >> 4) * 4, acc);
}

bool enter_fits(const JoinArgs& j, const LinArgs& a) {
  return j.width <= 4 * ENTER_NT && !(j.width & 3) && (!j.conv.w || sandwich_fits(j)) && !j.h_f && a.parts <= 1 && !(a.a_seg % (16 * ENTER_TILES)) && a.rows <= ENTER_ROWS &&
         a.rows * enter_stride(a.kt) <= ENTER_LDS && a.kt <= 1 << 16;
}
int launch_enter(hipStream_t st, const JoinArgs& j, const LinArgs& a, const EnterSync& s) {
  const int n = j.only_want ? j.p.n_want : j.p.rows;
  if (!enter_fits(j, a) || n != a.rows || n < 1 || !j.norm_w || !a.w || !a.a_t || a.kt < 2 || (a.kt & 1) || a.rt < 1 || a.lda < a.kt * 32 || a.row_seq)
    DSK_FAIL(DSK_ERR_INVALID, "enter: width %d, %d of %d rows, kt %d rt %d lda %d", j.width, n, a.rows, a.kt, a.rt, a.lda);
  const int lds = n * enter_stride(a.kt);
  const EnterArgs e{j, a, s};
  const dim3 grid((j.conv.w ? n * ENTER_SPLIT : n) + (a.rt + ENTER_TILES - 1) / ENTER_TILES);
  auto k = !j.conv.w ? enter_kernel<0> : !j.conv.mu ? enter_kernel<1> : enter_kernel<2>;
  HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, ENTER_LDS));
  hipLaunchKernelGGL(k, grid, dim3(ENTER_NT), lds, st, a.w, a.kt, a.rt, n, j.p.seqs, s.tag, e);
  return DSK_OK;
}
