// hyd_rounds.h -- workgroups of a plain matrix of a batched prompt (kernels_hydrate.hip), for the launch, the kernel and the host's check of them.
//
// (chunk of 32 tokens, group of strips) pairs, chunk-major, one workgroup to a compute unit.  What is left for a last round of at most half the units goes out as
// two workgroups of 16 tokens each: first the first halves of all that is left, then the second ones, of which a last chunk of up to 16 tokens has
// none.  (Halves beside each other, with those that have no tokens among them, had half of the chip's XCDs - workgroups go round them - take all the work:
// DeepSeek-V3's wo at 129 and 144 tokens 97 and 101 us as whole pairs, 115 and 117 so.)
#pragma once
#if defined(__HIPCC__)
#define HYD_ROUNDS_FN __host__ __device__ __forceinline__
#else
#define HYD_ROUNDS_FN inline
#endif

struct HydRounds { int full, left; };  // pairs as one workgroup of 32 tokens, and those behind them as halves (0: none)
inline HydRounds hyd_rounds(long long pairs, int cus) {
  const long long left = pairs % cus;
  return left > 0 && left <= cus / 2 && pairs + left < (1ll << 30) ? HydRounds{(int)(pairs - left), (int)left} : HydRounds{(int)(pairs < (1ll << 30) ? pairs : 0), 0};
}
inline int hyd_rounds_grid(const HydRounds& R, int groups, int m) {
  const int empty = (m + 31) % 32 < 16 ? (R.left < groups ? R.left : groups) : 0;  // pairs of a last chunk of up to 16 tokens
  return R.full + 2 * R.left - empty;
}
struct HydRound { int base, group; bool half; };  // first token, strip group; half: 16 tokens
HYD_ROUNDS_FN HydRound hyd_round(const HydRounds& R, int groups, int b) {
  const int k = b - R.full, second = b >= R.full && k >= R.left ? 1 : 0, pair = b < R.full ? b : R.full + k - second * R.left;
  return {pair / groups * 32 + second * 16, pair % groups, b >= R.full};
}
