// head_rows.h -- which bytes of a layer's key and value caches a head of kernels_head.hip requests, for the kernels and for the host's check of them.
//
// The caches are as long as the context allows, without rows behind it.  A raw buffer load of an offset at or past the descriptor's records
// returns zeros and reads nothing; that test is of the lane's offset (the scalar one is taken off the records, which says nothing once it is larger than they
// are).  So the whole offset is the lane's, steps that begin behind the context are not requested at all, and nothing here passes 32 bits (head_rows_fit).
#pragma once
#if defined(__HIPCC__)
#define HEAD_ROWS_FN __host__ __device__ __forceinline__
#else
#define HEAD_ROWS_FN inline
#endif

enum { HEAD_KEY_STEP = 64 };                        // positions of a workgroup's step over the keys: 16 lanes each
constexpr unsigned HEAD_NOWHERE = 0x80000000u;      // (a value lane without a place: stays past the records with any position added)

// keys: lanes (pos in a step, sl); + 128 and + 256 bytes for the lane's second and third values
HEAD_ROWS_FN unsigned head_key_at(int pos, int sl, int H, int h, int hd) { return ((unsigned)pos * (unsigned)H + (unsigned)h) * (unsigned)hd * 2u + (unsigned)sl * 8u; }
// values: threads (g, i4) of TG groups
HEAD_ROWS_FN unsigned head_value_at(int g, int i4, int TG, int H, int h, int vd) {
  return g < TG ? ((unsigned)g * (unsigned)H + (unsigned)h) * (unsigned)vd * 2u + (unsigned)i4 * 8u : HEAD_NOWHERE;
}
// a row's bytes, and a step's distance: `first` positions into the context
HEAD_ROWS_FN unsigned head_row_bytes(int H, int d) { return (unsigned)H * (unsigned)d * 2u; }
HEAD_ROWS_FN bool head_step_there(int first, int kv_len) { return first < kv_len; }
// records below 2^31 (a descriptor's are an int), and no offset past 32 bits: a step's last lanes are up to 1024 positions of vd = 4 or 64 of hd behind the context
inline bool head_rows_fit(int max_kv, int H, int hd, int vd) {
  const double row = (double)H * (hd > vd ? hd : vd) * 2.0;
  return max_kv * row < 2147483648.0 && (double)H * hd * 2.0 * HEAD_KEY_STEP + 512.0 < 1073741824.0 && (double)H * vd * 2.0 * (1024 / (vd / 4 > 0 ? vd / 4 : 1)) < 1073741824.0;
}
