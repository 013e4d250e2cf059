// context.h -- the device context and the model-family seam shared by every family of models.
#pragma once
#include "dsk_internal.h"

#include <rccl/rccl.h>

#include <atomic>

// Where a tensor's bytes come from: host memory (dsk_model_bind) or a byte range of an open file (the .dseek
// loader, loader.cpp).  Either way they travel through the context's pinned staging ring (context.cpp stage_copy).
struct HostSrc {
  const void* ptr = nullptr;
  int fd = -1;
  uint64_t off = 0;  // file offset of byte 0 (fd >= 0)
};

struct dsk_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  ncclComm_t comm = nullptr;
  int rank = 0, world = 1;
  int n_cus = 256;       // compute units of the device (resident-grid kernels size themselves by it)
  int live_models = 0;   // models created on this context and not yet destroyed
  bool closing = false;  // dsk_ctx_destroy was called while models were alive: freed by the last dsk_model_destroy
  // scratch for op-level entry points
  void* op_buf[8] = {nullptr};
  size_t op_cap[8] = {0};
  // host -> HBM staging ring: STAGE_BUFS pinned buffers filled by reader threads (memcpy / pread) while the previous
  // one is in flight on the stream (hipMemcpyAsync); an event per buffer says when it may be refilled
  static const int STAGE_BUFS = 3;
  static const size_t STAGE_BYTES = (size_t)64 << 20;
  void* pin[STAGE_BUFS] = {nullptr};
  hipEvent_t pin_ev[STAGE_BUFS] = {nullptr};
  bool pin_busy[STAGE_BUFS] = {false};
  int pin_next = 0;
  double staged_bytes = 0, staged_fill_s = 0;  // bookkeeping for dsk_load_stats
};
void ctx_model_released(dsk_ctx* c);
int stage_copy(dsk_ctx* ctx, const HostSrc& src, uint64_t src_off, void* dev_dst, size_t bytes);

// ---- pinned rows that callers borrow (dsk_rows_lend) ----------------------------------------------
// Slots at the end of an allocation that a model makes and uses; it is freed when the model and every borrower have let go of it.
struct RowPool;
struct dsk_rows {
  RowPool* pool;
  unsigned slot;
};
struct RowPool {
  enum { SLOTS = 4 };
  char* mem;          // hipHostMalloc
  float* lent;        // slot i: lent + i * slot_floats
  size_t slot_floats;
  std::atomic<unsigned> taken{0};
  std::atomic<int> owners{1};
  dsk_rows slots[SLOTS];
  RowPool(void* m, float* first, size_t floats) : mem((char*)m), lent(first), slot_floats(floats) {
    for (unsigned i = 0; i < SLOTS; ++i) slots[i] = {this, i};
  }
  dsk_rows* lend();   // nullptr: none left
  bool take_all();    // nobody has borrowed any, and nobody can until give_all()
  void give_all() { taken.store(0, std::memory_order_release); }
  void let_go();      // one owner less
  float* rows(const dsk_rows* r) const { return lent + r->slot * slot_floats; }
  bool holds(const float* p, size_t n) const { return p >= lent && p + n <= lent + SLOTS * slot_floats; }
};

// ---- model families -------------------------------------------------------------------------------
// A dsk_model handle is one of several concrete types; all of them start with a ModelHead, whose table carries the calls
// every family answers (registry.cpp dispatches them).  Calls that exist for one family only check the table (family_is).
struct Family {
  const char* name;
  int (*destroy)(dsk_model*);
  int (*vocab_size)(const dsk_model*);
  int (*forward)(dsk_model*, int token, int pos, int mode, float* host_logits);
  int (*hydrate)(dsk_model*, const int32_t* tokens, int n, int pos0, int mode, float* host_logits);
  int (*forward_argmax)(dsk_model*, int token, int pos, int32_t* next);
  int (*forward_sample)(dsk_model*, int token, int pos, float temperature, float top_p, float coin, int32_t* next);
  int (*forward_prob)(dsk_model*, int token, int pos, int index, float* prob);
  float* (*host_logits)(dsk_model*);
  int (*set_graph)(dsk_model*, int);
  int (*set_trace)(dsk_model*, int);
  int (*get_trace_x)(dsk_model*, int layer, float* x);
  int (*trace_row)(dsk_model*, int layer, int row, float* x);  // row of the last pass
  int (*get_info)(dsk_model*, const char* key, int* value);
  double (*active_bytes)(const dsk_model*, int pos);
  double (*device_bytes)(const dsk_model*);
  int (*seq_open)(dsk_model*, int32_t* seq);
  int (*seq_close)(dsk_model*, int32_t seq);
  int (*seq_pos)(dsk_model*, int32_t seq, int32_t* pos);
  int (*step)(dsk_model*, const dsk_step_entry* entries, int n, float* logits);
  int (*step_sample)(dsk_model*, const dsk_step_entry* entries, int n, float temperature, float top_p, const float* coins, int32_t* next);
  int (*rows_lend)(dsk_model*, int n_rows, float** rows, dsk_rows** hold);  // nullptr: lends none
};
struct ModelHead {
  const Family* family = nullptr;
  dsk_ctx* ctx = nullptr;
};
static inline ModelHead* model_head(dsk_model* m) { return reinterpret_cast<ModelHead*>(m); }
static inline const ModelHead* model_head(const dsk_model* m) { return reinterpret_cast<const ModelHead*>(m); }
static inline bool family_is(const dsk_model* m, const Family& f) { return m && model_head(m)->family == &f; }

// How a family is found for a checkpoint directory: config.json's "architecture" when there is one, the metadata key "arch" of a
// .dseek shard otherwise.  `open` loads the model; families register themselves (static objects) in registry.cpp's list.
struct FamilyLoader {
  bool (*claims)(const char* architecture);
  int (*open)(dsk_ctx* ctx, const char* dir, int dtype, const char* options, dsk_model** out);
  const FamilyLoader* next;
  FamilyLoader(bool (*c)(const char*), int (*o)(dsk_ctx*, const char*, int, const char*, dsk_model**));
};
