// registry.cpp -- model families: which one a checkpoint directory belongs to, and the C ABI calls that every family answers.
#include "checkpoint.h"
#include "context.h"

#include <sys/stat.h>

static const FamilyLoader*& loaders() {  // (a function-local static: families register from static initialisers)
  static const FamilyLoader* first = nullptr;
  return first;
}
FamilyLoader::FamilyLoader(bool (*c)(const char*), int (*o)(dsk_ctx*, const char*, int, const char*, dsk_model**)) : claims(c), open(o), next(loaders()) {
  loaders() = this;
}

// the architecture a checkpoint directory names: config.json's "architecture", or the metadata key "arch" of its first shard
static int read_architecture(const char* dir, std::string* arch) {
  const std::string path = std::string(dir) + "/config.json";
  struct stat sb;
  if (stat(path.c_str(), &sb) == 0) {
    std::string text;
    DSK_TRY(read_text_file(path, &text));
    JVal root;
    if (!json_parse(text, &root) || root.kind != JVal::OBJ) DSK_FAIL(DSK_ERR_INVALID, "loader: %s is not a JSON object", path.c_str());
    const JVal* a = root.get("architecture");
    if (!a || a->kind != JVal::STR) DSK_FAIL(DSK_ERR_INVALID, "loader: %s names no architecture", path.c_str());
    *arch = a->str;
    return DSK_OK;
  }
  Checkpoint ck;
  DSK_TRY(open_checkpoint(dir, ck));
  auto it = ck.meta.find("arch");
  if (it == ck.meta.end()) DSK_FAIL(DSK_ERR_INVALID, "loader: %s names no architecture", dir);
  *arch = it->second;
  return DSK_OK;
}

static int find_loader(const char* dir, std::string* arch, const FamilyLoader** out) {
  DSK_TRY(read_architecture(dir, arch));
  for (const FamilyLoader* l = loaders(); l; l = l->next)
    if (l->claims(arch->c_str())) {
      *out = l;
      return DSK_OK;
    }
  DSK_FAIL(DSK_ERR_UNSUPPORTED, "loader: no model family of this library knows the architecture '%s'", arch->c_str());
}

extern "C" int dsk_dir_architecture(const char* dir, char* out, int cap) {
  if (!dir || !out || cap < 1) DSK_FAIL(DSK_ERR_INVALID, "dir_architecture: null argument");
  std::string arch;
  const FamilyLoader* l = nullptr;
  DSK_TRY(find_loader(dir, &arch, &l));
  if ((int)arch.size() >= cap) DSK_FAIL(DSK_ERR_INVALID, "dir_architecture: the name needs %zu bytes", arch.size() + 1);
  arch.copy(out, arch.size());
  out[arch.size()] = 0;
  return DSK_OK;
}

extern "C" int dsk_model_open(dsk_ctx* ctx, const char* dir, int dtype, const char* options, dsk_model** out) {
  if (!ctx || !dir || !out) DSK_FAIL(DSK_ERR_INVALID, "model_open: null argument");
  if (dtype != DSK_DTYPE_BF16 && dtype != DSK_DTYPE_F32) DSK_FAIL(DSK_ERR_INVALID, "model_open: dtype %d", dtype);
  *out = nullptr;
  std::string arch;
  const FamilyLoader* l = nullptr;
  DSK_TRY(find_loader(dir, &arch, &l));
  return l->open(ctx, dir, dtype, options, out);
}

// ---- calls every family answers -------------------------------------------------------------------
#define FAMILY(m, what)                                           \
  if (!(m)) DSK_FAIL(DSK_ERR_INVALID, what ": null model");       \
  const Family& F = *model_head(m)->family

extern "C" int dsk_model_destroy(dsk_model* m) { return m ? model_head(m)->family->destroy(m) : DSK_OK; }
extern "C" const char* dsk_model_family(const dsk_model* m) { return m ? model_head(m)->family->name : ""; }
extern "C" int dsk_model_vocab_size(const dsk_model* m) { return m ? model_head(m)->family->vocab_size(m) : 0; }
extern "C" int dsk_forward(dsk_model* m, int token, int pos, int mode, float* host_logits) {
  FAMILY(m, "forward");
  return F.forward(m, token, pos, mode, host_logits);
}
extern "C" int dsk_hydrate(dsk_model* m, const int32_t* tokens, int n_tokens, int pos0, int mode, float* host_logits) {
  FAMILY(m, "hydrate");
  return F.hydrate(m, tokens, n_tokens, pos0, mode, host_logits);
}
extern "C" int dsk_forward_argmax(dsk_model* m, int token, int pos, int32_t* next_token) {
  FAMILY(m, "forward_argmax");
  return F.forward_argmax(m, token, pos, next_token);
}
extern "C" int dsk_forward_sample(dsk_model* m, int token, int pos, float temperature, float top_p, float coin, int32_t* next_token) {
  FAMILY(m, "forward_sample");
  return F.forward_sample(m, token, pos, temperature, top_p, coin, next_token);
}
extern "C" int dsk_forward_prob(dsk_model* m, int token, int pos, int index, float* prob) {
  FAMILY(m, "forward_prob");
  return F.forward_prob(m, token, pos, index, prob);
}
extern "C" float* dsk_model_host_logits(dsk_model* m) { return m ? model_head(m)->family->host_logits(m) : nullptr; }
extern "C" int dsk_model_set_graph(dsk_model* m, int enable) {
  FAMILY(m, "set_graph");
  return F.set_graph(m, enable);
}
extern "C" int dsk_model_set_trace(dsk_model* m, int enable) {
  FAMILY(m, "set_trace");
  return F.set_trace(m, enable);
}
extern "C" int dsk_model_get_trace_x(dsk_model* m, int layer, float* x_out) {
  FAMILY(m, "get_trace_x");
  return F.get_trace_x(m, layer, x_out);
}
extern "C" int dsk_hydrate_get_trace_x(dsk_model* m, int layer, int index, float* x_out) {
  FAMILY(m, "hydrate_get_trace_x");
  return F.trace_row(m, layer, index, x_out);
}
extern "C" int dsk_model_get_info(dsk_model* m, const char* key, int* value) {
  FAMILY(m, "get_info");
  return F.get_info(m, key, value);
}
extern "C" double dsk_model_active_bytes(const dsk_model* m, int pos) { return m ? model_head(m)->family->active_bytes(m, pos) : 0; }
extern "C" double dsk_model_device_bytes(const dsk_model* m) { return m ? model_head(m)->family->device_bytes(m) : 0; }
extern "C" int dsk_seq_open(dsk_model* m, int32_t* seq) {
  FAMILY(m, "seq_open");
  if (!seq) DSK_FAIL(DSK_ERR_INVALID, "seq_open: null output");
  return F.seq_open(m, seq);
}
extern "C" int dsk_seq_close(dsk_model* m, int32_t seq) {
  FAMILY(m, "seq_close");
  return F.seq_close(m, seq);
}
extern "C" int dsk_seq_pos(dsk_model* m, int32_t seq, int32_t* pos) {
  FAMILY(m, "seq_pos");
  if (!pos) DSK_FAIL(DSK_ERR_INVALID, "seq_pos: null output");
  return F.seq_pos(m, seq, pos);
}

// the checks of a step that do not depend on the family
static int check_step(dsk_model* m, const dsk_step_entry* e, int n) {
  if (!e || n < 1) DSK_FAIL(DSK_ERR_INVALID, "step: no entries");
  const int V = dsk_model_vocab_size(m);
  for (int i = 0; i < n; ++i) {
    if (e[i].n_tokens < 1 || !e[i].tokens) DSK_FAIL(DSK_ERR_INVALID, "step: entry %d has no tokens", i);
    for (int t = 0; t < e[i].n_tokens; ++t)
      if (e[i].tokens[t] < 0 || e[i].tokens[t] >= V) DSK_FAIL(DSK_ERR_INVALID, "step: entry %d: token %d out of range", i, e[i].tokens[t]);
    if (e[i].n_want < 0 || (e[i].n_want > 0 && !e[i].want)) DSK_FAIL(DSK_ERR_INVALID, "step: entry %d: bad list of places", i);
    for (int w = 0; w < e[i].n_want; ++w)
      if (e[i].want[w] < 0 || e[i].want[w] >= e[i].n_tokens) DSK_FAIL(DSK_ERR_INVALID, "step: entry %d: place %d of %d tokens", i, e[i].want[w], e[i].n_tokens);
    for (int k = 0; k < i; ++k)
      if (e[k].seq == e[i].seq) DSK_FAIL(DSK_ERR_INVALID, "step: sequence %d comes twice", e[i].seq);
  }
  return DSK_OK;
}
extern "C" int dsk_step(dsk_model* m, const dsk_step_entry* entries, int n, float* logits) {
  FAMILY(m, "step");
  DSK_TRY(check_step(m, entries, n));
  for (int i = 0; i < n; ++i)
    if (entries[i].n_want > 0 && !logits) DSK_FAIL(DSK_ERR_INVALID, "step: logits are asked for and there is no buffer");
  return F.step(m, entries, n, logits);
}
extern "C" int dsk_rows_lend(dsk_model* m, int n_rows, float** rows, dsk_rows** hold) {
  FAMILY(m, "rows_lend");
  if (!rows || !hold || n_rows < 1) DSK_FAIL(DSK_ERR_INVALID, "rows_lend: bad argument");
  *rows = nullptr;
  *hold = nullptr;
  return F.rows_lend ? F.rows_lend(m, n_rows, rows, hold) : DSK_OK;
}
extern "C" void dsk_rows_return(dsk_rows* hold) {
  if (!hold) return;
  RowPool* p = hold->pool;
  p->taken.fetch_and(~(1u << hold->slot), std::memory_order_release);
  p->let_go();
}
dsk_rows* RowPool::lend() {
  unsigned t = taken.load(std::memory_order_relaxed);
  for (;;) {
    unsigned i = 0;
    while (i < SLOTS && (t >> i & 1)) ++i;
    if (i == SLOTS) return nullptr;
    if (taken.compare_exchange_weak(t, t | 1u << i, std::memory_order_acquire)) {
      owners.fetch_add(1, std::memory_order_relaxed);
      return &slots[i];
    }
  }
}
bool RowPool::take_all() {
  unsigned none = 0;
  return taken.compare_exchange_strong(none, (1u << SLOTS) - 1, std::memory_order_acquire);
}
void RowPool::let_go() {
  if (owners.fetch_sub(1, std::memory_order_acq_rel) > 1) return;
  hipHostFree(mem);
  delete this;
}
extern "C" int dsk_step_sample(dsk_model* m, const dsk_step_entry* entries, int n, float temperature, float top_p, const float* coins, int32_t* next) {
  FAMILY(m, "step_sample");
  if (!next || (temperature != 0.0f && !coins)) DSK_FAIL(DSK_ERR_INVALID, "step_sample: null argument");
  DSK_TRY(check_step(m, entries, n));
  return F.step_sample(m, entries, n, temperature, top_p, coins, next);
}
