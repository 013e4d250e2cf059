// deepseek_family.cpp -- the DeepSeek engine's row of the model-family table: the single-sequence engine behind dsk_step.
#include "engine.h"

#include <string.h>

static int ds_vocab_size(const dsk_model* m) { return m->c.vocab_size; }

// one KV cache per model, so one sequence at a time; its rows need no clearing (attention reads rows below the position only)
static int ds_seq_open(dsk_model* m, int32_t* seq) {
  if (!m->finalized) DSK_FAIL(DSK_ERR_STATE, "seq_open before finalize");
  if (m->live_seq >= 0) DSK_FAIL(DSK_ERR_UNSUPPORTED, "seq_open: a DeepSeek model holds one sequence at a time (sequence %d is live)", m->live_seq);
  m->live_seq = 0;
  m->live_pos = 0;
  *seq = 0;
  return DSK_OK;
}
static int ds_check_seq(dsk_model* m, int32_t seq) {
  if (seq != 0 || m->live_seq != 0) DSK_FAIL(DSK_ERR_INVALID, "sequence %d is not open", seq);
  return DSK_OK;
}
static int ds_seq_close(dsk_model* m, int32_t seq) {
  DSK_TRY(ds_check_seq(m, seq));
  m->live_seq = -1;
  return DSK_OK;
}
static int ds_seq_pos(dsk_model* m, int32_t seq, int32_t* pos) {
  DSK_TRY(ds_check_seq(m, seq));
  *pos = m->live_pos;
  return DSK_OK;
}
static int ds_step(dsk_model* m, const dsk_step_entry* e, int n, float* logits) {
  if (n != 1) DSK_FAIL(DSK_ERR_UNSUPPORTED, "step: a DeepSeek model runs one sequence at a time");
  DSK_TRY(ds_check_seq(m, e->seq));
  float* out = logits;
  int done = 0, w = 0;
  while (done < e->n_tokens) {  // up to the next wanted place in one prompt chunk
    if (w < e->n_want && e->want[w] < done) DSK_FAIL(DSK_ERR_UNSUPPORTED, "step: the wanted places must ascend");
    const bool want = w < e->n_want;
    const int end = want ? e->want[w] + 1 : e->n_tokens;
    const int mode = want ? DSK_MODE_OUTPUT_LOGITS : DSK_MODE_HYDRATE_KV_CACHE;
    if (end - done == 1) DSK_TRY(ds_forward(m, e->tokens[done], m->live_pos, mode, out));
    else DSK_TRY(ds_hydrate(m, e->tokens + done, end - done, m->live_pos, mode, out));
    m->live_pos += end - done;
    done = end;
    if (want) {
      out += m->c.vocab_size;
      ++w;
    }
  }
  return DSK_OK;
}
static int ds_step_sample(dsk_model* m, const dsk_step_entry* e, int n, float temperature, float top_p, const float* coins, int32_t* next) {
  if (n != 1) DSK_FAIL(DSK_ERR_UNSUPPORTED, "step: a DeepSeek model runs one sequence at a time");
  DSK_TRY(ds_check_seq(m, e->seq));
  if (e->n_tokens > 1) {
    DSK_TRY(ds_hydrate(m, e->tokens, e->n_tokens - 1, m->live_pos, DSK_MODE_HYDRATE_KV_CACHE, nullptr));
    m->live_pos += e->n_tokens - 1;
  }
  const int last = e->tokens[e->n_tokens - 1];
  DSK_TRY(temperature == 0.0f ? ds_forward_argmax(m, last, m->live_pos, next) : ds_forward_sample(m, last, m->live_pos, temperature, top_p, coins[0], next));
  m->live_pos++;
  return DSK_OK;
}

Family deepseek_family = {  // (not const: a const table of host functions would be emitted for the device too)
    "deepseek",       ds_destroy,  ds_vocab_size, ds_forward,     ds_hydrate,  ds_forward_argmax, ds_forward_sample, ds_forward_prob, ds_host_logits, ds_set_graph,
    ds_set_trace,     ds_get_trace_x, ds_trace_row, ds_get_info, ds_active_bytes, ds_device_bytes, ds_seq_open, ds_seq_close,     ds_seq_pos,      ds_step,        ds_step_sample, nullptr};

static bool ds_claims(const char* arch) { return !strncmp(arch, "Deepseek", 8); }
static int ds_open(dsk_ctx* ctx, const char* dir, int dtype, const char* options, dsk_model** out) {
  if (dtype == DSK_DTYPE_F32) DSK_FAIL(DSK_ERR_UNSUPPORTED, "a .dseek checkpoint runs in the precision its quantisation names");
  return dsk_model_load_dseek_opts(ctx, dir, 0, options, out, nullptr);
}
static FamilyLoader ds_loader(ds_claims, ds_open);
