// What the two kernels of the paged causal attention for prompt portions are handed, and the launcher of the one for the usual shapes.
#pragma once
#include "common.h"

struct PrefillArgs {
  const int* cu;
  const int* ctx;
  const int* table;
  int n_req, max_pages, page_size, num_pages;
  int page_shift;  // log2(page_size) if it is a power of two, else -1
  int nh, nkv, hd;
  long ldq, ldo;
  float scale;
  int window;
  int n_splits;    // slices of the key tiles (1: the workgroup writes the finished rows)
  // a bias on the scores by distance, or null: [nh, bias_len], row h entry d for keys d positions back (the last
  // entry for all farther ones), divided by `scale` already (it is added to the raw scores, which are scaled later)
  const float* bias;
  int bias_len;
  // a sink per head, or null: [nh]; the softmax's denominator also holds exp(sink[h]) (natural units, not scaled)
  const float* sink;
  int chunk;       // > 0: a row sees the keys of its own stretch of `chunk` positions (counted from 0) instead of a window
  float softcap;   // > 0: scaled scores are capped as softcap * tanh(s / softcap)
};

// What is done to the scores before the softmax: nothing, a bias by distance added, or a cap (and a bias, if there is one).
enum { SCORES_PLAIN = 0, SCORES_BIASED = 1, SCORES_CAPPED = 2 };

// Head sizes 64 and 128, pages of 8 keys or a larger power of two (a load of a wave covers 8 or 4 whole keys of one page), pools that start
// at 16 bytes.  (Which calls of those take it in a step: gibbs_rule_prefill.)
static inline bool prompt_attention_takes(int hd, int page_size, const void* kpages, const void* vpages) {
  return (hd == 64 || hd == 128) && page_size >= 8 && (page_size & (page_size - 1)) == 0 && ((uintptr_t)kpages | (uintptr_t)vpages) % 16 == 0;
}
// n_rows: of the requests cu[0] .. cu[n_req].
void launch_prompt_attention(const bf16* q, const bf16* kpages, const bf16* vpages, bf16* out, float* partial, const PrefillArgs& a,
                             int n_rows, hipStream_t stream);
