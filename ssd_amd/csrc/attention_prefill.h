// Causal attention of many query rows (attention_prefill.hip), launched by ssd_attn_paged where its rule says so.
#pragma once
#include "common.h"

struct PrefillAttn {
  const bf16_t* q;            // [T][nh][hd]
  const bf16_t* kc;           // [pages][nkv][bs][hd]
  const bf16_t* vc;
  const int32_t* block_tables;
  const int32_t* context_lens;
  const int32_t* cu_q;        // [B + 1], or null: q_per_seq rows each
  bf16_t* out_rows;           // either may be null
  u32x2_t* out_frag;
  int max_blocks, q_per_seq, nh, nkv, bs_shift;
  float scale_log2e;
};
constexpr int PREFILL_ROWS = 128;       // (token, head) rows of one kv head per workgroup
constexpr int PREFILL_MIN_TOKENS = 161;       // in the batch
int attn_prefill_launch(const PrefillAttn& p, int B, int max_q, int hd, hipStream_t st);
