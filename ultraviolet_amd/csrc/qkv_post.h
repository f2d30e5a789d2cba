// The post-processing of the QKV projection as the kernels take it: model_ops.hip, and qkv_proj.hip, where it is part of the projection's launch.
#pragma once
#include "common.h"

namespace uvmi {

struct QkvArgs {
  const void* qkv; const void* xn; const void* ve_table; const float* ve_gate; const int64_t* tok;
  const int64_t* pos; const int64_t* rows; const int64_t* last_pos; const float* inv_freq;
  void* q_out; void* k_out; void* v_out;
  int8_t* k_cache; int8_t* v_cache; uint16_t* k_scale; uint16_t* v_scale;
  const float* gate_w; float* gate_out; float* vhat_out;
  int64_t scb, sch, scs, ssb, ssh;
  int64_t n, vocab;
  int H, KH, d, ve_ch, n_pairs, S, ring, has_ve, rope, q_dt, gate_ch;
  float eps, xsa_eps;
  const float* rope_tab; int rope_n;   // optional table of the rounded cos / sin per position (row: cos[n_pairs], sin[n_pairs])
  int64_t ld; int ext;                 // row pitch of qkv; gate logits read from columns W .. of the row instead of formed from xn
};

// model_ops.hip: uvmi_qkv_post's checks and the kernels' arguments.
int qkv_post_prepare(const uvmi_qkv_post_args* a, QkvArgs* out);
// 16-bit rows of 8 query heads on 1 kv head with the gates' logits behind them and a rotation of 16 pairs by table
bool qkv_post_engine_shape(const uvmi_qkv_post_args* a, const QkvArgs& A);

}  // namespace uvmi
