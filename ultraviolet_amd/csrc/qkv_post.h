// The post-processing of the QKV projection as the kernels take it: model_ops.hip, and qkv_proj.hip, where it is part of the projection's launch; and what
// else a launch of gemm_big.hip does beside its product.
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

// The query heads' part of it, as an epilogue of the projection takes it: columns 0 .. 511 are 8 heads, whose normed and rotated rows go to out
// (n, 512); a row whose position the table does not hold is normed only.
struct QueryPost { void* out; const int64_t* pos; const float* tab; int rope_n; float eps; };   // tab: null without a rotation

// The head's rows of the hidden (null: all of them) and the positions that its launch counts up (or null): uvmi_head.
struct HeadRows { const int64_t* rows; int a_rows; int64_t* advance; int64_t n_advance; };

// model_ops.hip: uvmi_qkv_post's checks and the kernels' arguments.
int qkv_post_prepare(const uvmi_qkv_post_args* a, QkvArgs* out);
// 16-bit rows of 8 query heads on 1 kv head with the gates' logits behind them and a rotation of 16 pairs by table
bool qkv_post_engine_shape(const uvmi_qkv_post_args* a, const QkvArgs& A);
// alignment that the rows' keys, values and caches need for 16-byte accesses
bool qkv_post_rows_ok(const uvmi_qkv_post_args* a);
// the rest of the post-processing behind such an epilogue (engine shape, qkv_post_rows_ok)
void qkv_post_kv_launch(int dtype, const QkvArgs& A, hipStream_t st);
// gemm.hip: the projection with that epilogue (sums: as uvmi_gemm_sums reads them, or null), if its tiles are loaded straight into LDS: whether it was launched
bool gemm_query_post(const uvmi_gemm_args* a, const QueryPost& q, float* sums, int64_t sums_ld, hipStream_t st);

}  // namespace uvmi
