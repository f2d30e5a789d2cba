// A pass as one call: the launches of all layers back to back, without a host language between them.  A decode step of
// UV-50M is 42 to 52 launches of ~5 us; prepared and issued one by one from Python they cost ~12 us of host time each, so
// the GPU waited for the host half of the time (0.65 ms a step on one row, 0.33 ms from this list, 0.18 ms now).
#include "common.h"

namespace uvmi {
int norm_run(const uvmi_norm_args* a, void* stream);   // model_ops.hip
}

extern "C" int uvmi_run_ops(const int* kinds, const void* const* args, int n_ops, void* stream) {
  UVMI_REQUIRE(n_ops >= 0 && (n_ops == 0 || (kinds && args)), UVMI_EINVAL, "uvmi_run_ops: null pointer or negative count");
  for (int i = 0; i < n_ops; i++) {
    const void* a = args[i];
    UVMI_REQUIRE(a, UVMI_EINVAL, "uvmi_run_ops: operation %d has no arguments", i);
    int rc;
    switch (kinds[i]) {
      case UVMI_OP_GEMM: rc = uvmi_gemm_tn_ex((const uvmi_gemm_args*)a, stream); break;
      case UVMI_OP_DECODE_ATTN: rc = uvmi_decode_attn((const uvmi_attn_args*)a, stream); break;
      case UVMI_OP_QKV_POST: rc = uvmi_qkv_post((const uvmi_qkv_post_args*)a, stream); break;
      case UVMI_OP_PREFILL_ATTN: rc = uvmi_prefill_attn((const uvmi_prefill_attn_args*)a, stream); break;
      case UVMI_OP_QKV_PROJ: rc = uvmi_qkv_proj((const struct uvmi_qkv_proj_args*)a, stream); break;
      case UVMI_OP_PREFILL_ATTN_O: rc = uvmi_prefill_attn_o((const struct uvmi_prefill_attn_o_args*)a, stream); break;
      case UVMI_OP_GEMM_RESID: rc = uvmi_gemm_resid((const uvmi_gemm_args*)a, stream); break;
      case UVMI_OP_GEMM_SUMS: rc = uvmi_gemm_sums((const struct uvmi_gemm_sums_args*)a, stream); break;
      case UVMI_OP_NORM: rc = uvmi::norm_run((const uvmi_norm_args*)a, stream); break;
      default: UVMI_REQUIRE(false, UVMI_EINVAL, "uvmi_run_ops: operation %d has the unknown kind %d", i, kinds[i]);
    }
    if (rc) return rc;
  }
  return UVMI_OK;
}
