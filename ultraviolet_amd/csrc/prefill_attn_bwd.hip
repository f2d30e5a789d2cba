// Backward of the packed (cu_seqlens) causal attention with an optional sliding window: dq, dk, dv from the output
// gradient (reference: mathk::varlen_attn_bwd, ultraviolet/kernels/varlen_attn.py:56-66, which calls
// aten._efficient_attention_backward on K / V expanded to the query heads and sums their gradients back over a group).
//
// With s_ij = scale q_i . k_j over the keys j query i sees (same segment, i - window < j <= i), p_ij = exp(s_ij - lse_i),
// D_i = go_i . o_i:   dv_j = sum_i p_ij go_i,   ds_ij = p_ij (go_i . v_j - D_i),   dq_i = scale sum_j ds_ij k_j,
// dk_j = scale sum_i ds_ij q_i  (dk, dv also summed over the query heads of the group).
//
// Two forms.  The matrix-core form (bwd_dq_mfma, bwd_dkv_heads, described where they are defined) serves up to 8 query heads
// per kv head.  The plain form below it serves the rest: fp32 arithmetic on the vector units, no atomics, no
// cross-workgroup state.
//   bwd_dq_kernel   lane = query token (64 per wave), one query head per workgroup: the wave walks the union of its
//                   queries' key ranges; a key / value row is the same address in every lane.  Pass 1 recomputes the
//                   row's log-sum-exp (the forward does not keep it), pass 2 accumulates dq in registers.  Writes
//                   lse and D for the second kernel.
//   bwd_dkv_kernel  two lanes per key (32 head dims each, 32 keys per wave), one kv head per workgroup: the wave walks
//                   the queries that see its keys and the heads of the group; dk and dv stay in registers.
#include "common.h"
#include "attn_mfma_util.h"
#include "gemm_util.h"

#include <climits>

namespace uvmi {

struct BwdParams {
  const void* q; const void* k; const void* v; const void* o; const void* go;
  void* dq; void* dk; void* dv;
  float* lse; float* dsum;   // (N, H) each
  const void* cu; int idx64, n_seg, N, H, KH, G, window;
  float scale;
};

template <int DT>
__device__ __forceinline__ void bld8(const void* p, int64_t i, float* o) {  // 8 consecutive 16-bit elements from element i
  const uint4 w = *(const uint4*)((const uint16_t*)p + i);
  const uint32_t r[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (DT == UVMI_BF16) {
      o[2 * j] = __uint_as_float(r[j] << 16);
      o[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u);
    } else {
      o[2 * j] = half_bits_to_float((uint16_t)(r[j] & 0xffff));
      o[2 * j + 1] = half_bits_to_float((uint16_t)(r[j] >> 16));
    }
  }
}
template <int DT>
__device__ __forceinline__ void bst8(void* p, int64_t i, const float* v) {
  uint32_t r[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (DT == UVMI_BF16) r[j] = float2_to_bf16x2(v[2 * j], v[2 * j + 1]);
    else r[j] = (uint32_t)float_to_half_bits(v[2 * j]) | ((uint32_t)float_to_half_bits(v[2 * j + 1]) << 16);
  }
  *(uint4*)((uint16_t*)p + i) = uint4{r[0], r[1], r[2], r[3]};
}

__device__ __forceinline__ int wave_min_i(int v) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// index s of the segment that holds token t: the last s < n_seg with cu[s] <= t (empty segments are skipped)
__device__ __forceinline__ int segment_of(const BwdParams& P, int t) {
  int lo = 0, hi = P.n_seg;  // invariant: cu[lo] <= t, and hi == n_seg or cu[hi] > t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (load_index(P.cu, P.idx64, mid) <= t) lo = mid; else hi = mid;
  }
  return lo;
}

template <int DT>
__global__ __launch_bounds__(64) void bwd_dq_kernel(BwdParams P) {
  const int lane = threadIdx.x, h = blockIdx.y, kh = h / P.G;
  const int i = blockIdx.x * 64 + lane;
  int n_end = (int)load_index(P.cu, P.idx64, P.n_seg);   // tokens at or after it are padding
  n_end = n_end < 0 ? 0 : (n_end > P.N ? P.N : n_end);
  const bool live = i < n_end;
  int lo = 0x7fffffff, hi = -1;   // keys lo..hi (inclusive)
  if (live) {
    int seg0 = (int)load_index(P.cu, P.idx64, segment_of(P, i));
    if (seg0 < 0) seg0 = 0;
    lo = P.window > 0 && i - P.window + 1 > seg0 ? i - P.window + 1 : seg0;
    hi = i;
  }
  const int jmin = __builtin_amdgcn_readfirstlane(wave_min_i(lo)), jmax = __builtin_amdgcn_readfirstlane(wave_max_i(hi));
  const int64_t qrow = ((int64_t)(live ? i : 0) * P.H + h) * 64;
  float q[64], g[64], dq[64];
  float D = 0.f;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    float o8[8];
    bld8<DT>(P.q, qrow + 8 * c, q + 8 * c);
    bld8<DT>(P.go, qrow + 8 * c, g + 8 * c);
    bld8<DT>(P.o, qrow + 8 * c, o8);
#pragma unroll
    for (int d = 0; d < 8; d++) {
      D = fmaf(g[8 * c + d], o8[d], D);
      dq[8 * c + d] = 0.f;
    }
  }
  auto score = [&](int j) {
    const int64_t kr = ((int64_t)j * P.KH + kh) * 64;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      float k8[8];
      bld8<DT>(P.k, kr + 8 * c, k8);
#pragma unroll
      for (int d = 0; d < 8; d++) s = fmaf(q[8 * c + d], k8[d], s);
    }
    return s * P.scale;
  };
  // ---- pass 1: log-sum-exp of the row
  float m = -INFINITY, l = 0.f;
  for (int j = jmin; j <= jmax; j++) {
    const float s = score(j);
    if (j >= lo && j <= hi) {
      const float mn = fmaxf(m, s);
      l = l * __expf(m - mn) + __expf(s - mn);
      m = mn;
    }
  }
  const float lse = live ? m + __logf(l) : 0.f;   // (a live query sees at least itself)
  // ---- pass 2: dq
  for (int j = jmin; j <= jmax; j++) {
    const float s = score(j);
    const bool ok = j >= lo && j <= hi;
    const float p = ok ? __expf(s - lse) : 0.f;
    const int64_t kr = ((int64_t)j * P.KH + kh) * 64;
    float dp = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      float v8[8];
      bld8<DT>(P.v, kr + 8 * c, v8);
#pragma unroll
      for (int d = 0; d < 8; d++) dp = fmaf(g[8 * c + d], v8[d], dp);
    }
    const float ds = p * (dp - D);
#pragma unroll
    for (int c = 0; c < 8; c++) {
      float k8[8];
      bld8<DT>(P.k, kr + 8 * c, k8);
#pragma unroll
      for (int d = 0; d < 8; d++) dq[8 * c + d] = fmaf(ds, k8[d], dq[8 * c + d]);
    }
  }
  if (i < P.N) {
    const int64_t orow = ((int64_t)i * P.H + h) * 64;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      float o8[8];
#pragma unroll
      for (int d = 0; d < 8; d++) o8[d] = live ? dq[8 * c + d] * P.scale : 0.f;
      bst8<DT>(P.dq, orow + 8 * c, o8);
    }
    P.lse[(int64_t)i * P.H + h] = lse;
    P.dsum[(int64_t)i * P.H + h] = live ? D : 0.f;
  }
}

template <int DT>
__global__ __launch_bounds__(64) void bwd_dkv_kernel(BwdParams P) {
  const int lane = threadIdx.x, jj = lane >> 1, half = lane & 1, kh = blockIdx.y;
  const int j = blockIdx.x * 32 + jj;
  int n_end = (int)load_index(P.cu, P.idx64, P.n_seg);
  n_end = n_end < 0 ? 0 : (n_end > P.N ? P.N : n_end);
  const bool live = j < n_end && j >= (int)load_index(P.cu, P.idx64, 0);   // (in a sequence)
  int lo = 0x7fffffff, hi = 0;   // queries lo .. hi - 1 see key j
  if (live) {
    int se = (int)load_index(P.cu, P.idx64, segment_of(P, j) + 1);
    se = se > n_end ? n_end : se;
    lo = j;
    hi = P.window > 0 && j + P.window < se ? j + P.window : se;
  }
  const int imin = __builtin_amdgcn_readfirstlane(wave_min_i(lo)), imax = __builtin_amdgcn_readfirstlane(wave_max_i(hi)) - 1;
  const int64_t krow = ((int64_t)(live ? j : 0) * P.KH + kh) * 64 + 32 * half;
  float kk[32], vv[32], dk[32], dv[32];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    bld8<DT>(P.k, krow + 8 * c, kk + 8 * c);
    bld8<DT>(P.v, krow + 8 * c, vv + 8 * c);
#pragma unroll
    for (int d = 0; d < 8; d++) { dk[8 * c + d] = 0.f; dv[8 * c + d] = 0.f; }
  }
  for (int i = imin; i <= imax; i++) {
    const bool ok = live && i >= lo && i < hi;
    for (int hh = 0; hh < P.G; hh++) {
      const int h = kh * P.G + hh;
      const int64_t qrow = ((int64_t)i * P.H + h) * 64 + 32 * half;
      float qh[32], gh[32];
      float s = 0.f, dp = 0.f;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        bld8<DT>(P.q, qrow + 8 * c, qh + 8 * c);
        bld8<DT>(P.go, qrow + 8 * c, gh + 8 * c);
#pragma unroll
        for (int d = 0; d < 8; d++) {
          s = fmaf(qh[8 * c + d], kk[8 * c + d], s);
          dp = fmaf(gh[8 * c + d], vv[8 * c + d], dp);
        }
      }
      s += __shfl_xor(s, 1, 64);
      dp += __shfl_xor(dp, 1, 64);
      const float p = ok ? __expf(s * P.scale - P.lse[(int64_t)i * P.H + h]) : 0.f;
      const float ds = p * (dp - P.dsum[(int64_t)i * P.H + h]);
#pragma unroll
      for (int d = 0; d < 32; d++) {
        dv[d] = fmaf(p, gh[d], dv[d]);
        dk[d] = fmaf(ds, qh[d], dk[d]);
      }
    }
  }
  if (j < P.N) {
    const int64_t orow = ((int64_t)j * P.KH + kh) * 64 + 32 * half;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      float a8[8], b8[8];
#pragma unroll
      for (int d = 0; d < 8; d++) { a8[d] = live ? dk[8 * c + d] * P.scale : 0.f; b8[d] = live ? dv[8 * c + d] : 0.f; }
      bst8<DT>(P.dk, orow + 8 * c, a8);
      bst8<DT>(P.dv, orow + 8 * c, b8);
    }
  }
}

// ------------------------------------------------------------------------------------------------ the MFMA form
// Same mathematics on the matrix cores, on the forward kernel's operand layouts (prefill_attn.hip):
//   * the rows' log-sum-exp (log2 domain) is the forward's, or comes from one more run of the forward kernel without output;
//   * bwd_dq_mfma: a workgroup owns 16 query rows of one kv head, wave w the query heads 2w, 2w+1 of the group (w up to four of them).  K and V
//     super-tiles (32 keys) are staged once per workgroup in LDS, two tiles to a barrier, as in the forward.  S^T = K Q^T and dP^T = V dO^T have the same shape: a lane
//     of either accumulator holds 4 consecutive keys of one query row for two 16-key tiles, so p = exp2(c s - lse) and
//     ds = p (dp - D) are lane-local, and the 8 values of ds, rounded to the input type, are the lane's slice of the B
//     operand of dQ^T += K^T dS^T (K^T operands from the transposing LDS read, as V^T in the
//     forward);
//   * bwd_dkv_heads: the transposed problem.  A workgroup owns 32 keys of one kv head and walks the 32-query tiles of the heads, a head to a wave:
//     S = Q K^T and dP = dO V^T leave 4 consecutive queries of one key in a lane for two 16-query tiles, exactly the B-operand slices
//     of dV^T += dO^T P and dK^T += Q^T dS, which accumulate over the tiles in registers and over the heads in LDS at the end.
// The accumulators of dP start at -D.  Probabilities and ds are rounded to the input type for their second products; everything else is
// fp32.  Both kernels keep a tile's mask in a branch of its own, with the products on both sides of it outside: as two versions of the
// whole tile the accumulators of the two met in copies, 32 and 64 registers of them a tile.
//
struct BwdMParams {
  const void* q; const void* k; const void* v; const void* o; const void* go;
  void* dq; void* dk; void* dv;
  const float* lse; int64_t lse_ld;            // (H, lse_ld): log2-domain log-sum-exp of a row
  float* dsum; int64_t ls;                      // (H, ls): -D = -(go . o)
  const int32_t* seg_start;                     // (ls,) first token of each token's sequence (entries >= N unused)
  const void* cu; int idx64, n_seg;
  int N, H, KH, G, window, n_wg;
  float scale, scale_log2;
};

template <int DT>
__device__ __forceinline__ float dot2w(uint32_t a, uint32_t b, float acc) {  // acc + a.lo b.lo + a.hi b.hi of two packed 16-bit pairs
  float a0, a1, b0, b1;
  if constexpr (DT == UVMI_BF16) {
    a0 = __uint_as_float(a << 16); a1 = __uint_as_float(a & 0xffff0000u); b0 = __uint_as_float(b << 16); b1 = __uint_as_float(b & 0xffff0000u);
  } else {
    a0 = half_bits_to_float((uint16_t)(a & 0xffff)); a1 = half_bits_to_float((uint16_t)(a >> 16));
    b0 = half_bits_to_float((uint16_t)(b & 0xffff)); b1 = half_bits_to_float((uint16_t)(b >> 16));
  }
  return fmaf(a1, b1, fmaf(a0, b0, acc));
}

// A staged tile of 32 rows of 128 bytes: row r keeps its 16-byte chunks xor-ed with r & 6.  Rows r and r + 1 share a 256-byte line of banks.  Both
// kinds of read are free of conflicts so: the transposing one takes 32 lanes on two neighbouring chunks of 8 rows at a time, that of rows
// 16 lanes, rows 0 .. 3 and 12 .. 15 of an even chunk with rows 4 .. 11 of the odd one beside it, or the other way about.  (With bit 3 of the row as
// the lowest one of the pattern the latter met: 4 cycles for each 16-byte read.)
__device__ __forceinline__ int tile_swizzle(int row) { return row & 6; }

// Operands of a staged tile.  Rows: [tile A dims 0..31, A dims 32..63, B dims 0..31, B dims 32..63], lane = row m, dims 8 g .. ;
// transposed: operand t is dim 16 t + m, slots 0..3 are rows 4 g + j of tile A, 4..7 of tile B.
struct TileReads {
  uint32_t row[2], col[4];
  __device__ __forceinline__ TileReads(int m, int g) {
#pragma unroll
    for (int s = 0; s < 2; s++) row[s] = (uint32_t)(m * 128 + (((4 * s + g) ^ tile_swizzle(m)) << 4));
    const int r = 4 * g + (m >> 2);   // the row that this lane names to the transposing read, 4 dims from 4 (m % 4)
#pragma unroll
    for (int t = 0; t < 4; t++) col[t] = (uint32_t)(r * 128 + (((2 * t + ((m & 3) >> 1)) ^ tile_swizzle(r)) << 4) + 8 * (m & 1));
  }
  __device__ __forceinline__ void rows(const unsigned char* s, pu4* a) const {
    a[0] = *(const pu4*)(s + row[0]);
    a[1] = *(const pu4*)(s + row[1]);
    a[2] = *(const pu4*)(s + 2048 + row[0]);
    a[3] = *(const pu4*)(s + 2048 + row[1]);
  }
  __device__ __forceinline__ pu4 cols(const unsigned char* s, int t) const {
    const pu2 a = ld_tr16(s + col[t]), b = ld_tr16(s + 2048 + col[t]);
    return pu4{a.x, a.y, b.x, b.y};
  }
};

template <int DT>
__device__ __forceinline__ void store_dims16(void* base, int64_t off, const pf4* acc, float mul) {  // acc[t][i] is dim 16 t + i from `off` on
  uint16_t* p = (uint16_t*)base + off;
#pragma unroll
  for (int t = 0; t < 4; t++)
    *(uint2*)(p + 16 * t) = uint2{pack2<DT>(acc[t][0] * mul, acc[t][1] * mul), pack2<DT>(acc[t][2] * mul, acc[t][3] * mul)};
}

// HB: heads of a wave.  Two for a group of five to eight, 164 registers and three waves per SIMD (at four, 128, 51 of them spill; a head to each of
// eight waves, 102 registers, reads the staged tiles twice as often and is no faster: 61 sequences of up to 1024 tokens, no window, dq and dk / dv,
// 149 us against 143); one for up to four, where two left two or three waves without a head.  What bounds it: issue (vector instructions 47 % and
// matrix ones 30 % of the cycles of a SIMD).  us, dq and dk / dv together, with a barrier for every tile -> for two: 64 x 64 .. 512 tokens 75.7 -> 73.8, 4 x
// 2048 106.2 -> 103.1, 61 x 16 .. 1024 145.8 -> 143.1 and with a window of 256 88.5 -> 86.3; 4 query heads, two kv heads, 10 x 300 19.9 -> 16.9, one, 20 x 700
// 55.6 -> 48.7.
template <int DT, int HB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HB == 1 ? 4 : 3))) void bwd_dq_mfma(BwdMParams P) {
  // one object per stage: the compiler can then tell that reads of one do not touch the one a load is filling
  __shared__ __attribute__((aligned(1024))) unsigned char s0[2][2][4096], s1[2][2][4096];  // [tile][K, V][32 keys x 128 B]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per = gridDim.x >> 3;
  const int bid = (blockIdx.x & 7) * per + (blockIdx.x >> 3);   // an XCD (ids congruent mod 8) gets a contiguous range
  if (bid >= P.n_wg) return;
  const int kvh = bid % P.KH, qb = bid / P.KH;
  const int m = lane & 15, g = lane >> 4;
  const int G = P.G;
  const float c = P.scale_log2;
  const int r0 = qb * 16, row = r0 + m;
  const int rowc = row < P.N ? row : P.N - 1;
  // ---- what depends on the row alone goes out first: Q^T, dO^T and O operands (lane = row m, dims 32 s + 8 g ..), the row's statistics
  pu4 Q[HB][2], GO[HB][2], Ov[HB][2];
  float lse2[HB];
  bool hok[HB];
  int lo_n = P.seg_start[rowc];
  int n_end = (int)load_index(P.cu, P.idx64, P.n_seg);   // tokens at or after it are padding
#pragma unroll
  for (int hh = 0; hh < HB; hh++) {
    const int hq = HB * wave + hh;
    hok[hh] = hq < G;
    const int head = kvh * G + (hok[hh] ? hq : G - 1);
    const int64_t base = ((int64_t)rowc * P.H + head) * 64 + 8 * g;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      Q[hh][s] = *(const pu4*)((const uint16_t*)P.q + base + 32 * s);
      GO[hh][s] = *(const pu4*)((const uint16_t*)P.go + base + 32 * s);
      Ov[hh][s] = *(const pu4*)((const uint16_t*)P.o + base + 32 * s);
    }
    lse2[hh] = P.lse[(int64_t)head * P.lse_ld + rowc];
  }
  __builtin_amdgcn_sched_barrier(0);
  n_end = n_end < 0 ? 0 : (n_end > P.N ? P.N : n_end);
  const bool row_ok = row < n_end;
  if (P.window > 0 && row - P.window + 1 > lo_n) lo_n = row - P.window + 1;
  if (!row_ok) lo_n = INT_MAX;
  // the block's key range: from its first live row's lower bound to its last live row (none: no tile)
  const int rl = min(r0 + 15, n_end - 1);
  const bool any = r0 < n_end;
  const int lo_first = __builtin_amdgcn_readfirstlane(lo_n);
  const int lo_last = __builtin_amdgcn_readfirstlane(__shfl(lo_n, any ? rl - r0 : 0, 64));
  const int kbeg = any ? lo_first & ~31 : 0, kend = any ? rl + 1 : 0;
  const int nk = __builtin_amdgcn_readfirstlane((kend - kbeg + 31) >> 5);
  const uint32_t n_keys = row_ok ? (uint32_t)(row - lo_n + 1) : 0u;   // the row sees keys lo_n .. lo_n + n_keys - 1 (none ahead of the first sequence)

  // ---- K / V tiles go from global memory straight into one of two LDS stages of two tiles, a stage ahead: wave w moves rows 8 w .. 8 w + 7
  const uint32_t rstride = (uint32_t)P.KH * 128;
  const int kv_bytes = (int)((uint32_t)P.N * rstride - (uint32_t)kvh * 128);
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint16_t*)P.k + (int64_t)kvh * 64), 0, kv_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rV = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint16_t*)P.v + (int64_t)kvh * 64), 0, kv_bytes, 0x00020000);
  const int lkey = 8 * wave + (lane >> 3);
  const uint32_t lch = (uint32_t)(((lane & 7) ^ tile_swizzle(lkey)) << 4);
  auto issue = [&](unsigned char (*S)[4096], int k) {   // (keys are clamped: a clamped key is masked)
    const uint32_t off = (uint32_t)min(kbeg + 32 * k + lkey, P.N - 1) * rstride + lch;
    load_lds16(rK, S[0] + 1024 * wave, off, 0);
    load_lds16(rV, S[1] + 1024 * wave, off, 0);
  };
  const bool odd = nk & 1;   // an odd count's first tile is a step of its own, ahead of the pairs, in the second stage
  if (odd) issue(s1[0], 0);
  if (nk > 1) issue(s0[0], odd), issue(s0[1], odd + 1);
  if (!odd && nk > 3) issue(s1[0], 2), issue(s1[1], 3);

  // ---- D = dO . O; -D is where the accumulators of dP^T start
  pf4 nD[HB], dQ[HB][4];
#pragma unroll
  for (int hh = 0; hh < HB; hh++) {
    float d = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) d = dot2w<DT>(GO[hh][1][i], Ov[hh][1][i], dot2w<DT>(GO[hh][0][i], Ov[hh][0][i], d));
    d = -psum32(psum16(d));
    nD[hh] = pf4{d, d, d, d};
    if (!row_ok) lse2[hh] = INFINITY;
#pragma unroll
    for (int t = 0; t < 4; t++) dQ[hh][t] = pf4{0.f, 0.f, 0.f, 0.f};
  }
  const TileReads at(m, g);
  auto step = [&](const unsigned char (*S)[4096], int tb) __attribute__((always_inline)) {
    pu4 KA[4], VA[4], KT[4];
    at.rows(S[0], KA);
    at.rows(S[1], VA);
#pragma unroll
    for (int t = 0; t < 4; t++) KT[t] = at.cols(S[0], t);
    float p[HB][8];
    pf4 dP[HB][2];
#pragma unroll
    for (int hh = 0; hh < HB; hh++) {
      pf4 sA = pf4{0.f, 0.f, 0.f, 0.f}, sB = sA, pA = nD[hh], pB = pA;
      sA = mfma16<DT>(KA[0], Q[hh][0], sA);
      sB = mfma16<DT>(KA[2], Q[hh][0], sB);
      pA = mfma16<DT>(VA[0], GO[hh][0], pA);
      pB = mfma16<DT>(VA[2], GO[hh][0], pB);
      sA = mfma16<DT>(KA[1], Q[hh][1], sA);
      sB = mfma16<DT>(KA[3], Q[hh][1], sB);
      dP[hh][0] = mfma16<DT>(VA[1], GO[hh][1], pA);
      dP[hh][1] = mfma16<DT>(VA[3], GO[hh][1], pB);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        p[hh][i] = __builtin_amdgcn_exp2f(fmaf(sA[i], c, -lse2[hh]));
        p[hh][4 + i] = __builtin_amdgcn_exp2f(fmaf(sB[i], c, -lse2[hh]));
      }
    }
    if (!(tb >= lo_last && tb + 31 <= r0)) {   // some row of the block does not see all keys of the tile
      const uint32_t kA = (uint32_t)(tb + 4 * g - lo_n);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const bool out = kA + (i & 3) + 16 * (i >> 2) >= n_keys;
#pragma unroll
        for (int hh = 0; hh < HB; hh++)
          if (out) p[hh][i] = 0.f;
      }
    }
#pragma unroll
    for (int hh = 0; hh < HB; hh++) {
      float ds[8];
#pragma unroll
      for (int i = 0; i < 8; i++) ds[i] = p[hh][i] * dP[hh][i >> 2][i & 3];
      const pu4 dsB = pu4{pack2<DT>(ds[0], ds[1]), pack2<DT>(ds[2], ds[3]), pack2<DT>(ds[4], ds[5]), pack2<DT>(ds[6], ds[7])};
#pragma unroll
      for (int t = 0; t < 4; t++) dQ[hh][t] = mfma16<DT>(KT[t], dsB, dQ[hh][t]);
    }
  };
  const bool work = hok[0];   // (wave-uniform: a wave without a head only helps with the loads)
  // a stage's tiles have landed (own loads: the wait; the other waves': the barrier) and every wave is done with the other stage
  auto landed = [&] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto full = [&](unsigned char (*S)[2][4096], unsigned char (*SN)[2][4096], int k) __attribute__((always_inline)) {   // tiles k and k + 1
    if (k == 0 && nk > 3) wait_vm<4>(); else wait_vm<0>();
    landed();
    if (k > 0 && k + 2 < nk) issue(SN[0], k + 2), issue(SN[1], k + 3);
    if (work) {
      step(S[0], kbeg + 32 * k);
      step(S[1], kbeg + 32 * k + 32);
    }
  };
  int k = 0;
  if (odd) {
    if (nk > 1) wait_vm<4>(); else wait_vm<0>();
    landed();
    if (work) step(s1[0], kbeg);
    k = 1;
  }
  for (; k + 4 <= nk; k += 4) {
    full(s0, s1, k);
    full(s1, s0, k + 2);
  }
  if (k < nk) full(s0, s1, k);
  // ---- dq = scale dQ; lane (row m, group g) holds head dims 16 t + 4 g + i (zeros for padding rows)
  if (row < P.N) {
#pragma unroll
    for (int hh = 0; hh < HB; hh++) {
      if (!hok[hh]) continue;
      const int head = kvh * G + HB * wave + hh;
      if (g == 0) P.dsum[(int64_t)head * P.ls + row] = row_ok ? nD[hh][0] : 0.f;
      store_dims16<DT>(P.dq, ((int64_t)row * P.H + head) * 64 + 4 * g, dQ[hh], P.scale);
    }
  }
}

// dk / dv.  A workgroup owns 32 keys of one kv head, and its NW waves are the heads of the group (GP: 1, 2, 4 or 8, the group padded; two
// passes over 8 heads with 4 waves) times strides of query tiles:
//   * a wave multiplies the Q and dO tiles of its own head, which nothing else in the workgroup reads, so it loads them straight into two LDS
//     stages of its own and waits for its own loads only: no barrier until the sums of the waves meet in LDS behind the loop.  A tile's
//     operands are all in registers before its products begin, so its stage is filled again, two tiles ahead, while they run;
//   * whatever the start needs is requested at once - the ends of the sequences (a lane each, up to 64 of them), the keys' own rows, the
//     first two tiles, which are made again or dropped where a head has fewer;
//   * the queries a key sees are an index range, key .. min(end of its sequence, key + window), found once per lane: the loop
//     reads no tables, and only the tiles at the ends of the range are masked.
// What bounds it: issue (vector instructions 41 % and matrix ones 33 % of the cycles of a SIMD, 70 % of them with some instruction; two waves per
// SIMD, for three it would have to hold 168 registers instead of 230), and for few keys the launch and its first trip, ~8 us.
// Before, four waves - two groups of 32 keys, two heads of a pair - shared the tiles behind a barrier per pair of heads and a workgroup
// of 64 keys walked its queries four times: 1.3 us a step, so a launch lasted as long as its longest row of steps.  us: 2 sequences of up to 778
// tokens 64.7 -> 25.1; 12 of up to 80 20.3 -> 10.6; 39 of up to 933 105 -> 56; 61 of up to 1024, window 256, 55.3 -> 52.6.
template <int DT, int GP, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_dkv_heads(BwdMParams P) {
  struct Stage { unsigned char q[4096], g[4096]; float lse[64], nd[64]; };   // 32 rows of 128 B of Q and dO; statistics of 32 (64 loaded)
  __shared__ __attribute__((aligned(1024))) Stage s0[NW], s1[NW];            // (an object per stage: the compiler can then tell that reads of one do not touch the one a load is filling)
  constexpr int LOADS = 10;                                                  // of a tile
  constexpr int HP = GP < NW ? GP : NW, TS = NW / HP;                        // heads at a time, tile strides
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per = gridDim.x >> 3;
  const int bid = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (bid >= P.n_wg) return;
  const int kvh = bid % P.KH, kb = bid / P.KH;
  const int n = lane & 15, g = lane >> 4;
  const int hq = wave % HP, t0 = wave / HP, G = P.G;
  const float c = P.scale_log2;
  const int jw = kb * 32, key0 = jw + n;
  // ---- requested together: the ends of the sequences (lane s: of sequence s, where there are at most 64), K^T / V^T operands, the first two tiles
  const bool few = P.n_seg <= 64;
  const int end_l = few ? (int)load_index(P.cu, P.idx64, min(lane + 1, P.n_seg)) : 0;
  int n_end = (int)load_index(P.cu, P.idx64, P.n_seg);
  const int n_beg = (int)load_index(P.cu, P.idx64, 0);
  pu4 Kb[2][2], Vb[2][2];
#pragma unroll
  for (int b = 0; b < 2; b++) {
    const int64_t base = ((int64_t)min(key0 + 16 * b, P.N - 1) * P.KH + kvh) * 64 + 8 * g;
    Kb[b][0] = *(const pu4*)((const uint16_t*)P.k + base);
    Kb[b][1] = *(const pu4*)((const uint16_t*)P.k + base + 32);
    Vb[b][0] = *(const pu4*)((const uint16_t*)P.v + base);
    Vb[b][1] = *(const pu4*)((const uint16_t*)P.v + base + 32);
  }
  // loader: tile t of the wave is rows jw + 32 (t0 + TS t) ..
  const uint32_t rstride = (uint32_t)P.H * 128;
  const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc((void*)P.q, 0, (int)((uint32_t)P.N * rstride), 0x00020000);
  const __amdgpu_buffer_rsrc_t rG = __builtin_amdgcn_make_buffer_rsrc((void*)P.go, 0, (int)((uint32_t)P.N * rstride), 0x00020000);
  const __amdgpu_buffer_rsrc_t rL = __builtin_amdgcn_make_buffer_rsrc((void*)P.lse, 0, (int)((P.lse_ld * (P.H - 1) + P.N + 32) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rD = __builtin_amdgcn_make_buffer_rsrc((void*)P.dsum, 0, (int)((P.ls * (P.H - 1) + P.N + 32) * 4), 0x00020000);
  uint32_t l_off[4];
  const uint32_t l_st = (uint32_t)(jw + 32 * t0 + (lane & 31)) * 4;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = 8 * i + (lane >> 3);
    l_off[i] = (uint32_t)(jw + 32 * t0 + r) * rstride + (uint32_t)(((lane & 7) ^ tile_swizzle(r)) << 4);
  }
  int f_t = 0, f_h = kvh * G + min(hq, G - 1);   // tile and head of the next request
  auto issue = [&](Stage* S) {                   // (rows past the last token come out as zeros: the descriptors' bounds)
    const uint32_t row = (uint32_t)(32 * TS * f_t), at = row * rstride + (uint32_t)f_h * 128;
#pragma unroll
    for (int i = 0; i < 4; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rQ, (__attribute__((address_space(3))) void*)(S[wave].q + 1024 * i), 16, l_off[i] + at, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rG, (__attribute__((address_space(3))) void*)(S[wave].g + 1024 * i), 16, l_off[i] + at, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rL, (__attribute__((address_space(3))) void*)S[wave].lse, 4, l_st + (row + (uint32_t)(f_h * P.lse_ld)) * 4, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rD, (__attribute__((address_space(3))) void*)S[wave].nd, 4, l_st + (row + (uint32_t)(f_h * P.ls)) * 4, 0, 0, 0);
  };
  if (hq < G) {   // (whether the keys are seen by these tiles is not known yet: the ends are on their way)
    issue(s0);
    f_t = 1;
    issue(s1);
  }
  // ---- the queries that see a key: n_q from the key on
  n_end = n_end < 0 ? 0 : (n_end > P.N ? P.N : n_end);
  int first_end = 0, qend = 0;
  uint32_t n_q[2] = {0, 0};
  if (jw < n_end) {
    const int j_last = min(jw + 31, n_end - 1);
    auto seq_of = [&](int j) {   // the last sequence s with cu[s] <= j
      if (few) return (int)__popcll(__ballot(lane + 1 < P.n_seg && end_l <= j));
      int lo = 0, hi = P.n_seg;
      while (hi - lo > 1) {      // 64 probes at a time
        const int step = (hi - lo + 63) >> 6, at = lo + (lane + 1) * step;
        const bool below = at < hi && load_index(P.cu, P.idx64, at) <= j;
        lo += __popcll(__ballot(below)) * step;
        hi = min(hi, lo + step);
      }
      return lo;
    };
    auto end_of = [&](int s) { return few ? __builtin_amdgcn_readlane(end_l, s) : (int)load_index(P.cu, P.idx64, s + 1); };
    const int sf = __builtin_amdgcn_readfirstlane(seq_of(jw)), sl = __builtin_amdgcn_readfirstlane(seq_of(j_last));
    qend = min(end_of(sl), n_end);
    int hi_q[2] = {qend, qend};
    for (int s = sl - 1; s >= sf; s--) {
      const int e = end_of(s);
#pragma unroll
      for (int b = 0; b < 2; b++)
        if (key0 + 16 * b < e) hi_q[b] = e;
    }
    first_end = __builtin_amdgcn_readfirstlane(hi_q[0]);
    if (P.window > 0) qend = min(qend, j_last + P.window);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (P.window > 0) hi_q[b] = min(hi_q[b], key0 + 16 * b + P.window);
      if (key0 + 16 * b < n_end && key0 + 16 * b >= n_beg) n_q[b] = (uint32_t)(hi_q[b] - key0 - 16 * b);
    }
  }
  // no mask in a query tile that starts in full_from .. full_to: every query follows every key, in the first key's sequence and window (nowhere
  // for first keys that lie ahead of the first sequence)
  const int full_from = jw + 31, full_to = jw < n_beg ? -1 : (P.window > 0 ? min(first_end, jw + P.window) : first_end) - 32;
  const int nt = qend > jw ? (qend - jw + 31) >> 5 : 0;                                            // query tiles that see some key,
  const int mine = __builtin_amdgcn_readfirstlane(nt > t0 ? (nt - t0 + TS - 1) / TS : 0);          // this wave's of them
  const int total = mine * __builtin_amdgcn_readfirstlane(hq < G ? (G - hq + HP - 1) / HP : 0);    // and for all its heads
  // (the second request was tile 1 of the first head; where there is no such tile it is made again)
  bool again = false;
  if (total > 1 && mine == 1) { f_t = 0; f_h += HP; again = true; }
  auto advance = [&]() {
    if (++f_t == mine) { f_t = 0; f_h += HP; }
  };
  if (again) {
    __builtin_amdgcn_s_waitcnt(0x0f70);   // (the one that it replaces has landed)
    issue(s1);
  }
  pf4 dK[2][4], dV[2][4];
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int t = 0; t < 4; t++) dK[b][t] = dV[b][t] = pf4{0.f, 0.f, 0.f, 0.f};
  const TileReads at(n, g);
  int c_t = 0;   // tile of the next arithmetic
  auto step = [&](Stage* SS, int i) __attribute__((always_inline)) {
    const int tq = jw + 32 * (t0 + TS * c_t);
    if (++c_t == mine) c_t = 0;
    if (i + 1 < total) __builtin_amdgcn_s_waitcnt(0x0f70 | LOADS); else __builtin_amdgcn_s_waitcnt(0x0f70);   // (the next tile's may be on their way)
    asm volatile("" ::: "memory");
    const Stage& S = SS[wave];
    pu4 QA[4], GA[4], TG[4], TQ[4];
    at.rows(S.q, QA);
    at.rows(S.g, GA);
    // statistics of this lane's queries tq + 4g + j (tile A) and tq + 16 + 4g + j (tile B)
    const pf4 lA = *(const pf4*)(S.lse + 4 * g), lB = *(const pf4*)(S.lse + 16 + 4 * g);
    const pf4 dA = *(const pf4*)(S.nd + 4 * g), dB = *(const pf4*)(S.nd + 16 + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; t++) TG[t] = at.cols(S.g, t);
#pragma unroll
    for (int t = 0; t < 4; t++) TQ[t] = at.cols(S.q, t);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (i + 2 < total) { advance(); issue(SS); }
    float p[2][8], ds[2][8];
#pragma unroll
    for (int b = 0; b < 2; b++) {
      pf4 sA = pf4{0.f, 0.f, 0.f, 0.f}, sB = sA, pA = dA, pB = dB;   // (dP starts at -D)
      sA = mfma16<DT>(QA[0], Kb[b][0], sA);
      sB = mfma16<DT>(QA[2], Kb[b][0], sB);
      pA = mfma16<DT>(GA[0], Vb[b][0], pA);
      pB = mfma16<DT>(GA[2], Vb[b][0], pB);
      sA = mfma16<DT>(QA[1], Kb[b][1], sA);
      sB = mfma16<DT>(QA[3], Kb[b][1], sB);
      pA = mfma16<DT>(GA[1], Vb[b][1], pA);
      pB = mfma16<DT>(GA[3], Vb[b][1], pB);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        p[b][j] = __builtin_amdgcn_exp2f(fmaf(sA[j], c, -lA[j]));
        p[b][4 + j] = __builtin_amdgcn_exp2f(fmaf(sB[j], c, -lB[j]));
        ds[b][j] = p[b][j] * pA[j];
        ds[b][4 + j] = p[b][4 + j] * pB[j];
      }
    }
    if (tq < full_from || tq > full_to) {
      // (selects, not products: the statistics of a query past the last token are whatever the workspace held)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const uint32_t from = (uint32_t)(tq + 4 * g - key0 - 16 * b);
#pragma unroll
        for (int j = 0; j < 8; j++)
          if (from + (j & 3) + 16 * (j >> 2) >= n_q[b]) { p[b][j] = 0.f; ds[b][j] = 0.f; }
      }
    }
    pu4 PB[2], SB[2];
#pragma unroll
    for (int b = 0; b < 2; b++) {
      PB[b] = pu4{pack2<DT>(p[b][0], p[b][1]), pack2<DT>(p[b][2], p[b][3]), pack2<DT>(p[b][4], p[b][5]), pack2<DT>(p[b][6], p[b][7])};
      SB[b] = pu4{pack2<DT>(ds[b][0], ds[b][1]), pack2<DT>(ds[b][2], ds[b][3]), pack2<DT>(ds[b][4], ds[b][5]), pack2<DT>(ds[b][6], ds[b][7])};
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int b = 0; b < 2; b++) dV[b][t] = mfma16<DT>(TG[t], PB[b], dV[b][t]);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
#pragma unroll
      for (int b = 0; b < 2; b++) dK[b][t] = mfma16<DT>(TQ[t], SB[b], dK[b][t]);
    }
  };
  for (int i = 0; i < total; i += 2) {
    step(s0, i);
    if (i + 1 < total) step(s1, i + 1);
  }
  // ---- the waves' sums meet in LDS, [register][lane], 16 KB a wave: wave w finishes registers 64 / NW w .. (dk: 0 .. 31, 16 of a key block)
  __builtin_amdgcn_s_waitcnt(0x0f70);   // (requests without a tile)
  __syncthreads();                      // (every wave has read its last tile)
  auto part = [&](int w) { return (float*)(w < NW / 2 ? (unsigned char*)s0 : (unsigned char*)s1) + (w & (NW / 2 - 1)) * 4096 + lane; };
  {
    float* o = part(wave);
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          o[((b * 4 + t) * 4 + j) * 64] = dK[b][t][j];
          o[(32 + (b * 4 + t) * 4 + j) * 64] = dV[b][t][j];
        }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 16 / NW; u++) {
    const int r = 64 / NW * wave + 4 * u, key = key0 + (r & 16);
    const bool is_v = r >= 32;
    float acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      float v = part(0)[(r + j) * 64];
#pragma unroll
      for (int w = 1; w < NW; w++) v += part(w)[(r + j) * 64];
      acc[j] = is_v ? v : v * P.scale;
    }
    if (key < P.N)   // (zeros for padding tokens)
      *(uint2*)((uint16_t*)(is_v ? P.dv : P.dk) + ((int64_t)key * P.KH + kvh) * 64 + 4 * (r & 12) + 4 * g) =
          uint2{pack2<DT>(acc[0], acc[1]), pack2<DT>(acc[2], acc[3])};
  }
}

}  // namespace uvmi

using namespace uvmi;

static int64_t bwd_row_stride(int N) { return (((int64_t)(N > 0 ? N : 0) + 31) & ~31LL) + 32; }   // statistics rows, padded for whole-tile reads

extern "C" size_t uvmi_prefill_attn_bwd_workspace_bytes(int N, int H) {
  const size_t ls = (size_t)bwd_row_stride(N);
  return ((size_t)2 * (size_t)(H > 0 ? H : 0) * ls + 2 * ls) * 4 + 256;   // lse, D (H, ls); segment table, scratch (ls)
}

// Whether dk / dv takes eight waves a workgroup rather than four: a wave for each of 8 heads, or twice the strides of query tiles, so the row of tiles
// of the keys that the most queries see, which a launch lasts as long as, is half as long.  Its waves have to have tiles: `keys` is the mean
// sequence, cut to the window.  us, dq and dk / dv, four / eight, workgroups with compute units of their own: 8 heads 2500 tokens in sequences of
// 16 14.3 / 15.1, of 40 15.2 / 15.5, of 100 19.2 / 18.4, of 250 34.5 / 30.0; 4 heads of 100 13.3 / 13.9, of 250 21.9 / 20.3; 2 heads of 250 14.8 / 15.3, of 700
// 27.7 / 25.8, 4096 tokens with a window of 256 13.2 / 13.9; one head 1500 tokens 26.4 / 25.8, with a window 11.7 / 12.6.  Eight waves leave a unit one
// workgroup: up to two rounds of them pay where sequences are long and no window shortens them (8 heads 16 of 1024 99.8 / 83.2, 24 of up to 1024 95.0 / 79.3, 3 of
// 4096 286 / 294, 30 of 512 58.1 / 61.3; 4 heads 57.8 / 50.4, 56.4 / 50.5, 158 / 163, 37.6 / 41.5; 2 heads 37.7 / 36.6, one 28.8 / 30.3), with short ones they do not
// (8 heads 20 000 tokens in sequences of 16 38.8 / 45.6, of 100 45.8 / 53.7; 10 000 of 40 26.3 / 31.4), nor with a window (24 of up to 1024 68.2 / 70.9) or a third round
// (10 of 2048 210 / 218; 39 of up to 933 95.0 / 93.4 is the exception).
static bool dkv_wide(int G, int64_t n_wg, int64_t mean, int window, int cus) {
  const int64_t keys = window > 0 && window < mean ? window : mean, least = G > 4 ? 64 : (G > 2 ? 160 : (G > 1 ? 640 : 1280));
  if (n_wg <= cus) return keys >= least;
  return window == 0 && G > 1 && n_wg <= 2 * (int64_t)cus && keys >= (least > 400 ? least : 400);
}

extern "C" int uvmi_prefill_attn_bwd(const uvmi_prefill_attn_bwd_args* a, void* stream) {
  UVMI_REQUIRE(a, UVMI_EINVAL, "uvmi_prefill_attn_bwd: null arguments");
  UVMI_REQUIRE(a->N >= 0 && a->H > 0 && a->KH > 0 && a->H % a->KH == 0 && a->n_seg >= 0, UVMI_EINVAL, "uvmi_prefill_attn_bwd: bad sizes");
  UVMI_REQUIRE(a->hd == 64, UVMI_EUNSUPPORTED, "uvmi_prefill_attn_bwd: head_dim %d (only 64)", a->hd);
  UVMI_REQUIRE(a->dtype == UVMI_F16 || a->dtype == UVMI_BF16, UVMI_EUNSUPPORTED, "uvmi_prefill_attn_bwd: q / k / v / o / go must be fp16 or bf16");
  UVMI_REQUIRE(a->idx_dtype == UVMI_I32 || a->idx_dtype == UVMI_I64, UVMI_EINVAL, "uvmi_prefill_attn_bwd: cu_seqlens must be int32 or int64");
  UVMI_REQUIRE(a->window >= 0 && a->N < (1 << 30), UVMI_EINVAL, "uvmi_prefill_attn_bwd: bad window / N");
  if (a->N == 0) return UVMI_OK;
  UVMI_REQUIRE(a->q && a->k && a->v && a->o && a->go && a->dq && a->dk && a->dv && a->cu_seqlens, UVMI_EINVAL, "uvmi_prefill_attn_bwd: null pointer");
  const void* ptrs[] = {a->q, a->k, a->v, a->o, a->go, a->dq, a->dk, a->dv};
  for (const void* p : ptrs) UVMI_REQUIRE(((uintptr_t)p % 16) == 0, UVMI_EINVAL, "uvmi_prefill_attn_bwd: tensors must be 16-byte aligned");
  UVMI_REQUIRE(a->workspace && ((uintptr_t)a->workspace % 16) == 0 && a->workspace_bytes >= uvmi_prefill_attn_bwd_workspace_bytes(a->N, a->H),
               UVMI_EWORKSPACE, "uvmi_prefill_attn_bwd: workspace of %zu bytes needed", uvmi_prefill_attn_bwd_workspace_bytes(a->N, a->H));
  const int window = a->window < a->N ? a->window : 0;   // (a window of all tokens hides none; the kernels add it to an index)
  hipStream_t st = (hipStream_t)stream;
  const int64_t ls = bwd_row_stride(a->N);
  float* lse = (float*)a->workspace;
  float* dsum = lse + (size_t)a->H * ls;
  int32_t* seg = (int32_t*)(dsum + (size_t)a->H * ls);
  int32_t* pidx = seg + ls;
  const int G = a->H / a->KH;
  if (G <= 8 && (int64_t)a->N * a->H * 64 < (1LL << 30)) {
    // the MFMA form: statistics from a forward pass without output, then dq and dk / dv
    uvmi_prefill_attn_args f = {};
    f.q = a->q; f.q_dtype = a->dtype; f.sqn = (int64_t)a->H * 64; f.sqh = 64;
    f.k = a->k; f.v = a->v; f.kv_dtype = a->dtype; f.skn = f.svn = (int64_t)a->KH * 64; f.skh = f.svh = 64;
    f.cu_seqlens = a->cu_seqlens; f.idx_dtype = a->idx_dtype; f.n_seg = a->n_seg;
    f.N = a->N; f.H = a->H; f.KH = a->KH; f.hd = a->hd; f.scale = a->scale; f.window = window;
    UVMI_REQUIRE(a->scale > 0.f, UVMI_EUNSUPPORTED, "uvmi_prefill_attn_bwd: scale must be positive");
    const float* stats = lse;
    int64_t stats_ld = ls;
    const int32_t* seg_start = seg;
    if (a->lse) {   // the forward kept them: no pass of its own (43 us of 290 for forward and backward of 31 700 tokens)
      UVMI_REQUIRE(a->fwd_workspace && ((uintptr_t)a->lse % 16) == 0 && a->lse_stride >= a->N + 32 && a->lse_stride % 4 == 0, UVMI_EINVAL,
                   "uvmi_prefill_attn_bwd: lse must be 16-byte aligned with a pitch of at least N + 32 that is a multiple of 4, beside fwd_workspace");
    }
    // (bwd_dkv_heads reaches the statistics by 32-bit offsets: those of a wider pitch are formed again)
    if (a->lse && a->lse_stride < (1LL << 29) / a->H) {
      stats = a->lse;
      stats_ld = a->lse_stride;
      seg_start = (const int32_t*)a->fwd_workspace;
    } else {
      int rc = prefill_attn_stats(&f, seg, pidx, lse, ls, stream);
      if (rc) return rc;
    }
    BwdMParams M;
    M.q = a->q; M.k = a->k; M.v = a->v; M.o = a->o; M.go = a->go; M.dq = a->dq; M.dk = a->dk; M.dv = a->dv;
    M.lse = stats; M.lse_ld = stats_ld; M.dsum = dsum; M.ls = ls; M.seg_start = seg_start;
    M.cu = a->cu_seqlens; M.idx64 = a->idx_dtype == UVMI_I64 ? 1 : 0; M.n_seg = a->n_seg;
    M.N = a->N; M.H = a->H; M.KH = a->KH; M.G = G; M.window = window;
    M.scale = a->scale; M.scale_log2 = a->scale * 1.4426950408889634f;
    M.n_wg = ((a->N + 15) / 16) * a->KH;
    const dim3 gq((unsigned)((M.n_wg + 7) / 8 * 8));
#define UVMI_DQ(DT)                                                                                    \
  do {                                                                                                 \
    if (M.G > 4) hipLaunchKernelGGL((bwd_dq_mfma<DT, 2>), gq, dim3(256), 0, st, M);                    \
    else hipLaunchKernelGGL((bwd_dq_mfma<DT, 1>), gq, dim3(256), 0, st, M);                            \
  } while (0)
    if (a->dtype == UVMI_F16) UVMI_DQ(UVMI_F16); else UVMI_DQ(UVMI_BF16);
#undef UVMI_DQ
    UVMI_CHECK_LAUNCH("uvmi_prefill_attn_bwd(dq)");
    int cus = uvmi_device_cus();
    if (cus <= 0) cus = 256;
    M.n_wg = ((a->N + 31) / 32) * a->KH;
    const bool wide = dkv_wide(G, M.n_wg, a->n_seg > 0 ? a->N / a->n_seg : a->N, window, cus);
    const dim3 gk((unsigned)((M.n_wg + 7) / 8 * 8));
#define UVMI_DKV_W(DT, GP)                                                                   \
  do {                                                                                       \
    if (wide) hipLaunchKernelGGL((bwd_dkv_heads<DT, GP, 8>), gk, dim3(512), 0, st, M);       \
    else hipLaunchKernelGGL((bwd_dkv_heads<DT, GP, 4>), gk, dim3(256), 0, st, M);            \
  } while (0)
#define UVMI_DKV(DT) do { if (G > 4) UVMI_DKV_W(DT, 8); else if (G > 2) UVMI_DKV_W(DT, 4); else if (G > 1) UVMI_DKV_W(DT, 2); else UVMI_DKV_W(DT, 1); } while (0)
    if (a->dtype == UVMI_F16) UVMI_DKV(UVMI_F16); else UVMI_DKV(UVMI_BF16);
#undef UVMI_DKV
#undef UVMI_DKV_W
    UVMI_CHECK_LAUNCH("uvmi_prefill_attn_bwd(dkv)");
    return UVMI_OK;
  }
  // more than 8 query heads per kv head: the plain kernels
  BwdParams P;
  P.q = a->q; P.k = a->k; P.v = a->v; P.o = a->o; P.go = a->go; P.dq = a->dq; P.dk = a->dk; P.dv = a->dv;
  P.lse = lse;
  P.dsum = P.lse + (size_t)a->N * a->H;
  P.cu = a->cu_seqlens; P.idx64 = a->idx_dtype == UVMI_I64 ? 1 : 0; P.n_seg = a->n_seg; P.N = a->N; P.H = a->H; P.KH = a->KH; P.G = a->H / a->KH;
  P.window = window; P.scale = a->scale;
  const dim3 blk(64), g1((unsigned)((a->N + 63) / 64), (unsigned)a->H), g2((unsigned)((a->N + 31) / 32), (unsigned)a->KH);
  if (a->dtype == UVMI_F16) hipLaunchKernelGGL((bwd_dq_kernel<UVMI_F16>), g1, blk, 0, st, P);
  else hipLaunchKernelGGL((bwd_dq_kernel<UVMI_BF16>), g1, blk, 0, st, P);
  UVMI_CHECK_LAUNCH("uvmi_prefill_attn_bwd(dq)");
  if (a->dtype == UVMI_F16) hipLaunchKernelGGL((bwd_dkv_kernel<UVMI_F16>), g2, blk, 0, st, P);
  else hipLaunchKernelGGL((bwd_dkv_kernel<UVMI_BF16>), g2, blk, 0, st, P);
  UVMI_CHECK_LAUNCH("uvmi_prefill_attn_bwd(dkv)");
  return UVMI_OK;
}
