// Packed causal self-attention with an optional sliding window over unquantized K/V: the attention of a packed prefill.
//
// Contract (ultraviolet/kernels/varlen_attn.py:87-115 of the reference): q (N, H, hd), k / v (N, KH, hd) hold the
// tokens of several sequences back to back, cu_seqlens their boundaries; query i sees keys j of its own sequence with
// i - window < j <= i.
//
// prefill_attn_mfma_hd64 (head_dim 64, 16-bit q/k/v of one dtype, up to 8 query heads per kv head):
//   * a wave owns 16 consecutive packed tokens x 2 query heads of one kv head, and walks the keys in 32-key
//     super-tiles, two of them a step where the four waves share a block (below).  Query blocks are aligned to the packed index, not to the sequences: a block that straddles a
//     boundary walks the union of its rows' key ranges and masks per (row, key), so the grid is ceil(N / 16) blocks
//     with no search for "which sequence is block i in";
//   * S^T = K . Q^T with v_mfma_f32_16x16x32 (A = 16 keys x 32 dims, B = 32 dims x 16 rows): a lane of the accumulator
//     holds 4 consecutive keys of one query row, for two 16-key tiles A and B.  Exactly these 8 values, rounded to
//     the 16-bit input type, are the lane's slice of the B operand of O^T = V^T . P^T when contraction slot 8g+j is
//     key 4g+j of tile A (j < 4) or of tile B (j >= 4): probabilities never move between lanes;
//   * V^T operands come out of LDS through the transposing read (ds_read_b64_tr_b16), once per super-tile for the wave's heads, as
//     do the K operands (16-byte reads, lane = key m, dims 8g..8g+7 of each half);
//   * the 4 waves of a workgroup are the 4 head pairs of a query block (2 blocks x 2 pairs for up to 4 query heads per kv head, 4
//     blocks for up to 2) of one kv head and walk the same keys, so a super-tile of K and V is fetched once per workgroup, from
//     global memory straight into one of two LDS stages of two tiles, a stage ahead; one barrier per stage, an odd count's first tile ahead of
//     the pairs (behind them, the accumulators of two step forms met in copies: 33 registers of the single form's spilled).  Where the
//     waves are of different blocks, a wave skips the tiles outside its own block's key range;
//   * a step of two tiles (PAIR) takes one maximum, one exponential and one rescale of the accumulators for 64 keys: of ~65 vector instructions a head and
//     tile 33 are a step's, not a key's.  It holds 158 registers, three waves per SIMD (at four, 128, 45 of them spill and everything
//     takes twice as long); single tiles at four waves in the same loop, both behind a launch for the segment table: 64 x 512 tokens 45.1 us
//     against 41.9, window 256 35.7 / 34.8;
//   * online softmax per (row, head) in the exp2 domain; tiles that every row of the block sees completely skip the
//     mask arithmetic: one branch per tile, around the mask alone (two versions of the whole tile would meet in copies of the accumulators);
//   * workgroup ids are remapped so that each XCD (one L2 each) owns a contiguous range of query blocks and therefore
//     whole sequences, the last blocks first: they see the most keys.
// What bounds it: vector instructions, at three waves per SIMD.  us of calls in a graph, one tile a step (118 registers, four waves) behind a launch
// for the segment table -> now, two tiles and the rows' sequences found here (up to 64 of them): 93 tokens 6.4 -> 5.0; 400 11.7 -> 9.1; 64 x 64 .. 512
// tokens 30.2 -> 25.2, window 256 24.7 -> 22.1; 64 x 512 42.4 -> 38.4 and 35.5 -> 31.8; 4 x 2048 45.3 -> 38.3; 61 x 16 .. 1024 58.9 -> 50.8, window 256 38.3 ->
// 33.5; 10 x 300 on 4 query and 2 kv heads 11.5 -> 9.9.  Groups of up to 4 query heads per kv head, table at hand, take single tiles from the same stages: 2 - 8 %
// faster (8 and 2 heads 1 x 4096 71.2 -> 66.2, 61 x 16 .. 1024 55.8 -> 55.1) but for equal long sequences whose workgroups come to between one and two a compute
// unit (2 x 4096 90.3 -> 94.7, 4 x 2048 43.5 -> 45.4); three stages of one tile are no faster there in this kernel (91.7) and slower elsewhere (1 x 4096 71.6).
//
// Everything else (fp32 K/V, other head dims) goes token by token through the decode kernel's generic path with the
// packed K/V as a batch-stride-0 "cache".
#include "common.h"
#include "attn_mfma_util.h"
#include "gemm_util.h"

#include <climits>
#include <type_traits>

namespace uvmi {

struct PrefillParams {
  const void* q; const void* k; const void* v; void* out;
  const int32_t* seg_start;  // (N,) packed index of the first token of each token's sequence
  // or found here, of at most 64 sequences: cu_seqlens (n_seg of them; null: seg_start holds the table), and where the table goes
  const void* cu; int idx64, n_seg; int32_t* seg_out; int32_t* pidx_out;
  int64_t sqn, sqh, skn, skh, svn, svh, son, soh;
  int N, H, KH, G, window, n_hg;   // n_hg: waves that share a query block of a kv head, HPW query heads each: 1, 2 or 4
  int n_wg;                        // workgroups with work: ceil(query blocks / (4 / n_hg)) * KH
  float scale_log2;
  const float* post_vhat; const float* post_gate; const float* post_xsa;  // fused Attention.post epilogue when post_vhat != null
  float* lse_out; int64_t lse_stride;  // optional (H, lse_stride) fp32: log2 of each row's sum of exp2(scale_log2 s) (the backward's statistics)
  // the output projection and residual update of the rows in the same launch (OP): y = o_ca r + o_cb (attention W^T), o_n columns
  const void* o_w; const void* o_r; void* o_out;
  int64_t o_ldw, o_ldr, o_ldo;
  int o_n;
  float o_ca, o_cb;
};

// seg_start[i] = cu[s] for the last s with cu[s] <= i (empty sequences are skipped); pidx[i] = i.
__global__ __launch_bounds__(256) void prefill_segments(const void* cu, int idx64, int n_seg, int N, int32_t* seg_start, int32_t* pidx) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  int lo = 0, hi = n_seg;  // invariant: cu[lo] <= i, and hi == n_seg or cu[hi] > i
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (load_index(cu, idx64, mid) <= i) lo = mid; else hi = mid;
  }
  const int first = (int)load_index(cu, idx64, lo);
  seg_start[i] = first <= i ? first : i + 1;   // (ahead of the first sequence: behind the token itself, so that it sees no key)
  pidx[i] = i;
}

constexpr int HPW = 2;  // query heads per wave

// The table's entry for token i, of at most 64 sequences; lane s has the start of sequence s.
__device__ __forceinline__ int first_token(int start, int n_seg, int i) {
  int lo = 0, hi = n_seg;
#pragma unroll
  for (int k = 0; k < 6; k++) {   // (as above)
    const int mid = (lo + hi) >> 1, c = __shfl(start, mid, 64);
    const bool le = c <= i;
    if (hi - lo > 1) { lo = le ? mid : lo; hi = le ? hi : mid; }
  }
  const int first = __shfl(start, lo, 64);
  return first <= i ? first : i + 1;
}

// maximum over lanes l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ float xmaximum(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __builtin_elementwise_maximum(__uint_as_float(r[0]), __uint_as_float(r[1]));
  auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __builtin_elementwise_maximum(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float max3(float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); }

// OP: blockIdx.y is a part of 64 OP columns of the output projection.  Every part's workgroup computes the block's attention for itself (8 heads on 1
// kv head: a wave has two of them, a workgroup all) while its rows of the weight go straight into LDS behind the first two tiles; the
// heads' outputs meet in LDS, and a wave forms 16 OP columns of the block's 16 rows from them.  For passes whose blocks leave most of
// the device idle: what is repeated takes no time, and a launch of the projection alone lasts 3.4 us at 93 rows, nearly all of it its start
// and a trip for the weights.  A whole prefill, us: 30 tokens 267 -> 245, 93 296 -> 274, 300 347 -> 323 (64 columns a part: up to 384 tokens),
// 500 400 -> 377, 700 444 -> 422 (128: up to 768; 780 tokens, where an XCD has more workgroups than compute units, 469 -> 479).
//
// PAIR: the waves of a workgroup share one query block (n_hg = 4), and a step takes both tiles of a stage.
template <int DT, int ODT, int OP, bool PAIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(OP ? 1 : (PAIR ? 3 : 4)))) void prefill_attn_mfma_hd64(PrefillParams P) {
  // one object per stage: the compiler can then tell that reads of one do not touch the one a load is filling
  __shared__ __attribute__((aligned(1024))) unsigned char s0[2][2][4096], s1[2][2][4096];  // [tile][K, V][32 keys x 128 B]
  constexpr int OW = 16 * OP;   // weight rows of a wave, a load each
  __shared__ __attribute__((aligned(1024))) unsigned char sw[OP ? 4 * OW * 1024 : 16];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // gridDim.x is a multiple of 8; ids congruent mod 8 run on one XCD and get a contiguous range of work
  const int per = gridDim.x >> 3;
  // from its end: a sequence's last blocks, which see the most keys, start first
  const int bid = (blockIdx.x & 7) * per + per - 1 - (blockIdx.x >> 3);
  if (bid >= P.n_wg) return;   // (the whole workgroup: no barrier is left waiting)
  const int kvh = bid % P.KH;
  const int qg = bid / P.KH;               // group of 4 / n_hg consecutive query blocks
  const int hsh = P.n_hg >> 1;             // n_hg is 1, 2 or 4
  const int qbw = 4 >> hsh;
  const int hg = wave & (P.n_hg - 1);
  const int qb = qg * qbw + (wave >> hsh);
  const int m = lane & 15, g = lane >> 4;
  const int G = P.G;
  const float c = P.scale_log2;

  // ---- this lane's query row (accumulator column m); a wave whose block starts past the last token (the tail of the last
  // group) has an empty key range and only helps with the loads
  const int r0 = qb * 16;
  const bool wave_ok = r0 < P.N;
  const int row = r0 + m;
  const bool row_ok = row < P.N;
  const int rowc = row_ok ? row : P.N - 1;
  const int row0 = qg * qbw * 16;          // < N
  // ---- what depends on the row alone goes out first: Q^T operands (lane (row m, group g) holds q[row][head][32 s + 8 g .. + 8] for
  // s = 0, 1; absent heads read the last one and are not stored), the row's segment, the epilogue's gates
  // (of at most 64 sequences a lane takes the start of one, and the row's is found between the lanes: the launch of a table in front goes away: us 93
  // tokens 6.6 -> 5.3, 400 10.9 -> 9.4, 61 x 16 .. 1024 with a window 37.2 -> 35.9; the table is written for the launches that read it)
  const bool find = P.cu != nullptr;
  int lo_n, lo0;
  if (find) {
    lo_n = lo0 = (int)min(max(load_index(P.cu, P.idx64, min(lane, P.n_seg - 1)), (int64_t)INT_MIN), (int64_t)INT_MAX);
  } else {
    lo_n = P.seg_start[rowc];
    lo0 = P.seg_start[row0];
  }
  pu4 Q[HPW][2];
  float gate[HPW], xsa[HPW];
  const bool has_post = P.post_vhat != nullptr;
#pragma unroll
  for (int hh = 0; hh < HPW; hh++) {
    const int head = kvh * G + min(hg * HPW + hh, G - 1);
    const uint16_t* qp = (const uint16_t*)P.q + (int64_t)rowc * P.sqn + (int64_t)head * P.sqh + 8 * g;
    Q[hh][0] = *(const pu4*)qp;
    Q[hh][1] = *(const pu4*)(qp + 32);
    gate[hh] = 1.0f;
    xsa[hh] = 0.f;
    if (has_post && P.post_gate) gate[hh] = P.post_gate[(int64_t)rowc * P.H + head];
    if (has_post && P.post_xsa) xsa[hh] = P.post_xsa[head];
  }
  const int on = OP * (64 * (int)blockIdx.y + 16 * wave);   // the wave's first output column
  uint2 ores[OP ? OP : 1];
#pragma unroll
  for (int j = 0; j < OP; j++) ores[j] = *(const uint2*)((const uint16_t*)P.o_r + (int64_t)rowc * P.o_ldr + on + 16 * j + 4 * g);
  __builtin_amdgcn_sched_barrier(0);
  if (find) {
    const int start = lo_n;
    lo_n = first_token(start, P.n_seg, rowc);
    lo0 = PAIR ? __builtin_amdgcn_readfirstlane(lo_n) : first_token(start, P.n_seg, row0);   // (PAIR: lane 0's row)
    if (g == 0 && row_ok && kvh == 0 && hg == 0 && (OP == 0 || blockIdx.y == 0)) {
      P.seg_out[row] = lo_n;
      P.pidx_out[row] = row;
    }
  }
  // ---- key ranges: the row's, the block's, and the workgroup's from its first row's lower bound (the smallest) to its last row
  if (P.window > 0 && row - P.window + 1 > lo_n) lo_n = row - P.window + 1;
  if (!row_ok) lo_n = INT_MAX;
  if (P.window > 0 && row0 - P.window + 1 > lo0) lo0 = row0 - P.window + 1;
  const uint32_t n_keys = row_ok ? (uint32_t)(row - lo_n + 1) : 0u;           // the row sees keys lo_n .. lo_n + n_keys - 1
  const int rl = min(r0 + 15, P.N - 1);                                       // last real row of the block
  const int lo_first = __builtin_amdgcn_readfirstlane(lo_n);                  // lo is non-decreasing in the row
  const int lo_last = __builtin_amdgcn_readfirstlane(__shfl(lo_n, wave_ok ? rl - r0 : 0, 64));
  const int kbeg = wave_ok ? lo_first & ~31 : 0, kend = wave_ok ? rl + 1 : 0;
  const int kbeg_wg = __builtin_amdgcn_readfirstlane(lo0) & ~31;
  const int kend_wg = min(row0 + qbw * 16, P.N);
  const int nk = (kend_wg - kbeg_wg + 31) >> 5;   // >= 1

  // ---- K / V tiles go from global memory straight into one of two LDS stages of two tiles each, a stage ahead: wave w moves keys
  // 8 w .. 8 w + 7 of K and of V, 16 bytes per lane.  Keys are clamped to N - 1 (a clamped key is masked).  K rows keep their 16-byte chunks
  // xor-ed with (key / 2) % 8, V rows theirs with 2 (key / 2 % 4), which makes the operand reads (lane = key m, chunk 4 s + g;
  // eight keys' 32 bytes per 32 lanes) free of bank conflicts.
  const uint16_t* kbase = (const uint16_t*)P.k + (int64_t)kvh * P.skh;
  const uint16_t* vbase = (const uint16_t*)P.v + (int64_t)kvh * P.svh;
  const uint32_t skn2 = (uint32_t)P.skn * 2, svn2 = (uint32_t)P.svn * 2;  // row strides in bytes
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void*)kbase, 0, (int)((uint32_t)(P.N - 1) * skn2 + 128), 0x00020000);
  const __amdgpu_buffer_rsrc_t rV = __builtin_amdgcn_make_buffer_rsrc((void*)vbase, 0, (int)((uint32_t)(P.N - 1) * svn2 + 128), 0x00020000);
  const int lkey = 8 * wave + (lane >> 3), lch = lane & 7;
  const uint32_t kch = (uint32_t)((lch ^ ((lkey >> 1) & 7)) << 4), vch = (uint32_t)((lch ^ (lkey & 6)) << 4);
  auto issue = [&](unsigned char (*S)[4096], int k) {   // tile k
    const uint32_t r = (uint32_t)min(kbeg_wg + 32 * k + lkey, P.N - 1);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rK, (__attribute__((address_space(3))) void*)(S[0] + 1024 * wave), 16, r * skn2 + kch, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rV, (__attribute__((address_space(3))) void*)(S[1] + 1024 * wave), 16, r * svn2 + vch, 0, 0, 0);
  };
  const bool odd = nk & 1;   // an odd count's first tile is a step of its own, ahead of the pairs, in the second stage
  if (odd) issue(s1[0], 0);
  if (nk > 1) issue(s0[0], odd), issue(s0[1], odd + 1);
  if (!odd && nk > 3) issue(s1[0], 2), issue(s1[1], 3);
  if constexpr (OP > 0) {   // row i of the wave's weight rows, 1 KB, keeps its 16-byte chunks xor-ed with i % 16
    const __amdgpu_buffer_rsrc_t rO = __builtin_amdgcn_make_buffer_rsrc((void*)P.o_w, 0, (int)((uint32_t)(P.o_n - 1) * (uint32_t)P.o_ldw * 2 + 1024u), 0x00020000);
#pragma unroll
    for (int i = 0; i < OW; i++) load_lds16(rO, sw + (wave * OW + i) * 1024, (uint32_t)(on + i) * (uint32_t)P.o_ldw * 2 + (uint32_t)((lane ^ (i & 15)) << 4), 0);
  }

  pf4 O[HPW][4];
  float mrun[HPW], lrun[HPW];
#pragma unroll
  for (int hh = 0; hh < HPW; hh++) {
#pragma unroll
    for (int t = 0; t < 4; t++) O[hh][t] = pf4{0.f, 0.f, 0.f, 0.f};
    mrun[hh] = -INFINITY;
    lrun[hh] = 0.f;
  }
  const uint32_t kld0 = (uint32_t)m * 128 + (uint32_t)((g ^ ((m >> 1) & 7)) << 4), kld1 = (uint32_t)m * 128 + (uint32_t)(((4 + g) ^ ((m >> 1) & 7)) << 4);
  // V^T operand t: lane m of group g names key 4 g + m / 4, dims 16 t + 4 (m % 4) ..; the transposing read hands it dim 16 t + m of keys
  // 4 g .. 4 g + 3
  uint32_t vld[4];
#pragma unroll
  for (int t = 0; t < 4; t++) vld[t] = (uint32_t)(4 * g + (m >> 2)) * 128 + (uint32_t)(((2 * t + ((m & 3) >> 1)) ^ ((4 * g + (m >> 2)) & 6)) << 4) + 8 * (m & 1);

  // NT tiles from tile k on: one maximum, one rescale of the accumulators for all of their keys
  auto step = [&](const unsigned char (*S)[2][4096], int k, auto nt) __attribute__((always_inline)) {
    constexpr int NT = decltype(nt)::value;
    const int tb = kbeg_wg + 32 * k;
    if (!PAIR && (tb < kbeg || tb >= kend)) return;   // (wave-uniform)
    float t[HPW][8 * NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
      pu4 K[4];      // [tile A dims 0..31, tile A dims 32..63, tile B dims 0..31, tile B dims 32..63]: key m, dims 8g..8g+7
      K[0] = *(const pu4*)(S[j][0] + kld0);
      K[1] = *(const pu4*)(S[j][0] + kld1);
      K[2] = *(const pu4*)(S[j][0] + 2048 + kld0);
      K[3] = *(const pu4*)(S[j][0] + 2048 + kld1);
#pragma unroll
      for (int hh = 0; hh < HPW; hh++) {
        pf4 sA = mfma16<DT>(K[0], Q[hh][0], pf4{0.f, 0.f, 0.f, 0.f});
        pf4 sB = mfma16<DT>(K[2], Q[hh][0], pf4{0.f, 0.f, 0.f, 0.f});
        sA = mfma16<DT>(K[1], Q[hh][1], sA);
        sB = mfma16<DT>(K[3], Q[hh][1], sB);
#pragma unroll
        for (int i = 0; i < 4; i++) { t[hh][8 * j + i] = sA[i]; t[hh][8 * j + 4 + i] = sB[i]; }
      }
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
      if (tb + 32 * j < lo_last || tb + 32 * j + 31 > r0) {   // some row of the block does not see all of the tile
        const uint32_t kA = (uint32_t)(tb + 32 * j + 4 * g - lo_n);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const bool out = kA + (i & 3) + 16 * (i >> 2) >= n_keys;
#pragma unroll
          for (int hh = 0; hh < HPW; hh++)
            if (out) t[hh][8 * j + i] = -INFINITY;
        }
      }
    float mc[HPW];
#pragma unroll
    for (int hh = 0; hh < HPW; hh++) {
      // (the maximum that hands NaN on: one instruction for three values, where the one that ignores it needs each made quiet first; a
      // score that is NaN makes its row NaN either way)
      float mx = max3(t[hh][0], t[hh][1], mrun[hh]);
#pragma unroll
      for (int i = 2; i < 8 * NT; i += 2) mx = max3(t[hh][i], t[hh][i + 1], mx);
      // rescale by alpha = exp2((m_old - m_new) c), 1 where the row's maximum did not grow.  Unconditional: a branch
      // here would split the heads into separate blocks and stop the scheduler from overlapping one head's
      // softmax arithmetic with the next head's MFMAs.  (A reference point that may lag behind the maximum, as the decode
      // kernel's, costs precision here: the largest probability is then no longer 1, which is exact in 16 bits.)
      const float mnew = xmaximum(mx);
      const float alpha = mnew == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((mrun[hh] - mnew) * c);
#pragma unroll
      for (int tt = 0; tt < 4; tt++) O[hh][tt] *= alpha;
      lrun[hh] *= alpha;
      mrun[hh] = mnew;
      mc[hh] = mnew == -INFINITY ? 0.f : mnew * c;
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
      pu4 VA[4];     // V^T operands: row m is head dim 16 t + m; slots 0..3 are keys 4g+j of tile A, 4..7 of tile B
#pragma unroll
      for (int tt = 0; tt < 4; tt++) {
        const pu2 a = ld_tr16(S[j][1] + vld[tt]), b = ld_tr16(S[j][1] + 2048 + vld[tt]);
        VA[tt] = pu4{a.x, a.y, b.x, b.y};
      }
#pragma unroll
      for (int hh = 0; hh < HPW; hh++) {
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; i++) p[i] = __builtin_amdgcn_exp2f(fmaf(t[hh][8 * j + i], c, -mc[hh]));
        lrun[hh] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        const pu4 PB = pu4{pack2<DT>(p[0], p[1]), pack2<DT>(p[2], p[3]), pack2<DT>(p[4], p[5]), pack2<DT>(p[6], p[7])};
#pragma unroll
        for (int tt = 0; tt < 4; tt++) O[hh][tt] = mfma16<DT>(VA[tt], PB, O[hh][tt]);
      }
    }
  };
  typedef std::integral_constant<int, 1> one;
  typedef std::integral_constant<int, 2> two;
  // a step's tiles have landed (own loads: the wait; the other waves': the barrier) and every wave is done with the other stage
  auto landed = [&] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto full = [&](unsigned char (*S)[2][4096], unsigned char (*SN)[2][4096], int k) __attribute__((always_inline)) {   // tiles k and k + 1
    if (k < 2) {   // (the weight rows were requested behind the tiles that went out at the start)
      if (k == 0 && nk > 3) wait_vm<4 + OP * 16>(); else wait_vm<OP * 16>();
    } else if (OP > 0 && k == 2) {
      wait_vm<OP * 16>();
    } else {
      wait_vm<0>();
    }
    landed();
    if (k > 0 && k + 2 < nk) issue(SN[0], k + 2), issue(SN[1], k + 3);
    if constexpr (PAIR) {
      step(S, k, two{});
    } else {
      step(S, k, one{});
      step(S + 1, k + 1, one{});
    }
  };
  int k = 0;
  if (odd) {
    if (nk > 1) wait_vm<4 + OP * 16>(); else wait_vm<OP * 16>();
    landed();
    step(s1, 0, one{});
    k = 1;
  }
  for (; k + 4 <= nk; k += 4) {
    full(s0, s1, k);
    full(s1, s0, k + 2);
  }
  if (k < nk) full(s0, s1, k);
  if constexpr (OP > 0) __syncthreads();   // (the stages take the heads' outputs)

  // ---- normalise and store: lane (row m, group g) holds head dims 16 t + 4 g + i, t, i = 0 .. 3
  // Optional epilogue, as in the decode kernel: z (rounded to the activation type, as the attention output tensor would be)
  // -> XSA with the token's normalised v -> per-head gate; the 4 lane groups of a row reduce z . v_hat between them.
  float vv[16];
  if (has_post) {
    const float* vp = P.post_vhat + ((int64_t)rowc * P.KH + kvh) * 64 + 4 * g;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float4 x = *(const float4*)(vp + 16 * i);
      vv[4 * i] = x.x; vv[4 * i + 1] = x.y; vv[4 * i + 2] = x.z; vv[4 * i + 3] = x.w;
    }
  }
  auto rnd = [&](float x) -> float { return DT == UVMI_BF16 ? bf16_to_float(float_to_bf16(x)) : (float)(half_t)x; };
#pragma unroll
  for (int hh = 0; hh < HPW; hh++) {
    const int hq = hg * HPW + hh;
    const float l = psum32(psum16(lrun[hh]));
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    if (P.lse_out && g == 0 && hq < G && row_ok)   // (+inf for a row without keys: its probabilities come out as 0)
      P.lse_out[(int64_t)(kvh * G + hq) * P.lse_stride + row] = l > 0.f ? mrun[hh] * c + __builtin_amdgcn_logf(l) : INFINITY;
    if (P.out == nullptr) continue;   // statistics only
    float o[16];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) o[4 * t + i] = O[hh][t][i] * inv;
    if (has_post) {  // (every lane takes part in the reduction; lanes of absent heads / rows compute on clamped operands)
      float proj = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        o[i] = rnd(o[i]);
        proj += o[i] * vv[i];
      }
      if (P.post_xsa) {
        proj = psum32(psum16(proj));
        const float ah = xsa[hh] * proj;
#pragma unroll
        for (int i = 0; i < 16; i++) o[i] = rnd(o[i] - ah * vv[i]);
      }
#pragma unroll
      for (int i = 0; i < 16; i++) o[i] *= gate[hh];
    }
    if constexpr (OP > 0) {   // into the tiles' first two stages, four heads each: 16 rows of 512 bytes, chunks xor-ed with the row
      unsigned char* sz = (unsigned char*)(hg < 2 ? s0 : s1) + m * 512 + 8 * (g & 1);
#pragma unroll
      for (int t = 0; t < 4; t++)
        *(uint2*)(sz + (((8 * (hq & 3) + 2 * t + (g >> 1)) ^ m) << 4)) = uint2{pack2<DT>(o[4 * t], o[4 * t + 1]), pack2<DT>(o[4 * t + 2], o[4 * t + 3])};
      continue;
    }
    if (hq >= G || !row_ok) continue;
    const int64_t off = (int64_t)row * P.son + (int64_t)(kvh * G + hq) * P.soh + 4 * g;
    if (ODT == UVMI_F32) {
      float* op = (float*)P.out + off;
#pragma unroll
      for (int i = 0; i < 4; i++) *(float4*)(op + 16 * i) = float4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
    } else {
      uint32_t w[8];
#pragma unroll
      for (int i = 0; i < 8; i++) w[i] = ODT == UVMI_BF16 ? pack2<UVMI_BF16>(o[2 * i], o[2 * i + 1]) : pack2<UVMI_F16>(o[2 * i], o[2 * i + 1]);
      uint16_t* op = (uint16_t*)P.out + off;
#pragma unroll
      for (int i = 0; i < 4; i++) *(uint2*)(op + 16 * i) = uint2{w[2 * i], w[2 * i + 1]};
    }
  }
  if constexpr (OP > 0) {
    wait_vm<0>();   // (the wave's own weight rows)
    __syncthreads();
    gf4 y[OP][2];
#pragma unroll
    for (int j = 0; j < OP; j++) y[j][0] = y[j][1] = gf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const gu4 z = *(const gu4*)((const unsigned char*)(s < 8 ? s0 : s1) + m * 512 + (((4 * (s & 7) + g) ^ m) << 4));
#pragma unroll
      for (int j = 0; j < OP; j++) {
        const gu4 w = *(const gu4*)(sw + (wave * OW + 16 * j + m) * 1024 + (((4 * s + g) ^ m) << 4));
        y[j][s & 1] = gmfma<DT>(w, z, y[j][s & 1]);   // (C^T: the lane has columns 16 j + 4 g .. of row m)
      }
    }
    if (!row_ok) return;
#pragma unroll
    for (int j = 0; j < OP; j++) {
      float x[4], q[4];
      gunpack<DT>(ores[j].x, x[0], x[1]);
      gunpack<DT>(ores[j].y, x[2], x[3]);
#pragma unroll
      for (int t = 0; t < 4; t++) q[t] = P.o_ca * x[t] + P.o_cb * ground<DT>(y[j][0][t] + y[j][1][t]);
      *(uint2*)((uint16_t*)P.o_out + (int64_t)row * P.o_ldo + on + 16 * j + 4 * g) = uint2{gpack<DT>(q[0], q[1]), gpack<DT>(q[2], q[3])};
    }
  }
}

// ---------------------------------------------------------------------------------------------------- host side
static int check_prefill(const uvmi_prefill_attn_args* a) {
  UVMI_REQUIRE(a, UVMI_EINVAL, "uvmi_prefill_attn: null args");
  UVMI_REQUIRE(a->N >= 0 && a->H > 0 && a->KH > 0 && a->hd > 0 && a->n_seg >= 0, UVMI_EINVAL, "uvmi_prefill_attn: bad sizes");
  if (a->N == 0) return UVMI_OK;
  UVMI_REQUIRE(a->q && a->k && a->v && a->cu_seqlens && a->out, UVMI_EINVAL, "uvmi_prefill_attn: null pointer");
  UVMI_REQUIRE(a->n_seg >= 1, UVMI_EINVAL, "uvmi_prefill_attn: N > 0 needs at least one sequence");
  UVMI_REQUIRE(a->H % a->KH == 0, UVMI_EINVAL, "uvmi_prefill_attn: H=%d is not a multiple of KH=%d", a->H, a->KH);
  UVMI_REQUIRE(a->q_dtype == UVMI_F16 || a->q_dtype == UVMI_BF16 || a->q_dtype == UVMI_F32, UVMI_EUNSUPPORTED,
               "uvmi_prefill_attn: q must be F16, BF16 or F32");
  UVMI_REQUIRE(is_float_dtype(a->kv_dtype), UVMI_EUNSUPPORTED, "uvmi_prefill_attn: k/v must be F16, BF16 or F32");
  UVMI_REQUIRE(is_float_dtype(a->out_dtype), UVMI_EUNSUPPORTED, "uvmi_prefill_attn: out must be F16, BF16 or F32");
  UVMI_REQUIRE(a->idx_dtype == UVMI_I64 || a->idx_dtype == UVMI_I32, UVMI_EINVAL, "uvmi_prefill_attn: cu_seqlens must be I32 or I64");
  UVMI_REQUIRE(a->window >= 0, UVMI_EINVAL, "uvmi_prefill_attn: negative window");
  UVMI_REQUIRE(a->hd <= 256 && a->H / a->KH <= 16, UVMI_EUNSUPPORTED, "uvmi_prefill_attn: head_dim %d / group %d beyond 256 / 16", a->hd,
               a->H / a->KH);
  const size_t need = uvmi_prefill_attn_workspace_bytes(a->N);
  UVMI_REQUIRE(a->workspace && a->workspace_bytes >= need, UVMI_EWORKSPACE, "uvmi_prefill_attn: workspace of %zu bytes needed, %zu given",
               need, a->workspace_bytes);
  UVMI_REQUIRE(((uintptr_t)a->workspace % 16) == 0, UVMI_EWORKSPACE, "uvmi_prefill_attn: workspace must be 16-byte aligned");
  UVMI_REQUIRE(!a->lse_out || a->lse_stride >= a->N, UVMI_EINVAL, "uvmi_prefill_attn: lse_stride %lld below N", (long long)a->lse_stride);
  return UVMI_OK;
}

static bool prefill_mfma_ok_stats(const uvmi_prefill_attn_args* a) {   // (as below, without an output tensor)
  if (a->hd != 64 || a->H / a->KH > 8 || a->kv_dtype != a->q_dtype || a->q_dtype == UVMI_F32) return false;   // 16-bit operands
  if (!(a->scale > 0.f)) return false;
  auto al = [](const void* p, int n) { return ((uintptr_t)p % n) == 0; };
  if (!al(a->q, 16) || a->sqn % 8 || a->sqh % 8) return false;
  if (!al(a->k, 16) || a->skn % 8 || a->skh % 8 || !al(a->v, 16) || a->svn % 8 || a->svh % 8) return false;
  if (a->skn <= 0 || a->svn <= 0) return false;
  if ((int64_t)a->N * a->skn * 2 >= (1LL << 31) || (int64_t)a->N * a->svn * 2 >= (1LL << 31)) return false;
  return true;
}

static bool prefill_mfma_ok(const uvmi_prefill_attn_args* a) {
  if (a->hd != 64 || a->H / a->KH > 8 || a->kv_dtype != a->q_dtype || a->q_dtype == UVMI_F32) return false;   // 16-bit operands
  if (!(a->scale > 0.f)) return false;  // the running maximum is tracked before the (positive) softmax scale
  auto al = [](const void* p, int n) { return ((uintptr_t)p % n) == 0; };
  if (!al(a->q, 16) || a->sqn % 8 || a->sqh % 8) return false;
  if (!al(a->k, 16) || a->skn % 8 || a->skh % 8 || !al(a->v, 16) || a->svn % 8 || a->svh % 8) return false;
  if (a->skn <= 0 || a->svn <= 0) return false;
  if ((int64_t)a->N * a->skn * 2 >= (1LL << 31) || (int64_t)a->N * a->svn * 2 >= (1LL << 31)) return false;  // 32-bit buffer offsets
  const int ob = a->out_dtype == UVMI_F32 ? 4 : 2;
  if (!al(a->out, 16) || (a->son * ob) % 16 || (a->soh * ob) % 16) return false;
  return true;
}

// 64-column pieces of an output projection's part that rides in the attention's launch, 0: a launch of its own.  8 heads on 1 kv head, the projection
// of what the attention writes, and a compute unit for every block's every part, the smaller one if it can.
static int oproj_pieces(const uvmi_prefill_attn_args* a, const uvmi_gemm_args* o) {
  if (a->H != 8 || a->KH != 1 || a->out_dtype != a->q_dtype || a->lse_out || a->soh != 64) return 0;
  if (!uvmi_gemm_tn_supported(o->dtype, o->M, o->N, o->K, o->lda, o->ldw, o->ldc, o->epilogue)) return 0;
  if (o->epilogue != UVMI_GEMM_RESID || o->norm_a || o->config != 0 || o->dtype != a->q_dtype || o->M != a->N || o->K != 512 || o->N % 64 != 0) return 0;
  if (o->a != a->out || o->lda != a->son || !o->w || !o->c || !o->resid) return 0;
  if (((uintptr_t)o->w % 16) != 0 || ((uintptr_t)o->c % 8) != 0 || ((uintptr_t)o->resid % 8) != 0 || o->ldr % 4 != 0 || o->ldr < o->N) return 0;
  int cus = uvmi_device_cus();
  if (cus <= 0) cus = 256;
  for (int pieces : {1, 2})
    if (o->N % (64 * pieces) == 0 && (int64_t)((a->N + 127) / 128) * (o->N / (64 * pieces)) <= cus / 8) return pieces;   // (of an XCD's blocks)
  return 0;
}

// find: the segment table has yet to be made; the launch does (n_seg <= 64)
static int launch_mfma(const uvmi_prefill_attn_args* a, int32_t* seg_start, int32_t* pidx, bool find, float* lse_out, int64_t lse_stride, hipStream_t st, const uvmi_gemm_args* o = nullptr, int pieces = 0) {
  PrefillParams P = {};
  if (find) { P.cu = a->cu_seqlens; P.idx64 = a->idx_dtype == UVMI_I64 ? 1 : 0; P.n_seg = a->n_seg; P.seg_out = seg_start; P.pidx_out = pidx; }
  P.q = a->q; P.k = a->k; P.v = a->v; P.out = a->out; P.seg_start = seg_start;
  P.sqn = a->sqn; P.sqh = a->sqh; P.skn = a->skn; P.skh = a->skh; P.svn = a->svn; P.svh = a->svh; P.son = a->son; P.soh = a->soh;
  P.N = a->N; P.H = a->H; P.KH = a->KH; P.G = a->H / a->KH; P.window = a->window;
  P.n_hg = P.G <= HPW ? 1 : (P.G <= 2 * HPW ? 2 : 4);   // (G <= 8)
  const int64_t n_qb = (a->N + 15) / 16, qbw = 4 / P.n_hg;
  const int64_t n_wg = (n_qb + qbw - 1) / qbw * a->KH;
  P.scale_log2 = a->scale * 1.4426950408889634f;
  P.post_vhat = a->post_vhat; P.post_gate = a->post_gate; P.post_xsa = a->post_xsa;
  P.lse_out = lse_out; P.lse_stride = lse_stride;
  UVMI_REQUIRE(n_wg < (1LL << 30), UVMI_EUNSUPPORTED, "uvmi_prefill_attn: too many work items");
  P.n_wg = (int)n_wg;
  const unsigned nblk = (unsigned)((n_wg + 7) / 8 * 8);
  const dim3 grid(nblk), blk(256);
  const int od = a->out_dtype;
  if (o) {
    P.o_w = o->w; P.o_r = o->resid; P.o_out = o->c; P.o_ldw = o->ldw; P.o_ldr = o->ldr; P.o_ldo = o->ldc; P.o_n = o->N; P.o_ca = o->ca; P.o_cb = o->cb;
    const dim3 parts(nblk, (unsigned)(o->N / (64 * pieces)));
#define UVMI_LO(DT)                                                                                                       \
  do {                                                                                                                    \
    if (pieces == 1) hipLaunchKernelGGL((prefill_attn_mfma_hd64<DT, DT, 1, true>), parts, blk, 0, st, P);                       \
    else hipLaunchKernelGGL((prefill_attn_mfma_hd64<DT, DT, 2, true>), parts, blk, 0, st, P);                                   \
  } while (0)
    if (a->q_dtype == UVMI_F16) UVMI_LO(UVMI_F16); else UVMI_LO(UVMI_BF16);
#undef UVMI_LO
    UVMI_CHECK_LAUNCH("uvmi_prefill_attn_o");
    return UVMI_OK;
  }
#define UVMI_LP(QD, OD)                                                                                                  \
  do {                                                                                                                   \
    if (P.n_hg == 4) hipLaunchKernelGGL((prefill_attn_mfma_hd64<QD, OD, 0, true>), grid, blk, 0, st, P);                  \
    else hipLaunchKernelGGL((prefill_attn_mfma_hd64<QD, OD, 0, false>), grid, blk, 0, st, P);                            \
  } while (0)
#define UVMI_L(QD)                                                                                                       \
  do {                                                                                                                   \
    if (od == UVMI_F16) UVMI_LP(QD, UVMI_F16);                                                                           \
    else if (od == UVMI_BF16) UVMI_LP(QD, UVMI_BF16);                                                                    \
    else UVMI_LP(QD, UVMI_F32);                                                                                          \
  } while (0)
  if (a->q_dtype == UVMI_F16) UVMI_L(UVMI_F16); else UVMI_L(UVMI_BF16);
#undef UVMI_L
#undef UVMI_LP
  UVMI_CHECK_LAUNCH("uvmi_prefill_attn");
  return UVMI_OK;
}

// For the backward (prefill_attn_bwd.hip): the segment table of cu_seqlens into seg_start (N ints; pidx: N ints of scratch) and
// the rows' softmax statistics into lse (H, lse_stride), from one forward pass that stores no output.  a->out may be null.
int prefill_attn_stats(const uvmi_prefill_attn_args* a, int32_t* seg_start, int32_t* pidx, float* lse, int64_t lse_stride, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(prefill_segments, dim3((unsigned)((a->N + 255) / 256)), dim3(256), 0, st, a->cu_seqlens, a->idx_dtype == UVMI_I64 ? 1 : 0,
                     a->n_seg, a->N, seg_start, pidx);
  UVMI_CHECK_LAUNCH("uvmi_prefill_attn_bwd(segments)");
  uvmi_prefill_attn_args b = *a;
  b.out = nullptr; b.out_dtype = a->q_dtype; b.son = (int64_t)a->H * 64; b.soh = 64;
  b.post_vhat = nullptr; b.post_gate = nullptr; b.post_xsa = nullptr;
  UVMI_REQUIRE(prefill_mfma_ok_stats(&b), UVMI_EUNSUPPORTED, "uvmi_prefill_attn_bwd: q / k / v layout not served by the MFMA kernels");
  return launch_mfma(&b, seg_start, pidx, false, lse, lse_stride, st);
}

}  // namespace uvmi

using namespace uvmi;

extern "C" size_t uvmi_prefill_attn_workspace_bytes(int N) {
  if (N <= 0) return 0;
  return (((size_t)N * 4 + 255) / 256 * 256) * 2;
}

extern "C" int uvmi_prefill_attn_path(const uvmi_prefill_attn_args* a) {
  int rc = check_prefill(a);
  if (rc) return rc;
  return prefill_mfma_ok(a) ? 1 : 0;
}

// o: the output projection that follows (uvmi_prefill_attn_o)
static int prefill_attn_run(const uvmi_prefill_attn_args* a, const uvmi_gemm_args* o, void* stream) {
  int rc = check_prefill(a);
  if (rc) return rc;
  if (a->N == 0) return o ? uvmi_gemm_resid(o, stream) : UVMI_OK;
  hipStream_t st = (hipStream_t)stream;
  int32_t* seg_start = (int32_t*)a->workspace;
  int32_t* pidx = (int32_t*)((char*)a->workspace + ((size_t)a->N * 4 + 255) / 256 * 256);
  const bool find = !a->segments_ready && a->n_seg <= 64 && prefill_mfma_ok(a);
  if (!a->segments_ready && !find) {
    hipLaunchKernelGGL(prefill_segments, dim3((unsigned)((a->N + 255) / 256)), dim3(256), 0, st, a->cu_seqlens, a->idx_dtype == UVMI_I64 ? 1 : 0,
                       a->n_seg, a->N, seg_start, pidx);
    UVMI_CHECK_LAUNCH("uvmi_prefill_attn(segments)");
  }
  if (a->post_vhat) {
    UVMI_REQUIRE(prefill_mfma_ok(a), UVMI_EUNSUPPORTED, "uvmi_prefill_attn: the fused post epilogue needs the MFMA kernel (head_dim 64, 16-bit q / k / v)");
    UVMI_REQUIRE(((uintptr_t)a->post_vhat % 16) == 0, UVMI_EINVAL, "uvmi_prefill_attn: post_vhat must be 16-byte aligned");
  }
  UVMI_REQUIRE(!a->lse_out || prefill_mfma_ok(a), UVMI_EUNSUPPORTED, "uvmi_prefill_attn: lse_out needs the MFMA kernel (head_dim 64, 16-bit q / k / v)");
  if (!prefill_mfma_ok(a)) {
    // every packed token is a decode row whose "cache" is the packed K / V of the call (batch stride 0)
    uvmi_attn_args d = {};
    d.q = a->q; d.q_dtype = a->q_dtype; d.sqb = a->sqn; d.sqh = a->sqh;
    d.k_cache = a->k; d.v_cache = a->v; d.kv_dtype = a->kv_dtype;
    d.skb = 0; d.skh = a->skh; d.sks = a->skn; d.svb = 0; d.svh = a->svh; d.svs = a->svn;
    d.pos = pidx; d.starts = seg_start; d.idx_dtype = UVMI_I32;
    d.out = a->out; d.out_dtype = a->out_dtype; d.sob = a->son; d.soh = a->soh;
    d.B = a->N; d.H = a->H; d.KH = a->KH; d.S = a->N; d.hd = a->hd;
    d.scale = a->scale; d.window = a->window; d.ring = 0; d.num_splits = 1;
    rc = uvmi_decode_attn(&d, stream);
    return rc || !o ? rc : uvmi_gemm_resid(o, stream);
  }
  if (const int pieces = o ? oproj_pieces(a, o) : 0) return launch_mfma(a, seg_start, pidx, find, nullptr, 0, st, o, pieces);
  rc = launch_mfma(a, seg_start, pidx, find, a->lse_out, a->lse_stride, st);
  return rc || !o ? rc : uvmi_gemm_resid(o, stream);
}

extern "C" int uvmi_prefill_attn(const uvmi_prefill_attn_args* a, void* stream) { return prefill_attn_run(a, nullptr, stream); }

extern "C" int uvmi_prefill_attn_o(const struct uvmi_prefill_attn_o_args* a, void* stream) {
  UVMI_REQUIRE(a && a->attn && a->gemm, UVMI_EINVAL, "uvmi_prefill_attn_o: null args");
  return prefill_attn_run(a->attn, a->gemm, stream);
}

