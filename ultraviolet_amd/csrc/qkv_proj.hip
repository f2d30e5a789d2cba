// The extended QKV projection of prompts and mixed passes with its post-processing in the same launch: q, k, v and the gates' logits of a
// block's rows (A W^T, the pre-norm as a row scale: uvmi_gemm_tn_ex), QK-norm, rotation, value embedding, the cache append and the
// attention epilogue's inputs (uvmi_qkv_post) - Attention.qkv and what follows it in the reference (ultraviolet/model.py:302-319,
// kernels/fast_decode.py:291-294, 315-317).
//
// For passes of up to a few hundred rows, where the two launches last as long as their trips to the last-level cache and the start of a launch
// (93 rows: 3.4 + 4.3 us of a layer's 27).  The projection streams as in gemm_stream.hip - the waves split K, a wave's slabs go straight into
// its own LDS, partial sums meet behind one barrier - but a tile is 16 FM rows of one head's 64 columns, so that what QK-norm, rotation and
// quantisation reduce over lies in one wave: lane (r, g) holds dims 16 j + 4 g + t (j, t = 0 .. 3) of row r, a rotated pair (d, d + 16) in one
// lane, the rest of a row in the lanes l ^ 16, l ^ 32.  Ten strips of columns: 8 query heads, the key, the value; the value's strip is 80 columns
// wide, for the value-embedding gate's logit (and the output gates', which it writes) sit behind the value's columns.
// The rows' positions are requested ahead of the first slab, what depends on them (rotation, value embedding) behind the slabs.  Roundings
// are those of the two launches: the projection to the activation type, then each operation's own (common.h: rope_rot, ve_add).
//
// What bounds it: a trip for the slabs, as long as a compute unit takes to pull 96 - 144 rows of operands, and the start of a launch.  A whole prefill, two
// launches a layer -> one, us: 30 rows 282 -> 267, 93 rows 311 -> 296, 300 rows 368 -> 347 (16-row tiles), 500 418 -> 400, 700 458 -> 444
// (32), 900 485 -> 476, 1200 510 -> 498, 1550 535 -> 519 (64).
#include "common.h"
#include "gemm_util.h"
#include "qkv_post.h"

namespace uvmi {

// FM: fragments of 16 rows; R: slabs of a wave in flight
template <int DT, int FM, int R, bool NORM>
__global__ __launch_bounds__(320) void qkv_proj_kernel(const void* a_a, const void* a_w, uint32_t lda2, uint32_t ldw2, int M, int K, int tiles_m,
                                                       float norm_eps, QkvArgs A) {
  constexpr int NW = 5, BM = 16 * FM, FN = 5, ROWS = BM + 16 * FN;
  constexpr int SLAB = ROWS * 128 > FM * FN * 1024 ? ROWS * 128 : FM * FN * 1024;   // a wave's slab, later its partial sums
  constexpr int LOADS = BM / 8 + 8;                                                 // of a slab (the value's strip: two more)
  __shared__ __attribute__((aligned(1024))) unsigned char s0[NW * SLAB];
  __shared__ __attribute__((aligned(1024))) unsigned char s1[R > 1 ? (NW - 1) * SLAB + ROWS * 128 : 16];
  __shared__ float sSS[NORM ? NW * BM : 1];
  static_assert(sizeof(s0) + (R > 1 ? sizeof(s1) : 0) + (NORM ? sizeof(sSS) : 0) <= 160 * 1024, "a compute unit's LDS");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = tiles_m * 10, per = (T + 7) / 8;
  const int L = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);   // (an XCD gets neighbouring tiles of a strip)
  if (L >= T) return;
  const int strip = L / tiles_m, m0 = (L % tiles_m) * BM;
  const bool is_v = strip == 9;
  const int r = lane & 15, g = lane >> 4;
  // ---- the row that this lane finishes (wave f: fragment f), its position and what else depends on the row alone
  const bool fin = wave < FM;
  const int row = m0 + 16 * wave + r;
  const bool row_ok = fin && row < M;
  const int64_t rowc = row_ok ? row : (M > 0 ? M - 1 : 0);
  int64_t p = 0, crow = 0, lastp = 0, tk = 0;
  if (fin) {
    p = A.pos[rowc];
    if (strip >= 8) {
      crow = A.rows ? A.rows[rowc] : rowc;
      if (A.last_pos) lastp = A.last_pos[rowc];
      if (is_v && A.has_ve) tk = A.tok[rowc];
    }
  }
  // ---- loader, as gemm_stream_kernel's: load i of a slab moves its rows 8 i .. 8 i + 7 (the tile's rows of A, then of W)
  const int lr = lane >> 3;
  const uint32_t c0 = (uint32_t)(((lane & 7) ^ (lr >> 1)) << 4), c1 = c0 ^ 64;
  const uint32_t ra = (uint32_t)(m0 + lr) * lda2, rw = (uint32_t)(64 * strip + lr) * ldw2;
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)a_a, 0, (int)((uint32_t)(M - 1) * lda2 + (uint32_t)K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void*)a_w, 0, (int)(655u * ldw2 + (uint32_t)K * 2), 0x00020000);
  const int nk = K / 64, nw = (nk - wave + NW - 1) / NW;   // slabs of this wave: wave, wave + NW, ..
  const int lds0 = wave * SLAB;
  auto issue = [&](unsigned char* S, int i) {
    const int ko = (wave + NW * i) * 128;
#pragma unroll
    for (int l = 0; l < BM / 8; l++) load_lds16(rA, S + lds0 + 1024 * l, ra + (l & 1 ? c1 : c0) + (uint32_t)(8 * l) * lda2, ko);
#pragma unroll
    for (int l = 0; l < 8; l++) load_lds16(rW, S + lds0 + BM * 128 + 1024 * l, rw + (l & 1 ? c1 : c0) + (uint32_t)(8 * l) * ldw2, ko);
    if (is_v) {
#pragma unroll
      for (int l = 8; l < 10; l++) load_lds16(rW, S + lds0 + BM * 128 + 1024 * l, rw + (l & 1 ? c1 : c0) + (uint32_t)(8 * l) * ldw2, ko);
    }
  };
  if (nw > 0) issue(s0, 0);
  if (R > 1 && nw > 1) issue(s1, 1);
  // ---- behind the slabs: the rotation of the lane's frequencies 4 g .. 4 g + 3, the value embedding of its dims
  const bool in_tab = p >= 0 && p < A.rope_n;
  float4 cs = float4{1.f, 1.f, 1.f, 1.f}, sn = float4{0.f, 0.f, 0.f, 0.f};
  uint2 ve[4];
  if (fin) {
    if (A.rope && strip < 9) {
      const float* tab = A.rope_tab + (in_tab ? p : 0) * 32 + 4 * g;
      cs = *(const float4*)tab;
      sn = *(const float4*)(tab + 16);
    }
    if (is_v && A.has_ve) {
      const int64_t t = tk < 0 ? 0 : (tk >= A.vocab ? A.vocab - 1 : tk);
#pragma unroll
      for (int j = 0; j < 4; j++) ve[j] = *(const uint2*)((const uint16_t*)A.ve_table + t * 64 + 16 * j + 4 * g);
    }
  }

  gf4 acc[FM][FN], sq[FM];
#pragma unroll
  for (int i = 0; i < FM; i++) {
    sq[i] = gf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = gf4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t ld0 = (uint32_t)r * 128 + (uint32_t)((g ^ ((r >> 1) & 7)) << 4), ld1 = (uint32_t)r * 128 + (uint32_t)(((4 + g) ^ ((r >> 1) & 7)) << 4);
  auto slab = [&](unsigned char* S, int i) {
    if (R > 1 && i + 1 < nw) wait_vm<LOADS>(); else wait_vm<0>();   // (loads land in order; what else is on its way makes it wait for more)
    asm volatile("" ::: "memory");
    const unsigned char* Sa = S + lds0;
    const unsigned char* Sw = Sa + BM * 128;
    gu4 af[2][FM], wf[2][FN];
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int j = 0; j < 4; j++) wf[s][j] = *(const gu4*)(Sw + 2048 * j + (s ? ld1 : ld0));
      if (is_v) wf[s][4] = *(const gu4*)(Sw + 2048 * 4 + (s ? ld1 : ld0));
#pragma unroll
      for (int f = 0; f < FM; f++) af[s][f] = *(const gu4*)(Sa + 2048 * f + (s ? ld1 : ld0));
    }
    if (i + R < nw) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slab is in registers: its place may be filled again
      issue(S, i + R);
    }
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int f = 0; f < FM; f++) {
#pragma unroll
        for (int j = 0; j < 4; j++) acc[f][j] = gmfma<DT>(wf[s][j], af[s][f], acc[f][j]);
        if (is_v) acc[f][4] = gmfma<DT>(wf[s][4], af[s][f], acc[f][4]);
        if (NORM) sq[f] = gmfma<DT>(af[s][f], af[s][f], sq[f]);
      }
    }
  };
  for (int i = 0; i < nw; i += R) {
    slab(s0, i);
    if constexpr (R > 1)
      if (i + 1 < nw) slab(s1, i + 1);
  }

  // ---- the waves' partial sums meet in LDS; wave f finishes fragment f
  if (NORM) {
#pragma unroll
    for (int f = 0; f < FM; f++) {   // (lane (r, g) holds elements (4 g + t, r) of X X^T)
      const float v = r & 2 ? (r & 1 ? sq[f][3] : sq[f][2]) : (r & 1 ? sq[f][1] : sq[f][0]);
      if (g == r >> 2) sSS[wave * BM + 16 * f + r] = v;
    }
  }
  auto part = [&](int w, int f) { return (gf4*)(s0 + w * SLAB + 1024 * f) + lane; };
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int j = 0; j < FN; j++)
      if (j < 4 || is_v) *part(wave, f * FN + j) = acc[f][j];
  __syncthreads();
  if (!fin) return;
  float rn = 1.0f;
  if (NORM) {
    float t = sSS[16 * wave + r];
#pragma unroll
    for (int w = 1; w < NW; w++) t += sSS[w * BM + 16 * wave + r];
    rn = rsqrtf(t / (float)K + norm_eps);
  }
  auto rnd = [](float f) { return ground<DT>(f); };
  auto column = [&](int j, float* x) {   // columns 16 j + 4 g .. of the strip, rounded to the activation type
    gf4 v = *part(0, wave * FN + j);
#pragma unroll
    for (int w = 1; w < NW; w++) v += *part(w, wave * FN + j);
#pragma unroll
    for (int t = 0; t < 4; t++) x[t] = rnd(v[t] * rn);
  };
  float x[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++) column(j, x[j]);
  auto sum_squares = [&]() {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int t = 0; t < 4; t++) ss = fmaf(x[j][t], x[j][t], ss);
    return xsum32(xsum16(ss));
  };
  if (!is_v) {   // ---- a query head or the key: norm, rotation of dims 0 .. 31 (d with d + 16)
    const float rs = rsqrtf(sum_squares() * (1.0f / 64.0f) + A.eps);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int t = 0; t < 4; t++) x[j][t] = rnd(x[j][t] * rs);
    if (A.rope) {
      float c4[4] = {cs.x, cs.y, cs.z, cs.w}, s4[4] = {sn.x, sn.y, sn.z, sn.w};
      if (!in_tab) {   // a position outside the table: the angles are formed here
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const float th = (float)p * A.inv_freq[4 * g + t];
          c4[t] = rnd(cosf(th));
          s4[t] = rnd(sinf(th));
        }
      }
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const float a = x[0][t], b = x[1][t];
        x[0][t] = rope_rot(a, b, c4[t], s4[t], true, rnd);
        x[1][t] = rope_rot(b, a, c4[t], s4[t], false, rnd);
      }
    }
  } else {       // ---- the value: its embedding, the output gates, its direction for the attention epilogue
    if (A.has_ve || A.gate_out) {
      float gl[4];   // columns 640 + 4 g ..: the heads' gates (g = 0, 1), the value embedding's (648)
      column(4, gl);
      if (A.gate_out && g < 2 && row_ok) {
        float o[4];
#pragma unroll
        for (int t = 0; t < 4; t++) o[t] = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-gl[t]))));
        *(float4*)(A.gate_out + (int64_t)row * 8 + 4 * g) = float4{o[0], o[1], o[2], o[3]};
      }
      if (A.has_ve) {
        const float vl = __shfl(gl[0], 32 + r, 64);
        const float gv = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-vl))));
#pragma unroll
        for (int j = 0; j < 4; j++) {
          float e[4];
          gunpack<DT>(ve[j].x, e[0], e[1]);
          gunpack<DT>(ve[j].y, e[2], e[3]);
#pragma unroll
          for (int t = 0; t < 4; t++) x[j][t] = ve_add(x[j][t], gv, e[t], rnd);
        }
      }
    }
    if (A.vhat_out) {
      const float nv = fmaxf(sqrtf(sum_squares()), A.xsa_eps);
      if (row_ok) {
#pragma unroll
        for (int j = 0; j < 4; j++)
          *(float4*)(A.vhat_out + (int64_t)row * 64 + 16 * j + 4 * g) = float4{x[j][0] / nv, x[j][1] / nv, x[j][2] / nv, x[j][3] / nv};
      }
    }
  }
  auto store = [&](void* base, int64_t off) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      *(uint2*)((uint16_t*)base + off + 16 * j + 4 * g) = uint2{gpack<DT>(x[j][0], x[j][1]), gpack<DT>(x[j][2], x[j][3])};
  };
  if (strip < 8) {
    if (row_ok) store(A.q_out, ((int64_t)row * 8 + strip) * 64);
    return;
  }
  void* out = is_v ? A.v_out : A.k_out;
  if (out && row_ok) store(out, (int64_t)row * 64);
  if (!A.k_cache) return;
  const int64_t slot = A.ring ? (p % A.S) : p;
  bool wr = row_ok && crow >= 0 && p >= 0 && slot < A.S;
  if (wr && A.ring && A.last_pos) wr = p > lastp - A.S;
  int8_t* cache = is_v ? A.v_cache : A.k_cache;
  const int64_t at = crow * A.scb + slot * A.scs;
  if (!A.k_scale) {
    if (wr) store(cache, at);
    return;
  }
  float am = 0.f;   // int8 codes and scale, the standalone quantizer's arithmetic
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int t = 0; t < 4; t++) am = fmaxf(am, fabsf(x[j][t]));
  am = xmax32(xmax16(am));
  const uint16_t sb = float_to_half_bits(__fdiv_rn(am, 127.0f));
  const float sf = fmaxf(half_bits_to_float(sb), 1e-30f);
  if (!wr) return;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint32_t word = 0;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const float qv = fminf(fmaxf(__builtin_rintf(__fdiv_rn(x[j][t], sf)), -127.0f), 127.0f);
      word |= (uint32_t)(uint8_t)(int8_t)(int)qv << (8 * t);
    }
    *(uint32_t*)(cache + at + 16 * j + 4 * g) = word;
  }
  if (g == 0) (is_v ? A.v_scale : A.k_scale)[crow * A.ssb + slot] = sb;
}

template <int DT, int FM, int R>
static void launch_qkv(const uvmi_gemm_args* g, const QkvArgs& A, hipStream_t st) {
  const int tiles = (int)((g->M + 16 * FM - 1) / (16 * FM)), T = 10 * tiles;
  const dim3 grid((unsigned)((T + 7) / 8 * 8)), blk(320);
  const uint32_t lda2 = (uint32_t)g->lda * 2, ldw2 = (uint32_t)g->ldw * 2;
  if (g->norm_a) hipLaunchKernelGGL((qkv_proj_kernel<DT, FM, R, true>), grid, blk, 0, st, g->a, g->w, lda2, ldw2, (int)g->M, g->K, tiles, g->eps, A);
  else hipLaunchKernelGGL((qkv_proj_kernel<DT, FM, R, false>), grid, blk, 0, st, g->a, g->w, lda2, ldw2, (int)g->M, g->K, tiles, g->eps, A);
}

// The extended projection of the engine's shape, of the rows that the post-processing reads.
static bool proj_shape(const uvmi_gemm_args* g, const uvmi_qkv_post_args* p, const QkvArgs& A) {
  if (!g->a || !g->w || !g->c || !uvmi_gemm_tn_supported(g->dtype, g->M, g->N, g->K, g->lda, g->ldw, g->ldc, g->epilogue)) return false;
  if (g->N != 656 || g->epilogue != UVMI_GEMM_STORE || g->M == 0 || g->M != p->n || g->dtype != p->dtype) return false;
  if (((uintptr_t)g->a | (uintptr_t)g->w) % 16 != 0 || (g->norm_a && g->eps < 0.f)) return false;
  return qkv_post_engine_shape(p, A) && A.ld == g->ldc && p->qkv == g->c;
}

// Rows of the tile that takes the projection with its post-processing in one launch; 0: two launches.
static int proj_rows(const uvmi_gemm_args* g, const uvmi_qkv_post_args* p, const QkvArgs& A) {
  if (g->config != 0 || !proj_shape(g, p, A)) return 0;
  const uintptr_t a16 = (uintptr_t)A.q_out | (uintptr_t)A.k_out | (uintptr_t)A.v_out | (uintptr_t)A.vhat_out | (uintptr_t)A.gate_out | (A.has_ve ? (uintptr_t)A.ve_table : 0);
  if (a16 % 16 != 0) return 0;
  if (A.k_cache && ((((uintptr_t)A.k_cache | (uintptr_t)A.v_cache) % 8) != 0 || A.scb % 4 != 0 || A.scs % 4 != 0)) return 0;
  int cus = uvmi_device_cus();
  if (cus <= 0) cus = 256;
  for (int rows : {16, 32, 64})   // the smallest tile that leaves a compute unit one workgroup; beyond, the projection has larger ones to gain by
    if (10 * ((g->M + rows - 1) / rows) <= cus) return rows;
  return 0;
}

}  // namespace uvmi

using namespace uvmi;

extern "C" int uvmi_qkv_proj(const struct uvmi_qkv_proj_args* a, void* stream) {
  UVMI_REQUIRE(a && a->gemm && a->post, UVMI_EINVAL, "uvmi_qkv_proj: null args");
  QkvArgs A;
  int rc = qkv_post_prepare(a->post, &A);
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  const uvmi_gemm_args* g = a->gemm;
  const int rows = g->a && g->w && g->c && !a->sums ? proj_rows(g, a->post, A) : 0;
  if (rows == 0) {
    // Many rows, on tiles loaded straight into LDS: the query heads' part is an epilogue of the projection, so they are not written, read and written
    // again (two thirds of what the post-processing moves).  Projection and post-processing, us: 3328 rows 18.2 -> 15.8, 5000 21.0 -> 16.5, 9000
    // 28.5 -> 22.8; with sums 18 432 rows 37.4 -> 33.7, 33 216 61.5 -> 55.9, 65 536 109 -> 87.  Below, on the streaming tiles, which cut heads apart
    // and split K over waves, the two launches stay: 2600 rows 15.7 against 15.4 on 128 x 128 tiles with it, 1700 13.1 / 15.3.
    if (proj_shape(g, a->post, A) && qkv_post_rows_ok(a->post)) {
      if (gemm_query_post(g, QueryPost{A.q_out, A.pos, A.rope ? A.rope_tab : nullptr, A.rope_n, A.eps}, a->sums, a->sums_ld, st)) {
        qkv_post_kv_launch(g->dtype, A, st);
        UVMI_CHECK_LAUNCH("uvmi_qkv_proj");
        return UVMI_OK;
      }
    }
    const struct uvmi_gemm_sums_args s = {g, a->sums, a->sums_ld};
    rc = a->sums ? uvmi_gemm_sums(&s, stream) : uvmi_gemm_tn_ex(g, stream);
    return rc ? rc : uvmi_qkv_post(a->post, stream);
  }
#define UVMI_Q(DT) do { if (rows == 16) launch_qkv<DT, 1, 2>(g, A, st); else if (rows == 32) launch_qkv<DT, 2, 2>(g, A, st); else launch_qkv<DT, 4, 1>(g, A, st); } while (0)
  if (g->dtype == UVMI_F16) UVMI_Q(UVMI_F16); else UVMI_Q(UVMI_BF16);
#undef UVMI_Q
  UVMI_CHECK_LAUNCH("uvmi_qkv_proj");
  return UVMI_OK;
}
