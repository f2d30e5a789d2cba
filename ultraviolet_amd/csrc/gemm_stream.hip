// 16-bit GEMM for steps of up to a few thousand rows: C[M, N] = A[M, K] . W[N, K]^T, fp32 accumulation, with the epilogues of
// the other forms - SwiGLU on interleaved gate / up slabs, the block's residual update, the RMS pre-norm as a row scale.  These
// are the F.linear calls of the reference's fused inference path (ultraviolet/model.py:302-335 attention projections,
// 388-391 MLP) with what surrounds them (:566-571).
//
// What bounds it: 0.7 - 4.3 MB of weights that the previous layers have pushed out of the L2, and activations that another XCD
// wrote: a launch lasts as long as the round trips to the last-level cache that it puts in sequence, then as long as a compute
// unit takes to pull its tiles through the L2 (64 bytes per clock).  To keep that pipe full for one trip of ~1 us takes ~150 KB in
// flight per compute unit, which is what LDS holds.  So:
//   * the NW waves of a workgroup split K: wave w takes the 64-wide slabs w, w + NW, .. of the tile's rows of A and W, from global
//     memory straight into its own part of LDS (16 bytes per lane, a 1 KB load is 8 rows), R slabs ahead, and multiplies them
//     into its own accumulators of the whole tile.  A wave waits for its own loads only: the loop has no barrier, no staging
//     registers and no LDS stores, and an operand fragment is read from LDS once per 16-row fragment of the other side;
//   * small problems have all their slabs in flight within the first few hundred cycles;
//   * LDS rows are 128 bytes with the 16-byte chunk index xor-ed with (row / 2) % 8 (the lane fetches the chunk that belongs at
//     its place), so the 16-row operand reads (lane (r, g) reads chunk 4 s + g of row r) touch every bank once;
//   * the MFMA's A input is the weight fragment and its B input the activation fragment, so an accumulator holds C^T: a lane
//     has 4 consecutive columns of one row and stores them as one 8-byte write;
//   * the partial sums meet in LDS (the slabs' space) behind the kernel's only barrier; a wave adds and finishes its share of the
//     fragments.  The residual of that share is requested before anything else; the squares of NORM are the diagonal of an
//     activation fragment's product with itself, one more matrix instruction for it (32 vector ones before: twice the time of the 64 x
//     64 tile's own products);
//   * rows past M or N are zeros (computed, not stored);
//   * individual scalar arguments rather than a parameter block: they arrive in SGPRs with the wave.
// us per launch in a stream of launches with 20 layers' weights in turn (N x K: 656 x 640 with NORM | 640 x 512 RESID | 3328 x 640
// NORM, SWIGLU | 640 x 1664 RESID), and in brackets what the forms took that it replaced (a whole weight strip parked in LDS
// behind a barrier below 448 rows, 64 x 64 tiles through registers from there on):
//      1 row   2.7 [3.9] | 2.5 [3.8] | 3.4 [4.7] | 2.9 [4.3]        64 rows   2.7 [4.4] | 2.5 [4.3] | 3.7 [6.0] | 3.2 [5.3]
//    256 rows  3.5 [5.6] | 3.0 [5.4] | 5.4 [6.5] | 4.6 [9.2]       512 rows   4.0 [6.2] | 3.4 [5.2] | 7.4 [8.7] | 5.3 [8.9]
//   2048 rows  7.3 [8.4] | 5.9 [7.4] |     -     | 9.5 [13.7]
#include "common.h"
#include "gemm_util.h"

namespace uvmi {

struct StreamParams {
  const void* a; const void* w; void* c; const void* r;
  int64_t ldc, ldr;     // elements
  uint32_t lda2, ldw2;  // row pitches in bytes
  int M, N, K, tiles_m, tiles_n, rowsplit;
  float eps, ca, cb;
};

// EPI 0: C = A W^T (M, N).  EPI 1: W rows are [gate 16 | up 16] slabs; C = silu(gate) * up, (M, N / 2); a tile of 16 columns
// takes 8 gate rows and their 8 up rows.  EPI 2: C = ca * R + cb * (A W^T).  NORM: A stands for its RMS-normalised rows.
template <int DT, int BM, int BN, int NW, int R, int EPI, bool NORM>
__global__ __launch_bounds__(64 * NW) void gemm_stream_kernel(const void* a_a, const void* a_w, uint32_t a_lda2, uint32_t a_ldw2, int a_M, int a_N,
                                                              int a_K, int a_tiles_m, int a_tiles_n, int a_rowsplit, const void* a_r,
                                                              void* a_c, int64_t a_ldc, int64_t a_ldr, float a_eps, float a_ca, float a_cb) {
  const StreamParams P = {a_a, a_w, a_c, a_r, a_ldc, a_ldr, a_lda2, a_ldw2, a_M, a_N, a_K, a_tiles_m, a_tiles_n, a_rowsplit, a_eps, a_ca, a_cb};
  constexpr int FM = BM / 16, FN = BN / 16, F = FM * FN;
  constexpr int ROWS = BM + BN, LOADS = ROWS / 8;          // a load instruction moves 8 rows of 128 bytes
  constexpr int FW = (F + NW - 1) / NW;                    // fragments per wave in the epilogue
  static_assert(R == 1 || R == 2, "slabs of a wave in flight");
  constexpr int SLAB = ROWS * 128 > F * 1024 ? ROWS * 128 : F * 1024;   // a wave's slab, later its partial sums
  // (one object per stage: the compiler can then tell that reads of one do not touch the one a load is filling)
  __shared__ __attribute__((aligned(1024))) unsigned char s0[NW * SLAB];
  __shared__ __attribute__((aligned(1024))) unsigned char s1[R > 1 ? (NW - 1) * SLAB + ROWS * 128 : 16];
  __shared__ float sSS[NORM ? NW * BM : 1];
  static_assert(sizeof(s0) + (R > 1 ? sizeof(s1) : 0) + (NORM ? sizeof(sSS) : 0) <= 160 * 1024, "a compute unit's LDS");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = P.tiles_m * P.tiles_n, per = (T + 7) / 8;
  const int L = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (L >= T) return;
  const int bn = P.rowsplit ? L % P.tiles_n : L / P.tiles_m, bm = P.rowsplit ? L / P.tiles_n : L % P.tiles_m;
  const int m0 = bm * BM, n0 = bn * BN;
  const int r = lane & 15, g = lane >> 4;

  // ---- loader: load i of a slab moves its rows 8 i .. 8 i + 7 (the tile's rows of A, then of W).  Rows past the last one come out as zeros:
  // the descriptors' bounds.  (One multiplication and an addition per load: 64-bit addresses of clamped rows took ~60 cycles a load
  // before the first one left, and twice the registers; 2 - 3 % of a launch of 400 to 2500 rows, 512 x 3328 x 640 7.76 -> 7.57 us.)
  const int lr = lane >> 3;
  uint32_t off[LOADS];
  {
    const uint32_t c0 = (uint32_t)(((lane & 7) ^ (lr >> 1)) << 4), c1 = c0 ^ 64;   // chunk of an even, an odd load
    const uint32_t ra = (uint32_t)(m0 + lr) * P.lda2;
#pragma unroll
    for (int i = 0; i < BM / 8; i++) off[i] = ra + (i & 1 ? c1 : c0) + (uint32_t)(8 * i) * P.lda2;
    // (EPI 1, 16 columns: 8 gate rows and, 16 rows on, their 8 up rows)
    constexpr bool SPLIT = EPI == 1 && BN == 16;
    const uint32_t rw = (uint32_t)((SPLIT ? (n0 & ~31) + ((n0 & 16) >> 1) : n0) + lr) * P.ldw2;
#pragma unroll
    for (int i = 0; i < BN / 8; i++) off[BM / 8 + i] = rw + (i & 1 ? c1 : c0) + (uint32_t)((SPLIT ? 16 : 8) * i) * P.ldw2;
  }
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)P.a, 0, (int)((uint32_t)(P.M - 1) * P.lda2 + (uint32_t)P.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void*)P.w, 0, (int)((uint32_t)(P.N - 1) * P.ldw2 + (uint32_t)P.K * 2), 0x00020000);
  const int nk = P.K / 64;
  const int nw = (nk - wave + NW - 1) / NW;                // slabs of this wave: wave, wave + NW, ..
  const int lds0 = wave * SLAB;
  auto issue = [&](unsigned char* S, int i) {
    const int ko = (wave + NW * i) * 128;
#pragma unroll
    for (int l = 0; l < BM / 8; l++) load_lds16(rA, S + lds0 + 1024 * l, off[l], ko);
#pragma unroll
    for (int l = BM / 8; l < LOADS; l++) load_lds16(rW, S + lds0 + 1024 * l, off[l], ko);
  };

  // ---- this wave's share of the output, and its residual
  uint2 res[FW];
  int f_of[FW];
#pragma unroll
  for (int i = 0; i < FW; i++) f_of[i] = wave * FW + i;
  if (EPI == 2) {
#pragma unroll
    for (int i = 0; i < FW; i++) {
      const int fi = f_of[i] / FN, fj = f_of[i] % FN;
      const int row = m0 + 16 * fi + r, n = n0 + 16 * fj;
      res[i] = uint2{0u, 0u};
      if (f_of[i] < F && row < P.M && n < P.N) res[i] = *(const uint2*)((const uint16_t*)P.r + (int64_t)row * P.ldr + n + 4 * g);
    }
  }
  if (nw > 0) issue(s0, 0);
  if (R > 1 && nw > 1) issue(s1, 1);

  gf4 acc[FM][FN];
  gf4 sq[FM];   // NORM: the squares of a row are the diagonal of X X^T, one more matrix instruction per fragment
#pragma unroll
  for (int i = 0; i < FM; i++) {
    sq[i] = gf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = gf4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t ld0 = (uint32_t)r * 128 + (uint32_t)((g ^ ((r >> 1) & 7)) << 4), ld1 = (uint32_t)r * 128 + (uint32_t)(((4 + g) ^ ((r >> 1) & 7)) << 4);
  auto slab = [&](unsigned char* S, int i) {
    if (R > 1 && i + 1 < nw) wait_vm<LOADS>(); else wait_vm<0>();   // (loads land in order)
    asm volatile("" ::: "memory");
    const unsigned char* A = S + lds0;
    const unsigned char* B = A + BM * 128;
    gu4 af[2][FM], wf[2][FN];
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int j = 0; j < FN; j++) wf[s][j] = *(const gu4*)(B + 2048 * j + (s ? ld1 : ld0));
#pragma unroll
      for (int f = 0; f < FM; f++) af[s][f] = *(const gu4*)(A + 2048 * f + (s ? ld1 : ld0));
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
        for (int j = 0; j < FN; j++) acc[f][j] = gmfma<DT>(wf[s][j], af[s][f], acc[f][j]);
        if (NORM) sq[f] = gmfma<DT>(af[s][f], af[s][f], sq[f]);
      }
    }
  };
  int i = 0;
  if constexpr (R == 1) {
    for (; i < nw; i++) slab(s0, i);
  } else {
    for (; i + 2 <= nw; i += 2) { slab(s0, i); slab(s1, i + 1); }
    if (i < nw) slab(s0, i);
  }

  // ---- the waves' partial sums meet in LDS
  if (NORM) {
#pragma unroll
    for (int f = 0; f < FM; f++) {   // (lane (r, g) holds elements (4 g + t, r) of X X^T)
      const float v = r & 2 ? (r & 1 ? sq[f][3] : sq[f][2]) : (r & 1 ? sq[f][1] : sq[f][0]);
      if (g == r >> 2) sSS[wave * BM + 16 * f + r] = v;
    }
  }
  auto part = [&](int w, int f) { return (gf4*)(s0 + w * SLAB + 1024 * f) + lane; };   // fragment f of wave w's sums
#pragma unroll
  for (int fi = 0; fi < FM; fi++)
#pragma unroll
    for (int fj = 0; fj < FN; fj++) *part(wave, fi * FN + fj) = acc[fi][fj];
  __syncthreads();
  gf4 o[FW];
  float rn[FW];
#pragma unroll
  for (int q = 0; q < FW; q++) {
    const int f = f_of[q];
    if (F % NW != 0 && f >= F) break;
    gf4 v = *part(0, f);
#pragma unroll
    for (int w = 1; w < NW; w++) v += *part(w, f);
    rn[q] = 1.0f;
    if (NORM) {
      const int rl = 16 * (f / FN) + r;
      float t = sSS[rl];
#pragma unroll
      for (int w = 1; w < NW; w++) t += sSS[w * BM + rl];
      rn[q] = rsqrtf(t / (float)P.K + P.eps);
    }
    o[q] = v;
  }
  if constexpr (EPI == 1 && BN == 16) {
#pragma unroll
    for (int q = 0; q < FW; q++) {
      const int f = f_of[q], row = m0 + 16 * f + r;
      float x[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const float gv = ground<DT>(o[q][t] * rn[q]), uv = __shfl_xor(gv, 32, 64);
        x[t] = silu_round<DT>(gv) * uv;
      }
      if (f >= F || row >= P.M || g >= 2) continue;
      uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + (n0 >> 1) + 4 * g;
      *(uint2*)cp = uint2{gpack<DT>(x[0], x[1]), gpack<DT>(x[2], x[3])};
    }
  } else if constexpr (EPI == 1) {
    if constexpr (FW % 2 == 0) {
#pragma unroll
      for (int q = 0; q < FW; q += 2) {
        const int f = f_of[q], row = m0 + 16 * (f / FN) + r, n = n0 + 16 * (f % FN);
        if (row >= P.M || n >= P.N) continue;
        float x[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const float gv = ground<DT>(o[q][t] * rn[q]), uv = ground<DT>(o[q + 1][t] * rn[q]);
          x[t] = silu_round<DT>(gv) * uv;
        }
        uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + (n >> 1) + 4 * g;
        *(uint2*)cp = uint2{gpack<DT>(x[0], x[1]), gpack<DT>(x[2], x[3])};
      }
    } else {                                               // one fragment per wave: the even ones take their pair's other half
      static_assert(FW == 1, "");
      const int f = f_of[0], row = m0 + 16 * (f / FN) + r, n = n0 + 16 * (f % FN);
      if (f >= F || f % 2 || row >= P.M || n >= P.N) return;
      gf4 u = *part(0, f + 1);
#pragma unroll
      for (int w = 1; w < NW; w++) u += *part(w, f + 1);
      float x[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const float gv = ground<DT>(o[0][t] * rn[0]), uv = ground<DT>(u[t] * rn[0]);
        x[t] = silu_round<DT>(gv) * uv;
      }
      uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + (n >> 1) + 4 * g;
      *(uint2*)cp = uint2{gpack<DT>(x[0], x[1]), gpack<DT>(x[2], x[3])};
    }
  } else {
#pragma unroll
    for (int q = 0; q < FW; q++) {
      const int f = f_of[q], row = m0 + 16 * (f / FN) + r, n = n0 + 16 * (f % FN);
      if (f >= F || row >= P.M || n >= P.N) continue;
      float x[4];
#pragma unroll
      for (int t = 0; t < 4; t++) x[t] = o[q][t] * rn[q];
      if (EPI == 2) {
        float y[4];
        if (DT == UVMI_BF16) {
          y[0] = __uint_as_float(res[q].x << 16); y[1] = __uint_as_float(res[q].x & 0xffff0000u);
          y[2] = __uint_as_float(res[q].y << 16); y[3] = __uint_as_float(res[q].y & 0xffff0000u);
        } else {
          y[0] = half_bits_to_float((uint16_t)(res[q].x & 0xffff)); y[1] = half_bits_to_float((uint16_t)(res[q].x >> 16));
          y[2] = half_bits_to_float((uint16_t)(res[q].y & 0xffff)); y[3] = half_bits_to_float((uint16_t)(res[q].y >> 16));
        }
#pragma unroll
        for (int t = 0; t < 4; t++) x[t] = P.ca * y[t] + P.cb * ground<DT>(x[t]);
      }
      uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + n + 4 * g;
      *(uint2*)cp = uint2{gpack<DT>(x[0], x[1]), gpack<DT>(x[2], x[3])};
    }
  }
}

// (a gate and an up fragment beside each other in every wave's share)
constexpr bool swiglu_tile(int bm, int bn) { return bn == 16 || (bn % 32 == 0 && bm != 48); }

template <int DT, int BM, int BN, int NW, int R>
static void launch_stream(const uvmi_gemm_args* a, StreamParams& P, hipStream_t st) {
  P.tiles_m = (int)((a->M + BM - 1) / BM);
  P.tiles_n = (a->N + BN - 1) / BN;
  const int T = P.tiles_m * P.tiles_n;
  const dim3 grid((unsigned)(((T + 7) / 8) * 8)), blk(64 * NW);
#define UVMI_GO(EPI, NORM) hipLaunchKernelGGL((gemm_stream_kernel<DT, BM, BN, NW, R, EPI, NORM>), grid, blk, 0, st, P.a, P.w, P.lda2, P.ldw2, P.M, P.N, P.K, P.tiles_m, P.tiles_n, P.rowsplit, P.r, P.c, P.ldc, P.ldr, P.eps, P.ca, P.cb)
  const bool norm = a->norm_a != 0;
  if (a->epilogue == UVMI_GEMM_SWIGLU) {
    if constexpr (swiglu_tile(BM, BN)) { if (norm) UVMI_GO(1, true); else UVMI_GO(1, false); }
  } else if constexpr (BN != 96) {   // (which serves SWIGLU alone)
    if (a->epilogue == UVMI_GEMM_RESID) { if (norm) UVMI_GO(2, true); else UVMI_GO(2, false); }
    else { if (norm) UVMI_GO(0, true); else UVMI_GO(0, false); }
  }
#undef UVMI_GO
}

// The tiles, by the rows of A and W that they load: (BM, BN, NW, R).  LDS: 64, 48, 64, 80, 96 / 48, 112, 64, 158 (159 with NORM, of 160), 96 KB.  The smallest
// tile takes 8 waves (K of 512 or 640: one or two slabs each, all in flight at once).
constexpr int TILE_M[9] = {16, 16, 32, 32, 32, 48, 64, 64, 64}, TILE_N[9] = {16, 32, 32, 48, 64, 64, 64, 80, 96};
constexpr int FORM_64 = 6, FORM_96 = 8;
template <int DT>
static void launch_form(const uvmi_gemm_args* a, int form, bool single_round, StreamParams& P, hipStream_t st) {
  switch (form) {
    case 0: launch_stream<DT, 16, 16, 8, 2>(a, P, st); break;
    case 1: launch_stream<DT, 16, 32, 4, 2>(a, P, st); break;
    case 2: launch_stream<DT, 32, 32, 4, 2>(a, P, st); break;
    case 3: launch_stream<DT, 32, 48, 4, 2>(a, P, st); break;
    case 4:   // two slabs per wave ahead where a compute unit has one workgroup; else one, and three workgroups fit (384 rows, N 3328: 7.3 against 11.3 us)
      if (single_round) launch_stream<DT, 32, 64, 4, 2>(a, P, st);
      else launch_stream<DT, 32, 64, 4, 1>(a, P, st);
      break;
    case 5: launch_stream<DT, 48, 64, 4, 2>(a, P, st); break;
    case 7: launch_stream<DT, 64, 80, 4, 2>(a, P, st); break;
    case FORM_96: launch_stream<DT, 64, 96, 4, 1>(a, P, st); break;
    default: launch_stream<DT, 64, 64, 4, 1>(a, P, st); break;
  }
}

static int64_t stream_tiles(const uvmi_gemm_args* a, int form) {
  return ((a->M + TILE_M[form] - 1) / TILE_M[form]) * ((a->N + TILE_N[form] - 1) / TILE_N[form]);
}

// The smallest tile that leaves a compute unit one workgroup: a launch lasts as long as a unit takes to load its tiles' rows, about 0.055 us
// a row at K 1664, and larger tiles leave units idle.  (640 columns, K 1664: 384 rows, 32 x 32, 64 rows of operands a unit, 5.4 us; 512 rows,
// where those come to 320 tiles, 7.4, 32 x 48, 80 rows, 6.0, 32 x 64 6.8; 1024 rows 48 x 64 7.7, 64 x 64 8.8; 2048 rows 64 x 80 9.8, two rounds of 64 x 64
// 12.4.  K 512: 512 rows 32 x 32 4.4, 32 x 48 4.0; 2048 rows 64 x 80 6.1, 64 x 64 6.9.)  Of the two smallest a short K ends before a second
// workgroup on the unit hurts: 7 / 4 per unit up to K = 768 (K 512, 256 rows: 16 x 32, 320 tiles, 3.0 us; 32 x 32, 160 tiles, 3.1); nor does it with
// 32 x 64 ones where 48 x 64 come to more than one (1280 rows 5.3, 64 x 64 5.5).  So with SWIGLU,
// whose tiles are multiples of 32 wide (N 3328, 256 rows: 32 x 64, 416 tiles, 5.9, 64 x 64 6.0), unless 64 x 96 ones fill one round where
// 64 x 64 ones begin a second (448 rows 7.2, 64 x 64 7.7; 320 rows 7.1 and 7.4).
// -1: more than that of every tile.
int gemm_stream_form(const uvmi_gemm_args* a, int cus) {
  const int64_t most = a->K <= 768 ? (int64_t)cus * 7 / 4 : cus;
  if (a->epilogue == UVMI_GEMM_SWIGLU) {
    for (int f = 0; f < FORM_64; f++)
      if (swiglu_tile(TILE_M[f], TILE_N[f]) && stream_tiles(a, f) <= most) return f;
    const int64_t t = stream_tiles(a, FORM_64);
    if (t > cus && stream_tiles(a, FORM_96) <= cus) return FORM_96;
    return t <= most ? FORM_64 : -1;
  }
  for (int f = 0; f < FORM_64; f++)
    if (stream_tiles(a, f) <= (f < 2 ? most : cus)) return f;
  if (stream_tiles(a, 4) <= most) return 4;
  for (int f = FORM_64; f < FORM_96; f++)
    if (stream_tiles(a, f) <= cus) return f;
  return -1;
}

void gemm_stream_tile(int form, int* rows, int* cols) { *rows = TILE_M[form]; *cols = TILE_N[form]; }

// Arguments are validated by the caller (uvmi_gemm_tn_ex).
void gemm_stream_launch(const uvmi_gemm_args* a, int form, int cus, hipStream_t st) {
  StreamParams P;
  P.a = a->a; P.w = a->w; P.c = a->c; P.r = a->resid;
  P.lda2 = (uint32_t)a->lda * 2; P.ldw2 = (uint32_t)a->ldw * 2; P.ldc = a->ldc; P.ldr = a->ldr;
  P.M = (int)a->M; P.N = a->N; P.K = a->K;
  P.eps = a->eps; P.ca = a->ca; P.cb = a->cb;
  // tiles are dealt to the XCDs in contiguous runs, by row blocks or by weight strips, whichever leaves the smaller working set
  // per XCD (an eighth of A plus all of W, or all of A plus an eighth of W)
  const double bytes_a = (double)a->M * a->K, bytes_w = (double)a->N * a->K;
  P.rowsplit = bytes_a / 8 + bytes_w < bytes_a + bytes_w / 8;
  const bool single_round = stream_tiles(a, form) <= cus;
  if (a->dtype == UVMI_F16) launch_form<UVMI_F16>(a, form, single_round, P, st);
  else launch_form<UVMI_BF16>(a, form, single_round, P, st);
}

}  // namespace uvmi
