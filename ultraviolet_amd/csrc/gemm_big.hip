// 16-bit GEMM for passes of many thousand rows (a packed prefill, a mixed prefill + decode pass): the same product and
// epilogues as the tiled kernel of gemm_tile.hip - C[M, N] = A[M, K] . W[N, K]^T with fp32 accumulation, SwiGLU on
// interleaved gate / up slabs, the block's residual update, the RMS pre-norm as a row scale (the F.linear calls of the
// reference's fused inference path, ultraviolet/model.py:302-335, 388-391, with what surrounds them, :566-571) - on a
// 256 x 256 tile.
//
// What bounds a GEMM of this size on gfx950 is not the matrix cores but what feeds them.  Measured on the part: a compute
// unit takes ~52 bytes per clock from the L2 when every request is a whole 128-byte line and half of that when requests
// are 64-byte row segments, and its LDS delivers ~128 bytes per clock.  Hence:
//   * a workgroup of 8 waves (2 x 4) owns a 256 x 256 tile, a wave 128 x 64 of it: per K-step of 32 a wave reads 12 operand
//     fragments from LDS for 32 MFMAs (the 64 x 64 wave tile of the smaller kernels reads 8 for 16), and the tile takes
//     half the L2 bytes per flop of a 128 x 128 tile;
//   * K is walked in slabs of 64: a row's share of a slab is one whole 128-byte line;
//   * slabs go from global memory straight into LDS (buffer loads, 16 bytes per lane): no staging registers, no LDS
//     store instructions, and 32-bit offsets where global loads keep eight 64-bit addresses per lane (33 216-row gate-up without the
//     norm 152 -> 149 us).  A wave-load lands as 1 KB of consecutive LDS - 8 rows of 128 bytes - so the xor swizzle that
//     keeps the operand reads conflict-free (16-byte chunk index ^ (row / 2) % 8) is applied on the global side: lane l
//     of a load fetches the chunk that belongs at physical position l % 8 of its row;
//   * two LDS stages of 64 KB (A and W slab each 256 rows x 128 B).  An iteration multiplies slab k out of one stage while
//     slab k + 1 lands in the other; its operand reads run one MFMA group (8 MFMAs) ahead of their use, and before its
//     last group it waits for slab k + 1, refills its own stage with slab k + 2 and requests slab k + 1's first operands:
//     one barrier per slab, no bubble between slabs;
//   * the accumulator holds C^T fragments (a lane has 4 consecutive columns of one row); the epilogue converts and swaps
//     lanes so that the 4 lane groups of a row store 64 consecutive bytes (RESID: 16 columns per lane).  fp32 logits are
//     stored as they lie: 4 columns are 16 bytes (512 x 32768 with the softcap 52.8 us behind the 4 x 4 transpose, 47.7 so,
//     33.7 on 256 x 256 tiles; 128 rows 17.8 / 14.2; 256 rows 24.2 / 18.0);
//   * the residual of the whole tile is requested at once behind the main loop, ahead of the first store (in place it may not be
//     moved across one by the compiler, and was requested row block by row block: 18 432 x 640 x 512 27.9 -> 23.8 us, x 1664 53.8 ->
//     50.8; 33 216 rows in 128 x 128 tiles 47.7 -> 45.3, 98.4 -> 96.7);
//   * a pass of more tiles than run at a time (K a multiple of 128) has a workgroup take several: the next tile's first two slabs are
//     requested in a tile's last two iterations, so they land under its epilogue (33 216-row gate-up 165 -> 160 us, without the norm 150 ->
//     142; 128 x 128 tiles 174 -> 161; 640 columns, K 1664, 97 -> 94).  Per-tile constants of the lane are computed anew between
//     tiles: there is no register for them in the main loop, and a spilled one is reloaded behind the loads in flight;
//   * the pre-norm's sums of squares are matrix instructions too, one for 16 rows and 32 columns, a sixteenth of the product's
//     (gate-up at 33 216 rows 160 -> 154 us, at 18 432 rows 96 -> 90; as vector instructions between the matrix ones they cost 12 % of
//     a launch, in 128 x 128 tiles 14 %: 177 -> 169).  The results' distance from 64 bits is the same to seven digits, K 512 .. 2560;
//   * in a pass of many rows they are not formed here at all: the residual updates leave them where they write the hidden (uvmi_gemm_sums;
//     gate-up at 33 216 rows 144 -> 133 us, at 18 432 rows 86 -> 79; without any norm 128 and 77).  Against 64 bits the products are as before
//     (2-norms of the error over 12 288 .. 40 000 rows, K 256 .. 1024, equal to eight digits, fp16 to six, the smaller of the two);
//   * no loads are made past the last slab (they were, to keep the loop free of branches: the epilogue then waited for them;
//     1 - 3 % of a launch);
//   * tiles are dealt to the XCDs in contiguous runs, as in the tiled kernel; a workgroup's tiles are a stride apart in its XCD's run.
// One workgroup per compute unit (128 KB of LDS, 2 waves per SIMD).  K >= 128; C and the residual 16-byte aligned with
// pitches that are multiples of 8 elements (the caller checks).
#include "common.h"
#include "gemm_util.h"
#include "qkv_post.h"

namespace uvmi {

struct BigParams {
  const void* a; const void* w; void* c; const void* r;
  uint32_t lda2, ldw2;  // row pitches in bytes
  int64_t ldc, ldr;     // elements
  int M, N, K, tiles_m, tiles_n;
  int rowsplit;
  float eps, ca, cb, cap_c;
  float* sums; uint32_t sums_ld4; int parts;   // NORM 2: read; EPI 2 (or null): written.  parts x sums_ld4 bytes
  QueryPost q;                                 // EPI 4
  HeadRows h;                                  // EPI 3
};
constexpr int SUM_PARTS = 16;

// Two dwords x, y per lane in lane groups g = lane / 16 (x0 .. x3, y0 .. y3) -> x = (x0, x2, y0, y2), y = (x1, x3, y1, y3).
// (permlane32_swap exchanges the upper 32 lanes of its first operand with the lower 32 of its second, permlane16_swap does the
// same inside each half.)
__device__ __forceinline__ void xpose_pair(uint32_t& x, uint32_t& y) {
  auto s = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  auto t = __builtin_amdgcn_permlane16_swap(s[0], s[1], false, false);
  x = t[0]; y = t[1];
}
// 4 x 4 transpose of one dword per (register j, lane group g = lane / 16): afterwards register j of group g holds what
// register g of group j held.
__device__ __forceinline__ void xpose4(uint32_t (&x)[4]) {
  auto s0 = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
  auto s1 = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
  x[0] = s0[0]; x[2] = s0[1]; x[1] = s1[0]; x[3] = s1[1];
  auto t0 = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
  auto t1 = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
  x[0] = t0[0]; x[1] = t0[1]; x[2] = t1[0]; x[3] = t1[1];
}
// 2 x 2 transpose between (register j, lane / 16 % 2)
__device__ __forceinline__ void xpose2(uint32_t& x0, uint32_t& x1) {
  auto t = __builtin_amdgcn_permlane16_swap(x0, x1, false, false);
  x0 = t[0]; x1 = t[1];
}

// The lane, computed anew: what is derived from it does not stay in registers across a tile's main loop, which has none to spare.
__device__ __forceinline__ int fresh_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

// EPI 0: C = A W^T (M, N).  EPI 1: W rows are [gate 16 | up 16] slabs; C = silu(gate) * up, (M, N / 2).
// EPI 2: C = ca * R + cb * (A W^T).  EPI 3: C fp32 = ca * sigmoid((x + cb) / cap_c) of the rounded product x, of rows of A that
// h.rows names (or all), with h.advance counted up behind it.  NORM: A stands
// for its RMS-normalised rows, whose squares are summed here (1) or were by the launches that wrote them (2: a number per row and 64
// columns, which an EPI 2 launch leaves).
// EPI 4: EPI 0 whose columns 0 .. 511, a wave's 64 of them a query head, are normed, rotated (QK-norm and RoPE, with the roundings of
// qkv_post_rows_kernel) and go to q.out: 18 432 rows 21.7 -> 25.8 us on 256 x 256 tiles, 33 216 rows 39.2 -> 45.5 on 128 x 128 ones, where an epilogue
// runs beside another workgroup's main loop.
// FI: 16-row fragments per wave along M: 8 - the 256 x 256 tile on 8 waves (2 x 4); 6 - 192 x 128 on 4 waves (2 x 2, 96 x 64 per wave, two
// workgroups per compute unit; no pre-norm); 4 - a 128 x 128 tile on 4 waves (64 x 64 per wave, two workgroups per compute unit) for passes whose 256 x 256 tiles would not fill the device.  (A
// 64 x 64 tile on 2 waves was measured too: no faster at 2 k rows than 64 x 64 tiles staged through registers.)
// MANY: a workgroup takes several tiles (an even number of slabs: a tile ends on the stage that it does not begin on).
template <int FI> constexpr int BIG_THREADS = FI == 8 ? 512 : 256;
template <int DT, int EPI, int NORM, int FI, bool MANY>
__global__ __launch_bounds__(BIG_THREADS<FI>) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_big_kernel(BigParams P) {
  constexpr int WN = BIG_THREADS<FI> / 128;    // waves along N (2 along M)
  constexpr int BM = 32 * FI, BN = 64 * WN, LA = BM / (16 * WN);   // LA: a wave's loads of A per slab (of W: 4)
  static_assert(NORM != 1 || FI / 2 == WN, "a wave along N for every pair of a wave's row fragments");
  // one array per stage and operand: the compiler can then tell that the operand reads of one stage do not touch the
  // stage a load in flight is writing, and does not wait for that load
  __shared__ __attribute__((aligned(1024))) unsigned char sA0[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char sA1[BM * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char sB0[BN * 128];
  __shared__ __attribute__((aligned(1024))) unsigned char sB1[BN * 128];
  __shared__ float sRS[NORM ? BM : 1];
  __shared__ __attribute__((aligned(1024))) unsigned char sPart[NORM == 2 ? SUM_PARTS * BM * 4 : 4];
  __shared__ __attribute__((aligned(1024))) unsigned char sPos[EPI == 4 ? BM * 8 : 4];
  __shared__ int sAt[EPI == 4 ? BM : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T = P.tiles_m * P.tiles_n;
  const int per = (T + 7) / 8;
  // the workgroup's tiles: every gridDim.x / 8 th of its XCD's run
  const int step = (int)(gridDim.x / 8), last = min((int)(blockIdx.x % 8 + 1) * per, T);
  int L = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (L >= last) return;
  const int nk = P.K / 64;
  int m0, n0;
  auto tile_at = [&](int l) {
    const int bn = P.rowsplit ? l % P.tiles_n : l / P.tiles_m, bm = P.rowsplit ? l / P.tiles_n : l % P.tiles_m;
    m0 = bm * BM;
    n0 = bn * BN;
  };
  tile_at(L);

  // ---- loader: wave w fills blocks LA w .. of A and 4 w .. 4 w + 3 of W (8 rows each).  Rows past M / N repeat the last row: what they
  // produce is never stored.
  uint32_t offA[LA], offB[4];
  auto offsets = [&]() {
    const int ln = fresh_lane();
#pragma unroll
    for (int i = 0; i < LA; i++) {
      const int rl = 8 * (LA * wave + i) + (ln >> 3);   // row inside the tile
      int m = min(m0 + rl, P.M - 1);
      if (EPI == 3 && P.h.rows) m = (int)min(max(P.h.rows[m], (int64_t)0), (int64_t)P.h.a_rows - 1);
      offA[i] = (uint32_t)m * P.lda2 + 16 * ((ln & 7) ^ ((rl >> 1) & 7));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int rl = 8 * (4 * wave + i) + (ln >> 3);
      offB[i] = (uint32_t)min(n0 + rl, P.N - 1) * P.ldw2 + 16 * ((ln & 7) ^ ((rl >> 1) & 7));
    }
  };
  offsets();
  // (buffer loads: 32-bit offsets and the slab as a scalar, where global ones keep eight 64-bit addresses)
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)P.a, 0, (int)((uint32_t)((EPI == 3 && P.h.rows ? P.h.a_rows : P.M) - 1) * P.lda2 + (uint32_t)P.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void*)P.w, 0, (int)((uint32_t)(P.N - 1) * P.ldw2 + (uint32_t)P.K * 2), 0x00020000);
  auto issue = [&](unsigned char* sa, unsigned char* sb, int kt) {
#pragma unroll
    for (int i = 0; i < LA; i++)
      load_lds16(rA, sa + (LA * wave + i) * 1024, offA[i], kt * 128);
#pragma unroll
    for (int i = 0; i < 4; i++)
      load_lds16(rW, sb + (4 * wave + i) * 1024, offB[i], kt * 128);
  };

  // ---- reader: wave (wm, wn) owns rows 16 FI wm .., columns 64 wn ..; lane (r, g) reads chunk (4 s + g) ^ ((r / 2) % 8) of
  // row r of a 16-row fragment for K-step s
  const int wm = wave / WN, wn = wave % WN;
  // The wave's pairs of row fragments are walked from pair wn on (NORM; accumulator rows 2 p, 2 p + 1 belong to pair (p + wn) mod
  // FI / 2), so that the rows whose squares a wave sums are the same in the code of every wave.
  constexpr int NP = FI / 2;
  uint32_t a_off[2], b_off[2], pair_at[NP];
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const uint32_t lo = (uint32_t)(lane & 15) * 128 + (uint32_t)((((4 * s + (lane >> 4)) ^ ((lane >> 1) & 7))) << 4);
    a_off[s] = (uint32_t)wm * (16 * FI * 128) + lo;
    b_off[s] = (uint32_t)wn * 8192 + lo;
  }
#pragma unroll
  for (int p = 0; p < NP; p++) pair_at[p] = (uint32_t)(NORM == 1 ? ((p + wn) & (NP - 1)) : p) * 4096;
  gf4 acc[FI][4];

  gu4 w0[4], w1[4], f0[2], f1[2], f2[2];
  auto read_b = [&](const unsigned char* sb, int s, gu4* w) {
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = *(const gu4*)(sb + b_off[s] + j * 2048);
  };
  auto read_a = [&](const unsigned char* sa, int s, int i, gu4* f) {
    uint32_t o;
    if constexpr (NORM == 1) asm volatile("v_add_u32 %0, %1, %2" : "=v"(o) : "s"(pair_at[i / 2]), "v"(a_off[s]));   // (kept out of registers between uses)
    else o = a_off[s] + pair_at[i / 2];
    f[0] = *(const gu4*)(sa + o);
    f[1] = *(const gu4*)(sa + o + 2048);
  };
  // (the MFMA's A input is the weight fragment, its B input the activation fragment: the accumulator holds C^T)
  auto mm1 = [&](int i, const gu4* f, const gu4* w) { acc[i][0] = gmfma<DT>(w[0], f[0], acc[i][0]); };
  auto mm7 = [&](int i, const gu4* f, const gu4* w) {
#pragma unroll
    for (int j = 1; j < 4; j++) acc[i][j] = gmfma<DT>(w[j], f[0], acc[i][j]);
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i + 1][j] = gmfma<DT>(w[j], f[1], acc[i + 1][j]);
  };
  // NORM: the squares of a row are the diagonal of X X^T: one more matrix instruction on an operand fragment with itself per 16 rows and
  // K-step.  Wave (wm, wn) takes row pair wn (rows 16 FI wm + 32 wn + 16 u + r, u = 0, 1),
  // which is its first pair (as a branch on wn it costs 4 us of 157).
  gf4 sq[2];
  auto sumsq = [&](int pair, const gu4* f) {
    if (NORM == 1 && pair == 0) {
#pragma unroll
      for (int u = 0; u < 2; u++) sq[u] = gmfma<DT>(f[u], f[u], sq[u]);
    }
  };
  auto frow = [&](int i) { return 16 * FI * wm + 16 * (NORM == 1 ? ((i + 2 * wn) & (FI - 1)) : i); };   // first tile row of accumulator row fragment i
#define UVMI_SB() __builtin_amdgcn_sched_barrier(0)

  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) acc[i][j] = gf4{0.f, 0.f, 0.f, 0.f};
    sq[0] = sq[1] = gf4{0.f, 0.f, 0.f, 0.f};
  };
  // NORM 2: the sums of the tile's rows, SUM_PARTS x BM, on their way with its first slab, and its scales, formed behind its first barrier, when all
  // waves are past the epilogue before; EPI 4: likewise the rows' positions and what they point to in the table (requested there the sums were waited for, added up in the epilogue they held it: 4 - 7 us
  // of 80 - 140)
  auto issue_sums = [&]() {
    if constexpr (NORM == 2) {
      const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc((void*)P.sums, 0, (int)(P.parts * P.sums_ld4), 0x00020000);
      const int ln = fresh_lane();
      for (int b = wave; b * 256 < P.parts * BM; b += 2 * WN)
        load_lds16(rS, sPart + b * 1024, (uint32_t)((b * 256 + 4 * ln) / BM) * P.sums_ld4 + 4 * (m0 + (b * 256 + 4 * ln) % BM), 0);
    }
    if constexpr (EPI == 4) {
      const __amdgpu_buffer_rsrc_t rP = __builtin_amdgcn_make_buffer_rsrc((void*)P.q.pos, 0, P.M * 8, 0x00020000);
      if (wave < BM / 128) load_lds16(rP, sPos + wave * 1024, (uint32_t)m0 * 8 + 1024 * wave + 16 * fresh_lane(), 0);
    }
  };
  auto scales = [&]() {
    if constexpr (NORM == 2) {
      if (wave < BM / 64) {   // (two lanes a row, for half of the numbers each, in batches: no faster)
        const int row = 64 * wave + fresh_lane();
        float v = 0.f;
        for (int p = 0; p < P.parts; p++) v += ((const float*)sPart)[p * BM + row];
        sRS[row] = rsqrtf(v / (float)P.K + P.eps);
      }
    }
    if constexpr (EPI == 4) {
      if (wave < BM / 64) {
        const int row = 64 * wave + fresh_lane();
        const int64_t p = ((const int64_t*)sPos)[row];
        sAt[row] = P.q.tab && p >= 0 && p < P.q.rope_n ? (int)p * 128 : -1;   // (bytes)
      }
    }
  };
  issue(sA0, sB0, 0);
  issue_sums();
  clear();
#pragma unroll
  for (int i = 0; i < FI; i++) asm volatile("" : "+v"(acc[i][0]), "+v"(acc[i][1]), "+v"(acc[i][2]), "+v"(acc[i][3]));   // (while the loads are on their way)
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  issue(sA1, sB1, 1);
  for (;;) {   // tiles
    const int cm0 = m0, cn0 = n0;
    const bool more = MANY && L + step < last;
    // slab k of this tile or, past its last one, slab k - nk of the next
    auto request = [&](unsigned char* sa, unsigned char* sb, int k) {
      if (k < nk) issue(sa, sb, k);
      else if (more) {
        if (k == nk) { tile_at(L + step); offsets(); issue_sums(); }
        issue(sa, sb, k - nk);
      }
    };
    read_b(sB0, 0, w0);
    read_a(sA0, 0, 0, f0);
    // Iteration k multiplies slab k out of stage S: 8 groups of 8 MFMAs (K-step s, row pair p); the operands of a group are
    // requested behind the first MFMA of the group before it, so a wait for them comes seven MFMAs after their request.
    // Before the last group: slab k + 1 has landed in the other stage (own loads: the wait; the other waves': the barrier)
    // and every read of stage S is complete, so S is refilled with slab k + 2 and the first operands of slab k + 1 are
    // requested.
#define UVMI_ITER(SA, SB_, SAN, SBN, k)                                                                                  \
  do {                                                                                                                   \
    mm1(0, f0, w0); UVMI_SB(); read_a(SA, 0, 2, f1); UVMI_SB(); mm7(0, f0, w0); sumsq(0, f0); UVMI_SB();                 \
    mm1(2, f1, w0); UVMI_SB(); read_a(SA, 0, 4, f2); UVMI_SB(); mm7(2, f1, w0); sumsq(1, f1); UVMI_SB();                 \
    mm1(4, f2, w0); UVMI_SB(); read_a(SA, 0, 6, f0); UVMI_SB(); mm7(4, f2, w0); sumsq(2, f2); UVMI_SB();                 \
    mm1(6, f0, w0); UVMI_SB(); read_b(SB_, 1, w1); read_a(SA, 1, 0, f1); UVMI_SB(); mm7(6, f0, w0); sumsq(3, f0); UVMI_SB(); \
    mm1(0, f1, w1); UVMI_SB(); read_a(SA, 1, 2, f2); UVMI_SB(); mm7(0, f1, w1); sumsq(0, f1); UVMI_SB();                 \
    mm1(2, f2, w1); UVMI_SB(); read_a(SA, 1, 4, f0); UVMI_SB(); mm7(2, f2, w1); sumsq(1, f2); UVMI_SB();                 \
    mm1(4, f0, w1); UVMI_SB(); read_a(SA, 1, 6, f1); UVMI_SB(); mm7(4, f0, w1); sumsq(2, f0); UVMI_SB();                 \
    __builtin_amdgcn_s_waitcnt(0x0f70);                                                                                  \
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                                                      \
    request(SA, SB_, (k) + 2);                                                                                           \
    read_b(SBN, 0, w0); read_a(SAN, 0, 0, f0); UVMI_SB();                                                                \
    mm1(6, f1, w1); mm7(6, f1, w1); sumsq(3, f1); UVMI_SB();                                                             \
  } while (0)
    // FI = 4: 4 groups per slab; the first operands of the next slab arrive in the buffer the iteration's second group used,
    // so two iterations alternate the roles of f0 and f1
#define UVMI_ITER4(SA, SB_, SAN, SBN, k, X, Y)                                                                           \
  do {                                                                                                                   \
    mm1(0, X, w0); UVMI_SB(); read_a(SA, 0, 2, Y); UVMI_SB(); mm7(0, X, w0); sumsq(0, X); UVMI_SB();                     \
    mm1(2, Y, w0); UVMI_SB(); read_b(SB_, 1, w1); read_a(SA, 1, 0, f2); UVMI_SB(); mm7(2, Y, w0); sumsq(1, Y); UVMI_SB(); \
    mm1(0, f2, w1); UVMI_SB(); read_a(SA, 1, 2, X); UVMI_SB(); mm7(0, f2, w1); sumsq(0, f2); UVMI_SB();                  \
    __builtin_amdgcn_s_waitcnt(0x0f70);                                                                                  \
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                                                      \
    request(SA, SB_, (k) + 2);                                                                                           \
    read_b(SBN, 0, w0); read_a(SAN, 0, 0, Y); UVMI_SB();                                                                 \
    mm1(2, X, w1); mm7(2, X, w1); sumsq(1, X); UVMI_SB();                                                                \
  } while (0)
    // FI = 6: 6 groups per slab, whose operands take the three buffers in turn
#define UVMI_ITER6(SA, SB_, SAN, SBN, k)                                                                                 \
  do {                                                                                                                   \
    mm1(0, f0, w0); UVMI_SB(); read_a(SA, 0, 2, f1); UVMI_SB(); mm7(0, f0, w0); UVMI_SB();                               \
    mm1(2, f1, w0); UVMI_SB(); read_a(SA, 0, 4, f2); UVMI_SB(); mm7(2, f1, w0); UVMI_SB();                               \
    mm1(4, f2, w0); UVMI_SB(); read_b(SB_, 1, w1); read_a(SA, 1, 0, f0); UVMI_SB(); mm7(4, f2, w0); UVMI_SB();           \
    mm1(0, f0, w1); UVMI_SB(); read_a(SA, 1, 2, f1); UVMI_SB(); mm7(0, f0, w1); UVMI_SB();                               \
    mm1(2, f1, w1); UVMI_SB(); read_a(SA, 1, 4, f2); UVMI_SB(); mm7(2, f1, w1); UVMI_SB();                               \
    __builtin_amdgcn_s_waitcnt(0x0f70);                                                                                  \
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                                                      \
    request(SA, SB_, (k) + 2);                                                                                           \
    read_b(SBN, 0, w0); read_a(SAN, 0, 0, f0); UVMI_SB();                                                                \
    mm1(4, f2, w1); mm7(4, f2, w1); UVMI_SB();                                                                           \
  } while (0)
    int k = 0;
    if constexpr (FI == 6) {
      for (; k + 2 <= nk; k += 2) {
        UVMI_ITER6(sA0, sB0, sA1, sB1, k);
        UVMI_ITER6(sA1, sB1, sA0, sB0, k + 1);
      }
      if (!MANY && k < nk) UVMI_ITER6(sA0, sB0, sA1, sB1, k);
    } else if constexpr (FI == 8) {
      for (; k + 2 <= nk; k += 2) {
        UVMI_ITER(sA0, sB0, sA1, sB1, k);
        if ((NORM == 2 || EPI == 4) && k == 0) scales();
        UVMI_ITER(sA1, sB1, sA0, sB0, k + 1);
      }
      if (!MANY && k < nk) UVMI_ITER(sA0, sB0, sA1, sB1, k);
    } else {
      for (; k + 2 <= nk; k += 2) {
        UVMI_ITER4(sA0, sB0, sA1, sB1, k, f0, f1);
        if ((NORM == 2 || EPI == 4) && k == 0) scales();
        UVMI_ITER4(sA1, sB1, sA0, sB0, k + 1, f1, f0);
      }
      if (!MANY && k < nk) UVMI_ITER4(sA0, sB0, sA1, sB1, k, f0, f1);
    }
#undef UVMI_ITER4
#undef UVMI_ITER6
#undef UVMI_ITER
#undef UVMI_SB

    const int el = fresh_lane(), r = el & 15, g = el >> 4;
    // ---- row scales of the pre-norm: the 4 lane groups of a row add their sums; LDS carries the scales to every wave
    float rn[FI];
#pragma unroll
    for (int i = 0; i < FI; i++) rn[i] = 1.0f;
    if constexpr (NORM == 2) {
#pragma unroll
      for (int i = 0; i < FI; i++) rn[i] = sRS[frow(i) + r];
    } else if constexpr (NORM == 1) {
      int kd = P.K;
      asm volatile("" : "+s"(kd));   // (not a register of its own through the main loop)
#pragma unroll
      for (int u = 0; u < 2; u++) {   // (lane (r, g) holds elements (4 g + t, r) of X X^T)
        const float v = r & 2 ? (r & 1 ? sq[u][3] : sq[u][2]) : (r & 1 ? sq[u][1] : sq[u][0]);
        if (g == r >> 2) sRS[16 * FI * wm + 32 * wn + 16 * u + r] = rsqrtf(v / (float)kd + P.eps);
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int i = 0; i < FI; i++) rn[i] = sRS[frow(i) + r];
    }

    // ---- EPI 4: rotations of row fragment i + 1 on their way while fragment i is finished
    const bool head = EPI == 4 && cn0 + 64 * wn < 512;
    int at[2];
    float4 cs[2], sn[2];
    auto rotation = [&](int i) {
      at[i & 1] = sAt[EPI == 4 ? frow(i) + r : 0];
      if (!P.q.tab) return;
      const float* t = (const float*)((const char*)P.q.tab + (uint32_t)max(at[i & 1], 0)) + 4 * g;
      cs[i & 1] = *(const float4*)t;
      sn[i & 1] = *(const float4*)(t + 16);
    };
    if (EPI == 4 && head) rotation(0);

    // ---- epilogue: accumulator (i, j): lane (r, g) holds C[m0 + 16 FI wm + 16 i + r][n0 + 64 wn + 16 j + 4 g + t], t = 0..3
    uint4 res[EPI == 2 ? FI : 1][2];
    if constexpr (EPI == 2) {
      const int n = cn0 + 64 * wn + 16 * g;
#pragma unroll
      for (int i = 0; i < FI; i++) {
        const int row = cm0 + frow(i) + r;
        res[i][0] = res[i][1] = uint4{0u, 0u, 0u, 0u};
        if (row < P.M && n < P.N) {
          const uint16_t* rp = (const uint16_t*)P.r + (int64_t)row * P.ldr + n;
          res[i][0] = *(const uint4*)rp;
          res[i][1] = *(const uint4*)(rp + 8);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < FI; i++) {
      const int row = cm0 + frow(i) + r;
      if (EPI == 1) {
        // gate slab j, up slab j + 1 -> 4 outputs per slab pair; after the 2 x 2 transpose lane (r, g) holds the 8 consecutive
        // output columns 16 (g % 2) + 8 (g / 2) .. of the wave's 32
        uint32_t x0[2], x1[2];
#pragma unroll
        for (int jp = 0; jp < 2; jp++) {
          const gf4 gv = acc[i][2 * jp] * rn[i], uv = acc[i][2 * jp + 1] * rn[i];
          (jp == 0 ? x0 : x1)[0] = gswiglu2<DT>(gv[0], gv[1], uv[0], uv[1]);
          (jp == 0 ? x0 : x1)[1] = gswiglu2<DT>(gv[2], gv[3], uv[2], uv[3]);
        }
        xpose2(x0[0], x1[0]);
        xpose2(x0[1], x1[1]);
        const int n = (cn0 >> 1) + 32 * wn + 16 * (g & 1) + 8 * (g >> 1);   // output column
        if (row < P.M && 2 * n < P.N) {
          uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + n;
          *(uint4*)cp = uint4{x0[0], x0[1], x1[0], x1[1]};
        }
      } else if (EPI == 3) {   // fp32: 4 columns are 16 bytes, the 4 lane groups of a row store 64 consecutive ones
        // (the hardware's exponential and reciprocal, with one scale for -x log2(e) / c: over every 16-bit x of the softcap's range 2.40e-8
        // from 64 bits in the 2-norm and 5.5e-7 at most; an exact quotient, expf and a division, as torch's expression has, 2.42e-8 and 6.4e-7)
        const float k2 = -1.4426950408889634f / P.cap_c;
        auto cap = [&](float x) { return P.ca * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f((ground<DT>(x * rn[i]) + P.cb) * k2)); };
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int n = cn0 + 64 * wn + 16 * j + 4 * g;
          if (row < P.M && n < P.N)
            *(float4*)((float*)P.c + (int64_t)row * P.ldc + n) = float4{cap(acc[i][j][0]), cap(acc[i][j][1]), cap(acc[i][j][2]), cap(acc[i][j][3])};
        }
      } else if (EPI == 0 || EPI == 4) {
        uint32_t w[4][2];   // columns 16 j + 4 g ..
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const gf4 v = acc[i][j] * rn[i];
          w[j][0] = gpack<DT>(v[0], v[1]);
          w[j][1] = gpack<DT>(v[2], v[3]);
        }
        if constexpr (EPI == 4) {
          if (head) {
            if (i + 1 < FI) rotation(i + 1);
            auto round2 = [](float& a, float& b) { gunpack<DT>(gpack<DT>(a, b), a, b); };
            float x[4][4], ss = 0.f;
#pragma unroll
            for (int j = 0; j < 4; j++) {
              gunpack<DT>(w[j][0], x[j][0], x[j][1]);
              gunpack<DT>(w[j][1], x[j][2], x[j][3]);
#pragma unroll
              for (int t = 0; t < 4; t++) ss = fmaf(x[j][t], x[j][t], ss);
            }
            const float rs = rsqrtf(xsum32(xsum16(ss)) * (1.0f / 64.0f) + P.q.eps);
#pragma unroll
            for (int j = 0; j < 4; j++) {
              w[j][0] = gpack<DT>(x[j][0] * rs, x[j][1] * rs);
              w[j][1] = gpack<DT>(x[j][2] * rs, x[j][3] * rs);
            }
            if (at[i & 1] >= 0) {   // dims d and d + 16, columns of fragments 0 and 1 (rope_rot, two at a time)
              const float c4[4] = {cs[i & 1].x, cs[i & 1].y, cs[i & 1].z, cs[i & 1].w}, s4[4] = {sn[i & 1].x, sn[i & 1].y, sn[i & 1].z, sn[i & 1].w};
#pragma unroll
              for (int t = 0; t < 4; t += 2) {
                float a0, a1, b0, b1;
                gunpack<DT>(w[0][t / 2], a0, a1);
                gunpack<DT>(w[1][t / 2], b0, b1);
                float ac0 = mul_sep(a0, c4[t]), ac1 = mul_sep(a1, c4[t + 1]), bs0 = mul_sep(b0, s4[t]), bs1 = mul_sep(b1, s4[t + 1]);
                float bc0 = mul_sep(b0, c4[t]), bc1 = mul_sep(b1, c4[t + 1]), as0 = mul_sep(a0, s4[t]), as1 = mul_sep(a1, s4[t + 1]);
                round2(ac0, ac1); round2(bs0, bs1); round2(bc0, bc1); round2(as0, as1);
                w[0][t / 2] = gpack<DT>(add_sep(ac0, -bs0), add_sep(ac1, -bs1));
                w[1][t / 2] = gpack<DT>(add_sep(bc0, as0), add_sep(bc1, as1));
              }
            }
          }
        }
        uint16_t* const base = head ? (uint16_t*)P.q.out : (uint16_t*)P.c;
        const int64_t pitch = head ? 512 : P.ldc;
#pragma unroll
        for (int s = 0; s < 2; s++) {
          // columns 16 (2 s + j) + 4 g .. of fragments j = 0, 1 -> the 8 consecutive columns 32 s + 8 g ..: the 4 lane groups of a row
          // store 64 consecutive bytes (pieces of 16 bytes 32 apart: 33 216 x 656 x 640 51.9 us, so 49.2)
          uint32_t(&x0)[2] = w[2 * s], (&x1)[2] = w[2 * s + 1];
          xpose_pair(x0[0], x1[0]);
          xpose_pair(x0[1], x1[1]);
          const int n = cn0 + 64 * wn + 32 * s + 8 * g;
          if (row < P.M && n < P.N) *(uint4*)(base + (int64_t)row * pitch + n) = uint4{x0[0], x0[1], x1[0], x1[1]};
        }
      } else {
        // (with the stores of EPI 0 here the residual's loads come in the same pieces: 0 - 3 % slower; requested in the last iteration
        // but one instead of behind the loop, the residual costs 56 registers and 10 % of the K = 1664 product)
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          lo[j] = gpack<DT>(acc[i][j][0] * rn[i], acc[i][j][1] * rn[i]);
          hi[j] = gpack<DT>(acc[i][j][2] * rn[i], acc[i][j][3] * rn[i]);
        }
        xpose4(lo);
        xpose4(hi);
        // lane (r, g) now holds columns 16 g .. 16 g + 15 of the wave's 64: words lo[0] hi[0] lo[1] hi[1] ...
        const int n = cn0 + 64 * wn + 16 * g;
        float s = 0.f;
        if (row < P.M && n < P.N) {
          uint32_t wds[8] = {lo[0], hi[0], lo[1], hi[1], lo[2], hi[2], lo[3], hi[3]};
          const uint4 q0 = res[i][0], q1 = res[i][1];
          const uint32_t rw[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
          for (int e = 0; e < 8; e++) {
            float p0, p1, x0, x1;
            gunpack<DT>(wds[e], p0, p1);   // the product, already rounded to the activation type
            gunpack<DT>(rw[e], x0, x1);
            wds[e] = gpack<DT>(P.ca * x0 + P.cb * p0, P.ca * x1 + P.cb * p1);
          }
          uint16_t* cp = (uint16_t*)P.c + (int64_t)row * P.ldc + n;
          *(uint4*)cp = uint4{wds[0], wds[1], wds[2], wds[3]};
          *(uint4*)(cp + 8) = uint4{wds[4], wds[5], wds[6], wds[7]};
          if (NORM == 0 && P.sums) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
              float x0, x1;
              gunpack<DT>(wds[e], x0, x1);
              s = fmaf(x1, x1, fmaf(x0, x0, s));
            }
          }
        }
        if (NORM == 0 && P.sums) {   // the squares of the row's 64 columns: its 4 lane groups
          auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
          s = __uint_as_float(t[0]) + __uint_as_float(t[1]);
          t = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
          s = __uint_as_float(t[0]) + __uint_as_float(t[1]);
          if (g == 0 && row < P.M && cn0 + 64 * wn < P.N) *(float*)((char*)P.sums + (uint32_t)(cn0 / 64 + wn) * P.sums_ld4 + 4 * (uint32_t)row) = s;
        }
      }
    }
    if (!more) break;
    L += step;
    clear();
  }
  if (EPI == 3 && P.h.advance && blockIdx.x == 0)
    for (int64_t i = 64 * wave + fresh_lane(); i < P.h.n_advance; i += BIG_THREADS<FI>) P.h.advance[i] += 1;
}

template <int DT, int FI>
static void launch_big(const uvmi_gemm_args* a, const BigParams& P, int cus, hipStream_t st) {
  const int T = P.tiles_m * P.tiles_n;
  const int slots = (FI == 8 ? cus : 2 * cus) / 8 * 8;   // workgroups that run at a time
  // (a launch of one round keeps the shorter code: it lost 0.5 us of 9 to the other's)
  // (nor are there registers in a 256 x 256 tile for several and the query heads' epilogue)
  const bool many = P.K % 128 == 0 && slots > 0 && T > slots && !(FI == 8 && P.q.out);
  const dim3 grid((unsigned)(many ? slots : ((T + 7) / 8) * 8)), blk(BIG_THREADS<FI>);
#define UVMI_GO(EPI, NORM)                                                                              \
  do {                                                                                                  \
    if (many) hipLaunchKernelGGL((gemm_big_kernel<DT, EPI, NORM, FI, FI != 8 || EPI != 4>), grid, blk, 0, st, P); \
    else hipLaunchKernelGGL((gemm_big_kernel<DT, EPI, NORM, FI, false>), grid, blk, 0, st, P);          \
  } while (0)
  const int norm = a->norm_a ? (P.sums ? 2 : 1) : 0;
  if constexpr (FI == 6) {
    UVMI_GO(2, 0);
  } else if (a->epilogue == UVMI_GEMM_RESID) { if (norm) UVMI_GO(2, 1); else UVMI_GO(2, 0); }
  else if (a->epilogue == UVMI_GEMM_SWIGLU) { if (norm == 2) UVMI_GO(1, 2); else if (norm) UVMI_GO(1, 1); else UVMI_GO(1, 0); }
  else if (a->epilogue == UVMI_GEMM_SOFTCAP) { if (norm) UVMI_GO(3, 1); else UVMI_GO(3, 0); }
  else if (P.q.out) { if (norm == 2) UVMI_GO(4, 2); else if (norm) UVMI_GO(4, 1); else UVMI_GO(4, 0); }
  else { if (norm == 2) UVMI_GO(0, 2); else if (norm) UVMI_GO(0, 1); else UVMI_GO(0, 0); }
#undef UVMI_GO
}

// Arguments are validated by the caller (uvmi_gemm_tn_ex), which also checks K >= 128.  tile: 256, 128 or (RESID without
// the pre-norm: uvmi_gemm_resid) 192 rows.  sums: as uvmi_gemm_sums has it, q: STORE of K >= 256 and the
// extended projection's columns, h: SOFTCAP; or null.
void gemm_big_launch(const uvmi_gemm_args* a, int tile, int cus, hipStream_t st, float* sums, int64_t sums_ld, const QueryPost* q, const HeadRows* h) {
  BigParams P;
  P.a = a->a; P.w = a->w; P.c = a->c; P.r = a->resid;
  P.lda2 = (uint32_t)a->lda * 2; P.ldw2 = (uint32_t)a->ldw * 2; P.ldc = a->ldc; P.ldr = a->ldr;
  P.M = (int)a->M; P.N = a->N; P.K = a->K;
  const int cols = tile == 192 ? 128 : tile;
  P.tiles_m = (int)((a->M + tile - 1) / tile);
  P.tiles_n = (a->N + cols - 1) / cols;
  P.q = q ? *q : QueryPost{};
  P.h = h ? *h : HeadRows{};
  P.sums = sums; P.sums_ld4 = (uint32_t)sums_ld * 4; P.parts = ((a->norm_a ? a->K : a->N) + 63) / 64;
  P.eps = a->eps; P.ca = a->ca; P.cb = a->cb; P.cap_c = a->cap_c;
  const double bytes_a = (double)a->M * a->K, bytes_w = (double)a->N * a->K;
  P.rowsplit = bytes_a / 8 + bytes_w < bytes_a + bytes_w / 8;
#define UVMI_T(DT) do { if (tile == 256) launch_big<DT, 8>(a, P, cus, st); else if (tile == 192) launch_big<DT, 6>(a, P, cus, st); else launch_big<DT, 4>(a, P, cus, st); } while (0)
  if (a->dtype == UVMI_F16) UVMI_T(UVMI_F16); else UVMI_T(UVMI_BF16);
#undef UVMI_T
}

}  // namespace uvmi
