// The 16-bit GEMM's entry points and the choice of its form: gemm_stream.hip (up to a few thousand rows), gemm_big.hip (128 x 128 and
// 256 x 256 tiles loaded straight into LDS), gemm_tile.hip (128 x 128 tiles through registers: outputs whose rows are not 16-byte
// aligned).
#include "common.h"
#include "qkv_post.h"

using namespace uvmi;

namespace uvmi {
void gemm_tile_launch(const uvmi_gemm_args* a, hipStream_t st);                     // gemm_tile.hip
void gemm_big_launch(const uvmi_gemm_args* a, int tile, int cus, hipStream_t st, float* sums = nullptr, int64_t sums_ld = 0, const QueryPost* q = nullptr, const HeadRows* h = nullptr);   // gemm_big.hip; tile: 128, 256, 192 (x 128: RESID)
int gemm_stream_form(const uvmi_gemm_args* a, int cus);                             // gemm_stream.hip
void gemm_stream_tile(int form, int* rows, int* cols);
void gemm_stream_launch(const uvmi_gemm_args* a, int form, int cus, hipStream_t st);
}

// Rows from which a product may take the 256 x 256 tile of gemm_big.hip (one workgroup per compute unit) by big_tiles_pay; below, its
// rounds of the device are too few and too empty on UV-50M's projections.
constexpr int64_t BIG_MIN_ROWS = 12288, BIG_MIN_ROWS_SWIGLU = 4096;

// what the 256 x 256 kernel assumes beyond uvmi_gemm_tn_supported: two slabs at least, 16-byte stores and residual loads
static bool big_ok(const uvmi_gemm_args* a) {
  if (a->K < 128 || ((uintptr_t)a->c % 16) != 0 || a->ldc % 8 != 0) return false;
  if (a->epilogue == UVMI_GEMM_RESID && (((uintptr_t)a->resid % 16) != 0 || a->ldr % 8 != 0)) return false;
  return true;
}

// Whether a pass of many rows takes 256 x 256 tiles rather than 128 x 128 ones.  A launch lasts as long as its rounds of the device: of
// one 256 x 256 tile per compute unit, or of two 128 x 128 ones, which take about 0.6 of that.  us, 256 against 128, activations in
// the last-level cache as a pass leaves them: gate-up with norm and SwiGLU 5000 rows, 2 rounds against 3, 41.0 / 31.1; 8192 rows, 2
// against 3 and a quarter, 42.0 / 41.5 and again 43.9 / 42.3 (the one size measured where the choice is not the faster, by 1 - 4 %; 7168 rows
// 47.1 / 37.9, 9216 rows 45.1 / 49.0); 10 000 rows, 3 against 5, 62.6 / 51.4; 18 432 rows, 4 against 8, 88.6 / 96.0; 20 000 rows, 5 against 8, 100.3 /
// 104.9; 33 216 rows, 7 against 14, 150 / 171.  640 columns, K 1664: 18 432 rows, 1 against 2, 51.2 / 59.4; 24 576 rows, 2 against 2, 97.1 /
// 66.4; 40 000 rows, 2 against 4, 103 / 112.  With a short K a last round of 128 x 128 tiles that fills a quarter of the device or
// less takes half a round (K 512: 16 384 rows 21.9 / 20.4, 18 432 rows, 0.4 of a round, 23.4 / 26.0).
static bool big_tiles_pay(const uvmi_gemm_args* a, int64_t t128, int64_t t256, int cus, int round256 = 17) {
  const int64_t r256 = (t256 + cus - 1) / cus, slots = 2 * (int64_t)cus, rest = t128 % slots;
  const int64_t halves128 = 2 * (t128 / slots) + (rest == 0 ? 0 : (a->K <= 768 && 4 * rest <= slots ? 1 : 2));
  return round256 * r256 <= 5 * halves128;
}

extern "C" int uvmi_gemm_tn_supported(int dtype, int64_t M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc, int epilogue) {
  if (dtype != UVMI_F16 && dtype != UVMI_BF16) return 0;
  if (epilogue != UVMI_GEMM_STORE && epilogue != UVMI_GEMM_SWIGLU && epilogue != UVMI_GEMM_RESID && epilogue != UVMI_GEMM_SOFTCAP) return 0;
  if (M < 0 || M > (1 << 16) || N <= 0 || K <= 0 || K % 64 != 0 || K > 8192) return 0;
  if (N % (epilogue == UVMI_GEMM_SWIGLU ? 32 : 16) != 0) return 0;
  if (lda < K || ldw < K || lda % 8 != 0 || ldw % 8 != 0 || ldc % 4 != 0) return 0;
  if (ldc < (epilogue == UVMI_GEMM_SWIGLU ? N / 2 : N)) return 0;
  if ((M + 64) * lda * 2 >= (1LL << 30) || ((int64_t)N + 64) * ldw * 2 >= (1LL << 30)) return 0;  // 32-bit offsets with room for the out-of-range mark
  return 1;
}

static int check_gemm(const uvmi_gemm_args* a) {
  UVMI_REQUIRE(a && a->a && a->w && a->c, UVMI_EINVAL, "uvmi_gemm_tn: null pointer");
  UVMI_REQUIRE(uvmi_gemm_tn_supported(a->dtype, a->M, a->N, a->K, a->lda, a->ldw, a->ldc, a->epilogue), UVMI_EUNSUPPORTED,
               "uvmi_gemm_tn: unsupported problem (dtype %d, M %lld, N %d, K %d, lda %lld, ldw %lld, ldc %lld, epilogue %d): needs F16 / BF16, "
               "K %% 64 == 0, N %% 16 == 0 (32 with SWIGLU), lda, ldw %% 8 == 0, ldc %% 4 == 0",
               a->dtype, (long long)a->M, a->N, a->K, (long long)a->lda, (long long)a->ldw, (long long)a->ldc, a->epilogue);
  UVMI_REQUIRE(((uintptr_t)a->a % 16) == 0 && ((uintptr_t)a->w % 16) == 0 && ((uintptr_t)a->c % 8) == 0, UVMI_EINVAL, "uvmi_gemm_tn: misaligned pointer");
  if (a->epilogue == UVMI_GEMM_RESID)
    UVMI_REQUIRE(a->resid && ((uintptr_t)a->resid % 8) == 0 && a->ldr % 4 == 0 && a->ldr >= a->N, UVMI_EINVAL,
                 "uvmi_gemm_tn: the RESID epilogue needs an 8-byte aligned residual with a pitch that is a multiple of 4 and >= N");
  if (a->epilogue == UVMI_GEMM_SOFTCAP)
    UVMI_REQUIRE(big_ok(a) && a->cap_c != 0.f && (a->config == 0 || a->config == 5 || a->config == 6), UVMI_EUNSUPPORTED,
                 "uvmi_gemm_tn: the SOFTCAP epilogue needs K >= 128, a 16-byte aligned C with ldc %% 8 == 0, a non-zero cap_c and config 0, 5 or 6");
  UVMI_REQUIRE(!a->norm_a || a->eps >= 0.f, UVMI_EINVAL, "uvmi_gemm_tn: negative eps");
  UVMI_REQUIRE(a->config >= 0 && a->config <= 8, UVMI_EINVAL, "uvmi_gemm_tn: config %d", a->config);
  UVMI_REQUIRE((a->config != 1 && a->config != 2) || a->K <= (a->epilogue == UVMI_GEMM_SWIGLU ? 960 : 1984), UVMI_EUNSUPPORTED,
               "uvmi_gemm_tn: K = %d is beyond config 1, 2 (1984; 960 with SWIGLU)", a->K);
  UVMI_REQUIRE(a->config != 5 || a->M == 0 || big_ok(a), UVMI_EUNSUPPORTED,
               "uvmi_gemm_tn: config 5 (256 x 256 tiles) needs K >= 128, C (and the residual) 16-byte aligned, ldc (ldr) %% 8 == 0");
  UVMI_REQUIRE(a->config != 6 || a->M == 0 || big_ok(a), UVMI_EUNSUPPORTED,
               "uvmi_gemm_tn: config 6 (tiles loaded straight into LDS) needs K >= 128, C (and the residual) 16-byte aligned, ldc (ldr) %% 8 == 0");
  return UVMI_OK;
}

// The kernel that takes the problem: through registers (a 128 x 128 tile), streaming (the tile of `form`) or direct to LDS (128 x 128 or 256 x 256).
struct Path {
  int kind;   // UVMI_GEMM_PATH_*
  int form;   // STREAM: gemm_stream.hip's form; BIG: 128 or 256
};
static Path gemm_path(const uvmi_gemm_args* a, int cus) {
  // (also a product of fewer rows whose 256 x 256 tiles still come to two rounds of the device or more - the tied head,
  // 2048 x 32768: 104 us against 129 us on 128 x 128 tiles - or, none of their columns padding, to one full round where 128 x 128
  // tiles, two to a compute unit, take a second one: 512 x 32768 26.6 us against 29.9, with the softcap 33.7 against 47.7 and
  // from 384 rows on 28.3 against 35.6; 288 rows 27.9 against 26.4, 384 without the softcap 26.6 against 24.1).  With the softcap two rounds are
  // taken from 769 rows on, where 128 x 128 tiles come to more than three: 800 rows 54.5 / 51.4 us in a stream of its own and 60.9 / 73.5 behind other
  // work, as a step has it, 900 rows 56.3 / 59.7 and 65.0 / 78.5, 1000 rows 58.9 / 61.8 and 71.2 / 97.8 (two decode steps of 800 rows 990 -> 976 us,
  // 900 rows 1066 -> 1032, 1000 rows 1107 -> 1052); one and a half rounds, 648 - 768 rows, and one of 257 - 352 are within half a percent of a step either way.
  const int64_t t128 = ((a->M + 127) / 128) * (((int64_t)a->N + 127) / 128), t256 = ((a->M + 255) / 256) * (((int64_t)a->N + 255) / 256);
  const bool one_round = a->N % 256 == 0 && a->M >= (a->epilogue == UVMI_GEMM_SOFTCAP ? 384 : 512) && t256 <= cus && 8 * t256 >= 7 * (int64_t)cus && t128 > 2 * (int64_t)cus;
  const bool many_big_tiles = one_round || (a->M >= (a->epilogue == UVMI_GEMM_SOFTCAP ? 769 : 1024) && t256 >= 2 * (int64_t)cus);
  const bool rows_ok = a->M >= (a->epilogue == UVMI_GEMM_SWIGLU ? BIG_MIN_ROWS_SWIGLU : BIG_MIN_ROWS);
  if (a->config == 5) return {UVMI_GEMM_PATH_BIG, 256};
  if (a->config == 0 && (many_big_tiles || rows_ok) && big_ok(a)) {
    // (a product of fewer rows whose many 256-wide tiles would be more than a tenth emptier than 128-wide ones takes those)
    const int64_t pad128 = ((int64_t)a->N + 127) / 128 * 128, pad256 = ((int64_t)a->N + 255) / 256 * 256;
    const bool small = rows_ok ? !big_tiles_pay(a, t128, t256, cus) : pad128 * 10 < pad256 * 9;
    return {UVMI_GEMM_PATH_BIG, small ? 128 : 256};
  }
  if (a->config == 6 || a->epilogue == UVMI_GEMM_SOFTCAP) return {UVMI_GEMM_PATH_BIG, 128};
  // The streaming form while one of its tiles leaves a compute unit about one workgroup (gemm_stream_form) and, on 64 x 64 tiles, while
  // they are at most two to a unit, which run at the same time (N 640, K 512: 3072 rows, 480 tiles, 7.7 us against 9.2 in 128 x 128 tiles; 3328
  // rows, 520 tiles, 10.6 / 9.3; gate-up 576 rows, 468 tiles, 7.9 / 9.5, 640 rows, 520 tiles, 11.0 / 9.9).  With a longer K, where rounds of
  // the small tiles overlap, until 128 x 128 tiles fill 3/4 of the device (640 columns, K 1664: 4608 rows 19.3 / 20.5, 5120 rows 23.3 / 20.5).
  static const int of_config[9] = {-1, 4, 0, -1, 6, -1, -1, 1, 2};
  int form = a->config == 0 ? gemm_stream_form(a, cus) : of_config[a->config];
  const int64_t t64 = ((a->M + 63) / 64) * (((int64_t)a->N + 63) / 64);
  if (a->config == 0 && form < 0 && (a->K <= 768 ? t64 <= 2 * (int64_t)cus : 4 * t128 < 3 * (int64_t)cus)) form = 6;
  if (form >= 0) return {UVMI_GEMM_PATH_STREAM, form};
  if (a->config == 0 && big_ok(a)) return {UVMI_GEMM_PATH_BIG, 128};
  return {UVMI_GEMM_PATH_TILED, 0};
}

static int compute_units() {
  const int cus = uvmi_device_cus();
  return cus > 0 ? cus : 256;
}

extern "C" int uvmi_gemm_tn_path(const uvmi_gemm_args* a, int* tile_rows, int* tile_cols) {
  const int rc = check_gemm(a);
  if (rc) return rc;
  const Path p = gemm_path(a, compute_units());
  int rows = 128, cols = 128;
  if (p.kind == UVMI_GEMM_PATH_BIG) rows = cols = p.form;
  else if (p.kind == UVMI_GEMM_PATH_STREAM) gemm_stream_tile(p.form, &rows, &cols);
  if (tile_rows) *tile_rows = rows;
  if (tile_cols) *tile_cols = cols;
  return p.kind;
}

extern "C" int uvmi_gemm_tn_ex(const uvmi_gemm_args* a, void* stream) {
  const int rc = check_gemm(a);
  if (rc) return rc;
  if (a->M == 0) return UVMI_OK;
  const int cus = compute_units();
  const Path p = gemm_path(a, cus);
  if (p.kind == UVMI_GEMM_PATH_STREAM) gemm_stream_launch(a, p.form, cus, (hipStream_t)stream);
  else if (p.kind == UVMI_GEMM_PATH_BIG) gemm_big_launch(a, p.form, cus, (hipStream_t)stream);
  else gemm_tile_launch(a, (hipStream_t)stream);
  UVMI_CHECK_LAUNCH("uvmi_gemm_tn");
  return UVMI_OK;
}

extern "C" int uvmi_gemm_tn(const void* a, const void* w, void* c, int dtype, int64_t M, int N, int K, int64_t lda, int64_t ldw,
                            int64_t ldc, int epilogue, void* stream) {
  uvmi_gemm_args g = {};
  g.a = a; g.w = w; g.c = c; g.dtype = dtype; g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldw = ldw; g.ldc = ldc; g.epilogue = epilogue;
  UVMI_REQUIRE(epilogue != UVMI_GEMM_RESID, UVMI_EINVAL, "uvmi_gemm_tn: the RESID epilogue takes its residual through uvmi_gemm_tn_ex");
  return uvmi_gemm_tn_ex(&g, stream);
}

// The residual update of a pass of many rows also has 192 x 128 tiles, two to a compute unit, to choose from: between the rounds of the
// device of the other two, and with two epilogues to overlap.  A launch lasts as long as its rounds, of which a last one that gives a unit one
// workgroup takes about six tenths (128 x 128) and four (192 x 128) of a full one; a full one of 192 x 128 tiles 1.48 and one of 256 x 256
// tiles 1.7 of one of 128 x 128 ones.  us, 128 / 192 / 256, 640 columns, K 1664 and 512: 12 288 rows 30.1 / 38.1 / 45.0 and 15.2 /
// 18.5 / 22.1; 14 000 46.3 / 38.3 / 45.3 and 21.2 / 19.7 / 22.5; 18 432 47.3 / 41.6 / 48.6 and 22.6 / 21.5 / 23.8; 20 000 52.1 / 56.9 / 47.7 and
// 26.2 / 28.1 / 24.3; 24 576 54.9 / 57.0 / 86.5 and 27.3 / 28.0 / 41.3; 28 000 71.6 / 61.6 / 88.9 and 32.7 / 29.6 / 41.8; 33 216 77.2 / 79.0 /
// 90.6 and 37.6 / 36.5 / 43.8; 50 000 106.8 / 116.2 / 131.9 and 49.4 / 52.4 / 60.4.  Those are last rounds, which start while the one before ends: an update
// whose 128 x 128 tiles are one round has no use for larger ones (256 columns, K 256, 512 and 2048: 16 000 rows 7.4 / 9.0, 9.7 / 11.7 and 26.8 / 28.7; 24 576 10.2 / 10.1,
// 15.2 / 14.5 and 30.9 / 32.8; two rounds, 33 216 rows, 16.4 / 14.2, 22.1 / 18.4 and 49.7 in 256 x 256 ones / 43.2; 128 columns, K 1664, 40 000 rows 31.1 / 34.9).
static bool resid_192(const uvmi_gemm_args* a, int cus) {
  if (a->epilogue != UVMI_GEMM_RESID || a->norm_a || a->config != 0 || a->M < BIG_MIN_ROWS || !big_ok(a)) return false;
  const int64_t slots = 2 * (int64_t)cus, n128 = ((int64_t)a->N + 127) / 128;
  auto rounds = [&](int64_t tiles, int full, int part) {
    const int64_t rest = tiles % slots;
    return tiles / slots * full + (rest == 0 ? 0 : (rest <= cus ? part : full));
  };
  const int64_t t256 = ((a->M + 255) / 256) * (((int64_t)a->N + 255) / 256);
  const int64_t t128 = ((a->M + 127) / 128) * n128;
  if (t128 <= slots) return false;
  const int64_t c192 = rounds(((a->M + 191) / 192) * n128, 148, 59);
  return c192 < rounds(t128, 100, 64) && c192 < (t256 + cus - 1) / cus * 170;
}

extern "C" int uvmi_gemm_resid_tile(const uvmi_gemm_args* a) {
  const int rc = check_gemm(a);
  return rc ? rc : (resid_192(a, compute_units()) ? 192 : 0);
}

extern "C" int uvmi_gemm_resid(const uvmi_gemm_args* a, void* stream) {
  if (a && a->M < BIG_MIN_ROWS) return uvmi_gemm_tn_ex(a, stream);
  const int rc = check_gemm(a);
  if (rc) return rc;
  const int cus = compute_units();
  if (!resid_192(a, cus)) return uvmi_gemm_tn_ex(a, stream);
  gemm_big_launch(a, 192, cus, (hipStream_t)stream);
  UVMI_CHECK_LAUNCH("uvmi_gemm_resid");
  return UVMI_OK;
}

// A pass of many rows takes the squares of a block's hidden where the residual updates write it, 64 columns at a time, not again in every
// column of tiles that reads it.
static int check_sums(const uvmi_gemm_args* a, const float* sums, int64_t ld) {
  const bool writes = a->epilogue == UVMI_GEMM_RESID && !a->norm_a, reads = a->norm_a && (a->epilogue == UVMI_GEMM_STORE || a->epilogue == UVMI_GEMM_SWIGLU);
  UVMI_REQUIRE((writes || reads) && (writes ? a->N : a->K) <= 1024 && (writes || a->K >= 256) && big_ok(a) && a->M > 0 &&
               (a->config == 5 || a->config == 6 || (a->config == 0 && a->M >= BIG_MIN_ROWS)), UVMI_EUNSUPPORTED,
               "uvmi_gemm_sums: RESID without a pre-norm or STORE / SWIGLU with one, of a hidden of 256 to 1024 columns, on tiles loaded straight into LDS");
  UVMI_REQUIRE((uintptr_t)sums % 16 == 0 && ld % 4 == 0 && ld >= a->M && ld <= (1 << 24), UVMI_EINVAL,
               "uvmi_gemm_sums: sums 16-byte aligned, with a pitch that is a multiple of 4, >= M");
  return UVMI_OK;
}

extern "C" int uvmi_gemm_sums(const struct uvmi_gemm_sums_args* s, void* stream) {
  UVMI_REQUIRE(s && s->gemm && s->sums, UVMI_EINVAL, "uvmi_gemm_sums: null pointer");
  const uvmi_gemm_args* a = s->gemm;
  int rc = check_gemm(a);
  if (!rc) rc = check_sums(a, s->sums, s->ld);
  if (rc) return rc;
  const int cus = compute_units();
  gemm_big_launch(a, resid_192(a, cus) ? 192 : gemm_path(a, cus).form, cus, (hipStream_t)stream, s->sums, s->ld);
  UVMI_CHECK_LAUNCH("uvmi_gemm_sums");
  return UVMI_OK;
}

bool uvmi::gemm_query_post(const uvmi_gemm_args* a, const QueryPost& q, float* sums, int64_t sums_ld, hipStream_t st) {
  const int cus = compute_units();
  if (check_gemm(a) || a->M == 0 || a->epilogue != UVMI_GEMM_STORE || a->K < 256 || q.rope_n > (1 << 23)) return false;
  if (sums && check_sums(a, sums, sums_ld)) return false;
  Path p = gemm_path(a, cus);
  if (p.kind != UVMI_GEMM_PATH_BIG) return false;
  // (256 x 256 tiles come one to a workgroup here, a round costs more: 33 216 rows 49.7 us against 45.2 in 128 x 128 tiles; 40 000
  // rows, two full rounds, 59.6 / 61.5 with the rest of the post-processing, 18 432 rows, one, 25.6 / 26.7)
  const int64_t t256 = ((a->M + 255) / 256) * 3, t128 = ((a->M + 127) / 128) * 6;
  if (a->config == 0 && p.form == 256 && t256 > cus && !big_tiles_pay(a, t128, t256, cus, 20)) p.form = 128;
  gemm_big_launch(a, p.form, cus, st, sums, sums_ld, &q);
  return true;
}

extern "C" int uvmi_head(const struct uvmi_head_args* s, void* stream) {
  UVMI_REQUIRE(s && s->gemm, UVMI_EINVAL, "uvmi_head: null pointer");
  const uvmi_gemm_args* a = s->gemm;
  const int rc = check_gemm(a);
  if (rc) return rc;
  UVMI_REQUIRE(a->epilogue == UVMI_GEMM_SOFTCAP, UVMI_EINVAL, "uvmi_head: the SOFTCAP epilogue only");
  UVMI_REQUIRE(!s->rows || (s->a_rows > 0 && s->a_rows <= (1 << 20) && (s->a_rows + 64) * a->lda * 2 < (1LL << 30)), UVMI_EUNSUPPORTED,
               "uvmi_head: rows of a hidden of %lld rows with a pitch of %lld", (long long)s->a_rows, (long long)a->lda);
  UVMI_REQUIRE(!s->advance || s->n_advance >= 0, UVMI_EINVAL, "uvmi_head: negative count");
  UVMI_REQUIRE(a->M > 0 || !s->advance || s->n_advance == 0, UVMI_EINVAL, "uvmi_head: positions to count up behind no rows");
  if (a->M == 0) return UVMI_OK;
  const int cus = compute_units();
  const HeadRows h = {s->rows, (int)s->a_rows, s->advance, s->n_advance};
  gemm_big_launch(a, gemm_path(a, cus).form, cus, (hipStream_t)stream, nullptr, 0, nullptr, &h);
  UVMI_CHECK_LAUNCH("uvmi_head");
  return UVMI_OK;
}
