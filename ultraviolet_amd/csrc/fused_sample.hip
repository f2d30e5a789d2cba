// Fused softcap + categorical draw (inverse CDF, one uniform per row) + behaviour log-prob, and greedy argmax.
//
// Contract (ultraviolet/kernels/fused_sample.py:31-77 of the reference): with z = a*sigmoid((x+b)/c) and
// e = exp((z-a)/T) in (exp(-a/T), 1] (the softcap bounds z, so there is no max pass), S = sum(e),
// target = (1-u)*S; the token is the first index whose running sum reaches target (clamped to V-1) and
// logp = (z_tok - a)/T - log S.  The running sum is hierarchical here (512-element chunks, then lanes, then the
// lane's 8 elements), so the token equals the flat-cumsum one up to fp32 summation order.
//
// e is evaluated as exp2(-(a/T)*log2(e) / (1 + exp2(t*log2(e)))), t = (x+b)/c: algebraically the same as above
// (z - a = -a*sigmoid(-t)) without the cancellation of z - a near the cap.
//
// One workgroup of 256 threads per row streams the row once (HBM-bound: 2 B per logit for bf16/fp16), keeps only
// the 64 chunk sums in LDS, then one wave re-reads the chosen 1 KB chunk (cache-hot).  When u is not supplied it is
// drawn from Philox4x32-10 keyed by the seed with counter (token index, request id lo, request id hi, "SAMP"), so a
// request's stream does not depend on the slot it occupies.
#include "common.h"
#include "sched_commit.h"

namespace uvmi {

constexpr int CHUNK = 512;          // elements per wave pass: 64 lanes x 8
constexpr uint32_t DOMAIN_SAMPLE = 0x53414D50u;

__host__ __device__ inline void philox4x32_10(const uint32_t c_in[4], const uint32_t k_in[2], uint32_t out[4]) {
  uint32_t c0 = c_in[0], c1 = c_in[1], c2 = c_in[2], c3 = c_in[3], k0 = k_in[0], k1 = k_in[1];
#pragma unroll
  for (int r = 0; r < 10; r++) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0, n1 = (uint32_t)p1, n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1, n3 = (uint32_t)p0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

struct SampleParams {
  const void* x; int64_t stride; const float* u; uint64_t seed; const int64_t* req_id; const int64_t* tok_idx;
  int64_t* tok; float* logp; float* u_out;
  int V;
  float inv_c_l2, b_over_c_l2;  // t*log2(e) = x*inv_c_l2 + b_over_c_l2
  float neg_a_over_t_l2;        // -(a/T)*log2(e)
  float neg_a_over_t;           // -(a/T)
  float cap_a, cap_b, cap_c, inv_c;
  int top_k; float top_p; float* thr_out;
  // optional: commit the drawn token to the slot table in the same launch (row = dense row of a decode step)
  int commit; float retire_p; uint64_t commit_seed; uvmi_sched_state S; DenseArrays D;
};

// The row's result; with P.commit also what uvmi_sched_commit_dense does for the row (one thread per row calls this; r: its commit_ahead).
__device__ __forceinline__ void emit(const SampleParams& P, int row, int tok, float logp, const CommitRow& r) {
  P.tok[row] = tok;
  P.logp[row] = logp;
  if (P.commit) commit_store<true>(P.S, P.D, row, r, tok, logp);
}
// what emit's commit reads, for thread 0, which emits: ahead of the draw, so that it is there by then (the kernels of 1024 threads that hold a row
// in registers request its logits first)
__device__ __forceinline__ CommitRow commit_ahead(const SampleParams& P, int row) {
  CommitRow r = {};
  if (P.commit && threadIdx.x == 0) r = commit_load<true>(P.S, P.D, row, P.retire_p, P.commit_seed);
  return r;
}
// the row's uniform (every thread of the wave that draws)
__device__ __forceinline__ float uniform_of(const SampleParams& P, int row) {
  if (P.u) return P.u[row];
  const uint64_t rid = (uint64_t)P.req_id[row], ti = (uint64_t)P.tok_idx[row];
  const uint32_t ctr[4] = {(uint32_t)ti, (uint32_t)rid, (uint32_t)(rid >> 32), DOMAIN_SAMPLE};
  const uint32_t key[2] = {(uint32_t)P.seed, (uint32_t)(P.seed >> 32)};
  uint32_t o[4];
  philox4x32_10(ctr, key, o);
  return (float)(o[0] >> 8) * 5.9604644775390625e-08f;  // 2^-24
}

template <int DT>
__device__ __forceinline__ void load8(const void* row, int i, float (&o)[8]) {  // elements 8i .. 8i+7
  if (DT == UVMI_F32) {
    const float4 a = ((const float4*)row)[2 * i], b = ((const float4*)row)[2 * i + 1];
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  } else {
    const uint4 w = ((const uint4*)row)[i];
    const uint32_t r[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (DT == UVMI_BF16) {
        o[2 * j] = __uint_as_float(r[j] << 16);
        o[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u);
      } else {
        o[2 * j] = half_bits_to_float(r[j] & 0xffff);
        o[2 * j + 1] = half_bits_to_float(r[j] >> 16);
      }
    }
  }
}

__device__ __forceinline__ float e_of(float x, const SampleParams& P) {
  const float E = __builtin_amdgcn_exp2f(fmaf(x, P.inv_c_l2, P.b_over_c_l2));  // exp(t), may be +inf (then e = 1)
  return __builtin_amdgcn_exp2f(P.neg_a_over_t_l2 * __builtin_amdgcn_rcpf(1.0f + E));
}

// (the row pointer's ingredients lead the argument list: leading scalar arguments are preloaded into SGPRs with the wave,
// so the first loads of the row do not wait for a load of the kernel arguments)
// NT threads per row: 256 when there are rows enough to fill the device, 1024 for small batches (the row's exponentials are
// the work of the launch; with one small workgroup per row and fewer rows than compute units most of the device would idle)
template <int DT, int NT>
__global__ __launch_bounds__(NT) void sample_kernel(const void* a_x, int64_t a_stride, int a_V, float a_inv_c_l2, float a_b_over_c_l2,
                                                    float a_neg_a_over_t_l2, SampleParams P) {
  P.x = a_x; P.stride = a_stride; P.V = a_V; P.inv_c_l2 = a_inv_c_l2; P.b_over_c_l2 = a_b_over_c_l2; P.neg_a_over_t_l2 = a_neg_a_over_t_l2;
  __shared__ float csum[64 + 4];
  __shared__ int sh_chunk;
  __shared__ float sh_before, sh_total, sh_target;
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const char* xr = (const char*)P.x + (int64_t)row * P.stride * (DT == UVMI_F32 ? 4 : 2);
  const int nchunks = P.V / CHUNK;  // host guarantees V % 512 == 0 and nchunks <= 64
  const float u = wave == 0 ? uniform_of(P, row) : 0.f;
  const CommitRow cr = commit_ahead(P, row);
  for (int c = wave; c < nchunks; c += NT / 64) {
    float v[8];
    load8<DT>(xr, c * 64 + lane, v);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) s += e_of(v[j], P);
    s = wave_sum(s);
    if (lane == 0) csum[c] = s;
  }
  __syncthreads();
  if (wave != 0) return;
  // ---- wave 0: pick the chunk, then the lane, then the element
  float mine = lane < nchunks ? csum[lane] : 0.f;
  float incl = mine;  // inclusive scan over chunks in lane order
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  const float S = __shfl(incl, 63, 64);
  const float target = (1.0f - u) * S;
  const unsigned long long below = __ballot(lane < nchunks && incl < target);
  int ck = __popcll(below);  // first chunk whose inclusive sum reaches target
  if (ck > nchunks - 1) ck = nchunks - 1;
  const float before = ck > 0 ? __shfl(incl, ck - 1, 64) : 0.f;
  float v[8], e[8];
  load8<DT>(xr, ck * 64 + lane, v);
  float ls = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    e[j] = e_of(v[j], P);
    ls += e[j];
  }
  float linc = ls;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float t = __shfl_up(linc, o, 64);
    if (lane >= o) linc += t;
  }
  linc += before;
  const unsigned long long lb = __ballot(linc < target);
  int ln = __popcll(lb);
  if (ln > 63) ln = 63;
  // every lane recomputes the winner lane's walk from broadcast values (uniform control flow)
  float run = ln > 0 ? __shfl(linc, ln - 1, 64) : before;
  int jsel = 7;
  bool found = false;
  float xsel = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float ej = __shfl(e[j], ln, 64), xj = __shfl(v[j], ln, 64);
    run += ej;
    if (!found && run >= target) { found = true; jsel = j; xsel = xj; }
    if (j == 7 && !found) xsel = xj;
  }
  if (lane == 0) {
    const int tok = ck * CHUNK + ln * 8 + jsel;
    // logp = (z_tok - a)/T - log S, with (z - a)/T = -(a/T) / (1 + exp(t))
    const float E = __builtin_amdgcn_exp2f(fmaf(xsel, P.inv_c_l2, P.b_over_c_l2));
    if (P.u_out) P.u_out[row] = u;
    emit(P, row, tok, P.neg_a_over_t * __builtin_amdgcn_rcpf(1.0f + E) - __logf(S), cr);
  }
}

// Top-k / nucleus sampling (sample() of the reference, ultraviolet/model.py:1194-1211): keep the tokens whose value is at
// least the k-th largest, then of those the smallest prefix by probability whose mass reaches top_p (the token that
// crosses it included, ties of the last kept value all kept), and draw from what is kept by inverse CDF in index order.
// Everything is decided on e = exp((z - a)/T), which is positive and monotone in the logit, so its fp32 bit pattern
// orders the tokens: both thresholds are found by a radix select over those 32 bits.  The behaviour log-prob is that of the
// unfiltered softmax, as the reference records it (model.py:1161-1169).
//
// What bounds it: one row per workgroup is a serial chain of selects, so the chain is kept short.  The row is read once and
// its exponentials stay in registers (1024 threads x 32 elements); the digits are 12 + 10 + 10 bits, so a threshold takes
// three histograms, and the first digit (8 exponent bits and 3 of the mantissa) already spreads a row over tens of
// bins, which keeps the LDS atomics of a wave from meeting on one address.  A bin holds the count (16 bits) and the mass
// (48 bits, 32.32 fixed point: sums do not depend on the order of the additions) of its keys in one 64-bit word, so one
// histogram serves both selects: the nucleus walk starts on the histograms that the top-k walk left and only builds new
// ones for the bins in which it ends elsewhere.  200 rows x 32768, top_k 50 + top_p 0.95: 203 us for eleven sweeps of the
// row with 8-bit digits, one thread walking each histogram; 13.9 us with a bound from 4096 64-bit bins that every thread scanned,
// ranks and masses gathered by LDS atomics and the chosen chunk read again for the draw; 11.9 us as it is now, where the bound is
// 256 bins that a wave scans in four words a lane, ranks are counted by ballots, one wave walks the sorted masses and the wave that
// holds the chosen chunk draws from its registers (75 rows, top_k 50 alone: 13.2 -> 10.9).  What is left: launch and loads 4, the exponentials
// 2.8, the selects and barriers behind them; 22 - 23 us for top_p alone, which needs the histogram of the whole row (9 us: 512
// wave-wide 64-bit LDS atomics of ~40 clocks each).
constexpr unsigned long long BIN_ONE = 1ull << 48, BIN_MASS = BIN_ONE - 1;
constexpr unsigned int CAND = 512;   // most candidates of a top-k select that are ranked key by key
constexpr unsigned int BOUND_BINS = 256, BOUND_SHIFT = 19;   // of the bound below them: sixteen bins an octave

// floor(e * 2^32) for 0 <= e <= 1
__device__ __forceinline__ unsigned long long fix32(float e) {
  const uint32_t b = __float_as_uint(e);
  const int sh = (int)(b >> 23) - 118;   // e = m * 2^(exponent - 150)
  const uint32_t m = (b & 0x7fffffu) | 0x800000u;
  return sh >= 0 ? (unsigned long long)m << sh : (unsigned long long)(sh > -24 ? m >> -sh : 0u);
}

// inclusive prefix sum over the 64 lanes by DPP row shifts and broadcasts (a shuffle through the LDS crossbar per step and word
// would be most of a pick's time)
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long scan_step(unsigned long long v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS, 0xf, false);
  return v + (((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ unsigned long long wave_scan(unsigned long long v) {
  v = scan_step<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
  v = scan_step<0x112, 0xf>(v);
  v = scan_step<0x114, 0xf>(v);
  v = scan_step<0x118, 0xf>(v);
  v = scan_step<0x142, 0xa>(v);   // lane 15 of rows 0, 2 -> rows 1, 3
  return scan_step<0x143, 0xc>(v);  // lane 31 -> rows 2, 3
}

struct BinPick { unsigned int digit, cnt_above; unsigned long long mass_above, mass; };

// The bin of a histogram of 1024 * PER bins in which a walk from the largest key down ends: by count (the bin with the
// want-th largest key) or by mass (the first bin at which the mass reaches `want`; the largest key's bin when want is 0).
// All 1024 threads call it; share > 0: `want` is set to that share of the whole histogram's mass first.
template <int PER, bool BY_MASS>
__device__ __forceinline__ BinPick pick_bin(const unsigned long long* h, unsigned long long& want, unsigned long long* wtot, BinPick* sh,
                                            double share = 0.0) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned long long v[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; i++) {
    v[i] = h[1024 * PER - 1 - (tid * PER + i)];
    sum += v[i];
  }
  const unsigned long long incl = wave_scan(sum);
  if (lane == 63) wtot[wave] = incl;
  __syncthreads();
  unsigned long long run = incl - sum;
  unsigned long long total = 0;
#pragma unroll
  for (int w = 0; w < 16; w++) {
    const unsigned long long t = wtot[w];
    if (w < wave) run += t;
    total += t;
  }
  if (BY_MASS && share > 0.0) want = (unsigned long long)(share * (double)(total & BIN_MASS));
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const unsigned long long above = run;
    run += v[i];
    const unsigned long long ca = above >> 48, c = v[i] >> 48, ma = above & BIN_MASS, m = v[i] & BIN_MASS;
    const bool here = BY_MASS ? c > 0 && (want == 0 ? ca == 0 : ma < want && ma + m >= want) : ca < want && ca + c >= want;
    if (here) *sh = BinPick{(unsigned int)(1024 * PER - 1 - (tid * PER + i)), (unsigned int)ca, ma, m};
  }
  __syncthreads();
  const BinPick r = *sh;
  __syncthreads();   // (the next pick writes wtot and sh)
  return r;
}

// inclusive prefix sum of 32-bit counts over the lanes, as wave_scan
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned int count_step(unsigned int v) { return v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false); }
__device__ __forceinline__ unsigned int wave_count(unsigned int v) {
  return count_step<0x143, 0xc>(count_step<0x142, 0xa>(count_step<0x118, 0xf>(count_step<0x114, 0xf>(count_step<0x112, 0xf>(count_step<0x111, 0xf>(v))))));
}

template <int DT>
__global__ __launch_bounds__(1024) void sample_filtered_kernel(SampleParams P) {
  __shared__ float csum[64 + 4], csum_all[64];
  __shared__ unsigned long long h1[4096], h2[1024], h3[1024], wtot[16];
  __shared__ BinPick sh;
  __shared__ __attribute__((aligned(16))) unsigned int bound[BOUND_BINS];
  __shared__ unsigned int cand[CAND], sorted[CAND], n_cand, wmax[16], sh_thr;
  __shared__ float sh_u, sh_lp;
  __shared__ int sh_tok;
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tid = threadIdx.x;
  const char* xr = (const char*)P.x + (int64_t)row * P.stride * (DT == UVMI_F32 ? 4 : 2);
  const int nchunks = P.V / CHUNK;   // <= 64: wave w holds chunks w, w + 16, w + 32, w + 48

  // the thread's logits, 16-bit ones kept beside their exponentials for the draw
  float e[4][8];
  uint4 raw[DT == UVMI_F32 ? 1 : 4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = wave + 16 * q;
    if (c < nchunks) {
      if constexpr (DT == UVMI_F32) load8<DT>(xr, c * 64 + lane, e[q]);
      else raw[q] = ((const uint4*)xr)[c * 64 + lane];
    }
  }
  // (requested with the row: the draw at the end of the chain needs it at once)
  if (wave == 0) {
    const float u = uniform_of(P, row);
    if (lane == 0) sh_u = u;
  }
  if (tid < BOUND_BINS) bound[tid] = 0;
  if (tid == 0) n_cand = 0;
  // ---- unfiltered chunk sums (for the log-prob), in the order of the unfiltered kernel, and the thread's largest key
  unsigned int mx = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = wave + 16 * q;
    if (c < nchunks) {
      if constexpr (DT != UVMI_F32) load8<DT>(&raw[q], 0, e[q]);
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        e[q][j] = e_of(e[q][j], P);
        s += e[q][j];
        mx = max(mx, __float_as_uint(e[q][j]));
      }
      s = wave_sum(s);
      if (lane == 0) csum_all[c] = s;
    }
  }
  {
    const float wm = wave_max(__uint_as_float(mx));
    if (lane == 0) wmax[wave] = __float_as_uint(wm);
  }
  const CommitRow cr = commit_ahead(P, row);
  __syncthreads();

  unsigned int thr = 0;   // keep keys >= thr
  const bool by_count = P.top_k > 0 && P.top_k < P.V;
  const double share = P.top_p > 0.f ? (double)P.top_p : 0.0;
  // ---- top-k of at most 256: the threads' largest keys bound the k-th largest key from below (k of them are at least as
  // large), so only keys from that bound's bin up can matter: the bins are sixteenths of an octave below the row's largest key.  They are about a
  // hundred of the 32 768 and are collected in LDS, and each is put in its place by its rank among them, which the waves count
  // with ballots; one wave then walks the sorted keys' masses.  Rows whose candidates are too many for that (long runs of equal
  // logits) take the histograms.
  bool ranked = false;
  if (by_count && P.top_k <= 256) {
    unsigned int top = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) top = max(top, wmax[w]);
    atomicAdd(&bound[min(BOUND_BINS - 1u, (top - mx) >> BOUND_SHIFT)], 1u);
    __syncthreads();
    unsigned int low;
    {   // (every wave for itself)
      const uint4 c4 = ((const uint4*)bound)[lane];
      const unsigned int incl = wave_count(c4.x + c4.y + c4.z + c4.w), k = (unsigned int)P.top_k;
      const unsigned long long reach = __ballot(incl >= k);
      const int at = __ffsll((long long)reach) - 1;   // (1024 keys in the bins, k <= 256)
      unsigned int run = incl - (c4.x + c4.y + c4.z + c4.w), b = 4 * lane;
      if (run + c4.x < k) { run += c4.x; b++; if (run + c4.y < k) { run += c4.y; b++; if (run + c4.z < k) b++; } }
      b = (unsigned int)__builtin_amdgcn_readlane((int)b, at);
      const unsigned int span = (b + 1) << BOUND_SHIFT;   // keys above top - span
      low = b == BOUND_BINS - 1 || span > top ? 0u : top - span + 1;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (wave + 16 * q < nchunks) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const unsigned int key = __float_as_uint(e[q][j]);
          if (key >= low) {
            const unsigned int at = atomicAdd(&n_cand, 1u);
            if (at < CAND) cand[at] = key;
          }
        }
      }
    __syncthreads();
    ranked = n_cand <= CAND;
  }
  if (ranked) {
    const int n = (int)n_cand, R = (n + 63) >> 6;
    unsigned int key[CAND / 64];
#pragma unroll
    for (int r = 0; r < (int)CAND / 64; r++) key[r] = 64 * r + lane < n ? cand[64 * r + lane] : 0u;
    for (int c = wave; c < n; c += 16) {
      const unsigned int mine = cand[c];
      int rank = 0;
#pragma unroll
      for (int r = 0; r < (int)CAND / 64; r++) {
        if (r >= R) break;
        rank += __popcll(__ballot(key[r] > mine || (key[r] == mine && 64 * r + lane < c)));
      }
      if (lane == 0) sorted[rank] = mine;
    }
    __syncthreads();
    if (wave == 0) {   // lane l has the sorted keys R l .. R l + R - 1
      unsigned int t = sorted[P.top_k - 1];
      if (P.top_p < 1.0f) {
        unsigned long long m[CAND / 64], mine = 0, kept = 0;
#pragma unroll
        for (int r = 0; r < (int)CAND / 64; r++) {
          m[r] = 0;
          if (r >= R) break;
          key[r] = R * lane + r < n ? sorted[R * lane + r] : 0u;
          m[r] = key[r] ? fix32(__uint_as_float(key[r])) : 0ull;
          mine += m[r];
          kept += key[r] >= t ? m[r] : 0ull;
        }
        const unsigned long long all = wave_scan(kept);
        const unsigned long long mass = ((unsigned long long)(unsigned int)__builtin_amdgcn_readlane((int)(all >> 32), 63) << 32) |
                                        (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)all, 63);
        const unsigned long long want = (unsigned long long)(share * (double)mass);
        // the first key whose mass of keys up to it reaches want (a run of equal keys is kept whole: the threshold is their value)
        const unsigned long long incl = wave_scan(mine);
        unsigned long long run = incl - mine;
        unsigned int pick = 0;
        bool found = false;
#pragma unroll
        for (int r = 0; r < (int)CAND / 64; r++) {
          if (r >= R) break;
          run += m[r];
          if (!found && key[r] && run >= want) { pick = key[r]; found = true; }
        }
        const unsigned long long reach = __ballot(found);
        if (reach) t = (unsigned int)__builtin_amdgcn_readlane((int)pick, __ffsll((long long)reach) - 1);
      }
      if (lane == 0) sh_thr = t;
    }
    __syncthreads();
    thr = sh_thr;
  }
  // ---- the general form: radix selects over histograms of the whole row, by digits of 12 + 10 + 10 bits.  (Digits counted from
  // the row's largest key in 128 bins per octave were measured too: no faster - a wave's 64-bit LDS atomics take ~40 clocks
  // whether their addresses meet or not.)
  if (!ranked) {
    auto histogram = [&](unsigned long long* h, int shift, int nbits, unsigned int prefix) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (wave + 16 * q < nchunks) {
#pragma unroll
          for (int j = 0; j < 8; j++) {
            unsigned int key = __float_as_uint(e[q][j]);
            asm volatile("" : "+v"(key));   // (what is derived from a key is formed again in every pass: kept, it would spill)
            if (nbits + shift == 32 || (key >> (shift + nbits)) == prefix)
              atomicAdd(&h[(key >> shift) & ((1u << nbits) - 1u)], BIN_ONE | fix32(__uint_as_float(key)));
          }
        }
      __syncthreads();
    };
    auto clear = [&]() { h2[tid] = 0; h3[tid] = 0; };
    for (int i = tid; i < 4096; i += 1024) h1[i] = 0;
    clear();
    __syncthreads();
    unsigned int d1 = 0, d2 = 0;
    unsigned long long above1 = 0, above2 = 0, want = 0;
    histogram(h1, 20, 12, 0);
    if (by_count) {
      unsigned long long krem = (unsigned long long)P.top_k;
      BinPick b = pick_bin<4, false>(h1, krem, wtot, &sh);
      d1 = b.digit; krem -= b.cnt_above; above1 = b.mass_above;
      histogram(h2, 10, 10, d1);
      b = pick_bin<1, false>(h2, krem, wtot, &sh);
      d2 = b.digit; krem -= b.cnt_above; above2 = b.mass_above;
      histogram(h3, 0, 10, (d1 << 10) | d2);
      b = pick_bin<1, false>(h3, krem, wtot, &sh);
      thr = (d1 << 20) | (d2 << 10) | b.digit;
      want = (unsigned long long)(share * (double)(above1 + above2 + b.mass_above + b.mass));
    }
    // ---- nucleus: the smallest key whose mass of strictly larger keys is below top_p * (mass of the top-k set).  Bins above
    // the top-k threshold's are whole, so a walk that ends in one of them never meets a key below the threshold.
    if (P.top_p < 1.0f) {
      bool same = by_count;   // the walk is still on the top-k threshold's path: its histogram of this level is there
      if (!(same && want > above1)) {
        const BinPick b = pick_bin<4, true>(h1, want, wtot, &sh, by_count ? 0.0 : share);
        same = same && b.digit == d1;
        d1 = b.digit; above1 = b.mass_above;
      }
      want -= want ? above1 : 0;
      if (!same) {
        clear();
        __syncthreads();
        histogram(h2, 10, 10, d1);
      }
      if (!(same && want > above2)) {
        const BinPick b = pick_bin<1, true>(h2, want, wtot, &sh);
        same = same && b.digit == d2;
        d2 = b.digit; above2 = b.mass_above;
      }
      want -= want ? above2 : 0;
      if (!same) {
        h3[tid] = 0;
        __syncthreads();
        histogram(h3, 0, 10, (d1 << 10) | d2);
      }
      const BinPick b = pick_bin<1, true>(h3, want, wtot, &sh);
      thr = (d1 << 20) | (d2 << 10) | b.digit;
    }
  }

  // ---- draw from the kept tokens: chunk sums, then the chunk, the lane, the element (as the unfiltered kernel)
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int c = wave + 16 * q;
    if (c < nchunks) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) s += __float_as_uint(e[q][j]) >= thr ? e[q][j] : 0.f;
      s = wave_sum(s);
      if (lane == 0) csum[c] = s;
    }
  }
  __syncthreads();
  float incl = lane < nchunks ? csum[lane] : 0.f;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  const float Sk = __shfl(incl, 63, 64);
  const float target = (1.0f - sh_u) * Sk;
  const unsigned long long below = __ballot(lane < nchunks && incl < target);
  int ck = __popcll(below);
  if (ck > nchunks - 1) ck = nchunks - 1;
  // (a chunk without kept tokens has the inclusive sum of its predecessor, which is < target whenever it is chosen over,
  // so the chosen chunk always holds a kept token unless rounding pushed target past the total: then walk back)
  while (ck > 0 && (ck > 0 ? __shfl(incl, ck - 1, 64) : 0.f) >= Sk) ck--;
  ck = __builtin_amdgcn_readfirstlane(ck);
  if (wave == (ck & 15)) {   // the wave that holds the chunk
    const float before = ck > 0 ? __shfl(incl, ck - 1, 64) : 0.f;
    float ek[8];
    uint4 w = uint4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (q == ck >> 4) {
#pragma unroll
        for (int j = 0; j < 8; j++) ek[j] = __float_as_uint(e[q][j]) >= thr ? e[q][j] : 0.f;
        if constexpr (DT != UVMI_F32) w = raw[q];
      }
    float ls = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) ls += ek[j];
    float linc = ls;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float t = __shfl_up(linc, o, 64);
      if (lane >= o) linc += t;
    }
    linc += before;
    // the lane: the first one whose inclusive sum reaches target and that holds a kept token; when rounding pushed target
    // past the chunk's total, the last lane that holds one
    const unsigned long long has = __ballot(ls > 0.f);
    int ln = __popcll(__ballot(linc < target));
    {
      const unsigned long long hi = ln < 64 ? has & ~((1ull << ln) - 1ull) : 0ull;
      ln = hi ? __ffsll((long long)hi) - 1 : (has ? 63 - __clzll((long long)has) : 0);
    }
    // every lane walks its own elements from the sum ahead of it, for that one is among them: the first kept element whose running sum
    // reaches target, else the lane's last kept element
    const float prev = __shfl_up(linc, 1, 64);
    float run = lane > 0 ? prev : before, xsel;
    int sel = 0;
    bool found = false;
    float v[8];
    if constexpr (DT == UVMI_F32) load8<DT>(xr, ck * 64 + lane, v);
    else load8<DT>(&w, 0, v);
    xsel = v[0];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if (ek[j] > 0.f && !found) {
        run += ek[j];
        sel = j; xsel = v[j];
        if (run >= target) found = true;
      }
    }
    if (lane == ln) {
      const float E = __builtin_amdgcn_exp2f(fmaf(xsel, P.inv_c_l2, P.b_over_c_l2));
      sh_tok = ck * CHUNK + ln * 8 + sel;
      sh_lp = __builtin_amdgcn_rcpf(1.0f + E);
    }
  }
  const float S = wave == 0 ? wave_sum(lane < nchunks ? csum_all[lane] : 0.f) : 0.f;
  __syncthreads();
  if (tid == 0) {
    if (P.u_out) P.u_out[row] = sh_u;
    if (P.thr_out) P.thr_out[row] = __uint_as_float(thr);
    emit(P, row, sh_tok, P.neg_a_over_t * sh_lp - __logf(S), cr);
  }
}

// Greedy: argmax of the raw head output (the softcap is strictly increasing, so argmax z = argmax x), first maximal
// index; logp = log softmax(z)[tok] at T = 1.
// What bounds it: three quarter-rate instructions an element (exp2, reciprocal, exp2) on the compute unit that has the row, behind the
// launch and a load; with a commit, what that reads.  us with a commit, its reads at the end -> ahead and 1024 threads up to a row per
// compute unit: 1 row 8.3 -> 7.4, 16 rows 9.2 -> 8.0, 256 rows 10.4 -> 8.9; 640 rows 17.8 -> 16.5, 1024 rows 21.0 -> 19.8.
// The sum of exponentials is formed in 16 parts - a wave's of 1024 threads - at either width, so a row's log-prob does not depend on how many rows are in the
// call: 256 threads keep four sums each and add up each part as wave_sum does.  us so at 256 threads, one sum -> four: bf16 300 rows 10.7 -> 10.4, 1024 rows
// 19.5 -> 18.5, 2048 rows 32.3 -> 31.6; fp32 12.4 -> 12.6, 22.8 -> 23.0, 45.1 -> 45.5.
template <int DT, int NT>
__global__ __launch_bounds__(NT) void argmax_kernel(SampleParams P) {
  constexpr int NW = NT / 64, NP = 1024 / NT;
  __shared__ float smax[NW];
  __shared__ int sidx[NW];
  __shared__ __attribute__((aligned(16))) float ssum[16];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const char* xr = (const char*)P.x + (int64_t)row * P.stride * (DT == UVMI_F32 ? 4 : 2);
  const int nvec = P.V / 8;
  float best = -INFINITY, esum[NP] = {};   // esum[p]: vectors threadIdx.x + NT p of every 1024
  int bi = 0x7fffffff;
  CommitRow cr = {};
  if constexpr (NT == 256) cr = commit_ahead(P, row);
  auto take = [&](const float (&v)[8], int i, float& sum) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      if (v[j] > best) { best = v[j]; bi = i * 8 + j; }
      // softmax(z) with T = 1: e = exp(z - a)
      const float E = __builtin_amdgcn_exp2f(fmaf(v[j], P.inv_c_l2, P.b_over_c_l2));
      sum += __builtin_amdgcn_exp2f(-P.cap_a * 1.4426950408889634f * __builtin_amdgcn_rcpf(1.0f + E));
    }
  };
  if constexpr (NT == 1024) {   // (at most four vectors a thread: all requested at once)
    float v[4][8];
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (threadIdx.x + 1024 * q < nvec) load8<DT>(xr, threadIdx.x + 1024 * q, v[q]);
    cr = commit_ahead(P, row);
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (threadIdx.x + 1024 * q < nvec) take(v[q], threadIdx.x + 1024 * q, esum[0]);
  } else {
    auto one = [&](int i, float& sum) {
      float v[8];
      load8<DT>(xr, i, v);
      take(v, i, sum);
    };
    int i0 = 0;
    for (; i0 + 1024 <= nvec; i0 += 1024) {
#pragma unroll
      for (int p = 0; p < NP; p++) {
        one(i0 + NT * p + threadIdx.x, esum[p]);
        // (16-bit rows request all four at once: 640 rows 16.0 -> 14.5 us; fp32 ones lose by it, 800 rows 19.6 -> 22.1)
        if (DT == UVMI_F32) __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int p = 0; p < NP; p++)
      if (i0 + NT * p + (int)threadIdx.x < nvec) one(i0 + NT * p + threadIdx.x, esum[p]);
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
  }
  if constexpr (NP == 1) {
    esum[0] = wave_sum(esum[0]);
    if (lane == 0) ssum[wave] = esum[0];
  } else {   // wave_sum of the four at once: a swap adds the halves of two sums; rows 0 .. 3 of 16 lanes end with those of p = 0, 2, 1, 3
    auto fold = [](auto r) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
    const float a = fold(__builtin_amdgcn_permlane32_swap(__float_as_uint(esum[0]), __float_as_uint(esum[1]), false, false));
    const float b = fold(__builtin_amdgcn_permlane32_swap(__float_as_uint(esum[2]), __float_as_uint(esum[3]), false, false));
    float e = fold(__builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false));
    e += lane_xor8(e);
    e += lane_xor4(e);
    e += lane_xor2(e);
    e += lane_xor1(e);
    if (lane % 16 == 0) ssum[wave + NW * ((lane >> 5) + 2 * ((lane >> 4) & 1))] = e;
  }
  if (lane == 0) { smax[wave] = best; sidx[wave] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float4 x = ((const float4*)ssum)[w];
      tot = tot + x.x + x.y + x.z + x.w;
    }
    for (int w = 0; w < NW; w++) {
      if (smax[w] > best || (smax[w] == best && sidx[w] < bi)) { best = smax[w]; bi = sidx[w]; }
    }
    const float E = __builtin_amdgcn_exp2f(fmaf(best, P.inv_c_l2, P.b_over_c_l2));
    if (P.u_out) P.u_out[row] = 0.f;
    emit(P, row, bi, -P.cap_a * __builtin_amdgcn_rcpf(1.0f + E) - __logf(tot), cr);
  }
}

}  // namespace uvmi

using namespace uvmi;

extern "C" void uvmi_philox4x32_10(const uint32_t ctr[4], const uint32_t key[2], uint32_t out[4]) { philox4x32_10(ctr, key, out); }

extern "C" int uvmi_fused_sample(const uvmi_sample_args* a, void* stream) {
  UVMI_REQUIRE(a, UVMI_EINVAL, "uvmi_fused_sample: null args");
  UVMI_REQUIRE(a->x && a->tok && a->logp, UVMI_EINVAL, "uvmi_fused_sample: null pointer");
  UVMI_REQUIRE(is_float_dtype(a->x_dtype), UVMI_EINVAL, "uvmi_fused_sample: x_dtype must be a float type");
  UVMI_REQUIRE(a->B >= 0 && a->V > 0 && a->stride >= a->V, UVMI_EINVAL, "uvmi_fused_sample: bad sizes");
  UVMI_REQUIRE(a->V % CHUNK == 0 && a->V / CHUNK <= 64, UVMI_EUNSUPPORTED,
               "uvmi_fused_sample: V=%d must be a multiple of 512 and at most 32768", a->V);
  UVMI_REQUIRE(a->cap_c != 0.f, UVMI_EINVAL, "uvmi_fused_sample: softcap c must be non-zero");
  const int eb = a->x_dtype == UVMI_F32 ? 4 : 2;
  UVMI_REQUIRE(((uintptr_t)a->x % 16) == 0 && (a->stride * eb) % 16 == 0, UVMI_EUNSUPPORTED,
               "uvmi_fused_sample: rows of x must be 16-byte aligned");
  const bool greedy = !(a->temperature > 0.f);
  if (!greedy) {
    UVMI_REQUIRE(a->cap_a / a->temperature <= 80.0f, UVMI_EUNSUPPORTED, "uvmi_fused_sample: a/T = %g exceeds 80 (fp32 underflow)",
                 (double)(a->cap_a / a->temperature));
    UVMI_REQUIRE(a->u || (a->req_id && a->tok_idx), UVMI_EINVAL, "uvmi_fused_sample: need u or (req_id, tok_idx)");
  }
  if (a->B == 0) return UVMI_OK;
  SampleParams P;
  P.x = a->x; P.stride = a->stride; P.u = a->u; P.seed = a->seed; P.req_id = a->req_id; P.tok_idx = a->tok_idx;
  P.tok = a->tok; P.logp = a->logp; P.u_out = a->u_out; P.V = a->V;
  const float l2e = 1.4426950408889634f;
  P.inv_c = 1.0f / a->cap_c;
  P.inv_c_l2 = l2e / a->cap_c;
  P.b_over_c_l2 = a->cap_b / a->cap_c * l2e;
  const float T = greedy ? 1.0f : a->temperature;
  P.neg_a_over_t = -a->cap_a / T;
  P.neg_a_over_t_l2 = P.neg_a_over_t * l2e;
  P.cap_a = a->cap_a; P.cap_b = a->cap_b; P.cap_c = a->cap_c;
  P.top_k = a->top_k > 0 && a->top_k < a->V ? a->top_k : 0;
  P.top_p = a->top_p > 0.f && a->top_p < 1.0f ? a->top_p : 1.0f;
  P.thr_out = a->thr_out;
  P.commit = 0;
  if (a->commit) {
    const uvmi_sample_commit* c = a->commit;
    UVMI_REQUIRE(c->state && c->act_slot && c->tok_c && c->pos_c && c->starts_c && c->req_c && c->cnt_c, UVMI_EINVAL,
                 "uvmi_fused_sample: null pointer in commit");
    const uvmi_sched_state* t = c->state;
    UVMI_REQUIRE(t->slot_req && t->slot_cnt && t->slot_limit && t->slot_tok && t->pos && t->starts && t->out_tok && t->counters && t->done_req &&
                     t->done_slot && t->done_cnt && t->B > 0 && t->max_new > 0 && t->done_cap > 0, UVMI_EINVAL,
                 "uvmi_fused_sample: bad slot table in commit");
    // the kernel reads req_id / tok_idx of a row before it rewrites the row's dense entries, so they may be the same arrays
    P.commit = 1; P.retire_p = c->retire_p; P.commit_seed = c->seed; P.S = *t;
    P.D = DenseArrays{c->act_slot, c->tok_c, c->pos_c, c->starts_c, c->req_c, c->cnt_c};
  }
  const bool filtered = !greedy && (P.top_k > 0 || P.top_p < 1.0f);
  hipStream_t st = (hipStream_t)stream;
  // Drawing, 1024 threads per row are faster up to ~640 rows (12.0 against 14.5 us at 384 rows), slower from 1024 on; its sums are formed per
  // chunk whatever the width, so the draw does not depend on it.  Greedy, whose sums do not either, up to a row per compute unit (256
  // rows 8.4 against 8.7, 300 rows 12.9 against 10.8).
  int cus = uvmi_device_cus();
  if (cus <= 0) cus = 256;
  const bool wide = filtered || a->B <= (greedy ? cus : 640);
  const dim3 grid(a->B), blk(wide ? 1024 : 256);
#define UVMI_S(...) hipLaunchKernelGGL((__VA_ARGS__), grid, blk, 0, st, P)
#define UVMI_SK(DT, NT) \
  hipLaunchKernelGGL((sample_kernel<DT, NT>), grid, blk, 0, st, P.x, P.stride, P.V, P.inv_c_l2, P.b_over_c_l2, P.neg_a_over_t_l2, P)
#define UVMI_DT(DT)                                                                                      \
  do {                                                                                                   \
    if (filtered) UVMI_S(sample_filtered_kernel<DT>);                                                    \
    else if (greedy) { if (wide) UVMI_S(argmax_kernel<DT, 1024>); else UVMI_S(argmax_kernel<DT, 256>); } \
    else { if (wide) UVMI_SK(DT, 1024); else UVMI_SK(DT, 256); }                                         \
  } while (0)
  if (a->x_dtype == UVMI_F16) UVMI_DT(UVMI_F16);
  else if (a->x_dtype == UVMI_BF16) UVMI_DT(UVMI_BF16);
  else UVMI_DT(UVMI_F32);
#undef UVMI_DT
#undef UVMI_SK
#undef UVMI_S
  UVMI_CHECK_LAUNCH("uvmi_fused_sample");
  return UVMI_OK;
}
