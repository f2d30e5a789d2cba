// Fused per-token kernels of the UV-50M decode / prefill step: everything between the GEMMs.
//
// One wave64 per token row.  All arithmetic is fp32; values are rounded to the activation type T (fp16 / bf16 / fp32)
// where the next GEMM reads them.  Weightless RMSNorm takes its eps from the caller: the reference calls
// torch.nn.functional.rms_norm(x, eps=None) (ultraviolet/model.py:190-191), whose default has been the machine epsilon
// of the input dtype in some torch releases and of fp32 in others, so the host passes what its torch does.
//
//   embed_norm   x = rmsnorm(E[tok]); n = rmsnorm(x)                                    (fast_decode.py:286, 305)
//   add_norm     h = a*x + b*y; n = rmsnorm(h)          residual lambdas + pre-norm     (model.py:567-571)
//   qkv_post     value-embedding gate, QK-norm, partial RoPE, q out, int8 K/V append    (model.py:302-319,
//                                                                                        fast_decode.py:291-294, 315-317)
//   attn_post    XSA projection removal + per-head sigmoid gate                         (model.py:321-333)
//   swiglu       silu(g) * u                                                            (model.py:388-391)
//
// All of them are HBM/launch-bound and tiny next to the GEMMs and attention; they exist to keep the step at a handful
// of launches per layer and to write K/V straight into the int8 cache without a round trip through HBM.
#include "common.h"
#include "qkv_post.h"

#include <type_traits>

namespace uvmi {

template <int DT> __device__ __forceinline__ float round_t(float v);
template <> __device__ __forceinline__ float round_t<UVMI_F32>(float v) { return v; }
template <> __device__ __forceinline__ float round_t<UVMI_F16>(float v) { return (float)(half_t)v; }
template <> __device__ __forceinline__ float round_t<UVMI_BF16>(float v) { return bf16_to_float(float_to_bf16(v)); }

template <int DT>
__device__ __forceinline__ void ld2(const void* p, int64_t i, float& a, float& b) {  // elements i, i+1 (i even)
  if (DT == UVMI_F32) { const float2 v = *(const float2*)((const float*)p + i); a = v.x; b = v.y; }
  else {
    const uint32_t w = *(const uint32_t*)((const uint16_t*)p + i);
    if (DT == UVMI_BF16) { a = __uint_as_float(w << 16); b = __uint_as_float(w & 0xffff0000u); }
    else { a = half_bits_to_float(w & 0xffff); b = half_bits_to_float(w >> 16); }
  }
}
template <int DT>
__device__ __forceinline__ void st2(void* p, int64_t i, float a, float b) {
  if (DT == UVMI_F32) *(float2*)((float*)p + i) = float2{a, b};
  else {
    const uint32_t lo = DT == UVMI_BF16 ? float_to_bf16(a) : float_to_half_bits(a);
    const uint32_t hi = DT == UVMI_BF16 ? float_to_bf16(b) : float_to_half_bits(b);
    *(uint32_t*)((uint16_t*)p + i) = lo | (hi << 16);
  }
}

template <int DT>
__device__ __forceinline__ void unpack8(uint4 w, float (&o)[8]) {  // 8 elements of a 16-bit type
  const uint32_t r[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (DT == UVMI_BF16) { o[2 * j] = __uint_as_float(r[j] << 16); o[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u); }
    else { o[2 * j] = half_bits_to_float(r[j] & 0xffff); o[2 * j + 1] = half_bits_to_float(r[j] >> 16); }
  }
}
template <int DT>
__device__ __forceinline__ void ld8(const void* p, int64_t i, float (&o)[8]) {  // 8 consecutive elements starting at i
  if (DT == UVMI_F32) {
    const float4 a = *(const float4*)((const float*)p + i), b = *(const float4*)((const float*)p + i + 4);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  } else {
    unpack8<DT>(*(const uint4*)((const uint16_t*)p + i), o);
  }
}
template <int DT>
__device__ __forceinline__ void st8(void* p, int64_t i, const float (&v)[8]) {
  if (DT == UVMI_F32) {
    *(float4*)((float*)p + i) = float4{v[0], v[1], v[2], v[3]};
    *(float4*)((float*)p + i + 4) = float4{v[4], v[5], v[6], v[7]};
  } else {
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (DT == UVMI_BF16) r[j] = float2_to_bf16x2(v[2 * j], v[2 * j + 1]);
      else r[j] = (uint32_t)float_to_half_bits(v[2 * j]) | ((uint32_t)float_to_half_bits(v[2 * j + 1]) << 16);
    }
    *(uint4*)((uint16_t*)p + i) = uint4{r[0], r[1], r[2], r[3]};
  }
}

// ------------------------------------------------------------------------------------------------ embed / residual
// MODE 0: src = E[tok[r]] ; x = rmsnorm(src)        MODE 1: x = a*xin + b*yin
// then n = rmsnorm(x) (of the rounded x).  NP: pairs per lane, d <= 64 * 2 * NP.
// A row is a chain of trips - its token, its elements, its stores - and its elements are requested together: pairs past the row are read from its last one
// and count as zeros.  (With a branch around each pair every load was waited for by itself, five of them at d = 640.)  Embedding
// and norm, d = 640, us in a stream: 1 row 3.3 -> 2.9, 512 rows 3.8 -> 2.9, 18 432 rows 17.5 -> 13.3, 33 216 29.2 -> 21.5 (5.9 TB/s); the same bits.
// Requests past the row's end cost what the row's own do, so NP is the width's: residual norm of 33 216 rows with branches / in the form of 5 or 16 pairs /
// now, d = 64 9.3 / 11.9 / 6.4, 642 29.0 / 31.9 / 26.7, 768 31.6 / 32.3 / 30.0, 1280 67.0 / 60.1 / 60.2; 4096 rows of 768 6.0 / 7.1 / 5.1.
template <int DT, int MODE, int NP>
__global__ __launch_bounds__(256) void norm_kernel(const void* __restrict__ xin, const void* __restrict__ yin,
                                                   const int64_t* __restrict__ tok, int64_t vocab, float a, float b,
                                                   void* __restrict__ xout, void* __restrict__ nout, int64_t rows, int d, float eps,
                                                   int64_t* __restrict__ advance) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int np = d / 2;
  float v0[NP], v1[NP], y0[NP], y1[NP];
  float ss = 0.f;
  int64_t src = r;
  if (advance && lane == 0) atomicAdd((unsigned long long*)advance + r, 1ull);   // (nothing waits for it)
  if (MODE == 0) {
    src = tok[r];
    if (src < 0) src = 0;
    if (src >= vocab) src = vocab - 1;
  }
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int pidx = min(lane + 64 * i, np - 1);
    ld2<DT>(xin, src * d + 2 * pidx, v0[i], v1[i]);
    if (MODE == 1) ld2<DT>(yin, r * d + 2 * pidx, y0[i], y1[i]);
  }
#pragma unroll
  for (int i = 0; i < NP; i++) {
    if (MODE == 1) {
      v0[i] = round_t<DT>(fmaf(a, v0[i], b * y0[i]));   // (which product is rounded is said, for the forms' results to be the same bits)
      v1[i] = round_t<DT>(fmaf(a, v1[i], b * y1[i]));
    }
    if (lane + 64 * i >= np) v0[i] = v1[i] = 0.f;
    ss += v0[i] * v0[i] + v1[i] * v1[i];
  }
  if (MODE == 0) {
    const float rs = rsqrtf(wave_sum(ss) / (float)d + eps);
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      v0[i] = round_t<DT>(v0[i] * rs); v1[i] = round_t<DT>(v1[i] * rs);
      ss += v0[i] * v0[i] + v1[i] * v1[i];
    }
  }
  const float rn = rsqrtf(wave_sum(ss) / (float)d + eps);
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int pidx = lane + 64 * i;
    if (pidx < np) {
      if (xout) st2<DT>(xout, r * d + 2 * pidx, v0[i], v1[i]);
      st2<DT>(nout, r * d + 2 * pidx, v0[i] * rn, v1[i] * rn);
    }
  }
}

// ------------------------------------------------------------------------------------------------ qkv_post (hd = 64)
template <int DT>
__global__ __launch_bounds__(256) void qkv_post_kernel(QkvArgs A) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= A.n) return;
  const int W = (A.H + 2 * A.KH) * 64;
  const int64_t base = r * A.ld;
  const int64_t p = A.pos[r];
  const int np_ = A.n_pairs;
  const float* tab = A.rope_tab && p >= 0 && p < A.rope_n ? A.rope_tab + p * 2 * np_ : nullptr;   // (wave-uniform)
  // ---- queries: lane (hh = lane / 8, c = lane % 8) owns dims 8c..8c+7 of head 8*pass + hh
  {
    const int hh = lane >> 3, c = lane & 7;
    // RoPE angles of this lane's 8 dims (dims < 2 n_pairs rotate; dim j pairs with j +- n_pairs): one cos / sin per
    // frequency is computed by lanes 0..n_pairs-1 and fetched by shuffle
    float cs[8], sn[8];
    {
      float cl = 1.f, sl = 0.f;
      if (A.rope && lane < np_) {
        if (tab) {
          cl = tab[lane];
          sl = tab[np_ + lane];
        } else {
          const float th = (float)p * A.inv_freq[lane];
          cl = round_t<DT>(cosf(th));
          sl = round_t<DT>(sinf(th));
        }
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int dim = 8 * c + j;
        const int src = A.rope ? dim % np_ : 0;
        const float cj = __shfl(cl, src, 64), sj = __shfl(sl, src, 64);
        const bool rot = A.rope && dim < 2 * np_;
        cs[j] = rot ? cj : 1.f;
        sn[j] = rot ? sj : 0.f;
      }
    }
    const int pl = np_ / 8;  // lane distance of the RoPE partner chunk (n_pairs is a multiple of 8, host-checked)
    for (int h0 = 0; h0 < A.H; h0 += 8) {
      const int h = h0 + hh;
      float x[8];
      if (h < A.H) ld8<DT>(A.qkv, base + h * 64 + 8 * c, x);
      else {
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = 0.f;
      }
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) ss += x[j] * x[j];
      ss += lane_xor1(ss); ss += lane_xor2(ss); ss += lane_xor4(ss);
      const float rs = rsqrtf(ss * (1.0f / 64.0f) + A.eps);
#pragma unroll
      for (int j = 0; j < 8; j++) x[j] = round_t<DT>(x[j] * rs);
      if (A.rope) {
        const bool first = 8 * c < np_, rot = 8 * c < 2 * np_;
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; j++) y[j] = pl == 2 ? lane_xor2(x[j]) : __shfl_xor(x[j], pl, 64);  // partner chunk: c <-> c ^ pl inside the head
        if (rot) {
#pragma unroll
          for (int j = 0; j < 8; j++) x[j] = rope_rot(x[j], y[j], cs[j], sn[j], first, [](float f) { return round_t<DT>(f); });
        }
      }
      if (h < A.H) {
        const int64_t o = (r * A.H + h) * 64 + 8 * c;
        if (A.q_dt == UVMI_BF16) st8<UVMI_BF16>(A.q_out, o, x); else if (A.q_dt == UVMI_F32) st8<UVMI_F32>(A.q_out, o, x); else st8<UVMI_F16>(A.q_out, o, x);
      }
    }
    // ---- per-head output gate 2 sigmoid(W_h . xn[:gate_ch]) for the attention epilogue (model.py:330-333)
    if (A.gate_out) {
      const int cpl = A.gate_ch / 8;  // channels per lane (a multiple of 8 when gate_ch % 64 == 0, else the scalar loop)
      for (int h0 = 0; h0 < A.H; h0 += 8) {
        const int h = h0 + hh;
        float dot = 0.f;
        if (A.ext) {   // the projection formed the logit (already rounded to the activation type)
          if (h < A.H && c == 0) dot = elem<DT>::ld(A.qkv, base + W + h);
        } else if (h < A.H) {
          if (cpl % 8 == 0 && (A.d % 8) == 0) {
            for (int j = 0; j < cpl; j += 8) {
              float xv[8];
              ld8<DT>(A.xn, r * A.d + c * cpl + j, xv);
              const float4 w0 = *(const float4*)(A.gate_w + h * A.gate_ch + c * cpl + j), w1 = *(const float4*)(A.gate_w + h * A.gate_ch + c * cpl + j + 4);
              dot += xv[0] * w0.x + xv[1] * w0.y + xv[2] * w0.z + xv[3] * w0.w + xv[4] * w1.x + xv[5] * w1.y + xv[6] * w1.z + xv[7] * w1.w;
            }
          } else {
            for (int j = 0; j < cpl; j++) dot += elem<DT>::ld(A.xn, r * A.d + c * cpl + j) * A.gate_w[h * A.gate_ch + c * cpl + j];
          }
        }
        dot += lane_xor1(dot); dot += lane_xor2(dot); dot += lane_xor4(dot);
        dot = round_t<DT>(dot);
        if (h < A.H && c == 0) A.gate_out[r * A.H + h] = round_t<DT>(2.0f * round_t<DT>(1.0f / (1.0f + __expf(-dot))));
      }
    }
  }
  // ---- keys / values per kv head: lane = dim
  float cs1 = 1.f, sn1 = 0.f;
  const bool rot1 = A.rope && lane < 2 * np_;
  if (rot1) {
    if (tab) {
      cs1 = tab[lane % np_];
      sn1 = tab[np_ + lane % np_];
    } else {
      const float th = (float)p * A.inv_freq[lane % np_];
      cs1 = round_t<DT>(cosf(th));
      sn1 = round_t<DT>(sinf(th));
    }
  }
  const int64_t row = A.rows ? A.rows[r] : r;
  const int64_t slot = A.ring ? (p % A.S) : p;
  bool wr = A.k_cache && row >= 0 && p >= 0 && slot < A.S;
  if (wr && A.ring && A.last_pos) wr = p > A.last_pos[r] - A.S;  // only the last S positions of a prompt survive in a ring
  for (int kh = 0; kh < A.KH; kh++) {
    float k = elem<DT>::ld(A.qkv, base + (A.H + kh) * 64 + lane);
    {
      const float rs = rsqrtf(wave_sum(k * k) * (1.0f / 64.0f) + A.eps);
      k = round_t<DT>(k * rs);
      if (A.rope) {
        const float other = np_ == 16 ? lane_xor16(k) : __shfl_xor(k, np_, 64);
        if (rot1) k = rope_rot(k, other, cs1, sn1, lane < np_, [](float f) { return round_t<DT>(f); });
      }
    }
    float v = elem<DT>::ld(A.qkv, base + (A.H + A.KH + kh) * 64 + lane);
    if (A.has_ve) {  // v += 2 sigmoid(W xn[:ve_ch]) * value_embed[tok]
      float dot = 0.f;
      if (A.ext) dot = elem<DT>::ld(A.qkv, base + W + A.H + kh);
      else {
        if (lane < A.ve_ch) dot = elem<DT>::ld(A.xn, r * A.d + lane) * A.ve_gate[kh * A.ve_ch + lane];
        dot = round_t<DT>(wave_sum(dot));
      }
      const float g = round_t<DT>(2.0f * round_t<DT>(1.0f / (1.0f + __expf(-dot))));
      int64_t t = A.tok[r];
      if (t < 0) t = 0;
      if (t >= A.vocab) t = A.vocab - 1;
      const float ve = elem<DT>::ld(A.ve_table, (t * A.KH + kh) * 64 + lane);
      v = ve_add(v, g, ve, [](float f) { return round_t<DT>(f); });
    }
    if (A.k_out) elem<DT>::st(A.k_out, (r * A.KH + kh) * 64 + lane, k);
    if (A.v_out) elem<DT>::st(A.v_out, (r * A.KH + kh) * 64 + lane, v);
    if (A.vhat_out) {  // v / max(|v|, eps) in fp32 for the XSA epilogue (model.py:327)
      const float nv = sqrtf(wave_sum(v * v));
      A.vhat_out[(r * A.KH + kh) * 64 + lane] = v / fmaxf(nv, A.xsa_eps);
    }
    if (wr && !A.k_scale) {   // an unquantized cache: the values as they are
      const int64_t at = row * A.scb + kh * A.sch + slot * A.scs + lane;
      elem<DT>::st(A.k_cache, at, k);
      elem<DT>::st(A.v_cache, at, v);
    } else if (wr) {  // int8 append, same arithmetic as the standalone quantizer
      const float vals[2] = {k, v};
      int8_t* caches[2] = {A.k_cache, A.v_cache};
      uint16_t* scales[2] = {A.k_scale, A.v_scale};
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const float am = wave_max(fabsf(vals[j]));
        const uint16_t sb = float_to_half_bits(__fdiv_rn(am, 127.0f));
        const float sf = fmaxf(half_bits_to_float(sb), 1e-30f);
        float qv = __builtin_rintf(__fdiv_rn(vals[j], sf));
        qv = fminf(fmaxf(qv, -127.0f), 127.0f);
        caches[j][row * A.scb + kh * A.sch + slot * A.scs + lane] = (int8_t)(int)qv;
        if (lane == 0) scales[j][row * A.ssb + kh * A.ssh + slot] = sb;
      }
    }
  }
}

// The same post-processing for the engine's shape - 8 query heads on one kv head, 16 rotated pairs with the rotation
// table, gate logits formed by the projection (ext), q written in the activation type - with everything a row needs
// requested in two batches: first what depends on the row index alone (position, cache row, token, the row's q / k / v and
// logits), then what depends on those (the rotation table's row, the value embedding).  The general kernel above meets
// these loads one after the other between branches and loops, a chain of six memory latencies per row; the arithmetic,
// its order and its roundings are the same, so the two kernels agree bit for bit.
template <int DT>
__global__ __launch_bounds__(256) void qkv_post_fast_kernel(QkvArgs A) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= A.n) return;
  constexpr int W = 10 * 64;
  auto rnd = [](float f) { return round_t<DT>(f); };
  const int64_t base = r * A.ld;
  const int hh = lane >> 3, c = lane & 7;
  // ---- requests that depend on the row index alone
  const int64_t p = A.pos[r];
  const int64_t row = A.rows ? A.rows[r] : r;
  const int64_t lastp = A.last_pos ? A.last_pos[r] : 0;
  int64_t t = A.has_ve ? A.tok[r] : 0;
  float x[8];
  ld8<DT>(A.qkv, base + hh * 64 + 8 * c, x);
  float k = elem<DT>::ld(A.qkv, base + 8 * 64 + lane);
  float v = elem<DT>::ld(A.qkv, base + 9 * 64 + lane);
  const float glog = A.gate_out ? elem<DT>::ld(A.qkv, base + W + hh) : 0.f;
  const float vlog = A.has_ve ? elem<DT>::ld(A.qkv, base + W + 8) : 0.f;
  // ---- requests that depend on the position and the token
  const bool in_tab = p >= 0 && p < A.rope_n;   // (wave-uniform)
  const float* tab = A.rope_tab + (in_tab ? p : 0) * 32;
  float cs[8], sn[8], cs1 = 1.f, sn1 = 0.f;
  if (A.rope) {
    const float* tq = tab + 8 * (c & 1);   // dim 8 c + j turns by frequency (8 c + j) % 16
    const float4 c0 = *(const float4*)tq, c1 = *(const float4*)(tq + 4), s0 = *(const float4*)(tq + 16), s1 = *(const float4*)(tq + 20);
    cs[0] = c0.x; cs[1] = c0.y; cs[2] = c0.z; cs[3] = c0.w; cs[4] = c1.x; cs[5] = c1.y; cs[6] = c1.z; cs[7] = c1.w;
    sn[0] = s0.x; sn[1] = s0.y; sn[2] = s0.z; sn[3] = s0.w; sn[4] = s1.x; sn[5] = s1.y; sn[6] = s1.z; sn[7] = s1.w;
    cs1 = tab[lane & 15];
    sn1 = tab[16 + (lane & 15)];
  }
  if (t < 0) t = 0;
  if (t >= A.vocab) t = A.vocab - 1;
  const float ve = A.has_ve ? elem<DT>::ld(A.ve_table, t * 64 + lane) : 0.f;
  if (A.rope && !in_tab) {   // a position outside the table: the angles are formed here, as the general kernel does
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float th = (float)p * A.inv_freq[8 * (c & 1) + j];
      cs[j] = rnd(cosf(th));
      sn[j] = rnd(sinf(th));
    }
    const float th = (float)p * A.inv_freq[lane & 15];
    cs1 = rnd(cosf(th));
    sn1 = rnd(sinf(th));
  }
  // ---- queries: lane (hh, c) owns dims 8c..8c+7 of head hh
  {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) ss += x[j] * x[j];
    ss += lane_xor1(ss); ss += lane_xor2(ss); ss += lane_xor4(ss);
    const float rs = rsqrtf(ss * (1.0f / 64.0f) + A.eps);
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = rnd(x[j] * rs);
    if (A.rope) {
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; j++) y[j] = lane_xor2(x[j]);   // partner chunk: c <-> c ^ 2 inside the head
      if (c < 4) {
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = rope_rot(x[j], y[j], cs[j], sn[j], c < 2, rnd);
      }
    }
    st8<DT>(A.q_out, (r * 8 + hh) * 64 + 8 * c, x);
    if (A.gate_out && c == 0) A.gate_out[r * 8 + hh] = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-glog))));
  }
  // ---- key and value: lane = dim
  {
    const float rs = rsqrtf(wave_sum(k * k) * (1.0f / 64.0f) + A.eps);
    k = rnd(k * rs);
    if (A.rope) {
      const float other = lane_xor16(k);
      if (lane < 32) k = rope_rot(k, other, cs1, sn1, lane < 16, rnd);
    }
  }
  if (A.has_ve) {
    const float g = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-vlog))));
    v = ve_add(v, g, ve, rnd);
  }
  if (A.k_out) elem<DT>::st(A.k_out, r * 64 + lane, k);
  if (A.v_out) elem<DT>::st(A.v_out, r * 64 + lane, v);
  if (A.vhat_out) {
    const float nv = sqrtf(wave_sum(v * v));
    A.vhat_out[r * 64 + lane] = v / fmaxf(nv, A.xsa_eps);
  }
  const int64_t slot = A.ring ? (p % A.S) : p;
  bool wr = A.k_cache && row >= 0 && p >= 0 && slot < A.S;
  if (wr && A.ring && A.last_pos) wr = p > lastp - A.S;
  if (wr && !A.k_scale) {
    elem<DT>::st(A.k_cache, row * A.scb + slot * A.scs + lane, k);
    elem<DT>::st(A.v_cache, row * A.scb + slot * A.scs + lane, v);
  } else if (wr) {
    const float vals[2] = {k, v};
    int8_t* caches[2] = {A.k_cache, A.v_cache};
    uint16_t* scales[2] = {A.k_scale, A.v_scale};
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float am = wave_max(fabsf(vals[j]));
      const uint16_t sb = float_to_half_bits(__fdiv_rn(am, 127.0f));
      const float sf = fmaxf(half_bits_to_float(sb), 1e-30f);
      float qv = __builtin_rintf(__fdiv_rn(vals[j], sf));
      qv = fminf(fmaxf(qv, -127.0f), 127.0f);
      caches[j][row * A.scb + slot * A.scs + lane] = (int8_t)(int)qv;
      if (lane == 0) scales[j][row * A.ssb + slot] = sb;
    }
  }
}

// The same again for passes of many rows: a wave owns 8 rows, lane (i, c) dims 8 c .. 8 c + 7 of row i, for the keys and values too, and
// walks the query heads.  What bounded the kernel above there was its vector instructions (the key and value of a row, an element per lane:
// six-step reductions, divisions and rounding for one row at a time) and the rotation table's row read per head; here a reduction serves 8
// rows, the table's row all heads and the key, every access is 16 bytes per lane, and all rows of a pass of 33 000 are in flight at once.
// wave_sum's order of additions (dims d ^ 32, 16, 8, 4, 2, 1) is kept, so the three kernels agree bit for bit.  us, one row per wave -> 8:
// 33 216 rows 34.2 -> 26.5, with a value embedding 42.6 -> 28.1; 18 432 rows 18.3 -> 16.7 and 20.4 -> 17.3 (100 MB at 33 216 rows: what bounds it
// is memory now, behind ~4 us of latencies; with the queries before the keys the stores come in a burst, 30 us).
__device__ __forceinline__ float row_sum(const float (&e)[8], int c) {   // of 8 lanes x 8 elements, in wave_sum's order
  float a[4], b[2];
#pragma unroll
  for (int j = 0; j < 4; j++) a[j] = add_sep(c & 4 ? e[4 + j] : e[j], lane_xor4(c & 4 ? e[j] : e[4 + j]));
#pragma unroll
  for (int j = 0; j < 2; j++) b[j] = add_sep(c & 2 ? a[2 + j] : a[j], lane_xor2(c & 2 ? a[j] : a[2 + j]));
  float u = add_sep(c & 1 ? b[1] : b[0], lane_xor1(c & 1 ? b[0] : b[1]));   // sum over the lanes of element c
  u = add_sep(u, lane_xor4(u));
  u = add_sep(u, lane_xor2(u));
  return add_sep(u, lane_xor1(u));
}
// Q false: the projection's epilogue has the query heads (QueryPost); what is left of them here is the rotation of rows whose position the table does
// not hold.  18 432 rows 16.1 us with the query heads, 8.5 without (a copy of what is left would take 4), 33 216 rows 24.7 / 11.9; with arguments and arrays
// asked for one by one and divisions in the quantiser 9.3 and 13.6: it is bound by its chain of trips and, at many rows, by its instructions.
template <int DT, bool Q>
__global__ __launch_bounds__(64) void qkv_post_rows_kernel(QkvArgs A) {
  const int lane = threadIdx.x & 63, c = lane & 7;
  const int64_t r0 = (int64_t)blockIdx.x * 8, r1 = r0 + (lane >> 3);
  // (the arguments that branches further down ask for, with the first ones: each was a trip of its own)
  asm volatile("" :: "s"(A.k_out), "s"(A.v_out), "s"(A.vhat_out), "s"(A.gate_out), "s"(A.k_cache), "s"(A.v_cache), "s"(A.k_scale), "s"(A.v_scale), "s"(A.scb),
               "s"(A.scs), "s"(A.ssb), "s"(A.S), "s"(A.ring), "s"(A.rope), "s"(A.rope_tab), "s"(A.rope_n), "s"(A.ve_table), "s"(A.vocab), "s"(A.eps), "s"(A.xsa_eps));
  if (r0 >= A.n) return;
  const bool live = r1 < A.n;
  const int64_t r = live ? r1 : A.n - 1;   // (a lane past the last row computes it again and stores nothing)
  auto rnd = [](float f) { return round_t<DT>(f); };
  const uint16_t* src = (const uint16_t*)A.qkv + r * A.ld + 8 * c;
  // ---- requests that depend on the row index alone
  // (all at once, an array that is not there read as another: behind a branch each, they were waited for one by one)
  const int64_t p = A.pos[r], rows_r = (A.rows ? A.rows : A.pos)[r], lastp = (A.last_pos ? A.last_pos : A.pos)[r];
  int64_t t = (A.has_ve ? A.tok : A.pos)[r];
  const int64_t row = A.rows ? rows_r : r;
  const uint4 kw = *(const uint4*)(src + 512), vw = *(const uint4*)(src + 576);
  const uint16_t gw = ((const uint16_t*)A.qkv)[r * A.ld + 640 + c], tw = ((const uint16_t*)A.qkv)[r * A.ld + 648];   // head c's gate, the value embedding's
  uint4 qw[Q ? 8 : 1];
  if constexpr (Q) {
#pragma unroll
    for (int h = 0; h < 8; h++) qw[h] = *(const uint4*)(src + 64 * h);
  }
  // ---- requests that depend on the position and the token
  const bool in_tab = p >= 0 && p < A.rope_n;
  float cs[8], sn[8];   // dim 8 c + j turns by frequency (8 c + j) % 16
  if (A.rope) {
    const float* tq = A.rope_tab + (in_tab ? p : 0) * 32 + 8 * (c & 1);
    const float4 c0 = *(const float4*)tq, c1 = *(const float4*)(tq + 4), s0 = *(const float4*)(tq + 16), s1 = *(const float4*)(tq + 20);
    cs[0] = c0.x; cs[1] = c0.y; cs[2] = c0.z; cs[3] = c0.w; cs[4] = c1.x; cs[5] = c1.y; cs[6] = c1.z; cs[7] = c1.w;
    sn[0] = s0.x; sn[1] = s0.y; sn[2] = s0.z; sn[3] = s0.w; sn[4] = s1.x; sn[5] = s1.y; sn[6] = s1.z; sn[7] = s1.w;
  }
  const float glog = elem<DT>::ld(&gw, 0), vlog = elem<DT>::ld(&tw, 0);
  if (t < 0) t = 0;
  if (t >= A.vocab) t = A.vocab - 1;
  uint4 ew = uint4{0u, 0u, 0u, 0u};
  if (A.has_ve) ew = *(const uint4*)((const uint16_t*)A.ve_table + t * 64 + 8 * c);
  if (A.rope && __any(!in_tab)) {   // a position outside the table: the angles are formed here (one at a time: there are few, and cosf is long)
#pragma unroll 1
    for (int j = 0; j < 8; j++) {
      const float th = (float)p * A.inv_freq[8 * (c & 1) + j];
      const float cj = rnd(cosf(th)), sj = rnd(sinf(th));
#pragma unroll
      for (int q = 0; q < 8; q++)
        if (!in_tab && q == j) { cs[q] = cj; sn[q] = sj; }
    }
  }
  if (A.rope && c < 2) {
#pragma unroll
    for (int j = 0; j < 8; j++) sn[j] = -sn[j];
  }
  auto round8 = [&](float (&x)[8]) {   // (in pairs: three instructions for two bf16 values)
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      if constexpr (DT == UVMI_BF16) {
        const uint32_t w = float2_to_bf16x2(x[j], x[j + 1]);
        x[j] = __uint_as_float(w << 16);
        x[j + 1] = __uint_as_float(w & 0xffff0000u);
      } else {
        x[j] = rnd(x[j]);
        x[j + 1] = rnd(x[j + 1]);
      }
    }
  };
  auto rotate = [&](float (&x)[8]) {   // (rope_rot)
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; j++) y[j] = lane_xor2(x[j]);   // partner chunk: c <-> c ^ 2 inside the head
    if (c < 4) {
#pragma unroll
      for (int j = 0; j < 8; j++) { x[j] = mul_sep(x[j], cs[j]); y[j] = mul_sep(y[j], sn[j]); }
      round8(x);
      round8(y);
#pragma unroll
      for (int j = 0; j < 8; j++) x[j] = add_sep(x[j], y[j]);
      round8(x);
    }
  };
  // ---- key and value
  float k[8], v[8];
  unpack8<DT>(kw, k);
  unpack8<DT>(vw, v);
  {
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; j++) e[j] = mul_sep(k[j], k[j]);
    const float rs = rsqrtf(row_sum(e, c) * (1.0f / 64.0f) + A.eps);
#pragma unroll
    for (int j = 0; j < 8; j++) k[j] = k[j] * rs;
    round8(k);
    if (A.rope) rotate(k);
  }
  if (A.has_ve) {
    const float g = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-vlog))));
    float e[8];
    unpack8<DT>(ew, e);
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = ve_add(v[j], g, e[j], rnd);
  }
  if (live && A.k_out) st8<DT>(A.k_out, r * 64 + 8 * c, k);
  if (live && A.v_out) st8<DT>(A.v_out, r * 64 + 8 * c, v);
  if (A.vhat_out) {
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; j++) e[j] = mul_sep(v[j], v[j]);
    const float nv = fmaxf(sqrtf(row_sum(e, c)), A.xsa_eps);
#pragma unroll
    for (int j = 0; j < 8; j++) e[j] = v[j] / nv;
    if (live) st8<UVMI_F32>(A.vhat_out, r * 64 + 8 * c, e);
  }
  const int64_t slot = A.ring ? (p % A.S) : p;
  bool wr = live && A.k_cache && row >= 0 && p >= 0 && slot < A.S;
  if (A.ring && A.last_pos && p <= lastp - A.S) wr = false;   // only the last S positions of a prompt survive in a ring
  if (A.k_cache && !A.k_scale) {
    if (wr) {
      st8<DT>(A.k_cache, row * A.scb + slot * A.scs + 8 * c, k);
      st8<DT>(A.v_cache, row * A.scb + slot * A.scs + 8 * c, v);
    }
  } else if (A.k_cache) {
    int8_t* caches[2] = {A.k_cache, A.v_cache};
    uint16_t* scales[2] = {A.k_scale, A.v_scale};
#pragma unroll
    for (int u = 0; u < 2; u++) {
      float am = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) am = fmaxf(am, fabsf(u ? v[j] : k[j]));
      am = fmaxf(am, lane_xor4(am));
      am = fmaxf(am, lane_xor2(am));
      am = fmaxf(am, lane_xor1(am));
      const uint16_t sb = float_to_half_bits(__fdiv_rn(am, 127.0f));
      const float sf = fmaxf(half_bits_to_float(sb), 1e-30f);
      // 8 quotients by one divisor, rounded as a division rounds: the reciprocal rounded to nearest, the product and its remainder (Markstein).  An
      // infinite divisor leaves the product as it is.
      const float r0f = __builtin_amdgcn_rcpf(sf);
      const bool fin = sf < __builtin_inff();
      const float d = fin ? sf : 0.f, rc = fin ? fmaf(fmaf(-sf, r0f, 1.0f), r0f, r0f) : 0.f;
      uint32_t b[2] = {0u, 0u};
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float x = u ? v[j] : k[j], q0 = x * rc;
        const float qv = fminf(fmaxf(__builtin_rintf(fmaf(fmaf(-q0, d, x), rc, q0)), -127.0f), 127.0f);
        b[j / 4] |= (uint32_t)(uint8_t)(int8_t)(int)qv << (8 * (j % 4));
      }
      if (wr) {
        *(uint2*)(caches[u] + row * A.scb + slot * A.scs + 8 * c) = uint2{b[0], b[1]};
        if (c == 0) scales[u][row * A.ssb + slot] = sb;
      }
    }
  }
  // ---- queries
  if (live && A.gate_out) A.gate_out[r * 8 + c] = rnd(2.0f * rnd(1.0f / (1.0f + __expf(-glog))));
  if constexpr (!Q) {
    if (A.rope && __any(!in_tab)) {
      for (int h = 0; h < 8; h++) {
        float x[8];
        unpack8<DT>(*(const uint4*)((const uint16_t*)A.q_out + (r * 8 + h) * 64 + 8 * c), x);
        rotate(x);
        if (live && !in_tab) st8<DT>(A.q_out, (r * 8 + h) * 64 + 8 * c, x);
      }
    }
    return;
  }
#pragma unroll
  for (int h = 0; h < 8; h++) {
    float x[8], ss = 0.f;
    unpack8<DT>(qw[Q ? h : 0], x);
#pragma unroll
    for (int j = 0; j < 8; j++) ss += x[j] * x[j];
    ss += lane_xor1(ss); ss += lane_xor2(ss); ss += lane_xor4(ss);
    const float rs = rsqrtf(ss * (1.0f / 64.0f) + A.eps);
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = x[j] * rs;
    round8(x);
    if (A.rope) rotate(x);
    if (live) st8<DT>(A.q_out, (r * 8 + h) * 64 + 8 * c, x);
  }
}

// ------------------------------------------------------------------------------------------------ attn_post (hd = 64)
struct PostArgs {
  const void* z; const void* v; const void* xn; const float* gate_w; const float* xsa;
  void* out; int64_t n; int H, KH, d, gate_ch, z_dt; float xsa_eps;
};

template <int DT>
__global__ __launch_bounds__(256) void attn_post_kernel(PostArgs A) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= A.n) return;
  const int G = A.H / A.KH;
  for (int h = 0; h < A.H; h++) {
    const int kh = h / G;
    const int64_t zi = (r * A.H + h) * 64 + lane;
    float z = A.z_dt == UVMI_BF16 ? elem<UVMI_BF16>::ld(A.z, zi) : (A.z_dt == UVMI_F32 ? elem<UVMI_F32>::ld(A.z, zi) : elem<UVMI_F16>::ld(A.z, zi));
    if (A.xsa) {  // z -= tanh(alpha_h) (z . v_hat) v_hat, v_hat = v / max(|v|, eps), in fp32
      const float v = elem<DT>::ld(A.v, (r * A.KH + kh) * 64 + lane);
      const float nv = sqrtf(wave_sum(v * v));
      const float vh = v / fmaxf(nv, A.xsa_eps);
      const float proj = wave_sum(z * vh);
      z = round_t<DT>(z - A.xsa[h] * proj * vh);
    }
    if (A.gate_w) {  // z *= 2 sigmoid(W_h . xn[:gate_ch])
      float dot = 0.f;
      for (int c = lane; c < A.gate_ch; c += 64) dot += elem<DT>::ld(A.xn, r * A.d + c) * A.gate_w[h * A.gate_ch + c];
      dot = round_t<DT>(wave_sum(dot));
      const float g = round_t<DT>(2.0f * round_t<DT>(1.0f / (1.0f + __expf(-dot))));
      z = z * g;
    }
    elem<DT>::st(A.out, (r * A.H + h) * 64 + lane, z);
  }
}

// ------------------------------------------------------------------------------------------------ swiglu
// f % 8 == 0 (host-checked): thread t handles 8 consecutive columns of one row
template <int DT>
__global__ __launch_bounds__(256) void swiglu_kernel(const void* __restrict__ gu, void* __restrict__ out, int64_t rows, int f) {
  const int f8 = f / 8;
  const int64_t total = rows * f8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / f8;
    const int j = (int)(i % f8) * 8;
    float g[8], u[8], o[8];
    ld8<DT>(gu, r * 2 * f + j, g);
    ld8<DT>(gu, r * 2 * f + f + j, u);
#pragma unroll
    for (int k = 0; k < 8; k++) o[k] = round_t<DT>(g[k] / (1.0f + __expf(-g[k]))) * u[k];
    st8<DT>(out, r * (int64_t)f + j, o);
  }
}

// SwiGLU on the gate/up product of the UN-normalised hidden h: the block's pre-norm is the row scale rn = rsqrt(mean(h^2) + eps)
// of that product, so the norm never needs a launch (or a buffer) of its own.  One workgroup per row; every wave sums
// the row's squares itself (d / 64 elements per lane), which needs no LDS and no barrier.  f % 8 == 0, d % 2 == 0.
template <int DT>
__global__ __launch_bounds__(256) void swiglu_norm_kernel(const void* __restrict__ gu, const void* __restrict__ h, void* __restrict__ out, int f,
                                                          int d, float eps) {
  const int64_t r = blockIdx.x;
  const int lane = threadIdx.x & 63;
  // the thread's first 8 gate / up columns are requested before the row's squares, so that both round trips to memory
  // overlap (f <= 2048: the only ones)
  int j = threadIdx.x * 8;
  float g[8], u[8], o[8];
  if (j < f) {
    ld8<DT>(gu, r * 2 * f + j, g);
    ld8<DT>(gu, r * 2 * f + f + j, u);
  }
  float ss = 0.f;
  for (int i = 2 * lane; i < d; i += 128) {
    float a, b;
    ld2<DT>(h, r * d + i, a, b);
    ss = fmaf(a, a, ss);
    ss = fmaf(b, b, ss);
  }
  const float rn = rsqrtf(wave_sum(ss) / (float)d + eps);
  while (j < f) {
    if (DT == UVMI_BF16) {
      // pairs share a conversion, and silu divides through the hardware reciprocal (1 ulp in fp32, before the rounding
      // to bf16): a third fewer instructions in a launch that is bound by them
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        const uint32_t gw = float2_to_bf16x2(g[k] * rn, g[k + 1] * rn), uw = float2_to_bf16x2(u[k] * rn, u[k + 1] * rn);
        const float g0 = __uint_as_float(gw << 16), g1 = __uint_as_float(gw & 0xffff0000u);
        const float s0 = g0 * __builtin_amdgcn_rcpf(1.0f + __expf(-g0)), s1 = g1 * __builtin_amdgcn_rcpf(1.0f + __expf(-g1));
        const uint32_t sw = float2_to_bf16x2(s0, s1);
        o[k] = __uint_as_float(sw << 16) * __uint_as_float(uw << 16);
        o[k + 1] = __uint_as_float(sw & 0xffff0000u) * __uint_as_float(uw & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const float gv = round_t<DT>(g[k] * rn), uv = round_t<DT>(u[k] * rn);
        o[k] = round_t<DT>(gv / (1.0f + __expf(-gv))) * uv;
      }
    }
    st8<DT>(out, r * (int64_t)f + j, o);
    j += 256 * 8;
    if (j < f) {
      ld8<DT>(gu, r * 2 * f + j, g);
      ld8<DT>(gu, r * 2 * f + f + j, u);
    }
  }
}

}  // namespace uvmi

using namespace uvmi;

template <typename F>
static void dispatch_dt(int dt, F&& f) {
  if (dt == UVMI_F16) f(std::integral_constant<int, UVMI_F16>{});
  else if (dt == UVMI_BF16) f(std::integral_constant<int, UVMI_BF16>{});
  else f(std::integral_constant<int, UVMI_F32>{});
}

// the smallest of the forms (ascending) that has `need` pairs a lane, the last one if none has
template <int NP, int... MORE, typename F>
static void norm_form(int need, F&& go) {
  if constexpr (sizeof...(MORE) > 0) {
    if (need > NP) return norm_form<MORE...>(need, go);
  }
  go(std::integral_constant<int, NP>{});
}

namespace uvmi {
int norm_run(const uvmi_norm_args* a, void* stream) {
  const bool embed = a->tok != nullptr;
  UVMI_REQUIRE(a->x && (embed || a->y) && a->n_out, UVMI_EINVAL, "uvmi_%s_norm: null pointer", embed ? "embed" : "add");
  UVMI_REQUIRE(is_float_dtype(a->dtype) && a->rows >= 0 && a->d > 0 && a->d % 2 == 0 && a->d <= 2048 && (!embed || a->vocab > 0), UVMI_EINVAL,
               "uvmi_%s_norm: bad arguments", embed ? "embed" : "add");
  if (a->rows == 0) return UVMI_OK;
  const dim3 grid((unsigned)((a->rows + 3) / 4)), blk(256);
  dispatch_dt(a->dtype, [&](auto DT) {
    constexpr int D = decltype(DT)::value;
    auto go = [&](auto NP) {
      constexpr int n = decltype(NP)::value;
      if (embed) hipLaunchKernelGGL((norm_kernel<D, 0, n>), grid, blk, 0, (hipStream_t)stream, a->x, nullptr, a->tok, a->vocab, 0.f, 0.f, a->h_out, a->n_out, a->rows, a->d, a->eps, a->advance);
      else hipLaunchKernelGGL((norm_kernel<D, 1, n>), grid, blk, 0, (hipStream_t)stream, a->x, a->y, nullptr, 0, a->a, a->b, a->h_out, a->n_out, a->rows, a->d, a->eps, a->advance);
    };
    norm_form<1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16>((a->d + 127) / 128, go);
  });
  UVMI_CHECK_LAUNCH(embed ? "uvmi_embed_norm" : "uvmi_add_norm");
  return UVMI_OK;
}
}  // namespace uvmi

extern "C" int uvmi_embed_norm(const void* table, int dtype, int64_t vocab, const int64_t* tok, int64_t rows, int d, float eps,
                               void* x_out, void* n_out, void* stream) {
  UVMI_REQUIRE(tok, UVMI_EINVAL, "uvmi_embed_norm: null pointer");
  const uvmi_norm_args a{table, nullptr, tok, vocab, dtype, 0.f, 0.f, rows, d, eps, x_out, n_out, nullptr};
  return norm_run(&a, stream);
}

extern "C" int uvmi_add_norm(const void* x, const void* y, int dtype, float a, float b, int64_t rows, int d, float eps, void* h_out,
                             void* n_out, void* stream) {
  const uvmi_norm_args n{x, y, nullptr, 0, dtype, a, b, rows, d, eps, h_out, n_out, nullptr};
  return norm_run(&n, stream);
}

namespace uvmi {
int qkv_post_prepare(const uvmi_qkv_post_args* a, QkvArgs* out) {
  UVMI_REQUIRE(a, UVMI_EINVAL, "uvmi_qkv_post: null args");
  UVMI_REQUIRE(a->qkv && a->pos && a->q_out, UVMI_EINVAL, "uvmi_qkv_post: null pointer");
  UVMI_REQUIRE(a->hd == 64, UVMI_EUNSUPPORTED, "uvmi_qkv_post: head_dim %d (only 64)", a->hd);
  UVMI_REQUIRE(is_float_dtype(a->dtype) && is_float_dtype(a->q_dtype), UVMI_EINVAL, "uvmi_qkv_post: bad dtype");
  UVMI_REQUIRE(a->n >= 0 && a->H > 0 && a->KH > 0 && a->H % a->KH == 0, UVMI_EINVAL, "uvmi_qkv_post: bad sizes");
  UVMI_REQUIRE(!a->rope || (a->inv_freq && a->n_pairs >= 8 && a->n_pairs <= 32 && (a->n_pairs & (a->n_pairs - 1)) == 0), UVMI_EUNSUPPORTED,
               "uvmi_qkv_post: rope needs inv_freq and 8, 16 or 32 rotated pairs");
  UVMI_REQUIRE(!a->gate_out || a->ext_logits || (a->gate_w && a->xn && a->gate_ch > 0 && a->gate_ch % 8 == 0 && a->gate_ch <= a->d), UVMI_EINVAL,
               "uvmi_qkv_post: gate_out needs gate_w, xn and a gate_ch that is a multiple of 8 (or ext_logits)");
  const int64_t qkv_w = (int64_t)(a->H + 2 * a->KH) * a->hd;
  UVMI_REQUIRE(a->qkv_ld == 0 || a->qkv_ld >= qkv_w, UVMI_EINVAL, "uvmi_qkv_post: qkv_ld below the row width");
  UVMI_REQUIRE(a->qkv_ld % 8 == 0, UVMI_EUNSUPPORTED, "uvmi_qkv_post: qkv_ld must be a multiple of 8 (16-byte rows)");
  UVMI_REQUIRE(!a->ext_logits || a->qkv_ld >= qkv_w + a->H + a->KH, UVMI_EINVAL,
               "uvmi_qkv_post: ext_logits needs a row pitch that holds the H + KH logits behind q, k, v");
  UVMI_REQUIRE(((uintptr_t)a->qkv % 16) == 0 && ((uintptr_t)a->q_out % 16) == 0, UVMI_EUNSUPPORTED, "uvmi_qkv_post: qkv and q_out must be 16-byte aligned");
  UVMI_REQUIRE(!a->has_ve || (a->ve_table && a->tok && a->vocab > 0 && (a->ext_logits || (a->xn && a->ve_gate && a->ve_ch > 0 && a->ve_ch <= 64))), UVMI_EINVAL,
               "uvmi_qkv_post: value-embedding inputs missing");
  UVMI_REQUIRE(!a->k_cache || (a->v_cache && !a->k_scale == !a->v_scale && (a->k_scale || a->dtype != UVMI_F32) && a->S > 0), UVMI_EINVAL,
               "uvmi_qkv_post: incomplete cache arguments");
  QkvArgs& A = *out;
  A.qkv = a->qkv; A.xn = a->xn; A.ve_table = a->ve_table; A.ve_gate = a->ve_gate; A.tok = a->tok; A.pos = a->pos; A.rows = a->rows;
  A.last_pos = a->last_pos; A.inv_freq = a->inv_freq; A.q_out = a->q_out; A.k_out = a->k_out; A.v_out = a->v_out;
  A.k_cache = a->k_cache; A.v_cache = a->v_cache; A.k_scale = a->k_scale; A.v_scale = a->v_scale;
  A.scb = a->scb; A.sch = a->sch; A.scs = a->scs; A.ssb = a->ssb; A.ssh = a->ssh; A.n = a->n; A.vocab = a->vocab;
  A.H = a->H; A.KH = a->KH; A.d = a->d; A.ve_ch = a->ve_ch; A.n_pairs = a->n_pairs; A.S = a->S; A.ring = a->ring; A.has_ve = a->has_ve;
  A.rope = a->rope; A.q_dt = a->q_dtype; A.eps = a->eps;
  A.gate_w = a->gate_w; A.gate_out = a->gate_out; A.vhat_out = a->vhat_out; A.gate_ch = a->gate_ch; A.xsa_eps = a->xsa_eps;
  A.rope_tab = a->rope && a->rope_positions > 0 ? a->rope_table : nullptr;
  A.rope_n = a->rope_positions;
  A.ld = a->qkv_ld ? a->qkv_ld : qkv_w;
  A.ext = a->ext_logits != 0;
  return UVMI_OK;
}
bool qkv_post_engine_shape(const uvmi_qkv_post_args* a, const QkvArgs& A) {
  return (a->dtype == UVMI_F16 || a->dtype == UVMI_BF16) && a->q_dtype == a->dtype && a->H == 8 && a->KH == 1 && A.ext &&
         (!a->rope || (a->n_pairs == 16 && A.rope_tab && ((uintptr_t)A.rope_tab % 16) == 0));
}
bool qkv_post_rows_ok(const uvmi_qkv_post_args* a) {
  const uintptr_t wide = (uintptr_t)a->k_out | (uintptr_t)a->v_out | (uintptr_t)a->vhat_out | (a->has_ve ? (uintptr_t)a->ve_table : 0) |
                         (a->k_cache ? (uintptr_t)a->k_cache | (uintptr_t)a->v_cache : 0) * (a->k_scale ? 2 : 1);
  return wide % 16 == 0 && (!a->k_cache || (a->scb % 8 == 0 && a->scs % 8 == 0));
}
void qkv_post_kv_launch(int dtype, const QkvArgs& A, hipStream_t st) {
  const dim3 grid((unsigned)((A.n + 7) / 8)), blk(64);
  if (dtype == UVMI_F16) hipLaunchKernelGGL((qkv_post_rows_kernel<UVMI_F16, false>), grid, blk, 0, st, A);
  else hipLaunchKernelGGL((qkv_post_rows_kernel<UVMI_BF16, false>), grid, blk, 0, st, A);
}
}  // namespace uvmi

extern "C" int uvmi_qkv_post(const uvmi_qkv_post_args* a, void* stream) {
  QkvArgs A;
  const int rc = qkv_post_prepare(a, &A);
  if (rc) return rc;
  if (a->n == 0) return UVMI_OK;
  const dim3 grid((unsigned)((a->n + 3) / 4)), blk(256);
  const bool fast = qkv_post_engine_shape(a, A);
  // passes of many rows: 8 per wave, with wide accesses to everything that a row reads or writes.  A wave of 8 rows has the longer chain (2048
  // rows 7.1 us against 4.7, 4096 7.8 against 6.8, 6144 8.9 against 9.1, 8192 9.9 against 11.2)
  if (fast && a->n >= 6144 && qkv_post_rows_ok(a)) {
    const dim3 g8((unsigned)((a->n + 7) / 8)), blk(64);
    if (a->dtype == UVMI_F16) hipLaunchKernelGGL((qkv_post_rows_kernel<UVMI_F16, true>), g8, blk, 0, (hipStream_t)stream, A);
    else hipLaunchKernelGGL((qkv_post_rows_kernel<UVMI_BF16, true>), g8, blk, 0, (hipStream_t)stream, A);
  } else if (fast) {
    if (a->dtype == UVMI_F16) hipLaunchKernelGGL((qkv_post_fast_kernel<UVMI_F16>), grid, blk, 0, (hipStream_t)stream, A);
    else hipLaunchKernelGGL((qkv_post_fast_kernel<UVMI_BF16>), grid, blk, 0, (hipStream_t)stream, A);
  } else {
    dispatch_dt(a->dtype, [&](auto DT) { hipLaunchKernelGGL((qkv_post_kernel<decltype(DT)::value>), grid, blk, 0, (hipStream_t)stream, A); });
  }
  UVMI_CHECK_LAUNCH("uvmi_qkv_post");
  return UVMI_OK;
}

// cos / sin of position * inv_freq per frequency, rounded to the activation type as the rotation applies them
// (round_t(cosf(th)) above), as an fp32 table: row p holds cos[0..n_pairs) then sin[0..n_pairs)
template <int DT>
__global__ __launch_bounds__(256) void rope_table_kernel(const float* __restrict__ inv_freq, int n_pairs, int64_t n_pos, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_pos * n_pairs) return;
  const int64_t p = i / n_pairs;
  const int j = (int)(i % n_pairs);
  const float th = (float)p * inv_freq[j];
  out[p * 2 * n_pairs + j] = round_t<DT>(cosf(th));
  out[p * 2 * n_pairs + n_pairs + j] = round_t<DT>(sinf(th));
}

extern "C" int uvmi_rope_table(const float* inv_freq, int n_pairs, int64_t n_positions, int round_dtype, float* out, void* stream) {
  UVMI_REQUIRE(inv_freq && out, UVMI_EINVAL, "uvmi_rope_table: null pointer");
  UVMI_REQUIRE(n_pairs > 0 && n_positions >= 0 && is_float_dtype(round_dtype), UVMI_EINVAL, "uvmi_rope_table: bad arguments");
  if (n_positions == 0) return UVMI_OK;
  const dim3 grid((unsigned)((n_positions * n_pairs + 255) / 256)), blk(256);
  dispatch_dt(round_dtype, [&](auto DT) {
    hipLaunchKernelGGL((rope_table_kernel<decltype(DT)::value>), grid, blk, 0, (hipStream_t)stream, inv_freq, n_pairs, n_positions, out);
  });
  UVMI_CHECK_LAUNCH("uvmi_rope_table");
  return UVMI_OK;
}

extern "C" int uvmi_attn_post(const void* z, int z_dtype, const void* v, const void* xn, int dtype, const float* gate_w, const float* xsa,
                              float xsa_eps, int64_t n, int H, int KH, int hd, int d, int gate_ch, void* out, void* stream) {
  UVMI_REQUIRE(z && out, UVMI_EINVAL, "uvmi_attn_post: null pointer");
  UVMI_REQUIRE(hd == 64, UVMI_EUNSUPPORTED, "uvmi_attn_post: head_dim %d (only 64)", hd);
  UVMI_REQUIRE(is_float_dtype(dtype) && is_float_dtype(z_dtype), UVMI_EINVAL, "uvmi_attn_post: bad dtype");
  UVMI_REQUIRE(!xsa || v, UVMI_EINVAL, "uvmi_attn_post: XSA needs v");
  UVMI_REQUIRE(!gate_w || (xn && gate_ch > 0 && gate_ch <= d), UVMI_EINVAL, "uvmi_attn_post: gate needs xn and gate_ch");
  UVMI_REQUIRE(n >= 0 && H > 0 && KH > 0 && H % KH == 0, UVMI_EINVAL, "uvmi_attn_post: bad sizes");
  if (n == 0) return UVMI_OK;
  PostArgs A{z, v, xn, gate_w, xsa, out, n, H, KH, d, gate_ch, z_dtype, xsa_eps};
  const dim3 grid((unsigned)((n + 3) / 4)), blk(256);
  dispatch_dt(dtype, [&](auto DT) { hipLaunchKernelGGL((attn_post_kernel<decltype(DT)::value>), grid, blk, 0, (hipStream_t)stream, A); });
  UVMI_CHECK_LAUNCH("uvmi_attn_post");
  return UVMI_OK;
}

extern "C" int uvmi_swiglu(const void* gu, int dtype, int64_t rows, int f, void* out, void* stream) {
  UVMI_REQUIRE(gu && out, UVMI_EINVAL, "uvmi_swiglu: null pointer");
  UVMI_REQUIRE(is_float_dtype(dtype) && rows >= 0 && f > 0, UVMI_EINVAL, "uvmi_swiglu: bad arguments");
  UVMI_REQUIRE(f % 8 == 0 && ((uintptr_t)gu % 16) == 0 && ((uintptr_t)out % 16) == 0, UVMI_EUNSUPPORTED, "uvmi_swiglu: f %% 8 and 16-byte alignment needed");
  if (rows == 0) return UVMI_OK;
  int64_t blocks = (rows * (f / 8) + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  const dim3 grid((unsigned)blocks), blk(256);
  dispatch_dt(dtype, [&](auto DT) { hipLaunchKernelGGL((swiglu_kernel<decltype(DT)::value>), grid, blk, 0, (hipStream_t)stream, gu, out, rows, f); });
  UVMI_CHECK_LAUNCH("uvmi_swiglu");
  return UVMI_OK;
}

extern "C" int uvmi_swiglu_norm(const void* gu, const void* h, int dtype, int64_t rows, int f, int d, float eps, void* out, void* stream) {
  UVMI_REQUIRE(gu && h && out, UVMI_EINVAL, "uvmi_swiglu_norm: null pointer");
  UVMI_REQUIRE(is_float_dtype(dtype) && rows >= 0 && rows <= 0x7fffffff && f > 0 && d > 0 && eps >= 0.f, UVMI_EINVAL, "uvmi_swiglu_norm: bad arguments");
  UVMI_REQUIRE(f % 8 == 0 && d % 2 == 0 && ((uintptr_t)gu % 16) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)h % 8) == 0, UVMI_EUNSUPPORTED,
               "uvmi_swiglu_norm: f %% 8, d %% 2 and 16-byte alignment needed");
  if (rows == 0) return UVMI_OK;
  const dim3 grid((unsigned)rows), blk(256);
  dispatch_dt(dtype, [&](auto DT) { hipLaunchKernelGGL((swiglu_norm_kernel<decltype(DT)::value>), grid, blk, 0, (hipStream_t)stream, gu, h, out, f, d, eps); });
  UVMI_CHECK_LAUNCH("uvmi_swiglu_norm");
  return UVMI_OK;
}
