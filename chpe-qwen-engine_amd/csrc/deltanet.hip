// deltanet.hip -- one decode step of a gated-DeltaNet (linear-attention) layer of Qwen3.5.
//
// The reference engine has no code for these layers (its README only claims them); the
// arithmetic follows the published gated delta rule (Yang, Kautz, Hatamizadeh, ICLR 2025)
// in the form of the library that defines the Qwen3.5 layer (transformers 5.15.0,
// models/qwen3_5/modeling_qwen3_5.py: causal_conv1d_update :200-217, l2norm :242-245,
// torch_recurrent_gated_delta_rule :331-380, beta/g :497-499, head repetition :500-502,
// RMSNormGated :168-184).
//
// k_dn_conv: the depthwise causal conv over [state, x] + SiLU, one thread per channel, the
// state shifted in place (the decode step applies it in its in-projection's epilogue instead).
// k_dn_step_head: the gated delta rule and the gated RMSNorm of one value head per workgroup
// (the decode step's form); k_dn_step: a workgroup per (value head, 16-column block), its slab
// of the head's 128x128 f32 state read once and written once (the columns of the update are
// independent), with k_dn_gnorm for the gated RMSNorm of each head's output.  2 x 64 KiB of
// state per head and step.
//
// Several tokens in order (the block step and the panels of a prompt): k_dn_prep, k_dn_scan and
// k_dn_gnorm_block, each state read and written once.
#include <cstdio>

#include "device_common.hpp"
#include "kernels.hpp"

namespace chpe {
namespace {
using namespace dev;

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

__global__ void __launch_bounds__(256) k_dn_conv(DnConvArgs a) {
  const uint32_t c = blockIdx.x * 256 + threadIdx.x;
  if (c >= a.channels) return;
  const uint32_t T = a.taps;
  const float* w = a.w + size_t(c) * T;
  float* st = a.state + size_t(c) * (T - 1);
  float wv[kDnMaxTaps], sv[kDnMaxTaps];
#pragma unroll
  for (uint32_t k = 0; k < kDnMaxTaps; ++k) {
    wv[k] = k + 1 < T ? w[k] : 0.0f;
    sv[k] = k + 1 < T ? st[k] : 0.0f;
  }
  const float x = a.x[c], wl = w[T - 1];
  const bool keep = a.step && a.step->broken;  // (after the step's break: the state stays)
  float acc = 0.0f;  // oldest tap first, the new input last
#pragma unroll
  for (uint32_t k = 0; k < kDnMaxTaps; ++k)
    if (k + 1 < T) acc += wv[k] * sv[k];
  acc += wl * x;
  a.out[c] = silu_f(acc);
  if (keep) return;
#pragma unroll
  for (uint32_t k = 0; k + 1 < kDnMaxTaps; ++k)
    if (k + 2 < T) st[k] = sv[k + 1];
  st[T - 2] = x;
}

// grid (value head, column block of CW columns): the block's D x CW slab of the head's state
// (rows i, columns c0 + j) is read once and written once; every column of the update is
// independent (kv_mem[j], delta_j, S[:, j], o[j]), so the head's columns spread over D / CW
// workgroups.  Thread (row block rb, column j) holds rows rb * RPB .. of column c0 + j; the
// two column sums (S^T k before the update, S^T q after) meet over the row blocks of a wave
// (lanes 16 and 32 apart) and over the waves in LDS, in a fixed order.  q and k are
// l2-normalised by every workgroup of the head (D values each).  Writes o[j] = (S^T q)_j; the
// gated norm, a reduction over the whole head, is k_dn_gnorm.
template <int D, int CW>
__global__ void __launch_bounds__(256) k_dn_step(DnStepArgs a) {
  constexpr int NT = 256, RB = NT / CW, RPB = D / RB, NWV = NT / 64;
  static_assert(CW == 16 && NT % CW == 0 && D % RB == 0 && D % 64 == 0, "lanes 16 / 32 apart share a column");
  const uint32_t h = blockIdx.x, c0 = blockIdx.y * CW, kh = h / (a.n_v_heads / a.n_k_heads);
  const int t = threadIdx.x, j = t % CW, rb = t / CW, lane = t & 63, wave = t >> 6;
  __shared__ float s_qn[D], s_kn[D];
  __shared__ float s_part[NWV][CW];

  // 1. loads: the thread's state rows, then the head's inputs (all before any use)
  float* S = a.state + size_t(h) * D * D + c0 + j;
  float sr[RPB];
#pragma unroll
  for (int r = 0; r < RPB; ++r) sr[r] = S[size_t(rb * RPB + r) * D];
  constexpr int PL = D / 64;  // q/k values per lane (every wave normalises both vectors)
  float qv[PL], kv[PL];
#pragma unroll
  for (int m = 0; m < PL; ++m) {
    qv[m] = a.q[size_t(kh) * D + lane + 64 * m];
    kv[m] = a.k[size_t(kh) * D + lane + 64 * m];
  }
  const float vj = a.v[size_t(h) * D + c0 + j];
  const bool keep = a.step && a.step->broken;  // (after the step's break: the state stays)
  const float beta = 1.0f / (1.0f + expf(-a.b[h]));
  const float decay = expf(-expf(a.A_log[h]) * softplus_f(a.a[h] + a.dt_bias[h]));

  // 2. l2-normalised q (scaled by 1/sqrt(D)) and k, into LDS
  float q2 = 0.0f, k2 = 0.0f;
#pragma unroll
  for (int m = 0; m < PL; ++m) {
    q2 += qv[m] * qv[m];
    k2 += kv[m] * kv[m];
  }
  q2 = wave_sum(q2);
  k2 = wave_sum(k2);
  const float qi = 1.0f / sqrtf(q2 + 1e-6f), ki = 1.0f / sqrtf(k2 + 1e-6f), scale = 1.0f / sqrtf(float(D));
  if (wave == 0) {
#pragma unroll
    for (int m = 0; m < PL; ++m) {
      s_qn[lane + 64 * m] = qv[m] * qi * scale;
      s_kn[lane + 64 * m] = kv[m] * ki;
    }
  }
  __syncthreads();

  // the column sum of a per-thread partial: over the wave's 4 row blocks, then the waves
  auto column_sum = [&](float p) {
    p = pair_sum(p, 16);
    p = pair_sum(p, 32);
    if (lane < CW) s_part[wave][lane] = p;
    __syncthreads();
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) v += s_part[w][j];
    __syncthreads();  // s_part is reused by the next sum
    return v;
  };

  // 3. decayed state; kv_mem[j] = sum_i S[i][j] k[i]
  float p = 0.0f;
#pragma unroll
  for (int r = 0; r < RPB; ++r) {
    sr[r] *= decay;
    p += sr[r] * s_kn[rb * RPB + r];
  }
  const float kvm = column_sum(p);
  const float delta = (vj - kvm) * beta;

  // 4. S += k delta^T, written back; o[j] = sum_i S[i][j] q[i]
  float o = 0.0f;
#pragma unroll
  for (int r = 0; r < RPB; ++r) {
    sr[r] += s_kn[rb * RPB + r] * delta;
    if (!keep) S[size_t(rb * RPB + r) * D] = sr[r];
    o += sr[r] * s_qn[rb * RPB + r];
  }
  o = column_sum(o);
  if (t < CW) a.out[size_t(h) * D + c0 + j] = o;
}

// The gated delta rule and the gated RMSNorm of one value head in one workgroup of kDnRb * D
// threads (thread (row block rb, column j): rows rb * D / kDnRb .. of column j; the column sums
// meet in LDS over the row blocks in order), so that the norm, a reduction over the head's D
// outputs, needs no second launch.  The same arithmetic as k_dn_step + k_dn_gnorm up to the
// order of the float sums.
constexpr int kDnRb = 8;
template <int D>
__global__ void __launch_bounds__(kDnRb * D) k_dn_step_head(DnStepArgs a) {
  constexpr int NT = kDnRb * D, RPB = D / kDnRb, NWV = NT / 64;
  static_assert(D % 64 == 0 && D % kDnRb == 0, "");
  const uint32_t h = blockIdx.x, kh = h / (a.n_v_heads / a.n_k_heads);
  const int t = threadIdx.x, j = t % D, rb = t / D, lane = t & 63, wave = t >> 6;
  __shared__ float s_qn[D], s_kn[D];
  __shared__ float s_part[kDnRb][D];
  __shared__ float s_red[NWV];

  // 1. loads: the thread's state rows, then the head's inputs (all before any use)
  float* S = a.state + size_t(h) * D * D + j;
  float sr[RPB];
#pragma unroll
  for (int r = 0; r < RPB; ++r) sr[r] = S[size_t(rb * RPB + r) * D];
  constexpr int PL = D / 64;
  float qv[PL], kv[PL];
#pragma unroll
  for (int m = 0; m < PL; ++m) {
    qv[m] = a.q[size_t(kh) * D + lane + 64 * m];
    kv[m] = a.k[size_t(kh) * D + lane + 64 * m];
  }
  const float vj = a.v[size_t(h) * D + j], zj = a.z[size_t(h) * D + j], wj = a.norm_w[j];
  const bool keep = a.step && a.step->broken;  // (after the step's break: the state stays)
  const float beta = 1.0f / (1.0f + expf(-a.b[h]));
  const float decay = expf(-expf(a.A_log[h]) * softplus_f(a.a[h] + a.dt_bias[h]));

  // 2. l2-normalised q (scaled by 1/sqrt(D)) and k, into LDS
  float q2 = 0.0f, k2 = 0.0f;
#pragma unroll
  for (int m = 0; m < PL; ++m) {
    q2 += qv[m] * qv[m];
    k2 += kv[m] * kv[m];
  }
  q2 = wave_sum(q2);
  k2 = wave_sum(k2);
  const float qi = 1.0f / sqrtf(q2 + 1e-6f), ki = 1.0f / sqrtf(k2 + 1e-6f), scale = 1.0f / sqrtf(float(D));
  if (wave == 0) {
#pragma unroll
    for (int m = 0; m < PL; ++m) {
      s_qn[lane + 64 * m] = qv[m] * qi * scale;
      s_kn[lane + 64 * m] = kv[m] * ki;
    }
  }
  __syncthreads();

  // the column sum of a per-thread partial over the row blocks, in order (every thread gets it)
  auto column_sum = [&](float p) {
    s_part[rb][j] = p;
    __syncthreads();
    float v = 0.0f;
#pragma unroll
    for (int b = 0; b < kDnRb; ++b) v += s_part[b][j];
    __syncthreads();  // s_part is reused by the next sum
    return v;
  };

  // 3. decayed state; kv_mem[j] = sum_i S[i][j] k[i]
  float p = 0.0f;
#pragma unroll
  for (int r = 0; r < RPB; ++r) {
    sr[r] *= decay;
    p += sr[r] * s_kn[rb * RPB + r];
  }
  const float kvm = column_sum(p);
  const float delta = (vj - kvm) * beta;

  // 4. S += k delta^T, written back; o[j] = sum_i S[i][j] q[i]
  float o = 0.0f;
#pragma unroll
  for (int r = 0; r < RPB; ++r) {
    sr[r] += s_kn[rb * RPB + r] * delta;
    if (!keep) S[size_t(rb * RPB + r) * D] = sr[r];
    o += sr[r] * s_qn[rb * RPB + r];
  }
  o = column_sum(o);

  // 5. the gated RMSNorm over the head's D outputs (row block 0's threads): w * (o * rr) * silu(z)
  if (rb == 0) {
    const float s2 = wave_sum(o * o);
    if (lane == 0) s_red[wave] = s2;
  }
  __syncthreads();
  if (rb != 0) return;
  float tot = 0.0f;
#pragma unroll
  for (int w = 0; w < D / 64; ++w) tot += s_red[w];
  const float rr = 1.0f / sqrtf(tot / float(D) + a.eps);
  a.out[size_t(h) * D + j] = wj * (o * rr) * silu_f(zj);
}

// the gated RMSNorm of each value head's output (one workgroup of D threads per head):
// w * (o * rsqrt(mean o^2 + eps)) * silu(z)
template <int D>
__global__ void __launch_bounds__(D) k_dn_gnorm(DnStepArgs a) {
  const uint32_t h = blockIdx.x;
  const int j = threadIdx.x, lane = j & 63, wave = j >> 6;
  __shared__ float s_red[D / 64];
  const float o = a.out[size_t(h) * D + j], z = a.z[size_t(h) * D + j], w = a.norm_w[j];
  const float s2 = wave_sum(o * o);
  if (lane == 0) s_red[wave] = s2;
  __syncthreads();
  float tot = 0.0f;
#pragma unroll
  for (int k = 0; k < D / 64; ++k) tot += s_red[k];
  const float rr = 1.0f / sqrtf(tot / float(D) + a.eps);
  a.out[size_t(h) * D + j] = w * (o * rr) * silu_f(z);
}

// ---- m tokens in order: each state read and written once (the block step and the panels) --------
// The recurrence alone is serial over the tokens, so everything else comes before or after it,
// parallel over the tokens: k_dn_prep (conv + SiLU, l2 norms, decay, beta), k_dn_scan (the delta
// rule), k_dn_gnorm_block (the gated norm).

// The input of channel c as the causal conv sees it before token t: the last three inputs of
// tokens that did not break (a broken token's state update is skipped), oldest first, continuing
// into the state of before the call.
__device__ __forceinline__ void dn_taps(const DnBlockArgs& a, uint32_t c, uint32_t t, float (&tap)[kDnConvTaps - 1]) {
  constexpr int P = int(kDnConvTaps) - 1;
  bool plain = t >= uint32_t(P);
#pragma unroll
  for (int k = 0; k < P; ++k) plain = plain && a.brk[t >= uint32_t(P) ? t - 1 - uint32_t(k) : 0u] == 0u;
  if (plain) {  // (uniform)
#pragma unroll
    for (int k = 0; k < P; ++k) tap[P - 1 - k] = a.x[size_t(t - 1 - uint32_t(k)) * a.x_stride + c];
    return;
  }
  const float* st = a.conv_state + size_t(c) * P;
  int s = int(t) - 1, from = P - 1;
#pragma unroll
  for (int k = P - 1; k >= 0; --k) {
    while (s >= 0 && a.brk[s] != 0u) --s;
    if (s >= 0) tap[k] = a.x[size_t(s--) * a.x_stride + c];
    else tap[k] = st[from--];
  }
}

// grid (n_k_heads + n_v_heads / 2, tokens), 256 threads: block b < n_k_heads the query and key head
// b (128 threads each), the others two value heads; rows of conv_out: q (l2-normalised, times
// 1/sqrt(128)), k (l2-normalised), v, then decay and beta per value head
__global__ void __launch_bounds__(256) k_dn_prep(DnBlockArgs a) {
  constexpr uint32_t D = 128;
  const uint32_t b = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t nk = a.n_k_heads, hi = tid >> 7, i = tid & 127u;
  const bool qk = b < nk;
  const uint32_t c = qk ? (hi ? nk * D : 0u) + b * D + i : 2 * nk * D + (b - nk) * 256 + tid;
  float* row = a.conv_out + size_t(t) * a.conv_stride;
  float tap[kDnConvTaps - 1];
  const float x = a.x[size_t(t) * a.x_stride + c];
  const float* w = a.w + size_t(c) * kDnConvTaps;
  dn_taps(a, c, t, tap);
  float acc = 0.0f;  // oldest tap first, the new input last (k_dn_conv)
#pragma unroll
  for (uint32_t k = 0; k + 1 < kDnConvTaps; ++k) acc += w[k] * tap[k];
  acc += w[kDnConvTaps - 1] * x;
  float y = silu_f(acc);
  if (!qk) {  // (uniform)
    row[c] = y;
    if (i == 0) {
      const uint32_t h = (b - nk) * 2 + hi;
      const float at = a.a[size_t(t) * a.ab_stride + h], bt = a.b[size_t(t) * a.ab_stride + h];
      row[a.channels + h] = expf(-expf(a.A_log[h]) * softplus_f(at + a.dt_bias[h]));
      row[a.channels + a.n_v_heads + h] = 1.0f / (1.0f + expf(-bt));
    }
    return;
  }
  __shared__ float s_red[4];
  const float s2 = wave_sum(y * y);
  if (lane == 0) s_red[wave] = s2;
  __syncthreads();
  const float inv = 1.0f / sqrtf((s_red[2 * hi] + s_red[2 * hi + 1]) + 1e-6f);
  y *= inv;
  if (hi == 0) y *= 1.0f / sqrtf(float(D));
  row[c] = y;
}

// The delta rule over the m tokens: workgroup (value head, 16 columns of its 128 x 128 state), wave =
// 4 columns x 16 lanes of 8 rows each.  The columns do not meet, so a token costs a lane 32 products,
// two 16-lane sums and no barrier: 0.34 us a token over 250 tokens (four waves of a column block
// meeting at two barriers per sum: 1.4 us).  32 tokens' q, k and v are staged in LDS, the next 32 on the way meanwhile.
// Bound by the chain of a token's products and sums.
__global__ void __launch_bounds__(256) k_dn_scan(DnBlockArgs a) {
  constexpr uint32_t D = 128, CT = 32, CW = 16;
  __shared__ __align__(16) float s_q[2][CT][D], s_k[2][CT][D];
  __shared__ __align__(16) float s_v[2][CT][CW];
  __shared__ float s_ab[2][CT][2], s_o[CT][CW];
  __shared__ uint32_t s_brk[2][CT];
  const uint32_t h = blockIdx.x, c0 = blockIdx.y * CW, kh = h / (a.n_v_heads / a.n_k_heads), nk = a.n_k_heads * D;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rb = lane & 15, col = wave * 4 + (lane >> 4);
  {  // the conv state after the tokens (the prep launch has read the one before)
    const uint32_t c = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + tid;
    if (c < a.channels) {
      float tap[kDnConvTaps - 1];
      dn_taps(a, c, a.m, tap);
#pragma unroll
      for (uint32_t k = 0; k + 1 < kDnConvTaps; ++k) a.conv_state[size_t(c) * (kDnConvTaps - 1) + k] = tap[k];
    }
  }
  float* S = a.state + size_t(h) * D * D + c0 + col;
  float sr[8];  // rows 4 rb .. + 3 and 64 + 4 rb .. + 3
#pragma unroll
  for (uint32_t r = 0; r < 8; ++r) sr[r] = S[size_t((r < 4 ? 0u : 60u) + rb * 4 + r) * D];
  float4 kq[8], vv;
  float ab = 0.0f;
  uint32_t bk = 0;
  auto load = [&](uint32_t t0) {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t e = (tid + 256 * i) & 1023u, t = t0 + (e >> 5), tt = t < a.m ? t : a.m - 1;
      kq[i] = ld_f4(a.conv_out + size_t(tt) * a.conv_stride + (i < 4 ? nk : 0u) + kh * D + 4 * (e & 31u));
    }
    const uint32_t t = t0 + ((tid & 127u) >> 2), tt = t < a.m ? t : a.m - 1;
    vv = ld_f4(a.conv_out + size_t(tt) * a.conv_stride + 2 * nk + h * D + c0 + 4 * (tid & 3u));
    const uint32_t u = t0 + ((tid & 63u) >> 1), uu = u < a.m ? u : a.m - 1;
    ab = a.conv_out[size_t(uu) * a.conv_stride + a.channels + (tid & 1u) * a.n_v_heads + h];
    bk = a.brk[uu];
  };
  auto stage = [&](uint32_t b) {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t e = (tid + 256 * i) & 1023u;
      *reinterpret_cast<float4*>(i < 4 ? &s_k[b][e >> 5][4 * (e & 31u)] : &s_q[b][e >> 5][4 * (e & 31u)]) = kq[i];
    }
    if (tid < 128) *reinterpret_cast<float4*>(&s_v[b][tid >> 2][4 * (tid & 3u)]) = vv;
    if (tid < 64) {
      s_ab[b][tid >> 1][tid & 1u] = ab;
      if ((tid & 1u) == 0) s_brk[b][tid >> 1] = bk;
    }
  };
  load(0);
  stage(0);
  __syncthreads();
  for (uint32_t t0 = 0, b = 0; t0 < a.m; t0 += CT, b ^= 1u) {
    const uint32_t n = a.m - t0 < CT ? a.m - t0 : CT;
    load(t0 + CT);  // (past the last token: that token again, not used)
    // a token's operands come out of LDS one token ahead of its chain, and a lane keeps the sum
    // of the token its index names until 16 are there: no branch and no LDS wait in the chain
    struct Tok {
      float4 ka, kb, qa, qb;
      float decay, beta, v;
    };
    auto read = [&](uint32_t tt) {
      Tok x;
      x.ka = *reinterpret_cast<const float4*>(&s_k[b][tt][4 * rb]);
      x.kb = *reinterpret_cast<const float4*>(&s_k[b][tt][64 + 4 * rb]);
      x.qa = *reinterpret_cast<const float4*>(&s_q[b][tt][4 * rb]);
      x.qb = *reinterpret_cast<const float4*>(&s_q[b][tt][64 + 4 * rb]);
      x.decay = s_ab[b][tt][0];
      x.beta = s_ab[b][tt][1];
      x.v = s_v[b][tt][col];
      return x;
    };
    auto token = [&](const Tok& x) {
      const float kv[8] = {x.ka.x, x.ka.y, x.ka.z, x.ka.w, x.kb.x, x.kb.y, x.kb.z, x.kb.w};
      const float qv[8] = {x.qa.x, x.qa.y, x.qa.z, x.qa.w, x.qb.x, x.qb.y, x.qb.z, x.qb.w};
      float p0 = 0.0f, p1 = 0.0f;
#pragma unroll
      for (int r = 0; r < 8; ++r) sr[r] *= x.decay;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        p0 = fmaf(sr[r], kv[r], p0);
        p1 = fmaf(sr[r + 4], kv[r + 4], p1);
      }
      float p = p0 + p1;
      p = pair_sum(p, 1);
      p = pair_sum(p, 2);
      p = pair_sum(p, 4);
      p = pair_sum(p, 8);
      const float delta = (x.v - p) * x.beta;
      float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
      for (int r = 0; r < 8; ++r) sr[r] = fmaf(kv[r], delta, sr[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        o0 = fmaf(sr[r], qv[r], o0);
        o1 = fmaf(sr[r + 4], qv[r + 4], o1);
      }
      float o = o0 + o1;
      o = pair_sum(o, 1);
      o = pair_sum(o, 2);
      o = pair_sum(o, 4);
      return pair_sum(o, 8);
    };
    if (n == CT && __syncthreads_or(tid < 64 && s_brk[b][tid >> 1] != 0u) == 0) {  // (no break in the chunk)
      Tok x = read(0);
#pragma unroll
      for (uint32_t t16 = 0; t16 < CT; t16 += 16) {
        float keep = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < 16; ++k) {
          const Tok nx = read(t16 + k + 1 < CT ? t16 + k + 1 : CT - 1);
          const float o = token(x);
          keep = rb == k ? o : keep;
          x = nx;
        }
        s_o[t16 + rb][col] = keep;
      }
    } else {
      for (uint32_t tt = 0; tt < n; ++tt) {
        float o = 0.0f;
        if (s_brk[b][tt] == 0u) o = token(read(tt));  // (uniform; a broken token: the state stays, the output is not used)
        if (rb == 0) s_o[tt][col] = o;
      }
    }
    stage(b ^ 1u);
    __syncthreads();
    for (uint32_t e = tid; e < n * CW; e += 256)
      a.out[size_t(t0 + e / CW) * a.out_stride + h * D + c0 + e % CW] = s_o[e / CW][e % CW];
    __syncthreads();
  }
#pragma unroll
  for (uint32_t r = 0; r < 8; ++r) S[size_t((r < 4 ? 0u : 60u) + rb * 4 + r) * D] = sr[r];
}

// the gated norm (k_dn_gnorm): grid (value heads / 8, tokens), wave = 2 heads, lane = 2 outputs of each
__global__ void __launch_bounds__(256) k_dn_gnorm_block(DnBlockArgs a) {
  constexpr uint32_t D = 128;
  const uint32_t tk = blockIdx.y, lane = threadIdx.x & 63, h0 = blockIdx.x * 8 + (threadIdx.x >> 6) * 2;
  float* out = a.out + size_t(tk) * a.out_stride + h0 * D + 2 * lane;
  const float* z = a.z + size_t(tk) * a.z_stride + h0 * D + 2 * lane;
  const float2 w = *reinterpret_cast<const float2*>(a.norm_w + 2 * lane);
  float2 o[2], g[2];
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) {
    o[k] = *reinterpret_cast<const float2*>(out + k * D);
    g[k] = *reinterpret_cast<const float2*>(z + k * D);
  }
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) {
    const float tot = wave_sum(o[k].x * o[k].x + o[k].y * o[k].y);
    const float rr = 1.0f / sqrtf(tot / float(D) + a.eps);
    *reinterpret_cast<float2*>(out + k * D) = make_float2(w.x * (o[k].x * rr) * silu_f(g[k].x), w.y * (o[k].y * rr) * silu_f(g[k].y));
  }
}

}  // namespace

bool launch_dn_block(const DnBlockArgs& a, hipStream_t st) {
  // (the engine plans the 9B layers: 4 taps, 128-wide heads, an even number of value heads in eights)
  if (a.taps != kDnConvTaps || a.head_dim != 128 || a.n_v_heads % 8 || a.n_v_heads % a.n_k_heads ||
      a.channels != (2 * a.n_k_heads + a.n_v_heads) * 128 || a.channels > a.n_v_heads * 8 * 256) {
    std::fprintf(stderr, "chpe: the multi-token DeltaNet kernels are built for the 9B layers\n");
    return false;
  }
  launch_kernel(&k_dn_prep, dim3(a.n_k_heads + a.n_v_heads / 2, a.m), dim3(256), st, a);
  launch_kernel(&k_dn_scan, dim3(a.n_v_heads, 8), dim3(256), st, a);
  launch_kernel(&k_dn_gnorm_block, dim3(a.n_v_heads / 8, a.m), dim3(256), st, a);
  return true;
}

bool deltanet_supported(uint32_t n_v_heads, uint32_t n_k_heads, uint32_t head_dim, uint32_t taps) {
  return n_k_heads > 0 && n_v_heads % n_k_heads == 0 && (head_dim == 64 || head_dim == 128) && taps >= 2 &&
         taps <= kDnMaxTaps;
}

void launch_dn_conv(const DnConvArgs& a, hipStream_t st) {
  launch_kernel(&k_dn_conv, dim3((a.channels + 255) / 256), dim3(256), st, a);
}

void launch_dn_step(const DnStepArgs& a, uint32_t head_dim, hipStream_t st) {
  constexpr uint32_t CW = 16;
  if (a.norm_w && head_dim == 128) {  // the gated form: a workgroup per head, the norm included
    launch_kernel(&k_dn_step_head<128>, dim3(a.n_v_heads), dim3(kDnRb * 128), st, a);
    return;
  }
  if (head_dim == 128) {
    launch_kernel(&k_dn_step<128, CW>, dim3(a.n_v_heads, 128 / CW), dim3(256), st, a);
    if (a.norm_w) launch_kernel(&k_dn_gnorm<128>, dim3(a.n_v_heads), dim3(128), st, a);
  } else {
    launch_kernel(&k_dn_step<64, CW>, dim3(a.n_v_heads, 64 / CW), dim3(256), st, a);
    if (a.norm_w) launch_kernel(&k_dn_gnorm<64>, dim3(a.n_v_heads), dim3(64), st, a);
  }
}

}  // namespace chpe
