// panel.hip -- a prompt's positions in panels of up to kMaxPanel tokens: every weight is read once
// per panel and the products run on the matrix cores, in 8-bit integers (4- and 2-bit codes) or fp16.
//
// Per projection:
// 1. k_panel_split: the input rows (RMS-normalised, (x * inv) * gamma, rmsNorm :187-191, when gamma
//    is set) as matrix-core operands, each 128-column group of a token with a scale of its own, as in
//    the block step (one scale per token let a channel 2^12 times the others take 12 of their bits).
//    For 4- and 2-bit codes: X = x * 2^(30 - e), max |x| of the group < 2^e, rounded to nearest, in
//    four balanced signed-byte limbs: within 2^-30 of the group's largest value (X is exact where
//    |x| is 2^-6 of it or more), below what f32 sums over 2048 columns and more resolve.  For fp16 weights: x * 2^(14 - e)
//    as the sum of three fp16 numbers of 11 bits each, f32's 24 bits and more down to 2^-14 of the
//    group's largest value, within 2^-38 of that below.  (Two fp16 numbers carry 23
//    bits: half the time the last bit of an f32 is lost, and the logits of the 3B model were 1.25
//    to 2 times as far from their 64-bit values.)
// 2. k_panel_gemm / k_panel_gemm_h: workgroup = 256 (128) weight rows x one token tile x a range of
//    128-column groups.
// 3. k_panel_epi: the ranges' sums, the outlier corrections and the decode step's epilogue.
// Attention (k_panel_attn_*): a wave owns 16 (token, head) rows of a kv head and walks the
// positions with a running softmax; no partial results go through memory.
#include "device_common.hpp"
#include "kernels.hpp"

namespace chpe {
namespace {
using namespace dev;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ half8_t as_half8(uint4 v) { return __builtin_bit_cast(half8_t, v); }
__device__ __forceinline__ uint32_t pack2(float a, float b) {  // (each rounded to nearest)
  const half2_t h = {_Float16(a), _Float16(b)};
  return __builtin_bit_cast(uint32_t, h);
}
__device__ __forceinline__ float f16_round(float x) { return float(_Float16(x)); }
// 2^(b - e) for a largest magnitude below 2^e (given as its bits), kept a normal number; a
// non-finite magnitude: NaN (every product of the group is then NaN)
__device__ __forceinline__ float scale_up(uint32_t max_bits, int b) {
  if (max_bits >= 0x7f800000u) return __uint_as_float(0x7fc00000u);
  int e = int(max_bits >> 23) - 126;  // (subnormal maxima: as 2^-126)
  e = e < -90 ? -90 : e;
  return ldexpf(1.0f, b - e);
}

__global__ void k_panel_begin(StepState* state, uint32_t token, uint32_t pos) { *state = StepState{token, pos, 0, 0}; }

// grid (128-column groups, 64-token tiles): 64 tokens x 128 columns.  Thread (token, 8 columns)
// four times.  The images are what the GEMM copies to LDS linearly, 16-byte pieces placed so that
// the 16 tokens of one LDS read fall on distinct banks:
//   limbs: [limb][token][8 pieces of 16 columns], piece c of token t at slot c ^ ((t >> 1) & 7), its
//     columns in the unpacked codes' order (4-bit {0,2,4,6}, {1,3,5,7}, {8,..}, {9,..}; 2-bit
//     {0,4,8,12}, {1,..}, {2,..}, {3,..}); thread pairs hold the two halves of a piece;
//   fp16: [part][token][16 pieces of 8 columns], piece c of token t at slot c ^ (t & 15);
//   then kScales floats, the factors from the tokens' products in this group to their values.
// The f32 values go out token-minor for the outlier corrections, through LDS.  Bound by memory: 4
// bytes in, 4 + 4 out per element.
template <bool kNorm, int BITS>
__global__ void __launch_bounds__(256) k_panel_split(PanelSplitArgs a) {
  __shared__ float s_x[128][65];
  __shared__ double s_red[4][64];
  __shared__ float s_inv[64];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t g = blockIdx.x, tok0 = blockIdx.y * 64, C = a.C, ng = C >> 7;
  float4 xa[4], xb[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t idx = tid + 256 * i, t = tok0 + (idx >> 4), c = g * 128 + (idx & 15) * 8;
    const float* row = a.x + size_t(t < a.m ? t : 0u) * C + c;
    xa[i] = ld_f4(row);
    xb[i] = ld_f4(row + 4);
  }
  [[maybe_unused]] const uint32_t tl = tok0 + lane < a.m ? tok0 + lane : a.m - 1;
  constexpr int kUp = BITS == 16 ? 14 : 30;
  if constexpr (kNorm) {  // the producers' partial sums of squares, each wave a quarter of them
    // (in 64 bits: the norm's factor scales the whole row, its error is not averaged out by the sums)
    double ss = 0.0;
#pragma unroll 8
    for (uint32_t i = wave; i < a.n_ssp; i += 4) ss += double(a.ssp[size_t(i) * kMaxPanel + tl]);
    s_red[wave][lane] = ss;
    __syncthreads();
    if (wave == 0) {
      const float tot = float((s_red[0][lane] + s_red[1][lane]) + (s_red[2][lane] + s_red[3][lane]));
      s_inv[lane] = 1.0f / sqrtf(tot / float(C) + a.eps);
      // forwardDecode's break test (StepState::broken) on the token's input
      if (g == 0 && tok0 + lane < a.m &&
          ((a.chk == 1u && !isfinite(tot)) || (a.chk == 2u && !isfinite(a.x[size_t(tl) * C]))))
        a.brk[tl] = 1u;
    }
    __syncthreads();
  }
  const uint32_t T = a.tile;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const uint32_t idx = tid + 256 * i, tok = idx >> 4, ch = idx & 15, t = tok0 + tok;
    float v[8] = {xa[i].x, xa[i].y, xa[i].z, xa[i].w, xb[i].x, xb[i].y, xb[i].z, xb[i].w};
    if constexpr (kNorm) {
      const float4 ga = ld_f4(a.gamma + g * 128 + ch * 8), gb = ld_f4(a.gamma + g * 128 + ch * 8 + 4);
      const float gv[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
      const float inv = s_inv[tok];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (v[k] * inv) * gv[k];
    }
    uint32_t mx = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (t >= a.m) v[k] = 0.0f;
      s_x[ch * 8 + k][tok] = v[k];
      const uint32_t b = __float_as_uint(v[k]) & 0x7fffffffu;
      mx = mx > b ? mx : b;
    }
    const float up = scale_up(lanes_umax<16>(mx), kUp);  // (the 16 lanes of a token)
    const bool in = t < a.n_tok;  // (not past the last token tile)
    uint4* img = a.xs + (size_t(in ? t / T : 0u) * ng + g) * panel_image(T, BITS);
    // (powers of two: exact; the codes enter the products times 16 or 64)
    if (in && ch == 0)
      reinterpret_cast<float*>(img + (panel_image(T, BITS) - kPanelScales / 4))[t % T] =
          (BITS == 4 ? 0.0625f : BITS == 2 ? 0.015625f : 1.0f) / up;
    if constexpr (BITS == 16) {
      float h[8], l[8], r[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float u = v[k] * up;
        h[k] = f16_round(u);
        l[k] = f16_round(u - h[k]);
        r[k] = (u - h[k]) - l[k];
      }
      if (!in) continue;
      uint4* dst = img + (t % T) * 16 + (ch ^ (t & 15u));
      dst[0] = make_uint4(pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7]));
      dst[T * 16] = make_uint4(pack2(l[0], l[1]), pack2(l[2], l[3]), pack2(l[4], l[5]), pack2(l[6], l[7]));
      dst[T * 32] = make_uint4(pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]), pack2(r[6], r[7]));
    } else {
      uint32_t z[8], lo[4], hi[4];  // z: bytes, the balanced limbs of X
#pragma unroll
      for (int k = 0; k < 8; ++k) z[k] = (uint32_t(__float2int_rn(v[k] * up)) + 0x808080u) ^ 0x808080u;
      if constexpr (BITS == 2) {  // (as k_block_limbs: each of a pair sends the four values its neighbour needs)
        const bool odd = (ch & 1u) != 0;
        const uint32_t r0 = pair_u(odd ? z[0] : z[2], 1), r1 = pair_u(odd ? z[1] : z[3], 1);
        const uint32_t r2 = pair_u(odd ? z[4] : z[6], 1), r3 = pair_u(odd ? z[5] : z[7], 1);
        if (odd) {
          limb_words(r0, r2, z[2], z[6], lo);
          limb_words(r1, r3, z[3], z[7], hi);
        } else {
          limb_words(z[0], z[4], r0, r2, lo);
          limb_words(z[1], z[5], r1, r3, hi);
        }
      } else {
        limb_words(z[0], z[2], z[4], z[6], lo);
        limb_words(z[1], z[3], z[5], z[7], hi);
      }
      if (!in) continue;
      uint2* dst = reinterpret_cast<uint2*>(img + (t % T) * 8 + ((ch >> 1) ^ ((t >> 1) & 7u))) + (ch & 1u);
#pragma unroll
      for (int L = 0; L < 4; ++L) dst[size_t(L) * T * 16] = make_uint2(lo[L], hi[L]);
    }
  }
  if (a.xt == nullptr) return;
  __syncthreads();
#pragma unroll 4
  for (uint32_t c = wave; c < 128; c += 4)
    if (tok0 + lane < a.n_tok) a.xt[(size_t(g) * 128 + c) * a.n_tok + tok0 + lane] = s_x[c][lane];
}

// ---- the GEMM -----------------------------------------------------------------------------------
// A workgroup of 4 waves: wave w owns U units (16 weight rows each) of the row tile's 4 U, all of a
// tile of T = 16 TT tokens and a range of groups.  The token tiles pass through LDS (two buffers, one
// barrier per group), the codes go from memory to registers.
struct PanelWork {
  uint32_t tt, rt, range, g_begin, g_end;
};
// workgroup -> (range, row tile, token tile), token tiles fastest; consecutive indexes on one XCD
// (workgroups go round robin over the 8), so that the token tiles of a row tile share its codes in that L2
__device__ __forceinline__ PanelWork panel_work(const PanelGemmArgs& a) {
  const uint32_t N = gridDim.x, xcd = blockIdx.x & 7u, Nq = N >> 3, Nr = N & 7u;
  const uint32_t w = xcd * Nq + (xcd < Nr ? xcd : Nr) + (blockIdx.x >> 3), rr = w / a.ntt;
  PanelWork p;
  p.tt = w % a.ntt;
  p.rt = rr % a.nrt;
  p.range = rr / a.nrt;
  p.g_begin = uint32_t(uint64_t(p.range) * a.ng / a.ranges);
  p.g_end = uint32_t(uint64_t(p.range + 1) * a.ng / a.ranges);
  return p;
}
// the units' parts (consecutive unit ranges); a unit past the last reads unit 0's rows and stores
// nothing, a row past a part's tiles reads row 0 and stores 0
template <int U>
struct PanelRows {
  const uint8_t* base[U];
  uint32_t stride[U], g[U];  // g: the lane's row's first group
  bool ok[U];
  __device__ __forceinline__ PanelRows(const PanelGemmArgs& a, uint32_t u0, uint32_t n) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t uu = u0 + uint32_t(u) < a.n_units ? u0 + uint32_t(u) : 0u;
      int p = 0;
#pragma unroll
      for (int k = 1; k < kMaxParts; ++k) p += (k < a.n_parts && uu >= a.unit_begin[k]) ? 1 : 0;
      p = int(__builtin_amdgcn_readfirstlane(p));
      base[u] = a.base[p];
      stride[u] = a.stride[p];
      const uint32_t r = (uu - a.unit_begin[p]) * 16 + n;
      ok[u] = r < a.wrows[p];
      g[u] = (ok[u] ? r : 0u) * a.ng;
    }
  }
};
// a group's image to LDS: XQ 16-byte pieces, the last kPanelScales / 4 of them in 4-byte loads, one a lane
template <uint32_t XQ>
__device__ __forceinline__ void panel_fetch(const uint4* src, uint4* dst, uint32_t wave, uint32_t lane) {
  constexpr uint32_t P = XQ - kPanelScales / 4;
  static_assert(P % 256 == 0 && kPanelScales == 256, "");
#pragma unroll
  for (uint32_t j = 0; j < P / 256; ++j) {
    const uint32_t i0 = (wave * (P / 256) + j) * 64;
    __builtin_amdgcn_global_load_lds(src + i0 + lane, dst + i0, 16, 0, 0);
  }
  __builtin_amdgcn_global_load_lds(reinterpret_cast<const float*>(src + P) + wave * 64 + lane,
                                   reinterpret_cast<float*>(dst + P) + wave * 64, 4, 0, 0);
}
// the factors of tokens 16 t + 4 q .. + 3 in an image
template <uint32_t XQ>
__device__ __forceinline__ f32x4_t panel_scale(const uint4* img, int t, uint32_t q) {
  return __builtin_bit_cast(f32x4_t, img[XQ - kPanelScales / 4 + 4 * uint32_t(t) + q]);
}
template <int U, int TT>
__device__ __forceinline__ void panel_store(const PanelGemmArgs& a, const PanelWork& p, const PanelRows<U>& R, uint32_t u0,
                                            uint32_t n, uint32_t q, const f32x4_t (&acc)[U][TT]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u0 + uint32_t(u) >= a.n_units) break;
    float* dst = a.partial + (size_t(p.range) * a.rows_all + (u0 + uint32_t(u)) * 16 + n) * a.n_tok + p.tt * (16 * TT) + 4 * q;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const f32x4_t v = acc[u][t];
      *reinterpret_cast<float4*>(dst + 16 * t) = R.ok[u] ? make_float4(v[0], v[1], v[2], v[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
}
// The group loop.  A group's codes are requested three groups ahead (four register sets in turn:
// one group ahead the codes' way from HBM was longer than a group's products, and every wave stood
// at the barrier for it), its token tile one group ahead.  Four groups per trip with no branch
// between them (after one the compiler would move a group's loads down to the block that uses
// them); past the last group the last one's codes are loaded again, not used.  The barrier is
// a bare s_barrier behind a wait for the token tile alone: the only loads younger than it are
// one group's codes (kCodeLoads of them, the order fixed by the scheduling barriers), and for the
// wave's own reads of the buffer that is overwritten next.  The wait is right only if the compiler issues
// at least kCodeLoads vector loads between a tile's and the next wait: one per unit's codes and one per unit's
// scale here (tests/test_panel_isa.py checks every path of every instance).
constexpr int kCodeLoads = 8;
template <class Codes, class Issue, class Fetch, class Compute, class Fold>
__device__ __forceinline__ void panel_loop(const PanelWork& p, uint4* x0, uint4* x1, const Issue& issue, const Fetch& fetch,
                                           const Compute& compute, const Fold& fold) {
  Codes C0, C1, C2, C3;
  const uint32_t last = p.g_end - 1;
  auto at = [&](uint32_t g) { return g < last ? g : last; };
  issue(p.g_begin, C0);
  issue(at(p.g_begin + 1), C1);
  __builtin_amdgcn_sched_barrier(0);
  fetch(p.g_begin, x0);
  __builtin_amdgcn_sched_barrier(0);
  issue(at(p.g_begin + 2), C2);
  __builtin_amdgcn_sched_barrier(0);
  // (restrict: the reads of one buffer do not wait for the loads into the other)
  auto body = [&](uint32_t g, const uint4* __restrict__ cur, uint4* __restrict__ nxt, const Codes& c, Codes& cn) {
    static_assert(kCodeLoads < 16, "");
    // group g's tile has landed (vmcnt), the last group's reads are done (lgkmcnt 0; expcnt at its maximum)
    __builtin_amdgcn_s_waitcnt(0x0070 | kCodeLoads);
    __builtin_amdgcn_s_barrier();                     // .. for every wave, and every wave is done with the other buffer
    fetch(at(g + 1), nxt);
    __builtin_amdgcn_sched_barrier(0);
    issue(at(g + 3), cn);
    __builtin_amdgcn_sched_barrier(0);  // (the loads go out before the products)
    compute(cur, c);
  };
  auto tail = [&](uint32_t g, const uint4* __restrict__ cur, uint4* __restrict__ nxt, const Codes& c) {
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    fetch(at(g + 1), nxt);
    __builtin_amdgcn_sched_barrier(0);
    compute(cur, c);
  };
  uint32_t g = p.g_begin;
  for (; g + 3 < p.g_end; g += 4) {
    body(g, x0, x1, C0, C3);
    body(g + 1, x1, x0, C1, C0);
    body(g + 2, x0, x1, C2, C1);
    body(g + 3, x1, x0, C3, C2);
    fold();
  }
  if (g < p.g_end) tail(g, x0, x1, C0);
  if (g + 1 < p.g_end) tail(g + 1, x1, x0, C1);
  if (g + 2 < p.g_end) tail(g + 2, x0, x1, C2);
  __builtin_amdgcn_s_waitcnt(0);  // (no load into LDS outlives the workgroup)
}

// The same with the codes one group ahead (fp16 weights: a group's codes are four times as many registers)
template <class Codes, class Issue, class Fetch, class Compute>
__device__ __forceinline__ void panel_loop_near(const PanelWork& p, uint4* x0, uint4* x1, const Issue& issue, const Fetch& fetch,
                                                const Compute& compute) {
  Codes CA, CB;
  fetch(p.g_begin, x0);
  issue(p.g_begin, CA);
  // (restrict: the reads of one buffer do not wait for the loads into the other)
  auto body = [&](uint32_t g, const uint4* __restrict__ cur, uint4* __restrict__ nxt, const Codes& c, Codes& cn) {
    __syncthreads();  // group g's tile has landed; every wave is done with the other buffer
    const uint32_t gn = g + 1 < p.g_end ? g + 1 : g;
    fetch(gn, nxt);
    issue(gn, cn);
    __builtin_amdgcn_sched_barrier(0);  // (the loads go out before the products)
    compute(cur, c);
  };
  uint32_t g = p.g_begin;
  for (; g + 1 < p.g_end; g += 2) {
    body(g, x0, x1, CA, CB);
    body(g + 1, x1, x0, CB, CA);
  }
  if (g < p.g_end) body(g, x0, x1, CA, CB);
  __builtin_amdgcn_s_waitcnt(0);  // (no load into LDS outlives the workgroup)
}

// 4- and 2-bit codes.  Lane layouts of v_mfma_i32_16x16x64_i8: A lane (m, q) = token m, k 16 q ..
// + 15; B lane (n, q) = weight row n; D lane (n, q) = row n, tokens 4 q .. 4 q + 3.  The k slots of
// step s hold columns 32 q + 16 s .. + 15 of the group, so a lane's codes are one contiguous piece of
// its row (4-bit: 16 bytes; 2-bit: 8).  The codes enter as bytes 16 (code - 8) (the nibble with its
// top bit flipped is the two's complement; in the high half of the byte it is 16 times it) or 64 times
// the 2-bit value: 4 (7) instructions for 8 (16) codes.  Per token tile and unit the four limbs' exact
// sums, put together exactly in pairs (|D| <= 2^21) and scaled by the token's and the row's group scales.
// (The token's scale, which varies by group, is one of seven instructions of such a sum: 72B gate/up at 300 tokens took 778 us
// with a scale per token, 808 with one per group; the kernels that had to find a token's largest value gained
// part of it back, 6 us a SwiGLU epilogue and 1 to 2 a k_panel_split.)
template <int BITS>
struct PanelCodes {
  uint4 v[4];
  uint32_t sc[4];
};
template <>
struct PanelCodes<2> {
  uint2 v[4];
  uint32_t sc[4];
};
// One wave per SIMD with all the registers: the products of one (token tile, unit) step
// alternate, one to three or four, with the vector instructions of the step before (order fixed by scheduling
// barriers: left to itself the compiler puts the eight products first, then the 28 instructions),
// and the next token tile's operands are read meanwhile.  (The file is built with the products'
// results in vector registers: with 512 registers the compiler otherwise keeps them in accumulator
// registers and copies each value out.  Tiles of 80 tokens and more spill two to four registers, once
// in four groups; 128 tokens spill in every group.)
template <int BITS, int TT>
__global__ void __launch_bounds__(256, 1) k_panel_gemm(PanelGemmArgs a) {
  constexpr uint32_t T = 16 * TT, XQ = panel_image(T, BITS);  // 16-byte pieces of one group's token tile
  __shared__ __align__(16) uint4 s_x0[XQ], s_x1[XQ];
  const uint32_t tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const PanelWork p = panel_work(a);
  const uint32_t u0 = p.rt * 16 + wave * 4;
  const PanelRows<4> R(a, u0, n);
  auto issue = [&](uint32_t g, PanelCodes<BITS>& c) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t G = R.g[u] + g, rec = (G >> 8) * R.stride[u], i = G & 255u;
      if constexpr (BITS == 4) c.v[u] = ld_u128(R.base[u] + (rec + 64u + i * 64u + 16u * q));
      else c.v[u] = ld_u64(R.base[u] + (rec + 64u + i * 32u + 8u * q));
      c.sc[u] = ld_u16(R.base[u] + (rec + 16448u + 48u + 2u * i));
    }
  };
  const uint4* xt = a.xs + size_t(p.tt) * a.ng * XQ;
  auto fetch = [&](uint32_t g, uint4* dst) { panel_fetch<XQ>(xt + size_t(g) * XQ, dst, wave, lane); };
  // acc: the sum over 4 groups, tot: those sums (the roundings of a row of 64 groups halve, and the
  // error stays below that of the block step's shorter column ranges)
  f32x4_t acc[4][TT], tot[4][TT];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t) tot[u][t] = acc[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t a0 = n * 8 + ((2 * q) ^ (n >> 1)), a1 = n * 8 + ((2 * q + 1) ^ (n >> 1));
  auto compute = [&](const uint4* xsrc, const PanelCodes<BITS>& c) {
    i32x4_t B[4][2], A[2][4][2], D[2][4];
    f32x4_t ts[2];
    float sc[4];
    auto read = [&](int t, int L, int s) {
      A[t & 1][L][s] = __builtin_bit_cast(i32x4_t, xsrc[uint32_t(L) * (T * 8) + uint32_t(t) * 128 + (s ? a1 : a0)]);
    };
#pragma unroll
    for (int k = 0; k < 8; ++k) read(0, k & 3, k >> 2);
    ts[0] = panel_scale<XQ>(xsrc, 0, q);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if constexpr (BITS == 4) {
          const uint32_t x = (s ? c.v[u].z : c.v[u].x) ^ 0x88888888u, y = (s ? c.v[u].w : c.v[u].y) ^ 0x88888888u;
          B[u][s] = i32x4_t{int((x << 4) & 0xF0F0F0F0u), int(x & 0xF0F0F0F0u), int((y << 4) & 0xF0F0F0F0u), int(y & 0xF0F0F0F0u)};
        } else {  // (the codebook {0, +1, -2, -1} is the 2-bit two's complement)
          const uint32_t x = s ? c.v[u].y : c.v[u].x;
          B[u][s] = i32x4_t{int((x << 6) & 0xC0C0C0C0u), int((x << 4) & 0xC0C0C0C0u), int((x << 2) & 0xC0C0C0C0u), int(x & 0xC0C0C0C0u)};
        }
      }
      sc[u] = h2f(uint16_t(c.sc[u]));
    }
    // step i: (token tile i / 4, unit i % 4); the last step only finishes the one before
#pragma unroll
    for (int i = 0; i <= 4 * TT; ++i) {
      const int t = i / 4, u = i % 4, b = i & 1, tp = (i - 1) / 4, up = (i - 1) & 3;
      const bool mul = i < 4 * TT, fin = i > 0;
      int lo[4], hi[4];
      float fl[4], fh[4];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (mul) {
          const int L = k & 3, s = k >> 2;
          D[b][L] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t & 1][L][s], B[u][s], s ? D[b][L] : i32x4_t{0, 0, 0, 0}, 0, 0, 0);
        }
        if (fin) {  // 28 instructions in eight threes and fours, the limbs' sums in the order they complete
          const i32x4_t(&E)[4] = D[b ^ 1];
#define CHPE_LO(j) lo[j] = E[0][j] + int(uint32_t(E[1][j]) << 8)
#define CHPE_HI(j) hi[j] = E[2][j] + int(uint32_t(E[3][j]) << 8)
#define CHPE_F(j) fh[j] = fmaf(fh[j], 65536.0f, fl[j])
#define CHPE_S(j) fh[j] *= ts[tp & 1][j]
#define CHPE_ACC(j) acc[up][tp][j] = fmaf(fh[j], sc[up], acc[up][tp][j])
          if (k == 0) CHPE_LO(0), CHPE_LO(1), CHPE_LO(2), CHPE_LO(3);
          if (k == 1) fl[0] = float(lo[0]), fl[1] = float(lo[1]), fl[2] = float(lo[2]);
          if (k == 2) fl[3] = float(lo[3]), CHPE_HI(0), CHPE_HI(1);
          if (k == 3) CHPE_HI(2), CHPE_HI(3), fh[0] = float(hi[0]), fh[1] = float(hi[1]);
          if (k == 4) fh[2] = float(hi[2]), fh[3] = float(hi[3]), CHPE_F(0);
          if (k == 5) CHPE_F(1), CHPE_F(2), CHPE_F(3), CHPE_S(0);
          if (k == 6) CHPE_S(1), CHPE_S(2), CHPE_S(3);
          if (k == 7) CHPE_ACC(0), CHPE_ACC(1), CHPE_ACC(2), CHPE_ACC(3);
#undef CHPE_LO
#undef CHPE_HI
#undef CHPE_F
#undef CHPE_S
#undef CHPE_ACC
        }
        if (mul && t + 1 < TT && (k & 3) == 1) {  // two reads of the next tile per step
          const int r = 2 * u + (k >> 2);
          read(t + 1, r & 3, r >> 2);
        }
        if (mul && t + 1 < TT && u == 1 && k == 2) ts[(t + 1) & 1] = panel_scale<XQ>(xsrc, t + 1, q);  // (the tile before t is done)
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto fold = [&] {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        tot[u][t] += acc[u][t];
        acc[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
  };
  panel_loop<PanelCodes<BITS>>(p, s_x0, s_x1, issue, fetch, compute, fold);
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[u][t] += tot[u][t];
  panel_store<4, TT>(a, p, R, u0, n, q, acc);
}

// fp16 weights: v_mfma_f32_16x16x32_f16, D lane (n, q) = row n, tokens 4 q .. + 3; the k slots of step
// d hold columns 32 q + 8 d .. + 7.  The products are exact; the small parts have a sum of their own, each
// step of 16 columns of the high parts has one, and those are scaled and added up in 64 bits (measured on random
// weights, 128 columns: 0.74 x 2^-24 of the sum, against 1.29 in one chain).  U = 2 units per wave:
// 64 bytes of codes per lane, unit and group.
// The small parts' sum is not the starting value of the first 16 columns' product: that is another opcode, and
// the compiler puts no wait between two products that hand on exactly the same registers.  Where its
// schedule brought the 16x16x16 product within 32 cycles of the 16x16x32 one it starts from, the sum was
// taken too early (the last small part missing) and the logits were 2e-5 to 2e-4 off.
struct PanelHalves {
  uint4 v[2][4];
};
__global__ void __launch_bounds__(256, 2) k_panel_gemm_h(PanelGemmArgs a) {
  constexpr int U = 2, TT = 2;
  constexpr uint32_t T = 16 * TT, XQ = panel_image(T, 16);
  __shared__ __align__(16) uint4 s_x0[XQ], s_x1[XQ];
  const uint32_t tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const PanelWork p = panel_work(a);
  const uint32_t u0 = p.rt * (4 * U) + wave * U;
  const PanelRows<U> R(a, u0, n);
  auto issue = [&](uint32_t g, PanelHalves& c) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int d = 0; d < 4; ++d) c.v[u][d] = ld_u128(R.base[u] + ((R.g[u] + g) * 256u + 64u * q + 16u * uint32_t(d)));
  };
  const uint4* xt = a.xs + size_t(p.tt) * a.ng * XQ;
  auto fetch = [&](uint32_t g, uint4* dst) { panel_fetch<XQ>(xt + size_t(g) * XQ, dst, wave, lane); };
  double acc[U][TT][4];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[u][t][j] = 0.0;
  auto compute = [&](const uint4* xsrc, const PanelHalves& c) {
    auto operand = [&](int part, int d, int t) {
      return as_half8(xsrc[uint32_t(part) * (T * 16) + uint32_t(t) * 256 + n * 16 + ((4 * q + uint32_t(d)) ^ n)]);
    };
    f32x4_t D[U][TT], ts[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) ts[t] = panel_scale<XQ>(xsrc, t, q);
#pragma unroll
    for (int part = 2; part >= 1; --part)
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const f32x4_t c0 = part == 2 && d == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : D[u][t];
            D[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(part, d, t), as_half8(c.v[u][d]), c0, 0, 0, 0);
          }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const half8_t A = operand(0, d, t);
        const half4_t A0 = __builtin_shufflevector(A, A, 0, 1, 2, 3), A1 = __builtin_shufflevector(A, A, 4, 5, 6, 7);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const half8_t B = as_half8(c.v[u][d]);
          const half4_t B0 = __builtin_shufflevector(B, B, 0, 1, 2, 3), B1 = __builtin_shufflevector(B, B, 4, 5, 6, 7);
          const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
          const f32x4_t E0 = __builtin_amdgcn_mfma_f32_16x16x16f16(A0, B0, z, 0, 0, 0);
          const f32x4_t E1 = __builtin_amdgcn_mfma_f32_16x16x16f16(A1, B1, z, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[u][t][j] = fma(double(E0[j]) + double(E1[j]), double(ts[t][j]), acc[u][t][j]);
        }
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[u][t][j] = fma(double(D[u][t][j]), double(ts[t][j]), acc[u][t][j]);
  };
  panel_loop_near<PanelHalves>(p, s_x0, s_x1, issue, fetch, compute);
  f32x4_t sum[U][TT];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[u][t][j] = float(acc[u][t][j]);
  panel_store<U, TT>(a, p, R, u0, n, q, sum);
}

// ---- the epilogue -------------------------------------------------------------------------------
// grid (tiles of 4 OPW outputs, 64-token tiles, x fastest: the tokens' slice of the token-minor
// input, 256 bytes a column, stays in the L2s), 4 waves x OPW consecutive outputs, lane = token.
// The ranges' sums of the OPW rows in flight together; then the rows' packed correction entries,
// which are one consecutive run: 64 entries in one load, one per lane, and 16 columns' loads in
// flight at a time, whatever row they belong to (row by row, with an entry load and a column load
// chain each, the SwiGLU launch of the 72B model at 300 tokens took 334 us; this way 92).  Then
// through LDS to outputs-fastest order for the writes.  Bound by the corrections' reads (4 bytes
// per entry and token, from L2) and the partial sums.
template <int MODE, int OPW>
__global__ void __launch_bounds__(256) k_panel_epi(PanelEpiArgs a) {
  constexpr bool kSwi = MODE == int(GemvMode::SwiGlu);
  constexpr bool kRope = MODE == int(GemvMode::QkvRope);
  constexpr bool kAcc = MODE == int(GemvMode::Accum);
  constexpr int NR = (kSwi || kRope) ? 2 : 1;
  constexpr uint32_t TILE = 4 * OPW;
  __shared__ float s_o[NR][64][TILE + 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tok0 = blockIdx.y * 64, m = a.m, half = a.head_dim / 2;
  const uint32_t tl = tok0 + lane < m ? tok0 + lane : m - 1;
  const size_t rstride = size_t(a.rows_all) * a.n_tok;
  // output o -> part and row (the first of its pair); OPW outputs from a multiple of OPW are
  // consecutive rows (the parts' outputs and half are multiples of 8)
  auto rows_of = [&](uint32_t o, int* part, uint32_t* r0) {
    int p = 0;
    if constexpr (kRope) {
      while (p + 1 < a.n_parts && o >= a.part[p].rows / 2) {
        o -= a.part[p].rows / 2;
        ++p;
      }
      *r0 = (o / half) * (2 * half) + o % half;
    } else {
      *r0 = o;
    }
    *part = p;
  };
  const uint32_t ow = blockIdx.x * TILE + wave * OPW;
  if (ow < a.total) {
    int p;
    uint32_t r0;
    rows_of(ow, &p, &r0);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const PanelPart& P = a.part[kSwi ? k : p];
      const uint32_t r = kRope ? r0 + (k ? half : 0u) : r0;
      const bool has = P.coff != nullptr && r < P.wrows;  // (rows past wrows have no entries)
      uint32_t off = 0;
      if (has) off = P.coff[r + (lane < uint32_t(OPW) ? lane : uint32_t(OPW))];
      const float* ps = a.partial + size_t(P.unit_begin * 16 + r) * a.n_tok + tl;
      double s[OPW];  // (up to 32 ranges one after another: in 64 bits)
#pragma unroll
      for (int i = 0; i < OPW; ++i) s[i] = 0.0;
#pragma unroll 2
      for (uint32_t rg = 0; rg < a.ranges; ++rg)
#pragma unroll
        for (int i = 0; i < OPW; ++i) s[i] += double(ps[rg * rstride + size_t(i) * a.n_tok]);
#pragma unroll
      for (int i = 0; i < OPW; ++i) s_o[k][lane][wave * OPW + i] = float(s[i]);
      const uint32_t eb = __builtin_amdgcn_readlane(off, 0), ee = __builtin_amdgcn_readlane(off, OPW);
      float c = 0.0f;
      uint32_t row = 0, bound = __builtin_amdgcn_readlane(off, 1);
      for (uint32_t e0 = eb; e0 < ee; e0 += 64) {
        const float2 mine = P.cpack[e0 + lane < ee ? e0 + lane : ee - 1];
        const uint32_t n = ee - e0 < 64u ? ee - e0 : 64u;
        for (uint32_t j = 0; j < n; j += 16) {
          float xc[16];
#pragma unroll
          for (uint32_t jj = 0; jj < 16; ++jj) {  // (lanes past the last entry hold it again)
            const uint32_t col = __builtin_amdgcn_readlane(__float_as_uint(mine.x), j + jj);
            xc[jj] = a.xt[size_t(col) * a.n_tok + tl];
          }
#pragma unroll
          for (uint32_t jj = 0; jj < 16; ++jj) {  // (uniform)
            if (j + jj >= n) break;
            while (e0 + j + jj >= bound) {  // the entry's row
              s_o[k][lane][wave * OPW + row] += c;
              c = 0.0f;
              ++row;
              bound = __builtin_amdgcn_readlane(off, row + 1);
            }
            c = fmaf(__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine.y), j + jj)), xc[jj], c);
          }
        }
      }
      if (ee > eb) s_o[k][lane][wave * OPW + row] += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < TILE / 4; ++i) {
    const uint32_t idx = tid + 256 * i, tok = idx / TILE, oi = idx % TILE, t = tok0 + tok, o = blockIdx.x * TILE + oi;
    const bool ok = t < m && o < a.total;
    if constexpr (kAcc) {
      float sq = 0.0f;
      if (ok) {
        float* y = a.part[0].y + size_t(t) * a.part[0].rows + o;
        const bool upd = o < a.part[0].wrows && a.brk[t] == 0u;  // rows past the tiles and broken tokens stay
        const float yo = *y, yn = upd ? yo + s_o[0][tok][oi] : yo;
        if (upd) *y = yn;
        sq = yn * yn;
      }
#pragma unroll
      for (int x = 1; x < int(TILE); x <<= 1) sq = pair_sum(sq, x);
      if (oi == 0 && t < m) a.ssp_out[size_t(blockIdx.x) * kMaxPanel + t] = sq;
    } else if constexpr (kSwi) {
      const float g = s_o[0][tok][oi];
      if (ok) a.part[0].y[size_t(t) * a.part[0].rows + o] = g / (1.0f + expf(-g)) * s_o[1][tok][oi];  // silu(g)*u: :159-161, :1746-1748
    } else if constexpr (kRope) {
#pragma clang fp contract(off)
      if (!ok) continue;
      int p;
      uint32_t r;
      rows_of(o, &p, &r);
      const PanelPart& P = a.part[p];
      const float lo = s_o[0][tok][oi] + (P.bias ? P.bias[r] : 0.0f);
      const float hi = s_o[1][tok][oi] + (P.bias ? P.bias[r + half] : 0.0f);
      const uint32_t pos = a.pos + t, d = r % (2 * half);
      float o0 = lo, o1 = hi;
      if (P.role < kRoleV && pos < a.rope_rows) {  // applyRope :195-216
        const float cc = a.rope_cos[size_t(pos) * half + d], sn = a.rope_sin[size_t(pos) * half + d];
        o0 = lo * cc - hi * sn;
        o1 = lo * sn + hi * cc;
      }
      if (P.role == kRoleQ || P.role == kRoleStore) {
        P.y[size_t(t) * P.rows + r] = o0;
        P.y[size_t(t) * P.rows + r + half] = o1;
      } else if (a.brk[t] == 0u) {  // (a broken token appends no row)
        const uint32_t hd = a.head_dim, head = r / hd;
        void* cache = P.role == kRoleK ? a.k_cache : a.v_cache;
        if (a.kv_f16 && P.role == kRoleV) {  // 4-position blocks: [pos/4][dim][pos%4]
          const size_t blk = (size_t(head) * a.max_seq + (pos & ~3u)) * hd + (pos & 3u);
          reinterpret_cast<__half*>(cache)[blk + size_t(d) * 4] = __float2half_rn(o0);
          reinterpret_cast<__half*>(cache)[blk + size_t(d + half) * 4] = __float2half_rn(o1);
        } else {
          const size_t at = (size_t(head) * a.max_seq + pos) * hd + d;
          if (a.kv_f16) {
            reinterpret_cast<__half*>(cache)[at] = __float2half_rn(o0);
            reinterpret_cast<__half*>(cache)[at + half] = __float2half_rn(o1);
          } else {
            reinterpret_cast<float*>(cache)[at] = o0;
            reinterpret_cast<float*>(cache)[at + half] = o1;
          }
        }
      }
    }
  }
}

// ---- attention ----------------------------------------------------------------------------------
// Workgroup = 16 rows of a kv head: 16 / G tokens x G query heads; wave w takes every fourth step
// of positions (32 or 16) from the w-th, and the four waves' sums meet at the end (one wave per 16
// rows left most SIMDs without work: 98 us per layer of the 3B model at 389 tokens, against 36).  S^T = K Q^T puts row n's scores in
// lanes n, n + 16, n + 32, n + 48, and its layout is the operand layout of O^T = V^T P^T, so
// neither scores nor weights leave the registers.  fp16 cache: query and weights as hi + lo (each
// row's query scaled so that its largest value is near 2^14, weights scaled by 2^14), two products
// each; f32 cache: f32 products.  In the last steps, where some of the wave's tokens see a
// position and others do not, each token runs alone with the positions past it taken out of V, and only
// its own rows keep the sums (0 times a non-finite row is not 0, neither for the token itself nor for the
// ones before it, which do not see that row).  A step's products have a sum of their own, added to the
// rescaled one of the steps before (in one chain over the context the 777-position prompt of the 3B model, f32 cache,
// was 7.8e-6 from its 64-bit logits; this way 7.6e-6, as in the decode steps).
constexpr float kPUp = 16384.0f;

struct SoftRow {
  float m = -INFINITY, l = 0.0f;
};

// The four waves' sums of the 16 rows put together: wave w's running maximum, weight sum and
// weighted values (times `post`) in LDS, each wave's part rescaled to the common maximum; thread
// (row, 4 of 64 dims) writes.
template <int HD, int G>
__device__ __forceinline__ void panel_attn_out(const PanelAttnArgs& a, const f32x4_t (&O)[HD / 16], SoftRow sr,
                                               float post, uint32_t t0, uint32_t kvh) {
  constexpr int DT = HD / 16;
  __shared__ __align__(16) float s_O[4][16][HD + 4];
  __shared__ float s_m[4][16], s_l[4][16];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  float l = pair_sum(sr.l, 16);
  l = pair_sum(l, 32);
  if (q == 0) {
    s_m[wave][n] = sr.m;
    s_l[wave][n] = l;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    *reinterpret_cast<float4*>(&s_O[wave][n][16 * dt + 4 * q]) = make_float4(O[dt][0], O[dt][1], O[dt][2], O[dt][3]);
  __syncthreads();
  const uint32_t row = threadIdx.x >> 4, c = threadIdx.x & 15;
  const uint32_t t = t0 + row / G, head = kvh * G + row % G;
  float M = s_m[0][row], f[4], L = 0.0f;
#pragma unroll
  for (int w = 1; w < 4; ++w) M = fmaxf(M, s_m[w][row]);
#pragma unroll
  for (int w = 0; w < 4; ++w) {  // (a wave with no position: weight 0)
    f[w] = s_l[w][row] == 0.0f ? 0.0f : expf(s_m[w][row] - M);
    L = fmaf(s_l[w][row], f[w], L);
  }
#pragma unroll
  for (int i = 0; i < HD / 64; ++i) {
#pragma clang fp contract(off)
    const uint32_t d = 64 * uint32_t(i) + 4 * c;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float x = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) x = fmaf(f[w] == 0.0f ? 0.0f : s_O[w][row][d + uint32_t(j)], f[w], x);
      v[j] = x * post / L;
    }
    if (a.gate && t < a.m) {  // the hybrid's output gate: times sigmoid(g)
      const float4 g = ld_f4(a.gate + (size_t(t) * a.H + head) * 2 * HD + HD + d);
      v[0] = v[0] * (1.0f / (1.0f + expf(-g.x)));
      v[1] = v[1] * (1.0f / (1.0f + expf(-g.y)));
      v[2] = v[2] * (1.0f / (1.0f + expf(-g.z)));
      v[3] = v[3] * (1.0f / (1.0f + expf(-g.w)));
    }
    if (t < a.m)
      *reinterpret_cast<float4*>(a.out + (size_t(t) * a.H + head) * HD + d) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

template <int HD, int G>
__global__ void __launch_bounds__(256) k_panel_attn_h(PanelAttnArgs a) {
  constexpr int TT = 16 / G, KB = HD / 32, DT = HD / 16;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t n = lane & 15, q = lane >> 4, kvh = blockIdx.y;
  const uint32_t t0 = (gridDim.x - 1 - blockIdx.x) * TT;  // (the longest first)
  const uint32_t t = t0 + n / G, tl = t < a.m ? t : a.m - 1, head = kvh * G + n % G;
  const uint8_t* kc = reinterpret_cast<const uint8_t*>(a.k_cache) + size_t(kvh) * a.max_seq * HD * 2;
  const uint8_t* vc = reinterpret_cast<const uint8_t*>(a.v_cache) + size_t(kvh) * a.max_seq * HD * 2;
  half8_t Qh[KB], Ql[KB];
  float sscale;
  {
    const float* qr = a.q + (size_t(tl) * a.H + head) * HD;
    float4 qa[KB], qb[KB];
    uint32_t mx = 0;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      qa[kb] = ld_f4(qr + 32 * kb + 8 * q);
      qb[kb] = ld_f4(qr + 32 * kb + 8 * q + 4);
      const float v[8] = {qa[kb].x, qa[kb].y, qa[kb].z, qa[kb].w, qb[kb].x, qb[kb].y, qb[kb].z, qb[kb].w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t b = __float_as_uint(v[j]) & 0x7fffffffu;
        mx = mx > b ? mx : b;
      }
    }
    uint32_t o = pair_u(mx, 16);
    mx = mx > o ? mx : o;
    o = pair_u(mx, 32);
    mx = mx > o ? mx : o;
    const float up = scale_up(mx, 14);
    sscale = a.scale / up;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const float v[8] = {qa[kb].x * up, qa[kb].y * up, qa[kb].z * up, qa[kb].w * up,
                          qb[kb].x * up, qb[kb].y * up, qb[kb].z * up, qb[kb].w * up};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        Qh[kb][j] = _Float16(v[j]);
        Ql[kb][j] = _Float16(v[j] - float(Qh[kb][j]));
      }
    }
  }
  f32x4_t O[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  SoftRow sr;
  const uint32_t lim = a.pos + tl, first = a.pos + t0;
  const uint32_t pmax = a.pos + (t0 + TT < a.m ? t0 + TT : a.m) - 1;
  for (uint32_t p0 = wave * 32; p0 <= pmax; p0 += 4 * 32) {
    f32x4_t S[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    uint4 kv[2][KB];
    uint2 vv[2][DT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t p = p0 + 16 * uint32_t(h) + n, pr = p < a.max_seq ? p : a.max_seq - 1;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) kv[h][kb] = ld_u128(kc + (size_t(pr) * HD + 32 * kb + 8 * q) * 2);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t p = p0 + 16 * uint32_t(h) + 4 * q, pr = p < a.max_seq ? p : a.max_seq - 4;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) vv[h][dt] = ld_u64(vc + (size_t(pr / 4) * HD + 16 * dt + n) * 8);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int h = 0; h < 2; ++h) S[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(kv[h][kb]), Ql[kb], S[h], 0, 0, 0);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int h = 0; h < 2; ++h) S[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(kv[h][kb]), Qh[kb], S[h], 0, 0, 0);
    float s[8], mn = sr.m;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t p = p0 + 16 * uint32_t(i / 4) + 4 * q + uint32_t(i % 4);
      s[i] = p <= lim ? S[i / 4][i % 4] * sscale : -INFINITY;
      mn = fmaxf(mn, s[i]);
    }
    mn = pair_max(mn, 16);
    mn = pair_max(mn, 32);
    // (a row that has seen no position yet stays at sum 0)
    const float corr = sr.m == mn ? 1.0f : expf(sr.m - mn);
    sr.m = mn;
    float ls = 0.0f;
    half8_t Ph, Pl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t p = p0 + 16 * uint32_t(i / 4) + 4 * q + uint32_t(i % 4);
      const float e = p <= lim ? expf(s[i] - mn) : 0.0f;
      ls += e;
      const float eu = e * kPUp;
      Ph[i] = _Float16(eu);
      Pl[i] = _Float16(eu - float(Ph[i]));
    }
    sr.l = fmaf(sr.l, corr, ls);
    if (p0 + 31 <= first) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const half8_t V = as_half8(make_uint4(vv[0][dt].x, vv[0][dt].y, vv[1][dt].x, vv[1][dt].y));
        f32x4_t R = __builtin_amdgcn_mfma_f32_16x16x32_f16(V, Pl, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        R = __builtin_amdgcn_mfma_f32_16x16x32_f16(V, Ph, R, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) O[dt][j] = fmaf(O[dt][j], corr, R[j]);
      }
    } else {
      for (uint32_t u = 0; u < uint32_t(TT); ++u) {
        const bool mine = n / G == u;
        const uint32_t last = first + u < pmax ? first + u : pmax;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          uint32_t x[4] = {vv[0][dt].x, vv[0][dt].y, vv[1][dt].x, vv[1][dt].y};
#pragma unroll
          for (int k = 0; k < 4; ++k) {  // (dword k: positions 16 (k / 2) + 4 q + 2 (k % 2), + 1)
            const uint32_t p = p0 + 16 * uint32_t(k / 2) + 4 * q + 2 * uint32_t(k % 2);
            x[k] = (p <= last ? x[k] & 0xFFFFu : 0u) | (p + 1 <= last ? x[k] & 0xFFFF0000u : 0u);
          }
          const half8_t V = as_half8(make_uint4(x[0], x[1], x[2], x[3]));
          f32x4_t R = __builtin_amdgcn_mfma_f32_16x16x32_f16(V, Pl, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          R = __builtin_amdgcn_mfma_f32_16x16x32_f16(V, Ph, R, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) O[dt][j] = mine ? fmaf(O[dt][j], corr, R[j]) : O[dt][j];
        }
      }
    }
  }
  panel_attn_out<HD, G>(a, O, sr, 1.0f / kPUp, t0, kvh);
}

// f32 cache: steps of 16 positions, v_mfma_f32_16x16x4_f32 (A lane (m, q): k = q).  K: lane (p, q)
// dims 16 kb + 4 q .. + 3 (component c of every lane is one product); V: lane (d, q), position
// 4 q + j is product j's k = q, the row's weight of S^T's element j.
template <int HD, int G>
__global__ void __launch_bounds__(256) k_panel_attn_f(PanelAttnArgs a) {
  constexpr int TT = 16 / G, KB = HD / 16, DT = HD / 16;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint32_t n = lane & 15, q = lane >> 4, kvh = blockIdx.y;
  const uint32_t t0 = (gridDim.x - 1 - blockIdx.x) * TT;
  const uint32_t t = t0 + n / G, tl = t < a.m ? t : a.m - 1, head = kvh * G + n % G;
  const float* kc = reinterpret_cast<const float*>(a.k_cache) + size_t(kvh) * a.max_seq * HD;
  const float* vc = reinterpret_cast<const float*>(a.v_cache) + size_t(kvh) * a.max_seq * HD;
  float4 Q[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) Q[kb] = ld_f4(a.q + (size_t(tl) * a.H + head) * HD + 16 * kb + 4 * q);
  f32x4_t O[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  SoftRow sr;
  const uint32_t lim = a.pos + tl, first = a.pos + t0;
  const uint32_t pmax = a.pos + (t0 + TT < a.m ? t0 + TT : a.m) - 1;
  for (uint32_t p0 = wave * 16; p0 <= pmax; p0 += 4 * 16) {
    float4 kv[KB];
    float vv[4][DT];
    {
      const uint32_t p = p0 + n, pr = p < a.max_seq ? p : a.max_seq - 1;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) kv[kb] = ld_f4(kc + size_t(pr) * HD + 16 * kb + 4 * q);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t p = p0 + 4 * q + uint32_t(j), pr = p < a.max_seq ? p : a.max_seq - 1;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) vv[j][dt] = gld(vc + size_t(pr) * HD + 16 * dt + n);
    }
    // sums of 8 products on the matrix cores, then a tree (one chain over a component's 32 products
    // took two and a half times its roundings; a score's error reaches the whole head)
    f32x4_t S[KB / 2][4];
#pragma unroll
    for (int kb = 0; kb < KB; kb += 2) {
      const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
      const float* k0 = &kv[kb].x;
      const float* k1 = &kv[kb + 1].x;
      const float* q0 = &Q[kb].x;
      const float* q1 = &Q[kb + 1].x;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        S[kb / 2][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1[c], q1[c], __builtin_amdgcn_mfma_f32_16x16x4f32(k0[c], q0[c], z, 0, 0, 0), 0, 0, 0);
    }
#pragma unroll
    for (int w = KB / 4; w > 0; w >>= 1)
#pragma unroll
      for (int i = 0; i < w; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) S[i][c] += S[i + w][c];
    float s[4], mn = sr.m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = (S[0][0][i] + S[0][1][i]) + (S[0][2][i] + S[0][3][i]);
      s[i] = p0 + 4 * q + uint32_t(i) <= lim ? v * a.scale : -INFINITY;
      mn = fmaxf(mn, s[i]);
    }
    mn = pair_max(mn, 16);
    mn = pair_max(mn, 32);
    const float corr = sr.m == mn ? 1.0f : expf(sr.m - mn);
    sr.m = mn;
    float e[4], ls = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      e[i] = p0 + 4 * q + uint32_t(i) <= lim ? expf(s[i] - mn) : 0.0f;
      ls += e[i];
    }
    sr.l = fmaf(sr.l, corr, ls);
    if (p0 + 15 <= first) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        f32x4_t R = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) R = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[j][dt], e[j], R, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) O[dt][j] = fmaf(O[dt][j], corr, R[j]);
      }
    } else {
      for (uint32_t u = 0; u < uint32_t(TT); ++u) {
        const bool mine = n / G == u;
        const uint32_t last = first + u < pmax ? first + u : pmax;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          f32x4_t R = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 4; ++j)
            R = __builtin_amdgcn_mfma_f32_16x16x4f32(p0 + 4 * q + uint32_t(j) <= last ? vv[j][dt] : 0.0f, e[j], R, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) O[dt][j] = mine ? fmaf(O[dt][j], corr, R[j]) : O[dt][j];
        }
      }
    }
  }
  panel_attn_out<HD, G>(a, O, sr, 1.0f, t0, kvh);
}

}  // namespace

void launch_panel_begin(StepState* state, uint32_t token, uint32_t pos, hipStream_t st) {
  launch_kernel(&k_panel_begin, dim3(1), dim3(1), st, state, token, pos);
}

void launch_panel_split(const PanelSplitArgs& a, uint32_t bits, hipStream_t st) {
  const dim3 grid(a.C / 128, (a.n_tok + 63) / 64);
  auto go = [&](auto norm, auto plain) {
    if (a.gamma) launch_kernel(norm, grid, dim3(256), st, a);
    else launch_kernel(plain, grid, dim3(256), st, a);
  };
  if (bits == 16) go(&k_panel_split<true, 16>, &k_panel_split<false, 16>);
  else if (bits == 2) go(&k_panel_split<true, 2>, &k_panel_split<false, 2>);
  else go(&k_panel_split<true, 4>, &k_panel_split<false, 4>);
}

// The cut with the least time: the workgroups in rounds over the 256 CUs -- a group takes a workgroup
// about 0.35 us per 16 tokens, a range starts and ends in about three groups' time --, and a
// range's partial sums written and read back at 4 TB/s.  Tiles of 64 to 112 tokens (a longer one reads
// fewer codes per product, a shorter one may leave fewer rows of the last tile empty), 32 for
// panels of up to 32 tokens and for fp16 weights.
PanelShape panel_shape(uint32_t n_units, uint32_t ng, uint32_t m, uint32_t bits, size_t max_partials) {
  PanelShape best{};
  float best_us = 1e30f;
  const uint32_t rt_units = bits == 16 ? 8u : 16u, nrt = (n_units + rt_units - 1) / rt_units;
  const bool small = m <= 32 || bits == 16;
  for (uint32_t tt = small ? 2 : 4; tt <= (small ? 2u : 7u); ++tt) {
    const uint32_t tile = 16 * tt, ntt = (m + tile - 1) / tile;
    const size_t sums = size_t(n_units) * 16 * ntt * tile;
    for (uint32_t R = 1; R <= ng && R <= 32 && R * sums <= max_partials; ++R) {
      const uint32_t rounds = (nrt * ntt * R + 255) / 256;
      const float us = float(rounds) * (float((ng + R - 1) / R) + 3.0f) * (0.35f * float(tt)) + float(R) * float(sums) * 8.0f / 4e6f;
      if (us < best_us) {
        best_us = us;
        best = PanelShape{tile, ntt, nrt, R};
      }
    }
  }
  return best;
}

template <int BITS>
bool launch_panel_gemm_of(const PanelGemmArgs& a, uint32_t tile, dim3 grid, hipStream_t st) {
  switch (tile) {
    case 32: launch_kernel(&k_panel_gemm<BITS, 2>, grid, dim3(256), st, a); break;
    case 64: launch_kernel(&k_panel_gemm<BITS, 4>, grid, dim3(256), st, a); break;
    case 80: launch_kernel(&k_panel_gemm<BITS, 5>, grid, dim3(256), st, a); break;
    case 96: launch_kernel(&k_panel_gemm<BITS, 6>, grid, dim3(256), st, a); break;
    case 112: launch_kernel(&k_panel_gemm<BITS, 7>, grid, dim3(256), st, a); break;
    default: return false;
  }
  return true;
}

bool launch_panel_gemm(const PanelGemmArgs& a, uint32_t bits, uint32_t tile, hipStream_t st) {
  const dim3 grid(a.nrt * a.ntt * a.ranges);
  if (bits == 16) {
    if (tile != 32) return false;
    launch_kernel(&k_panel_gemm_h, grid, dim3(256), st, a);
    return true;
  }
  return bits == 2 ? launch_panel_gemm_of<2>(a, tile, grid, st) : launch_panel_gemm_of<4>(a, tile, grid, st);
}

// outputs per workgroup: 32, or 16 where that leaves the CUs short of workgroups
uint32_t panel_epi_tile(uint32_t total, uint32_t m) {
  return ((total + 31) / 32) * ((m + 63) / 64) < 1024 ? 16u : 32u;
}

void launch_panel_epi(const PanelEpiArgs& a, GemvMode mode, hipStream_t st) {
  const uint32_t tile = panel_epi_tile(a.total, a.m);
  const dim3 grid((a.total + tile - 1) / tile, (a.m + 63) / 64);
  auto go = [&](auto k32, auto k16) {
    if (tile == 32) launch_kernel(k32, grid, dim3(256), st, a);
    else launch_kernel(k16, grid, dim3(256), st, a);
  };
  if (mode == GemvMode::Accum) go(&k_panel_epi<int(GemvMode::Accum), 8>, &k_panel_epi<int(GemvMode::Accum), 4>);
  else if (mode == GemvMode::SwiGlu) go(&k_panel_epi<int(GemvMode::SwiGlu), 8>, &k_panel_epi<int(GemvMode::SwiGlu), 4>);
  else go(&k_panel_epi<int(GemvMode::QkvRope), 8>, &k_panel_epi<int(GemvMode::QkvRope), 4>);
}

void launch_panel_attention(const PanelAttnArgs& a, hipStream_t st) {
  const uint32_t G = a.H / a.KV, TT = 16 / G;  // (attention_supported: 128 / 8 or 256 / 4)
  const dim3 grid((a.m + TT - 1) / TT, a.KV);
  if (a.hd == 128) {
    if (a.kv_f16) launch_kernel(&k_panel_attn_h<128, 8>, grid, dim3(256), st, a);
    else launch_kernel(&k_panel_attn_f<128, 8>, grid, dim3(256), st, a);
  } else {
    if (a.kv_f16) launch_kernel(&k_panel_attn_h<256, 4>, grid, dim3(256), st, a);
    else launch_kernel(&k_panel_attn_f<256, 4>, grid, dim3(256), st, a);
  }
}

}  // namespace chpe
