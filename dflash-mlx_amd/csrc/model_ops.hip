// The non-GEMM operators of the Qwen3.5 hybrid target's verify step on gfx950.
//
// Around the gated-delta layers (gdn_layer_ops.hip, gdn_scan.hip) the
// reference's target model (DecoderLayer, dflash_mlx/custom_qwen35_model.py:
// 815-846; Qwen3_5TextModel.__call__ :860-881) runs, per decoder layer:
//   residual add + RMSNorm (nn.RMSNorm input/post-attention layernorms,
//   :824-827, applied :841-845; final norm :881), the MLP silu(gate) * up
//   (mlx-lm Qwen3NextMLP, :845),
//   and on every 4th layer the gated full attention of
//   forward_full_attention_layer_explicit (:487-540): q/k RMSNorm, partial
//   rotary embedding at the cache offset, KV-cache append, causal SDPA over the
//   cache, output * sigmoid(gate).
// The projections are this package's GEMMs (skinny_gemm.hip at verify
// sizes, prefill_gemm.hip over a prompt) and stay with the caller.  Cache
// lengths live in device memory, so a whole verify step (append, attend,
// accept, commit) runs without a host round trip.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <stdint.h>

#include "dflash_gdn.h"
#include "device_common.h"
#include "host_common.h"

namespace dflash {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u32x4 ld16(const void* p) { return *reinterpret_cast<const u32x4*>(p); }

__device__ __forceinline__ void unpack8(u32x4 w, float* f) {
  f[0] = bf16_lo(w.x); f[1] = bf16_hi(w.x);
  f[2] = bf16_lo(w.y); f[3] = bf16_hi(w.y);
  f[4] = bf16_lo(w.z); f[5] = bf16_hi(w.z);
  f[6] = bf16_lo(w.w); f[7] = bf16_hi(w.w);
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return (uint32_t)f32_to_bf16_rne(a) | ((uint32_t)f32_to_bf16_rne(b) << 16);
}

__device__ __forceinline__ u32x4 pack8(const float* f) {
  return u32x4{pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7])};
}

__device__ __forceinline__ float bf16_round(float x) { return bf16_bits_to_f32(f32_to_bf16_rne(x)); }

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Max over the 16 lanes of one DPP row; every lane of the row gets it.
__device__ __forceinline__ float row16_max(float x) {
  x = fmaxf(x, dpp_mov<kDppQuadSwap1>(x));
  x = fmaxf(x, dpp_mov<kDppQuadSwap2>(x));
  x = fmaxf(x, dpp_mov<kDppRowHalfMirror>(x));
  x = fmaxf(x, dpp_mov<kDppRowMirror>(x));
  return x;
}

__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }

// ------------------------------------------------------------ add + RMSNorm
// h = bf16(x + r) (the residual stream, stored to h_out), y = bf16(h *
// rsqrt(mean(h^2) + eps) * w), fp32 arithmetic.  The branch r is either bf16
// [M, H] or (PART) the fp32 split-K partial sums of the projection that
// produced it, rp[nsplit][M][H], rounded to bf16 after the sum (where the
// projection's own output would be rounded).  One workgroup per row (verify
// steps have only B*T rows) of one thread per 8-element chunk (H / 8 threads,
// up to 1024): every thread issues all of its loads (x, and every split of
// r: NS of them, a compile-time count for the common split factors) before
// using any, so a row costs one memory round trip.  With tok != nullptr, x
// is the embedding table and row m reads table row tok[m] (clamped to
// [0, vocab)), stored to h_out as the residual stream's start.  With hc !=
// nullptr, h is also stored to row m of hc (row stride hc_stride elements):
// the target hidden state a drafter reads at selected layers.
template <bool PART, int NS>
__global__ __launch_bounds__(1024) void add_rmsnorm_kernel(const uint16_t* x, const int32_t* tok,
                                                           int vocab, const uint16_t* r,
                                                           const float* rp, int nsplit,
                                                           const uint16_t* w, uint16_t* h_out,
                                                           uint16_t* hc, int64_t hc_stride,
                                                           uint16_t* y, int M, int H, float eps) {
  __shared__ float wsum[16];
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const int ch = tid;
  const bool live = ch < (H >> 3);
  const int chc = live ? ch : 0;  // idle threads load chunk 0 and drop it
  const int64_t xrow = tok != nullptr ? (int64_t)min(max(tok[row], 0), vocab - 1) : row;
  const u32x4 wraw = ld16(w + chc * 8);  // the norm weight, up front with the row's loads
  float v[8];
  unpack8(ld16(x + xrow * H + chc * 8), v);
  if (PART) {
    const float* src = rp + (int64_t)row * H + chc * 8;
    const int64_t sstride = (int64_t)M * H;
    f32x4 p0[NS > 0 ? NS : 1], p1[NS > 0 ? NS : 1];
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
    if (NS > 0) {
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        p0[k] = *reinterpret_cast<const f32x4*>(src + k * sstride);
        p1[k] = *reinterpret_cast<const f32x4*>(src + k * sstride + 4);
      }
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        s0 += p0[k];
        s1 += p1[k];
      }
    } else {
#pragma unroll 8
      for (int k = 0; k < nsplit; ++k) {
        s0 += *reinterpret_cast<const f32x4*>(src + k * sstride);
        s1 += *reinterpret_cast<const f32x4*>(src + k * sstride + 4);
      }
    }
    const float rv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_round(v[e] + bf16_round(rv[e]));
  } else if (r != nullptr) {
    float rv[8];
    unpack8(ld16(r + (int64_t)row * H + chc * 8), rv);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_round(v[e] + rv[e]);
  }
  float ss = 0.f;
  if (live) {
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) wsum[tid >> 6] = ss;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) tot += wsum[i];
  const float inv = 1.f / sqrtf(tot / (float)H + eps);
  if (live) {
    if ((PART || r != nullptr || tok != nullptr) && h_out != nullptr)
      *reinterpret_cast<u32x4*>(h_out + (int64_t)row * H + ch * 8) = pack8(v);
    if (hc != nullptr) *reinterpret_cast<u32x4*>(hc + (int64_t)row * hc_stride + ch * 8) = pack8(v);
    float wv[8], o[8];
    unpack8(wraw, wv);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = v[e] * inv * wv[e];
    *reinterpret_cast<u32x4*>(y + (int64_t)row * H + ch * 8) = pack8(o);
  }
}

// ------------------------------------------------------------------ SwiGLU
// out[m][i] = bf16(silu(gu[m][i]) * gu[m][I + i]).
__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t* gu, uint16_t* out, int M,
                                                     int I) {
  const int per_row = I >> 3;
  const int64_t n = (int64_t)M * per_row;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int m = (int)(e / per_row);
    const int c = (int)(e - (int64_t)m * per_row);
    const uint16_t* row = gu + (int64_t)m * 2 * I;
    float g[8], u[8], o[8];
    unpack8(ld16(row + c * 8), g);
    unpack8(ld16(row + I + c * 8), u);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = silu(g[k]) * u[k];
    *reinterpret_cast<u32x4*>(out + (int64_t)m * I + c * 8) = pack8(o);
  }
}

// ------------------------------------------------------- attention: prepare
// One wave per (token, head slot); D = 128, lane l holds features 2l, 2l+1.
// Slots [0, Hq): query heads (RMSNorm with q_norm_w, rotary, -> q_out);
// [Hq, Hq+Hkv): key heads (RMSNorm with k_norm_w, rotary, -> K cache row);
// [Hq+Hkv, Hq+2Hkv): value heads (-> V^T cache column).  Position of token t
// of sequence b: lens[b] + t.  Rotary (non-interleaved, first `rot` features):
// feature i < rot/2 pairs with i + rot/2 at angle pos * base^(-2i/rot).
struct AttnPrepParams {
  const uint16_t* proj;  // [B*T, row_stride]: Hq x (q | gate) of D each, then Hkv x k, Hkv x v
  int64_t row_stride;
  const uint16_t* q_norm_w;
  const uint16_t* k_norm_w;
  const int32_t* lens;
  uint16_t* k_cache;   // [B, Hkv, Smax, D]
  uint16_t* vt_cache;  // [B, Hkv, D, Smax]
  uint16_t* q_out;     // [B, T, Hq, D]
  int32_t* overflow;   // [B] or null: set to 1 when a block position falls outside [0, Smax)
  int B, T, Hq, Hkv, Smax, rot;
  int skip_v;          // value heads left to attn_prep_vt_kernel
  int heads, groups;   // attn_prep_rows_kernel: heads a wave, waves a token
  double log2_base;
  float eps;
};

constexpr int kHD = 128;  // attention head dim supported by these kernels

// pos * base^(-2i/rot) reduced to [0, 2*pi), computed in fp64.
__device__ __forceinline__ float rope_angle(int pos, int i, int rot, double log2_base) {
  const double inv_freq = exp2(-(double)(2 * i) / (double)rot * log2_base);
  const double a = (double)pos * inv_freq;
  const double two_pi = 6.283185307179586476925286766559;
  return (float)(a - two_pi * floor(a / two_pi));
}

// Rotation of a lane's features 2l and 2l + 1 at position pos (sine and cosine
// of both; only lanes below rot / 2 rotate).
struct Rotation {
  float s0, c0, s1, c1;
};

__device__ __forceinline__ Rotation rotation_of(int pos, int d0, int rot, double log2_base) {
  Rotation r{0.f, 1.f, 0.f, 1.f};
  if (d0 < rot) {
    const int half = rot >> 1;
    const int i0 = d0 < half ? d0 : d0 - half;
    // Angles in fp64, reduced modulo 2*pi before the fp32 sincos: at
    // positions of several thousand an fp32 angle would carry ~1e-4 rad of
    // rounding.
    sincosf(rope_angle(pos, i0, rot, log2_base), &r.s0, &r.c0);
    sincosf(rope_angle(pos, i0 + 1, rot, log2_base), &r.s1, &r.c1);
  }
  return r;
}

// A head's row (this lane's two features of it): RMSNorm and rotary by rotation(),
// packed.  x c and the product p s round once each, whatever the compiler would
// contract where this is inlined: every kernel rotates to the same bits.
template <class Rot>
__device__ __forceinline__ uint32_t norm_rotate(uint32_t xv, uint32_t wv, Rot rotation, int d0, int rot,
                                                float eps) {
  float x0 = bf16_lo(xv), x1 = bf16_hi(xv);
  const float ss = wave_sum(x0 * x0 + x1 * x1);
  const float inv = 1.f / sqrtf(ss / (float)kHD + eps);
  x0 = x0 * inv * bf16_lo(wv);
  x1 = x1 * inv * bf16_hi(wv);
  if (rot > 0) {
    const float p0 = __shfl_xor(x0, rot >> 2, 64);
    const float p1 = __shfl_xor(x1, rot >> 2, 64);
    if (d0 < rot) {
      const Rotation r = rotation();
      const float q0 = p0 * r.s0, q1 = p1 * r.s1;
      const bool low = d0 < (rot >> 1);
      x0 = fmaf(x0, r.c0, low ? -q0 : q0);
      x1 = fmaf(x1, r.c1, low ? -q1 : q1);
    }
  }
  return pack2(x0, x1);
}

__global__ __launch_bounds__(256) void attn_prep_kernel(const AttnPrepParams p) {
  const int bt = blockIdx.x;
  const int slot = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (slot >= p.Hq + 2 * p.Hkv) return;
  const int b = bt / p.T;
  const int t = bt - b * p.T;
  const int pos = p.lens[b] + t;
  // A position outside the cache is never written; the sequence's overflow
  // word records it so the host can refuse the step's output.
  const bool in_cache = pos >= 0 && pos < p.Smax;
  if (!in_cache && slot == 0 && lane == 0 && p.overflow != nullptr) p.overflow[b] = 1;
  const uint16_t* row = p.proj + (int64_t)bt * p.row_stride;
  const int d0 = 2 * lane;
  if (slot >= p.Hq + p.Hkv) {  // value head: V^T cache column
    if (p.skip_v) return;
    const int h = slot - p.Hq - p.Hkv;
    const uint32_t vv = *reinterpret_cast<const uint32_t*>(row + p.Hq * 2 * kHD + p.Hkv * kHD + h * kHD + d0);
    if (in_cache) {
      uint16_t* col = p.vt_cache + (((int64_t)b * p.Hkv + h) * kHD + d0) * p.Smax + pos;
      col[0] = (uint16_t)vv;
      col[p.Smax] = (uint16_t)(vv >> 16);
    }
    return;
  }
  const bool is_q = slot < p.Hq;
  const int h = is_q ? slot : slot - p.Hq;
  const uint16_t* src = is_q ? row + h * 2 * kHD : row + p.Hq * 2 * kHD + h * kHD;
  const uint32_t xv = *reinterpret_cast<const uint32_t*>(src + d0);
  const uint32_t wv = *reinterpret_cast<const uint32_t*>((is_q ? p.q_norm_w : p.k_norm_w) + d0);
  const uint32_t packed = norm_rotate(
      xv, wv, [&] { return rotation_of(pos, d0, p.rot, p.log2_base); }, d0, p.rot, p.eps);
  if (is_q) {
    *reinterpret_cast<uint32_t*>(p.q_out + ((int64_t)bt * p.Hq + h) * kHD + d0) = packed;
  } else if (in_cache) {
    *reinterpret_cast<uint32_t*>(p.k_cache + (((int64_t)b * p.Hkv + h) * p.Smax + pos) * kHD + d0) =
        packed;
  }
}

// The query and key heads of a long input, a wave walking `heads` of a token's
// in turn: the fp64 angles and their sines, the longest part of a head's work,
// are the token's and are computed once, and the next heads' rows are loaded
// while these are normalized.  What is left is mostly the traffic of the q
// and k rows.  With the value launch, 16 query and 4 key heads, a wave a head
// (attn_prep_kernel) -> this: 420 tokens 10.5 -> 9.9 us, 1024 16.2 -> 11.9, 2048
// 26.5 -> 16.0, 4096 46.7 -> 23.8, 8192 84.4 -> 33.6; both kernels give the same bits.
constexpr int kPrepBatch = 4;  // heads loaded together
__global__ __launch_bounds__(256) void attn_prep_rows_kernel(const AttnPrepParams p) {
  // (waves < 2^32: more than one a token only below 16 waves a compute unit)
  const uint32_t w = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t bt = w / (uint32_t)p.groups;
  if (bt >= (int64_t)p.B * p.T) return;
  const int lane = threadIdx.x & 63, d0 = 2 * lane;
  const int first = (int)(w - bt * p.groups) * p.heads;
  const int end = min(first + p.heads, p.Hq + p.Hkv);
  const int b = (int)((uint32_t)bt / (uint32_t)p.T);
  const uint16_t* row = p.proj + bt * p.row_stride + d0;
  auto load = [&](uint32_t (&x)[kPrepBatch], int s0) {
#pragma unroll
    for (int u = 0; u < kPrepBatch; ++u) {
      const int s = min(s0 + u, end - 1);
      x[u] = *reinterpret_cast<const uint32_t*>(row + (s < p.Hq ? 2 * s : p.Hq + s) * kHD);
    }
  };
  uint32_t xv[kPrepBatch], next[kPrepBatch];
  load(xv, first);
  const uint32_t wq = *reinterpret_cast<const uint32_t*>(p.q_norm_w + d0);
  const uint32_t wk = *reinterpret_cast<const uint32_t*>(p.k_norm_w + d0);
  const int pos = p.lens[b] + (int)(bt - (int64_t)b * p.T);
  const bool in_cache = pos >= 0 && pos < p.Smax;
  if (!in_cache && first == 0 && lane == 0 && p.overflow != nullptr) p.overflow[b] = 1;
  const Rotation r = rotation_of(pos, d0, p.rot, p.log2_base);
  for (int s0 = first; s0 < end; s0 += kPrepBatch) {
    load(next, min(s0 + kPrepBatch, end - 1));
#pragma unroll
    for (int u = 0; u < kPrepBatch; ++u) {
      const int s = s0 + u;
      if (s >= end) break;
      const bool is_q = s < p.Hq;
      const uint32_t packed = norm_rotate(xv[u], is_q ? wq : wk, [&] { return r; }, d0, p.rot, p.eps);
      if (is_q) {
        *reinterpret_cast<uint32_t*>(p.q_out + (bt * p.Hq + s) * kHD + d0) = packed;
      } else if (in_cache) {
        *reinterpret_cast<uint32_t*>(p.k_cache +
                                     (((int64_t)b * p.Hkv + s - p.Hq) * p.Smax + pos) * kHD + d0) = packed;
      }
    }
#pragma unroll
    for (int u = 0; u < kPrepBatch; ++u) xv[u] = next[u];
  }
}

// The value heads of a long input (a prompt pass) into the transposed cache:
// workgroup (block of kVtTile tokens, value head h, sequence b).  Per token
// the value row is one 256-byte run of proj, but in vt_cache each of its 128
// features lands in another row (Smax positions apart), so one wave a token
// scatters 2-byte stores.  Here the block's rows go to LDS (16 bytes a
// thread) and each feature's kVtTile positions are then stored by
// consecutive lanes: one 128-byte run a store.  Positions outside
// [0, Smax) are not written (attn_prep_kernel's query head 0 records them
// in the overflow word).  The values are copied bit for bit.
constexpr int kVtTile = 64;

__global__ __launch_bounds__(256) void attn_prep_vt_kernel(const AttnPrepParams p) {
  __shared__ uint32_t sv[kVtTile][kHD / 2 + 1];  // a row of 128 bf16, 4 bytes of pad
  const int t0 = blockIdx.x * kVtTile, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int nt = min(kVtTile, p.T - t0);
  // piece e: token e / 16, features 8 (e % 16) .. +7
#pragma unroll
  for (int i = 0; i < kVtTile * kHD / 8 / 256; ++i) {
    const int e = tid + 256 * i;
    const int tk = e >> 4, c = e & 15;
    if (tk < nt) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(
          p.proj + ((int64_t)b * p.T + t0 + tk) * p.row_stride + p.Hq * 2 * kHD + p.Hkv * kHD +
          h * kHD + 8 * c);
#pragma unroll
      for (int w = 0; w < 4; ++w) sv[tk][4 * c + w] = v[w];
    }
  }
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6;
  const int pos = p.lens[b] + t0 + lane;
  if (lane >= nt || pos < 0 || pos >= p.Smax) return;
  uint16_t* col = p.vt_cache + ((int64_t)b * p.Hkv + h) * kHD * p.Smax + pos;
  for (int d = wave; d < kHD; d += 4) {
    const uint32_t pair = sv[lane][d >> 1];
    col[(int64_t)d * p.Smax] = (uint16_t)((d & 1) ? (pair >> 16) : pair);
  }
}

// ------------------------------------------------ attention: split-K partials
// Workgroup per (key split s, kv head h, sequence b), one wave per query head
// of the group (REP = Hq / Hkv waves).  Wave rows are the T <= 16 block
// tokens; keys are the split's KC = 64 cache positions.  The split's K rows
// (64 x 256 B) and V^T rows (128 x 128 B) are read once per workgroup, every
// thread loading its share of 16-byte pieces, into LDS (rows padded by 16 B
// against bank conflicts); each wave then reads its MFMA fragments from LDS.
// (With one global read per wave, the REP waves fetched the same 32 KB REP
// times: 12.9 us per call at the Qwen3.5-4B shape against 7.4 us staged.)
// S = Q K^T and O = P V on v_mfma_f32_16x16x32_bf16 (A lane = (row l%16,
// k 8(l/16)..+7), B lane = (col l%16, same k), D lane = (col l%16, rows
// 4(l/16)+e)).  Keys at or past lens[b] + T, and keys past lens[b] + t for
// row t (causal), get no weight.  Writes per (row, split): the running max
// m, the sum l of exp(S - m) and the unnormalised O.
constexpr int KC = 64;

struct AttnParams {
  const uint16_t* q;         // [B, T, Hq, D]
  const uint16_t* k_cache;   // [B, Hkv, Smax, D]
  const uint16_t* vt_cache;  // [B, Hkv, D, Smax]
  const int32_t* lens;
  const uint16_t* gate_src;  // proj rows: gate of head qh at qh*2D + D
  int64_t gate_row_stride;
  uint16_t* out;             // [B, T, Hq*D]
  float* part_o;             // [B, Hkv, nsplit, rep, 16, D]
  float* part_ml;            // [B, Hkv, nsplit, rep, 16, 2]
  int B, T, Hq, Hkv, Smax, nsplit;
  float scale;
};

template <int REP>
__global__ __launch_bounds__(256) void attn_partial_kernel(const AttnParams p) {
  constexpr int NT = 64 * REP;                      // threads
  constexpr int PIECES = KC * kHD * 2 / 16;         // 16-byte pieces of K (and of V^T)
  constexpr int PER = (PIECES + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) uint16_t sK[KC][kHD + 8];
  __shared__ __attribute__((aligned(16))) uint16_t sV[kHD][KC + 8];
  __shared__ __attribute__((aligned(16))) uint16_t sP[REP][16][KC + 8];
  const int s = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int qh = h * REP + wave;
  const int base_len = p.lens[b];
  const int L = base_len + p.T;
  const int k0 = s * KC;
  const int64_t prow = (((int64_t)b * p.Hkv + h) * p.nsplit + s) * REP + wave;  // x 16 rows
  if (k0 >= L) {  // split past the keys: no weight
    if (r16 == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p.part_ml[(prow * 16 + 4 * g4 + e) * 2] = -INFINITY;
        p.part_ml[(prow * 16 + 4 * g4 + e) * 2 + 1] = 0.f;
      }
    }
    return;
  }
  // The split's K and V^T, every piece's load issued before any is stored.
  const uint16_t* kbase = p.k_cache + (((int64_t)b * p.Hkv + h) * p.Smax + k0) * kHD;
  const uint16_t* vbase = p.vt_cache + ((int64_t)b * p.Hkv + h) * kHD * p.Smax + k0;
  u32x4 kv[PER], vv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = min(tid + NT * i, PIECES - 1);
    kv[i] = ld16(kbase + (int64_t)(e >> 4) * kHD + (e & 15) * 8);
    vv[i] = ld16(vbase + (int64_t)(e >> 3) * p.Smax + (e & 7) * 8);
  }
  // Q rows (block tokens), 4 k-steps of 32 features.
  const int tq = r16 < p.T ? r16 : p.T - 1;
  const uint16_t* qr = p.q + (((int64_t)b * p.T + tq) * p.Hq + qh) * kHD + g4 * 8;
  u32x4 qa[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const u32x4 v = ld16(qr + 32 * k);
    qa[k] = r16 < p.T ? v : u32x4{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = tid + NT * i;
    if (e < PIECES) {
      *reinterpret_cast<u32x4*>(&sK[e >> 4][(e & 15) * 8]) = kv[i];
      *reinterpret_cast<u32x4*>(&sV[e >> 3][(e & 7) * 8]) = vv[i];
    }
  }
  __syncthreads();
  // S tiles for the 4 groups of 16 keys.
  f32x4 sacc[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, qa[k]),
          __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&sK[16 * n + r16][32 * k + 8 * g4])),
          acc, 0, 0, 0);
    sacc[n] = acc;
  }
  // Masked, scaled scores; row max and sum over the split (row = 4 g4 + e,
  // spread over the 16 lanes of DPP row g4 and the 4 key groups).
  float sv[4][4];
  float m[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int t = 4 * g4 + e;
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int key = k0 + 16 * n + r16;
      const bool ok = (t < p.T) && (key < L) && (key <= base_len + t);
      sv[n][e] = ok ? sacc[n][e] * p.scale : -INFINITY;
      mx = fmaxf(mx, sv[n][e]);
    }
    m[e] = row16_max(mx);
    const float ms = m[e] == -INFINITY ? 0.f : m[e];
    float sum = 0.f;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const float pe = __expf(sv[n][e] - ms);
      sv[n][e] = pe;
      sum += pe;
    }
    l[e] = row16_sum(sum);
  }
  // P (bf16) through LDS into A-operand order: rows t, keys contiguous.
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int n = 0; n < 4; ++n) sP[wave][4 * g4 + e][16 * n + r16] = f32_to_bf16_rne(sv[n][e]);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's P writes are visible to it
  u32x4 pa[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) pa[k] = *reinterpret_cast<const u32x4*>(&sP[wave][r16][32 * k + 8 * g4]);
  // O = P V over 8 tiles of 16 features; V^T rows hold the keys contiguously.
  float* po = p.part_o + prow * 16 * kHD;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 2; ++k)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, pa[k]),
          __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&sV[16 * dt + r16][32 * k + 8 * g4])),
          acc, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) po[(4 * g4 + e) * kHD + 16 * dt + r16] = acc[e];
  }
  if (r16 == 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p.part_ml[(prow * 16 + 4 * g4 + e) * 2] = m[e];
      p.part_ml[(prow * 16 + 4 * g4 + e) * 2 + 1] = l[e];
    }
  }
}

// ------------------------------------------------- attention: combine + gate
// One workgroup per (token, query head): wave w merges the live splits
// s = w, w+4, ... (lane l holds features 2l, 2l+1), then the four partial
// (max, sum, O) merge through LDS; normalise, multiply by sigmoid(gate),
// write bf16.  Splits past lens[b] + T are never read.
__global__ __launch_bounds__(256) void attn_combine_kernel(const AttnParams p) {
  __shared__ float sm[4], sl[4];
  __shared__ f32x2 so[4][64];
  const int bt = blockIdx.x;
  const int qh = blockIdx.y;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int b = bt / p.T;
  const int t = bt - b * p.T;
  const int rep = p.Hq / p.Hkv;
  const int h = qh / rep, w = qh - h * rep;
  const int live = min(p.nsplit, (p.lens[b] + p.T + KC - 1) / KC);
  const int64_t prow0 = (((int64_t)b * p.Hkv + h) * p.nsplit) * rep + w;  // split 0
  // running merge over this wave's splits, 4 loads in flight per step
  float m = -INFINITY, l = 0.f, a0 = 0.f, a1 = 0.f;
  for (int s0 = wave; s0 < live; s0 += 16) {
    float ms[4], ls[4];
    f32x2 os[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = min(s0 + 4 * u, live - 1);
      const int64_t r = (prow0 + (int64_t)s * rep) * 16 + t;
      ms[u] = (s0 + 4 * u < live) ? p.part_ml[r * 2] : -INFINITY;
      ls[u] = p.part_ml[r * 2 + 1];
      os[u] = *reinterpret_cast<const f32x2*>(p.part_o + r * kHD + 2 * lane);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (ms[u] == -INFINITY) continue;  // no visible key in that split (wave-uniform)
      const float mn = fmaxf(m, ms[u]);
      const float ca = (m == -INFINITY) ? 0.f : __expf(m - mn);
      const float cb = __expf(ms[u] - mn);
      l = l * ca + ls[u] * cb;
      a0 = a0 * ca + os[u].x * cb;
      a1 = a1 * ca + os[u].y * cb;
      m = mn;
    }
  }
  if (lane == 0) {
    sm[wave] = m;
    sl[wave] = l;
  }
  so[wave][lane] = f32x2{a0, a1};
  __syncthreads();
  if (wave != 0) return;
  float mm = -INFINITY;
#pragma unroll
  for (int k = 0; k < 4; ++k) mm = fmaxf(mm, sm[k]);
  float lsum = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (sm[k] == -INFINITY) continue;
    const float c = __expf(sm[k] - mm);
    lsum = fmaf(sl[k], c, lsum);
    o0 = fmaf(so[k][lane].x, c, o0);
    o1 = fmaf(so[k][lane].y, c, o1);
  }
  const float inv = 1.f / lsum;
  const uint32_t gv = *reinterpret_cast<const uint32_t*>(
      p.gate_src + (int64_t)bt * p.gate_row_stride + qh * 2 * kHD + kHD + 2 * lane);
  const float g0 = 1.f / (1.f + __expf(-bf16_lo(gv)));
  const float g1 = 1.f / (1.f + __expf(-bf16_hi(gv)));
  *reinterpret_cast<uint32_t*>(p.out + ((int64_t)bt * p.Hq + qh) * kHD + 2 * lane) =
      pack2(o0 * inv * g0, o1 * inv * g1);
}

// ------------------------------------------------ attention over a prompt
// The same causal SDPA + gate for the P rows of a prompt pass (one sequence,
// cache length lens[0] before the prompt; prompt row i sees keys 0 ..
// lens[0] + i).  A workgroup owns RB blocks of 32 query rows of one KV head's REP
// query heads: two waves per head and block, which walk the keys 128 at a time,
// wave half hf the 64 keys from 64 hf of each turn; the halves merge through LDS
// at the end.  The turns' LDS lets a compute unit hold one workgroup, so it has
// eight waves, two a SIMD (one wave's softmax beside the other's products; six with
// REP = 3): RB = 4, 2, 1, 1 for REP = 1 to 4 (ap_row_blocks).
//   - Products on v_mfma_f32_32x32x16_bf16 in transposed form, S^T = K Q^T and
//     O^T = V^T P^T: a lane holds one query's column (32 of a tile's 64
//     scores, the other 32 in lane ^ 32), so a row's max is in-lane but for
//     one exchange, its sum and the rescale of O are in-lane altogether, and
//     P^T never leaves registers: result row 8 (i / 4) + 4 (lane / 32) + i % 4
//     is element i, so elements 8 s' .. 8 s' + 7 are the operand of keys
//     16 s' + 4 hl + {0..3, 8..11} (hl = lane / 32), and V^T's 16-byte LDS
//     pieces hold keys in that order.
//   - A turn's K (128 keys x 256 bytes) and V^T (2 x 128 features x 128 bytes)
//     are loaded once per workgroup, a turn ahead, into the other of two LDS
//     buffers: 16-byte piece c of row r at slot c ^ (r % 8).
//   - Running max m (in units of log2, the scale folded in), sum and O per
//     query; O is rescaled whenever some row's max grew, so that the heaviest
//     key's weight is 1 exactly.  With O left alone up to a growth of 2^8 that
//     weight is rounded to bf16 like the others: 5-8 % faster, but 3 % further
//     from 64 bits with flat scores and 24 % with peaked ones (queries of std 3 on
//     2560 keys 1.74e-3 -> 2.17e-3; the kernel before 1.77e-3).
// Row blocks are launched last first: later blocks see more keys and set the
// launch's end.
// What bounds it: per 64 keys and wave 1024 MFMA cycles against about as many
// of softmax arithmetic (32 exponentials at a quarter of the VALU rate), LDS
// reads 32 KB a wave.  Measured on MI355X (16 query heads, 4 KV heads; the kernel
// before, 16-row blocks on 16x16x32 MFMA with the softmax across lanes, after
// "against"): 4096 rows 94 us = 730 TFLOP/s against 252, 2048 rows 44 against 94,
// 600 rows 19 against 29, 120 rows 10.6 against 12.5, 60 and 256 rows after 14336
// keys 237 against 450 and 456.  Other groups, 2048 and 4096 rows: 3 heads (12:4) 49
// and 101 against 94 and 266, 2 (16:8) 44 and 97 against 104 and 291, 1 (8:8) 42 and
// 75 against 92 and 295, 1 (16:16) 47 and 150 against 162 and 467; 32 and 120 rows
// 7.2-10.5 and 10.6-11.2 against 10.0-10.7 and 12.1-12.6.  With one row block a
// workgroup groups of 1 and 2 had two and four waves on a compute unit: 16:16 173
// and 500, 16:8 53 and 177, after 14336 keys 303 and 277 for 234 and 238, but 120
// rows after none 9.2 for 11.1.  Also: rows stored from the lanes' columns cost 3 us
// a launch; all heads' blocks in one order 128 us at 4096 rows (a KV head's blocks
// now stay on 8 / Hkv XCDs, whose L2 then holds its keys).
struct AttnPrefillParams {
  const uint16_t* q;         // [P, Hq, D]
  const uint16_t* k_cache;   // [Hkv, Smax, D]
  const uint16_t* vt_cache;  // [Hkv, D, Smax]
  const int32_t* lens;       // [1]
  const uint16_t* gate_src;  // prompt row i's gate of head qh at i*gate_row_stride + qh*2D + D
  int64_t gate_row_stride;
  uint16_t* out;             // [P, Hq*D]
  int P, Hq, Hkv, Smax, nblk;
  float scale;
  int vec;   // gate and output rows hold whole 16-byte pieces
  int xcds;  // XCDs a KV head owns (0: heads in order)
};

constexpr int kAPRows = 32;              // query rows of a wave
constexpr int kAPKeys = 128;             // keys per turn, 64 per wave half
constexpr int kAPBuf = 2 * kAPKeys * kHD * 2;  // bytes of one turn's K and V^T
constexpr int kAPMerge = 66 * 64;        // floats of a wave's O, m and l
constexpr int kAPPitch = kHD + 4;        // floats of a normalized row in LDS (16 bytes of pad)

typedef float f32x16 __attribute__((ext_vector_type(16)));

// x of this lane and of lane ^ 32.
__device__ __forceinline__ f32x2 both_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return f32x2{__uint_as_float(r[0]), __uint_as_float(r[1])};
}

__device__ __forceinline__ u32x4 cvt8_bf16(const float* v) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2 * i], v[2 * i + 1]}, bf16x2));
  return u32x4{o[0], o[1], o[2], o[3]};
}

// The turns' two buffers, then (aliased) the merge and the normalized rows of a
// workgroup's pairs of head and row block.
constexpr int ap_lds_bytes(int pairs) {
  const int merge = 4 * pairs * (kAPMerge + kAPRows * kAPPitch);
  return merge > 2 * kAPBuf ? merge : 2 * kAPBuf;
}

template <int REP, int RB>
__global__ __launch_bounds__(128 * REP * RB, 2) void attn_prefill_kernel(const AttnPrefillParams p) {
  constexpr int PAIRS = REP * RB;  // of a query head and a block of 32 rows
  constexpr int NT = 128 * PAIRS;
  constexpr int PIECES = kAPKeys * kHD * 2 / 16;  // 16-byte pieces of K (and of V^T) a turn
  constexpr int PER = (PIECES + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) unsigned char lds[ap_lds_bytes(PAIRS)];
  const int xcd = blockIdx.x & 7;
  const int h = p.xcds ? xcd / p.xcds : (int)blockIdx.x / p.nblk;
  const int rank = p.xcds ? (int)(blockIdx.x >> 3) * p.xcds + xcd % p.xcds : (int)blockIdx.x % p.nblk;
  if (rank >= p.nblk) return;
  const int blk = p.nblk - 1 - rank;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r32 = lane & 31, hl = lane >> 5;
  const int hf = wave / PAIRS;  // key half of each turn
  const int pair = wave % PAIRS;
  const int qh = h * REP + (RB == 1 ? pair : pair % REP);
  const int base = min(max(p.lens[0], 0), p.Smax);
  const int t0 = blk * RB * kAPRows;          // the workgroup's first row
  const int tw = RB == 1 ? t0 : t0 + pair / REP * kAPRows;  // this wave's first row (past the last: it only loads)
  const int turns = (min(base + min(t0 + RB * kAPRows, p.P), p.Smax) + kAPKeys - 1) / kAPKeys;
  const int L = RB == 1 || tw < p.P ? min(base + min(tw + kAPRows, p.P), p.Smax) : 0;  // keys its last row sees
  const uint16_t* kbase = p.k_cache + (int64_t)h * p.Smax * kHD;
  const uint16_t* vbase = p.vt_cache + (int64_t)h * kHD * p.Smax;
  u32x4 kv[PER], vv[PER];
  // K piece e: key e / 16, piece e % 16; V^T piece e: feature e / 16, keys
  // 8 (e % 16) .. +7 (keys past the cache's last are clamped: never visible).
  auto load_turn = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = min(tid + NT * i, PIECES - 1);
      kv[i] = ld16(kbase + (int64_t)min(k0 + (e >> 4), p.Smax - 1) * kHD + (e & 15) * 8);
      vv[i] = ld16(vbase + (int64_t)(e >> 4) * p.Smax + min(k0 + (e & 15) * 8, p.Smax - 8));
    }
  };
  auto store_turn = [&](unsigned char* buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + NT * i;
      if (PIECES % NT != 0 && e >= PIECES) continue;
      const int key = e >> 4, c = e & 15;
      *reinterpret_cast<u32x4*>(buf + key * 256 + ((c ^ (key & 7)) << 4)) = kv[i];
      // half c / 8 of the turn, group (c % 8) / 2 of 16 keys; its first (second)
      // 8 keys are the first (second) 8 bytes of the pieces of hl = 0 and 1
      unsigned char* row = buf + kAPBuf / 2 + (c >> 3) * (kHD * 128) + key * 128 + (c & 1) * 8;
      const int slot = c & 6, sw = key & 7;  // (here `key` is the feature row)
      *reinterpret_cast<u32x2*>(row + ((slot ^ sw) << 4)) = u32x2{vv[i].x, vv[i].y};
      *reinterpret_cast<u32x2*>(row + (((slot + 1) ^ sw) << 4)) = u32x2{vv[i].z, vv[i].w};
    }
  };
  load_turn(0);
  const uint16_t* qr = p.q + ((int64_t)min(tw + r32, p.P - 1) * p.Hq + qh) * kHD + hl * 8;
  u32x4 qb[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) qb[k] = ld16(qr + 16 * k);
  // The loop takes maxima and masks before it scales, so its scale is positive:
  // the sign of a negative one goes to q, and with a zero one q is zero.
  if (!(p.scale > 0.f)) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      qb[k] = p.scale < 0.f ? qb[k] ^ 0x80008000u : p.scale == 0.f ? u32x4{0u, 0u, 0u, 0u} : qb[k];
  }
  store_turn(lds);
  if (turns > 1) load_turn(kAPKeys);
  float m = -INFINITY, l = 0.f;
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  const float sl = (p.scale == 0.f ? 1.f : fabsf(p.scale)) * 1.44269504088896340736f;
  const int last = min(base + tw + r32, L - 1);  // the last key this lane's row sees
  __syncthreads();
  for (int j = 0; j < turns; ++j) {
    const unsigned char* buf = lds + (j & 1) * kAPBuf;
    if (j + 1 < turns) {
      store_turn(lds + ((j + 1) & 1) * kAPBuf);
      if (j + 2 < turns) load_turn((j + 2) * kAPKeys);
    }
    const int k0 = j * kAPKeys + 64 * hf;
    if (k0 < L) {
      const unsigned char* sk = buf + 64 * hf * 256;
      const unsigned char* sv = buf + kAPBuf / 2 + hf * (kHD * 128);
      f32x16 st[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        st[kt] = f32x16{};
#pragma unroll
        for (int k = 0; k < 8; ++k)
          st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                             sk + (32 * kt + r32) * 256 + (((2 * k + hl) ^ (r32 & 7)) << 4))),
              __builtin_bit_cast(bf16x8, qb[k]), st[kt], 0, 0, 0);
      }
      if (k0 + 63 > base + tw) {  // some row does not see the whole tile
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * kt + 8 * (i >> 2) + 4 * hl + (i & 3);
            if (key > last) st[kt][i] = -INFINITY;
          }
      }
      float mx = st[0][0];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[kt][i]);
      const f32x2 mb = both_halves(mx);
      mx = fmaxf(mb.x, mb.y) * sl;
      if (__any(mx > m)) {
        const float mn = fmaxf(m, mx);
        const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
        m = mn;
      }
      const float ms = m == -INFINITY ? 0.f : m;
      u32x4 pb[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float pe[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          pe[i] = __builtin_amdgcn_exp2f(fmaf(st[s >> 1][8 * (s & 1) + i], sl, -ms));
          l += pe[i];
        }
        pb[s] = cvt8_bf16(pe);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                             sv + (32 * dt + r32) * 128 + (((2 * s + hl) ^ (r32 & 7)) << 4))),
              __builtin_bit_cast(bf16x8, pb[s]), o[dt], 0, 0, 0);
    }
    __syncthreads();
  }
  // The second key half's sums go to the first through LDS, which leaves the
  // normalized rows there; every wave then gates and stores whole rows (lanes
  // hold columns: stored from there, each piece would be a line of its own).
  float* red = reinterpret_cast<float*>(lds) + pair * kAPMerge + lane;
  float* rows = reinterpret_cast<float*>(lds) + PAIRS * kAPMerge;  // [PAIRS][32][kAPPitch]
  if (hf == 1) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) red[(16 * dt + i) * 64] = o[dt][i];
    red[64 * 64] = m;
    red[65 * 64] = l;
  }
  // this thread's pieces of 8 features: piece e is row (e / 16) % 32 of pair
  // e / 512, features 8 (e % 16) .. +7
  constexpr int OUT = PAIRS * kAPRows * 16 / NT;  // 4
  auto row_of = [&](int e) { return t0 + (RB == 1 ? 0 : (e >> 9) / REP * kAPRows) + ((e >> 4) & 31); };
  auto head_of = [&](int e) { return h * REP + (RB == 1 ? e >> 9 : (e >> 9) % REP); };
  u32x4 gt[OUT];
#pragma unroll
  for (int i = 0; i < OUT; ++i) {
    const int e = tid + NT * i;
    const uint16_t* gr = p.gate_src + (int64_t)min(row_of(e), p.P - 1) * p.gate_row_stride +
                         head_of(e) * 2 * kHD + kHD + (e & 15) * 8;
    if (p.vec) {
      gt[i] = ld16(gr);
    } else {
      uint32_t w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = (uint32_t)gr[2 * u] | ((uint32_t)gr[2 * u + 1] << 16);
      gt[i] = u32x4{w[0], w[1], w[2], w[3]};
    }
  }
  __syncthreads();
  if (hf == 0) {
    const float m1 = red[64 * 64], l1 = red[65 * 64];
    const float mn = fmaxf(m, m1);  // finite: key 0 is in the first half
    float c0 = __builtin_amdgcn_exp2f(m - mn), c1 = __builtin_amdgcn_exp2f(m1 - mn);
    const f32x2 lb = both_halves(l * c0 + l1 * c1);
    const float inv = 1.f / (lb.x + lb.y);
    c0 *= inv;
    c1 *= inv;
    float* row = rows + (pair * kAPRows + r32) * kAPPitch;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {  // features 32 dt + 8 i4 + 4 hl .. +3
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = o[dt][4 * i4 + e] * c0 + red[(16 * dt + 4 * i4 + e) * 64] * c1;
        *reinterpret_cast<f32x4*>(row + 32 * dt + 8 * i4 + 4 * hl) = v;
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < OUT; ++i) {
    const int e = tid + NT * i, t = row_of(e);
    if (t >= p.P) continue;
    const float* row = rows + (e >> 4) * kAPPitch + (e & 15) * 8;
    float g[8], v[8];
    unpack8(gt[i], g);
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = row[u] * (1.f / (1.f + __expf(-g[u])));
    uint16_t* orow = p.out + ((int64_t)t * p.Hq + head_of(e)) * kHD + (e & 15) * 8;
    if (p.vec) {
      *reinterpret_cast<u32x4*>(orow) = pack8(v);
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) orow[u] = f32_to_bf16_rne(v[u]);
    }
  }
}

// 32-row blocks of a workgroup: with 1 or 2 query heads a KV head as many as make
// eight waves, two a SIMD (kernel comment).
constexpr int ap_row_blocks(int rep) { return rep == 1 ? 4 : rep == 2 ? 2 : 1; }

template <int REP>
void launch_attn_prefill(const AttnPrefillParams& p, dim3 grid, hipStream_t s) {
  constexpr int RB = ap_row_blocks(REP);
  hipLaunchKernelGGL((attn_prefill_kernel<REP, RB>), grid, dim3(128 * REP * RB), 0, s, p);
}

// --------------------------------------------------------- commit an accept
// keep[b] = matched[b] + 1 (the block's first token plus the accepted drafts,
// runtime.py:146), lens[b] += keep[b] (the KV trim of adapters.py:505-508
// seen from the other side: the cache keeps lens + keep positions).
__global__ void commit_accept_kernel(const int32_t* matched, int32_t* keep, int32_t* lens, int B,
                                     int T) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const int k = min(max(matched[b], 0), T - 1) + 1;
  keep[b] = k;
  if (lens != nullptr) lens[b] += k;
}

}  // namespace
}  // namespace dflash

using namespace dflash;

namespace dflash {
namespace {
int launch_add_rmsnorm(const void* x, const int32_t* tok, int vocab, const void* r, const float* rp,
                       int nsplit, const void* weight, void* h_out, void* h_copy,
                       int64_t h_copy_stride, void* y, int M, int H, float eps, void* stream) {
  if (M < 0 || H <= 0 || H % 8 != 0 || H > 1024 * 8 || nsplit < 0) return DFLASH_ERR_SHAPE;
  if (h_copy != nullptr && h_copy_stride < H) return DFLASH_ERR_SHAPE;
  if (M == 0) return DFLASH_OK;
  if (x == nullptr || weight == nullptr || y == nullptr) return DFLASH_ERR_NULL;
  if (((uintptr_t)x & 15) || ((uintptr_t)r & 15) || ((uintptr_t)rp & 15) ||
      ((uintptr_t)weight & 15) || ((uintptr_t)h_out & 15) || ((uintptr_t)y & 15) ||
      ((uintptr_t)h_copy & 15) || (h_copy != nullptr && (h_copy_stride % 8)))
    return DFLASH_ERR_ALIGN;
  auto* hcp = static_cast<uint16_t*>(h_copy);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)M);
  const dim3 block((unsigned)ceil_div(H / 8, 64) * 64);
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* rpb = static_cast<const uint16_t*>(r);
  const auto* wp = static_cast<const uint16_t*>(weight);
  auto* hp = static_cast<uint16_t*>(h_out);
  auto* yp = static_cast<uint16_t*>(y);
  if (rp != nullptr) {
    switch (nsplit) {
#define DFLASH_ARN(ns)                                                                           \
  case ns:                                                                                       \
    hipLaunchKernelGGL((add_rmsnorm_kernel<true, ns>), grid, block, 0, s, xp, tok, vocab, nullptr, \
                       rp, nsplit, wp, hp, hcp, h_copy_stride, yp, M, H, eps);                   \
    break;
      DFLASH_ARN(1) DFLASH_ARN(2) DFLASH_ARN(3) DFLASH_ARN(4) DFLASH_ARN(5) DFLASH_ARN(6)
      DFLASH_ARN(7) DFLASH_ARN(8)
#undef DFLASH_ARN
      default:
        hipLaunchKernelGGL((add_rmsnorm_kernel<true, 0>), grid, block, 0, s, xp, tok, vocab, nullptr,
                           rp, nsplit, wp, hp, hcp, h_copy_stride, yp, M, H, eps);
    }
  } else {
    hipLaunchKernelGGL((add_rmsnorm_kernel<false, 0>), grid, block, 0, s, xp, tok, vocab, rpb,
                       nullptr, 0, wp, hp, hcp, h_copy_stride, yp, M, H, eps);
  }
  return to_status(hipGetLastError());
}
}  // namespace
}  // namespace dflash

extern "C" int dflash_add_rmsnorm(const void* x, const void* r, const void* weight, void* h_out,
                                  void* y, int M, int H, float eps, void* stream) {
  return launch_add_rmsnorm(x, nullptr, 0, r, nullptr, 0, weight, h_out, nullptr, 0, y, M, H, eps,
                            stream);
}

extern "C" int dflash_add_rmsnorm_splitk(const void* x, const float* r_partials, int nsplit,
                                         const void* weight, void* h_out, void* y, int M, int H,
                                         float eps, void* stream) {
  if (r_partials == nullptr || nsplit < 1) return DFLASH_ERR_NULL;
  return launch_add_rmsnorm(x, nullptr, 0, nullptr, r_partials, nsplit, weight, h_out, nullptr, 0,
                            y, M, H, eps, stream);
}

extern "C" int dflash_add_rmsnorm_capture(const void* x, const void* r, const float* r_partials,
                                          int nsplit, const void* weight, void* h_out,
                                          void* h_copy, int64_t h_copy_row_stride, void* y, int M,
                                          int H, float eps, void* stream) {
  if (r_partials != nullptr && (r != nullptr || nsplit < 1)) return DFLASH_ERR_SHAPE;
  if (h_copy == nullptr) return DFLASH_ERR_NULL;
  return launch_add_rmsnorm(x, nullptr, 0, r, r_partials, r_partials ? nsplit : 0, weight, h_out,
                            h_copy, h_copy_row_stride, y, M, H, eps, stream);
}

extern "C" int dflash_embed_rmsnorm(const void* table, const int32_t* tokens, int vocab,
                                    const void* weight, void* h_out, void* y, int M, int H,
                                    float eps, void* stream) {
  if (vocab <= 0) return DFLASH_ERR_SHAPE;
  if (tokens == nullptr || h_out == nullptr) return DFLASH_ERR_NULL;
  return launch_add_rmsnorm(table, tokens, vocab, nullptr, nullptr, 0, weight, h_out, nullptr, 0, y,
                            M, H, eps, stream);
}

extern "C" int dflash_swiglu(const void* gate_up, void* out, int M, int I, void* stream) {
  if (M < 0 || I <= 0 || I % 8 != 0) return DFLASH_ERR_SHAPE;
  if (M == 0) return DFLASH_OK;
  if (gate_up == nullptr || out == nullptr) return DFLASH_ERR_NULL;
  if (((uintptr_t)gate_up & 15) || ((uintptr_t)out & 15)) return DFLASH_ERR_ALIGN;
  const int64_t n = (int64_t)M * (I / 8);
  const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(n, 256), 2048);
  hipLaunchKernelGGL(swiglu_kernel, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(gate_up), static_cast<uint16_t*>(out), M, I);
  return to_status(hipGetLastError());
}

extern "C" int dflash_attn_prep(const void* proj, int64_t proj_row_stride, const void* q_norm_w,
                                const void* k_norm_w, const int32_t* lens, void* k_cache,
                                void* vt_cache, void* q_out, int32_t* overflow, int B, int T,
                                int Hq, int Hkv, int D, int Smax, int rot_dims, float rope_base,
                                float eps, void* stream) {
  if (B < 0 || T < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Smax <= 0) return DFLASH_ERR_SHAPE;
  if (D != kHD) return DFLASH_ERR_UNSUPPORTED;
  if (!(rot_dims == 0 || rot_dims == 16 || rot_dims == 32 || rot_dims == 64 || rot_dims == 128))
    return DFLASH_ERR_UNSUPPORTED;
  if (proj_row_stride < (int64_t)(2 * Hq + 2 * Hkv) * D) return DFLASH_ERR_SHAPE;
  if ((int64_t)B * T > INT32_MAX) return DFLASH_ERR_SHAPE;  // grid.x = B * T
  if (B == 0 || T == 0) return DFLASH_OK;
  if (proj == nullptr || q_norm_w == nullptr || k_norm_w == nullptr || lens == nullptr ||
      k_cache == nullptr || vt_cache == nullptr || q_out == nullptr)
    return DFLASH_ERR_NULL;
  if (((uintptr_t)proj & 3) || (proj_row_stride % 2) || ((uintptr_t)q_norm_w & 3) ||
      ((uintptr_t)k_norm_w & 3) || ((uintptr_t)k_cache & 3) || ((uintptr_t)q_out & 3))
    return DFLASH_ERR_ALIGN;
  AttnPrepParams p{};
  p.proj = static_cast<const uint16_t*>(proj);
  p.row_stride = proj_row_stride;
  p.q_norm_w = static_cast<const uint16_t*>(q_norm_w);
  p.k_norm_w = static_cast<const uint16_t*>(k_norm_w);
  p.lens = lens;
  p.k_cache = static_cast<uint16_t*>(k_cache);
  p.vt_cache = static_cast<uint16_t*>(vt_cache);
  p.q_out = static_cast<uint16_t*>(q_out);
  p.overflow = overflow;
  p.B = B; p.T = T; p.Hq = Hq; p.Hkv = Hkv; p.Smax = Smax; p.rot = rot_dims;
  p.log2_base = log2((double)rope_base);
  p.eps = eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Long inputs with 16-byte aligned value rows: the value heads through
  // attn_prep_vt_kernel's tiles instead of a wave a token.
  p.skip_v = T >= kVtTile && ((uintptr_t)proj & 15) == 0 && proj_row_stride % 8 == 0;
  const int slots = p.skip_v ? Hq + Hkv : Hq + 2 * Hkv;
  // Heads a wave: as many as leave 16 waves a compute unit.  Below two (under
  // 410 tokens of 20 heads) a wave a head is as fast: 256 tokens 8.6 us, and the
  // fewer the tokens, the more the walk along the heads would be all there is.
  p.heads = (int)std::min<int64_t>((int64_t)B * T * slots / (16 * std::max(device_cus(), 1)), slots);
  if (p.skip_v && p.heads > 1) {
    p.groups = (int)ceil_div(slots, p.heads);
    const dim3 rgrid((unsigned)ceil_div((int64_t)B * T * p.groups, 4));
    hipLaunchKernelGGL(attn_prep_rows_kernel, rgrid, dim3(256), 0, s, p);
  } else {
    const dim3 grid((unsigned)(B * T), (unsigned)ceil_div(slots, 4));
    hipLaunchKernelGGL(attn_prep_kernel, grid, dim3(256), 0, s, p);
  }
  if (p.skip_v) {
    const dim3 vgrid((unsigned)ceil_div(T, kVtTile), (unsigned)Hkv, (unsigned)B);
    hipLaunchKernelGGL(attn_prep_vt_kernel, vgrid, dim3(256), 0, s, p);
  }
  return to_status(hipGetLastError());
}

extern "C" size_t dflash_attn_verify_workspace_bytes(int B, int Hq, int Hkv, int max_len) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || max_len <= 0) return 0;
  const int64_t nsplit = ceil_div(max_len, KC);
  const int64_t rows = (int64_t)B * Hq * nsplit * 16;  // Hkv * rep = Hq
  return (size_t)(rows * (kHD + 2) * sizeof(float));
}

extern "C" int dflash_attn_verify(const void* q, const void* k_cache, const void* vt_cache,
                                  const int32_t* lens, const void* gate_src,
                                  int64_t gate_row_stride, void* out, int B, int T, int Hq,
                                  int Hkv, int D, int Smax, int max_len, float scale,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  if (B < 0 || T < 0 || T > 16 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Hq / Hkv > 4)
    return DFLASH_ERR_SHAPE;
  if (D != kHD) return DFLASH_ERR_UNSUPPORTED;
  if (Smax <= 0 || Smax % KC != 0 || max_len <= 0 || max_len > Smax) return DFLASH_ERR_SHAPE;
  if (B > 65535) return DFLASH_ERR_SHAPE;  // grid.z of the partials = B
  if (B == 0 || T == 0) return DFLASH_OK;
  if (q == nullptr || k_cache == nullptr || vt_cache == nullptr || lens == nullptr ||
      gate_src == nullptr || out == nullptr || workspace == nullptr)
    return DFLASH_ERR_NULL;
  if (workspace_bytes < dflash_attn_verify_workspace_bytes(B, Hq, Hkv, max_len))
    return DFLASH_ERR_WORKSPACE;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)vt_cache & 15) ||
      ((uintptr_t)gate_src & 3) || (gate_row_stride % 2) || ((uintptr_t)out & 3) ||
      ((uintptr_t)workspace & 15))
    return DFLASH_ERR_ALIGN;
  AttnParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k_cache = static_cast<const uint16_t*>(k_cache);
  p.vt_cache = static_cast<const uint16_t*>(vt_cache);
  p.lens = lens;
  p.gate_src = static_cast<const uint16_t*>(gate_src);
  p.gate_row_stride = gate_row_stride;
  p.out = static_cast<uint16_t*>(out);
  p.B = B; p.T = T; p.Hq = Hq; p.Hkv = Hkv; p.Smax = Smax;
  p.nsplit = (int)ceil_div(max_len, KC);
  p.scale = scale;
  const int64_t rows = (int64_t)B * Hq * p.nsplit * 16;
  p.part_o = static_cast<float*>(workspace);
  p.part_ml = p.part_o + rows * kHD;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rep = Hq / Hkv;
  const dim3 pgrid(p.nsplit, Hkv, B);
  switch (rep) {
    case 1: hipLaunchKernelGGL(attn_partial_kernel<1>, pgrid, dim3(64), 0, s, p); break;
    case 2: hipLaunchKernelGGL(attn_partial_kernel<2>, pgrid, dim3(128), 0, s, p); break;
    case 3: hipLaunchKernelGGL(attn_partial_kernel<3>, pgrid, dim3(192), 0, s, p); break;
    default: hipLaunchKernelGGL(attn_partial_kernel<4>, pgrid, dim3(256), 0, s, p); break;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(attn_combine_kernel, dim3(B * T, Hq), dim3(256), 0, s, p);
  return to_status(hipGetLastError());
}

extern "C" int dflash_attn_prefill(const void* q, const void* k_cache, const void* vt_cache,
                                   const int32_t* lens, const void* gate_src,
                                   int64_t gate_row_stride, void* out, int P, int Hq, int Hkv,
                                   int D, int Smax, float scale, void* stream) {
  if (P < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || Hq / Hkv > 4) return DFLASH_ERR_SHAPE;
  if (D != kHD) return DFLASH_ERR_UNSUPPORTED;
  if (Smax <= 0 || Smax % KC != 0 || Hkv > 65535) return DFLASH_ERR_SHAPE;
  if (gate_row_stride < (int64_t)2 * Hq * D) return DFLASH_ERR_SHAPE;
  if (P == 0) return DFLASH_OK;
  if (q == nullptr || k_cache == nullptr || vt_cache == nullptr || lens == nullptr ||
      gate_src == nullptr || out == nullptr)
    return DFLASH_ERR_NULL;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)vt_cache & 15) ||
      ((uintptr_t)gate_src & 1) || ((uintptr_t)out & 1))
    return DFLASH_ERR_ALIGN;
  AttnPrefillParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k_cache = static_cast<const uint16_t*>(k_cache);
  p.vt_cache = static_cast<const uint16_t*>(vt_cache);
  p.lens = lens;
  p.gate_src = static_cast<const uint16_t*>(gate_src);
  p.gate_row_stride = gate_row_stride;
  p.out = static_cast<uint16_t*>(out);
  p.P = P; p.Hq = Hq; p.Hkv = Hkv; p.Smax = Smax;
  p.nblk = (int)ceil_div(P, kAPRows * ap_row_blocks(Hq / Hkv));
  p.scale = scale;
  p.vec = !((uintptr_t)gate_src & 15) && gate_row_stride % 8 == 0 && !((uintptr_t)out & 15);
  hipStream_t s = static_cast<hipStream_t>(stream);
  p.xcds = 8 % Hkv == 0 ? 8 / Hkv : 0;
  const dim3 grid((unsigned)(p.xcds ? 8 * ceil_div(p.nblk, p.xcds) : (int64_t)p.nblk * Hkv));
  switch (Hq / Hkv) {
    case 1: launch_attn_prefill<1>(p, grid, s); break;
    case 2: launch_attn_prefill<2>(p, grid, s); break;
    case 3: launch_attn_prefill<3>(p, grid, s); break;
    default: launch_attn_prefill<4>(p, grid, s); break;
  }
  return to_status(hipGetLastError());
}

extern "C" int dflash_commit_accept(const int32_t* matched, int32_t* keep, int32_t* lens, int B,
                                    int T, void* stream) {
  if (B < 0 || T <= 0) return DFLASH_ERR_SHAPE;
  if (B == 0) return DFLASH_OK;
  if (matched == nullptr || keep == nullptr) return DFLASH_ERR_NULL;
  hipLaunchKernelGGL(commit_accept_kernel, dim3((unsigned)ceil_div(B, 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), matched, keep, lens, B, T);
  return to_status(hipGetLastError());
}
