// The k-loop of the block-sized products out[M, N] = x[M, K] . W[N, K]^T with
// 1 <= M <= 128 over a fragment-tiled weight, shared by the block GEMMs
// (block_gemm.hip) and the LM-head argmax (lm_head_argmax.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace dflash {

typedef __bf16 block_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kBlockWaves = 4;  // k-quarters (waves) of a workgroup
constexpr int kBlockThreads = 64 * kBlockWaves;
// Activation rows further apart than this leave the 32-bit offsets within a
// group of 8 rows (7 * 2 bytes * stride < 2^32).
constexpr int64_t kBlockMaxRowStride = (int64_t)1 << 28;
// Weight rows up to which a row tile's 2 KB fragments stay in 32-bit offsets.
constexpr int kBlockMaxN = 1 << 24;

// LDS bytes of a workgroup: each wave's k-step of MT x 16 activation rows,
// then (aliased) the merge of two row tiles.
template <int MT>
constexpr int block_lds_bytes() { return kBlockWaves * MT * 2048; }

// Orders this wave's LDS operations before and after it for the compiler, which
// could otherwise take one lane's stores and reads for independent ones; global
// loads may still move across.  No instruction of its own.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// A wave's activation rows, 16 MT of them (rows past M read row M - 1; their
// sums are never stored), k-steps counted from ks_begin.  A k-step is loaded as
// whole 128-byte lines (load i takes rows 8i .. 8i+7, 8 lanes a row) and goes
// through the wave's own LDS rows `tile`, 16-byte piece c of row r at slot
// c ^ (r % 8), so that the 8 rows a fragment read touches at once fall in
// different bank groups.  No workgroup barrier: the rows are the wave's own and its
// LDS operations complete in order; wave_sync keeps them in that order in the
// compiled code, between one lane's store and another's read.
template <int MT>
struct BlockRows {
  const char* base[2 * MT];
  uint32_t off[2 * MT];
  unsigned char* wslot;
  const unsigned char *rslot0, *rslot1;

  __device__ __forceinline__ BlockRows(const uint16_t* x, int64_t xs, int M, int ks_begin,
                                       unsigned char* tile, int lane) {
    const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
      const int first = min(8 * i, M - 1);
      base[i] = reinterpret_cast<const char*>(x + (int64_t)first * xs) + (int64_t)ks_begin * 128;
      off[i] = (uint32_t)(min(8 * i + (lane >> 3), M - 1) - first) * (uint32_t)(xs * 2) + (lane & 7) * 16;
    }
    wslot = tile + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    rslot0 = tile + r16 * 128 + (((2 * g) ^ (r16 & 7)) << 4);
    rslot1 = tile + r16 * 128 + (((2 * g + 1) ^ (r16 & 7)) << 4);
  }
  __device__ __forceinline__ void load(u32x4 (&xr)[2 * MT], int ks) const {
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) xr[i] = *reinterpret_cast<const u32x4*>(base[i] + ks * 128 + off[i]);
  }
  __device__ __forceinline__ void store(const u32x4 (&xr)[2 * MT]) const {
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) *reinterpret_cast<u32x4*>(wslot + i * 1024) = xr[i];
    wave_sync();  // before any lane reads them
  }
  // acc += the stored k-step against weight fragments a (tile, half).
  template <int VT>
  __device__ __forceinline__ void mma(const u32x4 (&a)[2 * VT], f32x4 (&acc)[VT][MT]) const {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const u32x4 b0 = *reinterpret_cast<const u32x4*>(rslot0 + mt * 2048);
      const u32x4 b1 = *reinterpret_cast<const u32x4*>(rslot1 + mt * 2048);
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        acc[vt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(block_bf16x8, a[2 * vt]), __builtin_bit_cast(block_bf16x8, b0),
            acc[vt][mt], 0, 0, 0);
        acc[vt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(block_bf16x8, a[2 * vt + 1]), __builtin_bit_cast(block_bf16x8, b1),
            acc[vt][mt], 0, 0, 0);
      }
    }
    wave_sync();  // every lane has read them before the next store
  }
};

// VT row tiles of a tiled weight of NT tiles, from tile rt0 (clamped to the
// last; such sums are never stored), k-steps counted from ks_begin: fragment
// (k-step, tile, half) is 1 KB at ((ks * NT + rt) * 2 + h) KB, straight into
// registers (nontemporal: read once).
template <int VT>
struct BlockWeight {
  const char* base;
  int64_t stride;
  uint32_t off[VT];

  __device__ __forceinline__ BlockWeight(const uint16_t* w, int NT, int rt0, int ks_begin, int lane)
      : base(reinterpret_cast<const char*>(w) + (int64_t)ks_begin * NT * 2048), stride((int64_t)NT * 2048) {
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) off[vt] = (uint32_t)min(rt0 + vt, NT - 1) * 2048 + lane * 16;
  }
  __device__ __forceinline__ void load(u32x4 (&r)[2 * VT], int ks) const {
    const char* b = base + ks * stride;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const u32x4* src = reinterpret_cast<const u32x4*>(b + off[vt]);
      r[2 * vt] = __builtin_nontemporal_load(src);
      r[2 * vt + 1] = __builtin_nontemporal_load(src + 64);
    }
  }
};

// This wave's sums over its nks k-steps: acc[vt][mt] is row tile vt against
// activation rows 16 mt .. +15; lane (r16, g) of it holds out[m = 16 mt + r16]
// [n = 16 (rt0 + vt) + 4g .. +3].  The weight runs D k-steps ahead, the
// activations DX (1 or D; loads complete in order, so with DX = 1 a wait for
// the activations is one for the weight loads issued before them).  Full turns
// of the weight ring issue every load without a condition (so the compiler's
// count of loads in flight is exact at each wait); the last turns only what is
// left.
template <int MT, int VT, int D, int DX>
__device__ __forceinline__ void block_accumulate(const BlockRows<MT>& rows, const BlockWeight<VT>& w,
                                                 int nks, f32x4 (&acc)[VT][MT]) {
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[vt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (nks <= 0) return;
  static_assert(DX == 1 || DX == D, "activation ring");
  u32x4 wr[D][2 * VT], xr[DX][2 * MT];
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < nks) {
      if (d < DX) rows.load(xr[d], d);
      w.load(wr[d], d);
    }
  int ks0 = 0;
  for (; ks0 + 2 * D <= nks; ks0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      rows.store(xr[d % DX]);
      rows.load(xr[d % DX], ks0 + d + DX);
      rows.template mma<VT>(wr[d], acc);
      w.load(wr[d], ks0 + d + D);
    }
  }
  for (; ks0 < nks; ks0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int ks = ks0 + d;
      if (ks < nks) {
        rows.store(xr[d % DX]);
        if (ks + DX < nks) rows.load(xr[d % DX], ks + DX);
        rows.template mma<VT>(wr[d], acc);
        if (ks + D < nks) w.load(wr[d], ks + D);
      }
    }
  }
}

// Sums of row tiles v0 and v0 + 1 (below VT) over the four k-quarters, in
// quarter order, handed to take(mt, s) by the wave that owns column tile mt
// (mt % 4 == wave).  `red` is the workgroup's LDS.  Every wave calls it.
template <int MT, int VT, class Take>
__device__ __forceinline__ void block_merge(f32x4* red, const f32x4 (&acc)[VT][MT], int wave,
                                            int lane, int v0, Take take) {
  __syncthreads();
#pragma unroll
  for (int v = 0; v < VT; ++v)
    if (v == v0 || v == v0 + 1) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        red[((wave * 2 + (v - v0)) * MT + mt) * 64 + lane] = acc[v][mt];
    }
  __syncthreads();
  for (int mt = wave; mt < MT; mt += kBlockWaves) {
    f32x4 s[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      s[j] = red[(j * MT + mt) * 64 + lane];
#pragma unroll
      for (int q = 1; q < kBlockWaves; ++q) s[j] += red[((q * 2 + j) * MT + mt) * 64 + lane];
    }
    take(mt, s);
  }
}

// out[M, N] for 1 <= M <= 128 (block_gemm.hip; a verify step's projections use
// it from 17 rows on, a prompt pass for its last rows, however few): bf16 (out, row stride os), the
// gated form over paired rows (swiglu), or fp32 partial sums of nsplit k-ranges
// of ks_per_split k-steps each into part [nsplit][M][N] (part != null).
hipError_t launch_block_gemm(const uint16_t* x, int64_t xs, const uint16_t* w_tiled, uint16_t* out,
                             int64_t os, float* part, int M, int N, int K, int nsplit,
                             int ks_per_split, bool swiglu, hipStream_t s);

}  // namespace dflash
