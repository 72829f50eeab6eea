// Block GEMMs: out[M, N] = x[M, K] . W[N, K]^T with 1 <= M <= 128 rows (built for
// more than 16; the prompt pass sends its last rows here, however few): the verify projections of two to four sequences' draft blocks and the prompt
// projections of a short prompt (dflash_mlx/custom_qwen35_model.py:726-736 and
// the Linear layers of mlx-lm's Qwen3NextAttention / Qwen3NextMLP).
//
// Between the two other families: the verify GEMMs (M = 16) stream the weight
// past activations that cost little, the prompt GEMMs (M in the hundreds)
// re-use a staged weight tile.  Here the weight is still streamed once, but
// every workgroup reads all M activation rows, as many bytes as its weights,
// so what counts is bytes per compute unit (about 50 GB/s each whatever the
// pattern) and keeping the loads of both apart from the products:
//   - a workgroup (4 waves) owns VT row tiles of the weight for all M rows, so
//     the activations are read N / (16 VT) times; each wave takes a contiguous
//     quarter of the k-range (no wave waits for another until the end) and
//     holds all VT x MT sums;
//   - activations arrive as whole 128-byte lines and are transposed through
//     the wave's own swizzled LDS rows (a fragment read straight from memory
//     touches 16 rows of half lines, twice);
//   - the quarters are added through LDS in k order, each wave finishing the
//     column tiles mt % 4 == wave.
// With the quarters and their order those of the verify GEMM's four k-waves,
// the sums are that kernel's bit for bit.
//
// Measured on MI355X (cold weights, us; the kernels that ran before, with their
// split-K reduce, after "against") at M = 32 / 64 / 128: gate|up (N 18432, K
// 2560) 18.6 / 22.2 / 29.5 against 23.9 / 33.4 / 36.6; in_proj (12352 x 2560)
// 14.3 / 17.3 / 23.7 against 15.8 / 21.6 / 33.5; q|k|v (5120 x 2560) 9.6 / 12.4
// / 17.9 against 10.8 / 16.2 / 25.9; down (2560 x 9216, 6 splits) 10.6 / 12.4 /
// 16.7 against 11.5 / 15.0 / 20.6; out_proj (2560 x 4096) 6.6 / 7.8 / 10.7
// against 7.6 / 10.5 / 18.2; o_proj (2560 x 2048) 5.1 / 6.2 / 8.7 against 6.6 /
// 9.0 / 17.1.  Of that, wave_sync (block_gemm.h): gate|up at 96 / 128 rows 27.9 /
// 32.3 without it, 26.2 / 29.5 with it, q|k|v 15.4 / 18.8 -> 15.1 / 17.9; at 64
// rows gate|up 21.9 -> 22.2, elsewhere within 0.2 us.  At M = 16 the verify kernel
// is as fast or faster (gate|up 18.1 against 18.6).  With timing copies (before
// wave_sync) at gate|up, M = 64: the weight stream alone
// 19.1, everything but the weight loads 14.4; at M = 128: no activation loads
// 27.0, no weight loads 22.9.  Tried: ring depth 3 (the same or slower), two
// LDS halves with the next step's rows stored between the products (24.7
// against 24.0 at in_proj, M = 128), the rows split over two waves of 4 column
// tiles each, the weight read twice (23.3 at in_proj, 44 at gate|up).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "block_gemm.h"
#include "dflash_gdn.h"
#include "device_common.h"
#include "host_common.h"

namespace dflash {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct BlockParams {
  const uint16_t* x;  // [M][xs]
  int64_t xs;
  const uint16_t* w;  // fragment-tiled [K/64][N/16][2][64][8]
  uint16_t* out;      // [M][os]
  int64_t os;
  float* part;  // split-K partial sums [nsplit][M][N], else null
  int M, N, K, ks_per_split, swiglu;
};

__device__ __forceinline__ u32x2 pack4(f32x4 v) {
  return u32x2{(uint32_t)f32_to_bf16_rne(v.x) | ((uint32_t)f32_to_bf16_rne(v.y) << 16),
               (uint32_t)f32_to_bf16_rne(v.z) | ((uint32_t)f32_to_bf16_rne(v.w) << 16)};
}

// Two waves a SIMD while the sums and the ring fit 256 registers, else one.
template <int MT, int VT>
constexpr int block_occupancy() { return MT * VT <= 16 ? 2 : 1; }

template <int MT, int VT, int DX>
__global__ __launch_bounds__(kBlockThreads, (block_occupancy<MT, VT>())) void block_gemm_kernel(const BlockParams p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[block_lds_bytes<MT>()];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int rt0 = blockIdx.x * VT;
  const int split = blockIdx.y;
  const int split_begin = split * p.ks_per_split;
  const int split_len = min(p.ks_per_split, (p.K >> 6) - split_begin);
  const int part_len = (split_len + kBlockWaves - 1) / kBlockWaves;
  const int ks_begin = split_begin + min(wave * part_len, split_len);
  const int nks = min(part_len, split_begin + split_len - ks_begin);

  f32x4 acc[VT][MT];
  const BlockRows<MT> rows(p.x, p.xs, p.M, ks_begin, lds + wave * MT * 2048, lane);
  const BlockWeight<VT> w(p.w, p.N >> 4, rt0, ks_begin, lane);
  block_accumulate<MT, VT, 2, DX>(rows, w, nks, acc);

  f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int v0 = 0; v0 < VT; v0 += 2)
    block_merge<MT, VT>(red, acc, wave, lane, v0, [&](int mt, const f32x4 (&s)[2]) {
      const int m = mt * 16 + r16;
      const int n = (rt0 + v0) * 16 + 4 * g;
      if (m >= p.M) return;
      if (p.swiglu) {  // tile v0 the gate rows, v0 + 1 the matching up rows (N % 32 == 0)
        if (n >= p.N) return;
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = s[0][e] / (1.f + __expf(-s[0][e])) * s[1][e];
        *reinterpret_cast<u32x2*>(p.out + (int64_t)m * p.os + (rt0 + v0) * 8 + 4 * g) = pack4(o);
        return;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (n + 16 * j >= p.N) continue;
        if (p.part != nullptr)
          *reinterpret_cast<f32x4*>(p.part + ((int64_t)split * p.M + m) * p.N + n + 16 * j) = s[j];
        else
          *reinterpret_cast<u32x2*>(p.out + (int64_t)m * p.os + n + 16 * j) = pack4(s[j]);
      }
    });
}

// Activation k-steps in flight.  Up to 64 rows two fit the registers beside the
// weight's, and above that with 4 row tiles (one wave a SIMD either way): worth it
// in long walks, in_proj (10 k-steps a wave) 21.1 -> 20.6 us at 96 rows and 23.85 ->
// 23.73 at 128; in down (6) they cost as much, 16.7 -> 17.0 and 14.6 -> 14.7, and
// with 2 or 3 (o_proj, out_proj) the longer start shows, 8.7 -> 9.1 and 10.7 ->
// 11.3.  With 6 row tiles all registers would be taken, with 2 some spill.
constexpr int kBlockDeepSteps = 8;

template <int MT, int VT>
void launch_mt(const BlockParams& p, dim3 grid, hipStream_t s) {
  const dim3 block(kBlockThreads);
  if constexpr (MT <= 4) {
    hipLaunchKernelGGL((block_gemm_kernel<MT, VT, 2>), grid, block, 0, s, p);
  } else {
    if constexpr (VT == 4) {
      if (ceil_div(std::min(p.ks_per_split, p.K >> 6), kBlockWaves) >= kBlockDeepSteps) {
        hipLaunchKernelGGL((block_gemm_kernel<MT, VT, 2>), grid, block, 0, s, p);
        return;
      }
    }
    hipLaunchKernelGGL((block_gemm_kernel<MT, VT, 1>), grid, block, 0, s, p);
  }
}

template <int VT>
hipError_t launch_vt(const BlockParams& p, int nsplit, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(p.N, 16 * VT), (unsigned)nsplit);
  switch ((int)ceil_div(p.M, 16)) {
    case 1:
    case 2: launch_mt<2, VT>(p, grid, s); break;
    case 3: launch_mt<3, VT>(p, grid, s); break;
    case 4: launch_mt<4, VT>(p, grid, s); break;
    case 5:
    case 6: launch_mt<6, VT>(p, grid, s); break;
    default: launch_mt<8, VT>(p, grid, s); break;
  }
  return hipGetLastError();
}

}  // namespace

// Row tiles a workgroup (2, 4 or 6): the choice whose busiest compute unit
// reads the fewest bytes, (16 VT weight rows + M activation rows) times whole
// rounds of the units, the larger on a tie.  Measured at 64 rows: gate|up
// (N 18432) 22.0 us with 6 (192 units, one round), 28.4 with 4 (288, two
// rounds), 28.7 with 2; in_proj (12352) 16.7 with 4 (193 units), 20.4 with 6,
// 19.7 with 2; q|k|v (5120) 12.2 with 2 (160 units), 15.9 with 4 (80).
hipError_t launch_block_gemm(const uint16_t* x, int64_t xs, const uint16_t* w_tiled, uint16_t* out,
                             int64_t os, float* part, int M, int N, int K, int nsplit,
                             int ks_per_split, bool swiglu, hipStream_t s) {
  BlockParams p{};
  p.x = x; p.xs = xs; p.w = w_tiled; p.out = out; p.os = os; p.part = part;
  p.M = M; p.N = N; p.K = K; p.ks_per_split = ks_per_split; p.swiglu = swiglu;
  const int64_t cus = std::max(device_cus(), 1);
  auto cost = [&](int vt) { return (16 * vt + M) * ceil_div(ceil_div(N, 16 * vt) * nsplit, cus); };
  const int64_t c2 = cost(2), c4 = cost(4), c6 = cost(6);
  return c6 <= c4 && c6 <= c2 ? launch_vt<6>(p, nsplit, s)
         : c4 <= c2           ? launch_vt<4>(p, nsplit, s)
                              : launch_vt<2>(p, nsplit, s);
}

}  // namespace dflash

using namespace dflash;

// Internal to this package (its prompt pass); not part of the C interface.
// out [M, N] (swiglu: [M, N / 2]) when nsplit == 0, else fp32 partial sums
// [dflash_gemm_splits(K, nsplit)][M][N] into partials.  M <= 128.
extern "C" int dflash_gemm_bf16_tiled_block(const void* x, int64_t x_row_stride, const void* w_tiled,
                                            void* out, int64_t out_row_stride, float* partials,
                                            int nsplit, int M, int N, int K, int swiglu,
                                            void* stream) {
  if (M < 0 || M > 128 || N <= 0 || N % (swiglu ? 32 : 16) != 0 || N > kBlockMaxN || K <= 0 ||
      K % 64 != 0 || nsplit < 0 || (swiglu && nsplit > 0))
    return DFLASH_ERR_SHAPE;
  if (x_row_stride < K || x_row_stride > kBlockMaxRowStride) return DFLASH_ERR_SHAPE;
  if (nsplit == 0 && out_row_stride < (swiglu ? N / 2 : N)) return DFLASH_ERR_SHAPE;
  if (M == 0) return DFLASH_OK;
  if (x == nullptr || w_tiled == nullptr || (nsplit == 0 ? out == nullptr : partials == nullptr))
    return DFLASH_ERR_NULL;
  if (((uintptr_t)x & 15) || (x_row_stride % 8) || ((uintptr_t)w_tiled & 15)) return DFLASH_ERR_ALIGN;
  if (nsplit == 0 ? (((uintptr_t)out & 7) || (out_row_stride % 4)) : ((uintptr_t)partials & 15))
    return DFLASH_ERR_ALIGN;
  const int nks = K / 64;
  const int per = (int)ceil_div(nks, nsplit > 0 ? std::min(nsplit, nks) : 1);
  return to_status(launch_block_gemm(static_cast<const uint16_t*>(x), x_row_stride,
                                     static_cast<const uint16_t*>(w_tiled),
                                     static_cast<uint16_t*>(out), out_row_stride,
                                     nsplit > 0 ? partials : nullptr, M, N, K,
                                     (int)ceil_div(nks, per), per, swiglu != 0,
                                     static_cast<hipStream_t>(stream)));
}
