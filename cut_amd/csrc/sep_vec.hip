// One or two rows of A on the separated layout (compat.hip says what it is): C[m,n] = sum_k A[m,k] * w[k,n], fp32.
//
// What bounds it: HBM and the start-up on large matrices, launches on small ones.  The layout is column-major in n, so the parallelism
// of a product with one row comes from K.  A workgroup owns a strip of columns and one of a few K ranges; its waves take the range's blocks of
// 32 k-rows in turn, two of them in flight in each, and meet in LDS at the end:
//   * strips of a whole cache line of the weights (128 int8 columns, 256 of nibbles) where there are enough of them: half lines arrive
//     at a lower rate (14336 x 4096 int8 as 224 workgroups, us: strips of 128 15.8, of 64 19.4, of 32 27, of 16 42);
//   * as many ranges as fill the 256 CUs once, and at most 16, so that the partial sums that meet in memory are 2 to 16 sets and not one for
//     every 128 k-rows (16 columns a lane and one block a wave: 32 sets for K = 4096, 112 for 14336); few columns over a long K then run on
//     16 workgroups for each strip (128 x 14336 7.5, 512 x 14336 8.7, 1024 x 14336 9.5, that form 13.4, 9.3, 10.6);
//   * a short K in one range: strips of 64 columns and sixteen waves, and no second launch;
//   * the activations come straight from the caches with the block they belong to: no staging, no barrier ahead of the weights.
// Against that form, both launches, us, graph replay over 600 MB of weights: int8 one row 14336 x 4096 (N x K) 16.4 -> 15.8, 4096 x 14336
// 18.2 -> 15.6 (4.0 TB/s), 4096 x 4096 9.9 -> 7.9, 1024 x 4096 7.8 -> 5.7, 4096 x 1024 7.8 -> 4.2, 28672 x 4096 28.2 -> 25.6; two rows
// 4096 x 14336 20.0 -> 16.5, 4096 x 4096 11.6 -> 8.1; nibbles with minima 4096 x 14336 14.6 -> 12.3, 4096 x 4096 9.2 -> 7.1.
// Columns in a multiple of eight that is none of 16 took the byte-wise form: 1000 x 2560 51 -> 5.8.  On weights that were written just
// before, the launches of the seven matmuls of such a layer take 102 -> 92 together, with all caches flushed 137 -> 121.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "sep_rows.hpp"

namespace cuthip {

struct SepVecRest {
  float *C;          // the output, or the sums of the K ranges [nsplit][MT][N]
  Epilogue epi;
  uint32_t strideC;
};

// MT rows of A; LC lanes of 8 columns to a k-row, so that a workgroup owns 8 LC columns and a wave's load takes 64 / LC k-rows;
// W waves share the blocks of 32 k-rows, D of them in flight in each.
template <bool Q4, bool AFF, int MT, int LC, int W, int D>
__global__ void __launch_bounds__(64 * W) sep_vec_kernel(const float *A, const uint8_t *B, const uint16_t *S, uint32_t N, uint32_t blocks,
                                                         uint32_t per, uint32_t strideA, uint32_t strideB, uint32_t scaleStride,
                                                         uint32_t tiles, uint32_t pieces, SepVecRest p) {
  constexpr uint32_t TC = 8 * LC;
  constexpr int RPL = LC / 2;   // k-rows of a block in one lane
  static_assert(LC == 8 || LC == 16 || LC == 32, "whole 16-byte pieces of A, eight columns halved up to three times");
  __shared__ float red[W][MT][TC];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // ids id, id + 8, ... share an XCD and take neighbouring column tiles of one range: a cache line that two tiles share is fetched once
  const uint32_t piece = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (piece >= pieces) return;
  const uint32_t split = __builtin_amdgcn_readfirstlane(piece / tiles), tile = piece - split * tiles;
  const uint32_t sub = lane / LC, c0 = tile * TC + 8 * (lane % LC), cb = min(c0, N - 8);
  const uint32_t b0 = split * per, b1 = min(b0 + per, blocks), iters = (b1 - b0 + W - 1) / W;

  struct Slot {
    u32x2 q[Q4 ? (RPL + 1) / 2 : RPL];   // Q4: a dword a row
    u32x4 s, m;
    float x[MT][RPL];
  } slot[D];
  const uint32_t woff = sub * RPL * strideB + (Q4 ? cb / 2 : cb);
  auto fetch = [&](Slot &t, uint32_t i) __attribute__((always_inline)) {
    const uint32_t b = min(b0 + wave + W * i, b1 - 1);
    const float *x = A + (size_t)b * 32;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float *xr = x + (size_t)m * strideA + sub * RPL;
#pragma unroll
      for (int j = 0; j < RPL; j += 4) {
        const f32x4 v = __builtin_bit_cast(f32x4, ld_u32x4(reinterpret_cast<const uint8_t *>(xr + j)));
#pragma unroll
        for (int e = 0; e < 4; ++e) t.x[m][j + e] = v[e];
      }
    }
    const uint8_t *w = B + (size_t)b * 32 * strideB;
#pragma unroll
    for (int j = 0; j < RPL; ++j) {
      if constexpr (Q4) t.q[j / 2][j & 1] = ld_u32(w + (woff + j * strideB));
      else t.q[j] = ld_u32x2(w + (woff + j * strideB));
    }
    t.s = ld_u32x4(reinterpret_cast<const uint8_t *>(S + (size_t)b * scaleStride + cb));
    if constexpr (AFF) t.m = ld_u32x4(reinterpret_cast<const uint8_t *>(S + (size_t)(blocks + b) * scaleStride + cb));
  };

  float acc[MT][8];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[m][c] = 0.0f;
  auto use = [&](const Slot &t) __attribute__((always_inline)) {
    float bs[MT][8], sx[MT];
#pragma unroll
    for (int j = 0; j < RPL; ++j) {
      float q[8];
      if constexpr (Q4) {
        const uint32_t w = t.q[j / 2][j & 1];
        uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
        asm("" : "+v"(lo), "+v"(hi));   // known bits would turn every conversion into a bit-field extract + convert
        q[0] = cvt_ubyte0(lo); q[1] = cvt_ubyte0(hi); q[2] = cvt_ubyte1(lo); q[3] = cvt_ubyte1(hi);
        q[4] = cvt_ubyte2(lo); q[5] = cvt_ubyte2(hi); q[6] = cvt_ubyte3(lo); q[7] = cvt_ubyte3(hi);
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) q[c] = (float)(int)(int8_t)((t.q[j][c >> 2] >> (8 * (c & 3))) & 0xFF);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float x = t.x[m][j];
        sx[m] = j == 0 ? x : sx[m] + x;
#pragma unroll
        for (int c = 0; c < 8; ++c) bs[m][c] = j == 0 ? x * q[c] : fmaf(x, q[c], bs[m][c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float s = f16bits_to_f32((t.s[c >> 1] >> (16 * (c & 1))) & 0xFFFFu);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        acc[m][c] = fmaf(Q4 ? fmaf(-8.0f, sx[m], bs[m][c]) : bs[m][c], s, acc[m][c]);
        if constexpr (AFF) acc[m][c] = fmaf(f16bits_to_f32((t.m[c >> 1] >> (16 * (c & 1))) & 0xFFFFu), sx[m], acc[m][c]);
      }
    }
  };

#pragma unroll
  for (int d = 0; d < D; ++d) {
    fetch(slot[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  uint32_t i = 0;
  for (; i + D < iters; i += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      use(slot[d]);
      fetch(slot[d], i + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (b0 + wave + W * (i + d) < b1) use(slot[d]);

  // the lanes of a column: each step keeps half of the columns, in registers that are known at compile time (left to the unroller, the
  // array went to LDS: + 10 us)
  constexpr int STEPS = LC == 32 ? 1 : LC == 16 ? 2 : 3, KEEP = 8 >> STEPS;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    uint32_t first = 0;
    auto halve = [&](auto kc, uint32_t x) __attribute__((always_inline)) {
      constexpr int keep = decltype(kc)::value;
      const bool up = (lane & x) != 0;
#pragma unroll
      for (int c = 0; c < keep; ++c) {
        const float send = up ? acc[m][c] : acc[m][c + keep], mine = up ? acc[m][c + keep] : acc[m][c];
        acc[m][c] = mine + __shfl_xor(send, (int)x);
      }
      first += up ? keep : 0;
    };
    halve(std::integral_constant<int, 4>{}, 32);
    if constexpr (STEPS > 1) halve(std::integral_constant<int, 2>{}, 16);
    if constexpr (STEPS > 2) halve(std::integral_constant<int, 1>{}, 8);
#pragma unroll
    for (int c = 0; c < KEEP; ++c) red[wave][m][8 * (lane % LC) + first + c] = acc[m][c];
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < MT * TC; t += 64 * W) {
    const uint32_t m = t / TC, c = t % TC, n = tile * TC + c;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) v += red[w][m][c];
    if (n < N) {
      if (pieces > tiles) p.C[((size_t)split * MT + m) * N + n] = v;
      else store_out(p.C, p.epi, 0, (size_t)m * p.strideC + n, v);
    }
  }
}

// The sums of up to 16 ranges, one column a lane, all of them requested at once: against eight waves that share the ranges and meet in LDS
// (sep_reduce4_kernel, for the 32 and more of other kernels) 0.1 to 0.3 us less at 1024 to 14336 columns.
constexpr uint32_t kVecSplits = 16;
template <uint32_t U>
__global__ void __launch_bounds__(64) sep_vec_reduce_kernel(const float *ws, uint32_t N, uint32_t nsplit, uint32_t tiles, size_t step,
                                                            SepVecRest p) {
  const uint32_t r = blockIdx.x / tiles, n = (blockIdx.x - r * tiles) * 64 + threadIdx.x;
  const float *src = ws + (size_t)r * N + min(n, N - 1);
  float t[U], v = 0.0f;
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) t[u] = src[min(u, nsplit - 1) * step];
#pragma unroll
  for (uint32_t u = 0; u < U; ++u)
    if (u < nsplit) v += t[u];
  if (n < N) store_out(p.C, p.epi, 0, (size_t)r * p.strideC + n, v);
}

// p.t: LC.  us, int8 / nibbles with minima, one row:
//   a K of up to 1024 in one range, strips of 64 columns on sixteen waves, while those run at once: 4096 x 1024 (N x K) 4.2 / 4.4, two or
//   more ranges 5.8 / 5.5; 14336 x 1024 7.0 / 5.8 against 7.7 / 6.5; 32000 x 1024 9.2 / 9.2, strips of 128 8.3 / 7.1; at K = 1536, 2048 columns 6.1 / 6.0
//   against 5.8 / 5.5;
//   nibbles take strips of 256 columns on four waves where there are 48 million weights and more: 14336 x 4096 12.7, strips of 128
//   13.2, 4096 x 14336 12.3 / 13.7, 28672 x 4096 19.7 / 20.8; 5120 x 5120 8.8 / 8.8, 4096 x 4096 7.2 / 7.1, 1024 x 4096 5.9 / 5.4;
//   ranges: as many as leave every wave a block and fit the chip once; two workgroups a CU where that leaves a quarter of it idle and K is
//   long (20000 x 4096, 157 strips: one range 22.9 / 18.5, three 21.4 / 16.9; 20000 x 2048 one 12.7 / 10.8, three 13.1 / 11.6).
bool sep_vec_cut(SepRowsParams &p, bool q4) {
  if (p.M > 2 || p.N % 8 != 0 || p.strideB > 1u << 26 || p.N > 1u << 29) return false;
  const uint32_t blocks = p.K / 32, strips64 = (p.N - 1) / 64 + 1;
  const bool one = blocks <= 32 && strips64 <= 256;
  p.t = one ? 8 : q4 && (uint64_t)p.K * p.N >= 48000000u ? 32 : 16;
  p.tiles = (p.N - 1) / (8 * p.t) + 1;
  uint32_t ns = 1;
  if (blocks > 32) {
    ns = std::max(1u, 256 / p.tiles);
    if (p.tiles * ns <= 192 && p.tiles > 64 && blocks >= 96) ns = 512 / p.tiles;
    ns = std::min(std::min(ns, blocks / (p.t == 32 ? 4 : 8)), kVecSplits);   // (the workspace holds blocks / 4 sets of sums: matmul_sep)
  }
  p.per = (blocks - 1) / ns + 1;
  p.nsplit = (blocks - 1) / p.per + 1;
  return true;
}

template <bool Q4, bool AFF, int MT> static void launch_vec(const SepRowsParams &p, const SepVecRest &r, hipStream_t stream) {
  const uint32_t pieces = p.tiles * p.nsplit, grid = (pieces + 7) / 8 * 8;
  auto go = [&](auto kernel, uint32_t waves) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), 0, stream, p.A, p.B, p.S, p.N, p.K / 32, p.per, p.strideA, p.strideB, p.scaleStride,
                       p.tiles, pieces, r);
  };
  if constexpr (Q4)
    if (p.t == 32) return go(sep_vec_kernel<Q4, AFF, MT, 32, 4, 2>, 4);
  if (p.t == 16) go(sep_vec_kernel<Q4, AFF, MT, 16, 8, 2>, 8);
  else go(sep_vec_kernel<Q4, AFF, MT, 8, 16, 2>, 16);
}

int launch_sep_vec(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream) {
  const SepVecRest out{p.C, p.epi, p.strideC}, r = p.nsplit > 1 ? SepVecRest{p.partial, Epilogue{CUTHIP_EPI_NONE, 0, nullptr}, p.N} : out;
  if (!q4) p.M == 1 ? launch_vec<false, false, 1>(p, r, stream) : launch_vec<false, false, 2>(p, r, stream);
  else if (!affine) p.M == 1 ? launch_vec<true, false, 1>(p, r, stream) : launch_vec<true, false, 2>(p, r, stream);
  else p.M == 1 ? launch_vec<true, true, 1>(p, r, stream) : launch_vec<true, true, 2>(p, r, stream);
  if (int rc = check_hip(hipGetLastError(), "separated-layout matmul launch")) return rc;
  if (p.nsplit == 1) return CUTHIP_OK;
  const uint32_t tiles = (p.N - 1) / 64 + 1;
  hipLaunchKernelGGL(p.nsplit <= 8 ? sep_vec_reduce_kernel<8> : sep_vec_reduce_kernel<kVecSplits>, dim3(tiles * p.M), dim3(64), 0, stream,
                     (const float *)p.partial, p.N, p.nsplit, tiles, (size_t)p.M * p.N, out);
  return check_hip(hipGetLastError(), "separated-layout reduce launch");
}

}  // namespace cuthip
