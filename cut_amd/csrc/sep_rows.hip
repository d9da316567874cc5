// Matmul on the reference's separated weight layout (see compat.hip) for several rows of A, fp32 throughout:
//   C[m,n] = sum_k A[m,k] * w[k,n]
// on the matrix cores, with products as exact as fp32 fused multiply-adds have them: an integer of 8 bits or less is a bf16
// number, and an fp32 activation is the sum of three (its leading, middle and last eight significant bits), so the three
// v_mfma_f32_16x16x32_bf16 of a fragment multiply without rounding and add in fp32.  One matrix instruction's k range is one
// quantization block, whose sum is scaled in fp32 as in the vector kernel.
//
//   * A wave owns 128 columns and a range of blocks.  Lane (c, g) loads columns 8 c .. 8 c + 7 of the k-rows 8 g .. 8 g + 7
//     of a block: 128 (nibbles: 64) contiguous bytes of each k-row per load.  Byte f of the eight rows is the lane's part of
//     the B operand for column 8 c + f, so the K-major layout needs no transposition: eight operands, eight columns a lane.
//   * A is read from global memory in the operand's own shape (16 rows of 128 bytes) and split in registers; no LDS and no
//     barrier until the ranges of the workgroup meet at the end.
//   * Two blocks of loads are in flight per wave, in a ring of registers.
//
// What bounds it: the memory up to 16 rows (about 180 vector instructions and 24 matrix instructions a block and wave, 4 KB of
// int8), the vector ALU beyond (44 instructions to split 16 rows, 32 to scale their results).  Measured, us, both launches
// (graph replay, weights from memory), passes of four rows on the vector ALU -> this kernel:
//   14336 x 4096  int8     4 rows 22.3 -> 19.7,  8 rows 33.4 -> 20.3,  16 rows 54.5 -> 21.9,  31 rows 96.5 -> 29.5
//                 nibbles  4 rows 19.3 -> 18.0,  8 rows 31.6 -> 18.4,  16 rows 53.8 -> 19.9,  31 rows 96.0 -> 28.7
//   4096 x 14336  int8     8 rows 34.2 -> 20.4,  31 rows 99.3 -> 28.1;   1024 x 4096  int8  8 rows 13.4 -> 9.5, 31 rows 15.6 -> 13.6
// Distance to float64 (2-norm, the shapes above): int8 1.0e-7 to 1.4e-7 of the result (vector kernel 1.3e-7 to 1.5e-7), nibbles
// 1.1e-7 to 1.6e-7 (2.2e-7 to 3.4e-7).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "sep_rows.hpp"

namespace cuthip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kSepRowsK = 4;         // K ranges of a workgroup: two waves side by side in each
constexpr uint32_t kSepRowsTile = 256;

enum { kSepQ8 = 0, kSepQ4 = 1, kSepAffine = 2 };

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// the upper halves of two floats: a pair of bf16, truncated
__device__ __forceinline__ uint32_t upper_pair(float a, float b) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}
__device__ __forceinline__ float upper(float v) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u); }

// Eight activations as three bf16 operands whose sum they are (8 + 8 + 8 significant bits, truncated each time, so that the
// differences are exact).  An infinity is its first part alone: infinity minus itself would make the others NaN.
__device__ __forceinline__ void split3(f32x4 x, f32x4 y, u32x4 &hi, u32x4 &mid, u32x4 &lo) {
  float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]}, r[8], s[8];
  bool inf = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    r[e] = v[e] - upper(v[e]);
    inf |= __builtin_isinf(v[e]);
  }
  if (__builtin_amdgcn_ballot_w64(inf) != 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = __builtin_isinf(v[e]) ? 0.0f : r[e];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = r[e] - upper(r[e]);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = upper_pair(v[2 * e], v[2 * e + 1]);
    mid[e] = upper_pair(r[2 * e], r[2 * e + 1]);
    lo[e] = upper_pair(s[2 * e], s[2 * e + 1]);
  }
}

template <int KIND, int T>
__global__ void __launch_bounds__(512, T == 1 ? 4 : 2) sep_rows_kernel(SepRowsParams p) {
  constexpr bool Q4 = KIND != kSepQ8;
  constexpr int D = 2;   // blocks in flight (three of them leave one workgroup on a CU: 14336 x 4096 at 8 rows 21.9 us, 20.3)
  __shared__ f32x4 red[kSepRowsK][T][8][64];   // two ranges of two waves at a time; [fragment][lane]: no bank conflicts
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c = lane & 15, g = lane >> 4, side = wave & 1, kw = wave >> 1;
  // Ids id, id + 8, ... share an XCD: the passes over one piece of the weights run there one after the other, and all but
  // the first find it in that XCD's L2.
  const uint32_t slot = blockIdx.x >> 3, group = __builtin_amdgcn_readfirstlane(slot / p.passes), pass = slot - group * p.passes;
  const uint32_t piece = group * 8 + (blockIdx.x & 7), split = __builtin_amdgcn_readfirstlane(piece / p.tiles);
  if (split >= p.nsplit) return;   // the last group of eight may be short
  const uint32_t tile = piece - split * p.tiles, m0 = pass * (16 * T);
  const uint32_t c0 = tile * kSepRowsTile + side * 128 + 8 * c;
  const bool live = c0 < p.N;
  const uint32_t blocks = p.K / 32, b0 = (split * kSepRowsK + kw) * p.per, b1 = min(b0 + p.per, blocks);

  // lane offsets inside a block (32 bits); lanes past the last column read column 0, rows past the last the last row
  const uint32_t cb = live ? c0 : 0u, woff = 8 * g * p.strideB + (Q4 ? cb / 2 : cb), soff = cb * 2;
  uint32_t aoff[T];
#pragma unroll
  for (int t = 0; t < T; ++t) aoff[t] = (min(16 * t + c, p.M - 1 - m0) * p.strideA + 8 * g) * 4;
  const uint8_t *abase = reinterpret_cast<const uint8_t *>(p.A + (size_t)m0 * p.strideA);

  using Row = typename std::conditional<Q4, uint32_t, u32x2>::type;
  Row w[D][8];
  f32x4 a[D][T][2];
  u32x4 sc[D], mn[KIND == kSepAffine ? D : 1];
  auto request = [&](int d, uint32_t b) __attribute__((always_inline)) {
    b = min(b, blocks - 1);
    const uint8_t *ab = abase + (size_t)b * 128;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      a[d][t][0] = __builtin_bit_cast(f32x4, ld_u32x4(ab + aoff[t]));
      a[d][t][1] = __builtin_bit_cast(f32x4, ld_u32x4(ab + aoff[t] + 16));
    }
    const uint8_t *wb = p.B + (size_t)b * 32 * p.strideB;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (Q4) w[d][j] = ld_u32(wb + woff + j * p.strideB);
      else w[d][j] = ld_u32x2(wb + woff + j * p.strideB);
    }
    const uint8_t *sb = reinterpret_cast<const uint8_t *>(p.S + (size_t)b * p.scaleStride);
    sc[d] = ld_u32x4(sb + soff);
    if constexpr (KIND == kSepAffine) mn[d] = ld_u32x4(sb + (size_t)blocks * p.scaleStride * 2 + soff);
    __builtin_amdgcn_sched_barrier(0);
  };

  f32x4 acc[T][8];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int f = 0; f < 8; ++f) acc[t][f] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

  auto work = [&](int d) __attribute__((always_inline)) {
    u32x4 hi[T], mid[T], lo[T];
    f32x4 sx[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      split3(a[d][t][0], a[d][t][1], hi[t], mid[t], lo[t]);
      if constexpr (Q4) {   // sums of x over the block, in every column
        const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
        sx[t] = mfma_bf16(hi[t], ones, mfma_bf16(mid[t], ones, mfma_bf16(lo[t], ones, zero)));
      }
    }
    uint32_t n[8][2];   // Q4: nibbles of the even and the odd columns, a byte each
    if constexpr (Q4) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        n[j][0] = w[d][j] & 0x0F0F0F0Fu;
        n[j][1] = (w[d][j] >> 4) & 0x0F0F0F0Fu;
        asm volatile("" : "+v"(n[j][0]), "+v"(n[j][1]));   // known bits would turn every conversion into a bit-field extract + convert
      }
    }
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      auto value = [&](int j) __attribute__((always_inline)) {
        if constexpr (Q4) return (float)((n[j][f & 1] >> (8 * (f >> 1))) & 0xFFu);
        else return (float)(int)(int8_t)((w[d][j][f >> 2] >> (8 * (f & 3))) & 0xFFu);
      };
      u32x4 b;
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = upper_pair(value(2 * e), value(2 * e + 1));
      const float s = f16bits_to_f32((sc[d][f >> 1] >> (16 * (f & 1))) & 0xFFFFu);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        f32x4 v = mfma_bf16(hi[t], b, mfma_bf16(mid[t], b, mfma_bf16(lo[t], b, zero)));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (Q4) v[i] = fmaf(-8.0f, sx[t][i], v[i]);
          acc[t][f][i] = fmaf(v[i], s, acc[t][f][i]);
          if constexpr (KIND == kSepAffine)
            acc[t][f][i] = fmaf(f16bits_to_f32((mn[d][f >> 1] >> (16 * (f & 1))) & 0xFFFFu), sx[t][i], acc[t][f][i]);
        }
      }
    }
  };

  if (b0 < b1) {
#pragma unroll
    for (int d = 0; d < D; ++d) request(d, b0 + d);
    for (uint32_t b = b0; b < b1; b += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (b + d < b1) work(d);
        request(d, b + d + D);   // unconditional, so that the waits count the loads in flight exactly
      }
    }
  }

  // the four ranges of the workgroup meet in LDS: 2 + 3 -> 0 + 1, then 1 -> 0
#pragma unroll
  for (int step = 2; step >= 1; --step) {
    if (step == 1) __syncthreads();
    if (kw >= (uint32_t)step && kw < 2 * (uint32_t)step) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int f = 0; f < 8; ++f) red[(kw - step) * 2 + side][t][f][lane] = acc[t][f];
    }
    __syncthreads();
    if (kw < (uint32_t)step) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int f = 0; f < 8; ++f) acc[t][f] += red[kw * 2 + side][t][f][lane];
    }
  }
  if (kw > 0 || !live) return;
  if (p.nsplit > 1) {   // to the workspace [split][M][N], 16-byte aligned
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = m0 + 16 * t + 4 * g + i;
        if (row >= p.M) continue;
        f32x4 *dst = reinterpret_cast<f32x4 *>(p.partial + ((size_t)split * p.M + row) * p.N + c0);
        dst[0] = f32x4{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
        dst[1] = f32x4{acc[t][4][i], acc[t][5][i], acc[t][6][i], acc[t][7][i]};
      }
    return;
  }
  // every operator of the epilogue behind each of 32 T stores would be most of the kernel's code: the lane's results go
  // through its own part of LDS into a loop
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int f = 0; f < 8; ++f) red[side][t][f][lane] = acc[t][f];
#pragma unroll 1
  for (uint32_t e = 0; e < 32u * T; ++e) {
    const uint32_t f = e & 7, i = (e >> 3) & 3, t = e >> 5, row = m0 + 16 * t + 4 * g + i;
    if (row < p.M) store_out(p.C, p.epi, 0, (size_t)row * p.strideC + c0 + f, red[side][t][f][lane][i]);
  }
}

// K ranges over workgroups: as many as run at once (a second round, or more partial sums than that, costs more than it
// gives: 14336 x 4096, 8 rows, int8, two / four / eight ranges of 56 column tiles 27.3 / 20.3 / 22.0 us; 4096 x 14336, 8 / 16 /
// 28 ranges of 16 tiles 25.6 / 20.4 / 20.2), at least one block a wave.
void sep_rows_cut(SepRowsParams &p) {
  const uint32_t blocks = p.K / 32;
  p.tiles = (p.N - 1) / kSepRowsTile + 1;
  p.passes = p.M <= 16 ? 1 : (p.M - 1) / 32 + 1;
  const uint64_t panels = (uint64_t)p.tiles * p.passes;
  uint32_t want = g_tuning.gemm_ksplit ? (uint32_t)g_tuning.gemm_ksplit : panels < 256 ? (uint32_t)(256 / panels) : 1u;
  want = std::min(want, (blocks - 1) / kSepRowsK + 1);
  p.per = (blocks - 1) / (want * kSepRowsK) + 1;
  p.nsplit = (blocks - 1) / (p.per * kSepRowsK) + 1;
}

static uint64_t sep_rows_grid(const SepRowsParams &p) { return ((uint64_t)p.tiles * p.nsplit + 7) / 8 * 8 * p.passes; }

// Whole lanes of eight columns; offsets inside a block and inside a pass over 32 rows of A are 32-bit, and so are the threads
// of the launch and of the reduce.
bool sep_rows_fits(const SepRowsParams &p) {
  const uint64_t reduce = ((uint64_t)(p.N - 1) / 256 + 1) * p.M;
  return p.N % 8 == 0 && (uint64_t)p.strideB * 32 <= 0xFFFFFFFFull && (uint64_t)p.strideA * 128 <= 0xFFFFFFFFull &&
         std::max(sep_rows_grid(p), reduce) * 512 <= 0xFFFFFFFFull;
}

template <int KIND> static int launch_kind(const SepRowsParams &p, uint32_t grid, hipStream_t stream) {
  if (p.M <= 16) hipLaunchKernelGGL((sep_rows_kernel<KIND, 1>), dim3(grid), dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((sep_rows_kernel<KIND, 2>), dim3(grid), dim3(512), 0, stream, p);
  return check_hip(hipGetLastError(), "separated-layout row matmul launch");
}

int launch_sep_rows(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream) {
  const uint32_t grid = (uint32_t)sep_rows_grid(p);
  return affine ? launch_kind<kSepAffine>(p, grid, stream) : q4 ? launch_kind<kSepQ4>(p, grid, stream) : launch_kind<kSepQ8>(p, grid, stream);
}

}  // namespace cuthip
