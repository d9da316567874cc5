// Matmul on the reference's separated weight layout (see compat.hip) for several rows of A, fp32 throughout:
//   C[m,n] = sum_k A[m,k] * w[k,n]
// on the matrix cores, with products as exact as fp32 fused multiply-adds have them: an integer of 8 bits or less is a bf16
// number, and an fp32 activation is the sum of three (its leading, middle and last eight significant bits), so the three
// v_mfma_f32_16x16x32_bf16 of a fragment multiply without rounding and add in fp32 (below 2^-110 times 2^24: see split3).  One matrix
// instruction's k range is one quantization block, whose sum is scaled in fp32 as in the vector kernel.
//
//   * A wave owns 128 columns and a range of blocks.  Lane (c, g) loads columns 8 c .. 8 c + 7 of the k-rows 8 g .. 8 g + 7
//     of a block: 128 (nibbles: 64) contiguous bytes of each k-row per load.  Byte f of the eight rows is the lane's part of
//     the B operand for column 8 c + f, so the K-major layout needs no transposition: eight operands, eight columns a lane.
//   * A is read from global memory in the operand's own shape (16 rows of 128 bytes) and split in registers; no LDS and no
//     barrier until the ranges of the workgroup meet at the end.
//   * Two blocks of loads are in flight per wave, in a ring of registers.
//
// What bounds it (14336 x 4096): int8 up to 16 rows the memory (3.4 of the 4.8 TB/s of a copy, vector ALU 41 % of the time: about 210
// vector instructions and 24 matrix instructions a block and wave, 4 KB of int8), nibbles the vector ALU (56 to 59 %), and int8 beyond
// 16 rows it (46 %: 44 instructions to split 16 rows, 32 to scale their results) beside chains of three matrix instructions (28 %).  Measured,
// us, both launches
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
// differences are exact).  True for one of which that does not hold: a third part that is a NaN (infinity minus itself) or
// subnormal (bf16 ends at 2^-133, so that below 2^-110 the last bits may be lost).
__device__ __forceinline__ bool split3(f32x4 x, f32x4 y, u32x4 &hi, u32x4 &mid, u32x4 &lo) {
  const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  float r[8], s[8];
  bool odd = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    r[e] = v[e] - upper(v[e]);
    s[e] = r[e] - upper(r[e]);
    odd |= __builtin_amdgcn_classf(s[e], 0x1 | 0x2 | 0x10 | 0x80);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = upper_pair(v[2 * e], v[2 * e + 1]);
    mid[e] = upper_pair(r[2 * e], r[2 * e + 1]);
    lo[e] = upper_pair(s[2 * e], s[2 * e + 1]);
  }
  return odd;
}
// For waves that hold such values: times `up` (2^24 makes every part of a subnormal number normal), and an infinity as its first
// part alone.
__device__ __forceinline__ void split3_odd(f32x4 x, f32x4 y, float up, u32x4 &hi, u32x4 &mid, u32x4 &lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v[2], r[2], s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v[h] = (e < 2 ? x[2 * e + h] : y[2 * e + h - 4]) * up;
      r[h] = __builtin_isinf(v[h]) ? 0.0f : v[h] - upper(v[h]);
      s[h] = r[h] - upper(r[h]);
    }
    hi[e] = upper_pair(v[0], v[1]);
    mid[e] = upper_pair(r[0], r[1]);
    lo[e] = upper_pair(s[0], s[1]);
  }
}

// Where a workgroup and a lane stand.
struct SepPlace {
  uint32_t lane, c, g, side, kw;   // columns 8 c .. 8 c + 7 of the 128 of this side, k-rows 8 g .. 8 g + 7, K range
  uint32_t split, m0, c0, b0, b1;  // c0: first column; blocks b0 .. b1 - 1
  bool live, any;                  // columns inside N; a range that exists
};
template <int T> __device__ __forceinline__ SepPlace sep_place(const SepRowsParams &p) {
  SepPlace s;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  s.lane = threadIdx.x & 63;
  s.c = s.lane & 15;
  s.g = s.lane >> 4;
  s.side = wave & 1;
  s.kw = wave >> 1;
  // Ids id, id + 8, ... share an XCD: the passes over one piece of the weights run there one after the other, and all but
  // the first find it in that XCD's L2.  Pieces go round the XCDs (neighbours on one XCD: 3 to 31 rows 3 % longer); the passes over
  // those that are left over, fewer than eight, are shared out (as whole pieces they are a second round of workgroups for
  // some XCDs: 828 rows of 4816 x 5888 on nibbles, 19 pieces of 13 passes, 140 us, so 81).
  const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, pieces = p.tiles * p.nsplit, even = (pieces >> 3) * p.passes;
  const uint32_t item = slot < even ? slot : xcd * (((pieces & 7) * p.passes + 7) >> 3) + slot - even;
  const uint32_t group = __builtin_amdgcn_readfirstlane(item / p.passes), pass = item - group * p.passes;
  const uint32_t piece = slot < even ? group * 8 + xcd : (pieces & ~7u) + group;
  s.split = __builtin_amdgcn_readfirstlane(piece / p.tiles);
  s.any = s.split < p.nsplit;   // the last XCD's share may be short
  s.m0 = pass * (16 * T);
  s.c0 = (piece - s.split * p.tiles) * kSepRowsTile + s.side * 128 + 8 * s.c;
  s.live = s.c0 < p.N;
  s.b0 = (s.split * kSepRowsK + s.kw) * p.per;
  s.b1 = min(s.b0 + p.per, p.K / 32);
  return s;
}

// four outputs of one row through the epilogue (vec: C and D take 16-byte accesses)
__device__ __forceinline__ void sep_store4(const SepRowsParams &p, size_t idx, f32x4 v, bool vec) {
  if (!vec) {
#pragma unroll
    for (int f = 0; f < 4; ++f) store_out(p.C, p.epi, 0, idx + f, v[f]);
    return;
  }
  if (p.epi.kind == CUTHIP_EPI_UNARY) {
#pragma unroll
    for (int f = 0; f < 4; ++f) v[f] = apply_unary(p.epi.op, v[f]);
  } else if (p.epi.kind == CUTHIP_EPI_BINARY) {
    const f32x4 d = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(p.epi.D) + idx);
#pragma unroll
    for (int f = 0; f < 4; ++f) v[f] = apply_binary(p.epi.op, v[f], d[f]);
  }
  *reinterpret_cast<f32x4 *>(p.C + idx) = v;
}

// The four K ranges of the workgroup meet in LDS (T x 32 KB: 2 + 3 -> 0 + 1, then 1 -> 0) and leave for C or the partial sums.
template <int T> __device__ __forceinline__ void sep_finish(const SepRowsParams &p, const SepPlace &s, f32x4 (&acc)[T][8], uint8_t *lds) {
  f32x4 (*red)[T][8][64] = reinterpret_cast<f32x4 (*)[T][8][64]>(lds);   // [fragment][lane]: no bank conflicts
#pragma unroll
  for (int step = 2; step >= 1; --step) {
    if (step == 1) __syncthreads();
    if (s.kw >= (uint32_t)step && s.kw < 2 * (uint32_t)step) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int f = 0; f < 8; ++f) red[(s.kw - step) * 2 + s.side][t][f][s.lane] = acc[t][f];
    }
    __syncthreads();
    if (s.kw < (uint32_t)step) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int f = 0; f < 8; ++f) acc[t][f] += red[s.kw * 2 + s.side][t][f][s.lane];
    }
  }
  if (s.kw > 0 || !s.live) return;
  if (p.nsplit > 1) {   // to the workspace [split][M][N], 16-byte aligned
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = s.m0 + 16 * t + 4 * s.g + i;
        if (row >= p.M) continue;
        f32x4 *dst = reinterpret_cast<f32x4 *>(p.partial + ((size_t)s.split * p.M + row) * p.N + s.c0);
        dst[0] = f32x4{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
        dst[1] = f32x4{acc[t][4][i], acc[t][5][i], acc[t][6][i], acc[t][7][i]};
      }
    return;
  }
  // every operator of the epilogue behind each of 8 T stores would be most of the kernel's code: the lane's results go
  // through its own part of LDS into a loop
  f32x4 *own = &red[s.side][0][0][0];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      own[(8 * t + 2 * i) * 64 + s.lane] = f32x4{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
      own[(8 * t + 2 * i + 1) * 64 + s.lane] = f32x4{acc[t][4][i], acc[t][5][i], acc[t][6][i], acc[t][7][i]};
    }
  const bool vec = ((uintptr_t)p.C | (p.epi.kind == CUTHIP_EPI_BINARY ? (uintptr_t)p.epi.D : 0)) % 16 == 0 && p.strideC % 4 == 0;
#pragma unroll 1
  for (uint32_t e = 0; e < 8u * T; ++e) {
    const uint32_t row = s.m0 + 16 * (e >> 3) + 4 * s.g + ((e >> 1) & 3);
    if (row < p.M) sep_store4(p, (size_t)row * p.strideC + s.c0 + 4 * (e & 1), own[e * 64 + s.lane], vec);
  }
}

// Blocks b0 .. b1 - 1 of a wave, two of them in flight in a ring of registers.  Every step requests, a step behind the last block
// that one again (from the caches): with requests under a condition the waits count for the worst case, and behind an early
// return they sink past it.  Three blocks in flight give nothing (16 to 512 rows within 3 %) and cost the third workgroup's registers.
template <class RQ, class WK> __device__ __forceinline__ void sep_walk(uint32_t b0, uint32_t b1, RQ request, WK work) {
  if (b0 >= b1) return;
  request(0, b0);
  request(1, b0 + 1);
  for (uint32_t b = b0; b < b1; b += 2) {
    work(0);
    request(0, b + 2);
    if (b + 1 < b1) work(1);
    request(1, b + 3);
  }
}

template <int KIND, int T>
__global__ void __launch_bounds__(512, T == 1 ? 4 : 2) sep_rows_kernel(SepRowsParams p) {
  constexpr bool Q4 = KIND != kSepQ8;
  __shared__ __attribute__((aligned(16))) uint8_t lds[T * 32 * 1024];
  const SepPlace s = sep_place<T>(p);
  if (!s.any) return;
  const uint32_t blocks = p.K / 32;

  // lane offsets inside a block (32 bits); lanes past the last column read column 0, rows past the last the last row
  const uint32_t cb = s.live ? s.c0 : 0u, woff = 8 * s.g * p.strideB + (Q4 ? cb / 2 : cb), soff = cb * 2;
  uint32_t aoff[T];
#pragma unroll
  for (int t = 0; t < T; ++t) aoff[t] = (min(16 * t + s.c, p.M - 1 - s.m0) * p.strideA + 8 * s.g) * 4;
  const uint8_t *abase = reinterpret_cast<const uint8_t *>(p.A + (size_t)s.m0 * p.strideA);

  using Row = typename std::conditional<Q4, uint32_t, u32x2>::type;
  Row w[2][8];
  f32x4 a[2][T][2];
  u32x4 sc[2], mn[KIND == kSepAffine ? 2 : 1];
  auto request = [&](int d, uint32_t b) __attribute__((always_inline)) {
    b = min(b, s.b1 - 1);
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

  auto multiply = [&](int d, const u32x4 *hi, const u32x4 *mid, const u32x4 *lo, const f32x4 *sx) __attribute__((always_inline)) {
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
      const float scale = f16bits_to_f32((sc[d][f >> 1] >> (16 * (f & 1))) & 0xFFFFu);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        f32x4 v = mfma_bf16(hi[t], b, mfma_bf16(mid[t], b, mfma_bf16(lo[t], b, zero)));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (Q4) v[i] = fmaf(-8.0f, sx[t][i], v[i]);
          acc[t][f][i] = fmaf(v[i], scale, acc[t][f][i]);
          if constexpr (KIND == kSepAffine)
            acc[t][f][i] = fmaf(f16bits_to_f32((mn[d][f >> 1] >> (16 * (f & 1))) & 0xFFFFu), sx[t][i], acc[t][f][i]);
        }
      }
    }
  };
  auto sum = [&](const u32x4 &hi, const u32x4 &mid, const u32x4 &lo) __attribute__((always_inline)) {   // of x over the block, in every column
    const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    return Q4 ? mfma_bf16(hi, ones, mfma_bf16(mid, ones, mfma_bf16(lo, ones, zero))) : zero;
  };

  bool odd = false;
  sep_walk(s.b0, s.b1, request, [&](int d) __attribute__((always_inline)) {
    u32x4 hi[T], mid[T], lo[T];
    f32x4 sx[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      odd |= split3(a[d][t][0], a[d][t][1], hi[t], mid[t], lo[t]);
      sx[t] = sum(hi[t], mid[t], lo[t]);   // (one tile's beside the split of the next: behind both, 17 to 31 rows of nibbles take 4 % longer)
    }
    multiply(d, hi, mid, lo, sx);
  });

  // A wave that met numbers which split3 does not split exactly begins again, with activations and sums times 2^24 in the rows that
  // hold no number from 2^40 on (2^32 products of it with 127 and a scale of 2^16, times 2^24, stay below 2^119); beside such a number
  // the small ones of its own row keep what bf16 has.  8 x 14336 x 4096, us, with one such number / in every block: int8 25.2 / 32.2
  // (without 20.2), nibbles 23.0 / 28.8 (17.8).  Inside the walk, block by block, they take 23.6 there, but 720 calls of 3 to 31
  // rows without any 1.4 % longer, up to 7 (code and registers beside the loop), or 0.4 % with one scaling for all rows of the wave.
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd) != 0, 0)) {
    uint32_t most[T] = {};   // the largest magnitude of the lane's row, as bits: what is no number is above all
#pragma unroll 1
    for (uint32_t b = s.b0; b < s.b1; ++b) {
      request(0, b);
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) most[t] = max(most[t], __builtin_bit_cast(uint32_t, a[0][t][e >> 2][e & 3]) & 0x7FFFFFFFu);
    }
    uint32_t up = 0;   // (uniform) a bit for each row that is scaled
#pragma unroll
    for (int t = 0; t < T; ++t) {
      uint64_t large = __builtin_amdgcn_ballot_w64(most[t] >= __builtin_bit_cast(uint32_t, 0x1p40f));   // 16 g + row
      large |= large >> 32;
      up |= (uint32_t)(~(large | large >> 16) & 0xFFFF) << 16 * t;
#pragma unroll
      for (int f = 0; f < 8; ++f) acc[t][f] = zero;
    }
    sep_walk(s.b0, s.b1, request, [&](int d) __attribute__((always_inline)) {
      u32x4 hi[T], mid[T], lo[T];
      f32x4 sx[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        split3_odd(a[d][t][0], a[d][t][1], up >> (16 * t + s.c) & 1 ? 0x1p24f : 1.0f, hi[t], mid[t], lo[t]);
        sx[t] = sum(hi[t], mid[t], lo[t]);
      }
      multiply(d, hi, mid, lo, sx);
    });
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float by = up >> (16 * t + 4 * s.g + i) & 1 ? 0x1p-24f : 1.0f;
#pragma unroll
        for (int f = 0; f < 8; ++f) acc[t][f][i] *= by;
      }
  }
  sep_finish<T>(p, s, acc, lds);
}

// ---- 32 rows and more: operands rounded to fp16 -------------------------------------------------------------------
// The same walk over the weights with the operands of the dense GEMM (activations rounded to fp16 once, by a launch in front
// of this one; weights fp16(q * scale (+ min))), for as many rows as it takes until writing the weights out once as fp16 pays:
// no pass over memory but the blocks themselves.  A weight costs two vector instructions (two k-rows are paired by a byte
// permute with the 0x64 that makes 1024 + q of them, offset and scale are packed fp16) once per 16 T rows, and the sums over
// all of K stay in the accumulators.  What bounds it: those instructions and, from 64 rows on, the matrix cores.  Measured, us, all
// launches (graph replay), two passes -> this:
//   14336 x 4096  int8  32 rows 84 -> 25,  64 rows 86 -> 34,  128 rows 92 -> 46,  256 rows 97 -> 69;  nibbles 64 rows 87 -> 28
//   4096 x 14336  int8  64 rows 81 -> 36,  256 rows 96 -> 68;   4096 x 4096  int8  64 rows 33 -> 20,  256 rows 47 -> 32
//   1024 x 4096   int8  64 rows 24 -> 18,  512 rows 31 -> 27
__device__ __forceinline__ f32x4 mfma_f16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ half2_t as_pair(uint32_t v) { return __builtin_bit_cast(half2_t, v); }

template <int KIND, int T>
__global__ void __launch_bounds__(512, 2) sep_rows16_kernel(SepRowsParams p) {
  constexpr bool Q4 = KIND != kSepQ8;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // T x 32 KB
  const SepPlace s = sep_place<T>(p);
  if (!s.any) return;
  const uint32_t blocks = p.K / 32;
  const uint32_t cb = s.live ? s.c0 : 0u, woff = 8 * s.g * p.strideB + (Q4 ? cb / 2 : cb), soff = cb * 2;
  uint32_t aoff[T];
#pragma unroll
  for (int t = 0; t < T; ++t) aoff[t] = (min(16 * t + s.c, p.M - 1 - s.m0) * p.K + 8 * s.g) * 2;
  const uint8_t *abase = reinterpret_cast<const uint8_t *>(p.A16 + (size_t)s.m0 * p.K);

  using Row = typename std::conditional<Q4, uint32_t, u32x2>::type;
  Row w[2][8];
  u32x4 a[2][T], sc[2], mn[KIND == kSepAffine ? 2 : 1];
  auto request = [&](int d, uint32_t b) __attribute__((always_inline)) {
    b = min(b, s.b1 - 1);
    const uint8_t *ab = abase + (size_t)b * 64;
#pragma unroll
    for (int t = 0; t < T; ++t) a[d][t] = *reinterpret_cast<const u32x4 *>(ab + aoff[t]);
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

  auto work = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      const half_t sh = as_pair(sc[d][f >> 1])[f & 1];
      const half2_t scale{sh, sh};
      half2_t low{};
      if constexpr (KIND == kSepAffine) {
        const half_t m = as_pair(mn[d][f >> 1])[f & 1];
        low = half2_t{m, m};
      }
      u32x4 b;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        half2_t q;
        if constexpr (Q4) {
          constexpr uint32_t pick[4] = {0x0C040C00u, 0x0C050C01u, 0x0C060C02u, 0x0C070C03u};   // byte f / 2 of both rows
          const uint32_t v = __builtin_amdgcn_perm(w[d][2 * e + 1], w[d][2 * e], pick[f >> 1]);
          if (f & 1) q = __builtin_elementwise_fma(as_pair((v & 0x00F000F0u) | 0x64006400u), half2_t{(half_t)0.0625f, (half_t)0.0625f}, half2_t{(half_t)-72.0f, (half_t)-72.0f});
          else q = as_pair((v & 0x000F000Fu) | 0x64006400u) + half2_t{(half_t)-1032.0f, (half_t)-1032.0f};
        } else {
          constexpr uint32_t pair[4] = {0x05010400u, 0x05010400u, 0x07030602u, 0x07030602u};
          const uint32_t v = __builtin_amdgcn_perm(w[d][2 * e + 1][f >> 2], w[d][2 * e][f >> 2], pair[f & 3]) ^ 0x80808080u;   // columns f & ~1, f | 1
          q = as_pair(__builtin_amdgcn_perm(0x64646464u, v, f & 1 ? 0x04030402u : 0x04010400u)) + half2_t{(half_t)-1152.0f, (half_t)-1152.0f};
        }
        if constexpr (KIND == kSepAffine) b[e] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, scale, low));
        else b[e] = __builtin_bit_cast(uint32_t, q * scale);
      }
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t][f] = mfma_f16(a[d][t], b, acc[t][f]);
    }
  };

  sep_walk(s.b0, s.b1, request, work);
  sep_finish<T>(p, s, acc, lds);
}

static uint64_t sep_rows_grid(const SepRowsParams &p) {
  const uint64_t pieces = (uint64_t)p.tiles * p.nsplit;
  return (pieces / 8 * p.passes + (pieces % 8 * p.passes + 7) / 8) * 8;
}

// Whole lanes of eight columns; offsets inside a block and inside a pass over the rows of A are 32-bit, and so are the threads
// of the launch and of the reduce.
static bool sep_fits(const SepRowsParams &p, uint64_t a_row_bytes) {
  const uint64_t reduce = ((uint64_t)(p.N - 1) / 256 + 1) * p.M;
  return p.N % 8 == 0 && (uint64_t)p.strideB * 32 <= 0xFFFFFFFFull && a_row_bytes * 16 * p.t <= 0xFFFFFFFFull &&
         std::max(sep_rows_grid(p), reduce) * 512 <= 0xFFFFFFFFull;
}

// K ranges over workgroups: as many as run at once (a second round, or more partial sums than that, costs more than it
// gives: 14336 x 4096, 8 rows, int8, two / four / eight ranges of 56 column tiles 27.3 / 20.3 / 22.0 us; 4096 x 14336, 8 / 16 /
// 28 ranges of 16 tiles 25.6 / 20.4 / 20.2), at least one block a wave.
bool sep_rows_cut(SepRowsParams &p, size_t partial_bytes) {
  p.t = p.M <= 16 ? 1 : 2;
  const uint32_t blocks = p.K / 32;
  p.tiles = (p.N - 1) / kSepRowsTile + 1;
  p.passes = (p.M - 1) / (16 * p.t) + 1;
  const uint64_t panels = (uint64_t)p.tiles * p.passes;
  uint32_t want = g_tuning.gemm_ksplit ? (uint32_t)g_tuning.gemm_ksplit : panels < 256 ? (uint32_t)(256 / panels) : 1u;
  want = (uint32_t)std::min<uint64_t>(std::min(want, (blocks - 1) / kSepRowsK + 1), std::max<uint64_t>(1, partial_bytes / ((uint64_t)p.M * p.N * 4)));
  p.per = (blocks - 1) / (want * kSepRowsK) + 1;
  p.nsplit = (blocks - 1) / (p.per * kSepRowsK) + 1;
  return sep_fits(p, (uint64_t)p.strideA * 4);
}

// From 32 rows on.  Microseconds with the conversion of A in front and the sum over the ranges behind, fitted to 2,430 launches
// (three layouts, 32 .. 512 rows, nine weight shapes from 512 x 512 to 14336 x 4096, 1 .. 16 ranges forced; graph replay; 9 %
// rms; the ranges chosen are 1.4 % slower than the best of them on average): a fixed part, the blocks of a wave in every
// round of 256 workgroups, more for a full chip, the partial products, C, A.  No wave gets a single block if there are more (512 x 2048,
// 192 rows: 16 ranges 17.4, eight 15.4).
bool sep_rows16_cut(SepRowsParams &p, bool q4, bool affine, size_t partial_bytes) {
  static const double kBlock[3][3] = {{0.88, 1.18, 1.49}, {0.62, 0.87, 1.15}, {0.69, 0.94, 1.22}}, kFull[3] = {0.38, 0.34, 0.05};
  const uint32_t t16 = (p.M - 1) / 16 + 1, blocks = p.K / 32;
  p.t = std::max(2u, (t16 - 1) / ((t16 - 1) / 4 + 1) + 1);
  p.tiles = (p.N - 1) / kSepRowsTile + 1;
  p.passes = (p.M - 1) / (16 * p.t) + 1;
  const double block = kBlock[affine ? 2 : q4 ? 1 : 0][p.t - 2], mn = (double)p.M * p.N;
  const uint32_t forced = (uint32_t)g_tuning.gemm_ksplit;
  p.cost_us = 1e30;
  for (uint32_t ks = 1; ks <= 32; ++ks) {
    const uint32_t per = (blocks - 1) / (ks * kSepRowsK) + 1, ranges = (blocks - 1) / (per * kSepRowsK) + 1;
    const uint64_t all = (uint64_t)p.tiles * p.passes * ranges, full = (all - 1) / 256;
    if (ks > 1 && ((!forced && (all > 256 || per < 2)) || (uint64_t)ranges * p.M * p.N * 4 > partial_bytes)) break;
    if (forced && ks != forced && ks != 1) continue;
    double us = 10.7 + per * (block * (full + 1.0) + kFull[p.t - 2] * (full + (all - 256.0 * full) / 256.0)) + 2.2e-6 * mn + 2.1e-6 * p.M * p.K;
    if (ranges > 1) us += 1.33e-6 * ranges * mn;
    if (us < p.cost_us || ks == forced) {
      p.cost_us = us;
      p.per = per;
      p.nsplit = ranges;
    }
  }
  return sep_fits(p, (uint64_t)p.K * 2);
}

double sep_two_pass_us(uint32_t M, uint32_t K, uint32_t N);

// That way, or the weights written out as fp16 first (both estimated).  Not on a K below 512, where its waves have a block or two and the
// row tiles' code is most of the time: 64 x 256 x 256, us, two passes / this: int8 12.9 / 16.6, nibbles 13.1 / 14.7, affine 13.2 / 15.1;
// on int8 up to 512 x 512: 64 rows 14.5 / 15.5, 200 rows 15.3 / 15.8 (of 1024 x 512 16.6 / 16.2).
// (Nibbles of 11008 x 4096 and 14336 x 4096 from 350 rows on are up to 10 % faster in two passes by themselves, 512 rows 106 / 112, but a
// layer of 500 rows of the latter is 3 % slower so: the line by the estimates stays.)
bool sep_rows16_preferred(SepRowsParams &p, bool q4, bool affine, size_t partial_bytes) {
  const bool small = p.K < 512 || (!q4 && p.M >= 64 && p.K == 512 && p.N <= 512);
  return !small && sep_rows16_cut(p, q4, affine, partial_bytes) && p.cost_us < sep_two_pass_us(p.M, p.K, p.N);
}

template <int KIND> static int launch_kind(const SepRowsParams &p, uint32_t grid, hipStream_t stream) {
  if (p.t == 1) hipLaunchKernelGGL((sep_rows_kernel<KIND, 1>), dim3(grid), dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((sep_rows_kernel<KIND, 2>), dim3(grid), dim3(512), 0, stream, p);
  return check_hip(hipGetLastError(), "separated-layout row matmul launch");
}

int launch_sep_rows(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream) {
  const uint32_t grid = (uint32_t)sep_rows_grid(p);
  return affine ? launch_kind<kSepAffine>(p, grid, stream) : q4 ? launch_kind<kSepQ4>(p, grid, stream) : launch_kind<kSepQ8>(p, grid, stream);
}

template <int KIND, int T> static int launch_kind16(const SepRowsParams &p, uint32_t grid, hipStream_t stream) {
  auto kernel = sep_rows16_kernel<KIND, T>;
  if (T > 2) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, T * 32 * 1024),
                           "hipFuncSetAttribute"))
      return rc;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), T * 32 * 1024, stream, p);
  return check_hip(hipGetLastError(), "separated-layout row matmul launch");
}

template <int KIND> static int launch_tiles16(const SepRowsParams &p, uint32_t grid, hipStream_t stream) {
  return p.t == 2 ? launch_kind16<KIND, 2>(p, grid, stream) : p.t == 3 ? launch_kind16<KIND, 3>(p, grid, stream) : launch_kind16<KIND, 4>(p, grid, stream);
}

int launch_sep_rows16(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream) {
  const uint32_t grid = (uint32_t)sep_rows_grid(p);
  return affine ? launch_tiles16<kSepAffine>(p, grid, stream)
                : q4 ? launch_tiles16<kSepQ4>(p, grid, stream) : launch_tiles16<kSepQ8>(p, grid, stream);
}

}  // namespace cuthip
