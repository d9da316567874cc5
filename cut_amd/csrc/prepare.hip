// Load-time weight preparation on the GPU, for callers that keep the reference's
// separated [K, N] weight layout (cuthip_matmul_q8_sep / cuthip_matmul_q4_sep):
//   * GGUF blocks -> transposed separated tensors in one launch.  The reference
//     splits the blocks on the host (read_tensor_q8_separated / _q4_separated,
//     gguf_reader.cpp:389-501), uploads them and transposes on the GPU
//     (TransposeQ4Nibble.cu:17-61 for the nibbles, a generic transpose for the
//     int8 values and the scales; llama.cpp:940-965).
//   * Q4_K -> affine Q4 (requantizeQ4KToAffine, llama.cpp:573-619): per 32
//     elements scale = f16(d * sc), min = f16(8 * (d * sc) - dmin * m) (from the
//     unrounded scale), nibbles kept, written in the [K, N/2] orientation.
//   * fp32 rows -> Q8_0 blocks (quantizeRowsQ8_0, llama.cpp:488-505).
//
// All of it is byte shuffling bound by HBM.  A workgroup takes 256 elements of k of 128 (int8) or 256 (nibbles) weight
// rows, so that it writes runs of 128 bytes, whole cache lines.  It requests the blocks in 16-byte pieces (GGUF blocks are
// only 2-byte aligned), all of them before the first use, and puts the quants into LDS without the scales between them;
// then a thread reads a 16-byte piece of 4 (int8) or 8 (nibble) neighbouring rows, transposes 4 x 4 bytes at a time with
// v_perm_b32 and writes 16 (32) dwords.  14336 x 4096, us: Q8_0 52 -> 25, Q4_0 34 -> 15, Q4_K 38 -> 13.5 (before: 2-byte
// loads, one dword per row read from LDS, runs of 64 bytes for nibbles), all three 154 -> 67; with stores past the caches
// (nothing here reads the outputs back) 65, 4.0 TB/s.
#include <cstdint>

#include "common.hpp"

namespace cuthip {

constexpr int kPrepThreads = 256;
constexpr int kPrepK = 256;   // k extent of a tile

enum PrepMode { PREP_Q8_0 = 0, PREP_Q4_0 = 1, PREP_Q4_K_AFFINE = 2, PREP_NIBBLES = 3 };

// ROWS: weight rows of a tile.  PIECES: 16-byte pieces of a row's LDS image.  A row takes PIECES (made odd) x 16 bytes there
// and row r sits at (r % G) * 32 + r / G, G = rows of a transposition item: the 32 lanes that read row G * lane + j of
// their items then touch every bank once.
template <int MODE> struct PrepGeom {
  static constexpr int G = MODE == PREP_Q8_0 ? 4 : 8, ROWS = 32 * G;
  static constexpr int PIECES = MODE == PREP_Q8_0 ? 16 : MODE == PREP_Q4_K_AFFINE ? 9 : 8, PITCH = 16 * (PIECES | 1);
  static constexpr bool SCALES = MODE == PREP_Q8_0 || MODE == PREP_Q4_0;   // blocks of 32 with one fp16 scale
  static __device__ uint32_t slot(uint32_t row) { return (row % G) * 32 + row / G; }
};

struct PrepParams {
  const uint8_t *src;
  uint8_t *B;
  uint16_t *S;
  uint32_t N, K, strideB, scaleStride;
  uint32_t src_row_bytes;
  uint32_t tiles, ktiles, tiles_per_xcd;   // set by the launch
};

// 4 x 4 bytes: byte i of in[j] -> byte j of out[i]
__device__ __forceinline__ void transpose4(const uint32_t (&in)[4], uint32_t (&out)[4]) {
  const uint32_t t0 = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u), t1 = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);
  const uint32_t t2 = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u), t3 = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);
  out[0] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
  out[1] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
  out[2] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
  out[3] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
}

template <int MODE> __global__ void __launch_bounds__(kPrepThreads) prepare_sep_kernel(PrepParams p) {
  using G = PrepGeom<MODE>;
  __shared__ __attribute__((aligned(16))) uint8_t raw[G::ROWS * G::PITCH];
  __shared__ uint16_t sc[G::SCALES ? 8 * G::ROWS : 1];
  const uint32_t tid = threadIdx.x;
  // an XCD (block index modulo 8) walks along k before it goes to the next rows: the cache lines that two neighbouring
  // tiles of a row share are read once into its L2
  const uint32_t tile = (blockIdx.x & 7u) * p.tiles_per_xcd + (blockIdx.x >> 3);
  if (tile >= p.tiles) return;
  const uint32_t nt = tile / p.ktiles, n0 = nt * G::ROWS, k0 = (tile - nt * p.ktiles) * kPrepK;
  const uint32_t kt = min((uint32_t)kPrepK, p.K - k0);   // a multiple of 32

  // Rows past N and blocks past K read the last one instead and are not written.
  if constexpr (G::SCALES) {
    constexpr uint32_t BYTES = MODE == PREP_Q8_0 ? 34 : 18, Q = MODE == PREP_Q8_0 ? 2 : 1;   // Q: 16-byte pieces of quants
    constexpr int IT = 8 * G::ROWS / kPrepThreads;
    const uint32_t blk = tid & 7u, b = k0 / 32 + min(blk, kt / 32 - 1);
    u32x4 q[IT][Q];
    uint32_t d[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t n = min(n0 + it * 32u + (tid >> 3), p.N - 1);
      const uint8_t *src = p.src + (size_t)n * p.src_row_bytes + b * BYTES;
      d[it] = ld_u16(src);
#pragma unroll
      for (uint32_t u = 0; u < Q; ++u) q[it][u] = ld_u32x4(src + 2 + 16 * u);
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t row = it * 32u + (tid >> 3);
#pragma unroll
      for (uint32_t u = 0; u < Q; ++u) *reinterpret_cast<u32x4 *>(raw + G::slot(row) * G::PITCH + (blk * Q + u) * 16) = q[it][u];
      sc[blk * G::ROWS + row] = (uint16_t)d[it];
    }
  } else {
    constexpr uint32_t RUN = G::PIECES * 16;
    constexpr int IT = (G::ROWS * G::PIECES + kPrepThreads - 1) / kPrepThreads;
    static_assert(IT * kPrepThreads == G::ROWS * G::PIECES, "whole rounds of pieces");
    const uint32_t last = MODE == PREP_NIBBLES ? kt / 32 - 1 : G::PIECES - 1;
    const uint8_t *src = p.src + (size_t)(k0 / kPrepK) * RUN;
    u32x4 q[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t i = it * kPrepThreads + tid, row = i / G::PIECES, c = i - row * G::PIECES;
      q[it] = ld_u32x4(src + (size_t)min(n0 + row, p.N - 1) * p.src_row_bytes + min(c, last) * 16);
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const uint32_t i = it * kPrepThreads + tid, row = i / G::PIECES, c = i - row * G::PIECES;
      *reinterpret_cast<u32x4 *>(raw + G::slot(row) * G::PITCH + c * 16) = q[it];
    }
  }
  __syncthreads();

  const bool words = (p.strideB & 3u) == 0;
  const uint32_t lane = tid & 31u;   // rows G * lane .. of the tile
  const uint32_t col = (MODE == PREP_Q8_0 ? n0 : n0 / 2) + 4 * lane, cols = MODE == PREP_Q8_0 ? p.N : p.N / 2;
  auto put = [&](uint32_t k, uint32_t v) {   // columns col .. col + 3 of row k0 + k
    uint8_t *dst = p.B + (size_t)(k0 + k) * p.strideB + col;
    if (words && col + 3 < cols) {
      __builtin_nontemporal_store(v, reinterpret_cast<uint32_t *>(dst));   // nothing here reads it back
    } else {
      for (uint32_t j = 0; j < 4 && col + j < cols; ++j) dst[j] = (uint8_t)(v >> (8 * j));
    }
  };
  // Q8_0: piece c holds k = 16 c ..; nibbles: 32 k of block c, low half first (Q4_K: of 64 k, 16 low and 16 high ones)
  constexpr uint32_t QUANTS = MODE == PREP_Q8_0 ? 16 : 8, FIRST = MODE == PREP_Q4_K_AFFINE ? 1 : 0;
  for (uint32_t c = tid >> 5; c < QUANTS; c += kPrepThreads / 32) {
    const uint32_t k = MODE == PREP_Q8_0 ? 16 * c : MODE == PREP_Q4_K_AFFINE ? 64 * (c >> 1) + 16 * (c & 1) : 32 * c;
    if (k >= kt) break;
    u32x4 q[G::G];
#pragma unroll
    for (int j = 0; j < G::G; ++j) q[j] = *reinterpret_cast<const u32x4 *>(raw + (j * 32 + lane) * G::PITCH + (FIRST + c) * 16);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t in[4], out[4];
      if constexpr (MODE == PREP_Q8_0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) in[j] = q[j][w];
        transpose4(in, out);
#pragma unroll
        for (int e = 0; e < 4; ++e) put(k + 4 * w + e, out[e]);
      } else {
        constexpr uint32_t kLow = 0x0F0F0F0Fu, HIGH = MODE == PREP_Q4_K_AFFINE ? 32 : 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) in[j] = (q[2 * j][w] & kLow) | ((q[2 * j + 1][w] & kLow) << 4);   // even row in the low nibble
        transpose4(in, out);
#pragma unroll
        for (int e = 0; e < 4; ++e) put(k + 4 * w + e, out[e]);
#pragma unroll
        for (int j = 0; j < 4; ++j) in[j] = ((q[2 * j][w] >> 4) & kLow) | (q[2 * j + 1][w] & ~kLow);
        transpose4(in, out);
#pragma unroll
        for (int e = 0; e < 4; ++e) put(k + HIGH + 4 * w + e, out[e]);
      }
    }
  }
  if constexpr (G::SCALES) {
#pragma unroll
    for (int it = 0; it < 8 * G::ROWS / kPrepThreads; ++it) {
      const uint32_t i = it * kPrepThreads + tid, blk = i / G::ROWS, n = n0 + i % G::ROWS;
      if (n < p.N && blk * 32 < kt) __builtin_nontemporal_store(sc[i], &p.S[(size_t)(k0 / 32 + blk) * p.scaleStride + n]);
    }
  }
  if constexpr (MODE == PREP_Q4_K_AFFINE) {   // one thread per row: scales and minima of its eight sub-blocks
    static_assert(G::ROWS == kPrepThreads, "one row per thread");
    const uint32_t n = n0 + tid, blocksK = p.K / 32;
    if (n < p.N) {
      const u32x4 h = *reinterpret_cast<const u32x4 *>(raw + G::slot(tid) * G::PITCH);
      const float d = f16bits_to_f32(h.x & 0xFFFFu), dmin = f16bits_to_f32(h.x >> 16);
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t sh = 8 * (j & 3);
        uint32_t s, m;   // get_scale_min_k4 (llama.cpp:547-555) on the packed bytes h.y, h.z, h.w
        if (j < 4) {
          s = (h.y >> sh) & 63u;
          m = (h.z >> sh) & 63u;
        } else {
          s = ((h.w >> sh) & 15u) | (((h.y >> (sh + 6)) & 3u) << 4);
          m = ((h.w >> (sh + 4)) & 15u) | (((h.z >> (sh + 6)) & 3u) << 4);
        }
        // both products are exact in fp32 (11 x 6 bits), so the subtraction is the only rounding whether or not it is fused
        const float scale = d * (float)s;
        const float minv = 8.0f * scale - dmin * (float)m;
        const size_t b = k0 / 32 + j;
        __builtin_nontemporal_store((uint16_t)f32_to_f16bits_any(scale), &p.S[b * p.scaleStride + n]);
        __builtin_nontemporal_store((uint16_t)f32_to_f16bits_any(minv), &p.S[(blocksK + b) * p.scaleStride + n]);
      }
    }
  }
}

template <int MODE> static int launch_prepare(PrepParams p, hipStream_t stream) {
  using G = PrepGeom<MODE>;
  p.ktiles = (p.K - 1) / kPrepK + 1;
  const uint64_t tiles = (uint64_t)((p.N - 1) / G::ROWS + 1) * p.ktiles;
  if ((p.K - 1) / (MODE == PREP_Q8_0 ? 128 : 256) >= 65535u || tiles > 0x7FFFFFF0ull) {
    set_error("prepare: K = %u is too long for one launch", p.K);
    return CUTHIP_ERR_INVALID;
  }
  p.tiles = (uint32_t)tiles;
  p.tiles_per_xcd = (p.tiles + 7) / 8;
  hipLaunchKernelGGL(prepare_sep_kernel<MODE>, dim3(8 * p.tiles_per_xcd), dim3(kPrepThreads), 0, stream, p);
  return check_hip(hipGetLastError(), "prepare launch");
}

// 8 lanes per block of 32 values: 16-byte loads, absmax folded over the 8 lanes, one dword of int8 per lane
__global__ void __launch_bounds__(256) quantize_q8_0_kernel(const float *x, uint64_t nblocks, uint8_t *blocks) {
  const uint64_t t = (uint64_t)blockIdx.x * 256u + threadIdx.x, b = t >> 3;
  const uint32_t i = (uint32_t)t & 7u;
  const bool ok = b < nblocks;
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (ok) v = *reinterpret_cast<const f32x4 *>(x + b * 32 + i * 4);
  float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  const float d = amax / 127.0f;                      // correctly rounded fp32 division, as on the host
  const float id = d != 0.0f ? 1.0f / d : 0.0f;
  // lroundf: half away from zero; |x * id| <= 127 * (1 + 2^-22), so the cast cannot overflow int8
  const uint32_t q0 = (uint32_t)(int)roundf(v.x * id) & 0xFFu, q1 = (uint32_t)(int)roundf(v.y * id) & 0xFFu;
  const uint32_t q2 = (uint32_t)(int)roundf(v.z * id) & 0xFFu, q3 = (uint32_t)(int)roundf(v.w * id) & 0xFFu;
  if (!ok) return;
  uint8_t *blk = blocks + b * 34;
  uint16_t *dst = reinterpret_cast<uint16_t *>(blk + 2 + 4 * i);   // blocks are 2-byte aligned
  dst[0] = (uint16_t)(q0 | (q1 << 8));
  dst[1] = (uint16_t)(q2 | (q3 << 8));
  if (i == 0) *reinterpret_cast<uint16_t *>(blk) = (uint16_t)f32_to_f16bits_any(d);
}

}  // namespace cuthip

using namespace cuthip;

extern "C" {

int cuthip_prepare_sep(int fmt, const void *blocks, uint32_t N, uint32_t K, void *B, uint32_t strideB, uint16_t *scales,
                       uint32_t scaleStride, void *stream) {
  if (!blocks || !B || !scales) {
    set_error("cuthip_prepare_sep: null pointer");
    return CUTHIP_ERR_INVALID;
  }
  if (fmt != CUTHIP_Q8_0 && fmt != CUTHIP_Q4_0 && fmt != CUTHIP_Q4_K) {
    set_error("cuthip_prepare_sep: format %d has no separated layout (Q8_0, Q4_0 and Q4_K -> affine Q4 do)", fmt);
    return CUTHIP_ERR_INVALID;
  }
  if (N == 0 || K == 0 || K % (uint32_t)fmt_elems(fmt) != 0) {
    set_error("cuthip_prepare_sep: K = %u must be a positive multiple of %d, N = %u positive", K, fmt_elems(fmt), N);
    return CUTHIP_ERR_INVALID;
  }
  const bool q4 = fmt != CUTHIP_Q8_0;
  if (q4 && (N & 1u)) {   // TransposeQ4NibbleOp.cpp:13-15, llama.cpp:576
    set_error("cuthip_prepare_sep: N = %u must be even for packed nibbles", N);
    return CUTHIP_ERR_INVALID;
  }
  if (strideB < (q4 ? N / 2 : N) || scaleStride < N) {
    set_error("cuthip_prepare_sep: strideB = %u / scaleStride = %u shorter than a row of N = %u", strideB, scaleStride, N);
    return CUTHIP_ERR_INVALID;
  }
  if ((reinterpret_cast<uintptr_t>(B) & 3u) || (reinterpret_cast<uintptr_t>(scales) & 1u) ||
      (reinterpret_cast<uintptr_t>(blocks) & 1u)) {
    set_error("cuthip_prepare_sep: B must be 4-byte aligned, blocks and scales 2-byte aligned");
    return CUTHIP_ERR_INVALID;
  }
  PrepParams p{};
  p.src = reinterpret_cast<const uint8_t *>(blocks);
  p.B = reinterpret_cast<uint8_t *>(B);
  p.S = scales;
  p.N = N; p.K = K; p.strideB = strideB; p.scaleStride = scaleStride;
  p.src_row_bytes = K / (uint32_t)fmt_elems(fmt) * (uint32_t)fmt_bytes(fmt);
  if (fmt == CUTHIP_Q8_0) return launch_prepare<PREP_Q8_0>(p, (hipStream_t)stream);
  if (fmt == CUTHIP_Q4_0) return launch_prepare<PREP_Q4_0>(p, (hipStream_t)stream);
  return launch_prepare<PREP_Q4_K_AFFINE>(p, (hipStream_t)stream);
}

int cuthip_transpose_q4_nibble(const void *packed, void *packedT, uint32_t N, uint32_t K, uint32_t strideInHalf,
                               uint32_t strideOutHalf, void *stream) {
  if (!packed || !packedT) {
    set_error("cuthip_transpose_q4_nibble: null pointer");
    return CUTHIP_ERR_INVALID;
  }
  if (N == 0 || (N & 1u)) {
    set_error("TransposeQ4: N must be even");
    return CUTHIP_ERR_INVALID;
  }
  if (K == 0 || K % 32 != 0) {
    set_error("TransposeQ4: K must be a multiple of 32");
    return CUTHIP_ERR_INVALID;
  }
  if (strideInHalf < K / 2 || (strideInHalf & 1u) || strideOutHalf < N / 2) {
    set_error("cuthip_transpose_q4_nibble: strideInHalf = %u (even, >= K/2) / strideOutHalf = %u (>= N/2) do not fit", strideInHalf,
              strideOutHalf);
    return CUTHIP_ERR_INVALID;
  }
  if ((reinterpret_cast<uintptr_t>(packedT) & 3u) || (reinterpret_cast<uintptr_t>(packed) & 1u)) {
    set_error("cuthip_transpose_q4_nibble: output must be 4-byte aligned, input 2-byte aligned");
    return CUTHIP_ERR_INVALID;
  }
  PrepParams p{};
  p.src = reinterpret_cast<const uint8_t *>(packed);
  p.B = reinterpret_cast<uint8_t *>(packedT);
  p.S = nullptr;
  p.N = N; p.K = K; p.strideB = strideOutHalf; p.scaleStride = 0;
  p.src_row_bytes = strideInHalf;
  // only K / 2 bytes of a padded row are nibbles: the kernel stops at K
  return launch_prepare<PREP_NIBBLES>(p, (hipStream_t)stream);
}

int cuthip_quantize_rows_q8_0(const float *x, uint64_t n, void *blocks, void *stream) {
  if (!x || !blocks) {
    set_error("cuthip_quantize_rows_q8_0: null pointer");
    return CUTHIP_ERR_INVALID;
  }
  if (n == 0 || n % 32 != 0) {
    set_error("cuthip_quantize_rows_q8_0: n = %llu must be a positive multiple of 32", (unsigned long long)n);
    return CUTHIP_ERR_INVALID;
  }
  if ((reinterpret_cast<uintptr_t>(x) & 15u) || (reinterpret_cast<uintptr_t>(blocks) & 1u)) {
    set_error("cuthip_quantize_rows_q8_0: x must be 16-byte aligned, blocks 2-byte aligned");
    return CUTHIP_ERR_INVALID;
  }
  const uint64_t nblocks = n / 32, wgs = (nblocks * 8 + 255) / 256;
  if (wgs > 0x7FFFFFFFull) {
    set_error("cuthip_quantize_rows_q8_0: n = %llu is too large for one launch", (unsigned long long)n);
    return CUTHIP_ERR_INVALID;
  }
  hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((uint32_t)wgs), dim3(256), 0, (hipStream_t)stream, x, nblocks,
                     reinterpret_cast<uint8_t *>(blocks));
  return check_hip(hipGetLastError(), "quantize launch");
}

}  // extern "C"
