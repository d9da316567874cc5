// Streaming matmul on Q4_K and Q8_0 blocks for a handful of activation rows (M <= 32):
//   C[m,n] = sum_k A[m,k] * dequant(W)[n,k]
// between the 8-row GEMV (whose matrix-core path spends three quarters of every product on mismatched pieces)
// and the row-tile matmul (which rounds every weight to fp16).
// Supersedes MatMulQ4GemvKPar8.cu / MatMulQ4TiledReg.cu (operators/impl/matmul) at these batch sizes.
//
// Q4_K.  Two waves share 16 weight rows and each walks half of the workgroup's K range in steps of one 256-element
// super-block.  v_mfma_f32_16x16x32_f16 multiplies the 16 (or 32) activation rows with the 16 weight rows: lane l holds weights
// of row l & 15, 16 bytes of either half of the quants (32 nibbles of two sub-blocks each).  The nibbles are turned into fp16
// without a conversion: an integer q in the low bits of a half IS the subnormal q * 2^-24, and four bits up q * 2^-20; the 6-bit
// scale of the sub-block (for the upper nibbles a sixteenth of it) is multiplied in as fp16, q * sc below 1024 in units of 2^-24, exact.
// A mask thus takes two weights out of a dword, the eighth byte apart (the activations lie in LDS in that order), and all eight
// sub-blocks accumulate in one MFMA chain; the fp32 super-block scale d * 2^24 is applied once per step.  The "- dmin * m" term needs
// only the activations' sums over the sub-blocks: they are formed once, while the activations are staged, as two halves (the second
// what rounding to the first leaves, with its sign: 24 bits together), and one MFMA multiplies those of a super-block with the eight 6-bit minima.  Products and sums are therefore those of the
// fp32 reference expression (d * sc) * q - dmin * m up to the order of the fp32 additions: 3e-7 normwise against 64 bits, where a
// chain of products with the minima, which cancels against the first, had 1e-6 to 3e-6.
//
// Q8_0.  A step is eight blocks of 34 bytes.  Lane l holds bytes 8 (l >> 4) .. + 7 of a block, as the halves 1024 + (q + 128) less 1152,
// one MFMA multiplies a block, and its four sums are scaled by the block's fp32 d: again the reference's expression, 1e-7 to 3e-7
// against 64 bits (the row-tile matmul, on d q rounded to fp16: 2e-4).
//
// Activations are staged once per workgroup as fp16 rows in LDS (fp32 inputs rounded to nearest even), row pitch
// = range + 16 bytes so that the 16 rows of a fragment read hit different banks; the K range of a workgroup is
// bounded by LDS (132 KB of activations), longer rows are split over workgroups (fp32 partial products, summed by the reduce kernel
// of the two-pass GEMM, which applies the epilogue).  After the staging barrier the loop has no barrier: each lane
// keeps kStreamDepth steps of weight loads in flight in a register ring and waits only for the step it multiplies.
//
// Q4_K is bound by the vector instructions of the unpack (47 % of the time at 16 and at 32 rows) and by the staging in front of the loop
// (waits 43 %), well before HBM (2.6 TB/s); Q8_0 by HBM (3.5 of the 4.8 TB/s of a copy) beside 31 to 34 % of vector instructions and LDS
// bank conflicts in the strip (15 to 19 %).  Measured (MI355X, HIP-graph replay, fp16 activations): Q4_K 14336 x 4096 at 9 / 16 / 24 / 32
// rows 12.4 / 12.7 / 17.0 / 17.2 us (with eight pieces of 8 bytes per lane, integer products and the minima as a second chain of eight
// products 14.1 / 14.5 / 19.7 / 19.9), 28672 x 4096 23.2 / 23.6 / 28.4 / 29.7 (25.3 / 25.9 / 33.7 / 34.1), 4096 x 4096 8.5 / 8.8 / 10.3 /
// 10.3 (11.2 / 11.6 / 13.2 / 13.7).  A sum per piece as it is staged, every fourth thread storing one, took back 1.5 us of it at 16 rows
// and 2 at 32: hence four pieces at a time, a sum to every thread.  Q8_0 14336 x 4096 at 8 / 16 / 24 / 32 rows 17.6 / 17.8 / 21.6 / 22.3 us
// (8-row GEMV 19.8, row-tile matmul 22.7 / 22.6 / 23.0), 4096 x 14336 19.6 / 20.3 / 22.1 / 22.1 (20.7; 22.6 / 23.1 / 23.8), 28672 x 4096
// at 8 / 16 rows 32.6 / 32.7 (36.1; 37.3).  Q4_K at 8 rows and fewer: the 8-row GEMV is as fast for the widest matrices and faster for
// all others.
#include <type_traits>

#include "common.hpp"

namespace cuthip {

int launch_splitk_reduce(const float *partial, uint32_t ksplit, uint32_t M, uint32_t N, void *C, uint32_t strideC, Epilogue epi,
                         int c_f16, hipStream_t stream);

struct StreamParams {
  const uint8_t *W;
  const void *A;
  void *C;
  Epilogue epi;
  uint32_t M, K, N, strideA, strideC, row_bytes;
  int a_f16, c_f16;
  uint32_t nblocks;       // workgroups along N (16 RG weight rows each)
  uint32_t range_steps;   // 256-element steps per K range
  uint32_t ksplit;
  float *partial;         // [ksplit][M][N] when ksplit > 1
};

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) uint8_t lds_u8s;

constexpr int kStreamDepth = 2;   // steps of weight loads in flight per lane (14336 x 4096 at 16 rows, two / three / four: Q4_K 12.7 / 13.0 / 13.5 us, Q8_0 17.8 / 20.0 / 23.9)
constexpr uint32_t kStripBytes = 144 * 16;          // LDS per wave for the blocks of a step
constexpr uint32_t kStreamLdsMax = 132 * 1024;     // staged activations: 16 rows of 4096 (the strips of eight waves and the sums take 26 KB more)

__device__ __forceinline__ half2_t as_pair(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
__device__ __forceinline__ uint32_t bits(half2_t v) { return __builtin_bit_cast(uint32_t, v); }
// the value of the lane whose number differs in bit 0 (quad_perm 1 0 3 2) / bit 1 (2 3 0 1)
__device__ __forceinline__ float lane_xor1(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_xor2(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));
}
__device__ __forceinline__ half8_t as_frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(half8_t, u32x4{a, b, c, d});
}

// MT: activation tiles of 16 rows (1 or 2); RG: groups of 16 weight rows per workgroup; KW: waves that share a group,
// each on its own part of the steps.  RG x KW = 8 waves wherever the range is long enough (two waves per SIMD: one
// wave alone cannot hide its own LDS and matrix-core latencies).
template <int FMT, int SB, int MT, int KW, int RG>
__global__ void __launch_bounds__(64 * RG * KW) gemm_stream_kernel(StreamParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int D = kStreamDepth, THREADS = 64 * RG * KW;
  constexpr bool Q4K = FMT == CUTHIP_Q4_K;
  constexpr int NP = Q4K ? 3 : 5;   // 16-byte pieces per lane and step
  const uint32_t split = blockIdx.x / p.nblocks, bid = blockIdx.x - split * p.nblocks;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), rg = wave % RG, kw = wave / RG;
  const uint32_t s_lo = split * p.range_steps, nsteps = p.K / 256;
  const uint32_t rcnt = min(p.range_steps, nsteps - s_lo);   // steps of this workgroup; the host launches no empty range
  const uint32_t range_k = rcnt * 256, pitch = range_k * 2 + 16;   // bytes per staged activation row
  // behind the activations: the sums of their sub-blocks, [row][step][lane group][4 halves], then the weight strips
  const uint32_t sums0 = 16 * MT * (p.range_steps * 512 + 16), spitch = range_k / 8 + 16;
  const uint32_t strip0 = sums0 + (Q4K ? 16 * MT * (p.range_steps * 32 + 16) : 0);
  const uint32_t sb = rcnt * kw / KW, cnt = rcnt * (kw + 1) / KW - sb;   // this wave's steps: [sb, sb + cnt) of the range

  const uint32_t n = (bid * RG + rg) * 16 + (lane & 15), kq = lane >> 4;

  // The 16 blocks of a step (16 rows x 144 bytes) are fetched as 144 pieces of 16 bytes, piece c = row c / 9, part
  // c % 9, by lanes c, c - 64, c - 128: neighbouring lanes read neighbouring bytes, every cache line is requested
  // once.  (Fetched in the operand layout - 8 bytes per lane, the four lanes of a row 16 lanes apart - every line
  // was requested four times: 17.6 us against 15.7 for 14336 x 4096 at 16 rows.)  The pieces go through a wave-private
  // strip of LDS, from which each lane picks its row's header and its 16 bytes of either half of the quants.
  // Q8_0 (17 pieces a row): parts 0-7, parts 9-16 and, by 16 lanes, part 8 of every row, as the strip holds half a step at a time.
  constexpr uint32_t kStepBytes = Q4K ? 144 : 272;
  const uint8_t *piece[NP];
  uint32_t slot[NP];   // where the piece goes in the strip: 144 bytes a row
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const uint32_t c = min((uint32_t)lane + 64u * j, Q4K ? 143u : 271u);
    const uint32_t r = Q4K ? c / 9 : j < 4 ? c / 8 % 16 : c - 256, part = Q4K ? c - 9 * r : j < 4 ? c % 8 + (j < 2 ? 0 : 9) : 8;
    piece[j] = p.W + (size_t)min((bid * RG + rg) * 16 + r, p.N - 1) * p.row_bytes + (size_t)(s_lo + sb) * kStepBytes + 16 * part;
    slot[j] = r * 144 + 16 * (part < 9 ? part : part - 8);
  }
  struct Raw { u32x4 c[NP]; };
  auto load = [&](Raw &r, uint32_t step) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NP; ++j) r.c[j] = ld_u32x4(piece[j] + (size_t)step * kStepBytes);
  };

  // activations first (they must not queue behind the weight loads), in batches of SB 16-byte pieces per thread;
  // the weight ring is requested behind the first batch
  const uint32_t cpr = range_k / 8, chunks = p.M * cpr;   // 8-element pieces per row, in all
  const uint32_t k_lo = s_lo * 256;
  const uint32_t inv = 0xFFFFFFFFu / cpr + 1;   // c / cpr = c inv >> 32: exact, as c (inv cpr - 2^32) < chunks cpr < 2^32
  u32x4 xa[SB], xb[SB];
  auto stage_load = [&](uint32_t base) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SB; ++i) {
      const uint32_t c = min(base + (uint32_t)i * THREADS + (uint32_t)tid, chunks - 1), r = __umulhi(c, inv), col = c - r * cpr;
      const size_t off = (size_t)r * p.strideA + k_lo + col * 8;
      if (p.a_f16) {
        xa[i] = ld_u32x4(reinterpret_cast<const uint8_t *>(p.A) + off * 2);
      } else {
        xa[i] = ld_u32x4(reinterpret_cast<const uint8_t *>(p.A) + off * 4);
        xb[i] = ld_u32x4(reinterpret_cast<const uint8_t *>(p.A) + off * 4 + 16);
      }
    }
  };
  // Four pieces of a thread at a time: four neighbouring threads hold the four pieces of four sub-blocks of 32, and each of
  // them takes one sub-block's sum
  auto stage_store = [&](uint32_t base) __attribute__((always_inline)) {
    const half2_t one{(half_t)1.0f, (half_t)1.0f};
    const bool b0 = tid & 1, b1 = tid & 2;
#pragma unroll
    for (int i0 = 0; i0 < SB; i0 += 4) {
      if (base + (uint32_t)i0 * THREADS >= chunks) break;
      float sum[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + j;
        const uint32_t c = base + (uint32_t)i * THREADS + (uint32_t)tid;
        u32x4 o = xa[i];
        if (!p.a_f16) {
          const f32x4 lo = __builtin_bit_cast(f32x4, xa[i]), hi = __builtin_bit_cast(f32x4, xb[i]);
          const half8_t h{(half_t)lo.x, (half_t)lo.y, (half_t)lo.z, (half_t)lo.w, (half_t)hi.x, (half_t)hi.y, (half_t)hi.z, (half_t)hi.w};
          o = __builtin_bit_cast(u32x4, h);
        }
        if (Q4K) {
          sum[j] = __builtin_amdgcn_fdot2(as_pair(o.x), one, 0.0f, false);
          sum[j] = __builtin_amdgcn_fdot2(as_pair(o.y), one, sum[j], false);
          sum[j] = __builtin_amdgcn_fdot2(as_pair(o.z), one, sum[j], false);
          sum[j] = __builtin_amdgcn_fdot2(as_pair(o.w), one, sum[j], false);
        }
        if (c < chunks) {
          const uint32_t r = __umulhi(c, inv), col = c - r * cpr;
          // Q4_K: elements 0 2 1 3 4 6 5 7, the order in which a mask takes two nibbles out of a dword
          *reinterpret_cast<u32x4 *>(lds + r * pitch + col * 16) = !Q4K ? o :
              u32x4{__builtin_amdgcn_perm(o.y, o.x, 0x05040100u), __builtin_amdgcn_perm(o.y, o.x, 0x07060302u),
                    __builtin_amdgcn_perm(o.w, o.z, 0x05040100u), __builtin_amdgcn_perm(o.w, o.z, 0x07060302u)};
        }
      }
      if (!Q4K) continue;
      const float s01 = (b0 ? sum[1] : sum[0]) + lane_xor1(b0 ? sum[0] : sum[1]), s23 = (b0 ? sum[3] : sum[2]) + lane_xor1(b0 ? sum[2] : sum[3]);
      const float s = ((b1 ? s23 : s01) + lane_xor2(b1 ? s01 : s23)) * 0.03125f;   // of this thread's sub-block, / 32
      const uint32_t c = base + (uint32_t)(i0 + (tid & 3)) * THREADS + (uint32_t)(tid & ~3);
      if (c < chunks) {
        // in two parts (24 bits together): part h of sub-block j of a step to lane group 2 ((j >> 1) & 1) + h
        const uint32_t r = __umulhi(c, inv), col = c - r * cpr, j = (col >> 2) & 7;
        half_t *dst = reinterpret_cast<half_t *>(lds + sums0 + r * spitch + (col >> 5) * 32 + 16 * ((j >> 1) & 1)) + 2 * (j >> 2) + (j & 1);
        const half_t lead = (half_t)s;
        dst[0] = lead;
        dst[4] = (half_t)((s - (float)lead) * 2048.0f);
      }
    }
  };
  stage_load(0);
  Raw buf[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    load(buf[i], min((uint32_t)i, cnt ? cnt - 1 : 0u));
    __builtin_amdgcn_sched_barrier(0);   // issue order = ring order: step i waits for its own loads only
  }
  stage_store(0);
  for (uint32_t base = SB * THREADS; base < chunks; base += SB * THREADS) {
    stage_load(base);
    stage_store(base);
  }
  __syncthreads();

  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0, 0, 0, 0};
  // Lane (n, kq) multiplies bytes 16 kq .. + 15 of each half (64 bytes) of its row's quants: in half t sub-blocks 4 t + 2 p (low
  // nibbles) and 4 t + 2 p + 1, p = kq >> 1, elements 16 (kq & 1) .. + 15.  Fragment f = 4 t + 2 (high nibbles) + u of activation tile
  // i: row 16 i + (lane & 15), elements 128 t + 64 p + 32 (high) + 16 (kq & 1) + 8 u .. + 7 of the step; rows at and beyond M
  // hold whatever the LDS held: their products land in accumulator rows that are never stored
  const lds_u8s *xbase = (const lds_u8s *)(lds) + (size_t)(lane & 15) * pitch + 128 * (kq >> 1) + 32 * (kq & 1);
  const lds_u8s *sbase = (const lds_u8s *)(lds) + sums0 + (size_t)(lane & 15) * spitch + 8 * kq;
  const half_t part = (half_t)(kq & 1 ? 1.0f : 2048.0f);

  // wave-private strip: the 144 pieces of a step
  lds_u8s *strip = (lds_u8s *)(lds) + strip0 + (size_t)wave * kStripBytes;
  struct Blk { u32x4 hdr, q[2]; };   // what a lane multiplies in a step: its row's header, 16 bytes of each half of the quants
  // pieces of a step -> strip -> the lane's operands (same wave, LDS in order: the strip's earlier reads are done);
  // issuing this a step ahead of the products measured no different
  auto deliver = [&](const Raw &raw, Blk &r) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<lds_u32x4 *>(strip + ((size_t)lane + 64 * j) * 16) = raw.c[j];
    if (lane < 16) *reinterpret_cast<lds_u32x4 *>(strip + ((size_t)lane + 128) * 16) = raw.c[2];
    __builtin_amdgcn_wave_barrier();
    const lds_u8s *blk = strip + (size_t)(lane & 15) * 144;
    r.hdr = *reinterpret_cast<const lds_u32x4 *>(blk);
#pragma unroll
    for (int t = 0; t < 2; ++t) r.q[t] = *reinterpret_cast<const lds_u32x4 *>(blk + 16 + 64 * t + 16 * kq);
    __builtin_amdgcn_wave_barrier();
  };
  auto do_step = [&](const Blk &r, uint32_t step) __attribute__((always_inline)) {
    // scales and minima of the lane's four sub-blocks: bytes 2 p, 2 p + 1 of either half of the header's 6-bit fields
    const uint32_t sh = 16 * (kq >> 1), a0 = r.hdr.y >> sh, a1 = r.hdr.z >> sh, a2 = r.hdr.w >> sh;
    const uint32_t s6[2] = {a0 & 0x3F3Fu, (a2 & 0x0F0Fu) | ((a0 >> 2) & 0x3030u)};
    const uint32_t m6[2] = {a1 & 0x3F3Fu, ((a2 >> 4) & 0x0F0Fu) | ((a1 >> 2) & 0x3030u)};
    half2_t sc[2];   // (scale, scale / 16): 1024 + s in the low bits of a half
    uint32_t mn[2];  // min * 2^-24, or for the leading parts of the sums * 2^-13
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = __builtin_elementwise_fma(as_pair(__builtin_amdgcn_perm(0x64646464u, s6[t], 0x04010400u)), half2_t{(half_t)1.0f, (half_t)0.0625f},
                                        half2_t{(half_t)-1024.0f, (half_t)-64.0f});
      mn[t] = bits(as_pair(__builtin_amdgcn_perm(0u, m6[t], 0x0C010C00u)) * half2_t{part, part});
    }
    const lds_u8s *xs = xbase + (size_t)(sb + step) * 512, *ss = sbase + (size_t)(sb + step) * 32;
    f32x4 t_main[MT], t_min[MT];
    const f32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const u32x2 x = *reinterpret_cast<const __attribute__((address_space(3))) u32x2 *>(ss + (size_t)i * 16 * spitch);
      t_min[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_frag(x.x, x.y, 0, 0), as_frag(mn[0], mn[1], 0, 0), zero, 0, 0, 0);
    }
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      // nibbles of bits 0-3 are q 2^-24, of bits 4-7 q 2^-20; times the scale (scale / 16) an integer below 1024 times 2^-24
      const uint32_t mask = f & 2 ? 0x00F000F0u : 0x000F000Fu;
      const half_t k = sc[f >> 2][(f >> 1) & 1];
      const uint32_t w0 = r.q[f >> 2][2 * (f & 1)], w1 = r.q[f >> 2][2 * (f & 1) + 1];
      const half2_t kk{k, k};
      const half8_t w = as_frag(bits(as_pair(w0 & mask) * kk), bits(as_pair((w0 >> 8) & mask) * kk), bits(as_pair(w1 & mask) * kk), bits(as_pair((w1 >> 8) & mask) * kk));
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const half8_t x = *reinterpret_cast<const __attribute__((address_space(3))) half8_t *>(xs + (size_t)i * 16 * pitch + 256 * (f >> 2) + 64 * ((f >> 1) & 1) + 16 * (f & 1));
        t_main[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w, f == 0 ? zero : t_main[i], 0, 0, 0);
      }
    }
    // the sums are of x / 32, in units of 2^-13
    const float d = f16bits_to_f32(r.hdr.x & 0xFFFF) * 16777216.0f, dmin = f16bits_to_f32(r.hdr.x >> 16) * 262144.0f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] = fmaf(-dmin, t_min[i][e], fmaf(d, t_main[i][e], acc[i][e]));
  };

  // Q8_0, half a step (four blocks of 34 bytes) at a time: the first half lies in parts 0-8 of a row, the second 8 bytes into parts 8-16.
  // Lane (n, kq) multiplies bytes 8 kq .. + 7 of every block with elements 32 b + 8 kq .. + 7 of the step.
  auto q8_step = [&](const Raw &raw, uint32_t step) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    const lds_u8s *xs = (const lds_u8s *)(lds) + (size_t)(lane & 15) * pitch + 16 * kq + (size_t)(sb + step) * 512;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; ++j) *reinterpret_cast<lds_u32x4 *>(strip + slot[2 * h + j]) = raw.c[2 * h + j];
      if (lane < 16) *reinterpret_cast<lds_u32x4 *>(strip + slot[NP - 1] - 128 * h) = raw.c[NP - 1];
      __builtin_amdgcn_wave_barrier();
      uint32_t q[4][3];
      float d[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const lds_u8s *blk = strip + (size_t)(lane & 15) * 144 + 8 * h + 34 * b;
        d[b] = f16bits_to_f32(*reinterpret_cast<const __attribute__((address_space(3))) uint16_t *>(blk));
        // the quants begin two bytes into a dword in the even blocks
#pragma unroll
        for (int w = 0; w < (b & 1 ? 2 : 3); ++w) q[b][w] = *reinterpret_cast<const lds_u32 *>(blk + (b & 1 ? 2 : 0) + 8 * kq + 4 * w);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        // a byte q + 128 below 0x64 is the half 1024 + q + 128
        const half2_t bias{(half_t)-1152.0f, (half_t)-1152.0f};
        uint32_t u[3];
#pragma unroll
        for (int w = 0; w < (b & 1 ? 2 : 3); ++w) u[w] = q[b][w] ^ 0x80808080u;
        uint32_t f[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t w = b & 1 ? u[k / 2] : u[(k + 1) / 2];
          const bool upper = b & 1 ? k & 1 : !(k & 1);
          f[k] = bits(as_pair(__builtin_amdgcn_perm(0x64646464u, w, upper ? 0x04030402u : 0x04010400u)) + bias);
        }
        const half8_t w = as_frag(f[0], f[1], f[2], f[3]);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const half8_t x = *reinterpret_cast<const __attribute__((address_space(3))) half8_t *>(xs + (size_t)i * 16 * pitch + 256 * h + 64 * b);
          const f32x4 t = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w, f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] = fmaf(d[b], t[e], acc[i][e]);
        }
      }
    }
  };

  // Ring slot i % D holds the pieces of step i.  With no load under a condition the compiler counts the loads in flight exactly and
  // every step waits for its own pieces only: the last D steps, which request nothing, stand by themselves (requested past
  // the end of the range, at its last step again, their pieces cost Q8_0 2 to 3 %).
  const uint32_t last = cnt ? cnt - 1 : 0u;
  auto multiply = [&](const Raw &raw, uint32_t i) __attribute__((always_inline)) {
    if constexpr (Q4K) {
      Blk blk;
      deliver(raw, blk);
      do_step(blk, i);
    } else {
      q8_step(raw, i);
    }
  };
  uint32_t i0 = 0;
  for (; i0 + D < cnt; i0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      multiply(buf[u], i0 + u);
      load(buf[u], min(i0 + u + D, last));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (i0 + u < cnt) multiply(buf[u], i0 + u);   // uniform
  // the K parts of a row group meet in LDS (the staged activations are no longer needed)
  if constexpr (KW > 1) {
    __syncthreads();
    // [KW - 1][RG row groups][MT * 4 registers][64 lanes]
    float *red = reinterpret_cast<float *>(lds) + ((size_t)(kw > 0 ? kw - 1 : 0) * RG + rg) * 64 * MT * 4 + lane;
    if (kw > 0) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[(t * 4 + e) * 64] = acc[t][e];
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int w = 1; w < KW; ++w)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] += red[((size_t)(w - 1) * RG * 64 * MT * 4) + (t * 4 + e) * 64];
  }
  // accumulator register e of lane l, tile t: row 16 t + 4 (l >> 4) + e, column (weight row) n
  if (p.epi.kind == CUTHIP_EPI_SWIGLU_PAIRS) {   // (never with several K ranges) gate in the even weight rows, up in the odd ones
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t m = 16 * t + 4 * kq + e;
        const float up = lane_xor1(acc[t][e]);
        if ((n & 1) == 0 && n + 1 < p.N && m < p.M)
          store_plain(p.C, p.c_f16, (size_t)m * p.strideC + n / 2, apply_unary(CUTHIP_UNARY_SILU, acc[t][e]) * up);
      }
  } else if (n < p.N) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t m = 16 * t + 4 * kq + e;
        if (m < p.M) {
          if (p.ksplit > 1) p.partial[((size_t)split * p.M + m) * p.N + n] = acc[t][e];
          else store_out(p.C, p.epi, p.c_f16, (size_t)m * p.strideC + n, acc[t][e]);
        }
      }
  }
}

// K ranges of the streaming kernel: as few as LDS allows (one range of up to kStreamLdsMax bytes of staged
// activations), more where the workgroups still run at once, one to a CU, a range keeps at least 4 steps (Q4_K at 16 / 32 rows, one
// range in the place of two: 4096 x 4096 10.3 / 12.4 us and 9.4 / 10.7, 2048 x 8192 10.3 / 12.4 and 9.4 / 10.8; of eight steps in all only
// with two activation tiles: 4096 x 2048 8.0 / 10.0 and 8.4 / 9.7; beyond 256 workgroups, which then run in two rounds, 10240 x 4096 at
// 16 rows 12.6 in one range and 16.5 in two, Q8_0 17.6 and 21.7), and the scratch memory
// holds the partial products of twice as many.  (A workgroup that stages one range after the other, without partial
// products, needs the registers of the staging beside those of the loop: 35.9 us against 30.0 for 28672 x 4096 at 32 rows.)
// Weight rows per workgroup: 64 (four row groups, two waves each), or with two activation tiles 128 (eight row groups
// of one wave: half as many workgroups stage the activations; 14336 x 4096 at 32 rows 17.9 us) wherever that
// still leaves a workgroup for every second CU (4096 x 4096 at 32 rows: 12.6 us with 64)
static uint32_t stream_block_rows(uint32_t M, uint32_t K, uint32_t N) {
  if (M <= 16) return 64;
  const uint32_t ks_lds = (K / 256 + 7) / 8;   // ranges of at most eight steps with 32 staged rows
  return (N + 127) / 128 * ks_lds >= 128 ? 128 : 64;
}
static void stream_layout(uint32_t M, uint32_t K, uint32_t N, size_t scratch_bytes, uint32_t *range_steps, uint32_t *ksplit) {
  const uint32_t mt = (M + 15) / 16, nsteps = K / 256, nblocks = (N + stream_block_rows(M, K, N) - 1) / stream_block_rows(M, K, N);
  const uint32_t max_steps = (kStreamLdsMax / (16 * mt) - 16) / 512;
  uint32_t ks = (nsteps + max_steps - 1) / max_steps;
  auto more = [&] { return 2 * nblocks * ks <= 256 && nsteps / (2 * ks) >= 4 && (mt == 2 || nsteps >= 16); };
  while (ks < 16 && more() && scratch_bytes >= (size_t)2 * ks * M * N * sizeof(float)) ks *= 2;
  *range_steps = (nsteps + ks - 1) / ks;
  *ksplit = (nsteps + *range_steps - 1) / *range_steps;
}

// Whether Q8_0 takes this kernel by itself, with this much scratch memory.  Figures: us, the kernel that ran before this one / this one;
// both round fp32 activations to fp16.
bool stream_q8_preferred(uint32_t M, uint32_t K, uint32_t N, int a_f16, bool pairs, size_t scratch_bytes) {
  uint32_t range_steps, ksplit;
  stream_layout(M, K, N, scratch_bytes, &range_steps, &ksplit);
  const uint64_t weights = (uint64_t)N * K;
  const uint32_t rows = stream_block_rows(M, K, N), grid = (N + rows - 1) / rows * ksplit;
  if (M <= 8) {
    // In place of the 8-row GEMV (exact products as here).  8 rows: 14336 x 4096 19.8 / 17.0 (fp32 20.5 / 18.4), 4096 x 14336 20.7 / 18.7,
    // 5120 x 5120 18.7 / 13.0, 10240 x 2048 11.1 / 9.9, but 4096 x 4096 8.7 / 10.4, 1 x 28672 x 4096 29.8 / 33.0.  Not with few
    // workgroups: 8192 x 2560 (128) 9.7 / 10.6 (fp32 11.6 / 11.2), 8192 x 4096 without scratch 13.4 / 14.9, 7168 x 3584 (112) 12.9 / 14.9;
    if (M < 5 || weights < 20000000 || grid < (a_f16 && ksplit == 1 ? 144u : 128u)) return false;
    // nor on a short K that the GEMV takes in one round: 14336 x 1536 9.4 / 9.8, 16384 x 1536 9.6 / 10.2 (20480 x 1536 16.6 / 16.3);
    if (K < 2048 && grid <= 256) return false;
    if (ksplit == 1) return true;
    // a split only where its workgroups nearly run at once (13824 x 5120, 432 of two ranges, 23.9 / 26.2), and not where the GEMV's own
    // split suits it: 8192 x 4096 14.0 / 14.4 (fp32 16.8 / 14.6), 4096 x 5120 10.8 / 11.3 (12.8 / 11.7), 2048 x 11008 11.7 / 12.3.
    if (grid > 320 || pairs) return false;
    if (a_f16 && (K <= 4096 || (K <= 5120 && N <= 4096))) return false;
    return ksplit <= 4 || weights >= 25000000;
  }
  // In place of the row-tile matmul (weights rounded to fp16, 2e-4 of the norm) or of 8-row passes: 16 x 4096 x 4096 11.8 / 10.6,
  // 16 x 2048 x 2048 9.0 / 9.1, 16 x 9216 x 5120 (288 workgroups of two K ranges) 22.1 / 24.0; with two activation tiles from where
  // its workgroups run at once and fill the chip: 32 x 11264 x 2048 13.6 / 13.2, 32 x 8192 x 8192 26.0 / 23.4; below that the two
  // are level (17 / 24 / 32 rows of 5120 x 4096 14.1 / 13.6, 13.5 / 13.8, 14.0 / 14.4; of 4096 x 5120 13.9 / 13.2, 14.7 / 14.1, 15.5 / 14.3; of
  // 8192 x 2048 12.2 / 11.6, 11.4 / 11.9, 11.5 / 12.1; 32 x 4096 x 4096 12.6 / 12.1).  32 x 18432 x 4096 (288 workgroups) 33.1 / 35.8,
  // 32 x 6144 x 6144 (144) 20.5 / 21.3.  Exact weights are kept inside these lines also where they cost time: 16 x 20480 x 1024
  // 10.8 / 12.5, 16 x 32000 x 2048 19.1 / 20.1, 32 x 10240 x 2560 13.6 / 15.8, 32 x 12288 x 2048 with fp32 activations 13.2 / 14.3.
  return weights >= (M > 16 ? 22000000u : 16000000u) && (M <= 16 || grid >= 160) && (grid <= 256 || (M <= 16 && ksplit == 1));
}

bool stream_gemm_fits(int fmt, uint32_t M, uint32_t K, uint32_t N, uint32_t strideA, int a_f16, const void *A) {
  const size_t asz = a_f16 ? 2 : 4;
  return (fmt == CUTHIP_Q4_K || fmt == CUTHIP_Q8_0) && M >= 1 && M <= 32 && K % 256 == 0 && K >= 256 && (uintptr_t)A % 16 == 0 && (strideA * asz) % 16 == 0 &&
         (uint64_t)M * N < 0x7FFFFFFFull;
}
// bytes of scratch the launch cannot do without (0: the K range of a workgroup may cover all of K)
size_t stream_gemm_scratch(uint32_t M, uint32_t K, uint32_t N) {
  uint32_t rs, ks;
  stream_layout(M, K, N, 0, &rs, &ks);
  return ks > 1 ? (size_t)ks * M * N * sizeof(float) : 0;
}

template <int FMT, int SB>
static auto stream_kernel(uint32_t mt, uint32_t block_rows, bool two) {
  return block_rows == 128 ? gemm_stream_kernel<FMT, SB, 2, 1, 8>
         : mt == 1 ? (two ? gemm_stream_kernel<FMT, SB, 1, 2, 4> : gemm_stream_kernel<FMT, SB, 1, 1, 4>)
                   : (two ? gemm_stream_kernel<FMT, SB, 2, 2, 4> : gemm_stream_kernel<FMT, SB, 2, 1, 4>);
}

int launch_stream_gemm(int fmt, const void *W, const void *A, int a_f16, void *C, int c_f16, uint32_t M, uint32_t K, uint32_t N,
                       uint32_t strideA, uint32_t strideC, Epilogue epi, void *scratch, size_t scratch_bytes, hipStream_t stream) {
  StreamParams p;
  p.W = reinterpret_cast<const uint8_t *>(W);
  p.A = A;
  p.C = C;
  p.epi = epi;
  p.M = M; p.K = K; p.N = N; p.strideA = strideA; p.strideC = strideC;
  p.row_bytes = K / 256 * (fmt == CUTHIP_Q4_K ? 144 : 272);
  p.a_f16 = a_f16; p.c_f16 = c_f16;
  const uint32_t block_rows = stream_block_rows(M, K, N);
  p.nblocks = (N + block_rows - 1) / block_rows;
  if (!scratch || (uintptr_t)scratch % 16 != 0) scratch_bytes = 0;
  stream_layout(M, K, N, scratch_bytes, &p.range_steps, &p.ksplit);
  p.partial = reinterpret_cast<float *>(scratch);
  if (p.ksplit > 1 && scratch_bytes < (size_t)p.ksplit * M * N * sizeof(float)) {
    set_error("streaming matmul: K = %u at %u rows needs %zu bytes of scratch for its %u K ranges", K, M,
              (size_t)p.ksplit * M * N * sizeof(float), p.ksplit);
    return CUTHIP_ERR_INVALID;
  }
  const uint32_t mt = (M + 15) / 16;
  const size_t lds = (size_t)16 * mt * ((size_t)p.range_steps * 544 + 32) + 8 * kStripBytes;
  // four row groups: two waves each once a wave keeps at least two steps
  const bool two = block_rows == 64 && p.range_steps >= 4;
  const uint32_t threads = block_rows == 128 || two ? 512 : 256;
  // Activations are staged in batches of 16 pieces per thread, of 8 where those are all: a batch requests its last piece over and over
  // (Q4_K 4096 x 4096 at 16 rows 9.0 us against 9.5, 2048 x 2048 7.5 against 7.9; chosen inside the kernel it costs large calls 2 %)
  const bool few = (uint64_t)M * p.range_steps * 32 <= 8 * threads;
  auto kern = fmt == CUTHIP_Q4_K ? (few ? stream_kernel<CUTHIP_Q4_K, 8>(mt, block_rows, two) : stream_kernel<CUTHIP_Q4_K, 16>(mt, block_rows, two))
                                 : (few ? stream_kernel<CUTHIP_Q8_0, 8>(mt, block_rows, two) : stream_kernel<CUTHIP_Q8_0, 16>(mt, block_rows, two));
  if (lds > 64 * 1024) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)lds),
                           "hipFuncSetAttribute"))
      return rc;
  }
  hipLaunchKernelGGL(kern, dim3(p.nblocks * p.ksplit), dim3(threads), lds, stream, p);
  if (int rc = check_hip(hipGetLastError(), "streaming matmul launch")) return rc;
  if (p.ksplit == 1) return CUTHIP_OK;
  return launch_splitk_reduce(p.partial, p.ksplit, M, N, C, strideC, epi, c_f16, stream);
}

}  // namespace cuthip
