// Matmul on native GGUF blocks for tens to hundreds of activation rows (gfx950):
//   C[m,n] = sum_k A[m,k] * dequant(W)[n,k]
//
// What bounds it: up to a few hundred rows the decode - about 2.2 vector instructions per weight (Q4_K: a mask or a
// shift for two weights, a mixed-precision multiply-add each, one packed rounding), 1.75 for Q8_0 / Q4_0 - together
// with v_mfma_f32_32x32x16_f16, which leaves the vector units about half of their issue slots while it runs; on random
// data the clock falls with both busy.  Everything else is laid out to stay out of their way:
//   * One workgroup of eight waves owns 32 T rows of A (T = 1 .. 4) and 32 NW weight rows (NW = 2, 4); its 8 / NW K ranges
//     meet in LDS at the end, so that a 64-row panel still has eight waves to hide latency with.  A weight is decoded
//     by one lane of one wave, straight into the operand registers of the matrix instruction (lane l: weight row
//     l & 31), once per 32 T rows; it never goes through LDS as fp16.
//   * The blocks are fetched in pieces of 8 or 16 bytes, neighbouring lanes neighbouring pieces, and turned into rows
//     by an LDS image that belongs to the wave alone (no barrier).  Loads whose neighbouring lanes are in different
//     weight rows touch a cache line per lane: 14336 x 4096 at 32 rows took 33 us with them, 16 with the pieces.
//   * A goes through registers into two LDS buffers of one slice (128 / SU elements of every K range), or straight into three
//     (rows_direct); its fragments are read L matrix instructions ahead into a ring of registers.
//   * The instruction stream is written slot by slot, one matrix instruction and its share of the decode, the LDS reads,
//     the loads and the LDS stores in each: left to the compiler, the decode of a unit ends up in front of its eight
//     matrix instructions and the two do not overlap.
// A weight is rounded to fp16 once, from the fp32 expression of its format (Q8_0 / Q4_0: the fp16 product d * q, the same
// bits); fp16 activations are exact, fp32 ones rounded once; accumulation is fp32: 3e-4 of the result's norm.
//
// Measured, us (graph replay, MI355X), against 128 x 128 tiles of four waves that decoded through LDS with K split
// over workgroups, or the two-pass path where that was the choice:
//   14336 x 4096   Q4_K  64 rows 28.0 -> 21.4, 128 37.4 -> 27.9, 256 72.2 -> 42.4;  Q8_0  12 rows 30.3 -> 21.3,
//                  64 34.3 -> 28.8;  Q6_K  32 rows 35.5 -> 23.5, 128 49.6 -> 38.7
//   4096 x 14336   Q4_K  128 rows 38.3 -> 31.8, 512 96.4 -> 79.9
//   4096 x 4096    Q8_0  24 rows 16.6 -> 12.4;  Q4_0  512 rows 38.4 -> 23.1, 768 57.0 -> 33.1
//   28672 x 4096   Q4_K  64 rows 48.1 -> 29.5, 130 92.4 -> 65.9;  Q8_0  16 rows 55.3 -> 33.7
//   2048 x 14336 x 4096 in one launch (no scratch memory): Q4_K 331 -> 285, Q6_K 397 -> 329, Q8_0 327 -> 308
// On a short K with many tiles those tiles (gemm_lds.hip) stay the faster ones: see single_launch_choice.
#pragma once
#include "common.hpp"
#include "gemm_store.hpp"

namespace cuthip {

int launch_splitk_reduce(const float *partial, uint32_t ksplit, uint32_t M, uint32_t N, void *C, uint32_t strideC, Epilogue epi,
                         int c_f16, hipStream_t stream);

struct RowsParams {
  const uint8_t *W;
  const void *A;
  void *C;
  float *partial;          // [ksplit][M][N] fp32 when ksplit > 1
  Epilogue epi;
  uint32_t M, K, N, strideA, strideC, row_bytes;
  uint32_t ntiles, mtiles, ksplit;
  uint32_t rest_per_xcd;   // tiles of the last ntiles % 8 panels, shared by eight; set by the launch
  uint32_t units;          // 128-element units of K
  uint32_t per;            // units per K range (ksplit x KW ranges), a multiple of the format's group
  int c_f16, vec_store;
};

// Four tiles of 32 rows per workgroup at most.  Q6_K with fp32 activations: three, the instance with four does not fit
// 256 registers (40 spilled; 1024 x 14336 x 4096 347 us).
constexpr uint32_t rows_max_tiles(int fmt, bool af32) { return fmt == CUTHIP_Q6_K && af32 ? 3 : 4; }

// Where A goes to LDS without passing registers (global_load_lds, three buffers): fp16 activations, rows of A on 16 bytes, slices of half a
// unit.  Elsewhere it does not pay: with slices of a whole unit the two slices in flight are enough (100 x 14336 x 4096 on Q4_K 27.6 us, direct
// 28.0), and on Q8_0 and Q4_0 it gave between +2 and -3 %.  Q4_K / Q6_K, us: 64 x 14336 x 4096 24.1 -> 21.6 / 27.8 -> 26.8,
// 512 x 14336 x 4096 80.2 -> 72.7 / 85.1 -> 84.9, 100 x 28672 x 4096 on Q4_K 42.8 -> 39.1, 100 x 5120 x 4096 17.5 -> 15.8.
constexpr bool rows_direct(int fmt, int t, int nw) { return t > nw / 2 && (fmt == CUTHIP_Q4_K || fmt == CUTHIP_Q6_K); }

constexpr uint32_t kPanelGroup = 8;   // weight panels (of one XCD) that are walked together

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef __attribute__((address_space(3))) uint8_t lds_u8r;
template <class V> __device__ __forceinline__ V lds_get(const uint8_t *p) { return *reinterpret_cast<const V *>(p); }

// Two weights on their way to a packed pair of halves: fp32 until the rounding, or (formats whose scale is an fp16 number)
// the integer as halves.  Decoding is cut in steps so that the kernel can put other instructions between dependent ones.
__device__ __forceinline__ f32x2 mix2(half_t a, half_t b, float s, float o) {   // fp16 subnormals (integer x 2^-24 or 2^-20)
  return f32x2{__builtin_fmaf((float)a, s, o), __builtin_fmaf((float)b, s, o)};
}
__device__ __forceinline__ uint32_t round2(f32x2 v) { return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, half2_t)); }
__device__ __forceinline__ half2_t as_h2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
// bytes 2X, 2X + 1 of w as 1024 + byte in fp16
template <int X> __device__ __forceinline__ half2_t bytes_h2(uint32_t w) {
  return as_h2(__builtin_amdgcn_perm(0x64646464u, w, X & 1 ? 0x04030402u : 0x04010400u));
}

// What a format tells the kernel.  The lane (row r = lane & 31, half kg = lane >> 5) turns 64 of a unit's 128 elements into
// eight B fragments of v_mfma_f32_32x32x16_f16, the ones that lie together in the block: fragment J of half kg holds
// elements a_off(kg) + j_off(J) .. + 7 of the unit (A is read in the same order).
//   GROUP     units that are loaded together; PIECE bytes per lane and load, NP pieces per weight row and group
//   IMG       bytes of a weight row's image in LDS; piece p is fetched from off(p) of the group and lies at p * PIECE
// Where A is staged in halves of a unit, half `part` holds the elements of fragments 4 part .. 4 part + 3 of both lanes:
// chunk c (8 elements) of it is element chunk(c) + part * PART of the unit, and fragment J of lane kg lies at
// h_off(kg) + hj_off(J & 3).
template <int FMT, bool DIR> struct RowFmt;

template <> struct RowFmt<CUTHIP_Q4_K, false> {
  static constexpr int GROUP = 2, PIECE = 16, NP = 9, BYTES = 144, IMG = 144;
  __device__ static uint32_t off(uint32_t p) { return 16 * p; }
  struct Raw { u32x4 hdr, q[2]; };
  struct Sc { float s0, s1, o0, o1; };
  __device__ static uint32_t a_off(uint32_t kg) { return 64 * kg; }
  static constexpr uint32_t j_off(int j) { return 32 * (j >> 2) + 8 * (j & 3); }
  static constexpr uint32_t PART = 32;
  __device__ static uint32_t chunk(uint32_t c) { return 64 * (c >> 2) + 8 * (c & 3); }
  __device__ static uint32_t h_off(uint32_t kg) { return 32 * kg; }
  static constexpr uint32_t hj_off(int j) { return 8 * j; }
  // U: unit inside the group
  template <int U> __device__ static void read(Raw &r, const uint8_t *img, uint32_t kg) {
    r.hdr = lds_get<u32x4>(img);
    r.q[0] = lds_get<u32x4>(img + 16 + 64 * U + 32 * kg);
    r.q[1] = lds_get<u32x4>(img + 32 + 64 * U + 32 * kg);
  }
  template <int U> __device__ static Sc prep(const Raw &r, uint32_t kg, bool live0, bool) {
    const uint32_t sh = 16 * kg, dd = live0 ? r.hdr.x : 0u;
    const float d = f16bits_to_f32(dd & 0xFFFF), dmin = -f16bits_to_f32(dd >> 16);
    const uint32_t a0 = r.hdr.y >> sh, a1 = r.hdr.z >> sh, a2 = r.hdr.w >> sh;
    const uint32_t scp = U ? (a2 & 0x0F0Fu) | ((a0 >> 2) & 0x3030u) : a0 & 0x3F3Fu;
    const uint32_t mp = U ? ((a2 >> 4) & 0x0F0Fu) | ((a1 >> 2) & 0x3030u) : a1 & 0x3F3Fu;
    return Sc{d * 16777216.0f * cvt_ubyte0(scp), d * 1048576.0f * cvt_ubyte1(scp), dmin * cvt_ubyte0(mp), dmin * cvt_ubyte1(mp)};
  }
  // Fragment J (0-3 low nibbles, 4-7 high nibbles) in three steps: fields() picks the four nibbles of dword H out of the
  // block's bytes, two in each register; mid() makes the pair X (elements 2X, 2X + 1), fin() rounds it.
  template <int J, int H> __device__ static void fields(const Raw &r, uint32_t &a, uint32_t &b) {
    constexpr int p = J & 3;
    const uint32_t w = r.q[p >> 1][2 * (p & 1) + H];
    constexpr uint32_t m = J < 4 ? 0x000F000Fu : 0x00F000F0u;
    a = w & m;
    b = (w >> 8) & m;
    asm("" : "+v"(a), "+v"(b));   // one mask for two weights (left alone, the compiler masks every nibble by itself)
  }
  typedef f32x2 Mid;
  template <int J, int X> __device__ static Mid mid(uint32_t a, uint32_t b, const Sc &c) {
    const float s = J < 4 ? c.s0 : c.s1, o = J < 4 ? c.o0 : c.o1;
    return X & 1 ? mix2(as_h2(a).y, as_h2(b).y, s, o) : mix2(as_h2(a).x, as_h2(b).x, s, o);
  }
  template <int J> __device__ static uint32_t fin(Mid v, const Sc &) { return round2(v); }
};

// Where A goes to LDS directly (in halves of a unit) the lane takes 16 bytes of each 64 elements, so that a half is 64 neighbouring elements:
// whole cache lines of A (lines requested in halves arrive at half the rate, 17 TB/s for the chip against 34), for the scales of four
// sub-blocks in place of two.  Through registers this does not pay (100 x 1024 x 4096 9.3 us, with these scales 9.7; 50 x 7552 x 1280 11.8, 12.5).
template <> struct RowFmt<CUTHIP_Q4_K, true> {
  static constexpr int GROUP = 2, PIECE = 16, NP = 9, BYTES = 144, IMG = 144;
  __device__ static uint32_t off(uint32_t p) { return 16 * p; }
  struct Raw { u32x4 hdr, q[2]; };
  struct Sc { float s[4], o[4]; };
  static constexpr uint32_t PART = 64;
  __device__ static uint32_t chunk(uint32_t c) { return 8 * c; }
  __device__ static uint32_t h_off(uint32_t kg) { return 16 * kg; }
  static constexpr uint32_t hj_off(int j) { return 32 * (j >> 1) + 8 * (j & 1); }
  // U: unit inside the group
  template <int U> __device__ static void read(Raw &r, const uint8_t *img, uint32_t kg) {
    r.hdr = lds_get<u32x4>(img);
    r.q[0] = lds_get<u32x4>(img + 16 + 64 * U + 16 * kg);
    r.q[1] = lds_get<u32x4>(img + 48 + 64 * U + 16 * kg);
  }
  template <int U> __device__ static Sc prep(const Raw &r, uint32_t, bool live0, bool) {
    const uint32_t dd = live0 ? r.hdr.x : 0u;
    const float d = f16bits_to_f32(dd & 0xFFFF), dmin = -f16bits_to_f32(dd >> 16);
    const uint32_t sc = U ? (r.hdr.w & 0x0F0F0F0Fu) | ((r.hdr.y >> 2) & 0x30303030u) : r.hdr.y & 0x3F3F3F3Fu;
    const uint32_t mn = U ? ((r.hdr.w >> 4) & 0x0F0F0F0Fu) | ((r.hdr.z >> 2) & 0x30303030u) : r.hdr.z & 0x3F3F3F3Fu;
    const float dl = d * 16777216.0f, dh = d * 1048576.0f;
    return Sc{{dl * cvt_ubyte0(sc), dh * cvt_ubyte1(sc), dl * cvt_ubyte2(sc), dh * cvt_ubyte3(sc)},
              {dmin * cvt_ubyte0(mn), dmin * cvt_ubyte1(mn), dmin * cvt_ubyte2(mn), dmin * cvt_ubyte3(mn)}};
  }
  // Fragment J (sub-block J >> 1 of the unit: low nibbles of 32 bytes, then their high nibbles) in three steps: fields() picks the
  // four nibbles of dword H out of the block's bytes, two in each register; mid() makes the pair X (elements 2X, 2X + 1), fin() rounds it.
  template <int J, int H> __device__ static void fields(const Raw &r, uint32_t &a, uint32_t &b) {
    const uint32_t w = r.q[J >> 2][2 * (J & 1) + H];
    constexpr uint32_t m = J & 2 ? 0x00F000F0u : 0x000F000Fu;
    a = w & m;
    b = (w >> 8) & m;
    asm("" : "+v"(a), "+v"(b));   // one mask for two weights (left alone, the compiler masks every nibble by itself)
  }
  typedef f32x2 Mid;
  template <int J, int X> __device__ static Mid mid(uint32_t a, uint32_t b, const Sc &c) {
    const float s = c.s[J >> 1], o = c.o[J >> 1];
    return X & 1 ? mix2(as_h2(a).y, as_h2(b).y, s, o) : mix2(as_h2(a).x, as_h2(b).x, s, o);
  }
  template <int J> __device__ static uint32_t fin(Mid v, const Sc &) { return round2(v); }
};

template <bool DIR> struct RowFmt<CUTHIP_Q6_K, DIR> {
  // [ql:128][qh:64][sc:16][d]: 13 pieces in place, the last 16 bytes of the block (d at their end) as piece 13
  static constexpr int GROUP = 2, PIECE = 16, NP = 14, BYTES = 210, IMG = 224;
  __device__ static uint32_t off(uint32_t p) { return p < 13 ? 16 * p : 194u; }
  struct Raw { u32x4 l0, l1, h; u32x2 sc; uint32_t d; };
  struct Sc { float s[4], o[4]; };   // d * scale of quarter s (times the 2^24 or 2^20 of its subnormals), -32 d * scale
  __device__ static uint32_t a_off(uint32_t kg) { return 16 * kg; }
  static constexpr uint32_t j_off(int j) { return 32 * (j >> 1) + 8 * (j & 1); }
  static constexpr uint32_t PART = 64;
  __device__ static uint32_t chunk(uint32_t c) { return 8 * c; }
  __device__ static uint32_t h_off(uint32_t kg) { return 16 * kg; }
  static constexpr uint32_t hj_off(int j) { return 32 * (j >> 1) + 8 * (j & 1); }
  template <int U> __device__ static void read(Raw &r, const uint8_t *img, uint32_t kg) {
    r.l0 = lds_get<u32x4>(img + 64 * U + 16 * kg);
    r.l1 = lds_get<u32x4>(img + 64 * U + 32 + 16 * kg);
    r.h = lds_get<u32x4>(img + 128 + 32 * U + 16 * kg);
    r.sc = lds_get<u32x2>(img + 192 + 8 * U);
    r.d = lds_get<uint32_t>(img + 220);
  }
  template <int U> __device__ static Sc prep(const Raw &r, uint32_t kg, bool live0, bool) {
    const float d = live0 ? f16bits_to_f32(r.d >> 16) : 0.0f;
    Sc c;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float ds = d * (float)(int)__builtin_amdgcn_sbfe((int)(s < 2 ? r.sc.x : r.sc.y), 8 * kg + 16 * (s & 1), 8);
      c.s[s] = ds * (s < 2 ? 16777216.0f : 1048576.0f);
      c.o[s] = -32.0f * ds;
    }
    return c;
  }
  template <int J, int H> __device__ static void fields(const Raw &r, uint32_t &a, uint32_t &b) {
    constexpr int s = J >> 1, e = 2 * (J & 1) + H;   // quarter, dword of its 16 bytes
    const uint32_t w = (s & 1 ? r.l1 : r.l0)[e], h = r.h[e];
    constexpr uint32_t m = s < 2 ? 0x000F000Fu : 0x00F000F0u, mb = s < 2 ? 0x00300030u : 0x03000300u;
    // high bits 2 s, 2 s + 1 of a byte to bits 4, 5 (low nibble) or 8, 9 (high nibble in place, x 16)
    const uint32_t ha = s & 1 ? h << 2 : h << 4, hb = s & 1 ? h >> 6 : h >> 4;
    a = (w & m) | (ha & mb);
    b = ((w >> 8) & m) | (hb & mb);
    asm("" : "+v"(a), "+v"(b));
  }
  typedef f32x2 Mid;
  template <int J, int X> __device__ static Mid mid(uint32_t a, uint32_t b, const Sc &c) {
    constexpr int s = J >> 1;
    return X & 1 ? mix2(as_h2(a).y, as_h2(b).y, c.s[s], c.o[s]) : mix2(as_h2(a).x, as_h2(b).x, c.s[s], c.o[s]);
  }
  template <int J> __device__ static uint32_t fin(Mid v, const Sc &) { return round2(v); }
};

// Blocks of 32 with an fp16 scale in front: block 2 kg and 2 kg + 1 of the unit; the quants of the first lie two bytes off
// a dword boundary.  value = d * q with one rounding to fp16: a packed fp16 product.
template <> struct RowFmt<CUTHIP_Q8_0, false> {
  static constexpr int GROUP = 1, PIECE = 8, NP = 17, BYTES = 136, IMG = 136;
  __device__ static uint32_t off(uint32_t p) { return 8 * p; }
  struct Raw { uint32_t w[17]; };
  struct Sc { half2_t d0, d1; };
  __device__ static uint32_t a_off(uint32_t kg) { return 64 * kg; }
  static constexpr uint32_t j_off(int j) { return 8 * j; }
  static constexpr uint32_t PART = 32;
  __device__ static uint32_t chunk(uint32_t c) { return 64 * (c >> 2) + 8 * (c & 3); }
  __device__ static uint32_t h_off(uint32_t kg) { return 32 * kg; }
  static constexpr uint32_t hj_off(int j) { return 8 * j; }
  template <int U> __device__ static void read(Raw &r, const uint8_t *img, uint32_t kg) {
#pragma unroll
    for (int i = 0; i < 17; ++i) r.w[i] = lds_get<uint32_t>(img + 68 * kg + 4 * i);
  }
  template <int U> __device__ static Sc prep(const Raw &r, uint32_t kg, bool live0, bool live1) {
    const uint32_t a = live0 ? r.w[0] : 0u, b = live1 ? r.w[8] : 0u;
    return Sc{__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(a, a, 0x01000100u)), __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(b, b, 0x03020302u))};
  }
  template <int J, int H> __device__ static void fields(const Raw &r, uint32_t &a, uint32_t &) {
    constexpr int e = 2 * (J & 3) + H;   // dword of the block's quants
    a = (J < 4 ? __builtin_amdgcn_alignbyte(r.w[e + 1], r.w[e], 2) : r.w[9 + e]) ^ 0x80808080u;   // q + 128
  }
  typedef half2_t Mid;
  template <int J, int X> __device__ static Mid mid(uint32_t a, uint32_t, const Sc &) {
    return bytes_h2<X>(a) + half2_t{(half_t)-1152.0f, (half_t)-1152.0f};
  }
  template <int J> __device__ static uint32_t fin(Mid v, const Sc &c) { return __builtin_bit_cast(uint32_t, v * (J < 4 ? c.d0 : c.d1)); }
};

template <> struct RowFmt<CUTHIP_Q4_0, false> {
  static constexpr int GROUP = 1, PIECE = 8, NP = 9, BYTES = 72, IMG = 72;
  __device__ static uint32_t off(uint32_t p) { return 8 * p; }
  struct Raw { uint32_t w[9]; };
  struct Sc { half2_t d0, d1; };
  __device__ static uint32_t a_off(uint32_t kg) { return 64 * kg; }
  static constexpr uint32_t j_off(int j) { return 8 * j; }
  static constexpr uint32_t PART = 32;
  __device__ static uint32_t chunk(uint32_t c) { return 64 * (c >> 2) + 8 * (c & 3); }
  __device__ static uint32_t h_off(uint32_t kg) { return 32 * kg; }
  static constexpr uint32_t hj_off(int j) { return 8 * j; }
  template <int U> __device__ static void read(Raw &r, const uint8_t *img, uint32_t kg) {
#pragma unroll
    for (int i = 0; i < 9; ++i) r.w[i] = lds_get<uint32_t>(img + 36 * kg + 4 * i);
  }
  template <int U> __device__ static Sc prep(const Raw &r, uint32_t kg, bool live0, bool live1) {
    const uint32_t a = live0 ? r.w[0] : 0u, b = live1 ? r.w[4] : 0u;
    return Sc{__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(a, a, 0x01000100u)), __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(b, b, 0x03020302u))};
  }
  // J & 3: 0, 1 low nibbles of the block's 16 bytes (elements 0-15), 2, 3 high nibbles (16-31)
  template <int J, int H> __device__ static void fields(const Raw &r, uint32_t &a, uint32_t &) {
    constexpr int e = 2 * (J & 1) + H;
    a = (J < 4 ? __builtin_amdgcn_alignbyte(r.w[e + 1], r.w[e], 2) : r.w[5 + e]) & (J & 2 ? 0xF0F0F0F0u : 0x0F0F0F0Fu);
  }
  typedef half2_t Mid;
  template <int J, int X> __device__ static Mid mid(uint32_t a, uint32_t, const Sc &) {
    if constexpr ((J & 2) != 0) {   // 1024 + 16 q
      const half2_t s{(half_t)0.0625f, (half_t)0.0625f}, k{(half_t)-72.0f, (half_t)-72.0f};
      return __builtin_elementwise_fma(bytes_h2<X>(a), s, k);
    }
    return bytes_h2<X>(a) + half2_t{(half_t)-1032.0f, (half_t)-1032.0f};
  }
  template <int J> __device__ static uint32_t fin(Mid v, const Sc &c) { return __builtin_bit_cast(uint32_t, v * (J < 4 ? c.d0 : c.d1)); }
};

// T: 32-row tiles of A per workgroup; NW groups of 32 weight rows x KW ranges of K = eight waves; SU slices per unit
// (a slice is what is staged of A at a time: 128 / SU elements of every K range; two of them have to fit in LDS)
template <int FMT, int T, int NW, bool DIR> struct RowsGeom {
  static constexpr int KW = 8 / NW, SU = T > NW / 2 ? 2 : 1;
  using F = RowFmt<FMT, DIR>;
  static constexpr int R = 32 * NW, SK = 128 / SU, ROWB = KW * SK * 2, PITCH = ROWB + 16,
                       BUF = DIR ? 32 * T * ROWB : 32 * T * PITCH, NBUF = DIR ? 3 : 2, CH = ROWB / 16,
                       CPT = 32 * T * CH / 512, IMGS = 32 * F::IMG, IMG0 = NBUF * BUF, STAGE_LD = R + 4,
                       STAGE = KW * 32 * T * STAGE_LD * 4, LOOP = IMG0 + 8 * IMGS, LDS = LOOP > STAGE ? LOOP : STAGE,
                       NI = (32 * F::NP + 63) / 64;
  // DIR: a row of one K range is CR chunks of 16 bytes, an instruction of a wave fills RPI rows of it
  static constexpr int CR = SK / 8, RPI = 64 / CR;
  __device__ static uint32_t key(uint32_t row) { return (row >> 1) & 7; }
  static_assert(!DIR || (SU == 2 && CR == 8), "straight to LDS: slices of half a unit (rows_direct)");
  static_assert(NW * KW == 8 && 512 % CH == 0 && (32 * T * CH) % 512 == 0 && LDS <= 160 * 1024, "tile geometry");
};

__device__ __forceinline__ f32x16 mfma32(half8_t a, half8_t b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

__device__ const u32x4 kZeros1K[64] = {};

template <int PIECE> struct PieceType { typedef u32x4 type; };
template <> struct PieceType<8> { typedef u32x2 type; };

// RAG: K is not a multiple of 128, or the K ranges do not cover it exactly.
template <int FMT, int T, int NW, bool AF32, bool RAG, bool DIR>
__global__ void __launch_bounds__(512, 2) gemm_rows_kernel(RowsParams p) {
  static_assert(!DIR || !AF32, "LDS-direct loads do not convert");
  using G = RowsGeom<FMT, T, NW, DIR>;
  using F = typename G::F;
  constexpr int KW = G::KW, SU = G::SU;
  // slices of A in flight in registers: as many as leave the instance without spills
  constexpr int P = (T == 1 || T == 3) && !(AF32 && (T == 3 || NW == 2)) ? 4 : 2;
  using PT = typename PieceType<F::PIECE>::type;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // Ids id, id + 8, ... share an XCD: the row tiles of one weight panel run there one after the other, neighbouring panels on
  // neighbouring XCDs.  Of the panels beyond a multiple of eight each XCD takes an eighth of the tiles: dealt out whole, 20
  // panels were three for four of the XCDs and two for the others, and 1024 x 2560 x 2560 ran in two rounds instead of one.
  // (Neighbouring panels on one XCD throughout: 2048 x 4096 x 512 with fp32 activations 29 -> 33 us.)
  // Beyond eight row tiles an XCD walks them in groups of eight panels: the 32 workgroups that run there together then read
  // about as much of A as of the weights.  With all row tiles of one panel first, A came through the L2 once for every panel:
  // 4096 x 5632 x 2048 on Q4_0 with fp32 activations 226 -> 153 us, 4096 x 14336 x 4096 on Q8_0 762 -> 644.
  const uint32_t whole = p.ntiles & ~7u, body = whole * p.mtiles * p.ksplit, xcd = blockIdx.x & 7;
  uint32_t slot = blockIdx.x >> 3, panels = whole / 8;
  if (blockIdx.x >= body) {
    panels = p.ntiles - whole;
    slot = xcd * p.rest_per_xcd + ((blockIdx.x - body) >> 3);
    if (slot >= panels * p.mtiles * p.ksplit) return;
  }
  uint32_t mt, pt, split;   // (quotients leave the vector ALU: scalar)
  if (p.mtiles <= kPanelGroup) {
    const uint32_t rest = __builtin_amdgcn_readfirstlane(slot / p.mtiles);
    split = __builtin_amdgcn_readfirstlane(rest / panels);
    mt = slot - rest * p.mtiles;
    pt = rest - split * panels;
  } else {
    split = __builtin_amdgcn_readfirstlane(slot / (panels * p.mtiles));
    const uint32_t in_split = slot - split * panels * p.mtiles, group = __builtin_amdgcn_readfirstlane(in_split / (kPanelGroup * p.mtiles));
    const uint32_t in_group = in_split - group * kPanelGroup * p.mtiles, width = min(kPanelGroup, panels - group * kPanelGroup);
    mt = __builtin_amdgcn_readfirstlane(in_group / width);
    pt = group * kPanelGroup + in_group - mt * width;
  }
  const uint32_t nt = blockIdx.x < body ? pt * 8 + xcd : whole + pt;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nw = wave % NW, kw = wave / NW, r32 = lane & 31, kg = lane >> 5;
  const uint32_t m0 = mt * 32 * T, nrow0 = nt * G::R + nw * 32, rows = min(p.M - m0, 32u * T);
  const uint32_t slices = p.per * SU, nblk = p.K / 32;
  const uint32_t u0 = (split * KW + kw) * p.per, u1 = min(u0 + p.per, p.units);

  // Weights.  Piece c = 64 i + lane of a group is piece c % NP of weight row c / NP (the surplus lanes of the last load
  // repeat the last piece): fetched by neighbouring lanes, every cache line is requested once.
  const uint32_t n0 = min(nrow0, p.N - 1), glast = (p.units - 1) / F::GROUP;
  const uint8_t *wbase = p.W + (size_t)n0 * p.row_bytes;
  uint32_t poff[G::NI];
#pragma unroll
  for (int i = 0; i < G::NI; ++i) {
    const uint32_t c = min(64u * i + lane, 32u * F::NP - 1), row = c / F::NP;
    poff[i] = (min(nrow0 + row, p.N - 1) - n0) * p.row_bytes + F::off(c - row * F::NP);
  }
  PT pc[G::NI];
  // No byte past the end of the tensor: where K ends inside a unit, the last unit of the tensor's last rows would be read
  // beyond it.  Only a wave that holds them looks, and only there: the piece is fetched earlier and shifted into place when it
  // is stored (what it then lacks lies past K).  With the shift behind every load each group waited for its own loads: Q8_0 at
  // 12 rows, us, 4096 x 11008 39 -> 21, 3584 x 9728 32 -> 18.
  const bool edge = RAG && F::PIECE == 8 && (uint64_t)(p.N - min(nrow0 + 32, p.N) + 1) * p.row_bytes < (uint64_t)(glast + 1) * F::BYTES;
  auto piece_group = [&](uint32_t g) __attribute__((always_inline)) { return min(u0 / F::GROUP + g, glast); };   // g: group of this wave's range
  auto beyond = [&](const uint8_t *q) __attribute__((always_inline)) {   // bytes by which a piece of 8 at q crosses the end
    const uint8_t *end = p.W + (size_t)p.N * p.row_bytes - 8;
    return q > end ? (uint32_t)(q - end) : 0u;
  };
  auto load_pieces = [&](uint32_t g) __attribute__((always_inline)) {
    const uint32_t gg = piece_group(g);
    const uint8_t *base = wbase + (size_t)gg * F::BYTES;
    if (RAG && F::PIECE == 8 && edge && gg == glast) {
#pragma unroll
      for (int i = 0; i < G::NI; ++i) {
        const uint8_t *q = base + poff[i];
        if constexpr (F::PIECE == 8) pc[i] = ld_u32x2(q - beyond(q));
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < G::NI; ++i) {
      // the offset is made opaque in place: a 32-bit lane offset on a scalar base, no 64-bit vector add per load
      asm volatile("" : "+v"(poff[i]));
      if constexpr (F::PIECE == 16) pc[i] = ld_u32x4(base + poff[i]);
      else pc[i] = ld_u32x2(base + poff[i]);
    }
  };
  uint8_t *img = lds + G::IMG0 + wave * G::IMGS;
  uint32_t pdst[G::NI];
#pragma unroll
  for (int i = 0; i < G::NI; ++i) {
    const uint32_t c = min(64u * i + lane, 32u * F::NP - 1), row = c / F::NP;
    pdst[i] = row * F::IMG + (c - row * F::NP) * F::PIECE;
  }
  auto store_pieces = [&](uint32_t g) __attribute__((always_inline)) {
    if constexpr (RAG && F::PIECE == 8) {
      const uint32_t gg = piece_group(g);
      if (edge && gg == glast) {
        const uint8_t *base = wbase + (size_t)gg * F::BYTES;
#pragma unroll
        for (int i = 0; i < G::NI; ++i) {
          const uint64_t w = (((uint64_t)pc[i].y << 32) | pc[i].x) >> (8 * min(beyond(base + poff[i]), 7u));
          pc[i] = PT{(uint32_t)w, (uint32_t)(w >> 32)};
        }
      }
    }
#pragma unroll
    for (int i = 0; i < G::NI; ++i) *reinterpret_cast<PT *>(img + pdst[i]) = pc[i];
  };
  const uint8_t *mine = img + r32 * F::IMG;

  // Activations: thread -> 16-byte column chunk (the same for all its rows), rows 512 / CH apart.
  constexpr uint32_t RS = 512 / G::CH, ESZ = AF32 ? 4 : 2, CPK = G::SK / 8;   // CPK: chunks per K range
  const uint32_t col = tid % G::CH, rf = tid / G::CH, cc = col % CPK;
  const uint32_t abeg = (split * KW + col / CPK) * p.per * 128 + (SU == 1 ? 8 * cc : F::chunk(cc));
  const uint8_t *abase = reinterpret_cast<const uint8_t *>(p.A) + (size_t)m0 * p.strideA * ESZ;
  uint32_t aoff[G::CPT];
#pragma unroll
  for (int v = 0; v < G::CPT; ++v) aoff[v] = (min(rf + v * RS, rows - 1) * p.strideA + (RAG ? 0u : abeg)) * ESZ;
  u32x4 st[P][G::CPT], st2[AF32 ? P : 1][AF32 ? G::CPT : 1];
  // k of slice t relative to abeg
  auto slice_k = [&](uint32_t t) __attribute__((always_inline)) { return SU == 1 ? t * 128 : (t / SU) * 128 + (t % SU) * F::PART; };
  auto stage_load = [&](int s, int v, uint32_t t) __attribute__((always_inline)) {
    if constexpr (RAG) {
      const uint8_t *b = abase + (aoff[v] + min(abeg + slice_k(t), p.K - 8) * ESZ);
      st[s][v] = ld_u32x4(b);
      if constexpr (AF32) st2[s][v] = ld_u32x4(b + 16);
    } else {
      const uint8_t *b = abase + (size_t)slice_k(min(t, slices - 1)) * ESZ;
      asm volatile("" : "+v"(aoff[v]));
      st[s][v] = ld_u32x4(b + aoff[v]);
      if constexpr (AF32) st2[s][v] = ld_u32x4(b + 16 + aoff[v]);
    }
  };
  auto stage_store = [&](int s, int v, uint32_t t, uint32_t buf) __attribute__((always_inline)) {
    u32x4 o = st[s][v];
    if constexpr (AF32) {
      const f32x4 lo = __builtin_bit_cast(f32x4, st[s][v]), hi = __builtin_bit_cast(f32x4, st2[s][v]);
      o = __builtin_bit_cast(u32x4, half8_t{(half_t)lo.x, (half_t)lo.y, (half_t)lo.z, (half_t)lo.w, (half_t)hi.x, (half_t)hi.y, (half_t)hi.z, (half_t)hi.w});
    }
    if (RAG && abeg + slice_k(t) >= p.K) o = u32x4{0, 0, 0, 0};
    *reinterpret_cast<u32x4 *>(lds + buf * G::BUF + (rf + v * RS) * G::PITCH + col * 16) = o;
  };

  // DIR: instruction v of a wave fills RPI rows of one K range, lane l the chunk l % CR of row l / CR (chunk c of a row lies at
  // c ^ key(row), so that the 16 rows of a quarter of a fragment read lie in different banks)
  uint32_t doff[DIR ? G::CPT : 1];
  if constexpr (DIR) {
#pragma unroll
    for (int v = 0; v < G::CPT; ++v) {
      constexpr uint32_t per_kw = 32 * T / G::RPI;
      const uint32_t i = 8 * v + wave, dkw = i / per_kw, row = (i % per_kw) * G::RPI + lane / G::CR;
      const uint32_t c = (lane % G::CR) ^ G::key(row), beg = (split * KW + dkw) * p.per * 128 + F::chunk(c);
      doff[v] = (min(row, rows - 1) * p.strideA + beg) * 2;
    }
  }
  auto load_direct = [&](int v, uint32_t t, uint32_t buf) __attribute__((always_inline)) {   // buf: LDS offset of the buffer
    // as text (gemm_dense.hip says why); M0 is the LDS address of the wave's 1,024 bytes
    const uint32_t dst = (uint32_t)(uintptr_t)(lds_u8r *)lds + buf + (8 * v + wave) * 1024;
    const uint8_t *g = abase + (size_t)slice_k(min(t, slices - 1)) * 2;
    uint32_t off = doff[v];
    if constexpr (RAG) {   // a range that reaches beyond K takes zeros there: the weights are zero too, but an infinity times zero is not
      constexpr uint32_t per_kw = 32 * T / G::RPI;
      const bool live = (split * KW + (8 * v + wave) / per_kw) * p.per + min(t, slices - 1) / SU < p.units;
      g = live ? g : reinterpret_cast<const uint8_t *>(kZeros1K);
      off = live ? off : lane * 16;
    }
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(g), "s"(dst) : "memory");
  };

  f32x16 acc[T];
#pragma unroll
  for (int i = 0; i < T; ++i) acc[i] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

  constexpr int FR = 8 * T / SU;                 // MFMAs, and A fragments, per slice
  constexpr int L = FR < 16 ? 4 : 6, RING = 8;   // fragments read ahead
  constexpr int BAR = FR - L + 2;                // the barrier stands in front of this MFMA: the last read is two MFMAs old
  constexpr int TRIP = 2 * SU > P ? 2 * SU : P;   // slices per loop trip: everything indexed by a slice or unit is static in it
  static_assert(TRIP * FR % RING == 0 && TRIP % (2 * SU) == 0 && TRIP % P == 0, "compile-time slots over a loop trip");
  uint32_t aread = r32 * G::PITCH + kw * (G::SK * 2);
  if constexpr (SU == 1) aread += F::a_off(kg) * 2;
  else aread += F::h_off(kg) * 2;
  half8_t ring[RING];
  typename F::Raw raw[2];
  typename F::Sc sc;
  u32x4 b;
  // DIR: byte offsets of fragment j of the lane's row of the wave's K range (chunk c of row r lies at c ^ key(r))
  constexpr int NJ = 8 / SU;
  uint32_t joff[DIR ? NJ : 1], jaddr = 0;
  if constexpr (DIR) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      joff[j] = (kw * 32 * T + r32) * (G::SK * 2) + (((F::h_off(kg) + F::hj_off(j)) / 8) ^ G::key(r32)) * 16;
  }
  // LDS offsets of the buffers of the present slice, the next one and the one after that
  uint32_t bufr = 0, bufn = G::BUF, bufw = 2 * G::BUF;
  auto read_a = [&](uint32_t buf, int f) __attribute__((always_inline)) {
    if constexpr (DIR) {
      if (f % T == 0) jaddr = joff[f / T] + buf;
      return lds_get<half8_t>(lds + jaddr + (f % T) * 32 * G::SK * 2);
    } else if constexpr (SU == 1) {
      return lds_get<half8_t>(lds + buf * G::BUF + aread + (f % T) * 32 * G::PITCH + F::j_off(f / T) * 2);
    } else {
      return lds_get<half8_t>(lds + buf * G::BUF + aread + (f % T) * 32 * G::PITCH + F::hj_off(f / T) * 2);
    }
  };
  auto prep = [&](auto uc, const typename F::Raw &r, uint32_t i) __attribute__((always_inline)) {   // i: unit of this wave's range
    const uint32_t u = u0 + i;
    const bool live = !RAG || u < u1;
    if constexpr (F::GROUP == 1) return F::template prep<0>(r, kg, !RAG || (live && 4 * u + 2 * kg < nblk), !RAG || (live && 4 * u + 2 * kg + 1 < nblk));
    else return F::template prep<decltype(uc)::value>(r, kg, live, live);
  };

  // One slice: FR slots of one MFMA each, with the LDS read of the fragment L slots ahead, a share of the decode of the
  // next weight fragment, and the loads and LDS stores of what comes later spread among them.  Slots are fenced from each
  // other, so that the order of the memory instructions is the one written here.
  auto slice = [&](auto qc, uint32_t t) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value, part = q % SU, ui = q / SU, U = ui % F::GROUP, UN = (ui + 1) % F::GROUP;
    constexpr bool WSL = part == 0 && U == F::GROUP - 1;   // weights are requested in this slice
    constexpr int r0 = q * FR;                     // ring position of the slice's first fragment
    const uint32_t i = t / SU;
    u32x4 bn;
    uint32_t fa = 0, fb = 0;
    typename F::Mid mid[4];
    static_for<FR>([&](auto fc) __attribute__((always_inline)) {
      constexpr int f = decltype(fc)::value, m = f % T, j = part * (8 / SU) + f / T;
      if constexpr (f == BAR) {
        if constexpr (DIR) {   // A of the next slice is here; what was requested in this one is under way
          constexpr int younger = G::CPT + (WSL ? G::NI : 0);
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(younger) : "memory");
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      acc[m] = mfma32(ring[(r0 + f) % RING], __builtin_bit_cast(half8_t, b), acc[m]);
      if constexpr (f + L < FR) ring[(r0 + f + L) % RING] = read_a(DIR ? bufr : q & 1, f + L);
      if constexpr (f >= BAR) {   // the first L fragments of the next slice, over the last slots
        constexpr int g0 = (f - BAR) * L / (L - 2), g1 = (f - BAR + 1) * L / (L - 2);
        static_for<g1 - g0>([&](auto gc) __attribute__((always_inline)) {
          constexpr int g = g0 + decltype(gc)::value;
          ring[(r0 + FR + g) % RING] = read_a(DIR ? bufn : (q & 1) ^ 1, g);
        });
      }
      // the next group's pieces to LDS (the last unit of this one is in registers), its successor's on their way
      if constexpr (j == (DIR ? 0 : 1) && m == 0 && U == F::GROUP - 1) {
        store_pieces(i / F::GROUP + 1);
        load_pieces(i / F::GROUP + 2);
      }
      if constexpr (j == 5 && m == T - 1) F::template read<UN>(raw[(ui + 1) & 1], mine, kg);
      if constexpr (j == 7 && m == 0) sc = prep(std::integral_constant<int, UN>{}, raw[(ui + 1) & 1], i + 1);
      // the next fragment of weights: pair X is rounded a slot after its products (in the last slot nothing is left to do
      // that the next MFMA would have to wait for)
      constexpr int jn = (j + 1) % 8, sets = T == 1 ? 1 : T - 1;
      static_for<4>([&](auto xc) __attribute__((always_inline)) {
        constexpr int X = decltype(xc)::value;
        if constexpr (X * sets / 4 == m) {
          if constexpr (X % 2 == 0) F::template fields<jn, X / 2>(raw[(j < 7 ? ui : ui + 1) & 1], fa, fb);
          mid[X] = F::template mid<jn, X>(fa, fb, sc);
        }
      });
      static_for<4>([&](auto xc) __attribute__((always_inline)) {
        constexpr int X = decltype(xc)::value;
        if constexpr (X * sets / 4 + (T == 1 ? 0 : 1) == m) bn[X] = F::template fin<jn>(mid[X], sc);
      });
      if constexpr (m == T - 1) b = bn;
      // A of the next slice to LDS, A of slice t + P on its way
      constexpr int v0 = f * G::CPT / (FR * 3 / 4), v1 = (f + 1) * G::CPT / (FR * 3 / 4);
      if constexpr (DIR) {
        if constexpr (f >= 1 && f <= G::CPT) load_direct(f - 1, t + 2, bufw);
        static_assert(G::CPT < BAR, "the barrier counts this slice's requests");
        if constexpr (f == FR - 1) {
          const uint32_t b0 = bufr;
          bufr = bufn; bufn = bufw; bufw = b0;
        }
      } else if constexpr (v0 < G::CPT)
        static_for<(v1 < G::CPT ? v1 : G::CPT) - v0>([&](auto vc) __attribute__((always_inline)) {
          constexpr int v = v0 + decltype(vc)::value;
          stage_store((q + 1) % P, v, t + 1, (q & 1) ^ 1);
          stage_load(q % P, v, t + P);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  if constexpr (DIR) static_for<G::CPT>([&](auto vc) __attribute__((always_inline)) { load_direct(decltype(vc)::value, 0, 0); });
  else static_for<G::CPT>([&](auto vc) __attribute__((always_inline)) { stage_load(0, decltype(vc)::value, 0); });
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();   // the first slice of every wave is requested ahead of the weights of any
  __builtin_amdgcn_sched_barrier(0);
  load_pieces(0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (DIR) static_for<G::CPT>([&](auto vc) __attribute__((always_inline)) { load_direct(decltype(vc)::value, 1, G::BUF); });
  else static_for<P - 1>([&](auto sc2) __attribute__((always_inline)) {
    static_for<G::CPT>([&](auto vc) __attribute__((always_inline)) { stage_load(decltype(sc2)::value + 1, decltype(vc)::value, decltype(sc2)::value + 1); });
    __builtin_amdgcn_sched_barrier(0);
  });
  if constexpr (!DIR) static_for<G::CPT>([&](auto vc) __attribute__((always_inline)) { stage_store(0, decltype(vc)::value, 0, 0); });
  if constexpr (DIR) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // both slices and the first weights
  store_pieces(0);
  load_pieces(1);
  __builtin_amdgcn_sched_barrier(0);
  F::template read<0>(raw[0], mine, kg);
  __syncthreads();
  sc = prep(std::integral_constant<int, 0>{}, raw[0], 0);
  static_for<4>([&](auto xc) __attribute__((always_inline)) {
    constexpr int X = decltype(xc)::value;
    uint32_t fa, fb;
    F::template fields<0, X / 2>(raw[0], fa, fb);
    b[X] = F::template fin<0>(F::template mid<0, X>(fa, fb, sc), sc);
  });
  static_for<L>([&](auto fc) __attribute__((always_inline)) { ring[decltype(fc)::value] = read_a(0, decltype(fc)::value); });
  for (uint32_t t = 0; t < slices; t += TRIP)
    static_for<TRIP>([&](auto qc) __attribute__((always_inline)) {
      if (t + decltype(qc)::value < slices) slice(qc, t + decltype(qc)::value);
    });
  if constexpr (DIR) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in what the K parts are added in
  __syncthreads();

  // the K parts of the workgroup meet in LDS as fp32 [KW][32 T][R]; register e of lane l: row 8 (e / 4) + 4 (l >> 5) + e % 4
  float *stage = reinterpret_cast<float *>(lds) + (size_t)kw * 32 * T * G::STAGE_LD + nw * 32 + r32;
  static_for<T>([&](auto mc) __attribute__((always_inline)) {
    static_for<16>([&](auto ec) __attribute__((always_inline)) {
      constexpr int m = decltype(mc)::value, e = decltype(ec)::value;
      stage[(32 * m + 8 * (e >> 2) + 4 * kg + (e & 3)) * G::STAGE_LD] = acc[m][e];
    });
  });
  __syncthreads();
  const uint32_t nbase = nt * G::R;
  const bool to_partial = p.ksplit > 1;
  const bool vec = to_partial ? p.N % 4 == 0 : p.vec_store != 0;
  void *cbase = to_partial ? (void *)(p.partial + ((size_t)split * p.M + m0) * p.N) : p.C;
  const Epilogue epi{to_partial ? (int)CUTHIP_EPI_NONE : p.epi.kind, p.epi.op, p.epi.D};
  const uint32_t ldc = to_partial ? p.N : p.strideC, mrow = to_partial ? 0 : m0;
  const int c_f16 = to_partial ? 0 : p.c_f16;
  // the common epilogues in short loops of their own: none, or the residual add (whole panels only)
  const int fast = !vec || nbase + G::R > p.N ? 0 : epi.kind == CUTHIP_EPI_NONE ? (c_f16 ? 1 : 2) : epi.kind == CUTHIP_EPI_BINARY && epi.op == CUTHIP_BINARY_ADD ? (c_f16 ? 3 : 4) : 0;
  auto finish = [&](auto fastc) __attribute__((always_inline)) {
    constexpr int FAST = decltype(fastc)::value;
    for (uint32_t c = tid; c < (uint32_t)(4 * T * G::R); c += 512) {   // 32 T rows x R / 8 chunks
      const uint32_t row = c / (G::R / 8), c8 = (c % (G::R / 8)) * 8;
      const float *src = reinterpret_cast<const float *>(lds) + row * G::STAGE_LD + c8;
      f32x4 lo = *reinterpret_cast<const f32x4 *>(src), hi = *reinterpret_cast<const f32x4 *>(src + 4);
#pragma unroll
      for (int w = 1; w < KW; ++w) {
        lo += *reinterpret_cast<const f32x4 *>(src + (size_t)w * 32 * T * G::STAGE_LD);
        hi += *reinterpret_cast<const f32x4 *>(src + (size_t)w * 32 * T * G::STAGE_LD + 4);
      }
      if (row >= rows || nbase + c8 >= p.N) continue;
      const size_t idx = (size_t)(mrow + row) * ldc + nbase + c8;
      if constexpr (FAST != 0) {
        if constexpr (FAST == 3) {
          const half8_t d = *reinterpret_cast<const half8_t *>(reinterpret_cast<const half_t *>(epi.D) + idx);
          lo += f32x4{(float)d[0], (float)d[1], (float)d[2], (float)d[3]};
          hi += f32x4{(float)d[4], (float)d[5], (float)d[6], (float)d[7]};
        }
        if constexpr (FAST == 4) {
          const f32x4 *dp = reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(epi.D) + idx);
          lo += dp[0];
          hi += dp[1];
        }
        if constexpr (FAST == 1 || FAST == 3) {
          *reinterpret_cast<half8_t *>(reinterpret_cast<half_t *>(cbase) + idx) =
              half8_t{(half_t)lo[0], (half_t)lo[1], (half_t)lo[2], (half_t)lo[3], (half_t)hi[0], (half_t)hi[1], (half_t)hi[2], (half_t)hi[3]};
        } else {
          f32x4 *cp = reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(cbase) + idx);
          cp[0] = lo;
          cp[1] = hi;
        }
      } else {
        store_out8(cbase, epi, c_f16, idx, lo, hi, nbase + c8, p.N, vec);
      }
    }
  };
  if (fast == 1) finish(std::integral_constant<int, 1>{});
  else if (fast == 2) finish(std::integral_constant<int, 2>{});
  else if (fast == 3) finish(std::integral_constant<int, 3>{});
  else if (fast == 4) finish(std::integral_constant<int, 4>{});
  else finish(std::integral_constant<int, 0>{});
}

template <int FMT, int T, int NW, bool AF32, bool RAG, bool ALIGNED> static int launch_rows_tile(RowsParams p, hipStream_t stream) {
  constexpr bool DIR = ALIGNED && !AF32 && rows_direct(FMT, T, NW);
  using G = RowsGeom<FMT, T, NW, DIR>;
  auto kern = gemm_rows_kernel<FMT, T, NW, AF32, RAG, DIR>;
  if (G::LDS > 64 * 1024) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS),
                           "hipFuncSetAttribute"))
      return rc;
  }
  const uint64_t body = (uint64_t)(p.ntiles & ~7u) * p.mtiles * p.ksplit, rest = (uint64_t)(p.ntiles & 7u) * p.mtiles * p.ksplit;
  const uint64_t grid = body + (rest + 7) / 8 * 8;
  if (grid > 0x7FFFFFFFull) {
    set_error("cuthip_matmul_gguf: problem too large for one launch");
    return CUTHIP_ERR_INVALID;
  }
  p.rest_per_xcd = (uint32_t)((rest + 7) / 8);
  hipLaunchKernelGGL(kern, dim3((uint32_t)grid), dim3(512), G::LDS, stream, p);
  return check_hip(hipGetLastError(), "row-tile matmul launch");
}

template <int FMT, bool AF32, bool RAG, bool ALIGNED> static int launch_rows_af(const RowsParams &p, uint32_t t, uint32_t nw, hipStream_t stream) {
  if (nw == 2) return t == 1 ? launch_rows_tile<FMT, 1, 2, AF32, RAG, ALIGNED>(p, stream) : launch_rows_tile<FMT, 2, 2, AF32, RAG, ALIGNED>(p, stream);
  switch (t) {
  case 1: return launch_rows_tile<FMT, 1, 4, AF32, RAG, ALIGNED>(p, stream);
  case 2: return launch_rows_tile<FMT, 2, 4, AF32, RAG, ALIGNED>(p, stream);
  case 3: return launch_rows_tile<FMT, 3, 4, AF32, RAG, ALIGNED>(p, stream);
  default:
    if constexpr (rows_max_tiles(FMT, AF32) == 4) return launch_rows_tile<FMT, 4, 4, AF32, RAG, ALIGNED>(p, stream);
    return CUTHIP_ERR_INVALID;   // (never asked for)
  }
}

// t: 32-row tiles of A per workgroup; nw: groups of 32 weight rows per workgroup (2: the waves share them four ways in K); aligned: rows of A
// lie on 16 bytes
template <int FMT> int launch_rows_fmt(const RowsParams &p, int a_f16, int ragged, int aligned, uint32_t t, uint32_t nw, hipStream_t stream) {
  if (!a_f16) return ragged ? launch_rows_af<FMT, true, true, false>(p, t, nw, stream) : launch_rows_af<FMT, true, false, false>(p, t, nw, stream);
  if (aligned) return ragged ? launch_rows_af<FMT, false, true, true>(p, t, nw, stream) : launch_rows_af<FMT, false, false, true>(p, t, nw, stream);
  return ragged ? launch_rows_af<FMT, false, true, false>(p, t, nw, stream) : launch_rows_af<FMT, false, false, false>(p, t, nw, stream);
}

}  // namespace cuthip
