// Layout rule and launch of the row-tile matmul (gemm_rows.hpp).
#include <algorithm>

#include "gemm_rows.hpp"

namespace cuthip {

extern template int launch_rows_fmt<CUTHIP_Q8_0>(const RowsParams &, int, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q4_0>(const RowsParams &, int, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q4_K>(const RowsParams &, int, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q6_K>(const RowsParams &, int, int, int, uint32_t, uint32_t, hipStream_t);

// Q8_0 on fp32 activations, four tiles, a K that the ranges do not cover exactly: the one instance that spills more than a
// couple of registers, and its reloads wait for every load in flight (a unit takes 1.3 times as long).
static bool rows_spills(int fmt, uint32_t t, bool af32) { return fmt == CUTHIP_Q8_0 && af32 && t == 4; }

// How the launch is cut.  A workgroup fills a CU, so what counts is how many rounds of 256 workgroups there are and how many units
// a wave walks in each; a K split costs a second launch and its partial products a round trip; more row tiles decode a
// weight less often, fewer fill the chip without a split.  In microseconds, fitted to 67,000 launches (four formats, both
// activation types, 12 .. 4096 rows, 22 weight shapes from 512 x 512 to 28672 x 4096, graph replay, every t, nw and most
// ksplit forced in turn; 7.9 % rms, and the layout chosen is on average 0.5 % slower than the best of them):
//   2.1 + (1.9 + 0.5 t) rounds + per x unit(format, t, nw) x (1 + f) for each full round (1 + f x its share of the CUs for the
//   last), f = 0.31 + 0.05 (t - 1): the clock falls and the memory fills up with the chip
//   + 2 + 0.16 ksplit + 8 ksplit M N / 5.4 MB
//   fp32 activations: a unit takes 1.165 times as long; ranges that do not cover K exactly: 1.08 times
// so that e.g. Q4_K 64 x 14336 x 4096 runs as 224 workgroups of t = 2, nw = 2 (21.2 us; nw = 4 with two K ranges 21.9, with one
// 26.3), 64 x 28672 x 4096 as 224 of nw = 4 (29.7; nw = 2 in two rounds 40.4), 128 x 4096 x 14336 as 64 x 4 of t = 2, nw = 4
// (30.8; t = 4 with seven ranges 32.6), 100 x 14336 x 4096 as 224 of t = 2, nw = 4 (26.2; t = 4 with two ranges 29.6, with one
// 36.1).  With the largest t only, narrow matrices split K where fewer tiles need no second launch: Q4_0 with fp32 activations
// 300 x 2560 x 2560 20.3 us (t = 2, nw = 2 without a split: 13.9), 300 x 2048 x 2048 17.8 (11.7); Q8_0 384 x 14336 x 4096 93.8 (83.4).
static double unit_us(int fmt, uint32_t t, uint32_t nw) {
  static const double q4[2][4] = {{0.95, 1.25, 0, 0}, {0.74, 0.95, 1.19, 1.42}};
  static const double q6_k[2][4] = {{1.66, 1.84, 0, 0}, {1.38, 1.47, 1.64, 1.85}};
  static const double q8_0[2][4] = {{1.43, 1.71, 0, 0}, {1.15, 1.32, 1.57, 1.81}};
  const auto &u = fmt == CUTHIP_Q6_K ? q6_k : fmt == CUTHIP_Q8_0 ? q8_0 : q4;
  return u[nw == 4][t - 1];
}

// What a unit takes where fp16 rows of A lie on 16 bytes, against the table: the direct form (rows_direct), and on Q6_K also the
// tiles of 32 rows beside it, which the table has 10 % too high for such rows (without a factor of their own they lost to the direct tiles of 64
// where those are slower, us: 53 x 5788 x 12544 without scratch memory 56.0 -> 63.7, 229 x 1673 x 10752 46.4 -> 51.9, 340 x 1046 x 1792
// 14.1 -> 16.0).  270 problems (33 .. 1200 rows, every t and nw forced): the layout chosen is 0.4 % (Q6_K 0.8 %) slower than the best one, without
// these factors 5.3 % (4.3 %); against the layout without them 0.956 (0.969) of the time, 5 of 152 (0 of 118) slower by more than 3 %.
static double direct_gain(int fmt, uint32_t t, uint32_t nw) {
  if (fmt == CUTHIP_Q6_K) return t == 1 || (t == 2 && nw == 2) ? 0.9 : 1.0;
  if (!rows_direct(fmt, (int)t, (int)nw)) return 1.0;
  return t == 2 ? 0.88 : t == 3 ? 1.0 : 0.96;
}

static RowsLayout layout_of(int fmt, uint32_t M, uint32_t K, uint32_t N, int a_f16, size_t scratch_bytes, bool aligned) {
  const uint32_t tmax = rows_max_tiles(fmt, !a_f16), t32 = (M - 1) / 32 + 1, units = (K - 1) / 128 + 1;
  const uint32_t want = (uint32_t)g_tuning.gemm_ksplit;   // forced by a test or a sweep
  RowsLayout best{0, 0, 0, 0, 1e30};
  auto consider = [&](uint32_t t) {
    const uint32_t mtiles = (t32 - 1) / t + 1;
    for (uint32_t nw = t <= 2 ? 2 : 4; nw <= 4; nw += 2) {
      if (g_tuning.rows_nw && nw != (uint32_t)g_tuning.rows_nw) continue;
      const uint32_t kw = 8 / nw;
      const uint64_t tiles = (uint64_t)((N - 1) / (32 * nw) + 1) * mtiles;
      for (uint32_t ks = 1; ks <= 16; ++ks) {
        // no split that needs a second round of workgroups: 18 of the 1,542 measured shapes that split would take one, and
        // without it 6 of them are 2 to 5 % slower and 2 faster
        if (ks > 1 && ((uint64_t)ks * M * N * 4 > scratch_bytes || (!want && tiles * ks > 256))) break;
        if (want && ks != want && (uint64_t)want * M * N * 4 <= scratch_bytes) continue;
        uint32_t per = (units - 1) / (ks * kw) + 1;
        if (fmt == CUTHIP_Q4_K || fmt == CUTHIP_Q6_K) per = (per + 1) & ~1u;   // whole blocks of 256
        const uint32_t ranges = (units - 1) / (per * kw) + 1;                  // no empty range
        const double full = (double)((tiles * ranges - 1) / 256), last = (double)(tiles * ranges) - 256.0 * full;
        const double f = 0.31 + 0.05 * (t - 1);
        double unit = unit_us(fmt, t, nw) * (a_f16 ? 1.0 : 1.165);
        if (a_f16 && aligned) unit *= direct_gain(fmt, t, nw);
        if (K % 128 != 0 || per * kw * ranges != units) unit *= rows_spills(fmt, t, !a_f16) ? 1.08 * 1.3 : 1.08;
        double cost = 2.1 + (1.9 + 0.5 * t) * (full + 1.0) + per * unit * (full * (1.0 + f) + 1.0 + f * last / 256.0);
        if (ranges > 1) cost += 2.0 + 0.16 * ranges + 8.0 * ranges * M * N / 5.4e6;
        if (cost < best.cost) best = RowsLayout{t, nw, per, ranges, cost};
      }
    }
  };
  auto even = [&](uint32_t most) { return (t32 - 1) / ((t32 - 1) / most + 1) + 1; };   // tiles per workgroup, evenly spread
  if (g_tuning.rows_t) {   // forced by a test or a sweep (an instance that does not exist: the next smaller one)
    consider(std::min((uint32_t)g_tuning.rows_t, tmax));
    return best;
  }
  for (uint32_t t = 1; t <= tmax; ++t)
    if (even(t) == t) consider(t);   // (else a smaller one covers the rows in as many workgroups)
  return best;
}

// The layout for rows of A on 16 bytes (rows_aligned), and for others: those are staged through registers.  With the cut of the direct
// kernel they took, us, its cut / their own: Q4_K 49 x 14292 x 8704 57.4 / 44.1, 799 x 1523 x 6656 49.0 / 42.6, 40 x 13878 x 3584 28.2 / 24.9;
// Q6_K without scratch memory 51 x 6045 x 7680 54.5 / 43.4, 229 x 1673 x 10752 64.6 / 51.8.
RowsLayout rows_gemm_layout(int fmt, uint32_t M, uint32_t K, uint32_t N, int a_f16, size_t scratch_bytes) {
  return layout_of(fmt, M, K, N, a_f16, scratch_bytes, true);
}
RowsLayout rows_gemm_layout_off16(int fmt, uint32_t M, uint32_t K, uint32_t N, int a_f16, size_t scratch_bytes) {
  return layout_of(fmt, M, K, N, a_f16, scratch_bytes, false);
}

// Offsets inside a workgroup's rows of A and of the weights are 32-bit.
bool rows_gemm_fits(int fmt, uint32_t K, uint32_t strideA, int a_f16) {
  return (uint64_t)(K / fmt_elems(fmt)) * fmt_bytes(fmt) * 128 <= 0xFFFFFFFFull && (uint64_t)strideA * 128 * (a_f16 ? 2 : 4) <= 0xFFFFFFFFull;
}

// l: rows_gemm_layout's (rows_gemm_layout_off16's) for the same arguments; scratch: the room for fp32 partial products that it was given (16-byte aligned)
int launch_rows_gemm(int fmt, const void *W, const void *A, int a_f16, void *C, int c_f16, uint32_t M, uint32_t K, uint32_t N,
                     uint32_t strideA, uint32_t strideC, Epilogue epi, hipStream_t stream, const RowsLayout &l, void *scratch) {
  RowsParams p{};
  p.W = reinterpret_cast<const uint8_t *>(W);
  p.A = A;
  p.C = C;
  p.partial = reinterpret_cast<float *>(scratch);
  p.epi = epi;
  p.M = M; p.K = K; p.N = N; p.strideA = strideA; p.strideC = strideC;
  p.row_bytes = (uint32_t)((uint64_t)(K / fmt_elems(fmt)) * fmt_bytes(fmt));
  p.ntiles = (N - 1) / (32 * l.nw) + 1;
  p.mtiles = (M - 1) / (32 * l.t) + 1;
  p.units = (K - 1) / 128 + 1;
  p.per = l.per;
  p.ksplit = l.ksplit;
  const bool aligned = rows_aligned(A, strideA);
  const int ragged = K % 128 != 0 || p.per * (8 / l.nw) * p.ksplit != p.units;
  p.c_f16 = c_f16;
  p.vec_store = store8_aligned(C, strideC, c_f16, epi) ? 1 : 0;
  int rc;
  switch (fmt) {
  case CUTHIP_Q8_0: rc = launch_rows_fmt<CUTHIP_Q8_0>(p, a_f16, ragged, aligned, l.t, l.nw, stream); break;
  case CUTHIP_Q4_0: rc = launch_rows_fmt<CUTHIP_Q4_0>(p, a_f16, ragged, aligned, l.t, l.nw, stream); break;
  case CUTHIP_Q4_K: rc = launch_rows_fmt<CUTHIP_Q4_K>(p, a_f16, ragged, aligned, l.t, l.nw, stream); break;
  default: rc = launch_rows_fmt<CUTHIP_Q6_K>(p, a_f16, ragged, aligned, l.t, l.nw, stream); break;
  }
  if (rc || p.ksplit == 1) return rc;
  return launch_splitk_reduce(p.partial, p.ksplit, M, N, C, strideC, epi, c_f16, stream);
}

}  // namespace cuthip
