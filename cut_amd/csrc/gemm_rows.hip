// Layout rule and launch of the row-tile matmul (gemm_rows.hpp).
#include "gemm_rows.hpp"

namespace cuthip {

extern template int launch_rows_fmt<CUTHIP_Q8_0>(const RowsParams &, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q4_0>(const RowsParams &, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q4_K>(const RowsParams &, int, int, uint32_t, uint32_t, hipStream_t);
extern template int launch_rows_fmt<CUTHIP_Q6_K>(const RowsParams &, int, int, uint32_t, uint32_t, hipStream_t);

// Q8_0 on fp32 activations, four tiles, a K that the ranges do not cover exactly: the one instance that spills more than a
// couple of registers, and its reloads wait for every load in flight: 646 x 3584 x 9600 took 230 us where the model without
// this rule said 82.
static bool rows_spills(int fmt, uint32_t t, bool af32) { return fmt == CUTHIP_Q8_0 && af32 && t == 4; }

struct RowsLayout { uint32_t t, nw, per, ksplit; double cost; };

// How the launch is cut: t 32-row tiles of A and 32 nw weight rows per workgroup, K in ksplit x (8 / nw) ranges of per
// units of 128.  A workgroup fills a CU, so what counts is how many rounds of 256 workgroups there are and how many units
// a wave walks in each; a K split costs a second launch and its partial products a round trip.  In microseconds, fitted to
// 1500 launches (four formats, 12 .. 2048 rows, nine weight shapes from 1024 x 4096 to 28672 x 4096, graph replay, every nw
// and ksplit that fits forced in turn; 5.6 % rms):
//   2.6 + 2.25 rounds + per x unit(format, t, nw) x (1 + f) for each full round (1 + f x its share of the CUs for the last),
//   f = 0.73 - 0.1 (t - 1): the clock falls and the memory fills up with the chip
//   + 1.8 + 0.15 ksplit + 8 ksplit M N / 3.9 MB
// so that e.g. Q4_K 64 x 14336 x 4096 runs as 224 workgroups of nw = 2 (20.9 us; nw = 4 with two K ranges 22.0, with one 25.5),
// 64 x 28672 x 4096 as 224 of nw = 4 (31.7; nw = 2 in two rounds 42.8), 64 x 4096 x 4096 as 64 x 4 of nw = 2 (13.1; 2 ranges
// 13.9), 128 x 4096 x 14336 as 32 x 8 of nw = 4 (34.1; 4 ranges 37.1, 16 ranges 44.5).  fp32 activations: a tenth more.
static double unit_us(int fmt, uint32_t t, uint32_t nw) {
  static const double q4[2][4] = {{0.82, 1.27, 0, 0}, {0.67, 0.94, 1.35, 1.67}};
  static const double q6_k[2][4] = {{1.47, 1.84, 0, 0}, {1.27, 1.54, 1.85, 2.03}};
  static const double q8_0[2][4] = {{1.29, 1.81, 0, 0}, {1.05, 1.37, 1.85, 2.01}};
  const auto &u = fmt == CUTHIP_Q6_K ? q6_k : fmt == CUTHIP_Q8_0 ? q8_0 : q4;
  return u[nw == 4][t - 1];
}

static RowsLayout rows_layout(int fmt, uint32_t M, uint32_t K, uint32_t N, int a_f16, size_t scratch_bytes) {
  const uint32_t tmax = rows_max_tiles(fmt, !a_f16), t32 = (M - 1) / 32 + 1, units = (K - 1) / 128 + 1;
  const uint32_t want = (uint32_t)g_tuning.gemm_ksplit;   // forced by a test or a sweep
  RowsLayout best{0, 0, 0, 0, 1e30};
  auto consider = [&](uint32_t t) {
    const uint32_t mtiles = (t32 - 1) / t + 1;
    for (uint32_t nw = t <= 2 ? 2 : 4; nw <= 4; nw += 2) {
      const uint32_t kw = 8 / nw;
      const uint64_t tiles = (uint64_t)((N - 1) / (32 * nw) + 1) * mtiles;
      for (uint32_t ks = 1; ks <= 16; ++ks) {
        if (ks > 1 && (uint64_t)ks * M * N * 4 > scratch_bytes) break;
        if (want && ks != want && (uint64_t)want * M * N * 4 <= scratch_bytes) continue;
        uint32_t per = (units - 1) / (ks * kw) + 1;
        if (fmt == CUTHIP_Q4_K || fmt == CUTHIP_Q6_K) per = (per + 1) & ~1u;   // whole blocks of 256
        const uint32_t ranges = (units - 1) / (per * kw) + 1;                  // no empty range
        const double full = (double)((tiles * ranges - 1) / 256), last = (double)(tiles * ranges) - 256.0 * full;
        const double f = 0.73 - 0.1 * (t - 1);
        double unit = unit_us(fmt, t, nw) * (a_f16 ? 1.0 : 1.1);
        if (rows_spills(fmt, t, !a_f16) && (K % 128 != 0 || per * kw * ranges != units)) unit *= 2.4;
        double cost = 2.6 + 2.25 * (full + 1.0) + per * unit * (full * (1.0 + f) + 1.0 + f * last / 256.0);
        if (ranges > 1) cost += 1.8 + 0.15 * ranges + 8.0 * ranges * M * N / 3.9e6;
        if (cost < best.cost) best = RowsLayout{t, nw, per, ranges, cost};
      }
    }
  };
  auto even = [&](uint32_t most) { return (t32 - 1) / ((t32 - 1) / most + 1) + 1; };   // tiles per workgroup, evenly spread
  consider(even(tmax));
  if (rows_spills(fmt, best.t, !a_f16)) consider(even(best.t - 1));
  return best;
}

double rows_gemm_cost_us(int fmt, uint32_t M, uint32_t K, uint32_t N, int a_f16, size_t scratch_bytes) {
  return rows_layout(fmt, M, K, N, a_f16, scratch_bytes).cost;
}

// Offsets inside a workgroup's rows of A and of the weights are 32-bit.
bool rows_gemm_fits(int fmt, uint32_t K, uint32_t strideA, int a_f16) {
  return (uint64_t)(K / fmt_elems(fmt)) * fmt_bytes(fmt) * 128 <= 0xFFFFFFFFull && (uint64_t)strideA * 128 * (a_f16 ? 2 : 4) <= 0xFFFFFFFFull;
}

// scratch: 16-byte aligned room for fp32 partial products of a K split (nullptr / 0: none, one workgroup per tile)
int launch_rows_gemm(int fmt, const void *W, const void *A, int a_f16, void *C, int c_f16, uint32_t M, uint32_t K, uint32_t N,
                     uint32_t strideA, uint32_t strideC, Epilogue epi, hipStream_t stream, void *scratch, size_t scratch_bytes) {
  if (!scratch || (uintptr_t)scratch % 16 != 0) scratch_bytes = 0;
  const RowsLayout l = rows_layout(fmt, M, K, N, a_f16, scratch_bytes);
  RowsParams p;
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
  const int ragged = K % 128 != 0 || p.per * (8 / l.nw) * p.ksplit != p.units;
  p.c_f16 = c_f16;
  p.vec_store = store8_aligned(C, strideC, c_f16, epi) ? 1 : 0;
  int rc;
  switch (fmt) {
  case CUTHIP_Q8_0: rc = launch_rows_fmt<CUTHIP_Q8_0>(p, a_f16, ragged, l.t, l.nw, stream); break;
  case CUTHIP_Q4_0: rc = launch_rows_fmt<CUTHIP_Q4_0>(p, a_f16, ragged, l.t, l.nw, stream); break;
  case CUTHIP_Q4_K: rc = launch_rows_fmt<CUTHIP_Q4_K>(p, a_f16, ragged, l.t, l.nw, stream); break;
  default: rc = launch_rows_fmt<CUTHIP_Q6_K>(p, a_f16, ragged, l.t, l.nw, stream); break;
  }
  if (rc || p.ksplit == 1) return rc;
  return launch_splitk_reduce(p.partial, p.ksplit, M, N, C, strideC, epi, c_f16, stream);
}

}  // namespace cuthip
