// The matmuls on the separated layout beside the general one of compat.hip: one or two rows (sep_vec.hip), several (sep_rows.hip).
#pragma once
#include "common.hpp"

namespace cuthip {

struct SepRowsParams {
  const float *A;
  const uint8_t *B;
  const uint16_t *S;
  float *C;
  float *partial;   // [nsplit][M][N], 16-byte aligned, when nsplit > 1
  Epilogue epi;
  uint32_t M, K, N, strideA, strideB, strideC, scaleStride;
  const half_t *A16;   // sep_rows16: [M][K], 16-byte aligned
  uint32_t t;                           // 16-row tiles of A per pass (sep_vec: lanes to a k-row) } set by those that cut
  uint32_t nsplit, per, tiles, passes;  // K ranges over workgroups, blocks per wave (sep_vec: per range), column tiles, passes over the rows }
  double cost_us;                       // sep_rows16: estimate                  }
};

// How the launch is cut; false if it does not fit.  partial_bytes: room for the sums of several K ranges (nsplit is never
// more than K / 128 rounded up).
bool sep_vec_cut(SepRowsParams &p, bool q4);
bool sep_rows_cut(SepRowsParams &p, size_t partial_bytes);
bool sep_rows16_cut(SepRowsParams &p, bool q4, bool affine, size_t partial_bytes);
bool sep_rows16_preferred(SepRowsParams &p, bool q4, bool affine, size_t partial_bytes);   // cut, and the cheaper of the two ways
int launch_sep_vec(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream);
int launch_sep_rows(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream);
int launch_sep_rows16(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream);

}  // namespace cuthip
