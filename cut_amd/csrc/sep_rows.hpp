// The several-row matmul on the separated layout (sep_rows.hip).
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
  uint32_t nsplit, per;     // K ranges over workgroups, blocks per wave    } set by sep_rows_cut
  uint32_t tiles, passes;   // column tiles, groups of 16 or 32 rows of A   }
};

void sep_rows_cut(SepRowsParams &p);          // nsplit is never more than K / 128 rounded up
bool sep_rows_fits(const SepRowsParams &p);   // after sep_rows_cut
int launch_sep_rows(const SepRowsParams &p, bool q4, bool affine, hipStream_t stream);

}  // namespace cuthip
