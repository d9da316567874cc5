#include "gemm_rows.hpp"
namespace cuthip {
template int launch_rows_fmt<CUTHIP_Q4_0>(const RowsParams &, int, int, uint32_t, uint32_t, hipStream_t);
}
