// Kernels over rows of 5118..524287 entries (hold_row and stream_row of sky_build_long.h), one workgroup per row.
#include "sky_build_long.h"

namespace sky {

// The first n_first workgroups take the rows of first_list (the longest ones), the others the n of vlist from the last one on.
__global__ __launch_bounds__(ST_T, 4) void build_stream_kernel(const RowRef* __restrict__ first_list, uint32_t n_first,
                                                            const RowRef* __restrict__ vlist, uint32_t n,
                                                            const float* __restrict__ wgt,
                                                            AliasEntry* __restrict__ table,
                                                            int8_t* __restrict__ valid) {
  __shared__ StreamLds lds;
  const RowRef rr = blockIdx.x < n_first ? first_list[blockIdx.x] : vlist[n - 1 - (blockIdx.x - n_first)];
  const bool ok = stream_row(rr, lds, wgt, table);
  if (threadIdx.x == 0) valid[rr.v] = ok ? 1 : 0;
}

__global__ __launch_bounds__(HOLD_T, 4) void build_hold_kernel(const RowRef* __restrict__ vlist, const float* __restrict__ wgt,
                                                       AliasEntry* __restrict__ table, int8_t* __restrict__ valid) {
  extern __shared__ __align__(16) uint64_t smem[];
  __shared__ uint64_t s_aux[8 * (HOLD_T / 64)];
  const RowRef rr = vlist[blockIdx.x];
  const bool ok = hold_row(rr, smem, s_aux, wgt, table);
  if (threadIdx.x == 0) valid[rr.v] = ok ? 1 : 0;
}

static bool g_hold_lds_enabled = false;
// The n rows of `rows` (5118..HOLD_MAX_DEG entries each).
int build_rows_hold(sky_graph* g, const RowRef* rows, uint32_t n) {
  if (n == 0) return SKY_OK;
  if (!g_hold_lds_enabled) {
    SKY_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(build_hold_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)HOLD_LDS_BYTES));
    g_hold_lds_enabled = true;
  }
  hipLaunchKernelGGL(build_hold_kernel, dim3(n), dim3(HOLD_T), HOLD_LDS_BYTES, g->stream, rows, g->adjwgt, g->table, g->valid);
  return SKY_OK;
}

// Builds the n_first rows of `first_list` and the n rows of `rows_list` (8190..STREAM_MAX_DEG entries each) in one
// launch that starts with the former and goes through the latter backwards: their lists have the longer ones last.
int build_rows_stream(sky_graph* g, const RowRef* first_list, uint32_t n_first, const RowRef* rows_list, uint32_t n) {
  if (n + n_first == 0) return SKY_OK;
  hipLaunchKernelGGL(build_stream_kernel, dim3(n + n_first), dim3(ST_T), 0, g->stream, first_list, n_first, rows_list, n, g->adjwgt,
                     g->table, g->valid);
  return SKY_OK;
}

}  // namespace sky
