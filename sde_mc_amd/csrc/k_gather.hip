// k_gather.hip -- a training batch gathered from stored trajectories: the rows
// of several arrays [paths][rows][dim] of any strides (the solvers store
// [rows][dim][paths]) for a list of path indices, written contiguous, in one
// launch.  Bound by the scattered reads: each value of a stored row lies in
// another 64-byte sector; consecutive lanes take consecutive output values, so
// the writes are whole lines.  Batches of 1000 trajectories of about 50 rows:
// 7 us, where slicing them one by one and stacking the slices took 6000 views
// and 6 concatenations a batch (5 ms of host work).
#include "sdemc_core.h"

namespace sdemc {

struct GatherArgs {
  sdemc_gather a[SDEMC_GATHER_MAX];
};

__global__ __launch_bounds__(256) void k_gather(const GatherArgs g, const int64_t* __restrict__ index,
                                                int64_t n_index, int64_t n_paths) {
  const sdemc_gather& a = g.a[blockIdx.y];
  const int64_t per = (int64_t)a.rows * a.dim;
  const int64_t total = n_index * per;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += stride) {
    const int64_t b = e / per;
    const int32_t v = (int32_t)(e - b * per);
    const int32_t r = v / a.dim, d = v - r * a.dim;
    const int64_t p = index[b];
    const bool ok = p >= 0 && p < n_paths;  // nothing is read for an index outside
    a.dst_dev[e] = ok ? a.src_dev[p * a.stride_path + r * a.stride_row + d * a.stride_dim]
                      : __builtin_nanf("");
  }
}

}  // namespace sdemc

using namespace sdemc;

extern "C" int sdemc_gather_paths(const sdemc_gather* arrays, int32_t n_arrays,
                                  const int64_t* index_dev, int64_t n_index, int64_t n_paths,
                                  void* stream) {
  if (!arrays || n_arrays < 1 || n_arrays > SDEMC_GATHER_MAX) return SDEMC_ERR_ARG;
  if (n_index < 0 || n_paths < 0 || (n_index > 0 && !index_dev)) return SDEMC_ERR_ARG;
  GatherArgs g = {};
  int64_t most = 0;
  for (int i = 0; i < n_arrays; ++i) {
    const sdemc_gather& a = arrays[i];
    if (a.rows < 0 || a.dim < 0) return SDEMC_ERR_ARG;
    const int64_t per = (int64_t)a.rows * a.dim;
    if (per > 0x7fffffffLL) return SDEMC_ERR_ARG;
    if (per > 0 && n_index > 0 && (!a.src_dev || !a.dst_dev)) return SDEMC_ERR_ARG;
    if (per * n_index > most) most = per * n_index;
    g.a[i] = a;
  }
  if (most == 0) return SDEMC_OK;
  int64_t blocks = (most + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_gather, dim3((unsigned)blocks, (unsigned)n_arrays), dim3(256), 0,
                     (hipStream_t)stream, g, index_dev, n_index, n_paths);
  return hipGetLastError() == hipSuccess ? SDEMC_OK : SDEMC_ERR_LAUNCH;
}
