// k_linear_grads.hip -- gradients of a Linear layer's parameters in training
// the control-variate networks: dW = dY^T X and db = the column sums of dY, for
// tall X [rows][n_in], dY [rows][n_out] of at most 63 and 64 columns, fp32.
//
// The product's result is a few kilobytes and its inner dimension the number
// of trajectory points of a batch (5e4), so all parallelism lies along that
// dimension: each wavefront multiplies its own rows on
// v_mfma_f32_32x32x2_f32 (fp32 throughout), reading both operands straight
// from memory as the instruction takes them -- 32 consecutive columns of two
// rows, whole lines -- with no staging; the 1 in column n_in of X makes db a
// column of the same product.  Partial results are summed in a fixed order:
// wavefronts of a workgroup in LDS, workgroups by k_linear_grads_sum.
// Off 64 bits (units of 2^-24 sum |terms|, 2048 to 50000 points): dW 0.03 to 0.10, the
// library's product 0.12 to 0.48; db 0.02 to 0.08, the library's sum, a tree, 0.01 to
// 0.06 (in fp64 beside the product db came to 0.002 to 0.010 in the same time; an
// epoch's weights then moved by up to 2e-3 for 2 of 10 shuffles, where a gradient
// almost vanishes and the optimiser divides by it, so the sums stay as they are).
// Bound by the latency of the operands' reads (20 MB, 4 us at the copy rate, 12 of
// the kernel's) and the second launch: both gradients of 48000 x 50 x 50 take 16 us, launches included, against 128 us
// for the library's product (tiles of the result without a split of the inner
// dimension: two workgroups) and bias sum; 36 against 504 us at 200000 rows.
#include "sdemc_core.h"

namespace sdemc {

typedef float lg_f32x16 __attribute__((ext_vector_type(16)));

constexpr int LG_WAVES = 4;           // per workgroup
constexpr int LG_STEPS = 8;           // row pairs whose loads are issued together
constexpr int LG_MIN_ROWS = 64;       // per wavefront at least
constexpr int LG_MAX_BLOCKS = 256;

struct LgShape {
  int64_t rows;
  int32_t n_in, n_out, rows_per_wave, blocks;
};

static inline LgShape lg_shape(int64_t rows, int32_t n_in, int32_t n_out) {
  LgShape s;
  s.rows = rows;
  s.n_in = n_in;
  s.n_out = n_out;
  int64_t per = (rows + LG_MAX_BLOCKS * LG_WAVES - 1) / (LG_MAX_BLOCKS * LG_WAVES);
  if (per < LG_MIN_ROWS) per = LG_MIN_ROWS;
  per = (per + 2 * LG_STEPS - 1) / (2 * LG_STEPS) * (2 * LG_STEPS);
  s.rows_per_wave = (int32_t)per;
  s.blocks = (int32_t)((rows + per * LG_WAVES - 1) / (per * LG_WAVES));
  return s;
}

// MT, NT: 32-wide tiles over the columns of dY and over those of X and the 1.
template <int MT, int NT>
__global__ __launch_bounds__(WAVE * LG_WAVES) void k_linear_grads(
    const float* __restrict__ x, const float* __restrict__ dy, const LgShape s,
    float* __restrict__ partials) {
  __shared__ float tile[LG_WAVES][MT * NT * 16 * WAVE];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int col = lane & 31, half = lane >> 5;
  const int64_t r0 = ((int64_t)blockIdx.x * LG_WAVES + wave) * s.rows_per_wave;
  int64_t r1 = r0 + s.rows_per_wave;
  if (r1 > s.rows) r1 = s.rows;
  lg_f32x16 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = lg_f32x16{};
  for (int64_t r = r0; r < r1; r += 2 * LG_STEPS) {
    float a[LG_STEPS][MT], b[LG_STEPS][NT];
#pragma unroll
    for (int t = 0; t < LG_STEPS; ++t) {
      const int64_t row = r + 2 * t + half;
      const bool in = row < r1;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int c = 32 * m + col;
        a[t][m] = in && c < s.n_out ? dy[row * s.n_out + c] : 0.0f;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int c = 32 * n + col;
        b[t][n] = in && c < s.n_in ? x[row * s.n_in + c] : (c == s.n_in ? 1.0f : 0.0f);
      }
    }
#pragma unroll
    for (int t = 0; t < LG_STEPS; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t][m], b[t][n], acc[m][n], 0, 0, 0);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int q = 0; q < 16; ++q) tile[wave][((m * NT + n) * 16 + q) * WAVE + lane] = acc[m][n][q];
  __syncthreads();
  constexpr int SIZE = MT * NT * 16 * WAVE;
  for (int e = threadIdx.x; e < SIZE; e += WAVE * LG_WAVES) {
    float v = tile[0][e];
#pragma unroll
    for (int w = 1; w < LG_WAVES; ++w) v += tile[w][e];
    partials[(int64_t)blockIdx.x * SIZE + e] = v;
  }
}

// Sum of the workgroups' partials: workgroup e / 64 takes the 64 elements of one
// accumulator of one tile (lane l: row 8 (q / 4) + 4 (l / 32) + q % 4, column
// l % 32), its 16 wavefronts a sixteenth of the partials each.
__global__ __launch_bounds__(1024) void k_linear_grads_sum(const float* __restrict__ partials,
                                                           int32_t blocks, int32_t size,
                                                           int32_t nt, int32_t n_in, int32_t n_out,
                                                           float* __restrict__ dw,
                                                           float* __restrict__ db) {
  __shared__ float part[16][WAVE];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int e = blockIdx.x * WAVE + lane;
  float v = 0.0f;
  for (int b = wave; b < blocks; b += 16) v += partials[(int64_t)b * size + e];
  part[wave][lane] = v;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < 16; ++w) v += part[w][lane];
  const int q = blockIdx.x & 15, t = blockIdx.x >> 4;
  const int o = 32 * (t / nt) + 8 * (q / 4) + 4 * (lane >> 5) + q % 4;
  const int i = 32 * (t % nt) + (lane & 31);
  if (o >= n_out) return;
  if (i < n_in) dw[(int64_t)o * n_in + i] = v;
  else if (i == n_in && db) db[o] = v;
}

}  // namespace sdemc

using namespace sdemc;

extern "C" {

size_t sdemc_linear_grads_floats(int64_t rows, int32_t n_in, int32_t n_out) {
  if (rows < 1 || n_in < 1 || n_in > 63 || n_out < 1 || n_out > 64) return 0;
  const int mt = (n_out + 31) / 32, nt = (n_in + 32) / 32;
  return (size_t)lg_shape(rows, n_in, n_out).blocks * (size_t)(mt * nt * 16 * WAVE);
}

int sdemc_linear_grads(const float* x_dev, const float* dy_dev, int64_t rows, int32_t n_in,
                       int32_t n_out, float* dw_dev, float* db_dev, float* workspace_dev,
                       size_t workspace_floats, void* stream) {
  const size_t need = sdemc_linear_grads_floats(rows, n_in, n_out);
  if (need == 0 || rows > (1LL << 37)) return SDEMC_ERR_ARG;
  if (!x_dev || !dy_dev || !dw_dev || !workspace_dev) return SDEMC_ERR_ARG;
  if (workspace_floats < need) return SDEMC_ERR_WORKSPACE;
  const LgShape s = lg_shape(rows, n_in, n_out);
  const int mt = (n_out + 31) / 32, nt = (n_in + 32) / 32;
  const dim3 g((unsigned)s.blocks), b(WAVE * LG_WAVES);
  const hipStream_t st = (hipStream_t)stream;
#define SDEMC_LG(M, N) \
  hipLaunchKernelGGL((k_linear_grads<M, N>), g, b, 0, st, x_dev, dy_dev, s, workspace_dev)
  if (mt == 1 && nt == 1) SDEMC_LG(1, 1);
  else if (mt == 1) SDEMC_LG(1, 2);
  else if (nt == 1) SDEMC_LG(2, 1);
  else SDEMC_LG(2, 2);
#undef SDEMC_LG
  hipLaunchKernelGGL(k_linear_grads_sum, dim3((unsigned)(mt * nt * 16)), dim3(1024), 0, st,
                     workspace_dev, s.blocks, mt * nt * 16 * WAVE, nt, n_in, n_out, dw_dev, db_dev);
  return hipGetLastError() == hipSuccess ? SDEMC_OK : SDEMC_ERR_LAUNCH;
}

}  // extern "C"
