// k_cv_pack.hip -- a control-variate network's parameters, already on the
// device, packed into the bf16 MFMA operand words of include/sdemc.h in one
// launch: eval-mode batch norms folded into the neighbouring Linear layers in
// fp64 and each word rounded as the host packer rounds it (fp64 -> fp32 ->
// bf16, nearest even), so both give the same words.  A packed network of three
// hidden layers is 22 blocks of 512 words, one workgroup each; the cost of the
// host packer was its ten copies to the host, each waiting for the device
// (mc_apply_cvs of 2^18 Merton paths x 300 steps with an f and a g: 4.35 ms packed
// on the host, 2.58 ms packed here with workgroups of eight wavefronts).
#include "cv_mlp.h"

#pragma clang fp contract(off)

namespace sdemc {

struct CvPackArgs {
  sdemc_cv_layer l[SDEMC_CV_MAX_HIDDEN + 1];
  int32_t hidden;
};

// scale and shift of feature i of a batch norm (identity when absent)
static __device__ void bn_affine(const sdemc_cv_bn& b, int i, double& s, double& c) {
  s = 1.0;
  c = 0.0;
  if (!b.var_dev) return;
  s = (b.weight_dev ? (double)b.weight_dev[i] : 1.0) / sqrt((double)b.var_dev[i] + b.eps);
  c = (b.bias_dev ? (double)b.bias_dev[i] : 0.0) - s * (double)b.mean_dev[i];
}

// Element [o][i] of layer l's padded matrix (cv.padded_matrices).
static __device__ double cv_element(const sdemc_cv_layer& l, bool last, int o, int i) {
  if (o == l.out && i == l.in && !last) return 1.0;  // the constant unit carries on
  if (o >= l.out || i > l.in) return 0.0;
  double v;
  double s, c;
  if (i < l.in) {
    v = (double)l.weight_dev[(int64_t)o * l.in + i];
    if (l.pre.var_dev) {
      bn_affine(l.pre, i, s, c);
      v = v * s;
    }
  } else {
    v = l.bias_dev ? (double)l.bias_dev[o] : 0.0;
    if (l.pre.var_dev) {
      double dot = 0.0;
      for (int k = 0; k < l.in; ++k) {
        bn_affine(l.pre, k, s, c);
        dot += (double)l.weight_dev[(int64_t)o * l.in + k] * c;
      }
      v = v + dot;
    }
  }
  if (l.post.var_dev) {
    bn_affine(l.post, o, s, c);
    v = s * v;
    if (i == l.in) v = v + c;
  }
  return v;
}

__global__ __launch_bounds__(256) void k_cv_pack(const CvPackArgs a, uint16_t* __restrict__ words) {
  const int blk = blockIdx.x;
  const int H = a.hidden;
  int layer, m, c;
  if (blk < 2) {
    layer = 0;
    m = blk;
    c = 0;
  } else if (blk < 2 + 8 * (H - 1)) {
    layer = 1 + (blk - 2) / 8;
    m = ((blk - 2) % 8) / 4;
    c = (blk - 2) % 4;
  } else {
    layer = H;
    m = 0;
    c = blk - 2 - 8 * (H - 1);
  }
  const sdemc_cv_layer& l = a.l[layer];
  for (int w = threadIdx.x; w < CV_BLOCK_WORDS; w += 256) {
    const int lane = w / 8, q = w % 8, h = lane / 32;
    const int o = 32 * m + lane % 32;
    const int i = layer == 0 ? q : 16 * c + 8 * (q / 4) + 4 * h + q % 4;
    const uint32_t u = __float_as_uint((float)cv_element(l, layer == H, o, i));
    words[blk * CV_BLOCK_WORDS + w] =
        (uint16_t)(((uint64_t)u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
  }
}

}  // namespace sdemc

using namespace sdemc;

extern "C" int sdemc_cv_pack(const sdemc_cv_layer* layers, int32_t n_layers, int32_t n_in,
                             int32_t n_out, uint16_t* words_dev, void* stream) {
  if (!layers || !words_dev) return SDEMC_ERR_ARG;
  if (n_layers < 2 || n_layers > SDEMC_CV_MAX_HIDDEN + 1) return SDEMC_ERR_UNSUPPORTED;
  if (n_in < 1 || n_in + 1 > 8 || n_out < 1 || n_out > SDEMC_CV_MAX_OUT) return SDEMC_ERR_UNSUPPORTED;
  CvPackArgs a = {};
  a.hidden = n_layers - 1;
  int32_t width = n_in;
  for (int j = 0; j < n_layers; ++j) {
    const sdemc_cv_layer& l = layers[j];
    if (!l.weight_dev || l.in != width || l.out < 1) return SDEMC_ERR_ARG;
    if (j + 1 < n_layers ? l.out > 63 : l.out != n_out) return SDEMC_ERR_UNSUPPORTED;
    if ((l.pre.var_dev != nullptr) != (l.pre.mean_dev != nullptr) ||
        (l.post.var_dev != nullptr) != (l.post.mean_dev != nullptr))
      return SDEMC_ERR_ARG;
    a.l[j] = l;
    width = l.out;
  }
  hipLaunchKernelGGL(k_cv_pack, dim3((unsigned)cv_blocks(a.hidden)), dim3(256), 0,
                     (hipStream_t)stream, a, words_dev);
  return hipGetLastError() == hipSuccess ? SDEMC_OK : SDEMC_ERR_LAUNCH;
}
