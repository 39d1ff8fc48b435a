// Compression of one layer of a dense cache [H, T, D] into new tensors: what surrounds the scorer and the
// selection kernels (core/compressor.py:279-346).
//
//  dense_prologue_kernel : the step's scalars and the key pointer in device memory, where the scorer and
//                          the selection read them, and the folded statistics, in one launch
//  dense_gather_kernel   : kept rows of K and of V, and the keep lists as 64-bit indices
//
// A layer of 4096 tokens is 4 us of memory traffic; the step was host work: four host-to-device copies of a few
// numbers, twenty launches of ten libraries' operators around the scorer, 268 us a call.  One library call with seven
// launches (these two, preparation, scorer, statistics, combination, top-k) and no copy: 45 us.  Up to 16384 tokens three
// (tri_score_small.hip, which folds for itself, select_small_kernel and the gather): 28 us, of which the GPU works 20.
#include "tri_common.h"

namespace tri {
namespace {

// Head statistics [A][F][2], [A][F], [A][F] -> [A][3][F] (as fold_stats_kernel, whose real and imaginary
// parts come in arrays of their own), and the argument words.
__global__ void dense_prologue_kernel(DenseLaunch d, int n, int F) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx == 0) {
    *d.arg_key = d.k;
    d.arg_words[0] = d.T;
    d.arg_words[1] = d.round_start;
    d.arg_words[2] = d.budget;
  }
  if (idx >= n) return;
  const int a = idx / F, f = idx - a * F;
  const float r = d.q_mean[2 * idx], i = d.q_mean[2 * idx + 1], s = d.freq_scale[idx];
  const float qmag = __fsqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(r, r), __fmul_rn(i, i)), 1e-8f));
  const float coef = d.disable_mlr ? d.q_abs[idx] : __fsub_rn(d.q_abs[idx], qmag);
  float* o = d.folded + (int64_t)a * 3 * F;
  o[f] = d.disable_trig ? 0.f : s * r;
  o[F + f] = d.disable_trig ? 0.f : s * i;
  o[2 * F + f] = s * coef;
}

// 16 bytes per lane; blockIdx.y: K or V.  A copy of 256-byte rows from scattered places, a few MB in all: one
// launch for both sides instead of an expanded 64-bit index and a library gather each.
__global__ __launch_bounds__(256) void dense_gather_kernel(DenseLaunch d) {
  const bool is_v = blockIdx.y != 0;
  const int lanes = (is_v ? d.v_row_bytes : d.k_row_bytes) / 16;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / lanes;                              // h * budget + j
  const int c = (int)(i - row * lanes);
  if (row >= (int64_t)d.H * d.budget) return;
  const int h = (int)(row / d.budget);
  const int t = d.keep32[row];
  const char* src = reinterpret_cast<const char*>(is_v ? d.v : d.k) +
                    h * (is_v ? d.v_stride_head : d.k_stride_head) + t * (is_v ? d.v_stride_token : d.k_stride_token);
  uint4* dst = reinterpret_cast<uint4*>(is_v ? d.out_v : d.out_k) + i;
  *dst = reinterpret_cast<const uint4*>(src)[c];
  if (!is_v && c == 0) d.out_keep[row] = (int64_t)t;
}

}  // namespace

hipError_t launch_dense_prologue(const DenseLaunch& d, hipStream_t s) {
  const int F = d.D / 2, n = d.H * F;
  hipLaunchKernelGGL(dense_prologue_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, s, d, n, F);
  return hipGetLastError();
}

hipError_t launch_dense_gather(const DenseLaunch& d, hipStream_t s) {
  const int64_t items = (int64_t)d.H * d.budget * (max(d.k_row_bytes, d.v_row_bytes) / 16);
  hipLaunchKernelGGL(dense_gather_kernel, dim3((unsigned)ceil_div64(items, 256), 2), dim3(256), 0, s, d);
  return hipGetLastError();
}

}  // namespace tri
