// Test hook, not product code: one layer of 64 outputs over 32 or 64 inputs through the split products of
// ffn_mlp_split.h, and through the fp32 matrix instruction in the same order of inputs, so that a GPU test can compare
// both with float64 sums.  Built into tests/hip/libffn_probe_math.so beside the math probe.
#include <hip/hip_runtime.h>
#include "../../ffnerf-experimental_amd/csrc/ffn_mlp_split.h"

using namespace ffn;

// a wavefront per block: 16 samples
template <int KB, bool SPLIT>
__global__ __launch_bounds__(64) void k_probe_layer(const float* __restrict__ x, const float* __restrict__ W,
                                                    const float* __restrict__ B, float* __restrict__ out, int n) {
  constexpr int K = 32 * KB, P = K + 8, PLANE = 64 * P;
  __shared__ __align__(16) __bf16 sW[3 * PLANE];
  __shared__ float sB[64];
  const int lane = threadIdx.x, g = lane >> 4, s = lane & 15, b = blockIdx.x * 16 + s;
  for (int e = lane; e < 64 * K / 4; e += 64) {
    const int o = e / (K / 4), i = 4 * (e % (K / 4));
    const float w[4] = {W[o * K + i], W[o * K + i + 1], W[o * K + i + 2], W[o * K + i + 3]};
    put_split4(sW + o * P + neuron_kpos(i), PLANE, w);
  }
  sB[lane] = B[lane];
  __syncthreads();
  floatx4 in[2 * KB], res[4];
#pragma unroll
  for (int t = 0; t < 2 * KB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) in[t][r] = b < n ? x[(size_t)b * K + 16 * t + 4 * g + r] : 0.0f;
  if constexpr (SPLIT) {
    Split8 xs[KB];
    split_tiles(in, xs);
    float bad = 0.0f;
    fwd_split<4, KB>(sW, PLANE, P, sB, xs, res, g, s, false, bad);
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) res[t][r] = sB[16 * t + 4 * g + r];
#pragma unroll
      for (int tp = 0; tp < 2 * KB; ++tp)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          res[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(W[(16 * t + s) * K + 16 * tp + 4 * g + r], in[tp][r], res[t],
                                                        0, 0, 0);
    }
  }
  if (b < n) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(size_t)b * 64 + 16 * t + 4 * g + r] = res[t][r];
  }
}

// x [n][32 kb], W [64][32 kb], B [64] -> out [n][64], device arrays.  Returns 0, or 1 for bad arguments or a launch
// error.
extern "C" int ffn_probe_layer(int kb, int split, const float* x, const float* W, const float* B, float* out, int n) {
  if (kb < 1 || kb > 2 || n < 1) return 1;
  const dim3 grid((n + 15) / 16), block(64);
  if (kb == 1 && split) hipLaunchKernelGGL((k_probe_layer<1, true>), grid, block, 0, 0, x, W, B, out, n);
  else if (kb == 1) hipLaunchKernelGGL((k_probe_layer<1, false>), grid, block, 0, 0, x, W, B, out, n);
  else if (split) hipLaunchKernelGGL((k_probe_layer<2, true>), grid, block, 0, 0, x, W, B, out, n);
  else hipLaunchKernelGGL((k_probe_layer<2, false>), grid, block, 0, 0, x, W, B, out, n);
  if (hipGetLastError() != hipSuccess) return 1;
  return hipDeviceSynchronize() == hipSuccess ? 0 : 1;
}
