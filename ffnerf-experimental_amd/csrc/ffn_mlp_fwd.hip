// ffn_mlp_fwd.hip -- the fp32 networks' forward: forward-only steps (previews, snapshots) and the forward over
// indexed samples (the marched render and the marched step's compositing input).
//
// Reference: ffnerf_OG.cl:1373-1466 (MLP fwd), 1505-1591 (compositing).
//
// MI355X design
//   * Where no training follows, the layers' products are fp32 products on bfloat16 matrix instructions, three planes
//     a value and eight terms a product (ffn_mlp_split.h): half the matrix cycles of the fp32 instruction, beside
//     vector instructions, and sums no further from 64 bits.  The marched step's forward has the training kernel's
//     own sums (k_mlp_fwd).
//   * A block of 16 wavefronts, one per CU, shares the weights in LDS (three bfloat16 planes, K-ordered rows); a
//     wavefront works alone (no barrier after the staging): 16 samples through all layers, activations in registers
//     in the D layout of one layer = the B operand of the next (K slot j of lane group g in block kb is neuron
//     32 kb + 16 (j / 4) + 4 g + j % 4).  A forward-only step's wavefront takes a tile of 64 samples as four such
//     groups and composites it on its 64 lanes.
//   * What bounds it: matrix instructions and the vector instructions of the splits (5.5 per value) about alike.
//     Measured against the fp32-MFMA forward (three blocks of four wavefronts per CU, 16-byte weight staging): a
//     frame's first round of 3.0M samples 542 -> 418 us; a preview of 590,000 samples of the 64-feature model with two
//     density layers 166 -> 102 us.
//   * The split does not hold infinities (their m is not a number), and loses the lower planes of operands near the
//     smallest numbers.  A wavefront sees infinities in its sums (every sum of a sample with such a value is not a
//     number) and does those samples again on the fp32 instruction, with the weights from memory; a block whose staged
//     weights are not all in the split's range takes the fp32 instruction alone (a preview of 2^20 samples of a
//     diverged model: 0.58 ms, in the split's range 0.32; a sample and a lane per neuron at a time it took 15.8).
#include "ffn_device.h"
#include "ffn_kernels.h"
#include "ffn_mlp_common.h"
#include "ffn_mlp_split.h"

namespace ffn {

constexpr int VIEW_NT = 64 * MLP_VIEW_WAVES;

// LDS: the colour output layer, the biases, then the other layers' weights (three planes or fp32 rows)
template <int LF_, int ND_, int NC_>
struct ArchF {
  static constexpr int LF = LF_, ND = ND_, NC = NC_;
  static constexpr int OUT_P = FFN_M + 4;  // the colour output layer: four fp32 rows (the last one zero)
  static constexpr int b_off(int k) {
    int o = 4 * OUT_P;
    for (int j = 0; j < k; ++j) o += layer_active(j, ND, NC) ? (j == FFN_WC_OUT ? 4 : layer_out(j)) : 0;
    return o;
  }
  static constexpr int w_base() { return b_off(FFN_N_LAYERS); }
  static_assert(w_base() % 4 == 0, "16-byte aligned weights");
  // layers on the split products (the colour output layer's three rows stay on fp32 4x4x1 MFMAs)
  static constexpr bool split(int k) { return layer_active(k, ND, NC) && k != FFN_WC_OUT; }
  static constexpr int cols(int k) { return layer_in(k, LF) < 32 ? 32 : layer_in(k, LF); }
  // row pitch in halves: the 8-half pad keeps the 16-byte reads aligned and spreads a tile's rows over the banks
  static constexpr int pitch(int k) { return cols(k) + 8; }
  static constexpr int sz(int k) { return split(k) ? layer_out(k) * pitch(k) : 0; }
  static constexpr int w_off(int k) {  // of plane 0, in halves after w_base; plane p follows at p * plane()
    int o = 0;
    for (int j = 0; j < k; ++j) o += sz(j);
    return o;
  }
  static constexpr int plane() { return w_off(FFN_N_LAYERS); }
  static constexpr int w_floats() { return w_base() + 3 * plane() / 2; }
  static_assert(plane() % 8 == 0, "16-byte aligned planes");
  // the same as fp32 rows (pitch in + 4, as in the training kernel)
  static constexpr int pitch32(int k) { return layer_in(k, LF) + 4; }
  static constexpr int off32(int k) {
    int o = w_base();
    for (int j = 0; j < k; ++j) o += split(j) ? layer_out(j) * pitch32(j) : 0;
    return o;
  }
  static constexpr int floats32() { return off32(FFN_N_LAYERS); }
};

// position of input neuron n in a layer's K-ordered row: for the first layer lane group g holds neurons (LF / 4) g
// + kk as slots kk of its K blocks (LF = 16: slots 0 .. 3 of one block), for the others see the file comment
template <int LF, int K>
__device__ __forceinline__ constexpr int row_pos(int n) {
  if constexpr (K == FFN_WD_IN) {
    constexpr int KA = LF / 4;
    const int g = n / KA, kk = n % KA;
    return 32 * (kk / 8) + 8 * g + kk % 8;
  } else {
    return neuron_kpos(n);
  }
}

// Whether the split holds a weight: zero, or its exponent at most 64 from 1's.  Beyond, infinities and "not a number"
// apart, the instruction's flush of operands below 2^-126 could take more of a product than its rounding does: a
// weight's lower planes below 2^-110, an input's at weights so large that the lost 2^-125 counts.
__device__ __forceinline__ bool split_holds(float w) {
  const uint32_t e = (__float_as_uint(w) >> 23) & 255u;
  return w == 0.0f || (e >= 127u - 64u && e <= 127u + 64u);
}

// stage the weights into LDS (split into planes) and the biases; returns whether the split holds this thread's weights
template <int LF, int ND, int NC>
__device__ __forceinline__ bool stage_split(float* __restrict__ sm, const MlpPtrs& wp, int tid) {
  using A = ArchF<LF, ND, NC>;
  __bf16* sW = reinterpret_cast<__bf16*>(sm + A::w_base());
  bool holds = true;
  read_weights<LF, ND, NC, VIEW_NT>(
      wp, tid,
      [&](auto K, int o, int i, const float4& v) {
        constexpr int k = K;
        if constexpr (k == FFN_WC_OUT) {
          *reinterpret_cast<float4*>(sm + o * A::OUT_P + i) = v;
        } else {
          const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int q = 0; q < 4; ++q) holds = holds && split_holds(x[q]);
          put_split4(sW + A::w_off(k) + o * A::pitch(k) + row_pos<LF, k>(i), A::plane(), x);  // consecutive positions
        }
      },
      [&](auto K, int o, float v) { sm[A::b_off(K) + o] = v; });
  if (tid < A::OUT_P) sm[3 * A::OUT_P + tid] = 0.0f;
  if constexpr (LF == 16) {  // the first layer's rows have 16 neurons in 32 positions
    constexpr int P = A::pitch(FFN_WD_IN);
    for (int e = tid; e < 3 * FFN_M * 4; e += VIEW_NT) {
      const int p = e / (FFN_M * 4), o = (e >> 2) % FFN_M, g = e & 3;
      *reinterpret_cast<uint2*>(sW + p * A::plane() + A::w_off(FFN_WD_IN) + o * P + 8 * g + 4) = make_uint2(0u, 0u);
    }
  }
  return holds;
}

// the same with fp32 rows
template <int LF, int ND, int NC>
__device__ __forceinline__ void stage_fp32(float* __restrict__ sm, const MlpPtrs& wp, int tid) {
  using A = ArchF<LF, ND, NC>;
  read_weights<LF, ND, NC, VIEW_NT>(
      wp, tid,
      [&](auto K, int o, int i, const float4& v) {
        constexpr int k = K;
        constexpr int at = k == FFN_WC_OUT ? 0 : A::off32(k), P = k == FFN_WC_OUT ? A::OUT_P : A::pitch32(k);
        *reinterpret_cast<float4*>(sm + at + o * P + i) = v;
      },
      [&](auto K, int o, float v) { sm[A::b_off(K) + o] = v; });
  if (tid < A::OUT_P) sm[3 * A::OUT_P + tid] = 0.0f;
}

// out tiles (D layout) = act(W . in + b) on the fp32 instruction, with the sums' order of the training kernels; W: the
// layer's rows of P floats, the weight of k-step kk of input tile tp at col(tp) + kk
template <int OT, int IT, class Col>
__device__ __forceinline__ void fwd_fp32(const float* __restrict__ W, bool aligned16, int P, const float* __restrict__ B,
                                         const floatx4 (&in)[4], floatx4 (&out)[4], int g, int s, bool relu, Col col) {
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    floatx4 acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = B[16 * t + 4 * g + r];
#pragma unroll
    for (int tp = 0; tp < IT; ++tp) {
      const float* w = W + (16 * t + s) * P + col(tp);
      floatx4 w4;
      if (aligned16) w4 = *reinterpret_cast<const floatx4*>(w);
      else w4 = floatx4{w[0], w[1], w[2], w[3]};
#pragma unroll
      for (int rp = 0; rp < 4; ++rp) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w4[rp], in[tp][rp], acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);  // (all weights' loads at once would spill)
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) out[t][r] = relu ? relu_f(acc[r]) : acc[r];
  }
}

// forward of the wavefront's 16 samples through both networks with fp32 products, the training kernel's sums bit for
// bit; W(k): layer k's weights, rows of in + PAD floats.  Returns the colours and the density network's first output.
template <int LF, int ND, int NC, int PAD, class Wt, class Tap>
__device__ __forceinline__ float4 fwd_nets_fp32(Wt W, bool al, const float* __restrict__ sm,
                                                const float (&a0r)[LF / 4], const float (&dir)[3], float sh_mult,
                                                int g, int s, Tap tap) {
  using A = ArchF<LF, ND, NC>;
  auto d_col = [&](int tp) { return 16 * tp + 4 * g; };
  floatx4 x[4], h[4];
#pragma unroll
  for (int q = 0; q < LF / 16; ++q) x[q] = floatx4{a0r[4 * q], a0r[4 * q + 1], a0r[4 * q + 2], a0r[4 * q + 3]};
  fwd_fp32<4, LF / 16>(W(FFN_WD_IN), al, LF + PAD, sm + A::b_off(FFN_WD_IN), x, h, g, s, true,
                       [&](int q) { return LF / 4 * g + 4 * q; });
  tap(0, h);
#pragma unroll
  for (int i = 1; i < ND; ++i) {
    const int k = i == 1 ? FFN_WD_01 : FFN_WD_12;
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = h[t];
    fwd_fp32<4, 4>(W(k), al, FFN_M + PAD, sm + A::b_off(k), x, h, g, s, true, d_col);
    tap(i, h);
  }
  floatx4 o1[4];
  fwd_fp32<1, 4>(W(FFN_WD_OUT), al, FFN_M + PAD, sm + A::b_off(FFN_WD_OUT), h, o1, g, s, false, d_col);
#pragma unroll
  for (int r = 0; r < 4; ++r) o1[1][r] = sh_component(dir, 4 * g + r) * sh_mult;
  fwd_fp32<4, 2>(W(FFN_WC_IN), al, FFN_C_IN + PAD, sm + A::b_off(FFN_WC_IN), o1, h, g, s, true, d_col);
  tap(3, h);
#pragma unroll
  for (int i = 1; i < NC; ++i) {
    const int k = i == 1 ? FFN_WC_01 : (i == 2 ? FFN_WC_12 : FFN_WC_23);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = h[t];
    fwd_fp32<4, 4>(W(k), al, FFN_M + PAD, sm + A::b_off(k), x, h, g, s, true, d_col);
    tap(3 + i, h);
  }
  float rgb[3];
  fwd_color_out(sm, sm + A::b_off(FFN_WC_OUT), A::OUT_P, h, g, s, rgb);
  return make_float4(rgb[0], rgb[1], rgb[2], o1[0][0]);
}

// the same for samples and weights that the split cannot hold: the weights straight from memory (the caches hold
// them), the biases and the colour output layer from LDS.  Not inlined: its registers would be spilled on the split's
// path.  b: the lane's sample (< 0: none); relu: its record of the ReLU tap (NULL: not written).
template <int LF, int ND, int NC, int FEAT, bool TAPS>
__device__ __noinline__ float4 fwd_samples_fp32(const MlpPtrs* __restrict__ wp, const float* __restrict__ sm,
                                                const float* __restrict__ a0, const FeatLayout* __restrict__ feat,
                                                int64_t b, float dx, float dy, float dz, float sh_mult,
                                                uint32_t* __restrict__ relu) {
  const int lane = threadIdx.x & 63, g = lane >> 4, s = lane & 15;
  float a0r[LF / 4];
  load_enc<LF, FEAT>(a0, *feat, b, b >= 0, g, a0r);
  const float dir[3] = {dx, dy, dz};
  return fwd_nets_fp32<LF, ND, NC, 0>([&](int k) { return wp->W[k]; }, wp->aligned16, sm, a0r, dir, sh_mult, g, s,
                                      [&](int layer, const floatx4 (&v)[4]) {
                                        if constexpr (TAPS) tap_relu(relu, layer, v, g);
                                      });
}

// forward of the wavefront's 16 samples through both networks on the split products; hd, hc: the hidden activations (for
// the ReLU tap).  Returns the samples (bit per sample) whose sums are not finite, to be done again by fwd_samples_fp32.
template <int LF, int ND, int NC>
__device__ __forceinline__ uint32_t fwd_samples_split(const float* __restrict__ sm, const float (&a0r)[LF / 4],
                                                      const float (&dirv)[3], float sh_mult, int g, int s,
                                                      floatx4 (&hd)[ND][4], floatx4 (&hc)[NC][4], float& dout0,
                                                      float (&rgb)[3]) {
  using A = ArchF<LF, ND, NC>;
  constexpr int PL = A::plane(), KB0 = A::cols(FFN_WD_IN) / 32;
  // an offset of zero that the compiler cannot see through: it would read the weights before the caller's loop and
  // spill them (200 to 900 bytes a lane)
  int zero = 0;
  __asm__ volatile("" : "+s"(zero));
  sm += zero;
  const __bf16* sW = reinterpret_cast<const __bf16*>(sm + A::w_base());
  float bad = 0.0f;
  Split8 x0[KB0];
#pragma unroll
  for (int kb = 0; kb < KB0; ++kb) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 8 * kb + j < LF / 4 ? a0r[8 * kb + j] : 0.0f;
    x0[kb] = split8(v);
  }
  fwd_split<4, KB0>(sW + A::w_off(FFN_WD_IN), PL, A::pitch(FFN_WD_IN), sm + A::b_off(FFN_WD_IN), x0, hd[0], g, s, true,
                    bad);
  Split8 x[2];
#pragma unroll
  for (int i = 1; i < ND; ++i) {
    const int k = i == 1 ? FFN_WD_01 : FFN_WD_12;
    split_tiles(hd[i - 1], x);
    fwd_split<4, 2>(sW + A::w_off(k), PL, A::pitch(k), sm + A::b_off(k), x, hd[i], g, s, true, bad);
  }
  split_tiles(hd[ND - 1], x);
  floatx4 o1[1];
  fwd_split<1, 2>(sW + A::w_off(FFN_WD_OUT), PL, A::pitch(FFN_WD_OUT), sm + A::b_off(FFN_WD_OUT), x, o1, g, s, false,
                   bad);
  dout0 = o1[0][0];
  floatx4 cin[2];
  cin[0] = o1[0];
#pragma unroll
  for (int r = 0; r < 4; ++r) cin[1][r] = sh_component(dirv, 4 * g + r) * sh_mult;
  Split8 xc[1];
  split_tiles(cin, xc);
  fwd_split<4, 1>(sW + A::w_off(FFN_WC_IN), PL, A::pitch(FFN_WC_IN), sm + A::b_off(FFN_WC_IN), xc, hc[0], g, s, true,
                  bad);
#pragma unroll
  for (int i = 1; i < NC; ++i) {
    const int k = i == 1 ? FFN_WC_01 : (i == 2 ? FFN_WC_12 : FFN_WC_23);
    split_tiles(hc[i - 1], x);
    fwd_split<4, 2>(sW + A::w_off(k), PL, A::pitch(k), sm + A::b_off(k), x, hc[i], g, s, true, bad);
  }
  fwd_color_out(sm, sm + A::b_off(FFN_WC_OUT), A::OUT_P, hc[NC - 1], g, s, rgb);
  return (uint32_t)__ballot(bad != 0.0f) & 0xFFFFu;  // not a number in all four lanes of a sample alike
}

// The forward over indexed samples.  SPLIT: the render's.  Without it the marched training step's, whose backward
// recomputes the activations in fp32 (k_mlp): the forward's sums are the same bit for bit, so the loss gradients belong
// to the activations and ReLU branches that the backward uses (880,000 samples of the 32-feature model: 160 us; with the
// split's sums the step, 1.45 ms, was not 1 % faster).
template <int LF, int ND, int NC, int FEAT, bool SPLIT>
__global__ __launch_bounds__(VIEW_NT) void k_mlp_fwd(MlpPtrs wp, const float* __restrict__ a0, FeatLayout feat,
                                                     const float4* __restrict__ rays,
                                                     const uint32_t* __restrict__ ray_ids, int64_t n, float sh_mult,
                                                     float* __restrict__ sigma, float* __restrict__ rgb,
                                                     const uint32_t* __restrict__ n_dev) {
  extern __shared__ __align__(16) float smv[];
  if (n_dev) {  // the count of a launch sized for a capacity, read on the device
    const int64_t nd = (int64_t)*n_dev;
    n = nd < n ? nd : n;
  }
  if ((int64_t)blockIdx.x * 16 >= n) return;  // no samples for this block: skip staging the weights
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, s = lane & 15;
  bool split_ok = false;
  if constexpr (SPLIT) {
    split_ok = __syncthreads_and(stage_split<LF, ND, NC>(smv, wp, tid));
  } else {
    stage_fp32<LF, ND, NC>(smv, wp, tid);
    __syncthreads();
  }
  // groups of 16 samples: a block's first, then its second ..., so that few groups spread over the blocks
  for (int64_t grp = (int64_t)blockIdx.x + (int64_t)gridDim.x * wave; grp * 16 < n;
       grp += (int64_t)gridDim.x * MLP_VIEW_WAVES) {
    const int64_t b = grp * 16 + s;
    const bool valid = b < n;
    float dirv[3] = {0.0f, 0.0f, 1.0f};
    if (valid) {
      const float4 rd = rays[2 * (size_t)ray_ids[b] + 1];
      dirv[0] = rd.x;
      dirv[1] = rd.y;
      dirv[2] = rd.z;
    }
    float dout0, c[3];
    uint32_t redo = 0xFFFFu;
    if constexpr (!SPLIT) {
      float a0r[LF / 4];
      load_enc<LF, FEAT>(a0, feat, b, valid, g, a0r);
      int zero = 0;  // as in fwd_samples_split
      __asm__ volatile("" : "+s"(zero));
      const float* sm = smv + zero;
      const float4 f = fwd_nets_fp32<LF, ND, NC, 4>([&](int k) { return sm + ArchF<LF, ND, NC>::off32(k); }, true, sm,
                                                    a0r, dirv, sh_mult, g, s, [](int, const floatx4 (&)[4]) {});
      c[0] = f.x;
      c[1] = f.y;
      c[2] = f.z;
      dout0 = f.w;
      redo = 0u;
    } else if (split_ok) {
      float a0r[LF / 4];
      load_enc<LF, FEAT>(a0, feat, b, valid, g, a0r);
      floatx4 hd[ND][4], hc[NC][4];
      redo = fwd_samples_split<LF, ND, NC>(smv, a0r, dirv, sh_mult, g, s, hd, hc, dout0, c);
    }
    if (SPLIT && redo) {  // the other samples keep their results, which so do not depend on their neighbours
      const MlpPtrs w = wp;  // (a copy: a kernel argument whose address is taken is read from memory everywhere)
      const FeatLayout lay = feat;
      const float4 f = fwd_samples_fp32<LF, ND, NC, FEAT, false>(&w, smv, a0, &lay, valid ? b : -1, dirv[0],
                                                                 dirv[1], dirv[2], sh_mult, nullptr);
      if ((redo >> s) & 1u) {
        c[0] = f.x;
        c[1] = f.y;
        c[2] = f.z;
        dout0 = f.w;
      }
    }
    if (g == 0 && valid) {
      sigma[b] = softplus(fminf(fmaxf(dout0, -10.0f), 10.0f));
      rgb[3 * b] = c[0];
      rgb[3 * b + 1] = c[1];
      rgb[3 * b + 2] = c[2];
    }
  }
}

// A forward-only step: tiles of 64 samples, one per wavefront at a time (a.tile_order puts the busy ones first).
template <int LF, int ND, int NC, int FEAT, bool TAPS, int SC>
__global__ __launch_bounds__(VIEW_NT) void k_mlp_view(MlpArgs a) {
  using A = ArchF<LF, ND, NC>;
  extern __shared__ __align__(16) float smv[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, s = lane & 15;
  const int log2S = a.log2S;
  const uint64_t n_samples = (uint64_t)a.num_rays << log2S;
  const bool split_ok = __syncthreads_and(stage_split<LF, ND, NC>(smv, a.w, tid));
  float* sSig = smv + A::w_floats() + 256 * wave;  // sigma[64], rgb[64][3] of the wavefront's tile
  float* sRgb = sSig + 64;
  const float Dhalf = half_box_diagonal(a.c);
  const int64_t first = (int64_t)blockIdx.x + (int64_t)gridDim.x * wave, step = (int64_t)gridDim.x * MLP_VIEW_WAVES;
  int64_t n_full = a.n_tiles;
  if constexpr (!TAPS) {
    if (a.tile_order) n_full = (int64_t)*a.n_busy;
    else if (a.tile_busy && first < a.n_tiles && !a.tile_busy[first]) n_full = 0;
  }
  int64_t ti = first;
#pragma unroll 1
  for (; ti < n_full; ti += step) {
    const int64_t tile = a.tile_order ? (int64_t)a.tile_order[ti] : ti;
#pragma unroll 1
    for (int cb = 0; cb < 4; ++cb) {
      const int col = 16 * cb + s;
      const int64_t b = tile * 64 + col;
      const bool valid = (uint64_t)b < n_samples;
      const float4 rd = a.rays[2 * (valid ? (b >> log2S) : 0) + 1];
      const float dirv[3] = {rd.x, rd.y, rd.z};
      float dout0, c[3];
      uint32_t* rec = TAPS && a.t_relu && valid ? a.t_relu + (int64_t)RELU_WORDS * b : nullptr;
      uint32_t redo = 0xFFFFu;
      if (split_ok) {
        float a0r[LF / 4];
        load_enc<LF, FEAT>(a.a0, a.feat, b, valid, g, a0r);
        floatx4 hd[ND][4], hc[NC][4];
        redo = fwd_samples_split<LF, ND, NC>(smv, a0r, dirv, a.sh_mult, g, s, hd, hc, dout0, c);
        if constexpr (TAPS) {
          if (a.t_relu) {
#pragma unroll
            for (int i = 0; i < ND; ++i) tap_relu(rec, i, hd[i], g);
#pragma unroll
            for (int i = 0; i < NC; ++i) tap_relu(rec, 3 + i, hc[i], g);
          }
        }
      }
      if (redo) {
        const bool mine = (redo >> s) & 1u;
        const MlpPtrs w = a.w;  // (as in k_mlp_fwd)
        const FeatLayout lay = a.feat;
        const float4 f = fwd_samples_fp32<LF, ND, NC, FEAT, TAPS>(&w, smv, a.a0, &lay, valid ? b : -1, rd.x, rd.y,
                                                                  rd.z, a.sh_mult, mine ? rec : nullptr);
        if (mine) {
          c[0] = f.x;
          c[1] = f.y;
          c[2] = f.z;
          dout0 = f.w;
        }
      }
      if (g == 0) {
        const float dt_b = valid ? a.DTs[b] : 0.0f;
        const float sig = softplus(fminf(fmaxf(dout0, -10.0f), 10.0f));
        sSig[col] = dt_b <= 0.0f ? 0.0f : sig;
        sRgb[3 * col] = c[0];
        sRgb[3 * col + 1] = c[1];
        sRgb[3 * col + 2] = c[2];
      }
    }
    const CompLane CL = load_comp_lane<SC>(a, tile, lane, true, n_samples, log2S, false);
    wave_lds_sync();
    float dLds, dLdc[3];
    composite_tile<TAPS, SC>(a, sSig, sRgb, CL, lane, 0, true, false, false, Dhalf, dLds, dLdc);
    wave_lds_sync();
  }
#pragma unroll 1
  for (; ti < a.n_tiles; ti += step) {
    const int64_t tile = a.tile_order ? (int64_t)a.tile_order[ti] : ti;
    const CompLane CL = load_comp_lane<SC>(a, tile, lane, false, n_samples, log2S, false);
    empty_tile<LF, FEAT, SC>(a, CL, lane, 0, 0, false, false, g);
  }
}

// ---------------------------------------------------------------------------

template <int LF, int ND, int NC, int FEAT, bool SPLIT>
static hipError_t launch_fwd_f(const MlpPtrs& w, const float* a0, const FeatLayout& feat, const float4* rays,
                               const uint32_t* ray_ids, int64_t n, float sh_mult, float* sigma, float* rgb,
                               int n_blocks, hipStream_t st, const uint32_t* n_dev) {
  using A = ArchF<LF, ND, NC>;
  const size_t lds = sizeof(float) * (size_t)(SPLIT ? A::w_floats() : A::floats32());
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_fwd<LF, ND, NC, FEAT, SPLIT>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_mlp_fwd<LF, ND, NC, FEAT, SPLIT>), dim3(n_blocks), dim3(VIEW_NT), lds, st, w, a0, feat, rays,
                     ray_ids, n, sh_mult, sigma, rgb, n_dev);
  return hipGetLastError();
}

template <int LF, int ND, int NC>
static hipError_t launch_fwd_t(const DevCfg& c, const MlpPtrs& w, const float* a0, const FeatLayout& feat,
                               const float4* rays, const uint32_t* ray_ids, int64_t n, float sh_mult, float* sigma,
                               float* rgb, bool train, int n_blocks, hipStream_t st, const uint32_t* n_dev) {
#define FFN_FWD(F)                                                                                                  \
  train ? launch_fwd_f<LF, ND, NC, F, false>(w, a0, feat, rays, ray_ids, n, sh_mult, sigma, rgb, n_blocks, st, n_dev) \
        : launch_fwd_f<LF, ND, NC, F, true>(w, a0, feat, rays, ray_ids, n, sh_mult, sigma, rgb, n_blocks, st, n_dev)
  switch (c.F) {
    case 1: return FFN_FWD(1);
    case 2: return FFN_FWD(2);
    case 4: return FFN_FWD(4);
    default: return hipErrorInvalidValue;
  }
#undef FFN_FWD
}

template <int LF, int ND, int NC, int FEAT, bool TAPS, int SC>
static hipError_t launch_view_f(const MlpArgs& a, int n_blocks, hipStream_t st) {
  const size_t lds = sizeof(float) * ((size_t)ArchF<LF, ND, NC>::w_floats() + 256 * MLP_VIEW_WAVES);
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)k_mlp_view<LF, ND, NC, FEAT, TAPS, SC>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_mlp_view<LF, ND, NC, FEAT, TAPS, SC>), dim3(n_blocks), dim3(VIEW_NT), lds, st, a);
  return hipGetLastError();
}

template <int LF, int ND, int NC, int SC>
static hipError_t launch_view_t(const MlpArgs& a, int n_blocks, hipStream_t st) {
  const bool taps = taps_requested(a);
  switch (a.c.F) {
    case 1:
      return taps ? launch_view_f<LF, ND, NC, 1, true, SC>(a, n_blocks, st)
                  : launch_view_f<LF, ND, NC, 1, false, SC>(a, n_blocks, st);
    case 2:
      return taps ? launch_view_f<LF, ND, NC, 2, true, SC>(a, n_blocks, st)
                  : launch_view_f<LF, ND, NC, 2, false, SC>(a, n_blocks, st);
    case 4:
      return taps ? launch_view_f<LF, ND, NC, 4, true, SC>(a, n_blocks, st)
                  : launch_view_f<LF, ND, NC, 4, false, SC>(a, n_blocks, st);
    default: return hipErrorInvalidValue;
  }
}

#define FFN_MLP_FWD_CONFIGS(X) \
  X(16, 1, 2)                  \
  X(32, 1, 2)                  \
  X(64, 1, 2)                  \
  X(16, 2, 2)                  \
  X(32, 2, 2)                  \
  X(64, 2, 2)

hipError_t launch_mlp_fwd(const DevCfg& c, const MlpPtrs& w, const float* a0, const FeatLayout& feat,
                          const float4* rays, const uint32_t* ray_ids, int64_t n, float sh_mult, float* sigma,
                          float* rgb, bool train, int LF, int nd, int nc, int n_blocks, hipStream_t st,
                          const uint32_t* n_dev) {
  if (n <= 0) return hipSuccess;
#define X(l, d, nn)                   \
  if (LF == l && nd == d && nc == nn) \
    return launch_fwd_t<l, d, nn>(c, w, a0, feat, rays, ray_ids, n, sh_mult, sigma, rgb, train, n_blocks, st, n_dev);
  FFN_MLP_FWD_CONFIGS(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_mlp_view(const MlpArgs& a, int LF, int nd, int nc, int n_blocks, hipStream_t st) {
#define X(l, d, n)                   \
  if (LF == l && nd == d && nc == n) \
    return a.S == 64 ? launch_view_t<l, d, n, 64>(a, n_blocks, st) : launch_view_t<l, d, n, 0>(a, n_blocks, st);
  FFN_MLP_FWD_CONFIGS(X)
#undef X
  return hipErrorInvalidValue;
}

}  // namespace ffn
