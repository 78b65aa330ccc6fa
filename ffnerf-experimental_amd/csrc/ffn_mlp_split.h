// ffn_mlp_split.h -- fp32 products on bfloat16 matrix instructions (the forward-only networks' layers).
//
// Every fp32 value x is the exact sum of three bfloat16 values: h = x's top 16 bits, m = the top 16 bits of x - h,
// l = x - h - m (8 + 8 + 8 significand bits; the differences are exact while l is not below 2^-126).  With h in
// [1, 2) m is below 2^-7 and l below 2^-15, all of x's sign, so of the nine terms of a product a b the last, l l, is
// below 2^-30 of it; the other eight are taken, each exact on v_mfma_f32_16x16x32_bf16, which adds 32 products to its
// fp32 accumulator.  Left out, the two terms m l and l m would take up to 2^-21 from a product, always toward zero.
//
// The h h terms have an accumulator of their own, which starts at the bias; the seven smaller ones share another,
// whose roundings are 2^-7 of the sum's, and the two are added last.  So a sum of 32 products is rounded about twice
// in all, where the fp32 instruction rounds after each of eight K = 4 steps.  Error against 64-bit sums, 2-norm and
// (largest over the sum of |products|), K = 64; fp32 instruction / eight terms so / in one accumulator / six of them:
//   normal values     1.44e-7 (2.5e-7) / 4.9e-8 (0.9e-7) / 9.7e-8 (1.9e-7) / 1.10e-7 (2.3e-7)
//   positive values   1.15e-7 (5.6e-7) / 4.7e-8 (2.1e-7) / 7.4e-8 (4.3e-7) / 8.3e-8 (4.4e-7)
//   one product       2.5e-8 (6.0e-8) / 2.5e-8 (6.0e-8) / 3.5e-8 (1.2e-7) / 7.4e-8 (4.6e-7)
//   three products    3.6e-8 (1.5e-7) / 2.6e-8 (1.2e-7) / 5.2e-8 (2.9e-7) / 7.8e-8 (4.3e-7)
//
// What bounds it: matrix instructions of 16 cycles (the fp32 one: 32, measured), eight for 32 products as with fp32,
// so half the matrix cycles; unlike the fp32 ones they run beside vector instructions.
#pragma once
#include "ffn_device.h"

namespace ffn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float top16(float x) { return __int_as_float(__float_as_int(x) & (int)0xFFFF0000); }
// {x1's upper half, x0's upper half}
__device__ __forceinline__ uint32_t upper_halves(float x1, float x0) {
  return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}

// eight values of a K block, as three bfloat16 operands
struct Split8 {
  bf16x8 h, m, l;
};
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float x0 = x[2 * q], x1 = x[2 * q + 1];
    const float r0 = x0 - top16(x0), r1 = x1 - top16(x1);
    const float l0 = r0 - top16(r0), l1 = r1 - top16(r1);
    h[q] = upper_halves(x1, x0);
    m[q] = upper_halves(r1, r0);
    l[q] = upper_halves(l1, l0);
  }
  Split8 s;
  s.h = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
  s.m = __builtin_bit_cast(bf16x8, make_uint4(m[0], m[1], m[2], m[3]));
  s.l = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
  return s;
}
// four consecutive values of a K-ordered row into its three planes
__device__ __forceinline__ void put_split4(__bf16* w, int plane, const float (&x)[4]) {
  float r[4], l[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    r[q] = x[q] - top16(x[q]);
    l[q] = r[q] - top16(r[q]);
  }
  *reinterpret_cast<uint2*>(w) = make_uint2(upper_halves(x[1], x[0]), upper_halves(x[3], x[2]));
  *reinterpret_cast<uint2*>(w + plane) = make_uint2(upper_halves(r[1], r[0]), upper_halves(r[3], r[2]));
  *reinterpret_cast<uint2*>(w + 2 * plane) = make_uint2(upper_halves(l[1], l[0]), upper_halves(l[3], l[2]));
}
// the K blocks of D-layout tiles
template <int IT>
__device__ __forceinline__ void split_tiles(const floatx4 (&t)[IT], Split8 (&o)[IT / 2]) {
#pragma unroll
  for (int kb = 0; kb < IT / 2; ++kb) {
    const float x[8] = {t[2 * kb][0],     t[2 * kb][1],     t[2 * kb][2],     t[2 * kb][3],
                        t[2 * kb + 1][0], t[2 * kb + 1][1], t[2 * kb + 1][2], t[2 * kb + 1][3]};
    o[kb] = split8(x);
  }
}

// out tiles (D layout) = act(W . in + b), two output tiles at a time so that consecutive MFMAs are independent; the
// smaller terms have accumulators of their own (see above).  W: plane 0 of the layer's K-ordered rows, plane p p *
// plane halves further.  bad becomes not a number where the sample's sums are infinite or not numbers
template <int OT, int KB>
__device__ __forceinline__ void fwd_split(const __bf16* __restrict__ W, int plane, int P, const float* __restrict__ B,
                                          const Split8 (&in)[KB], floatx4 (&out)[OT], int g, int s, bool relu,
                                          float& bad) {
  const __bf16* wrow = W + s * P + 8 * g;
  constexpr int G = OT < 2 ? OT : 2;
#pragma unroll
  for (int t0 = 0; t0 < OT; t0 += G) {
    floatx4 acc[G], low[G];
#pragma unroll
    for (int t = 0; t < G; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] = B[16 * (t0 + t) + 4 * g + r];
      low[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      bf16x8 wh[G], wm[G], wl[G];
#pragma unroll
      for (int t = 0; t < G; ++t) {
        const __bf16* w = wrow + 16 * (t0 + t) * P + 32 * kb;
        wh[t] = *reinterpret_cast<const bf16x8*>(w);
        wm[t] = *reinterpret_cast<const bf16x8*>(w + plane);
        wl[t] = *reinterpret_cast<const bf16x8*>(w + 2 * plane);
      }
      auto term = [&](floatx4 (&sum)[G], const bf16x8 (&w)[G], const bf16x8& x) {
#pragma unroll
        for (int t = 0; t < G; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t], x, sum[t], 0, 0, 0);
      };
      term(low, wl, in[kb].m);
      term(low, wm, in[kb].l);
      term(low, wl, in[kb].h);
      term(low, wh, in[kb].l);
      term(low, wm, in[kb].m);
      term(low, wm, in[kb].h);
      term(low, wh, in[kb].m);
      term(acc, wh, in[kb].h);
    }
#pragma unroll
    for (int t = 0; t < G; ++t) acc[t] = acc[t] + low[t];
    if (t0 == 0) bad = fmaf(acc[0][0], 0.0f, bad);
#pragma unroll
    for (int t = 0; t < G; ++t) {
      if (relu) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = relu_f(acc[t][r]);
      }
      out[t0 + t] = acc[t];
    }
  }
}

}  // namespace ffn
