// ffn_order.hip -- a spatial order of query points for the encode entry point.
//
// Points in no order touch a table vertex from wavefronts all over the GPU at different times: every corner of a
// table beyond the L2 is a cache line from further away (2^24 uniform points, 16 x 2^22 entries: 7.3 times the
// algorithmic bytes).  In Morton order the points around a vertex are neighbours, so its line is fetched about
// once.
//
// The order is a stable least-significant-digit radix sort of (key, index) pairs: three passes over 8 bits of a
// 24-bit Morton key (256 cells per axis).  A pass counts digits per block of 4096 pairs, scans the counts
// (digit-major), and moves each pair to its digit's place behind the equal ones before it: ranks come from ballots
// over the wavefront's lanes, which hold consecutive pairs, so equal keys keep their order and the result depends
// on the points alone.  2^24 points: 1.13 ms, 0.75 of them the last move, which reads the points in random order (a
// 64-byte sector for 12 bytes); the gather of 16 x 2^22 entries behind it 20.9 -> 12.1 ms (uniform points).
#include "ffn_device.h"
#include "ffn_kernels.h"

namespace ffn {

constexpr int OR_NT = 256, OR_ITEMS = 16, OR_TILE = OR_NT * OR_ITEMS, OR_DIGITS = 256;

// every third bit of the result is a bit of v (8 bits)
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
  v = (v | (v << 8)) & 0x0000F00Fu;
  v = (v | (v << 4)) & 0x000C30C3u;
  return (v | (v << 2)) & 0x00249249u;
}

__device__ __forceinline__ uint32_t morton_key(const DevCfg& c, const float* __restrict__ x, int64_t i) {
  const float pos[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
  float p[3];
  normalize_pos(c, pos, p);  // in [0, 1), also for non-finite coordinates
  return spread3((uint32_t)(p[0] * 256.0f)) | (spread3((uint32_t)(p[1] * 256.0f)) << 1) |
         (spread3((uint32_t)(p[2] * 256.0f)) << 2);
}

// digit counts of each block's pairs, [digit][block]; FIRST: the keys are made from the points (and kept)
template <bool FIRST>
__global__ __launch_bounds__(OR_NT) void k_order_count(DevCfg c, const float* __restrict__ x, int64_t n,
                                                       uint32_t* __restrict__ keys, const uint2* __restrict__ pairs,
                                                       int shift, uint32_t* __restrict__ counts) {
  __shared__ uint32_t cnt[OR_DIGITS];
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t b0 = (int64_t)blockIdx.x * OR_TILE;
#pragma unroll
  for (int q = 0; q < OR_ITEMS; ++q) {
    const int64_t i = b0 + q * OR_NT + threadIdx.x;
    if (i < n) {
      uint32_t k;
      if constexpr (FIRST) {
        k = morton_key(c, x, i);
        keys[i] = k;
      } else {
        k = pairs[i].x;
      }
      atomicAdd(&cnt[(k >> shift) & (OR_DIGITS - 1)], 1u);
    }
  }
  __syncthreads();
  counts[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = cnt[threadIdx.x];
}

// LAST: the pair's index goes to perm and its point to pts (16 bytes each), in order
template <bool FIRST, bool LAST>
__global__ __launch_bounds__(OR_NT) void k_order_move(const float* __restrict__ x, int64_t n,
                                                      const uint32_t* __restrict__ keys,
                                                      const uint2* __restrict__ in, int shift,
                                                      const uint32_t* __restrict__ offsets, uint2* __restrict__ out,
                                                      uint32_t* __restrict__ perm, float4* __restrict__ pts) {
  constexpr int NW = OR_NT / 64;
  __shared__ uint32_t cnt[NW][OR_DIGITS];  // a wavefront's pairs of a digit so far, then its first place
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int w = 0; w < NW; ++w) cnt[w][tid] = 0u;
  __syncthreads();
  // wavefront w holds the block's pairs [w OR_TILE / NW, ...), 64 consecutive ones per trip
  const int64_t w0 = (int64_t)blockIdx.x * OR_TILE + (int64_t)wave * (OR_TILE / NW);
  const uint64_t below = (1ull << lane) - 1ull;
  uint32_t key[OR_ITEMS], idx[OR_ITEMS], rank[OR_ITEMS];
#pragma unroll
  for (int q = 0; q < OR_ITEMS; ++q) {
    const int64_t i = w0 + 64 * q + lane;
    key[q] = 0u;
    idx[q] = 0u;
    if (i < n) {
      if constexpr (FIRST) {
        key[q] = keys[i];
        idx[q] = (uint32_t)i;
      } else {
        const uint2 p = in[i];
        key[q] = p.x;
        idx[q] = p.y;
      }
    }
  }
  volatile uint32_t* wcnt = cnt[wave];
#pragma unroll
  for (int q = 0; q < OR_ITEMS; ++q) {
    const bool valid = w0 + 64 * q + lane < n;
    const uint32_t d = (key[q] >> shift) & (OR_DIGITS - 1);
    uint64_t same = __ballot(valid);  // the valid lanes with this lane's digit
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t m = __ballot((d >> b) & 1u);
      same &= (d >> b) & 1u ? m : ~m;
    }
    const uint32_t before = wcnt[d];
    rank[q] = before + (uint32_t)__popcll(same & below);
    __builtin_amdgcn_wave_barrier();
    if (valid && (same & below) == 0ull) wcnt[d] = before + (uint32_t)__popcll(same);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    uint32_t at = offsets[(int64_t)tid * gridDim.x + blockIdx.x];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const uint32_t own = cnt[w][tid];
      cnt[w][tid] = at;
      at += own;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < OR_ITEMS; ++q) {
    if (w0 + 64 * q + lane >= n) continue;
    const uint32_t to = cnt[wave][(key[q] >> shift) & (OR_DIGITS - 1)] + rank[q];
    if constexpr (LAST) {
      const int64_t i = idx[q];
      perm[to] = idx[q];
      pts[to] = make_float4(x[3 * i], x[3 * i + 1], x[3 * i + 2], 0.0f);
    } else {
      out[to] = make_uint2(key[q], idx[q]);
    }
  }
}

size_t order_count_words(int64_t n) { return (size_t)OR_DIGITS * (size_t)((n + OR_TILE - 1) / OR_TILE); }

hipError_t launch_order_points(const DevCfg& c, const float* x, int64_t n, const OrderScratch& s, uint32_t* perm,
                               float4* pts, hipStream_t st) {
  const unsigned blocks = (unsigned)((n + OR_TILE - 1) / OR_TILE);
  const int64_t words = (int64_t)order_count_words(n);
  uint32_t* keys = reinterpret_cast<uint32_t*>(s.pairs[1]);  // read by the first move only, which writes pairs[0]
  const dim3 grid(blocks), nt(OR_NT);
  hipError_t e;
  hipLaunchKernelGGL(k_order_count<true>, grid, nt, 0, st, c, x, n, keys, (const uint2*)nullptr, 0, s.counts);
  if ((e = launch_scan_u32(s.counts, words, s.offsets, s.sums, s.total, st)) != hipSuccess) return e;
  hipLaunchKernelGGL((k_order_move<true, false>), grid, nt, 0, st, x, n, keys, (const uint2*)nullptr, 0, s.offsets,
                     s.pairs[0], (uint32_t*)nullptr, (float4*)nullptr);
  hipLaunchKernelGGL(k_order_count<false>, grid, nt, 0, st, c, x, n, (uint32_t*)nullptr, s.pairs[0], 8, s.counts);
  if ((e = launch_scan_u32(s.counts, words, s.offsets, s.sums, s.total, st)) != hipSuccess) return e;
  hipLaunchKernelGGL((k_order_move<false, false>), grid, nt, 0, st, x, n, (const uint32_t*)nullptr, s.pairs[0], 8,
                     s.offsets, s.pairs[1], (uint32_t*)nullptr, (float4*)nullptr);
  hipLaunchKernelGGL(k_order_count<false>, grid, nt, 0, st, c, x, n, (uint32_t*)nullptr, s.pairs[1], 16, s.counts);
  if ((e = launch_scan_u32(s.counts, words, s.offsets, s.sums, s.total, st)) != hipSuccess) return e;
  hipLaunchKernelGGL((k_order_move<false, true>), grid, nt, 0, st, x, n, (const uint32_t*)nullptr, s.pairs[1], 16,
                     s.offsets, (uint2*)nullptr, perm, pts);
  return hipGetLastError();
}

}  // namespace ffn
