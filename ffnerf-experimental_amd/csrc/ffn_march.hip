// ffn_march.hip -- occupancy bitfield, DDA marcher with stream compaction, and
// the early-terminated front-to-back compositing of the forward render.
//
// The reference has no marcher: every ray gets S importance-resampled samples
// (ffnerf_OG.cl:1002-1250).  This path is new; its specification is the CPU
// definition in the oracle (ora_occ_bitfield, ora_march_ray, ora_render_ray),
// which these kernels follow operation for operation (no contraction), so the
// marched sample times are bit-identical.  Nearest reference analogues: the
// occupancy nibble read (ffnerf_OG.cl:477-483) and the compositing recurrence
// (ffnerf_OG.cl:1505-1591).
//
// MI355X design
//   * The bitfield holds one bit per cell (x fastest, 32 cells per word):
//     128^3 cells = 256 KiB, 256^3 = 2 MiB -- resident in each XCD's L2, so the
//     DDA's bit lookups never reach HBM after the first touch.
//   * Two walks give the same samples bit for bit.  The lattice walk (k_march_lattice) gives a ray's lattice
//     points to the wavefront's lanes and finds each one's cell by itself; the cell walk (k_march) gives a lane
//     a ray and steps from cell to cell, for lattices much finer than the grid (launch_march).
//   * The cell walk: one lane per ray.  Empty cells are skipped in one step: the first lattice
//     index past the cell's exit is computed directly and corrected to the exact
//     index the one-by-one walk of the specification reaches.
//   * Empty 8^3 blocks are crossed in one step: a summary (one bit per block,
//     4 KiB at 256^3) marks the blocks with any occupied cell, and in an empty
//     block the walk moves straight to the first cell past the block -- the
//     same cell, lattice index and step count the one-cell-at-a-time walk
//     reaches, because every crossing of a cell boundary is an event ordered
//     by (time, axis) and the block's first face event and the interior events
//     before it follow from the same boundary-time formula.  A jump costs
//     several cell steps and diverges from the lanes that step cells, so the
//     walk uses the summary only when at least half the blocks are empty (a
//     flag computed on the device with it): a field with isolated occupied
//     cells scattered everywhere, where nearly every block holds one, walks
//     cell by cell.
//   * Compaction: one walk writes each ray's samples to its own fixed run of
//     slots (max_steps, or the chunk, per ray) and its count; a scan of the
//     counts and a wavefront-per-ray copy pack them.  Where those slots do not
//     fit, two passes over the same deterministic walk: count, scan, emit to the
//     scanned slots.  A chunked variant keeps a 16-byte state per
//     ray so that the render can march, shade and composite a few samples per
//     ray per round and retire rays whose transmittance fell below T_stop.
#include <math.h>
#include <stdlib.h>

#include "ffn_device.h"
#include "ffn_kernels.h"
#include "ffn_mlp_common.h"

namespace ffn {

__global__ __launch_bounds__(256) void k_occ_bitfield(const uint32_t* __restrict__ occ, int G, uint32_t q_min,
                                                      uint32_t* __restrict__ bits, int64_t n_words) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= n_words) return;
  const int R = 2 * G;
  const int64_t n_cells = (int64_t)R * R * R;
  uint32_t out = 0;
  for (int j = 0; j < 32; ++j) {
    const int64_t i = w * 32 + j;
    if (i >= n_cells) break;
    const int x = (int)(i % R), y = (int)((i / R) % R), z = (int)(i / ((int64_t)R * R));
    const uint32_t word = occ[(x >> 1) + G * ((y >> 1) + G * (z >> 1))];
    const uint32_t sub = (uint32_t)((x & 1) | ((y & 1) << 1) | ((z & 1) << 2));
    const uint32_t q = ((word >> (4u * sub)) & 0xFu) + 1u;
    if (q >= q_min) out |= 1u << j;
  }
  bits[w] = out;
}

// Block summary: bit (bx + NB (by + NB bz)) of `blocks` is set when any cell of the 8^3 block (bx, by, bz) is
// occupied (NB = ceil(R / 8); the last block of an axis is partial when 8 does not divide R).  One lane per
// block, 64 blocks (two words) per wavefront.
__global__ __launch_bounds__(256) void k_occ_blocks(const uint32_t* __restrict__ bits, int R,
                                                    uint32_t* __restrict__ blocks, int64_t n_blocks) {
  constexpr int B = 8;
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int NB = (R + B - 1) / B;
  bool any = false;
  if (b < n_blocks) {
    const int bx = (int)(b % NB), by = (int)((b / NB) % NB), bz = (int)(b / ((int64_t)NB * NB));
    const int x0 = B * bx, n = (R - x0 < B ? R - x0 : B);
    const uint32_t mask = (1u << n) - 1u;
    const int y1 = (B * by + B < R ? B * by + B : R), z1 = (B * bz + B < R ? B * bz + B : R);
    uint32_t acc = 0;
    for (int z = B * bz; z < z1; ++z)
      for (int y = B * by; y < y1; ++y) {
        const int64_t i0 = x0 + (int64_t)R * (y + (int64_t)R * z);
        const uint32_t sh = (uint32_t)(i0 & 31);
        uint32_t w = bits[i0 >> 5] >> sh;
        if (sh + (uint32_t)n > 32u) w |= bits[(i0 >> 5) + 1] << (32u - sh);
        acc |= w & mask;
      }
    any = acc != 0;
  }
  const uint64_t bal = __ballot(any);
  const int lane = threadIdx.x & 63;
  const int64_t w0 = (b - lane) >> 5;  // the wavefront's first word (64 blocks, 64-aligned)
  const int64_t n_words = (n_blocks + 31) >> 5;
  if (lane == 0 && w0 < n_words) blocks[w0] = (uint32_t)bal;
  if (lane == 32 && w0 + 1 < n_words) blocks[w0 + 1] = (uint32_t)(bal >> 32);
}

// *use = 1 when at least half of the n_blocks summary bits are clear (one workgroup; fixed-order sum)
__global__ __launch_bounds__(256) void k_blocks_use(const uint32_t* __restrict__ blocks, int64_t n_blocks,
                                                    uint32_t* __restrict__ use) {
  __shared__ uint32_t part[256];
  const int64_t n_words = (n_blocks + 31) >> 5;
  uint32_t c = 0;
  for (int64_t w = threadIdx.x; w < n_words; w += 256) c += (uint32_t)__popc(blocks[w]);
  part[threadIdx.x] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t t = 0;
    for (int i = 0; i < 256; ++i) t += part[i];
    use[0] = 2 * t <= (uint64_t)n_blocks ? 1u : 0u;
  }
}

__device__ __forceinline__ float lattice_t(float t0, uint32_t k, float dt) { return t0 + ((float)k + 0.5f) * dt; }

// the first lattice index k' >= k with t_k' >= t_exit, as the one-cell-at-a-time walk reaches it
__device__ __forceinline__ uint32_t skip_lattice(float t0, uint32_t k, float dt, float t_exit) {
  if (!(lattice_t(t0, k, dt) < t_exit)) return k;
  float est = ceilf((t_exit - t0) / dt - 0.5f);
  uint32_t ke = k + 1;
  if (est > (float)ke) ke = est < 4.0e9f ? (uint32_t)est : 4000000000u;
  while (ke > k + 1 && !(lattice_t(t0, ke - 1, dt) < t_exit)) --ke;
  while (lattice_t(t0, ke, dt) < t_exit) ++ke;
  return ke;
}

// Rays per wavefront of k_march.  A lane walks one ray at a time and, when that ray is finished (or paused at
// the chunk budget), takes the next unclaimed ray of its wavefront's range: walks are 37 % as long as
// their wavefront's longest on average, so a lane per ray would leave most lanes idle.
constexpr uint32_t MARCH_RPW = 256;
constexpr int MARCH_CELLS_PER_CLAIM = 8;

// One lane's walk of one ray, advanced a cell at a time.  The sequence of operations per ray is the
// specification's (ora_march_ray): the same cells, exit times and lattice indices, so the emitted samples
// are bit-identical whatever order the lane meets its rays in.
template <bool EMIT>
struct RayWalk {
  MarchState st;
  float o[3], d[3], invd[3], t0, t1;
  int cc[3], step[3];
  uint32_t r, k, emitted;
  uint64_t base;
  int iter;
  // Exit time of the last empty cell walked, not yet applied to k.  The one-cell-at-a-time walk moves k past
  // every empty cell's exit time; those times never decrease along the walk and k' = first index >= k with
  // t_k' >= t is the same whether applied once per cell or once for the last cell of a run, so k is brought up
  // to date only where it is used: on entering an occupied cell and when the walk state is saved.
  float t_pend;
  bool done, paused;

  // claim ray rr; returns false when the ray has nothing to walk (it is then already finished)
  __device__ __forceinline__ bool start(const MarchArgs& a, uint32_t rr, const float (&cell)[3]) {
    r = rr;
    emitted = 0;
    iter = 0;
    t_pend = -__builtin_huge_valf();
    done = false;
    paused = false;
    st = a.state ? a.state[r] : MarchState{0u, 0u, 0u, MARCH_FRESH};
    if (st.flags & MARCH_DONE) return false;  // no state change, no samples
    const float4 ro = a.rays[2 * (size_t)r], rd = a.rays[2 * (size_t)r + 1];
    o[0] = ro.x; o[1] = ro.y; o[2] = ro.z;
    d[0] = rd.x; d[1] = rd.y; d[2] = rd.z;
    base = EMIT ? (a.slot_stride ? (uint64_t)r * a.slot_stride : (uint64_t)a.offsets[r]) : 0;
    float ta, tb;
    if (!ray_aabb(o, d, a.bmin, a.bmax, ta, tb)) {
      done = true;
      finish_state(a, false);
      return false;
    }
    t0 = fmaxf(ta, a.t_near);
    t1 = fminf(tb, a.t_far);
    if (!(t1 > t0)) {
      done = true;
      finish_state(a, false);
      return false;
    }
    const int R = a.res;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      invd[i] = (d[i] != 0.0f) ? (1.0f / d[i]) : __builtin_huge_valf();
      step[i] = d[i] > 0.0f ? 1 : (d[i] < 0.0f ? -1 : 0);
    }
    if (st.flags & MARCH_FRESH) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const float inv = (float)R / (a.bmax[i] - a.bmin[i]);
        const float p = o[i] + t0 * d[i];
        const int ci = (int)floorf((p - a.bmin[i]) * inv);
        cc[i] = ci < 0 ? 0 : (ci > R - 1 ? R - 1 : ci);
      }
      st.k = 0;
      st.n = 0;
    } else {
      cc[0] = (int)(st.cell & 1023u);
      cc[1] = (int)((st.cell >> 10) & 1023u);
      cc[2] = (int)((st.cell >> 20) & 1023u);
    }
    k = st.k;
    return true;
  }

  // The current cell's 8^3 block is empty: move to the first cell past it.  Every boundary crossing of the
  // one-cell-at-a-time walk is an event (time, axis) -- the walk takes the smallest time, the lower axis on
  // ties, and the ray's end t1 before any axis at equal time -- and an axis' crossing times do not decrease
  // along it.  So the walk leaves the block by the first of the block's faces in that order (or ends inside
  // it at t1), after exactly the interior crossings that precede that event; each time below is the walk's
  // own formula for the same boundary.  The caller guarantees at least 24 steps of iteration budget.
  __device__ __forceinline__ bool jump_block(const MarchArgs& a, const float (&cell)[3]) {
    constexpr int B = 8;
    const int R = a.res;
    int face[3];
    float e_best = t1;
    int j_best = -1;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int b0 = cc[i] & ~(B - 1), b1 = (b0 + B - 1 < R - 1 ? b0 + B - 1 : R - 1);
      face[i] = step[i] > 0 ? b1 : b0;
      if (step[i] == 0) continue;
      const float bound = a.bmin[i] + (float)(face[i] + (step[i] > 0 ? 1 : 0)) * cell[i];
      const float te = (bound - o[i]) * invd[i];
      if (te < e_best) {
        e_best = te;
        j_best = i;
      }
    }
    int n_steps = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (step[i] == 0) continue;
      if (i == j_best) {
        n_steps += (face[i] - cc[i]) * step[i] + 1;
        cc[i] = face[i] + step[i];
        continue;
      }
      // this axis' crossings before the exit event (at most B - 1: its own face comes after that event)
      int c = cc[i];
      for (;;) {
        const float bound = a.bmin[i] + (float)(c + (step[i] > 0 ? 1 : 0)) * cell[i];
        const float te = (bound - o[i]) * invd[i];
        if (!(te < e_best || (te == e_best && i < j_best))) break;
        c += step[i];
        ++n_steps;
      }
      cc[i] = c;
    }
    t_pend = e_best;  // k past the block's cells, where it is next used
    if (j_best < 0) {  // the ray ends inside the block
      done = true;
      return true;
    }
    bool out = false;  // static indices: a dynamic cc[j_best] would put the walk state in scratch memory
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i == j_best) out = cc[i] < 0 || cc[i] >= R;
    if (out) {
      done = true;
      return true;
    }
    iter += n_steps;
    return false;
  }

  // one cell of the walk; returns true when the ray is finished or paused for this call
  __device__ __forceinline__ bool advance(const MarchArgs& a, const float (&cell)[3], bool use_blocks) {
    const int R = a.res;
    // the cell's bit and its block's bit, loaded together
    const int64_t bi = cc[0] + (int64_t)R * (cc[1] + (int64_t)R * cc[2]);
    const uint32_t wcell = a.bits[bi >> 5];
    if (use_blocks && iter + 24 < 3 * R + 2) {
      const int NB = (R + 7) >> 3;
      const int64_t bb = (cc[0] >> 3) + (int64_t)NB * ((cc[1] >> 3) + (int64_t)NB * (cc[2] >> 3));
      if (!((a.blocks[bb >> 5] >> (bb & 31)) & 1u)) return jump_block(a, cell);
    }
    float t_exit = t1;
    int axis = -1;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (step[i] == 0) continue;
      const float bound = a.bmin[i] + (float)(cc[i] + (step[i] > 0 ? 1 : 0)) * cell[i];
      const float te = (bound - o[i]) * invd[i];
      if (te < t_exit) {
        t_exit = te;
        axis = i;
      }
    }
    const bool occ = (wcell >> (bi & 31)) & 1u;
    if (occ) {
      k = skip_lattice(t0, k, a.dt, t_pend);
      for (;;) {
        const float tk = lattice_t(t0, k, a.dt);
        if (!(tk < t_exit)) break;
        if (st.n + emitted >= a.max_steps) {
          done = true;
          break;
        }
        if (emitted >= a.chunk) {
          paused = true;
          break;
        }
        if (EMIT) {
          const uint64_t slot = base + emitted;
          if (slot < a.capacity) {
            a.samples[slot] = make_float4(o[0] + tk * d[0], o[1] + tk * d[1], o[2] + tk * d[2], tk);
            if (a.ray_ids) a.ray_ids[slot] = r;
          }
        }
        ++emitted;
        ++k;
      }
      if (done || paused) return true;
    } else {
      t_pend = t_exit;  // skip the empty cell (k is brought past t_exit where it is next used)
    }
    if (axis < 0) {
      done = true;
      return true;
    }
    // step into the next cell (static indices: the walk state stays in registers)
    int ncc = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i == axis) {
        cc[i] += step[i];
        ncc = cc[i];
      }
    }
    if (ncc < 0 || ncc >= R) {
      done = true;
      return true;
    }
    if (iter == 3 * R + 2) {
      done = true;
      return true;
    }
    ++iter;
    return false;
  }

  // the state kept for the next call (walked rays only)
  __device__ __forceinline__ void finish_state(const MarchArgs& a, bool walked) {
    if (EMIT && a.state) {
      if (walked) {
        st.k = skip_lattice(t0, k, a.dt, t_pend);
        st.cell = (uint32_t)cc[0] | ((uint32_t)cc[1] << 10) | ((uint32_t)cc[2] << 20);
      }
      st.n += emitted;
      st.flags = (st.flags & ~MARCH_FRESH) | (done ? MARCH_DONE : 0u);
      a.state[r] = st;
    }
  }
};

template <bool EMIT>
__global__ __launch_bounds__(256) void k_march(MarchArgs a) {
  if (a.gate && *a.gate == 0u) return;  // the whole launch: every ray has stopped
  const int lane = threadIdx.x & 63;
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint64_t r_begin = wave * MARCH_RPW;
  if (r_begin >= a.num_rays) return;  // the same on every lane of the wavefront
  const uint32_t r_end = (uint32_t)(r_begin + MARCH_RPW < a.num_rays ? r_begin + MARCH_RPW : a.num_rays);
  float cell[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) cell[i] = (a.bmax[i] - a.bmin[i]) / (float)a.res;
  const bool use_blocks = a.blocks && *a.blocks_use != 0u;  // the same for every lane
  uint32_t next = (uint32_t)r_begin;  // the wavefront's next unclaimed ray
  RayWalk<EMIT> w;
  bool have = false;  // this lane walks a ray
  for (;;) {
    // lanes without a ray claim the next rays of the range, in lane order
    const uint64_t need = __ballot(!have);
    if (!have) {
      const uint32_t rr = next + (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
      if (rr < r_end) {
        if (w.start(a, rr, cell)) {
          have = true;
        } else if (!EMIT || a.slot_stride) {
          a.counts[rr] = 0u;
        }
      }
    }
    next = next + (uint32_t)__popcll(need);
    if (next > r_end) next = r_end;
    if (__ballot(have) == 0ull) {
      if (next >= r_end) break;
      continue;
    }
    // a few cells per lane between claims: the claim's wavefront-wide bookkeeping is paid once per batch
#pragma unroll 1
    for (int j = 0; j < MARCH_CELLS_PER_CLAIM; ++j) {
      if (have && w.advance(a, cell, use_blocks)) {
        w.finish_state(a, true);
        if (!EMIT || a.slot_stride) a.counts[w.r] = w.emitted;
        have = false;
      }
    }
  }
}

// The lattice walk.  The cell walk's state at lattice point k follows from t_k alone: on every axis it has left
// exactly the cells whose exit time te(c) = (bmin + (c + (d > 0)) cell - o) / d is <= t_k, from the start cell on
// (it steps while the smallest exit time is <= t_k, and an axis' exit times never decrease along it).  So a
// lane takes a lattice point and finds its cell without walking: floor of the grid coordinate, which is that
// cell unless the point lies within the rounding of a face, where the exit times themselves decide.
//
// What bounds it: vector instructions (about 45 per point and lane) and the latency of the bit load, which the
// iterations of a ray overlap.  The cell walk serialises a ray's ~1.5 R cells on one lane: at 40,001 rays of the
// ball scene (R = 256, dt = sqrt(3)/1024) it left most of the chip idle (1.13 ms a walk; this one 0.05 ms).
// Both sides measured: march_takes_lattice.
//
// A wavefront sets up to 64 consecutive rays up at once, one per lane, and then takes them one at a time with
// the ray's values in scalar registers.
struct LatticeRay {
  float o[3], d[3], t0, t1;
  float p0[3], slope[3];  // grid coordinate at t0 and its slope per unit of t (the point's cell up to rounding)
  float eps;              // the largest rounding of a grid coordinate or exit time, in cells (any axis)
};

// the walk's exit time of cell c on an axis (dir = 1 when the ray ascends it)
__device__ __forceinline__ float cell_exit(float bmin, float cell, float o, float invd, int c, int dir) {
  const float bound = bmin + (float)(c + dir) * cell;
  return (bound - o) * invd;
}

// the walk's cell on one axis at lattice time tk, from the guess g; R or -1 once the walk has left the grid
__device__ __forceinline__ int exact_axis_cell(const MarchArgs& a, int i, float o, float d, float t0, float tk, float pf) {
  const int R = a.res;
  const float inv = (float)R / (a.bmax[i] - a.bmin[i]), cell = (a.bmax[i] - a.bmin[i]) / (float)R;
  const float p = o + t0 * d;
  int c0 = (int)floorf((p - a.bmin[i]) * inv);
  c0 = c0 < 0 ? 0 : (c0 > R - 1 ? R - 1 : c0);
  if (d == 0.0f || d != d) return c0;  // the walk never steps along this axis
  const float invd = 1.0f / d;
  const int step = d > 0.0f ? 1 : -1, dir = d > 0.0f ? 1 : 0;
  int g = (int)floorf(pf);
  g = g < 0 ? 0 : (g > R - 1 ? R - 1 : g);
  g = step > 0 ? (g > c0 ? g : c0) : (g < c0 ? g : c0);
  while (g != c0 && !(cell_exit(a.bmin[i], cell, o, invd, g - step, dir) <= tk)) g -= step;
  while (g >= 0 && g < R && cell_exit(a.bmin[i], cell, o, invd, g, dir) <= tk) g += step;
  return g;
}

constexpr int LATTICE_UNROLL = 2;  // 64-point groups whose bit loads are in flight together
// The most lattice points between a ray's entry and exit that the lattice walk takes; a longer ray (a direction
// far from unit length, whose steps are tiny) is walked cell by cell by its own lane.
constexpr float LATTICE_MAX_POINTS = 65536.0f;

template <bool EMIT>
__global__ __launch_bounds__(256) void k_march_lattice(MarchArgs a, uint32_t rays_per_wave) {
  if (a.gate && *a.gate == 0u) return;  // the whole launch: every ray has stopped
  const int lane = threadIdx.x & 63;
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint64_t r_begin = wave * rays_per_wave;
  if (r_begin >= a.num_rays) return;  // the same on every lane of the wavefront
  const uint32_t n_here = (uint32_t)(a.num_rays - r_begin < rays_per_wave ? a.num_rays - r_begin : rays_per_wave);
  const int R = a.res;

  // lane j sets up ray r_begin + j
  const uint32_t r_own = (uint32_t)r_begin + (uint32_t)lane;
  const bool own = (uint32_t)lane < n_here;
  LatticeRay L{};
  MarchState st{0u, 0u, 0u, MARCH_FRESH};
  bool have = false;
  if (own) {
    if (a.state) st = a.state[r_own];
    if (!(st.flags & MARCH_DONE)) {
      const float4 ro = a.rays[2 * (size_t)r_own], rd = a.rays[2 * (size_t)r_own + 1];
      L.o[0] = ro.x; L.o[1] = ro.y; L.o[2] = ro.z;
      L.d[0] = rd.x; L.d[1] = rd.y; L.d[2] = rd.z;
      float ta, tb;
      if (ray_aabb(L.o, L.d, a.bmin, a.bmax, ta, tb)) {
        L.t0 = fmaxf(ta, a.t_near);
        L.t1 = fminf(tb, a.t_far);
        have = L.t1 > L.t0;
      }
      if (have) {
        L.eps = 0.0f;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const float size = a.bmax[i] - a.bmin[i], inv = (float)R / size;
          const float p = L.o[i] + L.t0 * L.d[i];
          L.p0[i] = (p - a.bmin[i]) * inv;
          L.slope[i] = L.d[i] * inv;
          // With u = 2^-24, A the larger |bound| of the box, s its extent and D = max(|t0|, |t1|) |d| (with a negative
          // t_near the box can lie behind the origin), the coordinate p0 + tau slope is off by at most
          // u (2 D + A + 9 s) inv cells from the real one at t_k and a face's exit time by u (3 D + A + 3 s) inv; eps
          // doubles the sum (second-order terms, points a rounding outside the box).
          const float A = fmaxf(fabsf(a.bmin[i]), fabsf(a.bmax[i]));
          const float far = fmaxf(fabsf(L.t0), fabsf(L.t1));
          const float e = (5.0f * far * fabsf(L.d[i]) + 2.0f * A + 12.0f * size) * inv * (2.0f / 16777216.0f);
          L.eps = fmaxf(L.eps, e);
          if (!(e < 0.5f)) L.eps = 1.0f;  // (NaN included) every point takes the exact path
        }
      } else if (EMIT && a.state) {
        st.flags = (st.flags & ~MARCH_FRESH) | MARCH_DONE;
        a.state[r_own] = st;
      }
    }
  }
  if (st.flags & MARCH_FRESH) st.k = st.n = 0;
  uint32_t emitted = 0;  // of this lane's ray
  const bool by_cells = have && !(L.t1 - L.t0 <= LATTICE_MAX_POINTS * a.dt);
  if (by_cells) {
    float cell[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) cell[i] = (a.bmax[i] - a.bmin[i]) / (float)R;
    RayWalk<EMIT> w;
    if (w.start(a, r_own, cell)) {
      while (!w.advance(a, cell, false)) {
      }
      w.finish_state(a, true);
      emitted = w.emitted;
    }
    have = false;
  }
  const uint64_t below = (1ull << lane) - 1ull;

  for (uint64_t todo = __ballot(have); todo != 0ull; todo &= todo - 1ull) {
    const int j = (int)__builtin_ctzll(todo);
    auto rl = [&](float x) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), j)); };
    const uint32_t r = (uint32_t)r_begin + (uint32_t)j;
    float o[3], d[3], p0[3], slope[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      o[i] = rl(L.o[i]);
      d[i] = rl(L.d[i]);
      p0[i] = rl(L.p0[i]);
      slope[i] = rl(L.slope[i]);
    }
    const float t0 = rl(L.t0), t1 = rl(L.t1), near = 0.5f - rl(L.eps);
    const uint32_t n_before = (uint32_t)__builtin_amdgcn_readlane((int)st.n, j);
    uint32_t kb = (uint32_t)__builtin_amdgcn_readlane((int)st.k, j);
    // the call's samples: at most `chunk`, and max_steps over all calls
    const uint32_t left = a.max_steps > n_before ? a.max_steps - n_before : 0u;
    const uint32_t budget = left < a.chunk ? left : a.chunk;
    uint64_t base = 0;
    if (EMIT) base = a.slot_stride ? (uint64_t)r * a.slot_stride : (uint64_t)a.offsets[r];
    uint32_t found = 0;
    bool over = false;  // a sample past the budget: the ray pauses at it
    for (;;) {
      float tk[LATTICE_UNROLL];
      uint32_t word[LATTICE_UNROLL], bit[LATTICE_UNROLL];
      bool in[LATTICE_UNROLL];
#pragma unroll
      for (int u = 0; u < LATTICE_UNROLL; ++u) {
        const float tau = ((float)(kb + 64u * u + (uint32_t)lane) + 0.5f) * a.dt;
        tk[u] = t0 + tau;
        in[u] = tk[u] < t1;
        float pf[3];
        int c[3];
        bool exact = false;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          pf[i] = fmaf(tau, slope[i], p0[i]);
          const float fl = floorf(pf[i]);
          c[i] = (int)fl;
          exact |= !(fabsf((pf[i] - fl) - 0.5f) < near);
        }
        // c outside the grid and not within the rounding of its faces: the walk has left it (or the point
        // lies before the start cell, which the exact path decides)
        exact |= (uint32_t)c[0] >= (uint32_t)R || (uint32_t)c[1] >= (uint32_t)R || (uint32_t)c[2] >= (uint32_t)R;
        if (exact && in[u]) {
#pragma unroll
          for (int i = 0; i < 3; ++i) c[i] = exact_axis_cell(a, i, o[i], d[i], t0, tk[u], pf[i]);
        }
        const bool inside = (uint32_t)c[0] < (uint32_t)R && (uint32_t)c[1] < (uint32_t)R && (uint32_t)c[2] < (uint32_t)R;
        const uint32_t bi = (uint32_t)c[0] + (uint32_t)R * ((uint32_t)c[1] + (uint32_t)R * (uint32_t)c[2]);
        bit[u] = bi & 31u;
        word[u] = (in[u] && inside) ? a.bits[bi >> 5] : 0u;
      }
      bool end = false;
#pragma unroll
      for (int u = 0; u < LATTICE_UNROLL; ++u) {
        const bool occ = (word[u] >> bit[u]) & 1u;
        const uint64_t m = __ballot(occ);
        if (m != 0ull && !over) {
          const uint32_t idx = found + (uint32_t)__popcll(m & below);
          const uint32_t cnt = (uint32_t)__popcll(m);
          if (EMIT && occ && idx < budget) {
            const uint64_t slot = base + idx;
            if (slot < a.capacity) {
              a.samples[slot] = make_float4(o[0] + tk[u] * d[0], o[1] + tk[u] * d[1], o[2] + tk[u] * d[2], tk[u]);
              if (a.ray_ids) a.ray_ids[slot] = r;
            }
          }
          if (found + cnt > budget) {
            // the first sample past the budget is where the next call starts
            const uint64_t past = __ballot(occ && idx == budget);
            kb = kb + 64u * u + (uint32_t)__builtin_ctzll(past);
            found = budget;
            over = true;
          } else {
            found += cnt;
          }
        }
        end |= __ballot(in[u]) != ~0ull;
      }
      if (over || end) break;
      kb += 64u * LATTICE_UNROLL;
    }
    if (lane == j) {
      emitted = found;
      if (EMIT && a.state) {
        st.k = kb;
        st.n = n_before + found;
        st.flags = (st.flags & ~MARCH_FRESH) | ((!over || st.n >= a.max_steps) ? MARCH_DONE : 0u);
        a.state[r_own] = st;
      }
    }
  }
  if (own && (!EMIT || a.slot_stride)) a.counts[r_own] = emitted;
}

// One wavefront per ray at a time: the ray's samples from its slots to its compacted range, 64 at a time
__global__ __launch_bounds__(256) void k_march_compact(const uint32_t* __restrict__ counts,
                                                       const uint32_t* __restrict__ offsets,
                                                       const float4* __restrict__ slots, uint32_t stride,
                                                       uint32_t num_rays, float4* __restrict__ samples,
                                                       uint32_t* __restrict__ ray_ids,
                                                       const uint32_t* __restrict__ gate) {
  if (gate && *gate == 0u) return;
  const int lane = threadIdx.x & 63;
  const uint32_t n_waves = gridDim.x * (blockDim.x >> 6);
  for (uint32_t r = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); r < num_rays; r += n_waves) {
    const uint32_t c = counts[r], o = offsets[r];
    const float4* src = slots + (uint64_t)r * stride;
    for (uint32_t k = lane; k < c; k += 64) {
      samples[(uint64_t)o + k] = src[k];
      ray_ids[(uint64_t)o + k] = r;
    }
  }
}

// sample budget of a marched step (launch_march_clamp): offsets [num_rays + 1], offsets[r + 1] the end of ray r
__global__ __launch_bounds__(256) void k_march_clamp(uint32_t* __restrict__ counts, const uint32_t* __restrict__ offsets,
                                                     uint32_t num_rays, uint32_t cap, uint32_t* __restrict__ n_eff) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= num_rays) return;
  const uint32_t end = offsets[r + 1];
  const bool fits = end <= cap;
  if (!fits) counts[r] = 0u;
  // the rays that fit are a prefix (offsets never decrease): its last ray writes the samples kept
  const bool next_fits = r + 1 < num_rays && offsets[r + 2] <= cap;
  if (fits && !next_fits) *n_eff = end;
  if (r == 0 && !fits) *n_eff = 0u;
}

__global__ __launch_bounds__(256) void k_march_init(MarchState* __restrict__ state, float4* __restrict__ acc,
                                                    uint32_t* __restrict__ n_used, uint32_t num_rays,
                                                    uint32_t* __restrict__ prime) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (prime && r == 0) *prime = 1u;
  if (r >= num_rays) return;
  state[r] = MarchState{0u, 0u, 0u, MARCH_FRESH};
  acc[r] = make_float4(0.0f, 0.0f, 0.0f, 1.0f);
  if (n_used) n_used[r] = 0u;
}

// front-to-back compositing of this round's samples of each ray (alpha as ffnerf_OG.cl:1505-1520);
// a ray whose transmittance drops below T_stop is retired.
// What bounds it: the latency of a lane's loads, so a lane loads RENDER_AHEAD samples before it composites them in
// order (past the ray's end the last one again).  450x800 frame, three rounds: one at a time 81 us, four 61, eight 50.
constexpr uint32_t RENDER_AHEAD = 8;
__global__ __launch_bounds__(256) void k_render_composite(const uint32_t* __restrict__ offsets,
                                                          const uint32_t* __restrict__ counts, uint32_t num_rays,
                                                          const float* __restrict__ sigma,
                                                          const float* __restrict__ rgb, float dt, float T_stop,
                                                          MarchState* __restrict__ state, float4* __restrict__ acc,
                                                          uint32_t* __restrict__ n_used,
                                                          const uint32_t* __restrict__ gate) {
  if (gate && *gate == 0u) return;
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= num_rays) return;
  const uint32_t cnt = counts[r];
  if (cnt == 0) return;
  const uint32_t off = offsets[r];
  float4 cv = acc[r];
  float T = cv.w;
  if (!(T >= T_stop)) return;  // retired in an earlier round
  float C0 = cv.x, C1 = cv.y, C2 = cv.z;
  uint32_t used = 0;
  bool stopped = false;
  for (uint32_t j = 0; j < cnt && !stopped; j += RENDER_AHEAD) {
    float sg[RENDER_AHEAD], c[RENDER_AHEAD][3];
#pragma unroll
    for (uint32_t u = 0; u < RENDER_AHEAD; ++u) {
      const size_t b = (size_t)off + (j + u < cnt ? j + u : cnt - 1);
      sg[u] = sigma[b];
#pragma unroll
      for (int i = 0; i < 3; ++i) c[u][i] = rgb[3 * b + i];
    }
#pragma unroll
    for (uint32_t u = 0; u < RENDER_AHEAD; ++u) {
      if (j + u >= cnt || stopped) continue;
      const float alpha = 1.0f - fast_exp(fminf(fmaxf(-sg[u] * dt, -5.0f), 18.0f));
      const float w = T * alpha;
      C0 = C0 + w * c[u][0];
      C1 = C1 + w * c[u][1];
      C2 = C2 + w * c[u][2];
      T = T * (1.0f - alpha);
      ++used;
      stopped = T < T_stop;
    }
  }
  if (stopped) state[r].flags |= MARCH_DONE;
  acc[r] = make_float4(C0, C1, C2, T);
  if (n_used) n_used[r] += used;
}

__global__ __launch_bounds__(256) void k_render_finish(const float4* __restrict__ acc, uint32_t num_rays,
                                                       float4* __restrict__ out_rgb) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= num_rays) return;
  out_rgb[r] = acc[r];  // black background: C + T * 0; w = T_final
}

// (cell, subcell) of the occupancy grid holding the point at time t of ray (o, d), as the proposals compute it;
// kOutsideGrid for a point outside the grid
constexpr uint64_t kOutsideGrid = ~(uint64_t)1;
__device__ __forceinline__ uint64_t occ_run_key(const DevCfg& c, const float (&o)[3], const float (&d)[3], float t) {
  float gpos[3];
  occ_grid_pos(c, o, d, t, gpos);
  const int G = c.G;
  const int ix = (int)floorf(gpos[0]), iy = (int)floorf(gpos[1]), iz = (int)floorf(gpos[2]);
  if (!((uint32_t)ix < (uint32_t)G && (uint32_t)iy < (uint32_t)G && (uint32_t)iz < (uint32_t)G)) return kOutsideGrid;
  uint32_t sub = 0;
#pragma unroll
  for (int i = 0; i < 3; ++i) sub += ((gpos[i] - floorf(gpos[i])) >= 0.5f ? 1u : 0u) << i;
  return ((uint64_t)(ix + G * (iy + G * iz)) << 3) | sub;
}

// The occupancy proposals of marched ray r: its samples, in order, fall into runs of one (cell, subcell) of the
// occupancy grid, and each run inside the grid proposes as a run of the resampled step does
// (ffnerf_OG.cl:1640-1821), from the compositing's transmittances (T_end past a termination, so those runs
// propose nothing).  One wavefront per ray: a lane whose sample starts a run walks to the run's end and proposes.
__device__ __forceinline__ void propose_marched_runs(const CompMarchArgs& a, uint32_t r, uint32_t off, uint32_t cnt,
                                                     float T_end, int lane) {
  const float4 ro = a.rays[2 * (size_t)r], rdv = a.rays[2 * (size_t)r + 1];
  const float o[3] = {ro.x, ro.y, ro.z}, d[3] = {rdv.x, rdv.y, rdv.z};
  const float Dhalf = half_box_diagonal(a.c);
  for (uint32_t s = (uint32_t)lane; s < cnt; s += 64) {
    const float t_s = a.samples[off + s].w;
    const uint64_t key = occ_run_key(a.c, o, d, t_s);
    const uint32_t prev = s > 0 ? s - 1 : 0;
    const float t_prev = a.samples[off + prev].w;
    if (key == kOutsideGrid || (s > 0 && occ_run_key(a.c, o, d, t_prev) == key)) continue;
    uint32_t j = s + 1;  // the run's end
    float t_last = t_s, t_j = 0.0f;
    for (; j < cnt; ++j) {
      t_j = a.samples[off + j].w;
      if (occ_run_key(a.c, o, d, t_j) != key) break;
      t_last = t_j;
    }
    const bool has_next = j < cnt;
    occ_propose_run(a.c, o, d, t_s, a.Tr[off + s], t_prev, a.Tr[off + prev], t_last, a.Tr[off + j - 1], has_next,
                    has_next ? t_j : 0.0f, has_next ? a.Tr[off + j] : 0.0f, T_end, a.occ_in[key >> 3], a.seed, r, s,
                    Dhalf, a.occ_st);
  }
}

// dL/dT after each lane's sample of a group of 64: the sample's map x -> b + a x (a = 1 - alpha, b = g . (alpha c)),
// composed over the later lanes and applied to gT, dL/dT after the group; gT becomes the one before it.  Inside a
// 16-lane row the composition is a suffix scan by DPP row shifts; the four rows follow each other by readlane.
__device__ __forceinline__ float grad_T_after(float a, float b, int lane, float& gT) {
  auto step = [&](float ar, float br) {  // self, then the lane to the right
    b = b + a * br;
    a = a * ar;
  };
  step(dpp_or<0x101>(1.0f, a), dpp_or<0x101>(0.0f, b));  // row_shl:1, 2, 4, 8: the identity past the row's end
  step(dpp_or<0x102>(1.0f, a), dpp_or<0x102>(0.0f, b));
  step(dpp_or<0x104>(1.0f, a), dpp_or<0x104>(0.0f, b));
  step(dpp_or<0x108>(1.0f, a), dpp_or<0x108>(0.0f, b));
  const float ea = dpp_or<0x101>(1.0f, a), eb = dpp_or<0x101>(0.0f, b);  // the lanes after this one in its row
  auto rl = [](float x, int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i)); };
  const float g3 = gT;  // dL/dT after row 3, 2, 1, 0
  const float g2 = rl(b, 48) + rl(a, 48) * g3;
  const float g1 = rl(b, 32) + rl(a, 32) * g2;
  const float g0 = rl(b, 16) + rl(a, 16) * g1;
  gT = rl(b, 0) + rl(a, 0) * g0;
  const int row = lane >> 4;
  return eb + ea * (row == 3 ? g3 : (row == 2 ? g2 : (row == 1 ? g1 : g0)));
}

// Compositing of marched training rays and its backward, one wavefront per ray: the specification's recurrences
// over the ray's samples (ora_train_step_marched; ffnerf_OG.cl:1593-1634 restated: T_(i+1) = T_i (1 - alpha_i);
// gT_i = g . (alpha_i c_i) + (1 - alpha_i) gT_(i+1), gT_end = g . bg) as scans over 64 samples at a time.
// What bounds it: latency (a ray's groups follow each other, each a few dependent loads and two scans).  A lane
// per ray, each walking its own range of the sample arrays, waited for its loads: 40,001 rays with 880,000 samples
// 217 us, now 28; 2^18 rays 390, now 127.  The recurrences kept sequential over the lanes' values by readlane
// took 97 and 395 us.
// (rays_per_wave: consecutive rays of a wavefront)
__global__ __launch_bounds__(256) void k_composite_marched(CompMarchArgs a, uint32_t rays_per_wave) {
  const int lane = threadIdx.x & 63;
  const uint64_t r0 = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * rays_per_wave;
  auto rl = [](float x, int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), i)); };
  for (uint64_t rr = r0; rr < r0 + rays_per_wave && rr < a.num_rays; ++rr) {
    const uint32_t r = (uint32_t)rr;
    const uint32_t cnt = a.counts[r], off = a.offsets[r];
    float T = 1.0f, C0 = 0.0f, C1 = 0.0f, C2 = 0.0f;
    uint32_t used = 0;  // samples up to and including the one that leaves T < T_stop
    bool stopped = false;
    for (uint32_t b0 = 0; b0 < cnt && !stopped; b0 += 64) {
      const int n = (int)(cnt - b0 < 64 ? cnt - b0 : 64);
      const size_t b = (size_t)off + b0 + lane;
      float alpha = 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
      if (lane < n) {
        alpha = 1.0f - fast_exp(fminf(fmaxf(-a.sigma[b] * a.dt, -5.0f), 18.0f));
        c0 = a.rgb[3 * b];
        c1 = a.rgb[3 * b + 1];
        c2 = a.rgb[3 * b + 2];
      }
      const float oma = 1.0f - alpha;
      Seg tot;
      const Seg pre = comp_seg_prefix(Seg{oma, alpha * c0, alpha * c1, alpha * c2}, lane, 64, &tot);
      const float Tr = T * pre.a;  // before this lane's sample
      // the group's samples up to the first that leaves T < T_stop
      const uint64_t stop = __ballot(lane < n && Tr * oma < a.T_stop);
      const int m = stop != 0ull ? (int)__builtin_ctzll(stop) + 1 : n;
      stopped = stop != 0ull;
      if (stopped) {  // the colours up to sample m - 1
        const float w = pre.a * alpha;
        tot = Seg{rl(pre.a * oma, m - 1), rl(pre.v0 + w * c0, m - 1), rl(pre.v1 + w * c1, m - 1),
                  rl(pre.v2 + w * c2, m - 1)};
      }
      C0 = C0 + T * tot.v0;
      C1 = C1 + T * tot.v1;
      C2 = C2 + T * tot.v2;
      T = T * tot.a;
      if (lane < m) a.Tr[b] = Tr;
      used += (uint32_t)m;
    }
    float bg[3] = {0.0f, 0.0f, 0.0f};
    if (a.background == FFN_BG_WHITE) {
      bg[0] = bg[1] = bg[2] = 1.0f;
    } else if (a.background == FFN_BG_RANDOM) {
      uint32_t rb = hash_u32(a.seed ^ r * 747796405u ^ 0xA511E9B3u);
      bg[0] = rand01(rb);
      bg[1] = rand01(rb);
      bg[2] = rand01(rb);
    }
    const float4 tg = a.targets[r];
    const float Cf0 = C0 + T * bg[0], Cf1 = C1 + T * bg[1], Cf2 = C2 + T * bg[2];
    const float gr0 = charbonnier_prime(Cf0 - tg.x), gr1 = charbonnier_prime(Cf1 - tg.y),
                gr2 = charbonnier_prime(Cf2 - tg.z);
    if (lane == 0) {
      a.out_rgb[r] = make_float4(fminf(fmaxf(Cf0, 0.0f), 1.0f), fminf(fmaxf(Cf1, 0.0f), 1.0f),
                                 fminf(fmaxf(Cf2, 0.0f), 1.0f), 4.0f);
      if (a.n_used) a.n_used[r] = used;
      if (a.T_final) a.T_final[r] = T;
      if (a.color) a.color[r] = make_float4(Cf0, Cf1, Cf2, 0.0f);
    }
    // past the termination: no contribution, no gradient
    for (uint32_t s = used + (uint32_t)lane; s < cnt; s += 64) {
      const size_t b = (size_t)off + s;
      a.Tr[b] = T;
      a.dLds[b] = 0.0f;
      a.dLdc[3 * b] = a.dLdc[3 * b + 1] = a.dLdc[3 * b + 2] = 0.0f;
    }
    float gT = gr0 * bg[0] + gr1 * bg[1] + gr2 * bg[2];
    for (uint32_t e = used; e > 0;) {  // groups of 64 from the back, aligned as in the forward
      const uint32_t b0 = (e - 1) & ~63u;
      const int n = (int)(e - b0);
      const size_t b = (size_t)off + b0 + lane;
      float alpha = 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f, Ti = 0.0f;
      if (lane < n) {
        alpha = 1.0f - fast_exp(fminf(fmaxf(-a.sigma[b] * a.dt, -5.0f), 18.0f));
        c0 = a.rgb[3 * b];
        c1 = a.rgb[3 * b + 1];
        c2 = a.rgb[3 * b + 2];
        Ti = a.Tr[b];  // written by this lane above
      }
      const float oma = 1.0f - alpha;
      const float gc = gr0 * (alpha * c0) + gr1 * (alpha * c1) + gr2 * (alpha * c2);
      const float g_next = grad_T_after(oma, gc, lane, gT);  // dL/dT after this lane's sample
      if (lane < n) {
        const float gA = gr0 * (Ti * c0) + gr1 * (Ti * c1) + gr2 * (Ti * c2);
        const float gAlpha = gA - g_next * Ti;
        a.dLds[b] = gAlpha * (a.dt * oma) + a.regu;
        const float ws = Ti * alpha;
        a.dLdc[3 * b] = ws * gr0;
        a.dLdc[3 * b + 1] = ws * gr1;
        a.dLdc[3 * b + 2] = ws * gr2;
      }
      e = b0;
    }
    if (a.occ_st) {
      __threadfence_block();  // the lanes read each other's Tr
      propose_marched_runs(a, r, off, cnt, T, lane);
    }
  }
}

hipError_t launch_composite_marched(const CompMarchArgs& a, hipStream_t st) {
  if (a.num_rays == 0) return hipSuccess;
  // one ray per wavefront while the rays are few, so that rays with samples do not queue behind each other
  const uint32_t rpw = a.num_rays < (1u << 17) ? 1 : 4;
  const uint64_t waves = ((uint64_t)a.num_rays + rpw - 1) / rpw;
  hipLaunchKernelGGL(k_composite_marched, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a, rpw);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------

hipError_t launch_occ_bitfield(const uint32_t* occ, int G, uint32_t q_min, uint32_t* bits, hipStream_t st) {
  const int64_t R = 2 * (int64_t)G;
  const int64_t n_words = (R * R * R + 31) / 32;
  hipLaunchKernelGGL(k_occ_bitfield, dim3((unsigned)((n_words + 255) / 256)), dim3(256), 0, st, occ, G, q_min,
                     bits, n_words);
  return hipGetLastError();
}

hipError_t launch_occ_blocks(const uint32_t* bits, int R, uint32_t* blocks, uint32_t* use, hipStream_t st) {
  const int64_t NB = (R + 7) / 8;
  const int64_t n_blocks = NB * NB * NB;
  hipLaunchKernelGGL(k_occ_blocks, dim3((unsigned)((n_blocks + 255) / 256)), dim3(256), 0, st, bits, R, blocks,
                     n_blocks);
  hipLaunchKernelGGL(k_blocks_use, dim3(1), dim3(256), 0, st, blocks, n_blocks, use);
  return hipGetLastError();
}

// The rule between the two walks.  The lattice walk costs rays x lattice points, the cell walk rays x cells, but
// with few rays its serial walk per lane costs the same however few they are.  ffn_march (count, scan, emit) in
// us, lattice / cells, K points along the box diagonal, the ball and the shell field:
//   rays 1000, R 256:    K 1024 63 / 1709, 64 / 1898;      K 4096 166 / 2445, 164 / 3212
//   rays 40001, R 256:   K 1024 114 / 2118, 117 / 2227;    K 4096 297 / 3069, 297 / 3850
//   rays 2^18, R 256:    K 1024 480 / 1924, 481 / 2160;    K 4096 1458 / 2795, 1467 / 3609
//   rays 2^20, R 256:    K 1024 1444 / 2716, 1460 / 3468;  K 4096 4578 / 4245, 4602 / 6175
//   rays 2^20, R 128:    K 2048 2167 / 2320, 2172 / 3182;  K 4096 3883 / 3459, 3877 / 4988
// so the line lies at 16 R points for 2^20 rays and moves up in proportion for fewer.  FFN_MARCH_LATTICE=0 keeps
// the cell walk.
bool march_takes_lattice(const MarchArgs& a) {
  const char* env = getenv("FFN_MARCH_LATTICE");
  if (env && env[0] == '0') return false;
  double diag2 = 0.0;
  for (int i = 0; i < 3; ++i) diag2 += ((double)a.bmax[i] - a.bmin[i]) * ((double)a.bmax[i] - a.bmin[i]);
  const double points = sqrt(diag2) / (double)a.dt;
  const double fewer = a.num_rays < (1u << 20) ? (double)(1u << 20) / a.num_rays : 1.0;
  return points <= 16.0 * a.res * fewer;
}

hipError_t launch_march(const MarchArgs& a, bool emit, hipStream_t st) {
  if (a.num_rays == 0) return hipSuccess;
  if (a.lattice) {
    // rays a wavefront sets up at once: as many as leave 8192 wavefronts (8 per SIMD), at least 4
    uint32_t rpw = 64;
    while (rpw > 4 && (a.num_rays + rpw - 1) / rpw < 8192u) rpw >>= 1;
    const uint64_t waves = ((uint64_t)a.num_rays + rpw - 1) / rpw;
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    if (emit)
      hipLaunchKernelGGL(k_march_lattice<true>, grid, block, 0, st, a, rpw);
    else
      hipLaunchKernelGGL(k_march_lattice<false>, grid, block, 0, st, a, rpw);
    return hipGetLastError();
  }
  const uint64_t waves = (a.num_rays + MARCH_RPW - 1) / MARCH_RPW;
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  if (emit)
    hipLaunchKernelGGL(k_march<true>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(k_march<false>, grid, block, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_march_compact(const uint32_t* counts, const uint32_t* offsets, const float4* slots,
                                uint32_t stride, uint32_t num_rays, float4* samples, uint32_t* ray_ids,
                                hipStream_t st, const uint32_t* gate) {
  if (num_rays == 0) return hipSuccess;
  const uint32_t blocks = (num_rays + 3) / 4 < 4096 ? (num_rays + 3) / 4 : 4096;
  hipLaunchKernelGGL(k_march_compact, dim3(blocks), dim3(256), 0, st, counts, offsets, slots, stride, num_rays,
                     samples, ray_ids, gate);
  return hipGetLastError();
}

hipError_t launch_march_clamp(uint32_t* counts, const uint32_t* offsets, uint32_t num_rays, uint32_t cap,
                              uint32_t* n_eff, hipStream_t st) {
  if (num_rays == 0) return hipSuccess;
  hipLaunchKernelGGL(k_march_clamp, dim3((num_rays + 255) / 256), dim3(256), 0, st, counts, offsets, num_rays, cap,
                     n_eff);
  return hipGetLastError();
}

hipError_t launch_march_init(MarchState* state, float4* acc, uint32_t* n_used, uint32_t num_rays, hipStream_t st,
                             uint32_t* prime) {
  if (num_rays == 0) return hipSuccess;
  hipLaunchKernelGGL(k_march_init, dim3((num_rays + 255) / 256), dim3(256), 0, st, state, acc, n_used, num_rays,
                     prime);
  return hipGetLastError();
}

hipError_t launch_render_composite(const uint32_t* offsets, const uint32_t* counts, uint32_t num_rays,
                                   const float* sigma, const float* rgb, float dt, float T_stop, MarchState* state,
                                   float4* acc, uint32_t* n_used, hipStream_t st, const uint32_t* gate) {
  if (num_rays == 0) return hipSuccess;
  hipLaunchKernelGGL(k_render_composite, dim3((num_rays + 255) / 256), dim3(256), 0, st, offsets, counts, num_rays,
                     sigma, rgb, dt, T_stop, state, acc, n_used, gate);
  return hipGetLastError();
}

hipError_t launch_render_finish(const float4* acc, uint32_t num_rays, float4* out_rgb, hipStream_t st) {
  if (num_rays == 0) return hipSuccess;
  hipLaunchKernelGGL(k_render_finish, dim3((num_rays + 255) / 256), dim3(256), 0, st, acc, num_rays, out_rgb);
  return hipGetLastError();
}

}  // namespace ffn
