// Grid parameters of a scene from its work-groups' bounding boxes, in the
// reference's host FP32 sequence (sph_simulation.cpp:201-252: no contraction,
// correctly rounded division), and the layout of the batch's keys. Used by the
// grid stage and by the kernel that runs it with the hash and the sort.
#pragma once

#include "reduce.h"
#include "state.h"

namespace clsph {

// LSD passes and digit width of a substep whose batch holds `base` half-cell
// keys: the sort orders by cell id (key >> 3) in sort_passes passes; a state
// sized for three runs two while the cell ids fit them.
struct KeyLayout {
  uint32_t key_bits, passes, digit_bits;
};
__device__ inline KeyLayout key_layout(uint64_t base, uint32_t sort_passes) {
  KeyLayout k;
  k.key_bits = bitlen((uint32_t)base);
  uint32_t cb = k.key_bits > 3u ? k.key_bits - 3u : 1u;
  k.passes = sort_passes ? sort_passes : 1u;
  if (k.passes > 2u && cb <= 2u * (uint32_t)kMaxDigitBits) k.passes = 2u;
  uint32_t db = (cb + k.passes - 1u) / k.passes;
  k.digit_bits = db < 1u ? 1u : (db > (uint32_t)kMaxDigitBits ? (uint32_t)kMaxDigitBits : db);
  return k;
}

// Stores the batch's layout for `base` keys in all (one thread); `err` holds
// the error bits raised while laying them out.
__device__ inline void batch_layout(BatchParams* __restrict__ bp, uint64_t base, uint32_t err,
                                    uint32_t table_cap, uint32_t sort_passes) {
  if (base > table_cap) err |= kErrTableCap;
  const KeyLayout k = key_layout(base, sort_passes);
  bp->key_total = (uint32_t)base;
  bp->key_bits = k.key_bits;
  bp->lsd_passes = k.passes;
  bp->digit_bits = k.digit_bits;
  if (err) atomicOr(&bp->err, err);
}

// The scene's box (min xyz, max xyz) from its partial boxes, in every lane of
// the first wave of a work-group of WAVES (a power of two) waves, which all
// call it; true there.
template <int WAVES>
__device__ inline bool scene_box(const DevParams* __restrict__ dp,
                                 const float* __restrict__ partial, uint32_t stride,
                                 float (&red)[6][WAVES], float v[6]) {
  const float inf = __builtin_huge_valf();
  for (int k = 0; k < 6; ++k) v[k] = k < 3 ? inf : -inf;
  // eight partial boxes per thread in flight at a time
  const uint32_t b0 = dp->block_begin, b1 = dp->block_end;
  for (uint32_t b = b0 + threadIdx.x; b < b1; b += 8u * blockDim.x) {
    float q[8][6];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t bu = b + (uint32_t)u * blockDim.x;
#pragma unroll
      for (int k = 0; k < 6; ++k) q[u][k] = bu < b1 ? partial[k * stride + bu] : (k < 3 ? inf : -inf);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      for (int k = 0; k < 3; ++k) v[k] = fminf(v[k], q[u][k]);
      for (int k = 3; k < 6; ++k) v[k] = fmaxf(v[k], q[u][k]);
    }
  }
  for (int k = 0; k < 3; ++k) v[k] = wave_min(v[k]);
  for (int k = 3; k < 6; ++k) v[k] = wave_max(v[k]);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0)
    for (int k = 0; k < 6; ++k) red[k][w] = v[k];
  __syncthreads();
  if (threadIdx.x >= 64u) return false;  // the first wave joins the waves' boxes
  // the first WAVES lanes take one wave's box each; a butterfly over them
  // leaves the scene's box in every lane
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    float r = red[k][l & (WAVES - 1)];
#pragma unroll
    for (int o = WAVES / 2; o >= 1; o >>= 1) {
      const float y = __shfl_xor(r, o, 64);
      r = (k < 3) ? fminf(r, y) : fmaxf(r, y);
    }
    v[k] = r;
  }
  return true;
}

// The grid of one scene from its bounding box v = (min xyz, max xyz), its
// smoothing length h and particle count n, with the error bits it raises.
struct GridOf {
  float mn[3], mx[3];
  uint32_t gs[3], cells, err;
};
__device__ inline GridOf grid_of(const float v[6], float h, uint32_t n) {
#pragma clang fp contract(off)
  GridOf g = {};
  if (n == 0) return g;
  // Initial values are numeric_limits<cl_int>::max()/min() as float; a
  // position replaces them only when strictly smaller / larger.
  const float init_min = 2147483648.0f, init_max = -2147483648.0f;
  float L = h * 2;
  for (int a = 0; a < 3; ++a) {
    g.mn[a] = (v[a] < init_min) ? v[a] : init_min;
    g.mx[a] = (v[3 + a] > init_max) ? v[3 + a] : init_max;
    g.mn[a] -= L * 2;
    g.mx[a] += L * 2;
    g.gs[a] = (uint32_t)((g.mx[a] - g.mn[a]) / L);
    if (g.gs[a] >= 1024u) g.err |= kErrGridDim;
  }
  g.cells = morton3(g.gs[0], g.gs[1], g.gs[2]);
  if (g.cells >= (1u << 29)) g.err |= kErrFineKey;
  return g;
}

__device__ inline void store_grid(DevParams* __restrict__ dp, const GridOf& g, uint32_t n) {
  dp->capped = 0;
  dp->p.grid_cell_count = g.cells;
  if (n == 0) return;
  for (int a = 0; a < 3; ++a) {
    dp->p.min_point.s[a] = g.mn[a];
    dp->p.max_point.s[a] = g.mx[a];
  }
  dp->p.min_point.s[3] = 0.f;
  dp->p.max_point.s[3] = 0.f;
  dp->p.grid_size_x = (int32_t)g.gs[0];
  dp->p.grid_size_y = (int32_t)g.gs[1];
  dp->p.grid_size_z = (int32_t)g.gs[2];
  if (g.err) atomicOr(&dp->err, g.err);
}

// Half-cell keys of a state of one scene with `cells` cells and error bits
// err: its own, and all that batch_keys would lay out, clamped alike.
__device__ inline uint32_t single_keys(uint32_t cells, uint32_t err) {
  return (err & kErrFineKey) ? 0u : cells;
}
__device__ inline uint64_t single_total(uint32_t keyed_cells) {
  const uint64_t base = 8ull * ((uint64_t)keyed_cells + 1u);
  return base < 0xFFFFFFF0ull ? base : 0xFFFFFFF0ull;
}

// Stores the layout of such a state (one thread).
__device__ inline void single_layout(DevParams* __restrict__ dp, BatchParams* __restrict__ bp,
                                     uint32_t cells, uint32_t err, uint32_t table_cap,
                                     uint32_t sort_passes) {
  const uint32_t Gk = single_keys(cells, err);
  dp->key_base = 0;
  dp->key_end = 8u * Gk;
  const uint64_t base = single_total(Gk);
  batch_layout(bp, base, 8ull * ((uint64_t)Gk + 1u) > base ? kErrFineKey : 0u, table_cap,
               sort_passes);
}

}  // namespace clsph
