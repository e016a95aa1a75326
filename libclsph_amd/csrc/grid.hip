// Grid stages: bounding box, grid parameters and cell-id hashing, for every
// scene of a batch at once (the sort, the cell table and the reference's
// stable order are in sort.hip).
//
// The bounding box / grid arithmetic must reproduce the reference's host FP32
// sequence bit for bit (sph_simulation.cpp:201-252), and the cell id the
// kernel's (grid.cl:43-67): no contraction, correctly rounded division.
//
// Particles are hashed to the half-size cell (side h) they fall in. With
// u = (x - min) / (2h) per axis, the cell coordinate of the reference is
// (uint)u and the half-cell coordinate is (uint)(2u) = 2 (uint)u + [frac(u) >=
// 1/2], exact because 2u is exact. The Morton key of the half-cell is then
// (reference key << 3) | octant, so sorting by it keeps the reference's cells
// contiguous and in order, each grouped by octant. A scene's keys are offset
// by its key_base.
#include "grid_params.h"
#include "reduce.h"
#include "state.h"

#pragma clang fp contract(off)

namespace clsph {

__global__ __launch_bounds__(kMaxBlock) void k_aabb(const float4* __restrict__ pos,
                                                    const BlockDesc* __restrict__ blocks,
                                                    const DevParams* __restrict__ dps,
                                                    float* __restrict__ partial, uint32_t stride) {
  uint32_t scene;
  uint32_t i = particle_of(blocks, dps, scene);
  bool valid = i != 0xFFFFFFFFu;
  float4 p = valid ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  block_aabb_partial(p, valid, partial, stride);
}

// Lays the scenes' half-cell key ranges end to end (each scene gets
// 8 (G + 1) keys, its base clamped at 0xFFFFFFF0 with kErrFineKey raised
// once the running total passes it) and sizes the sort digits for the total.
// One wave, 64 scenes at a time: each scene's base is the exclusive sum of
// the keys before it, a wave scan.
__device__ void batch_keys(DevParams* __restrict__ dps, BatchParams* __restrict__ bp) {
  constexpr uint64_t kTop = 0xFFFFFFF0ull;
  const uint32_t lane = threadIdx.x & 63u, ns = bp->n_scenes;
  uint64_t carry = 0;
  for (uint32_t s0 = 0; s0 < ns; s0 += 64u) {
    const uint32_t s = s0 + lane;
    uint64_t G = 0, keys = 0;
    if (s < ns) {
      G = (dps[s].err & kErrFineKey) ? 0u : dps[s].p.grid_cell_count;
      keys = 8ull * (G + 1);
    }
    uint64_t incl = keys;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
      const uint32_t lo = __shfl_up((uint32_t)incl, o, 64), hi = __shfl_up((uint32_t)(incl >> 32), o, 64);
      if (lane >= o) incl += ((uint64_t)hi << 32) | lo;
    }
    if (s < ns) {
      const uint64_t ex = carry + incl - keys;
      const uint64_t base = ex < kTop ? ex : kTop;
      dps[s].key_base = (uint32_t)base;
      dps[s].key_end = (uint32_t)(base + 8ull * G);
    }
    const uint32_t tlo = __shfl((uint32_t)incl, 63, 64), thi = __shfl((uint32_t)(incl >> 32), 63, 64);
    carry += ((uint64_t)thi << 32) | tlo;
  }
  if (lane == 0)
    batch_layout(bp, carry < kTop ? carry : kTop, carry > kTop ? kErrFineKey : 0u, bp->table_cap,
                 bp->sort_passes);
}

// One work-group per scene: reduces the scene's partial boxes, then restates
// sph_simulation.cpp:201-252 in FP32. The last work-group to finish lays out
// the batch's keys (batch_keys); a single scene does so from the values in
// its registers. The parameters thread 0 needs are loaded before the
// reduction, so that their latency overlaps it.
__global__ __launch_bounds__(1024) void k_grid_params(DevParams* __restrict__ dps,
                                                      const float* __restrict__ partial,
                                                      uint32_t stride,
                                                      BatchParams* __restrict__ bp) {
  __shared__ float red[6][16];
  DevParams* dp = dps + blockIdx.x;
  const float h = dp->p.h;
  const uint32_t np = dp->n, err0 = dp->err;
  const uint32_t table_cap = bp->table_cap, sort_passes = bp->sort_passes;
  float v[6];
  if (!scene_box<16>(dp, partial, stride, red, v)) return;
  if (threadIdx.x != 0 && gridDim.x == 1u) return;
  if (threadIdx.x == 0) {
    const GridOf g = grid_of(v, h, np);
    store_grid(dp, g, np);
    if (gridDim.x == 1u) {
      single_layout(dp, bp, g.cells, err0 | g.err, table_cap, sort_passes);
      return;
    }
  }
  // the scenes' grids are in place once every work-group has passed here
  uint32_t last = 0;
  if (threadIdx.x == 0) {
    __threadfence();
    last = atomicAdd(&bp->ticket, 1u) == gridDim.x - 1u ? 1u : 0u;
  }
  if (!__shfl(last, 0, 64)) return;
  __threadfence();
  if (threadIdx.x == 0) bp->ticket = 0;
  batch_keys(dps, bp);
}

// Half-cell keys of every particle (hash_key).
__global__ __launch_bounds__(kMaxBlock) void k_hash(const float4* __restrict__ pos,
                                                    const BlockDesc* __restrict__ blocks,
                                                    const DevParams* __restrict__ dps,
                                                    uint32_t* __restrict__ key) {
  uint32_t scene;
  uint32_t i = particle_of(blocks, dps, scene);
  if (i == 0xFFFFFFFFu) return;
  key[i] = hash_key(pos[i], dps + scene);
}

void launch_aabb(clsph_state* s) {
  if (s->n == 0) return;
  hipLaunchKernelGGL(k_aabb, dim3(s->nblocks_of(kStageAdvect)), dim3(s->bs_of(kStageAdvect)), 0,
                     s->ctx->stream, s->pos, s->table_of(kStageAdvect), s->dps, s->aabb_partial,
                     s->aabb_stride);
}

void launch_grid_params(clsph_state* s) {
  hipLaunchKernelGGL(k_grid_params, dim3(s->n_scenes), dim3(1024), 0, s->ctx->stream, s->dps,
                     s->aabb_partial, s->aabb_stride, s->bp);
}

void launch_hash(clsph_state* s) {
  if (s->n == 0) return;
  hipLaunchKernelGGL(k_hash, dim3(s->nblocks_of(kStageHash)), dim3(s->bs_of(kStageHash)), 0,
                     s->ctx->stream, s->pos, s->table_of(kStageHash), s->dps, s->key_a);
}

}  // namespace clsph

// Identity tracking across a substep: the particle at sorted position k came
// from canonical index perm[k] and is written back to canonical slot[k].
__global__ __launch_bounds__(256) void k_track_ids(const uint32_t* __restrict__ perm,
                                                   const uint32_t* __restrict__ slot,
                                                   const uint32_t* __restrict__ ids,
                                                   uint32_t* __restrict__ out, uint32_t n) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  uint32_t s = slot[k], p = perm[k];
  if (s < n && p < n) out[s] = ids[p];
}

__global__ __launch_bounds__(256) void k_copy_u32(const uint32_t* __restrict__ in,
                                                  uint32_t* __restrict__ out, uint32_t n) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) out[k] = in[k];
}

__global__ __launch_bounds__(256) void k_iota(uint32_t* __restrict__ out, uint32_t n) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) out[k] = k;
}

namespace clsph {
void launch_reset_ids(clsph_state* s) {
  if (!s->n_cap) return;
  hipLaunchKernelGGL(k_iota, dim3((s->n_cap + 255) / 256), dim3(256), 0, s->ctx->stream, s->ids,
                     s->n_cap);
}

void launch_track_ids(clsph_state* s) {
  if (!s->n) return;
  dim3 g((s->n + 255) / 256);
  hipLaunchKernelGGL(k_track_ids, g, dim3(256), 0, s->ctx->stream, s->val_b, s->slot, s->ids,
                     s->ids_tmp, s->n);
  hipLaunchKernelGGL(k_copy_u32, g, dim3(256), 0, s->ctx->stream, s->ids_tmp, s->ids, s->n);
}
}  // namespace clsph

namespace clsph {

// Particle records in the reference's layout (80 B: position, velocity,
// intermediate velocity, acceleration as float4 with w = 0, then density,
// pressure, grid_index and padding) in canonical order, as the host download
// assembles them: positions and velocities are canonical already; density,
// pressure, cell id and, while the fields are canonical, the acceleration
// are in sorted order and go to canonical slot[k]. Single-scene states.
__global__ __launch_bounds__(256) void k_pack_aos(
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const float4* __restrict__ vh, const float4* __restrict__ acc_s,
    const float* __restrict__ rho_s, const float* __restrict__ prs_s,
    const uint32_t* __restrict__ key, const uint32_t* __restrict__ slot,
    const DevParams* __restrict__ dps, uint32_t n, int reorder, int want_acc,
    uint4* __restrict__ out) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  auto bits = [](float a, float b, float c) {
    return make_uint4(__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), 0u);
  };
  const float4 p = pos[k], v = vel[k], h = vh[k];
  uint4* r = out + 5 * (size_t)k;
  r[0] = bits(p.x, p.y, p.z);
  r[1] = bits(v.x, v.y, v.z);
  r[2] = bits(h.x, h.y, h.z);
  const uint32_t o = reorder ? slot[k] : k;
  if (o >= n) return;
  uint4* q = out + 5 * (size_t)o;
  uint4 a = make_uint4(0u, 0u, 0u, 0u);
  if (want_acc && !reorder) {
    const float4 ak = acc_s[k];
    a = bits(ak.x, ak.y, ak.z);
  }
  q[3] = a;
  const uint32_t gi = reorder ? (key[k] - dps[0].key_base) >> 3 : key[k];
  q[4] = make_uint4(__float_as_uint(rho_s[k]), __float_as_uint(prs_s[k]), gi, 0u);
}

void launch_pack_aos(clsph_state* s, clsph_particle* out) {
  if (s->n == 0) return;
  hipLaunchKernelGGL(k_pack_aos, dim3((s->n + 255) / 256), dim3(256), 0, s->ctx->stream, s->pos,
                     s->vel, s->vh, s->acc_s, s->rho_s, s->prs_s, s->key_b, s->slot, s->dps, s->n,
                     s->fields_canonical ? 0 : 1, s->acc_zero ? 0 : 1,
                     reinterpret_cast<uint4*>(out));
}

// ---- particle records to and from host memory --------------------------------
//
// Synchronous transfers go through two page-locked buffers of kTransferRecords
// records each: these kernels read and write the buffers themselves, a
// work-group's records as one contiguous range (bound by PCIe, about 50 GB/s),
// and turn them into the state's arrays, or the arrays into records, in LDS.
// One 16-byte field of a record per access would be one bus transaction each.
// A copy per array through pageable memory, with the records put together on
// the host, took 184 us for 4,096 particles down and 78 us up, 519 us for
// 50,021 down sorted; a substep between an upload and a download now takes
// 143 us with both (383 before).
constexpr int kRecBlock = 256;

// Sorted position of each canonical position: inv[slot[k] - b0] = k.
__global__ __launch_bounds__(kRecBlock) void k_invert_slots(const uint32_t* __restrict__ slot,
                                                            uint32_t b0, uint32_t n,
                                                            uint32_t* __restrict__ inv) {
  const uint32_t k = blockIdx.x * kRecBlock + threadIdx.x;
  if (k >= n) return;
  const uint32_t o = slot[k] - b0;
  if (o < n) inv[o] = k;
}

// Records [r0, r0 + count) of a scene of n particles at b0, and the transfer's
// status: the error bits of every scene and of the batch, and whether the
// canonical slots are not a permutation. With `inv`, density, pressure and
// cell id (and in a sorted download everything) are in half-cell order and
// record o takes them from position inv[o].
__global__ __launch_bounds__(kRecBlock) void k_pack_records(
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const float4* __restrict__ vh, const float4* __restrict__ acc,
    const float* __restrict__ rho, const float* __restrict__ prs,
    const uint32_t* __restrict__ key, const uint32_t* __restrict__ slot,
    const uint32_t* __restrict__ inv, const DevParams* __restrict__ dps,
    const BatchParams* __restrict__ bp, uint32_t scene, uint32_t b0, uint32_t n, uint32_t r0,
    uint32_t count, int sorted, uint4* __restrict__ out, TransferStatus* __restrict__ status) {
  __shared__ uint4 rec[5 * kRecBlock];
  __shared__ uint32_t err;
  const uint32_t t = threadIdx.x, l = blockIdx.x * kRecBlock + t;
  if (blockIdx.x == 0) {
    if (t == 0) err = bp->err;
    __syncthreads();
    for (uint32_t s = t; s < bp->n_scenes; s += kRecBlock)
      if (dps[s].err) atomicOr(&err, dps[s].err);
    __syncthreads();
    if (t == 0) status->err = err;
  }
  if (l < count) {
    auto bits = [](float4 a) {
      return make_uint4(__float_as_uint(a.x), __float_as_uint(a.y), __float_as_uint(a.z), 0u);
    };
    const uint32_t o = r0 + l;
    uint32_t k = inv ? inv[o] : o;
    if (k >= n || (inv && slot[k] - b0 != o)) {
      status->bad_slots = 1u;
      k = o;
    }
    const uint32_t p = sorted ? k : o;
    rec[5u * t] = bits(pos[p]);
    rec[5u * t + 1u] = bits(vel[p]);
    rec[5u * t + 2u] = bits(vh[p]);
    rec[5u * t + 3u] = acc ? bits(acc[k]) : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t id = inv ? (key[k] - dps[scene].key_base) >> 3 : key[k];
    rec[5u * t + 4u] = make_uint4(__float_as_uint(rho[k]), __float_as_uint(prs[k]), id, 0u);
  }
  __syncthreads();
  const uint32_t first = blockIdx.x * kRecBlock;
  const uint32_t words = 5u * (count - first < kRecBlock ? count - first : kRecBlock);
  for (uint32_t q = t; q < words; q += kRecBlock) out[5u * first + q] = rec[q];
}

// `count` records into a state's arrays (already at their first particle).
__global__ __launch_bounds__(kRecBlock) void k_unpack_records(
    const uint4* __restrict__ in, uint32_t count, float4* __restrict__ pos,
    float4* __restrict__ vel, float4* __restrict__ vh, float4* __restrict__ acc,
    float* __restrict__ rho, float* __restrict__ prs, uint32_t* __restrict__ key) {
  __shared__ uint4 rec[5 * kRecBlock];
  const uint32_t t = threadIdx.x, first = blockIdx.x * kRecBlock, l = first + t;
  const uint32_t words = 5u * (count - first < kRecBlock ? count - first : kRecBlock);
  for (uint32_t q = t; q < words; q += kRecBlock) rec[q] = in[5u * first + q];
  __syncthreads();
  if (l >= count) return;
  auto vec = [&](uint32_t f) {
    const uint4 w = rec[5u * t + f];
    return make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), 0.f);
  };
  pos[l] = vec(0u);
  vel[l] = vec(1u);
  vh[l] = vec(2u);
  acc[l] = vec(3u);
  const uint4 w = rec[5u * t + 4u];
  rho[l] = __uint_as_float(w.x);
  prs[l] = __uint_as_float(w.y);
  key[l] = w.z;
}

void launch_invert_slots(clsph_state* s, uint32_t scene) {
  const uint32_t n = s->scene_n[scene], b0 = s->scene_begin[scene];
  hipLaunchKernelGGL(k_invert_slots, dim3((n + kRecBlock - 1) / kRecBlock), dim3(kRecBlock), 0,
                     s->ctx->stream, s->slot + b0, b0, n, s->sort_hist);
}

void launch_pack_records(clsph_state* s, uint32_t scene, uint32_t n, uint32_t r0, uint32_t count,
                         bool sorted, void* out, TransferStatus* status) {
  const uint32_t b0 = s->scene_begin[scene];
  const bool reorder = !s->fields_canonical;
  const bool acc = sorted || (!s->acc_zero && !reorder);
  hipLaunchKernelGGL(k_pack_records, dim3((count + kRecBlock - 1) / kRecBlock), dim3(kRecBlock), 0,
                     s->ctx->stream, (sorted ? s->pos_s : s->pos) + b0,
                     (sorted ? s->vel_s : s->vel) + b0, (sorted ? s->vh_s : s->vh) + b0,
                     acc ? s->acc_s + b0 : nullptr, s->rho_s + b0, s->prs_s + b0, s->key_b + b0,
                     s->slot + b0, reorder ? s->sort_hist : nullptr, s->dps, s->bp, scene, b0, n,
                     r0, count, sorted ? 1 : 0, reinterpret_cast<uint4*>(out), status);
}

void launch_unpack_records(clsph_state* s, uint32_t first, uint32_t count, const void* in) {
  hipLaunchKernelGGL(k_unpack_records, dim3((count + kRecBlock - 1) / kRecBlock), dim3(kRecBlock),
                     0, s->ctx->stream, reinterpret_cast<const uint4*>(in), count, s->pos + first,
                     s->vel + first, s->vh + first, s->acc_s + first, s->rho_s + first,
                     s->prs_s + first, s->key_b + first);
}

}  // namespace clsph
