// Density/pressure and internal forces over the grid neighbourhood.
//
// Reference: density_pressure (sph.cl:9-40, forces.cl:15-43) and forces
// (sph.cl:42-62, forces.cl:45-112) with the kernels of smoothing.cl. The
// reference visits all 27 cells (side 2h) around a particle's cell and
// multiplies every candidate's term by chi = 1 - clamp(floor(r/h), 0, 1).
// Particles here are ordered by half-cell (side h), so every particle within
// h of particle i lies in the 3x3x3 block of half-cells around i's own:
// visiting that block drops exactly the terms chi zeroes, and the sums are
// the reference's up to FP32 rounding (summation order differs).
#include <algorithm>

#include "state.h"

namespace clsph {

// Half-cell coordinates, with the hash's arithmetic (grid.cl:55-61):
// (uint)(2 (x - min) / (2h)).
__device__ inline void half_cell(float4 x, const DevParams* __restrict__ dp, uint32_t hc[3]) {
#pragma clang fp contract(off)
  float L = dp->p.h * 2;
  hc[0] = (uint32_t)(2.f * ((x.x - dp->p.min_point.s[0]) / L));
  hc[1] = (uint32_t)(2.f * ((x.y - dp->p.min_point.s[1]) / L));
  hc[2] = (uint32_t)(2.f * ((x.z - dp->p.min_point.s[2]) / L));
}

// Morton key of a half-cell within its scene: (cell id << 3) | octant.
__device__ inline uint32_t half_key(uint32_t hx, uint32_t hy, uint32_t hz) {
  return (morton3(hx >> 1, hy >> 1, hz >> 1) << 3) | ((hz & 1u) << 2) | ((hy & 1u) << 1) |
         (hx & 1u);
}

// Particles of the half-cells [f, f + len) (Morton-adjacent, keys of the
// batch), from the half-cell table ht; keys at or beyond F (the end of the
// scene's keys) hold none of its particles. The clamps keep a table from a
// stage run out of order from indexing past the arrays.
__device__ inline void half_range(uint32_t f, uint32_t len, const uint32_t* __restrict__ ht,
                                  uint32_t F, uint32_t n, uint32_t& s, uint32_t& e) {
  if (f >= F) {
    s = e = 0;
    return;
  }
  uint32_t g = f + len;
  g = g > F ? F : g;
  s = ht[f];
  e = ht[g];
  e = e < n ? e : n;
  s = s < e ? s : e;
}

// End of the scene's keys usable for table lookups; 0 when the table
// overflowed (an error bit is raised in that case).
__device__ inline uint32_t usable_key_end(const DevParams* __restrict__ dp,
                                          const BatchParams* __restrict__ bp) {
  return (bp->err & (kErrTableCap | kErrFineKey)) ? 0u : dp->key_end;
}

// Visits the runs [s, e) of particles of the 3x3x3 half-cells around hc in
// z, y, x order. Along x the three cells form two Morton-contiguous runs: the
// pair starting at the even coordinate, and the remaining one.
template <typename F>
__device__ inline void for_each_run(const uint32_t hc[3], uint32_t base,
                                    const uint32_t* __restrict__ ht, uint32_t Fc, uint32_t n,
                                    F&& fn) {
  const uint32_t x0 = hc[0] - 1u;
  const bool even = (x0 & 1u) == 0u;
  // not unrolled: nine rows' addresses ahead cost its callers 22 registers
#pragma unroll 1
  for (uint32_t dz = 0; dz < 3; ++dz)
#pragma unroll 1
    for (uint32_t dy = 0; dy < 3; ++dy) {
      uint32_t y = hc[1] + dy - 1u, z = hc[2] + dz - 1u;
      uint32_t a = base + half_key(x0, y, z);
      uint32_t b = base + half_key(even ? x0 + 2u : x0 + 1u, y, z);
      uint32_t s, e;
      half_range(a, even ? 2u : 1u, ht, Fc, n, s, e);
      fn(s, e);
      half_range(b, even ? 1u : 2u, ht, Fc, n, s, e);
      fn(s, e);
    }
}

// Half-cell coordinates and the particle's fractional position inside its
// half-cell (in units of the half-cell side h), with the hash's arithmetic.
__device__ inline void half_cell_frac(float4 x, const DevParams* __restrict__ dp, uint32_t hc[3],
                                      float fr[3]) {
#pragma clang fp contract(off)
  float L = dp->p.h * 2;
  float u[3] = {2.f * ((x.x - dp->p.min_point.s[0]) / L),
                2.f * ((x.y - dp->p.min_point.s[1]) / L),
                2.f * ((x.z - dp->p.min_point.s[2]) / L)};
  for (int a = 0; a < 3; ++a) {
    hc[a] = (uint32_t)u[a];
    fr[a] = u[a] - (float)hc[a];
  }
}

// Squared reach, in half-cell units, beyond which a half-cell cannot hold a
// particle within h: (1.01)^2. The 1 % margin exceeds the FP32 rounding of
// the scaled coordinates (a few ulp of at most 2048 half-cells, < 1e-3).
constexpr float kReach2 = 1.0201f;

// Two- and four-lane unsigned vectors, held in aligned register pairs and
// quads; the neighbour list's rows are addressed as global memory.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) u32x4 global_u32x4;

// (p0, p1, p2, p3) <- (p1, p2, p3, tail.y): the quad as two register pairs,
// each filled by one 64-bit move that takes one 32-bit half from each of two
// pairs (dst.lo = src0 half op_sel[0], dst.hi = src1 half op_sel[1]).
__device__ inline void shift_in(u32x4& reg, u32x2 tail) {
  u32x2 lo = reg.xy, hi = reg.zw;
  asm("v_pk_mov_b32 %0, %0, %1 op_sel:[1,0]" : "+v"(lo) : "v"(hi));
  asm("v_pk_mov_b32 %0, %0, %1 op_sel:[1,1]" : "+v"(hi) : "v"(tail));
  reg = (u32x4){lo.x, lo.y, hi.x, hi.y};
}

// Squared distance of a candidate, with every rounding written out so that
// both walks (and any inlining of them) compute the same bits.
__device__ inline float dist2(float4 xi, float4 c) {
#pragma clang fp contract(off)
  const float dx = xi.x - c.x, dy = xi.y - c.y, dz = xi.z - c.z;
  return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Density sum and neighbour list of one particle i. The sum starts with i's
// own term (r = 0: (h^2)^3) and adds the other candidates within h in
// visiting order. The list holds those neighbours (self excluded) in
// visiting order, four to a uint4, at nbr[q * n + i] (q < kMaxNeighbours / 4);
// pending entries wait in the shift register `reg` (oldest in .x, newest in
// .w), and `row` points at the list row the next four go to (nbr + i, then
// one row of n entries further per store).
struct DensityWalk {
  float acc;
  u32x4 reg = {0u, 0u, 0u, 0u};
  uint32_t cnt = 0;
  global_u32x4* row;
  uint64_t n;

  __device__ DensityWalk(uint4* __restrict__ nbr, uint32_t i, uint32_t n_, float h2)
      : acc((h2 * h2) * h2), row((global_u32x4*)(nbr + i)), n(n_) {}

  // Candidate j = tail.y at squared distance d2; in_run is false for the
  // padding entries of a group of four. Testing j != i with the distance
  // keeps the append below unconditional for the lanes that take it.
  __device__ inline void visit(bool in_run, float d2, float h2, u32x2 tail, uint32_t i) {
    static_assert((kMaxNeighbours & (kMaxNeighbours - 1u)) == 0u && kMaxNeighbours >= 4u,
                  "the list-room test below needs a power of two");
    if (in_run && d2 < h2 && tail.y != i) {
      const float t = h2 - d2;
      acc = __builtin_fmaf(t, t * t, acc);
      // the register shifts on every neighbour and is stored after each
      // fourth one while the list has room: cnt % 4 == 3 and cnt < kMaxNeighbours
      const bool full = (cnt & (3u - kMaxNeighbours)) == 3u;
      shift_in(reg, tail);
      if (full) {
        *row = reg;
        // the next row, after the store has read `row`, in place
        asm volatile("v_lshl_add_u64 %0, %1, 4, %0" : "+v"(row) : "s"(n) : "memory");
      }
      ++cnt;
    }
  }

  // Entries still pending (cnt % 4 of them, the newest of the register) go
  // to row cnt / 4 while the list has room.
  __device__ inline void finish() {
    const uint32_t r = cnt & 3u;
    if (cnt < kMaxNeighbours && r)
      *row = r == 1 ? (u32x4){reg.w, 0u, 0u, 0u}
                    : (r == 2 ? (u32x4){reg.z, reg.w, 0u, 0u} : (u32x4){reg.y, reg.z, reg.w, 0u});
  }
};

// One lane's walk over its unit's halo staged in LDS: the half-cells of the
// unit (a cell, side 4, or a quad of 2x2 cells, side 6) with one half-cell
// around them, half-cell q = x + side y + side^2 z at cand[off[q], off[q + 1])
// in sorted order, each entry (x, y, z, sorted index). Each row (dy, dz) of
// the particle's 3x3x3 block is one contiguous range. A row is skipped when
// its nearest face is out of reach, and its x-range keeps the half-cells on
// either side only when they are in reach. Candidates are visited in z, y, x
// order, four loaded at a time.
__device__ inline void density_walk_halo(DensityWalk& w, uint32_t i, float4 xi,
                                         const uint32_t hc[3], const float fr[3], uint32_t side,
                                         const float4* cand, const uint32_t* off, float h2) {
  const uint32_t lx = 1u + (hc[0] & (side - 3u)), ly = 1u + (hc[1] & (side - 3u)),
                 lz = 1u + (hc[2] & 1u);
  const float lo_x = fr[0] * fr[0], hi_x = (1.f - fr[0]) * (1.f - fr[0]);
  for (int dz = -1; dz <= 1; ++dz) {
    const float az = dz < 0 ? fr[2] : (dz > 0 ? 1.f - fr[2] : 0.f);
    for (int dy = -1; dy <= 1; ++dy) {
      const float ay = dy < 0 ? fr[1] : (dy > 0 ? 1.f - fr[1] : 0.f);
      const float ryz = az * az + ay * ay;
      if (ryz >= kReach2) continue;
      const uint32_t row = side * (ly + (uint32_t)dy + side * (lz + (uint32_t)dz));
      const uint32_t xa = lo_x + ryz < kReach2 ? lx - 1u : lx;
      const uint32_t xb = hi_x + ryz < kReach2 ? lx + 1u : lx;
      // byte offsets into cand: the group at a holds entry u inside the
      // range when a < end[u] = 16 (e - u)
      const int s = (int)off[row + xa] * 16, e = (int)off[row + xb + 1u] * 16;
      const int end[4] = {e, e - 16, e - 32, e - 48};
      for (int a = s; a < e; a += 64) {
        const float4* g = (const float4*)((const char*)cand + a);
        float4 c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = g[u];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          // (z, index): the candidate's last register pair
          w.visit(u == 0 || a < end[u], dist2(xi, c[u]), h2,
                  (u32x2){__float_as_uint(c[u].z), __float_as_uint(c[u].w)}, i);
        }
      }
    }
  }
}

// One lane's walk of the sorted positions in HBM, for small work-groups: the
// same half-cells in the same order as density_walk_halo, as runs of adjacent
// half-cells, candidates loaded four at a time so that their latencies overlap
// (pos is padded by 4 entries past the particles, so a group needs no clamp).
__device__ inline void density_walk_global(DensityWalk& w, uint32_t i, float4 xi,
                                           const uint32_t hc[3], const float fr[3],
                                           const DevParams* __restrict__ dp, uint32_t F,
                                           const float4* __restrict__ pos,
                                           const uint32_t* __restrict__ table, float h2,
                                           uint32_t n) {
  const float lo_x = fr[0] * fr[0], hi_x = (1.f - fr[0]) * (1.f - fr[0]);
  for (int dz = -1; dz <= 1; ++dz) {
    const float az = dz < 0 ? fr[2] : (dz > 0 ? 1.f - fr[2] : 0.f);
    for (int dy = -1; dy <= 1; ++dy) {
      const float ay = dy < 0 ? fr[1] : (dy > 0 ? 1.f - fr[1] : 0.f);
      const float ryz = az * az + ay * ay;
      if (ryz >= kReach2) continue;
      const uint32_t y = hc[1] + (uint32_t)dy, z = hc[2] + (uint32_t)dz;
      const uint32_t xa = lo_x + ryz < kReach2 ? hc[0] - 1u : hc[0];
      const uint32_t xb = hi_x + ryz < kReach2 ? hc[0] + 1u : hc[0];
      uint32_t x = xa;
      // half-cells 2k and 2k + 1 share a cell: at most two runs per row
      for (int piece = 0; piece < 2 && x <= xb; ++piece) {
        const uint32_t xe = (x | 1u) < xb ? (x | 1u) : xb;
        uint32_t s, e;
        half_range(dp->key_base + half_key(x, y, z), xe - x + 1u, table, F, n, s, e);
        for (uint32_t j0 = s; j0 < e; j0 += 4) {
          const float4* pj = pos + j0;
          float4 c[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) c[u] = pj[u];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t j = j0 + (uint32_t)u;
            w.visit(j < e, dist2(xi, c[u]), h2, (u32x2){j, j}, i);
          }
        }
        x = xe + 1u;
      }
    }
  }
}

// Density and pressure of particle i from its kernel sum (sph.cl:36-39), and
// what the later stages read: its neighbour count, its force inputs
// fab[2i] = (x, p / rho^2), fab[2i + 1] = (v, m / rho) and, with `nu`, the
// learned surrogate's node inputs.
__device__ inline void density_store(const DevParams* __restrict__ dp, uint32_t i, float4 xi,
                                     float sum, uint32_t count, const float4* __restrict__ vel,
                                     float* __restrict__ rho, float* __restrict__ prs,
                                     float4* __restrict__ fab, uint32_t* __restrict__ nbr_count,
                                     float2* __restrict__ nu) {
  nbr_count[i] = count;
  // density = sum m * poly6 * (h^2 - r^2)^3 ; Tait pressure
  float m = dp->p.particle_mass;
  float d = m * (dp->t.poly_6 * sum);
  float q = d / dp->p.fluid_density;
  float q2 = q * q, q4 = q2 * q2;
  float p = dp->p.K * (q4 * q2 * q - 1.f);
  rho[i] = d;
  prs[i] = p;
  float4 vi = vel[i];
  fab[2u * i] = make_float4(xi.x, xi.y, xi.z, p / (d * d));
  fab[2u * i + 1u] = make_float4(vi.x, vi.y, vi.z, m / d);
  if (nu) nu[i] = node_in(d, p, dp->p.fluid_density, dp->p.K);
}

// Orders a wave's own LDS accesses (its lanes exchange data, no other wave
// is involved).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of one particle in a walk by L lanes; in arrays, every element's lists
// are read 16 bytes at a time.
constexpr uint32_t kRuns = 18;  // runs of a particle's half-cells: 9 rows of at most two
template <int L>
struct alignas(16) LaneWalk {
  static constexpr uint32_t kHits = L == 16 ? 64u : 32u;
  float t[kHits];                // neighbours not yet summed: h^2 - r^2
  uint32_t j[kHits];             // and their sorted indices
  uint32_t run_end[kRuns + 1];   // the runs laid end to end
  uint32_t run_shift[kRuns + 1]; // sorted index less laid-out index
};
static_assert(sizeof(LaneWalk<4>) % 16 == 0 && sizeof(LaneWalk<16>) % 16 == 0,
              "16-byte reads of every element are aligned");

// Density sum and neighbour list of one particle i by L consecutive lanes,
// straight from the sorted positions: its runs of half-cells are looked up by
// the lanes in parallel and laid end to end, and each round takes the next L
// candidates, four rounds' loads in flight. A ballot ranks the neighbours
// found in a round, so that they land in the particle's LDS list in visiting
// order; the sum then runs over that list: the additions, in their order, of
// DensityWalk over the same candidates. Every lane of the wave calls it
// (`live` false: nothing is written) and gets its particle's sum and count.
template <int L>
__device__ inline void density_walk_lanes(LaneWalk<L>& w, bool live, uint32_t i, float4 xi,
                                          const DevParams* __restrict__ dp, uint32_t F,
                                          const float4* __restrict__ pos,
                                          const uint32_t* __restrict__ table,
                                          uint4* __restrict__ nbr, uint32_t n, float& sum,
                                          uint32_t& count) {
  constexpr uint32_t kHits = LaneWalk<L>::kHits;
  const uint32_t sub = threadIdx.x % L, lane = threadIdx.x & 63u, first = lane - sub;
  const float h = dp->p.h, h2 = h * h;
  uint32_t hc[3];
  float fr[3];
  half_cell_frac(xi, dp, hc, fr);
  // run r: row r / 2 (dy fastest); along x the half-cells 2k and 2k + 1 share
  // a cell and are Morton-adjacent, so the reach's x-range is cut after the
  // first odd coordinate (r even: up to there, r odd: the rest)
  uint32_t laid = 0;
  const float lo_x = fr[0] * fr[0], hi_x = (1.f - fr[0]) * (1.f - fr[0]);
#pragma unroll
  for (uint32_t r0 = 0; r0 < kRuns; r0 += L) {
    const uint32_t r = r0 + sub, row = r >> 1;
    const int dy = (int)(row % 3u) - 1, dz = (int)(row / 3u) - 1;
    const float az = dz < 0 ? fr[2] : (dz > 0 ? 1.f - fr[2] : 0.f);
    const float ay = dy < 0 ? fr[1] : (dy > 0 ? 1.f - fr[1] : 0.f);
    const float ryz = az * az + ay * ay;
    uint32_t s = 0, e = 0;
    if (r < kRuns && live && ryz < kReach2) {
      const uint32_t xa = lo_x + ryz < kReach2 ? hc[0] - 1u : hc[0];
      const uint32_t xb = hi_x + ryz < kReach2 ? hc[0] + 1u : hc[0];
      const uint32_t mid = (xa | 1u) < xb ? (xa | 1u) : xb;
      const uint32_t x0 = (r & 1u) ? mid + 1u : xa, x1 = (r & 1u) ? xb : mid;
      if (x0 <= x1)
        half_range(dp->key_base + half_key(x0, hc[1] + (uint32_t)dy, hc[2] + (uint32_t)dz),
                   x1 - x0 + 1u, table, F, n, s, e);
    }
    uint32_t incl = e - s;
#pragma unroll
    for (uint32_t o = 1; o < (uint32_t)L; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o, L);
      if (sub >= o) incl += y;
    }
    if (r < kRuns) {
      w.run_end[r] = laid + incl;
      w.run_shift[r] = s - (laid + incl - (e - s));
    }
    laid += __shfl(incl, L - 1, L);
  }
  wave_lds_fence();

  float acc = (h2 * h2) * h2;    // the particle's own term
  uint32_t total = 0, pend = 0;  // neighbours summed and listed in nbr; waiting in LDS
  // sums and lists the waiting neighbours: all of them, or whole groups of
  // four (a group is one entry of nbr); what is left moves to the front
  auto drain = [&](bool all) {
    wave_lds_fence();
    const uint32_t whole = pend & ~3u, take = all ? pend : whole;
    for (uint32_t k = 0; k < take; k += 4u) {
      const float4 t4 = *(const float4*)(w.t + k);
      const float tt[4] = {t4.x, t4.y, t4.z, t4.w};
#pragma unroll
      for (uint32_t u = 0; u < 4u; ++u) {
        const float t = k + u < take ? tt[u] : 0.f;
        acc = __builtin_fmaf(t, t * t, acc);
      }
    }
    for (uint32_t k = 4u * sub; k < take && total + k < kMaxNeighbours; k += 4u * L) {
      const uint4 j4 = *(const uint4*)(w.j + k);
      const uint32_t left = take - k;
      nbr[(size_t)((total + k) >> 2) * n + i] =
          make_uint4(j4.x, left > 1u ? j4.y : 0u, left > 2u ? j4.z : 0u, left > 3u ? j4.w : 0u);
    }
    total += take;
    const uint32_t left = pend - take;
    float mt = 0.f;
    uint32_t mj = 0;
    if (sub < left) mt = w.t[whole + sub], mj = w.j[whole + sub];
    wave_lds_fence();
    if (sub < left) w.t[sub] = mt, w.j[sub] = mj;
    pend = left;
    wave_lds_fence();
  };

  constexpr uint32_t kAhead = 4;
  uint32_t r = 0, r_end = w.run_end[0], shift = w.run_shift[0];
  for (uint32_t a = 0; __any(a < laid); a += kAhead * L) {
    float4 c[kAhead];
    uint32_t j[kAhead];
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) {
      const uint32_t k = a + u * L + sub;
      if (k < laid) {
        while (k >= r_end) {  // ends: the last run ends at laid
          ++r;
          r_end = w.run_end[r];
          shift = w.run_shift[r];
        }
      }
      j[u] = k < laid ? k + shift : i;  // past the end: the particle itself, no neighbour
      c[u] = pos[j[u]];
    }
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) {
      if (__any(pend + L > kHits)) drain(false);
      const float d2 = dist2(xi, c[u]);
      const bool hit = d2 < h2 && j[u] != i;
      const uint32_t found = (uint32_t)(__ballot(hit) >> first) & ((1u << L) - 1u);
      if (hit) {
        const uint32_t at = pend + (uint32_t)__popc(found & ((1u << sub) - 1u));
        w.t[at] = h2 - d2;
        w.j[at] = j[u];
      }
      pend += (uint32_t)__popc(found);
    }
  }
  drain(true);
  sum = acc;
  count = total;
}

// The density stage by L lanes per particle, for states too small to fill the
// chip with one particle per lane (rule in launch_density). Bound by the
// latency of its four dependent loads (position, table, candidates twice) and
// the ordered sum: 12 us at 4,096 particles, where one lane's walk took 66.
constexpr int kLanesBlock = 256;
constexpr uint32_t kLanes16Max = 40960;   // particles up to which 16 lanes take one
constexpr uint32_t kLanes4Max = 180224;   // and up to which 4 lanes do
template <int L>
__global__ __launch_bounds__(kLanesBlock) void k_density_lanes(
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const uint32_t* __restrict__ table, const BlockDesc* __restrict__ blocks,
    const DevParams* __restrict__ dps, const BatchParams* __restrict__ bp,
    float* __restrict__ rho, float* __restrict__ prs, float4* __restrict__ fab,
    uint4* __restrict__ nbr, uint32_t* __restrict__ nbr_count, float2* __restrict__ nu,
    uint32_t n) {
  constexpr uint32_t kParts = kLanesBlock / L;  // particles per work-group
  __shared__ LaneWalk<L> walks[kParts];
  // a 64-particle entry of the work list is shared by 64 / kParts work-groups
  constexpr uint32_t kShare = 64u / kParts;
  const BlockDesc b = blocks[blockIdx.x / kShare];
  const DevParams* dp = dps + b.scene;
  const uint32_t part = threadIdx.x / L;
  const uint32_t p = b.first + (blockIdx.x % kShare) * kParts + part;
  const uint32_t se = dp->begin + dp->n;
  const bool live = p < se;
  if (!__any(live)) return;
  const uint32_t i = live ? p : se - 1u;
  const float4 xi = pos[i];
  float sum;
  uint32_t count;
  density_walk_lanes<L>(walks[part], live, i, xi, dp, usable_key_end(dp, bp), pos, table, nbr, n,
                        sum, count);
  if (live && threadIdx.x % L == 0u)
    density_store(dp, i, xi, sum, count, vel, rho, prs, fab, nbr_count, nu);
}

// Inverse of spread10: the 10 bits at positions 3k.
__device__ inline uint32_t compact10(uint32_t v) {
  v &= 0x09249249u;
  v = (v | (v >> 2)) & 0x030C30C3u;
  v = (v | (v >> 4)) & 0x0300F00Fu;
  v = (v | (v >> 8)) & 0x030000FFu;
  v = (v | (v >> 16)) & 0x000003FFu;
  return v;
}

// Halo staging of the density kernel, per work-group of WAVES waves: the
// half-cells around a unit of its particles' cells, kCap candidates (x, y, z,
// index: 16 B each) in all. A unit is a quad of 2x2 cells in x and y (one run
// of the Morton order; 6x6x4 half-cells, about 1,152 candidates at rest for
// 256 particles) where all the work-group's quads fit, otherwise a cell
// (4x4x4, 512 for 64): quads stage a quarter fewer candidates for the same
// particles, but when dense the first ones that fit hold fewer of them. At 8
// waves 4,888 candidates fill a work-group's half of a CU's LDS: in settled
// fluid a cell that just doesn't fit leaves a few particles to a walk of HBM
// after all others (with 4,820 candidates, 207,000 and 262,144 particles took
// 146 and 135 us after 1,800 substeps, now 82 and 88); below, 768 per wave and
// two cells per wave. One wave's particles nearly always span two quads of
// which one fits, so it stages cells only.
constexpr uint32_t kQuadBox = 144, kCellBox = 64;  // half-cells of a halo
template <int WAVES>
struct DensityHalos {
  static constexpr uint32_t kQuads = WAVES == 8 ? 6u : WAVES == 4 ? 3u : WAVES == 2 ? 1u : 0u;
  static constexpr uint32_t kCells = WAVES < 8 ? 2u * WAVES : 13u;
  static constexpr uint32_t kEntries =  // half-cells of the halos at most
      kQuads * kQuadBox > kCells * kCellBox ? kQuads * kQuadBox : kCells * kCellBox;
  static constexpr uint32_t kCap = WAVES < 8 ? 768u * WAVES - 4u : 4888u;
  float4 cand[kCap + 4];               // + the padding of a group of four
  uint32_t off[kEntries + 1u];         // halo by halo, half-cell by half-cell
  uint32_t unit[kCells];               // the units' Morton codes
  uint32_t wave_sum[WAVES];
  uint32_t wave_units[WAVES];
};
// Lanes per particle outside the staged halos, and what their walks keep in
// the candidates' bytes (two 80 KB work-groups per CU leave no others). One or
// two waves stage too little of dense fluid to leave many of their particles to
// four lanes each: those walk one to a lane, beside the staged ones (207,000
// particles after 20 and 1,800 substeps, work-groups of 64: 131 and 182 us by
// four lanes, 120 and 148 by one; of 128: 87 and 214, 91 and 169).
constexpr int kRestLanes = 4;
template <int WAVES>
struct DensityRest {
  LaneWalk<kRestLanes> walk[WAVES * 64 / kRestLanes];
  uint16_t thread[WAVES * 64];
};

// Density and pressure (sph.cl:9-40, forces.cl:15-43) of the particles
// [first, first + 64 WAVES) of one scene, with each particle's neighbour
// list (self excluded) in visiting order into nbr[q * n + i]. The work-group
// first stages the halos of the units its particles fall in (DensityHalos) in
// LDS (coalesced runs of the sorted positions); particles then walk their
// 3x3x3 half-cells there, one to a lane. Those of units beyond the staging
// capacity, and every particle when the table is unusable, are walked from HBM
// with the same visiting order: by four lanes each after the others (a lane's
// walk of HBM by itself took 30-50 us, in some work-group of every launch), in
// small work-groups by their own lanes (kRestLanes). With cells only, whose
// halos overlap more, 207,000 particles took 65 us instead of 41 after 20
// substeps, 1,048,576 209, 149 and 219 instead of 198, 147 and 203 after 20,
// 200 and 1,000, 2,097,152
// 389, 339 and 446 instead of 376, 325 and 398.
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void k_density(const float4* __restrict__ pos,
                                                        const float4* __restrict__ vel,
                                                        const uint32_t* __restrict__ keys,
                                                        const uint32_t* __restrict__ table,
                                                        const BlockDesc* __restrict__ blocks,
                                                        const DevParams* __restrict__ dps,
                                                        const BatchParams* __restrict__ bp,
                                                        float* __restrict__ rho,
                                                        float* __restrict__ prs,
                                                        float4* __restrict__ fab,
                                                        uint4* __restrict__ nbr,
                                                        uint32_t* __restrict__ nbr_count,
                                                        float2* __restrict__ nu, uint32_t n) {
  using Halos = DensityHalos<WAVES>;
  constexpr int kPer = 2;  // half-cells per thread
  static_assert(Halos::kEntries <= (uint32_t)kPer * 64u * WAVES, "every half-cell has a thread");
  __shared__ Halos sh;
  // runs of 16 work-groups per XCD: neighbouring halos share an L2
  const BlockDesc b = blocks[xcd_block<16>(blockIdx.x, gridDim.x)];
  const DevParams* dp = dps + b.scene;
  const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
  const uint32_t se = dp->begin + dp->n;
  const uint32_t i = b.first + t;
  const bool live = i < se;
  const float h = dp->p.h, h2 = h * h;
  const uint32_t F = usable_key_end(dp, bp);

  // Units of the work-group's particles, in order: a particle starts one
  // when it is the first particle or its unit differs from its predecessor's.
  const uint32_t key = live ? keys[i] - dp->key_base : 0u;
  const uint32_t prev = (live && t > 0) ? keys[i - 1] - dp->key_base : 0u;
  uint32_t units, ui, side = Halos::kQuads ? 6u : 4u;
  auto find_units = [&](uint32_t bits) {
    const bool starts = live && (t == 0 || (key >> bits) != (prev >> bits));
    const uint64_t mask = __ballot(starts);
    if (lane == 0) sh.wave_units[wv] = (uint32_t)__popcll(mask);
    __syncthreads();
    uint32_t before = 0;
    units = 0;
    for (int q = 0; q < WAVES; ++q) {
      const uint32_t c = sh.wave_units[q];
      before += (uint32_t)q < wv ? c : 0u;
      units += c;
    }
    // index of the particle's unit among the work-group's units
    ui = before + (uint32_t)__popcll(mask & (~0ull >> (63u - lane))) - 1u;
    if (starts && ui < Halos::kCells) sh.unit[ui] = key >> bits;
  };
  find_units(side == 6u ? 5u : 3u);
  uint32_t rs[kPer], rc[kPer], ex[kPer], staged, box;
  for (;;) {
    const uint32_t most = F == 0u ? 0u : (side == 6u ? Halos::kQuads : Halos::kCells);
    const uint32_t halos = units < most ? units : most;
    box = side == 6u ? kQuadBox : kCellBox;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const uint32_t q = (uint32_t)kPer * t + (uint32_t)u;
      rs[u] = rc[u] = 0u;
      const uint32_t hh = side == 6u ? q / kQuadBox : q / kCellBox;
      if (hh < halos) {
        const uint32_t un = sh.unit[hh], l = q - hh * box;
        const uint32_t r = side == 6u ? l / 6u : l >> 2, x = l - r * side;
        const uint32_t z = side == 6u ? r / 6u : r >> 2, y = r - z * side;
        // a cell's Morton code is un; a quad's (2x2 cells in x and y) lacks
        // their last bits
        const uint32_t hx = side == 6u ? 4u * compact10(un >> 1) : 2u * compact10(un);
        const uint32_t hy = side == 6u ? 4u * compact10(un >> 2) : 2u * compact10(un >> 1);
        const uint32_t hz = 2u * compact10(side == 6u ? un : un >> 2);
        const uint32_t gx = hx - 1u + x, gy = hy - 1u + y, gz = hz - 1u + z;
        if (gx < 2048u && gy < 2048u && gz < 2048u) {
          const uint32_t f = dp->key_base + half_key(gx, gy, gz);
          if (f < F) {
            uint32_t e = table[f + 1u];
            e = e < n ? e : n;
            uint32_t s = table[f];
            s = s < e ? s : e;
            rs[u] = s;
            rc[u] = e - s;
          }
        }
      }
    }
    // exclusive scan of the run lengths over the work-group
    uint32_t mine = 0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) mine += rc[u];
    uint32_t incl = mine;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    if (lane == 63) sh.wave_sum[wv] = incl;
    __syncthreads();
    uint32_t base = 0;
    for (int q = 0; q < WAVES; ++q) base += (uint32_t)q < wv ? sh.wave_sum[q] : 0u;
    uint32_t at = base + incl - mine;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const uint32_t q = (uint32_t)kPer * t + (uint32_t)u;
      if (q < Halos::kEntries) sh.off[q] = at;
      ex[u] = at;
      at += rc[u];
    }
    if (t == WAVES * 64u - 1u) sh.off[Halos::kEntries] = at;
    __syncthreads();
    // halos staged: the leading ones whose candidates fit
    staged = 0;
    while (staged < halos && sh.off[box * (staged + 1u)] <= Halos::kCap) ++staged;
    if (staged == units || side == 4u || F == 0u) break;
    // not all quads fit: cell by cell
    side = 4u;
    find_units(3u);
  }
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const uint32_t q = (uint32_t)kPer * t + (uint32_t)u;
    if ((side == 6u ? q / kQuadBox : q / kCellBox) < staged) {
      for (uint32_t k = 0; k < rc[u]; ++k) {
        const uint32_t j = rs[u] + k;
        const float4 p = pos[j];
        sh.cand[ex[u] + k] = make_float4(p.x, p.y, p.z, __uint_as_float(j));
      }
    }
  }
  __syncthreads();

  constexpr bool kRest = WAVES >= 4;  // the particles not staged follow, by several lanes
  if (live && (!kRest || ui < staged)) {
    const float4 xi = pos[i];
    uint32_t hc[3];
    float fr[3];
    half_cell_frac(xi, dp, hc, fr);
    DensityWalk w(nbr, i, n, h2);
    if (kRest || ui < staged)
      density_walk_halo(w, i, xi, hc, fr, side, sh.cand, sh.off + box * ui, h2);
    else
      density_walk_global(w, i, xi, hc, fr, dp, F, pos, table, h2, n);
    w.finish();
    density_store(dp, i, xi, w.acc, w.cnt, vel, rho, prs, fab, nbr_count, nu);
  }
  if (!kRest || staged == units) return;  // uniform: every particle has been walked
  // the rest, in the order of their threads
  const bool left = live && ui >= staged;
  const uint64_t lm = __ballot(left);
  if (lane == 0) sh.wave_sum[wv] = (uint32_t)__popcll(lm);
  __syncthreads();  // also: the staged walks are done with cand
  uint32_t at = 0, rest = 0;
  for (int q = 0; q < WAVES; ++q) {
    at += (uint32_t)q < wv ? sh.wave_sum[q] : 0u;
    rest += sh.wave_sum[q];
  }
  using Rest = DensityRest<WAVES>;
  static_assert(sizeof(Rest) <= sizeof(sh.cand), "it fits in the candidates' bytes");
  Rest& rest_lds = reinterpret_cast<Rest&>(sh.cand);
  if (left) rest_lds.thread[at + (uint32_t)__popcll(lm & ((1ull << lane) - 1ull))] = (uint16_t)t;
  __syncthreads();
  constexpr uint32_t kParts = WAVES * 64 / kRestLanes;
  LaneWalk<kRestLanes>& walk = rest_lds.walk[t / kRestLanes];
  for (uint32_t r0 = 0; r0 < rest; r0 += kParts) {
    const uint32_t r = r0 + t / kRestLanes;
    const bool on = r < rest;
    if (!__any(on)) break;
    const uint32_t ip = b.first + rest_lds.thread[on ? r : 0u];
    const float4 xi = pos[ip];
    float sum;
    uint32_t count;
    density_walk_lanes<kRestLanes>(walk, on, ip, xi, dp, F, pos, table, nbr, n, sum, count);
    if (on && t % kRestLanes == 0u)
      density_store(dp, ip, xi, sum, count, vel, rho, prs, fab, nbr_count, nu);
  }
}

// Pair terms of compute_internal_forces_with_grid (forces.cl:60-101) for one
// neighbour j != i at squared distance d2 < h^2; a = (x, p/rho^2) and
// b = (v, m/rho) of each particle.
struct ForceSums {
  float3 pt, vt, nrm;
  float lap;
};

struct ForceConsts {
  float h, h2, m, c_spiky, c_visc, c_grad, c_lap, spiky0;
};

// Every rounding of the sums is written out, so that both kernels below (and
// any inlining) compute the same bits.
__device__ inline float length2(float x, float y, float z) {
  return __builtin_fmaf(z, z, __builtin_fmaf(x, x, y * y));
}

// A pair's terms: each sum adds a weight times a value.
struct PairTerms {
  float g, vw, gw, lw;     // weights: pressure, viscosity, colour-field gradient and laplacian
  float3 dir, dv, dx;      // values of the first three
  float lv;
};

__device__ inline PairTerms pair_terms(const ForceConsts& k, float4 ai, float4 bi, float4 aj,
                                       float4 bj) {
#pragma clang fp contract(off)
  PairTerms p;
  float dx = ai.x - aj.x, dy = ai.y - aj.y, dz = ai.z - aj.z;
  float d2 = length2(dx, dy, dz);
  float r = __builtin_amdgcn_sqrtf(d2);
  float t = k.h2 - d2;
  float hr = k.h - r;
  // pressure (forces.cl:66-73): (p_j/rho_j^2 + p_i/rho_i^2) m grad W_spiky
  float ps = (aj.w + ai.w) * k.m;
  const bool coincident = r < 1e-7f;
  p.g = coincident ? ps * k.spiky0 : ps * k.c_spiky * hr * hr * __builtin_amdgcn_rcpf(r);
  p.dir = make_float3(coincident ? 1.f : dx, coincident ? 1.f : dy, coincident ? 1.f : dz);
  // viscosity (forces.cl:75-80): (v_j - v_i) (m/rho_j) lap W_visc
  p.vw = bj.w * k.c_visc * hr;
  p.dv = make_float3(bj.x - bi.x, bj.y - bi.y, bj.z - bi.z);
  // colour field gradient and laplacian (forces.cl:83-91)
  p.gw = bj.w * k.c_grad * t * t;
  p.dx = make_float3(dx, dy, dz);
  p.lw = bj.w * k.c_lap * t;
  p.lv = __builtin_fmaf(-7.f, d2, 3.f * k.h2);
  return p;
}

__device__ inline void force_pair(ForceSums& f, const ForceConsts& k, float4 ai, float4 bi,
                                  float4 aj, float4 bj) {
  const PairTerms p = pair_terms(k, ai, bi, aj, bj);
  f.pt.x = __builtin_fmaf(p.g, p.dir.x, f.pt.x);
  f.pt.y = __builtin_fmaf(p.g, p.dir.y, f.pt.y);
  f.pt.z = __builtin_fmaf(p.g, p.dir.z, f.pt.z);
  f.vt.x = __builtin_fmaf(p.vw, p.dv.x, f.vt.x);
  f.vt.y = __builtin_fmaf(p.vw, p.dv.y, f.vt.y);
  f.vt.z = __builtin_fmaf(p.vw, p.dv.z, f.vt.z);
  f.nrm.x = __builtin_fmaf(p.gw, p.dx.x, f.nrm.x);
  f.nrm.y = __builtin_fmaf(p.gw, p.dx.y, f.nrm.y);
  f.nrm.z = __builtin_fmaf(p.gw, p.dx.z, f.nrm.z);
  f.lap = __builtin_fmaf(p.lw, p.lv, f.lap);
}

__device__ inline ForceConsts force_consts(const DevParams* __restrict__ dp) {
  ForceConsts k;
  k.h = dp->p.h;
  k.h2 = k.h * k.h;
  k.m = dp->p.particle_mass;
  k.c_spiky = dp->t.spiky;
  k.c_visc = dp->t.viscosity;
  k.c_grad = dp->t.poly_6_gradient;
  k.c_lap = dp->t.poly_6_laplacian;
  // Coincident-particle branch of spiky_gradient (smoothing.cl:23-25).
  const float h3 = k.h2 * k.h;
  k.spiky0 = -45.f / (3.14159274f * (h3 * h3));
  return k;
}

// The sums before the first pair: the self term of the colour-field
// laplacian, (m/rho_i) poly6_lap h^2 (3 h^2).
__device__ inline ForceSums force_start(const ForceConsts& k, float4 bi) {
  ForceSums fs;
  fs.pt = make_float3(0.f, 0.f, 0.f);
  fs.vt = fs.pt;
  fs.nrm = fs.pt;
  fs.lap = bi.w * k.c_lap * k.h2 * (3.f * k.h2);
  return fs;
}

// The neighbours past those the list holds, of which `last` is the final one:
// walks the half-cells again from there, in density's order and with its test,
// W candidates' loads in flight (one where registers are short).
// (Walking them all from the start, one candidate after another, took the
// stage from 35 to 123 us once some lists overflowed, 131,071 particles.)
template <uint32_t W>
__device__ inline void force_walk(ForceSums& fs, const ForceConsts& k, uint32_t i, float4 ai,
                                  float4 bi, uint32_t last, const float4* __restrict__ fab,
                                  const uint32_t* __restrict__ table,
                                  const DevParams* __restrict__ dp, uint32_t F, uint32_t n) {
  uint32_t hc[3];
  half_cell(ai, dp, hc);
  bool past = false;
  for_each_run(hc, dp->key_base, table, F, n, [&](uint32_t s, uint32_t e) {
    if (!past) {
      if (last < s || last >= e) return;
      past = true;
      s = last + 1u;
    }
    for (uint32_t j0 = s; j0 < e; j0 += W) {
      float4 aj[W];
#pragma unroll
      for (uint32_t u = 0; u < W; ++u) aj[u] = fab[2u * (j0 + u < e ? j0 + u : j0)];
#pragma unroll
      for (uint32_t u = 0; u < W; ++u) {
        const uint32_t j = j0 + u;
        if (j < e && dist2(ai, aj[u]) < k.h2 && j != i)
          force_pair(fs, k, ai, bi, aj[u], fab[2u * j + 1u]);
      }
    }
  });
}

// The last entry of particle i's full list.
__device__ inline uint32_t last_listed(const uint4* __restrict__ nbr, uint32_t i, uint32_t n) {
  return nbr[(size_t)(kMaxNeighbours / 4u - 1u) * n + i].w;
}

// Acceleration from the sums (forces.cl:95-111 and sph.cl:53-58).
__device__ inline float4 force_close(const ForceSums& fs, float rho_i,
                                     const DevParams* __restrict__ dp) {
#pragma clang fp contract(off)
  const float3 pt = fs.pt, vt = fs.vt, nrm = fs.nrm;
  const float mu = dp->p.dynamic_viscosity;
  float3 f = make_float3(__builtin_fmaf(vt.x, mu, -(rho_i * pt.x)),
                         __builtin_fmaf(vt.y, mu, -(rho_i * pt.y)),
                         __builtin_fmaf(vt.z, mu, -(rho_i * pt.z)));
  const float nl = sqrtf(length2(nrm.x, nrm.y, nrm.z));
  if (nl > dp->p.surface_tension_threshold) {
    const float kk = -dp->p.surface_tension * fs.lap / nl;
    f.x = __builtin_fmaf(kk, nrm.x, f.x);
    f.y = __builtin_fmaf(kk, nrm.y, f.y);
    f.z = __builtin_fmaf(kk, nrm.z, f.z);
  }
  const clsph_float3& g = dp->p.constant_acceleration;
  return make_float4(f.x / rho_i + g.s[0], f.y / rho_i + g.s[1], f.z / rho_i + g.s[2], 0.f);
}

// The acceleration of particle i by sixteen consecutive lanes: a round takes
// the next sixteen neighbours of the list, one per lane, and leaves their terms
// in LDS (w, kForceTerms rows); ten lanes then each add one sum's terms in list
// order, so that every sum is the one lane's of k_forces to the bit. The next
// round's gathers are in flight meanwhile. Every lane of the wave calls it
// (`live` false: nothing is written).
constexpr int kForceLanes = 16, kForceLanesBlock = 256;
constexpr uint32_t kForceTerms = 14;  // PairTerms' floats, in order
constexpr uint32_t kForcePitch = 20;  // floats between terms: 16-byte reads, spread over banks
__device__ inline void force_lanes(float* w, bool live, uint32_t i,
                                   const float4* __restrict__ fab, const float* __restrict__ rho,
                                   const uint32_t* __restrict__ table,
                                   const uint4* __restrict__ nbr,
                                   const uint32_t* __restrict__ nbr_count,
                                   const DevParams* __restrict__ dp,
                                   const BatchParams* __restrict__ bp,
                                   float4* __restrict__ acc_out, uint32_t n) {
  constexpr uint32_t L = kForceLanes;
  const uint32_t sub = threadIdx.x % L;
  const ForceConsts k = force_consts(dp);
  const float4 ai = fab[2u * i], bi = fab[2u * i + 1u];
  const uint32_t all = nbr_count[i];
  const uint32_t cnt = live ? (all < kMaxNeighbours ? all : kMaxNeighbours) : 0u;
  auto index = [&](uint32_t q) {  // past the end: the particle itself
    return q < cnt ? reinterpret_cast<const uint32_t*>(nbr)[4u * ((size_t)(q >> 2) * n + i) + (q & 3u)]
                   : i;
  };
  // the sum this lane adds: its weight's and value's rows of the terms
  const uint32_t sum = sub < 10u ? sub : 9u, kind = sum / 3u;
  const uint32_t wrow = kind, vrow = 4u + sum;
  float acc = kind == 3u ? force_start(k, bi).lap : 0.f;
  uint32_t j = index(sub), jn = index(L + sub);
  float4 aj = fab[2u * j], bj = fab[2u * j + 1u];
  for (uint32_t q0 = 0; __any(q0 < cnt); q0 += L) {
    const float4 na = fab[2u * jn], nb = fab[2u * jn + 1u];
    jn = index(q0 + 2u * L + sub);
    const PairTerms t = pair_terms(k, ai, bi, aj, bj);
    const float v[kForceTerms] = {t.g,    t.vw,   t.gw,   t.lw,   t.dir.x, t.dir.y, t.dir.z,
                                  t.dv.x, t.dv.y, t.dv.z, t.dx.x, t.dx.y,  t.dx.z,  t.lv};
#pragma unroll
    for (uint32_t r = 0; r < kForceTerms; ++r) w[r * kForcePitch + sub] = v[r];
    wave_lds_fence();
    const uint32_t left = cnt > q0 ? cnt - q0 : 0u, take = left < L ? left : L;
#pragma unroll
    for (uint32_t g = 0; g < L; g += 4u) {
      const float4 wt = *(const float4*)(w + wrow * kForcePitch + g);
      const float4 va = *(const float4*)(w + vrow * kForcePitch + g);
      if (g < take) acc = __builtin_fmaf(wt.x, va.x, acc);
      if (g + 1u < take) acc = __builtin_fmaf(wt.y, va.y, acc);
      if (g + 2u < take) acc = __builtin_fmaf(wt.z, va.z, acc);
      if (g + 3u < take) acc = __builtin_fmaf(wt.w, va.w, acc);
    }
    wave_lds_fence();
    aj = na;
    bj = nb;
  }
  w[sub] = acc;  // sub >= 10 repeats the last sum, past the ten
  wave_lds_fence();
  if (!live || sub != 0u) return;
  ForceSums fs;
  fs.pt = make_float3(w[0], w[1], w[2]);
  fs.vt = make_float3(w[3], w[4], w[5]);
  fs.nrm = make_float3(w[6], w[7], w[8]);
  fs.lap = w[9];
  if (all > kMaxNeighbours)
    force_walk<1>(fs, k, i, ai, bi, last_listed(nbr, i, n), fab, table, dp,
                  usable_key_end(dp, bp), n);
  acc_out[i] = force_close(fs, rho[i], dp);
}

// The forces stage by sixteen lanes per particle, for states too small to
// fill the chip with one particle per lane (rule in launch_forces). Bound by
// the latency of the list, the two gathers and the serial sums (4,096
// particles: 4.3 us, a lane each 10.5).
constexpr uint32_t kForceLanesMax = 57344;  // particles up to which they do
constexpr uint32_t kSmallScene = 8192;      // particles of a scene up to which, with none
constexpr uint32_t kForceLanesSmallMax = 28672;  // larger, they do up to this many
__global__ __launch_bounds__(kForceLanesBlock) void k_forces_lanes(
    const float4* __restrict__ fab, const float* __restrict__ rho,
    const uint32_t* __restrict__ table, const uint4* __restrict__ nbr,
    const uint32_t* __restrict__ nbr_count, const BlockDesc* __restrict__ blocks,
    const DevParams* __restrict__ dps, const BatchParams* __restrict__ bp,
    float4* __restrict__ acc_out, uint32_t n) {
  constexpr uint32_t kParts = kForceLanesBlock / kForceLanes, kShare = 64u / kParts;
  __shared__ __attribute__((aligned(16))) float terms[kParts][kForceTerms * kForcePitch];
  // a 64-particle entry of the work list is shared by kShare work-groups
  const BlockDesc b = blocks[blockIdx.x / kShare];
  const DevParams* dp = dps + b.scene;
  const uint32_t part = threadIdx.x / kForceLanes;
  const uint32_t p = b.first + (blockIdx.x % kShare) * kParts + part;
  const uint32_t se = dp->begin + dp->n;
  const bool live = p < se;
  if (!__any(live)) return;
  force_lanes(terms[part], live, live ? p : se - 1u, fab, rho, table, nbr, nbr_count, dp, bp,
              acc_out, n);
}

// The forces stage for the particles whose neighbours overflow the list only
// (more than kMaxNeighbours), for callers that sum the others themselves. A
// wave reads the counts of a 64-particle entry of the work list, and nearly
// always leaves; its overflowing particles are taken four at a time, by
// sixteen lanes each. Bound by that one load while no list overflows: 4.5 us
// at 1,048,576 particles (by a lane each, whose pipelined list sum took 131
// registers and left three waves per SIMD, 7.1; a macro step of 262,144 whose
// lists overflow 526 and 534 us).
__global__ __launch_bounds__(kForceLanesBlock) void k_forces_overflow(
    const float4* __restrict__ fab, const float* __restrict__ rho,
    const uint32_t* __restrict__ table, const uint4* __restrict__ nbr,
    const uint32_t* __restrict__ nbr_count, const BlockDesc* __restrict__ blocks, uint32_t entries,
    const DevParams* __restrict__ dps, const BatchParams* __restrict__ bp,
    float4* __restrict__ acc_out, uint32_t n) {
  constexpr uint32_t kParts = kForceLanesBlock / kForceLanes;
  __shared__ __attribute__((aligned(16))) float terms[kParts][kForceTerms * kForcePitch];
  // the same in all lanes, so that the scene's parameters stay in scalar registers
  const uint32_t entry = blockIdx.x * (kForceLanesBlock / 64u) +
                         (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (entry >= entries) return;
  const BlockDesc b = blocks[entry];
  const DevParams* dp = dps + b.scene;
  const uint32_t lane = threadIdx.x & 63u, p = b.first + lane;
  uint64_t over = __ballot(p < dp->begin + dp->n && nbr_count[p] > kMaxNeighbours);
  while (over) {
    // the wave's four groups of lanes take the four lowest particles left
    uint64_t mine = over;
    for (uint32_t q = 0; q < lane / kForceLanes; ++q) mine &= mine - 1u;
    force_lanes(terms[threadIdx.x / kForceLanes], mine != 0u,
                b.first + (uint32_t)__builtin_ctzll(mine ? mine : over), fab, rho, table, nbr,
                nbr_count, dp, bp, acc_out, n);
    wave_lds_fence();  // the sums are read before the next round's terms
    for (int q = 0; q < 4; ++q) over &= over - 1u;
  }
}

// The forces stage by a lane per particle.
__global__ __launch_bounds__(kMaxBlock) void k_forces(const float4* __restrict__ fab,
                                                      const float* __restrict__ rho,
                                                      const uint32_t* __restrict__ table,
                                                      const uint4* __restrict__ nbr,
                                                      const uint32_t* __restrict__ nbr_count,
                                                      const BlockDesc* __restrict__ blocks,
                                                      const DevParams* __restrict__ dps,
                                                      const BatchParams* __restrict__ bp,
                                                      float4* __restrict__ acc_out, uint32_t n) {
  uint32_t scene;
  // runs of 4 work-groups per XCD: neighbour records shared in an L2
  uint32_t i = particle_of<4>(blocks, dps, scene);
  if (i == 0xFFFFFFFFu) return;
  const DevParams* dp = dps + scene;
  const ForceConsts k = force_consts(dp);
  const uint32_t F = usable_key_end(dp, bp);
  float4 ai = fab[2u * i], bi = fab[2u * i + 1u];
  float rho_i = rho[i];
  ForceSums fs = force_start(k, bi);
  const uint32_t all = nbr_count[i], cnt = all < kMaxNeighbours ? all : kMaxNeighbours;
  // groups of four neighbours, software-pipelined: while a group's pair
  // terms are summed, the next group's records and the indices of the one
  // after it are in flight
  const uint32_t groups = cnt >> 2;
  auto gather = [&](uint4 js, float4 ra[4], float4 rb[4]) {
    const uint32_t jj[4] = {js.x, js.y, js.z, js.w};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ra[u] = fab[2u * jj[u]];
      rb[u] = fab[2u * jj[u] + 1u];
    }
  };
  float4 ca[4], cb[4];
  uint4 jn = make_uint4(0u, 0u, 0u, 0u);
  if (groups) {
    gather(nbr[i], ca, cb);
    if (groups > 1) jn = nbr[(size_t)n + i];
  }
  for (uint32_t gq = 0; gq < groups; ++gq) {
    float4 na[4], nb[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) na[u] = ca[u], nb[u] = cb[u];
    if (gq + 1 < groups) gather(jn, na, nb);
    if (gq + 2 < groups) jn = nbr[(size_t)(gq + 2) * n + i];
#pragma unroll
    for (int u = 0; u < 4; ++u) force_pair(fs, k, ai, bi, ca[u], cb[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) ca[u] = na[u], cb[u] = nb[u];
  }
  const uint32_t q = groups << 2;
  if (q < cnt) {
    uint4 js = nbr[(size_t)(q >> 2) * n + i];
    uint32_t r = cnt - q;
    force_pair(fs, k, ai, bi, fab[2u * js.x], fab[2u * js.x + 1u]);
    if (r > 1) force_pair(fs, k, ai, bi, fab[2u * js.y], fab[2u * js.y + 1u]);
    if (r > 2) force_pair(fs, k, ai, bi, fab[2u * js.z], fab[2u * js.z + 1u]);
  }
  if (all > kMaxNeighbours)
    force_walk<4>(fs, k, i, ai, bi, last_listed(nbr, i, n), fab, table, dp, F, n);
  acc_out[i] = force_close(fs, rho_i, dp);
}

void launch_density(clsph_state* s, float2* nu) {
  if (s->n == 0) return;
  // Lanes per particle. One (k_density) does the least work, but its time is
  // at least a wave's walk, 30-50 us; below that many particles the chip has
  // lanes to spare. Stage time on evolved dam breaks, 1 / 4 / 16 lanes:
  // 16,384 particles 86 / 25 / 15 us, 50,021 49 / 31 / 30, 65,536
  // 48 / 34 / 36, 131,071 62 / 49 / 58. 1 / 4 lanes after 20, 200, 1,000 and
  // 1,800 substeps: 131,071 31, 46, 58, 81 / 46, 43, 39, 56 us, 160,000 40, 64,
  // 59, 84 / 50, 46, 51, 61, 180,225 74, 41, 62, 82 / 55, 50, 56, 70, 207,000
  // 41, 42, 63, 82 / 63, 58, 58, 77, 262,144 42, 58, 65, 88 / 74, 67, 71, 93,
  // 524,288 78, 85, 125, 165 / 133, 122, 129, 178 (settled fluid is two to
  // three times as dense).
  if (s->n <= kLanes4Max) {
    // 64-particle entries of the work list, whatever the stage's block size
    auto lanes = [&](auto kernel, uint32_t share) {
      hipLaunchKernelGGL(kernel, dim3(s->nblocks[0] * share), dim3(kLanesBlock), 0,
                         s->ctx->stream, s->pos_s, s->vel_s, s->table, s->blocks[0], s->dps, s->bp,
                         s->rho_s, s->prs_s, s->fab, s->nbr, s->nbr_count, nu, s->n);
    };
    if (s->n <= kLanes16Max) lanes(k_density_lanes<16>, 4);
    else lanes(k_density_lanes<4>, 1);
    return;
  }
  const int bs = s->bs_of(kStageDensity);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(s->nblocks_of(kStageDensity)), dim3(bs), 0, s->ctx->stream,
                       s->pos_s, s->vel_s, s->key_b, s->table, s->table_of(kStageDensity), s->dps,
                       s->bp, s->rho_s, s->prs_s, s->fab, s->nbr, s->nbr_count, nu, s->n);
  };
  switch (bs) {
    case 64: go(k_density<1>); break;
    case 128: go(k_density<2>); break;
    case 256: go(k_density<4>); break;
    default: go(k_density<8>); break;
  }
}

void launch_forces(clsph_state* s) {
  if (s->n == 0) return;
  // One lane per particle does half the work, but takes at least a lane's
  // whole list: 10.5 us with 35 neighbours, 24-29 us with the up to 128 of a
  // settled dam break. Stage times with 1 / 16 lanes, early and settled: 4,096
  // particles 10.5 / 4.3 and 15.5 / 5.6 us, 16,384 11.6 / 6.3 and 22.7 / 8.9,
  // 50,021 12.1 / 13.4 and 28.1 / 20.4, 65,536 12.1 / 15.6 and 28.9 / 24.3,
  // 98,304 12.2 / 22.1 and 28.2 / 32.4. Small scenes' lists stay short however
  // many scenes there are: 100 of 200 particles 7.9 / 8.7 and 9.3 / 9.3, 20 of
  // 1,500 10.8 / 9.8 and 14.1 / 11.6, 400 of 100 8.7 / 13.1 and 9.3 / 14.0, 100
  // of 500 10.3 / 13.8 and 11.5 / 16.3, 14 of 4,000 11.3 / 14.7 and 16.2 / 18.8.
  const uint32_t largest = *std::max_element(s->scene_n.begin(), s->scene_n.end());
  if (s->n <= (largest > kSmallScene ? kForceLanesMax : kForceLanesSmallMax)) {
    constexpr uint32_t kShare = 64u * kForceLanes / kForceLanesBlock;
    hipLaunchKernelGGL(k_forces_lanes, dim3(s->nblocks[0] * kShare), dim3(kForceLanesBlock), 0,
                       s->ctx->stream, s->fab, s->rho_s, s->table, s->nbr, s->nbr_count,
                       s->blocks[0], s->dps, s->bp, s->acc_s, s->n);
    return;
  }
  hipLaunchKernelGGL(k_forces, dim3(s->nblocks_of(kStageForces)),
                     dim3(s->bs_of(kStageForces)), 0, s->ctx->stream, s->fab, s->rho_s,
                     s->table, s->nbr, s->nbr_count, s->table_of(kStageForces), s->dps, s->bp,
                     s->acc_s, s->n);
}

void launch_forces_overflow(clsph_state* s) {
  if (s->n == 0) return;
  constexpr uint32_t kWaves = kForceLanesBlock / 64;
  hipLaunchKernelGGL(k_forces_overflow, dim3((s->nblocks[0] + kWaves - 1) / kWaves),
                     dim3(kForceLanesBlock), 0, s->ctx->stream, s->fab, s->rho_s, s->table, s->nbr,
                     s->nbr_count, s->blocks[0], s->nblocks[0], s->dps, s->bp, s->acc_s, s->n);
}

}  // namespace clsph
