// Kernels of the two-round message-passing network (gfx950): the
// neighbour-graph and edge-input builders, the fused edge-round and node-MLP
// inference kernels, activation / aggregation / loss kernels and Adam, with
// the bf16 matrix-core GEMM of nn.hip for the training products. The
// forward and backward passes are sequences of these launches on the
// context stream.
#include <hip/hip_runtime.h>

#include "gnn.h"
#include "nn.h"

namespace clsph {
namespace gnn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t to_bf16(float x) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(x));
}
__device__ inline float from_bf16(uint16_t b) {
  return __builtin_bit_cast(float, (uint32_t)b << 16);
}
// Logistic function from the hardware exp2 and reciprocal (1 ulp each): the
// activations it feeds are rounded to bf16, so IEEE division would only add
// instructions.
__device__ inline float sigmoid(float x) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * -1.44269504f));
}
__device__ inline float silu(float x) { return x * sigmoid(x); }
__device__ inline float dsilu(float x) {
  float s = sigmoid(x);
  return s * (1.f + x * (1.f - s));
}

// the bf16 matrix-core GEMM of the corrective surrogate (nn.hip)
using nn::colsum;
using nn::gemm;
using nn::gemm_dsilu;
using nn::gemm_silu;
using nn::gemm_weight_grad;

// ---------------------------------------------------------------------------
// Exclusive scan of min(count, kMaxEdges) into off[0..n], off[n] = total.
constexpr int kScanItems = 4;
constexpr int kScanBlock = 256;
constexpr int kScanChunk = kScanItems * kScanBlock;

__device__ inline uint32_t block_scan_256(uint32_t v, uint32_t* lds, uint32_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) lds[wave] = x;
  __syncthreads();
  uint32_t base = 0;
  for (int w = 0; w < wave; ++w) base += lds[w];
  total = lds[0] + lds[1] + lds[2] + lds[3];
  __syncthreads();
  return base + x - v;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_local(const uint32_t* __restrict__ count,
                                                           uint32_t n, uint32_t* __restrict__ off,
                                                           uint32_t* __restrict__ part) {
  __shared__ uint32_t lds[4];
  uint32_t base = blockIdx.x * kScanChunk + threadIdx.x * kScanItems;
  uint32_t v[kScanItems], sum = 0;
  bool cut = false;
  for (int t = 0; t < kScanItems; ++t) {
    uint32_t i = base + t;
    v[t] = i < n ? min(count[i], kMaxEdges) : 0u;
    cut = cut || (i < n && count[i] > kMaxEdges);
    sum += v[t];
  }
  // the chunk's second word: a list was cut short at kMaxEdges
  const int any = __syncthreads_or(cut ? 1 : 0);
  if (threadIdx.x == 0) part[2 * blockIdx.x + 1] = any ? 1u : 0u;
  uint32_t total;
  uint32_t ex = block_scan_256(sum, lds, total);
  for (int t = 0; t < kScanItems; ++t) {
    uint32_t i = base + t;
    if (i < n) off[i] = ex;
    ex += v[t];
  }
  if (threadIdx.x == 0) part[2 * blockIdx.x] = total;
}

// One work-group scans the chunk totals (any count) in place; total_out[0] is
// their sum, total_out[1] whether any chunk's second word is set.
__global__ __launch_bounds__(kScanBlock) void k_scan_parts(uint32_t* __restrict__ part,
                                                           uint32_t nparts,
                                                           uint32_t* __restrict__ total_out) {
  __shared__ uint32_t lds[4];
  uint32_t carry = 0;
  int cut = 0;
  for (uint32_t b = 0; b < nparts; b += kScanBlock) {
    uint32_t i = b + threadIdx.x;
    uint32_t v = i < nparts ? part[2 * i] : 0u;
    cut |= __syncthreads_or(i < nparts && part[2 * i + 1] ? 1 : 0);
    uint32_t total;
    uint32_t ex = block_scan_256(v, lds, total);
    if (i < nparts) part[2 * i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) {
    total_out[0] = carry;
    total_out[1] = cut ? 1u : 0u;
  }
}

__global__ __launch_bounds__(256) void k_scan_add(uint32_t* __restrict__ off,
                                                  const uint32_t* __restrict__ part, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) off[i] += part[2 * (i / kScanChunk)];
}

// ---------------------------------------------------------------------------
// src / dst of every edge (dst-major, the density kernel's neighbour order);
// blockIdx.y of gridDim.y takes every gridDim.y-th group of four neighbours.
__global__ __launch_bounds__(256) void k_graph(const uint4* __restrict__ nbr,
                                               const uint32_t* __restrict__ count,
                                               const uint32_t* __restrict__ off, uint32_t n,
                                               uint32_t* __restrict__ src,
                                               uint32_t* __restrict__ dst,
                                               float* __restrict__ degc) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint32_t deg = min(count[i], kMaxEdges), o = off[i];
  for (uint32_t q = 4 * blockIdx.y; q < deg; q += 4 * gridDim.y) {
    uint4 js = nbr[(size_t)(q >> 2) * n + i];
    uint32_t jj[4] = {js.x, js.y, js.z, js.w};
    for (uint32_t t = 0; t < 4 && q + t < deg; ++t) {
      src[o + q + t] = jj[t];
      dst[o + q + t] = i;
    }
  }
  if (blockIdx.y == 0) degc[i] = (float)deg / kAggC;
}

// The 16 edge inputs of edge (i <- j) in float32 (12 used, 4 zero).
__device__ inline void edge_features(float4 xi, float4 xj, float4 vi, float4 vj, float2 ni,
                                     float2 nj, float inv_h, float f[kFeat]) {
  float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
  float q = sqrtf(dx * dx + dy * dy + dz * dz) * inv_h;
  float w = 1.f - q * q;
  f[0] = dx * inv_h, f[1] = dy * inv_h, f[2] = dz * inv_h;
  f[3] = (vi.x - vj.x) / kVelScale, f[4] = (vi.y - vj.y) / kVelScale;
  f[5] = (vi.z - vj.z) / kVelScale;
  f[6] = q, f[7] = w * w * w;
  f[8] = ni.x, f[9] = ni.y, f[10] = nj.x, f[11] = nj.y;
  f[12] = f[13] = f[14] = f[15] = 0.f;
}

// Edge inputs e (16 bf16 per edge) and node inputs nu.
__global__ __launch_bounds__(256) void k_edge_inputs(
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const float* __restrict__ rho, const float* __restrict__ prs,
    const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst, uint32_t e, uint32_t n,
    float h, float rho0, float K, uint16_t* __restrict__ E1, float* __restrict__ nu) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) {
    float2 a = node_in(rho[k], prs[k], rho0, K);
    nu[2 * k] = a.x;
    nu[2 * k + 1] = a.y;
  }
  if (k >= e) return;
  uint32_t i = dst[k], j = src[k];
  float f[kFeat];
  edge_features(pos[i], pos[j], vel[i], vel[j], node_in(rho[i], prs[i], rho0, K),
                node_in(rho[j], prs[j], rho0, K), 1.f / h, f);
  uint32_t packed[8];
  for (int t = 0; t < 8; ++t)
    packed[t] = (uint32_t)to_bf16(f[2 * t]) | ((uint32_t)to_bf16(f[2 * t + 1]) << 16);
  u32x4* o = (u32x4*)(E1 + (size_t)k * kFeat);
  o[0] = u32x4{packed[0], packed[1], packed[2], packed[3]};
  o[1] = u32x4{packed[4], packed[5], packed[6], packed[7]};
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

// Eight floats to bf16 (round to nearest even).
__device__ __attribute__((always_inline)) inline u32x4 pack8(const float v[8]) {
  const f32x8 x = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
  return __builtin_bit_cast(u32x4, __builtin_convertvector(x, bf16x8));
}

// Orders a wave's own LDS accesses (its lanes exchange data, no other wave is
// involved).
__device__ __attribute__((always_inline)) inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Fused edge round for inference: S_i = bf16(sum_j silu(silu(e_ij W1 + b1
// [+ PA_i + PB_j]) W2 + b2) / C) over particle i's neighbour list (the density
// kernel's, at most kMaxEdges) without storing per-edge values.
//
// A wave takes up to 16 particles at a time (a run), every R-th of R runs, so
// that particles with many neighbours, which lie together, are shared by all
// waves (an evaluation of 131,072 particles in a macro step 902 us at 29
// neighbours on average and 1,367 at 34, with consecutive particles; now 892
// and 1,006. 14,000 at 37: 304 and 265).
// The run's edges, each particle's padded to quads, are cut into four equal
// streams, one per lane group g = l / 16, whichever particles that splits; a
// tile is the next quad of each stream. (A tile of 16 edges per particle would
// be 3/4 full at 30 neighbours.) 64 edges at a time, one per lane, compute
// their inputs and pass them to the tiles through LDS as 32 bf16 K slots:
//   0-11 the inputs, 12-14 ones, 16-31 one-hot of the edge's particle.
// W1's rows 12-14 are b1 split into three bf16 (8 + 8 + 8 bits, exact) and its
// rows 16-31 the particles' PA, so layer 1's bias and node terms cost no
// instruction; PB_j is the product's starting value.
//
// Layer 1 runs transposed on 16x16x32 bf16 matrix cores, output row 4 g + r of
// block ob being feature 32 g + 4 ob + r, so lane group g of edge l % 16 holds
// 32 consecutive features. They are layer 2's A operand as they stand (slot t
// of k-step ks: feature 32 g + 8 ks + t), whose output has edges as rows and
// feature 8 (l % 16) + ob as column: register r of lane group g is edge r of
// its stream's quad, and a particle's sum stays in the lane's registers until
// its last quad. The up to three particles that the streams' ends split are
// joined through LDS at the end of the run.
//
// An infinite or NaN PA would spread over its run through the one-hot product,
// so a run with one is taken particle by particle.
//
// Bound by vector instructions: per tile and lane 64 SiLUs, of whose
// instructions 128 (exp2, rcp) take twice the issue time of the other 320;
// the matrix cores are busy for 640 of about 2,350 cycles. 131,072 particles of
// 28 neighbours: 358 us without node terms, 400 with (a tile per particle,
// node inputs recomputed per edge and 16-lane sums: 687 and 713). Four waves
// per SIMD instead of three, products issued a block ahead and runs handed out
// by a queue measured the same; sums by 16x16x4 float products with a 0/1
// matrix 452 (those run on the vector units).
constexpr int kRunMax = 16;
// 16-byte unit u of edge e's record in LDS, on distinct banks for 16 edges
__device__ inline int rec_at(int e, int u) { return 4 * e + (u ^ ((e >> 2) & 3)); }

// Node inputs nu and scaled degrees.
__global__ __launch_bounds__(256) void k_node_inputs(const float* __restrict__ rho,
                                                     const float* __restrict__ prs,
                                                     const uint32_t* __restrict__ count,
                                                     uint32_t n, float rho0, float K,
                                                     float2* __restrict__ nu,
                                                     float* __restrict__ degc) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  nu[i] = node_in(rho[i], prs[i], rho0, K);
  degc[i] = (float)min(count[i], kMaxEdges) / kAggC;
}

// The high 16 bits of b, as a float: b less it is exact and 8 bits shorter.
__device__ inline float bf16_head(float b) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, b) & 0xFFFF0000u);
}

template <bool ROUND2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_edge_fused(
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const float2* __restrict__ nu, const uint32_t* __restrict__ nbr,
    const uint32_t* __restrict__ count, uint32_t n, float h, const uint16_t* __restrict__ W1,
    const float* __restrict__ b1, const uint16_t* __restrict__ W2, const float* __restrict__ b2,
    const uint16_t* __restrict__ PA, const uint16_t* __restrict__ PB,
    uint16_t* __restrict__ S) {
  __shared__ u32x4 w2s[8 * 4 * 64];  // [ob][ks][lane]
  __shared__ u32x4 recs[4][64 * 4];
  __shared__ uint32_t js[4][64];
  __shared__ uint32_t quads[4][16];  // slot, edges << 8, last of its particle << 16
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  {
    // k-step `wave` of W2: eight rows of eight columns per lane, turned
    u32x4 row[8];
    for (int t = 0; t < 8; ++t)
      row[t] = *(const u32x4*)(W2 + (size_t)(32 * g + 8 * wave + t) * kWidth + 8 * c);
    for (int ob = 0; ob < 8; ++ob) {
      u32x4 v;
      for (int t = 0; t < 4; ++t)
        v[t] = __builtin_amdgcn_perm(row[2 * t + 1][ob >> 1], row[2 * t][ob >> 1],
                                     ob & 1 ? 0x07060302u : 0x05040100u);
      w2s[(ob * 4 + wave) * 64 + lane] = v;
    }
  }
  // layer 1's weights: lane (c, g) holds feature 32 (c / 4) + 4 ob + c % 4 of K slots 8 g + t
  u32x4 w1[8];
  for (int ob = 0; ob < 8; ++ob) {
    const int col = 32 * (c >> 2) + 4 * ob + (c & 3);
    const float b = b1[col];
    const bool finite = __builtin_fabsf(b) < __builtin_inff();
    const float head = finite ? bf16_head(b) : b, rest = finite ? b - head : 0.f;
    uint16_t v[8];
    for (int t = 0; t < 8; ++t) {
      const uint16_t row = W1[min(8 * g + t, kFeat - 1) * kWidth + col];
      v[t] = 8 * g + t < 12 ? row : (uint16_t)0;
    }
    if (g == 1) {
      v[4] = to_bf16(head);
      v[5] = to_bf16(bf16_head(rest));
      v[6] = to_bf16(rest - bf16_head(rest));
    }
    for (int t = 0; t < 4; ++t) w1[ob][t] = (uint32_t)v[2 * t] | ((uint32_t)v[2 * t + 1] << 16);
  }
  float bias2[8];
  for (int ob = 0; ob < 8; ++ob) bias2[ob] = b2[8 * c + ob];
  __syncthreads();

  // this wave's runs; consecutive ones on the same XCD's L2
  const uint32_t blocks = gridDim.x, waves = blocks * 4;
  const uint32_t b = blocks % 8 ? blockIdx.x : (blockIdx.x % 8) * (blocks / 8) + blockIdx.x / 8;
  const uint32_t w = b * 4 + wave;
  const uint32_t rounds = (n + kRunMax * waves - 1) / (kRunMax * waves);
  const uint32_t stride = waves * rounds;
  const float inv_h = 1.f / h;
  u32x4* rec = recs[wave];
  uint32_t limit = kRunMax, redo_end = 0;
  for (uint32_t q = 0, o0 = 0; q < rounds;) {
    // run q of the wave: `size` particles from `first`, every stride-th
    const uint32_t first = w + waves * q, size = first < n ? (n - 1 - first) / stride + 1 : 0u;
    if (o0 >= size) {
      ++q, o0 = 0, limit = kRunMax, redo_end = 0;
      continue;
    }
    const uint32_t parts = min(size - o0, limit), i0 = first + o0 * stride;
    if (ROUND2) {
      bool odd = false;  // PA not finite
      if (g >= 2)
        for (int ob = 0; ob < 8; ++ob) {
          const int col = 32 * (c >> 2) + 4 * ob + (c & 3);
          uint16_t v[8];
          for (int t = 0; t < 8; ++t) {
            const uint32_t p = 8 * (g - 2) + t;
            const uint16_t pa = PA[(size_t)(i0 + min(p, parts - 1) * stride) * kWidth + col];
            v[t] = p < parts ? pa : (uint16_t)0;
            odd |= (v[t] & 0x7F80u) == 0x7F80u;
          }
          for (int t = 0; t < 4; ++t)
            w1[ob][t] = (uint32_t)v[2 * t] | ((uint32_t)v[2 * t + 1] << 16);
        }
      if (parts > 1 && __any(odd)) {
        limit = 1, redo_end = o0 + parts;
        continue;
      }
    }
    // lane p: degree and first quad of particle p of the run
    const uint32_t deg = (uint32_t)lane < parts ? min(count[i0 + lane * stride], kMaxEdges) : 0u;
    uint32_t start = (deg + 3) / 4;
    for (int o = 1; o < kRunMax; o <<= 1) {
      const uint32_t y = __shfl_up(start, o, 64);
      if (lane >= o) start += y;
    }
    const uint32_t total = __builtin_amdgcn_readlane(start, kRunMax - 1);
    start -= (deg + 3) / 4;
    uint32_t from[kRunMax];
    for (int p = 1; p < kRunMax; ++p) from[p] = __builtin_amdgcn_readlane(start, p);
    // the particle that owns a quad: the last to start at or before it (one
    // without edges starts where the next does)
    auto owner = [&](uint32_t quad) {
      uint32_t slot = 0;
      for (int p = 1; p < kRunMax; ++p) slot += quad >= from[p] ? 1u : 0u;
      return quad < total ? slot : 0u;
    };
    for (uint64_t none = __ballot((uint32_t)lane < parts && deg == 0); none; none &= none - 1)
      if (lane < 16)
        *(u32x4*)(S + (size_t)(i0 + __builtin_ctzll(none) * stride) * kWidth + 8 * c) =
            u32x4{0u, 0u, 0u, 0u};
    const uint32_t tiles = (total + 3) / 4;  // quads per stream
    float acc[8], lead[8];
    for (int ob = 0; ob < 8; ++ob) acc[ob] = lead[ob] = 0.f;
    // this stream's first quad continues a particle of the stream before
    const uint32_t slot0 = owner(g * tiles);
    bool pending = g * tiles < total && g * tiles != (uint32_t)__shfl(start, slot0, 64);
    bool led = false, open = false;
    uint32_t slot = 0;
    auto store = [&](const float* sum) {
      float v[8];
      for (int ob = 0; ob < 8; ++ob) v[ob] = sum[ob] * (1.f / kAggC);
      *(u32x4*)(S + (size_t)(i0 + slot * stride) * kWidth + 8 * c) = pack8(v);
    };
    for (uint32_t t0 = 0; t0 < tiles; t0 += 4) {
      // the inputs of four tiles' edges
      wave_fence();
      {
        const uint32_t t = t0 + g, quad = ((lane >> 2) & 3) * tiles + t, r = lane & 3;
        const uint32_t p = owner(quad);
        const uint32_t k = quad - (uint32_t)__shfl(start, p, 64);
        const uint32_t d = (uint32_t)__shfl(deg, p, 64);
        const bool on = t < tiles && quad < total;
        const uint32_t i = i0 + p * stride;
        uint32_t j = i0;
        u32x4 lo = {0u, 0u, 0u, 0u}, hi = {0u, 0u, 0u, 0u};
        if (on) {
          // past the list's end the quad's first edge again, with a factor of
          // zero: finite wherever that edge's own term is
          j = nbr[((size_t)k * n + i) * 4 + (4 * k + r < d ? r : 0u)];
          float f[kFeat];
          edge_features(pos[i], pos[j], vel[i], vel[j], nu[i], nu[j], inv_h, f);
          f[12] = f[13] = f[14] = 1.f;
          lo = pack8(f), hi = pack8(f + 8);
        }
        rec[rec_at(lane, 0)] = lo;
        rec[rec_at(lane, 1)] = hi;
        if (ROUND2) {
          const uint32_t one = on ? 0x3F80u << (16 * (p & 1)) : 0u, h = p >> 1;
          rec[rec_at(lane, 2)] =
              u32x4{h == 0 ? one : 0u, h == 1 ? one : 0u, h == 2 ? one : 0u, h == 3 ? one : 0u};
          rec[rec_at(lane, 3)] =
              u32x4{h == 4 ? one : 0u, h == 5 ? one : 0u, h == 6 ? one : 0u, h == 7 ? one : 0u};
          js[wave][lane] = j;
        }
        if (r == 0)
          quads[wave][lane >> 2] =
              on ? p | (min(d - 4 * k, 4u) << 8) | (4 * k + 4 >= d ? 0x10000u : 0u) : 0u;
      }
      wave_fence();
      // PB of the tile's edges, loaded a layer ahead
      const uint32_t here = min(tiles - t0, 4u);
      u32x4 pb[4];
      auto load_pb = [&](uint32_t t) {
        const u32x4* p = (const u32x4*)(PB + (size_t)js[wave][16 * t + c] * kWidth + 32 * g);
        for (int q = 0; q < 4; ++q) pb[q] = p[q];
      };
      if (ROUND2) load_pb(0);
#pragma unroll 1
      for (uint32_t t = 0; t < here; ++t) {
        u32x4 er = {0u, 0u, 0u, 0u};
        if (ROUND2 || g < 2) er = rec[rec_at(16 * t + c, g)];
        const bf16x8 eb = __builtin_bit_cast(bf16x8, er);
        const uint32_t info = quads[wave][4 * t + g], edges = (info >> 8) & 0xFFu;
        auto layer1 = [&](int ob) {
          f32x4 z = {0.f, 0.f, 0.f, 0.f};
          if (ROUND2) {
            const uint32_t x = pb[ob >> 1][2 * (ob & 1)], y = pb[ob >> 1][2 * (ob & 1) + 1];
            z = f32x4{__builtin_bit_cast(float, x << 16),
                      __builtin_bit_cast(float, x & 0xFFFF0000u),
                      __builtin_bit_cast(float, y << 16),
                      __builtin_bit_cast(float, y & 0xFFFF0000u)};
          }
          return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w1[ob]), eb, z,
                                                         0, 0, 0);
        };
        bf16x8 a2[4];
        auto layer2 = [&](int ob) {
          f32x4 y = {bias2[ob], bias2[ob], bias2[ob], bias2[ob]};
          for (int ks = 0; ks < 4; ++ks)
            y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a2[ks], __builtin_bit_cast(bf16x8, w2s[(ob * 4 + ks) * 64 + lane]), y, 0, 0, 0);
          return y;
        };
        for (int ks = 0; ks < 4; ++ks) {
          const f32x4 z0 = layer1(2 * ks), z1 = layer1(2 * ks + 1);
          float v8[8];
          for (int r = 0; r < 4; ++r) v8[r] = silu(z0[r]), v8[4 + r] = silu(z1[r]);
          a2[ks] = __builtin_bit_cast(bf16x8, pack8(v8));
          __builtin_amdgcn_sched_barrier(0);
        }
        if (ROUND2) load_pb(min(t + 1, here - 1));
        // SiLU's 1 + exp2(..), or infinity (a factor of zero) past the quad's edges
        float one[4];
        for (uint32_t r = 0; r < 4; ++r) one[r] = r < edges ? 1.f : __builtin_inff();
        for (int ob = 0; ob < 8; ++ob) {
          const f32x4 y = layer2(ob);
          for (int r = 0; r < 4; ++r)
            acc[ob] = __builtin_fmaf(
                y[r], __builtin_amdgcn_rcpf(one[r] + __builtin_amdgcn_exp2f(y[r] * -1.44269504f)),
                acc[ob]);
          __builtin_amdgcn_sched_barrier(0);  // one output block's reads at a time
        }
        if (edges) slot = info & 0xFFu, open = !(info >> 16);
        if (__any(info >> 16)) {
          if (info >> 16) {
            if (pending) {
              for (int ob = 0; ob < 8; ++ob) lead[ob] = acc[ob];
              led = true, pending = false;
            } else {
              store(acc);
            }
            for (int ob = 0; ob < 8; ++ob) acc[ob] = 0.f;
          }
        }
      }
    }
    if (__any(open)) {
      // a particle that goes on in later streams: their leading sums, and
      // whole streams of it
      wave_fence();
      float4* rows = (float4*)rec;  // [g][acc, lead][128]
      for (int q = 0; q < 2; ++q) {
        rows[(2 * g) * 32 + 2 * c + q] =
            make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        rows[(2 * g + 1) * 32 + 2 * c + q] =
            make_float4(lead[4 * q], lead[4 * q + 1], lead[4 * q + 2], lead[4 * q + 3]);
      }
      wave_fence();
      for (int h = 1; h < 4; ++h) {
        const bool whole = __shfl((int)(open && pending), 16 * h, 64);
        const bool part = __shfl((int)led, 16 * h, 64);
        const uint32_t of = __shfl(slot0, 16 * h, 64);
        if (h > g && open && of == slot && (whole || part))
          for (int q = 0; q < 2; ++q) {
            const float4 v = rows[(2 * h + (whole ? 0 : 1)) * 32 + 2 * c + q];
            acc[4 * q] += v.x, acc[4 * q + 1] += v.y;
            acc[4 * q + 2] += v.z, acc[4 * q + 3] += v.w;
          }
      }
      if (open && !pending) store(acc);
    }
    o0 += parts;
    if (o0 >= redo_end) limit = kRunMax;
  }
}

// ---------------------------------------------------------------------------
// Fused node MLPs for inference. A wave handles tiles of 16 particles; each
// layer runs transposed on 16x16x32 bf16 matrix cores (outputs as rows,
// particles as columns), chaining in registers as the edge kernel does. B
// operands come either from memory in the natural K order (slot t of k-step
// ks, lane group g: feature 32 ks + 8 g + t) or from the previous layer's
// registers in the permuted order (32 ks + 16 (t / 4) + 4 g + t % 4); each
// layer's weights are staged once per work-group in LDS in the matching
// order. Rounding points are those of the GEMM path (bf16 layer inputs,
// float32 accumulation).
constexpr int kNodeTile = 16;

// Stages W rows for k-steps [ks0, ks0 + nks) of a layer with `ks_total`
// k-steps and `nob` 16-wide output blocks: dst[(ob * ks_total + ks) * 64 +
// lane] holds W[k][16 ob + lane % 16] for the lane's 8 K slots; rows at or
// beyond `kvalid` are zero. `krow0` is the W row of the first staged k-step.
__device__ __attribute__((always_inline)) inline void stage_layer(u32x4* dst, int ks_total, int ks0, int nks, int nob,
                                   const uint16_t* __restrict__ Wm, int ld, int krow0, int kvalid,
                                   bool perm) {
  const int total = nob * nks * 64;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    int l = idx & 63, ks = (idx >> 6) % nks, ob = (idx >> 6) / nks, g = l >> 4;
    int col = 16 * ob + (l & 15);
    uint32_t w[4];
    for (int t2 = 0; t2 < 4; ++t2) {
      uint32_t half[2];
      for (int h = 0; h < 2; ++h) {
        int t = 2 * t2 + h;
        int k = krow0 + 32 * ks + (perm ? 16 * (t >> 2) + 4 * g + (t & 3) : 8 * g + t);
        half[h] = k < kvalid ? Wm[(size_t)k * ld + col] : 0u;
      }
      w[t2] = half[0] | (half[1] << 16);
    }
    dst[(ob * ks_total + ks0 + ks) * 64 + l] = u32x4{w[0], w[1], w[2], w[3]};
  }
}

template <int NOB, int NKS>
__device__ __attribute__((always_inline)) inline void mfma_layer(const u32x4* __restrict__ w, const bf16x8* bop, f32x4* y) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob) {
    f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[(ob * NKS + ks) * 64 + lane]),
                                                   bop[ks], a, 0, 0, 0);
    y[ob] = a;
    // keep each block's weight reads next to its products: hoisting all of
    // a layer's LDS reads would need 4 NOB NKS registers more
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Permuted-order B operands (4 k-steps, 128 features) from a 128-wide
// layer's registers, optionally through SiLU.
__device__ __attribute__((always_inline)) inline void to_operands(const f32x4* y, bool act, bf16x8* bop) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    float v8[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      float v = y[2 * ks + (t >> 2)][t & 3];
      v8[t] = act ? silu(v) : v;
    }
    bop[ks] = __builtin_bit_cast(bf16x8, pack8(v8));
  }
}

// Natural-order B operands: features 32 ks + 8 g .. + 7 of a bf16 row.
__device__ __attribute__((always_inline)) inline void load_operands(const uint16_t* __restrict__ row, bool valid, int nks,
                                     bf16x8* bop) {
  const int g = (threadIdx.x & 63) >> 4;
  for (int ks = 0; ks < nks; ++ks) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (valid) v = *(const u32x4*)(row + 32 * ks + 8 * g);
    bop[ks] = __builtin_bit_cast(bf16x8, v);
  }
}

// Adds bias[16 ob + 4 g + r] (+ scale * bias2) to a 128-wide layer.
__device__ __attribute__((always_inline)) inline void add_bias(f32x4* y, int nob, const float* __restrict__ b,
                                const float* __restrict__ b2, float scale) {
  const int g = (threadIdx.x & 63) >> 4;
  for (int ob = 0; ob < nob; ++ob)
    for (int r = 0; r < 4; ++r) {
      int f = 16 * ob + 4 * g + r;
      y[ob][r] += b[f] + (b2 ? scale * b2[f] : 0.f);
    }
}

// Writes features 16 ob + 4 g .. + 3 of a particle's bf16 row.
__device__ __attribute__((always_inline)) inline void store_row_bf16(uint16_t* __restrict__ row, const f32x4* y) {
  const int g = (threadIdx.x & 63) >> 4;
  for (int ob = 0; ob < 8; ++ob) {
    uint32_t lo = (uint32_t)to_bf16(y[ob][0]) | ((uint32_t)to_bf16(y[ob][1]) << 16);
    uint32_t hi = (uint32_t)to_bf16(y[ob][2]) | ((uint32_t)to_bf16(y[ob][3]) << 16);
    *(uint2*)(row + 16 * ob + 4 * g) = make_uint2(lo, hi);
  }
}

// Round-1 node part: M1 = S0 W3 + (deg / C) b3; H = MLP([M1, nu, 0]); Hb.
__global__ __launch_bounds__(512) void k_node1(const uint16_t* __restrict__ S0,
                                               const float* __restrict__ degc,
                                               const float* __restrict__ nu, uint32_t n,
                                               const uint16_t* __restrict__ wb,
                                               const float* __restrict__ params,
                                               uint16_t* __restrict__ Hb) {
  extern __shared__ u32x4 lds[];
  u32x4* w3 = lds;                 // 8 x 4
  u32x4* wa = w3 + 8 * 4 * 64;     // 8 x 5
  u32x4* wb2 = wa + 8 * 5 * 64;    // 8 x 4
  u32x4* wc = wb2 + 8 * 4 * 64;    // 8 x 4
  float* bias = (float*)(wc + 8 * 4 * 64);  // b3, ba, bb, bc
  stage_layer(w3, 4, 0, 4, 8, wb + param_offset(E1_W3), kWidth, 0, kWidth, false);
  stage_layer(wa, 5, 0, 4, 8, wb + param_offset(N1_W1), kWidth, 0, kIn1, true);
  stage_layer(wa, 5, 4, 1, 8, wb + param_offset(N1_W1), kWidth, kWidth, kWidth + 2, false);
  stage_layer(wb2, 4, 0, 4, 8, wb + param_offset(N1_W2), kWidth, 0, kWidth, true);
  stage_layer(wc, 4, 0, 4, 8, wb + param_offset(N1_W3), kWidth, 0, kWidth, true);
  for (int k = threadIdx.x; k < kWidth; k += blockDim.x) {
    bias[k] = params[param_offset(E1_B3) + k];
    bias[kWidth + k] = params[param_offset(N1_B1) + k];
    bias[2 * kWidth + k] = params[param_offset(N1_B2) + k];
    bias[3 * kWidth + k] = params[param_offset(N1_B3) + k];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const uint32_t tiles = (n + kNodeTile - 1) / kNodeTile;
  for (uint32_t tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); tile < tiles;
       tile += waves) {
    const uint32_t i = tile * kNodeTile + c;
    const bool valid = i < n;
    bf16x8 bop[5];
    f32x4 y[8];
    load_operands(S0 + (size_t)(valid ? i : 0) * kWidth, valid, 4, bop);
    mfma_layer<8, 4>(w3, bop, y);
    {
      const float dc = valid ? degc[i] : 0.f;  // M1 = S0 W3 + (deg / C) b3
      for (int ob = 0; ob < 8; ++ob)
        for (int r = 0; r < 4; ++r) y[ob][r] += dc * bias[16 * ob + 4 * g + r];
    }
    to_operands(y, false, bop);
    {
      float v8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (g == 0 && valid) {
        v8[0] = nu[2 * i];
        v8[1] = nu[2 * i + 1];
      }
      bop[4] = __builtin_bit_cast(bf16x8, pack8(v8));
    }
    mfma_layer<8, 5>(wa, bop, y);
    add_bias(y, 8, bias + kWidth, nullptr, 0.f);
    to_operands(y, true, bop);
    mfma_layer<8, 4>(wb2, bop, y);
    add_bias(y, 8, bias + 2 * kWidth, nullptr, 0.f);
    to_operands(y, true, bop);
    mfma_layer<8, 4>(wc, bop, y);
    add_bias(y, 8, bias + 3 * kWidth, nullptr, 0.f);
    if (valid) store_row_bf16(Hb + (size_t)i * kWidth, y);
  }
}

// Round-2 node terms: PA = bf16(Hb Wa), PB = bf16(Hb Wb).
__global__ __launch_bounds__(512) void k_node_terms(const uint16_t* __restrict__ Hb, uint32_t n,
                                                    const uint16_t* __restrict__ wb,
                                                    uint16_t* __restrict__ PA,
                                                    uint16_t* __restrict__ PB) {
  extern __shared__ u32x4 lds[];
  u32x4* wa = lds;
  u32x4* wbb = wa + 8 * 4 * 64;
  stage_layer(wa, 4, 0, 4, 8, wb + param_offset(E2_WA), kWidth, 0, kWidth, false);
  stage_layer(wbb, 4, 0, 4, 8, wb + param_offset(E2_WB), kWidth, 0, kWidth, false);
  __syncthreads();
  const int c = threadIdx.x & 15;
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const uint32_t tiles = (n + kNodeTile - 1) / kNodeTile;
  for (uint32_t tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); tile < tiles;
       tile += waves) {
    const uint32_t i = tile * kNodeTile + c;
    const bool valid = i < n;
    bf16x8 bop[4];
    f32x4 y[8];
    load_operands(Hb + (size_t)(valid ? i : 0) * kWidth, valid, 4, bop);
    mfma_layer<8, 4>(wa, bop, y);
    if (valid) store_row_bf16(PA + (size_t)i * kWidth, y);
    mfma_layer<8, 4>(wbb, bop, y);
    if (valid) store_row_bf16(PB + (size_t)i * kWidth, y);
  }
}

// Round-2 node part: M2 = S1 W3' + (deg / C) b3'; out = MLP([H, M2]);
// acc = g + A out[0:3]. Writes out (32 floats per particle) as well.
__global__ __launch_bounds__(512) void k_node2(const uint16_t* __restrict__ S1,
                                               const uint16_t* __restrict__ Hb,
                                               const float* __restrict__ degc, uint32_t n,
                                               const uint16_t* __restrict__ wb,
                                               const float* __restrict__ params,
                                               float* __restrict__ out, float4* __restrict__ acc,
                                               float gx, float gy, float gz) {
  extern __shared__ u32x4 lds[];
  u32x4* w3 = lds;                 // 8 x 4
  u32x4* wa = w3 + 8 * 4 * 64;     // 8 x 8
  u32x4* wb2 = wa + 8 * 8 * 64;    // 8 x 4
  u32x4* wc = wb2 + 8 * 4 * 64;    // 2 x 4
  float* bias = (float*)(wc + 2 * 4 * 64);  // b3, ba, bb (128 each), bc (32)
  stage_layer(w3, 4, 0, 4, 8, wb + param_offset(E2_W3), kWidth, 0, kWidth, false);
  stage_layer(wa, 8, 0, 4, 8, wb + param_offset(N2_W1), kWidth, 0, kWidth, false);
  stage_layer(wa, 8, 4, 4, 8, wb + param_offset(N2_W1), kWidth, kWidth, kIn2, true);
  stage_layer(wb2, 4, 0, 4, 8, wb + param_offset(N2_W2), kWidth, 0, kWidth, true);
  stage_layer(wc, 4, 0, 4, 2, wb + param_offset(N2_W3), kOut, 0, kWidth, true);
  for (int k = threadIdx.x; k < kWidth; k += blockDim.x) {
    bias[k] = params[param_offset(E2_B3) + k];
    bias[kWidth + k] = params[param_offset(N2_B1) + k];
    bias[2 * kWidth + k] = params[param_offset(N2_B2) + k];
    if (k < kOut) bias[3 * kWidth + k] = params[param_offset(N2_B3) + k];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const uint32_t waves = gridDim.x * (blockDim.x >> 6);
  const uint32_t tiles = (n + kNodeTile - 1) / kNodeTile;
  for (uint32_t tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); tile < tiles;
       tile += waves) {
    const uint32_t i = tile * kNodeTile + c;
    const bool valid = i < n;
    bf16x8 bop[8];
    f32x4 y[8];
    load_operands(S1 + (size_t)(valid ? i : 0) * kWidth, valid, 4, bop);
    mfma_layer<8, 4>(w3, bop, y);
    {
      const float dc = valid ? degc[i] : 0.f;
      for (int ob = 0; ob < 8; ++ob)
        for (int r = 0; r < 4; ++r) y[ob][r] += dc * bias[16 * ob + 4 * g + r];
    }
    load_operands(Hb + (size_t)(valid ? i : 0) * kWidth, valid, 4, bop);
    to_operands(y, false, bop + 4);
    mfma_layer<8, 8>(wa, bop, y);
    add_bias(y, 8, bias + kWidth, nullptr, 0.f);
    to_operands(y, true, bop);
    mfma_layer<8, 4>(wb2, bop, y);
    add_bias(y, 8, bias + 2 * kWidth, nullptr, 0.f);
    to_operands(y, true, bop);
    f32x4 o[2];
    mfma_layer<2, 4>(wc, bop, o);
    for (int ob = 0; ob < 2; ++ob)
      for (int r = 0; r < 4; ++r) o[ob][r] += bias[3 * kWidth + 16 * ob + 4 * g + r];
    if (valid) {
      float* orow = out + (size_t)i * kOut;
      for (int ob = 0; ob < 2; ++ob)
        *(float4*)(orow + 16 * ob + 4 * g) = make_float4(o[ob][0], o[ob][1], o[ob][2], o[ob][3]);
      if (g == 0)
        acc[i] = make_float4(gx + kAccScale * o[0][0], gy + kAccScale * o[0][1],
                             gz + kAccScale * o[0][2], 0.f);
    }
  }
}

// ---------------------------------------------------------------------------
// Elementwise and row kernels (grid-stride loops).
__global__ void k_cast_2d(const float* __restrict__ x, int ldx, uint16_t* __restrict__ y, int ldy,
                          size_t rows, int cols) {
  size_t count = rows * cols;
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x) {
    size_t r = k / cols;
    int c = (int)(k % cols);
    y[r * ldy + c] = to_bf16(x[r * ldx + c]);
  }
}

__global__ void k_copy_2d(const float* __restrict__ x, int ldx, float* __restrict__ y, int ldy,
                          size_t rows, int cols) {
  size_t count = rows * cols;
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x) {
    size_t r = k / cols;
    int c = (int)(k % cols);
    y[r * ldy + c] = x[r * ldx + c];
  }
}

// dz2[e] = bf16(dS[dst[e]] * silu'(z2[e])), 128 features per edge, eight per
// thread.
__global__ __launch_bounds__(256) void k_edge_dz(const float* __restrict__ dS,
                                                 const float* __restrict__ z2,
                                                 const uint32_t* __restrict__ dst,
                                                 uint16_t* __restrict__ dz, size_t e) {
  const size_t count = e * (kWidth / 8);
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x) {
    const size_t ed = k / (kWidth / 8), c = 8 * (k % (kWidth / 8));
    const float4* zp = (const float4*)(z2 + ed * kWidth + c);
    const float4* dp = (const float4*)(dS + (size_t)dst[ed] * kWidth + c);
    uint32_t w[4];
    for (int h = 0; h < 2; ++h) {
      const float4 zz = zp[h], dd = dp[h];
      w[2 * h] = (uint32_t)to_bf16(dd.x * dsilu(zz.x)) | ((uint32_t)to_bf16(dd.y * dsilu(zz.y)) << 16);
      w[2 * h + 1] =
          (uint32_t)to_bf16(dd.z * dsilu(zz.z)) | ((uint32_t)to_bf16(dd.w * dsilu(zz.w)) << 16);
    }
    *(u32x4*)(dz + ed * kWidth + c) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

// S[i] = bf16(scale * sum over i's edges of silu(z2)); one wave per node.
__global__ __launch_bounds__(256) void k_segsum_silu(const float* __restrict__ z2,
                                                     const uint32_t* __restrict__ off, uint32_t n,
                                                     float scale, uint16_t* __restrict__ S) {
  uint32_t i = blockIdx.x * 4 + (threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  if (i >= n) return;
  float a0 = 0.f, a1 = 0.f;
  for (uint32_t k = off[i]; k < off[i + 1]; ++k) {
    float2 z = *(const float2*)(z2 + (size_t)k * kWidth + 2 * lane);
    a0 += silu(z.x);
    a1 += silu(z.y);
  }
  S[(size_t)i * kWidth + 2 * lane] = to_bf16(a0 * scale);
  S[(size_t)i * kWidth + 2 * lane + 1] = to_bf16(a1 * scale);
}

// out[i] = sum over i's edges of x (bf16 rows, 128 wide); one wave per node.
__global__ __launch_bounds__(256) void k_segsum_rows(const uint16_t* __restrict__ x,
                                                     const uint32_t* __restrict__ off, uint32_t n,
                                                     float* __restrict__ out) {
  uint32_t i = blockIdx.x * 4 + (threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  if (i >= n) return;
  float a0 = 0.f, a1 = 0.f;
  for (uint32_t k = off[i]; k < off[i + 1]; ++k) {
    uint32_t v = *(const uint32_t*)(x + (size_t)k * kWidth + 2 * lane);
    a0 += from_bf16((uint16_t)(v & 0xFFFFu));
    a1 += from_bf16((uint16_t)(v >> 16));
  }
  out[(size_t)i * kWidth + 2 * lane] = a0;
  out[(size_t)i * kWidth + 2 * lane + 1] = a1;
}

// out[j] = sum over the edges e with src[e] = j of x[e] (bf16 rows, 128 wide),
// when no neighbour list was cut short: neighbours are then mutual, so those
// edges are j's own neighbours i, each at the place of j in i's list. One wave
// per particle; four neighbours' lists, then their rows, in flight. (Adding
// every row with atomics instead takes 357 us for 557,000 edges, this 53.)
__global__ __launch_bounds__(256) void k_gather_rows(const uint16_t* __restrict__ x,
                                                     const uint32_t* __restrict__ off,
                                                     const uint32_t* __restrict__ src, uint32_t n,
                                                     float* __restrict__ out) {
  const uint32_t j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (j >= n) return;
  const uint32_t k0 = off[j], k1 = off[j + 1];
  float a0 = 0.f, a1 = 0.f;
  for (uint32_t k = k0; k < k1; k += 4) {
    uint32_t lo[4], hi[4], v[4][2];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      const bool on = k + u < k1;
      const uint32_t i = on ? src[k + u] : j;
      lo[u] = off[i];
      hi[u] = on ? off[i + 1] : lo[u];
    }
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      static_assert(kMaxEdges == 128, "a list is two lanes' worth");
      v[u][0] = lo[u] + lane < hi[u] ? src[lo[u] + lane] : 0xFFFFFFFFu;
      v[u][1] = lo[u] + lane + 64u < hi[u] ? src[lo[u] + lane + 64u] : 0xFFFFFFFFu;
    }
    uint32_t w[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      const uint64_t b0 = __ballot(v[u][0] == j), b1 = __ballot(v[u][1] == j);
      w[u] = 0u;
      if (b0 | b1) {
        const uint32_t e = lo[u] + (b0 ? (uint32_t)__builtin_ctzll(b0)
                                       : 64u + (uint32_t)__builtin_ctzll(b1));
        w[u] = *(const uint32_t*)(x + (size_t)e * kWidth + 2 * lane);
      }
    }
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      a0 += from_bf16((uint16_t)(w[u] & 0xFFFFu));
      a1 += from_bf16((uint16_t)(w[u] >> 16));
    }
  }
  *(float2*)(out + (size_t)j * kWidth + 2 * lane) = make_float2(a0, a1);
}

// out[src[e]] += x[e] (atomics; 128 wide).
__global__ void k_scatter_rows(const uint16_t* __restrict__ x, const uint32_t* __restrict__ src,
                               size_t e, float* __restrict__ out) {
  size_t count = e * (kWidth / 2);
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x) {
    size_t ed = k / (kWidth / 2);
    int c = 2 * (int)(k % (kWidth / 2));
    uint32_t v = *(const uint32_t*)(x + ed * kWidth + c);
    float* o = out + (size_t)src[ed] * kWidth + c;
    atomicAdd(o, from_bf16((uint16_t)(v & 0xFFFFu)));
    atomicAdd(o + 1, from_bf16((uint16_t)(v >> 16)));
  }
}

// u1[:, 128:] = bf16([nu, 0...]) (the GEMM of M1 writes the first 128 of 144).
__global__ __launch_bounds__(256) void k_tail_u1(const float* __restrict__ nu, uint32_t n,
                                                 uint16_t* __restrict__ u1) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  u32x4* o = (u32x4*)(u1 + (size_t)i * kIn1 + kWidth);
  o[0] = u32x4{(uint32_t)to_bf16(nu[2 * i]) | ((uint32_t)to_bf16(nu[2 * i + 1]) << 16), 0u, 0u, 0u};
  o[1] = u32x4{0u, 0u, 0u, 0u};
}

// u2[:, :128] = H (the GEMM of M2 writes the second half of 256); eight
// features per thread.
__global__ __launch_bounds__(256) void k_head_u2(const uint16_t* __restrict__ Hb, uint32_t n,
                                                 uint16_t* __restrict__ u2) {
  const size_t k = blockIdx.x * (size_t)256 + threadIdx.x;
  if (k >= (size_t)n * (kWidth / 8)) return;
  const size_t i = k / (kWidth / 8), c = 8 * (k % (kWidth / 8));
  *(u32x4*)(u2 + i * kIn2 + c) = *(const u32x4*)(Hb + i * kWidth + c);
}

// Loss = sum over particles and the 3 used outputs of (out - target)^2 / n;
// dout = d loss / d out.
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ out,
                                              const float* __restrict__ target, uint32_t n,
                                              float* __restrict__ dout, float* __restrict__ loss) {
  __shared__ float red[4];
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  float l = 0.f;
  if (i < n) {
    for (int c = 0; c < kOut; ++c) {
      float d = c < 3 ? out[(size_t)i * kOut + c] - target[3 * (size_t)i + c] : 0.f;
      dout[(size_t)i * kOut + c] = 2.f * d / (float)n;
      l += d * d;
    }
  }
  for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(loss, (red[0] + red[1] + red[2] + red[3]) / (float)n);
}

__global__ void k_fill(float* __restrict__ x, size_t count, float v) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x)
    x[k] = v;
}

// Adam (Kingma & Ba 2015) with bias correction; refreshes the bf16 copy.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, size_t count, float lr, float b1, float b2,
                       float eps, float bc1, float bc2, uint16_t* __restrict__ wb) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x) {
    float gk = g[k];
    float mk = b1 * m[k] + (1.f - b1) * gk;
    float vk = b2 * v[k] + (1.f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    float pk = p[k] - lr * (mk / bc1) / (sqrtf(vk / bc2) + eps);
    p[k] = pk;
    wb[k] = to_bf16(pk);
  }
}

__global__ void k_cast(const float* __restrict__ x, uint16_t* __restrict__ y, size_t count) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < count;
       k += (size_t)gridDim.x * blockDim.x)
    y[k] = to_bf16(x[k]);
}

// acc[i] = g + A * out[i, 0:3]
__global__ void k_write_acc(const float* __restrict__ out, uint32_t n, float gx, float gy,
                            float gz, float4* __restrict__ acc) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float* o = out + (size_t)i * kOut;
  acc[i] = make_float4(gx + kAccScale * o[0], gy + kAccScale * o[1], gz + kAccScale * o[2], 0.f);
}

// ---------------------------------------------------------------------------
// Work-groups of a grid-stride kernel over `count` items.
inline dim3 grid_for(size_t count, size_t per_block = 256) {
  size_t b = (count + per_block - 1) / per_block;
  if (b > 65536) b = 65536;
  if (b == 0) b = 1;
  return dim3((uint32_t)b);
}

// Work-groups of a kernel whose threads take one item each, all of them.
inline dim3 grid_of_all(size_t count, size_t per_block = 256) {
  const size_t b = (count + per_block - 1) / per_block;
  return dim3((uint32_t)(b ? b : 1));
}

void fill(float* x, size_t count, float v, hipStream_t s) {
  if (count) hipLaunchKernelGGL(k_fill, grid_for(count), dim3(256), 0, s, x, count, v);
}

void launch_graph(clsph_gnn* m, clsph_state* st) {
  hipStream_t s = st->ctx->stream;
  uint32_t n = st->n;
  m->n = n;
  uint32_t chunks = (n + kScanChunk - 1) / kScanChunk;
  if (!chunks) chunks = 1;
  hipLaunchKernelGGL(k_scan_local, dim3(chunks), dim3(kScanBlock), 0, s, st->nbr_count, n, m->off,
                     m->scan_part);
  hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(kScanBlock), 0, s, m->scan_part, chunks,
                     m->off + n);
  hipLaunchKernelGGL(k_scan_add, grid_of_all(n), dim3(256), 0, s, m->off, m->scan_part, n);
}

void launch_edge_inputs(clsph_gnn* m, clsph_state* st) {
  hipStream_t s = st->ctx->stream;
  uint32_t n = m->n, e = m->e;
  const DevParams& d = st->host_dps[0];
  hipLaunchKernelGGL(k_graph, dim3(n ? (n + 255) / 256 : 1, 8), dim3(256), 0, s, st->nbr,
                     st->nbr_count, m->off, n, m->src, m->dst, m->degc);
  uint32_t cnt = e > n ? e : n;
  hipLaunchKernelGGL(k_edge_inputs, grid_of_all(cnt), dim3(256), 0, s, st->pos_s, st->vel_s,
                     st->rho_s, st->prs_s, m->src, m->dst, e, n, d.p.h, d.p.fluid_density,
                     d.p.K, m->E1, m->nu);
}

static inline const float* P(const clsph_gnn* m, int id) { return m->params + param_offset(id); }
static inline const uint16_t* W(const clsph_gnn* m, int id) { return m->wb + param_offset(id); }
static inline float* G(clsph_gnn* m, int id) { return m->grad + param_offset(id); }

// bf16(A B [+ rowscale bias]) into out16 (row stride ldo).
static void gemm_cast(hipStream_t s, const uint16_t* A, const uint16_t* B, uint16_t* out16, int ldo,
                      int M, const float* bias = nullptr, const float* rowscale = nullptr) {
  nn::GemmArgs g{};
  g.A = A, g.lda = kWidth, g.B = B, g.ldb = kWidth, g.out16 = out16, g.ldc = ldo;
  g.M = M, g.N = kWidth, g.K = kWidth, g.alpha = 1.f, g.bias = bias, g.rowscale = rowscale;
  gemm<false, false, nn::kEpiCast>(s, g);
}

// Second and third layer of an edge round: s1 -> z2 -> S = bf16(sum silu(z2) / C).
static void edge_tail(clsph_gnn* m, int r, int w2, int b2, hipStream_t s) {
  gemm(s, false, false, false, m->s1[r], kWidth, W(m, w2), kWidth, m->z2[r], kWidth, (int)m->e,
       kWidth, kWidth, 1.f, P(m, b2));
  hipLaunchKernelGGL(k_segsum_silu, dim3((m->n + 3) / 4), dim3(256), 0, s, m->z2[r], m->off,
                     m->n, 1.f / kAggC, m->S[r]);
}

// First two layers of a three-layer SiLU MLP over n rows: input u (bf16, kin
// wide) -> pre1/act1 -> pre2/act2.
static void mlp2(clsph_gnn* m, const uint16_t* u, int kin, int w1, float* pre1, uint16_t* act1,
                 float* pre2, uint16_t* act2, hipStream_t s) {
  int n = (int)m->n;
  gemm_silu(s, u, kin, W(m, w1), kWidth, P(m, w1 + 1), pre1, act1, n, kWidth, kin);
  gemm_silu(s, act1, kWidth, W(m, w1 + 2), kWidth, P(m, w1 + 3), pre2, act2, n, kWidth, kWidth);
}

// Node part of round 1: M1 from S[0], node MLP 1 -> H (bf16), and the
// round-2 node terms PA = bf16(H Wa), PB = bf16(H Wb).
static void node_round1(clsph_gnn* m, hipStream_t s) {
  int n = (int)m->n;
  gemm_cast(s, m->S[0], W(m, E1_W3), m->u1, kIn1, n, P(m, E1_B3), m->degc);
  hipLaunchKernelGGL(k_tail_u1, grid_of_all(n), dim3(256), 0, s, m->nu, m->n, m->u1);
  mlp2(m, m->u1, kIn1, N1_W1, m->p1, m->y1, m->p2, m->y2, s);
  gemm_cast(s, m->y2, W(m, N1_W3), m->Hb, kWidth, n, P(m, N1_B3));
  gemm_cast(s, m->Hb, W(m, E2_WA), m->PA, kWidth, n);
  gemm_cast(s, m->Hb, W(m, E2_WB), m->PB, kWidth, n);
}

// Node part of round 2: M2 from S[1], node MLP 2 -> out, accelerations.
static void node_round2(clsph_gnn* m, float4* acc, float gx, float gy, float gz, hipStream_t s) {
  int n = (int)m->n;
  gemm_cast(s, m->S[1], W(m, E2_W3), m->u2 + kWidth, kIn2, n, P(m, E2_B3), m->degc);
  hipLaunchKernelGGL(k_head_u2, grid_of_all((size_t)n * (kWidth / 8)), dim3(256), 0, s, m->Hb, m->n,
                     m->u2);
  mlp2(m, m->u2, kIn2, N2_W1, m->q1, m->w1, m->q2, m->w2, s);
  gemm(s, false, false, false, m->w2, kWidth, W(m, N2_W3), kOut, m->out, kOut, n, kOut, kWidth,
       1.f, P(m, N2_B3));
  if (acc)
    hipLaunchKernelGGL(k_write_acc, grid_of_all(n), dim3(256), 0, s, m->out, m->n, gx, gy, gz, acc);
}

void forward(clsph_gnn* m, const DevParams* dp, float4* acc, float gx, float gy, float gz) {
  (void)dp;
  hipStream_t s = m->ctx->stream;
  int e = (int)m->e;
  // round 1 edges
  gemm_silu(s, m->E1, kFeat, W(m, E1_W1), kWidth, P(m, E1_B1), m->z1[0], m->s1[0], e, kWidth,
            kFeat);
  edge_tail(m, 0, E1_W2, E1_B2, s);
  node_round1(m, s);
  // round 2 edges, with the node terms PA[dst] + PB[src]
  nn::GemmArgs g{};
  g.A = m->E1, g.lda = kFeat, g.B = W(m, E2_W1), g.ldb = kWidth, g.C = m->z1[1], g.ldc = kWidth;
  g.M = e, g.N = kWidth, g.K = kFeat, g.alpha = 1.f, g.bias = P(m, E2_B1);
  g.out16 = m->s1[1], g.row_add = m->PA, g.row_of = m->dst, g.row_add2 = m->PB, g.row_of2 = m->src;
  gemm<false, false, nn::kEpiEdgeSilu>(s, g);
  edge_tail(m, 1, E2_W2, E2_B2, s);
  node_round2(m, acc, gx, gy, gz, s);
}

void forward_fused(clsph_gnn* m, clsph_state* st, float4* acc, float gx, float gy, float gz,
                   hipEvent_t* ev) {
  hipStream_t s = m->ctx->stream;
  uint32_t n = st->n;
  m->n = n;
  const DevParams& d = st->host_dps[0];
  // persistent grid: the work-groups that fit at once (three per compute
  // unit at the kernels' register and LDS use) stage the weights once each
  uint32_t blocks = (uint32_t)st->ctx->cus * 3;
  if (blocks * 4 > n) blocks = (n + 3) / 4;
  if (blocks == 0) blocks = 1;
  if (ev) (void)hipEventRecord(ev[0], s);
  hipLaunchKernelGGL(k_node_inputs, grid_of_all(n), dim3(256), 0, s, st->rho_s, st->prs_s,
                     st->nbr_count, n, d.p.fluid_density, d.p.K, (float2*)m->nu, m->degc);
  hipLaunchKernelGGL((k_edge_fused<false>), dim3(blocks), dim3(256), 0, s, st->pos_s, st->vel_s,
                     (const float2*)m->nu, (const uint32_t*)st->nbr, st->nbr_count, n, d.p.h, W(m, E1_W1),
                     P(m, E1_B1), W(m, E1_W2), P(m, E1_B2), (const uint16_t*)nullptr,
                     (const uint16_t*)nullptr, m->S[0]);
  if (ev) (void)hipEventRecord(ev[1], s);
  // node part of round 1 (fused)
  constexpr size_t kLdsNode1 = (size_t)(8 * 4 + 8 * 5 + 8 * 4 + 8 * 4) * 64 * 16 + 4 * kWidth * 4;
  constexpr size_t kLdsTerms = (size_t)(8 * 4 + 8 * 4) * 64 * 16;
  constexpr size_t kLdsNode2 =
      (size_t)(8 * 4 + 8 * 8 + 8 * 4 + 2 * 4) * 64 * 16 + (3 * kWidth + kOut) * 4;
  static bool lds_set = false;
  if (!lds_set) {
    (void)hipFuncSetAttribute((const void*)k_node1, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kLdsNode1);
    (void)hipFuncSetAttribute((const void*)k_node_terms,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsTerms);
    (void)hipFuncSetAttribute((const void*)k_node2, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kLdsNode2);
    lds_set = true;
  }
  uint32_t tiles = (n + kNodeTile - 1) / kNodeTile;
  uint32_t nblocks = (uint32_t)st->ctx->cus;
  if (nblocks * 8 > tiles) nblocks = (tiles + 7) / 8;
  if (nblocks == 0) nblocks = 1;
  hipLaunchKernelGGL(k_node1, dim3(nblocks), dim3(512), kLdsNode1, s, m->S[0], m->degc, m->nu, n,
                     m->wb, m->params, m->Hb);
  hipLaunchKernelGGL(k_node_terms, dim3(nblocks), dim3(512), kLdsTerms, s, m->Hb, n, m->wb, m->PA,
                     m->PB);
  if (ev) (void)hipEventRecord(ev[2], s);
  hipLaunchKernelGGL((k_edge_fused<true>), dim3(blocks), dim3(256), 0, s, st->pos_s, st->vel_s,
                     (const float2*)m->nu, (const uint32_t*)st->nbr, st->nbr_count, n, d.p.h, W(m, E2_W1),
                     P(m, E2_B1), W(m, E2_W2), P(m, E2_B2), m->PA, m->PB, m->S[1]);
  if (ev) (void)hipEventRecord(ev[3], s);
  hipLaunchKernelGGL(k_node2, dim3(nblocks), dim3(512), kLdsNode2, s, m->S[1], m->Hb, m->degc, n,
                     m->wb, m->params, m->out, acc, gx, gy, gz);
  if (ev) (void)hipEventRecord(ev[4], s);
}

// Backward of a three-layer MLP given dy (f32, kout wide, in dY-compatible
// storage `dy` with stride ldy). Leaves d(input) in m->dY (f32, kin_used wide).
static void mlp3_back(clsph_gnn* m, int w1, const uint16_t* u, int kin, const float* pre1,
                      const uint16_t* act1, const float* pre2, const uint16_t* act2,
                      const uint16_t* dy_b, const float* dy, int ldy, int kout, int kin_used,
                      hipStream_t s) {
  int n = (int)m->n;
  // layer 3
  gemm(s, true, false, true, act2, kWidth, dy_b, kout, G(m, w1 + 4), kout, kWidth, kout, n, 1.f);
  colsum(s, dy, ldy, n, kout, nullptr, G(m, w1 + 5));
  gemm_dsilu(s, dy_b, kout, W(m, w1 + 4), kout, pre2, m->dpb, n, kWidth, kout);
  // layer 2; each work-group's rows of dpb are its own input and output
  gemm_weight_grad(s, act1, kWidth, m->dpb, kWidth, G(m, w1 + 2), G(m, w1 + 3), kWidth, kWidth, n);
  gemm_dsilu(s, m->dpb, kWidth, W(m, w1 + 2), kWidth, pre1, m->dpb, n, kWidth, kWidth);
  // layer 1
  gemm_weight_grad(s, u, kin, m->dpb, kWidth, G(m, w1), G(m, w1 + 1), kin, kWidth, n);
  gemm(s, false, true, false, m->dpb, kWidth, W(m, w1), kWidth, m->dY, kIn2, n, kin_used, kWidth,
       1.f);
}

// Backward of an edge round given dM (f32, stride ldm): gradients of W3/b3,
// W2/b2, W1/b1; leaves dz1 (bf16, e x 128) in m->dz1.
static void edge_back(clsph_gnn* m, int r, int w1, int w2, int w3, const float* dM, int ldm,
                      hipStream_t s) {
  int n = (int)m->n, e = (int)m->e;
  // bf16(dM) into dpb (n x 128)
  hipLaunchKernelGGL(k_cast_2d, grid_for((size_t)n * kWidth), dim3(256), 0, s, dM, ldm, m->dpb,
                     kWidth, (size_t)n, kWidth);
  gemm(s, true, false, true, m->S[r], kWidth, m->dpb, kWidth, G(m, w3), kWidth, kWidth, kWidth, n,
       1.f);
  colsum(s, dM, ldm, n, kWidth, m->degc, G(m, w3 + 1));
  gemm(s, false, true, false, m->dpb, kWidth, W(m, w3), kWidth, m->dS, kWidth, n, kWidth, kWidth,
       1.f / kAggC);
  // edges
  hipLaunchKernelGGL(k_edge_dz, grid_for((size_t)e * (kWidth / 8)), dim3(256), 0, s, m->dS,
                     m->z2[r], m->dst, m->dz2, (size_t)e);
  gemm_weight_grad(s, m->s1[r], kWidth, m->dz2, kWidth, G(m, w2), G(m, w2 + 1), kWidth, kWidth, e);
  gemm_dsilu(s, m->dz2, kWidth, W(m, w2), kWidth, m->z1[r], m->dz1, e, kWidth, kWidth);
  gemm_weight_grad(s, m->E1, kFeat, m->dz1, kWidth, G(m, w1), G(m, w1 + 1), kFeat, kWidth, e);
}

void backward(clsph_gnn* m) {
  hipStream_t s = m->ctx->stream;
  int n = (int)m->n;
  size_t nw = (size_t)n * kWidth;
  fill(m->grad, kParamTotal, 0.f, s);
  fill(m->loss, 1, 0.f, s);
  hipLaunchKernelGGL(k_loss, grid_of_all(n), dim3(256), 0, s, m->out, m->target, m->n, m->dout,
                     m->loss);
  // dpb (n x 256 bf16): the first half is mlp3_back's scratch, the second
  // half holds the bf16 gradient fed into it.
  uint16_t* dy_b = m->dpb + nw;
  hipLaunchKernelGGL(k_cast, grid_for((size_t)n * kOut), dim3(256), 0, s, m->dout, dy_b,
                     (size_t)n * kOut);
  // node MLP 2: dY (stride 256) = [d H | d M2]
  mlp3_back(m, N2_W1, m->u2, kIn2, m->q1, m->w1, m->q2, m->w2, dy_b, m->dout, kOut, kOut, kIn2,
            s);
  hipLaunchKernelGGL(k_copy_2d, grid_for(nw), dim3(256), 0, s, m->dY, kIn2, m->dH, kWidth,
                     (size_t)n, kWidth);
  // edge round 2 and its node terms
  edge_back(m, 1, E2_W1, E2_W2, E2_W3, m->dY + kWidth, kIn2, s);
  hipLaunchKernelGGL(k_segsum_rows, dim3((n + 3) / 4), dim3(256), 0, s, m->dz1, m->off, m->n,
                     m->dPA);
  if (!m->cut) {
    hipLaunchKernelGGL(k_gather_rows, dim3((m->n + 3) / 4), dim3(256), 0, s, m->dz1, m->off,
                       m->src, m->n, m->dPB);
  } else {
    fill(m->dPB, nw, 0.f, s);
    hipLaunchKernelGGL(k_scatter_rows, grid_for((size_t)m->e * (kWidth / 2)), dim3(256), 0, s,
                       m->dz1, m->src, (size_t)m->e, m->dPB);
  }
  hipLaunchKernelGGL(k_cast, grid_for(nw), dim3(256), 0, s, m->dPA, m->dPA_b, nw);
  hipLaunchKernelGGL(k_cast, grid_for(nw), dim3(256), 0, s, m->dPB, m->dPB_b, nw);
  gemm(s, true, false, true, m->Hb, kWidth, m->dPA_b, kWidth, G(m, E2_WA), kWidth, kWidth, kWidth,
       n, 1.f);
  gemm(s, true, false, true, m->Hb, kWidth, m->dPB_b, kWidth, G(m, E2_WB), kWidth, kWidth, kWidth,
       n, 1.f);
  gemm(s, false, true, true, m->dPA_b, kWidth, W(m, E2_WA), kWidth, m->dH, kWidth, n, kWidth,
       kWidth, 1.f);
  gemm(s, false, true, true, m->dPB_b, kWidth, W(m, E2_WB), kWidth, m->dH, kWidth, n, kWidth,
       kWidth, 1.f);
  // node MLP 1: dY[:, :128] = d M1
  hipLaunchKernelGGL(k_cast, grid_for(nw), dim3(256), 0, s, m->dH, dy_b, nw);
  mlp3_back(m, N1_W1, m->u1, kIn1, m->p1, m->y1, m->p2, m->y2, dy_b, m->dH, kWidth, kWidth,
            kWidth, s);
  // edge round 1
  edge_back(m, 0, E1_W1, E1_W2, E1_W3, m->dY, kIn2, s);
}

void adam(clsph_gnn* m, float lr, float beta1, float beta2, float eps) {
  m->adam_step += 1;
  float bc1 = 1.f - powf(beta1, (float)m->adam_step);
  float bc2 = 1.f - powf(beta2, (float)m->adam_step);
  hipLaunchKernelGGL(k_adam, grid_for(kParamTotal), dim3(256), 0, m->ctx->stream, m->params,
                     m->grad, m->adam_m, m->adam_v, (size_t)kParamTotal, lr, beta1, beta2, eps,
                     bc1, bc2, m->wb);
}

void cast_params(clsph_gnn* m) {
  hipLaunchKernelGGL(k_cast, grid_for(kParamTotal), dim3(256), 0, m->ctx->stream, m->params,
                     m->wb, (size_t)kParamTotal);
}

}  // namespace gnn
}  // namespace clsph
