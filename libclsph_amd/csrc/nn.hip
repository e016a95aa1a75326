// Kernels of the learned force surrogate (gfx950): a bf16 matrix-core GEMM
// with float32 accumulation, the neighbour-graph and edge-input builders,
// activation / aggregation / loss kernels and Adam. The forward and
// backward passes are sequences of these launches on the context stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "nn.h"

namespace clsph {
namespace nn {

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

// Eight floats to bf16 (round to nearest even), as one vector conversion so
// that each pair becomes one two-operand v_cvt_pk_bf16_f32.
typedef float f32x8 __attribute__((ext_vector_type(8)));

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
// GEMM: op(A) op(B) of bf16 operands, accumulated in f32. op(A) is M x K: A
// row-major M x K (lda), or with TA stored K x M. op(B) is K x N: B row-major
// K x N (ldb), or with TB stored N x K. Tiles of 128 x 128, K steps of 64
// through LDS (both operands as rows of K), four waves of 2 x 2 32x32x16 bf16
// matrix-core blocks. blockIdx.z splits K into chunks of k_chunk (a multiple
// of the step); with more than one chunk the epilogue adds. What becomes of
// the product v = alpha op(A) op(B) [+ rowscale[m] * bias[n]] is the epilogue
// (GemmArgs::epi). The contiguous dimension of each operand must be a
// multiple of 8 and 16-byte aligned (checked by the host wrapper).
//
// The shapes here are long and thin (edges x 128, or a 128 x 128 weight
// gradient over all edges), so a work-group does few steps and each is bound
// by the latency of its loads: a step's loads are issued before the previous
// step's products. An operand whose rows run across K is turned by 4 x 8
// blocks in registers (16 byte permutes) on its way to LDS.
constexpr int kTile = 128;
constexpr int kStep = 64;
// u16 per LDS row: 144 bytes put 16 rows' 16-byte reads on distinct banks
constexpr int kLds = kStep + 8;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// A 128 x 64 tile of an operand in flight: 64 bytes per thread.
template <bool ACROSS>  // the operand's rows run across K
struct TileLoad {
  u32x4 v[4];
  // row r0 + .. of `rows` (along M or N), K from k0 up to ke
  __device__ inline void load(const uint16_t* __restrict__ P, int ld, int r0, int rows, int k0,
                              int ke) {
    const int t = threadIdx.x;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int r = ACROSS ? r0 + (t >> 4) * 8 : r0 + (t >> 3) + 32 * it;
      const int k = ACROSS ? k0 + (t & 15) * 4 + it : k0 + (t & 7) * 8;
      v[it] = u32x4{0u, 0u, 0u, 0u};
      if (r < rows && k < ke)
        v[it] = *(const u32x4*)(P + (ACROSS ? (size_t)k * ld + r : (size_t)r * ld + k));
    }
  }
  __device__ inline void store(uint16_t* lds) const {
    const int t = threadIdx.x;
    if constexpr (!ACROSS) {
#pragma unroll
      for (int it = 0; it < 4; ++it)
        *(u32x4*)(lds + ((t >> 3) + 32 * it) * kLds + (t & 7) * 8) = v[it];
    } else {
      uint16_t* at = lds + (t >> 4) * 8 * kLds + (t & 15) * 4;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        // rows 2p and 2p + 1: the low and high halves of dword p of each k
        const uint2 lo = make_uint2(__builtin_amdgcn_perm(v[1][p], v[0][p], 0x05040100u),
                                    __builtin_amdgcn_perm(v[3][p], v[2][p], 0x05040100u));
        const uint2 hi = make_uint2(__builtin_amdgcn_perm(v[1][p], v[0][p], 0x07060302u),
                                    __builtin_amdgcn_perm(v[3][p], v[2][p], 0x07060302u));
        *(uint2*)(at + (2 * p) * kLds) = lo;
        *(uint2*)(at + (2 * p + 1) * kLds) = hi;
      }
    }
  }
};

template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t tiles[2 * kTile * kLds];
  uint16_t* As = tiles;
  uint16_t* Bs = tiles + kTile * kLds;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.x * kTile, n0 = blockIdx.y * kTile;
  const int kb = blockIdx.z * g.k_chunk;
  const int ke = min(g.K, kb + g.k_chunk);
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  f32x16 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j)
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  // column sums of B, in the first row of tiles' upper waves
  const bool sums = EPI == kEpiAdd && g.colsum != nullptr && blockIdx.x == 0 && wm == 0;
  float csum[2] = {0.f, 0.f};
  TileLoad<TA> la;
  TileLoad<!TB> lb;
  la.load(g.A, g.lda, m0, g.M, kb, ke);
  lb.load(g.B, g.ldb, n0, g.N, kb, ke);
  for (int k0 = kb; k0 < ke; k0 += kStep) {
    la.store(As);
    lb.store(Bs);
    __syncthreads();
    if (k0 + kStep < ke) {
      la.load(g.A, g.lda, m0, g.M, k0 + kStep, ke);
      lb.load(g.B, g.ldb, n0, g.N, k0 + kStep, ke);
    }
    for (int ks = 0; ks < kStep && k0 + ks < ke; ks += 16) {
      const int kk = ks + 8 * (lane >> 5);
      bf16x8 a[2], b[2];
      for (int i = 0; i < 2; ++i)
        a[i] = __builtin_bit_cast(bf16x8,
                                  *(const u32x4*)(As + (wm + 32 * i + (lane & 31)) * kLds + kk));
      for (int j = 0; j < 2; ++j)
        b[j] = __builtin_bit_cast(bf16x8,
                                  *(const u32x4*)(Bs + (wn + 32 * j + (lane & 31)) * kLds + kk));
      for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      if (EPI == kEpiAdd && sums) {
        const bf16x2 one = {(__bf16)1.f, (__bf16)1.f};
        for (int j = 0; j < 2; ++j)
          for (int q = 0; q < 4; ++q)
            csum[j] = __builtin_amdgcn_fdot2_f32_bf16(
                (bf16x2){b[j][2 * q], b[j][2 * q + 1]}, one, csum[j], false);
      }
    }
    __syncthreads();
  }
  if (EPI == kEpiAdd && sums)
    for (int j = 0; j < 2; ++j) {
      const float c = csum[j] + __shfl_xor(csum[j], 32, 64);
      const int col = n0 + wn + 32 * j + (lane & 31);
      if (lane < 32 && col < g.N) atomicAdd(g.colsum + col, c);
    }
  // D layout of the 32x32 block: register r of lane l holds
  // row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
  if constexpr (EPI == kEpiAdd || EPI == kEpiStore) {
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j)
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const int col = n0 + wn + 32 * j + (lane & 31);
          if (row < g.M && col < g.N) {
            float v = g.alpha * acc[i][j][r];
            if (g.bias && blockIdx.z == 0)
              v = __builtin_fmaf(g.bias[col], g.rowscale ? g.rowscale[row] : 1.f, v);
            float* at = g.C + (size_t)row * g.ldc + col;
            if constexpr (EPI == kEpiAdd) atomicAdd(at, v);
            else *at = v;
          }
        }
  } else {
    // The wave's 32 x 64 half turned through LDS, so that a lane has eight
    // consecutive columns and its reads and bf16 stores are 16 bytes (N a
    // multiple of 8). A 2-byte access per lane and register left these
    // epilogues waiting on their loads: over 557,000 edges the silu' one took
    // 196 us and the one with two gathered rows 255, now 78 and 98.
    constexpr int kPitch = 64 + 4;
    static_assert(4 * 32 * kPitch * sizeof(float) <= sizeof(tiles), "fits in the tiles' bytes");
    float* turn = reinterpret_cast<float*>(tiles) + wave * 32 * kPitch;
    for (int i = 0; i < 2; ++i) {
      wave_fence();
      for (int j = 0; j < 2; ++j)
        for (int r = 0; r < 16; ++r)
          turn[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kPitch + 32 * j + (lane & 31)] =
              acc[i][j][r];
      wave_fence();
      const int col = n0 + wn + (lane & 7) * 8;
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int lr = 8 * it + (lane >> 3), row = m0 + wm + 32 * i + lr;
        if (row >= g.M || col >= g.N) continue;
        const float* tv = turn + lr * kPitch + (lane & 7) * 8;
        float v[8];
        if (g.bias) {
          const float rs = g.rowscale ? g.rowscale[row] : 1.f;
          for (int q = 0; q < 8; ++q) v[q] = __builtin_fmaf(g.bias[col + q], rs, g.alpha * tv[q]);
        } else {
          for (int q = 0; q < 8; ++q) v[q] = g.alpha * tv[q];
        }
        const size_t at = (size_t)row * g.ldc + col;
        if constexpr (EPI == kEpiDsilu) {
          const float4 x = *(const float4*)(g.C + at), y = *(const float4*)(g.C + at + 4);
          const float pre[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
          for (int q = 0; q < 8; ++q) v[q] *= dsilu(pre[q]);
        }
        if constexpr (EPI == kEpiEdgeSilu) {
          const u32x4 x = *(const u32x4*)(g.row_add + (size_t)g.row_of[row] * g.ldc + col);
          const u32x4 y = *(const u32x4*)(g.row_add2 + (size_t)g.row_of2[row] * g.ldc + col);
          for (int q = 0; q < 8; ++q) {
            v[q] += from_bf16((uint16_t)(x[q >> 1] >> (16 * (q & 1))));
            v[q] += from_bf16((uint16_t)(y[q >> 1] >> (16 * (q & 1))));
          }
        }
        if constexpr (EPI == kEpiSilu || EPI == kEpiEdgeSilu) {
          *(float4*)(g.C + at) = make_float4(v[0], v[1], v[2], v[3]);
          *(float4*)(g.C + at + 4) = make_float4(v[4], v[5], v[6], v[7]);
          for (int q = 0; q < 8; ++q) v[q] = silu(v[q]);
        }
        *(u32x4*)(g.out16 + at) = pack8(v);
      }
    }
  }
}

// Fills the shape's split of K and launches. Adding products are split over K
// until about two work-groups per compute unit share it, 256 of K each at
// least: a weight gradient over 16,384 particles runs on 64 work-groups, not
// on 4 (311 -> 15 us), over 557,000 edges on 512, not on 136 (357 -> 55).
void gemm_launch(hipStream_t s, bool ta, bool tb, int epi, GemmArgs g) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return;
  const int mt = (g.M + kTile - 1) / kTile, nt = (g.N + kTile - 1) / kTile;
  int splits = 1;
  if (epi == kEpiAdd) {
    splits = 512 / (mt * nt);
    if (splits > g.K / 256) splits = g.K / 256;
    if (splits < 1) splits = 1;
  }
  int chunk = (g.K + splits - 1) / splits;
  chunk = (chunk + kStep - 1) / kStep * kStep;
  splits = (g.K + chunk - 1) / chunk;
  g.k_chunk = chunk;
  dim3 grid(mt, nt, splits);
#define GEMM_CASE(a, b, c)                                                   \
  if (ta == a && tb == b && epi == c) {                                      \
    hipLaunchKernelGGL((k_gemm<a, b, c>), grid, dim3(256), 0, s, g);         \
    return;                                                                  \
  }
  GEMM_CASE(false, false, kEpiStore) GEMM_CASE(false, false, kEpiAdd)
  GEMM_CASE(false, true, kEpiStore) GEMM_CASE(false, true, kEpiAdd)
  GEMM_CASE(true, false, kEpiStore) GEMM_CASE(true, false, kEpiAdd)
  GEMM_CASE(true, true, kEpiStore) GEMM_CASE(true, true, kEpiAdd)
  GEMM_CASE(false, false, kEpiSilu) GEMM_CASE(false, false, kEpiEdgeSilu)
  GEMM_CASE(false, false, kEpiCast) GEMM_CASE(false, true, kEpiDsilu)
#undef GEMM_CASE
}

// C = alpha op(A) op(B) [+ rowscale[m] * bias[n]], or added to C with `add`.
void gemm(hipStream_t s, bool ta, bool tb, bool add, const uint16_t* A, int lda,
          const uint16_t* B, int ldb, float* C, int ldc, int M, int N, int K, float alpha,
          const float* bias, const float* rowscale) {
  GemmArgs g{};
  g.A = A, g.lda = lda, g.B = B, g.ldb = ldb, g.C = C, g.ldc = ldc;
  g.M = M, g.N = N, g.K = K, g.alpha = alpha, g.bias = bias, g.rowscale = rowscale;
  gemm_launch(s, ta, tb, add ? kEpiAdd : kEpiStore, g);
}

// A weight gradient and its bias gradient: W (M x N) += A^T B, b (N) += the
// column sums of B; A is K x M, B is K x N.
void gemm_weight_grad(hipStream_t s, const uint16_t* A, int lda, const uint16_t* B, int ldb,
                      float* W, float* b, int M, int N, int K) {
  GemmArgs g{};
  g.A = A, g.lda = lda, g.B = B, g.ldb = ldb, g.C = W, g.ldc = N;
  g.M = M, g.N = N, g.K = K, g.alpha = 1.f, g.colsum = b;
  gemm<true, false, kEpiAdd>(s, g);
}

// Column sums (optionally row-weighted) of f32 rows, `cols` of them (a
// multiple of 4, at most 128), added into out: 256 rows per work-group, 16
// bytes per thread and row, joined through LDS.
__global__ __launch_bounds__(256) void k_colsum(const float* __restrict__ x, int ldx, int rows,
                                                int cols, const float* __restrict__ rowscale,
                                                float* __restrict__ out) {
  __shared__ float4 red[256];
  const int quads = cols / 4, per = 256 / quads;  // threads per row, rows in flight
  const int q = threadIdx.x % quads, r = threadIdx.x / quads;
  const int r0 = blockIdx.x * 256, r1 = min(r0 + 256, rows);
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  if (r < per) {
#pragma unroll 4
    for (int k = r0 + r; k < r1; k += per) {
      const float4 v = *(const float4*)(x + (size_t)k * ldx + 4 * q);
      const float w = rowscale ? rowscale[k] : 1.f;
      a.x += v.x * w, a.y += v.y * w, a.z += v.z * w, a.w += v.w * w;
    }
  }
  red[threadIdx.x] = a;
  __syncthreads();
  if (r == 0) {
    for (int k = 1; k < per; ++k) {
      const float4 v = red[k * quads + q];
      a.x += v.x, a.y += v.y, a.z += v.z, a.w += v.w;
    }
    atomicAdd(out + 4 * q, a.x);
    atomicAdd(out + 4 * q + 1, a.y);
    atomicAdd(out + 4 * q + 2, a.z);
    atomicAdd(out + 4 * q + 3, a.w);
  }
}

void colsum(hipStream_t s, const float* x, int ldx, int rows, int cols, const float* rowscale,
            float* out) {
  if (rows > 0)
    hipLaunchKernelGGL(k_colsum, dim3((rows + 255) / 256), dim3(256), 0, s, x, ldx, rows, cols,
                       rowscale, out);
}

// C = A B + bias and out16 = bf16(silu(C)).
void gemm_silu(hipStream_t s, const uint16_t* A, int lda, const uint16_t* B, int ldb,
               const float* bias, float* C, uint16_t* out16, int M, int N, int K) {
  GemmArgs g{};
  g.A = A, g.lda = lda, g.B = B, g.ldb = ldb, g.C = C, g.ldc = N, g.out16 = out16;
  g.M = M, g.N = N, g.K = K, g.alpha = 1.f, g.bias = bias;
  gemm<false, false, kEpiSilu>(s, g);
}

// out16 = bf16(A B^T silu'(pre)); out16 may be A itself when N fits one tile
// (a work-group's rows are then read by no other).
void gemm_dsilu(hipStream_t s, const uint16_t* A, int lda, const uint16_t* B, int ldb,
                const float* pre, uint16_t* out16, int M, int N, int K) {
  GemmArgs g{};
  g.A = A, g.lda = lda, g.B = B, g.ldb = ldb, g.C = const_cast<float*>(pre), g.ldc = N;
  g.out16 = out16;
  g.M = M, g.N = N, g.K = K, g.alpha = 1.f;
  gemm<false, true, kEpiDsilu>(s, g);
}

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
  for (int t = 0; t < kScanItems; ++t) {
    uint32_t i = base + t;
    v[t] = i < n ? min(count[i], kMaxEdges) : 0u;
    sum += v[t];
  }
  uint32_t total;
  uint32_t ex = block_scan_256(sum, lds, total);
  for (int t = 0; t < kScanItems; ++t) {
    uint32_t i = base + t;
    if (i < n) off[i] = ex;
    ex += v[t];
  }
  if (threadIdx.x == 0) part[blockIdx.x] = total;
}

// One work-group scans the chunk totals (any count) in place.
__global__ __launch_bounds__(kScanBlock) void k_scan_parts(uint32_t* __restrict__ part,
                                                           uint32_t nparts,
                                                           uint32_t* __restrict__ total_out) {
  __shared__ uint32_t lds[4];
  uint32_t carry = 0;
  for (uint32_t b = 0; b < nparts; b += kScanBlock) {
    uint32_t i = b + threadIdx.x;
    uint32_t v = i < nparts ? part[i] : 0u;
    uint32_t total;
    uint32_t ex = block_scan_256(v, lds, total);
    if (i < nparts) part[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) *total_out = carry;
}

__global__ __launch_bounds__(256) void k_scan_add(uint32_t* __restrict__ off,
                                                  const uint32_t* __restrict__ part, uint32_t n) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) off[i] += part[i / kScanChunk];
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

// Constants of the edge inputs (one scene).
struct EdgeConsts {
  float h, h2, inv_h, rho0, inv_rho0, K, m, mu_over_m, c_spiky, c_visc, c_grad, c_lap;
  // the edge inputs' constant factors, multiplied out once (edge_features)
  float kp, kv, kg, kl, kr, kd, kx;
};

inline EdgeConsts edge_consts(const DevParams& d) {
  EdgeConsts k;
  k.h = d.p.h;
  k.h2 = d.p.h * d.p.h;
  k.inv_h = 1.f / d.p.h;
  k.rho0 = d.p.fluid_density;
  k.inv_rho0 = 1.f / d.p.fluid_density;
  k.K = d.p.K;
  k.m = d.p.particle_mass;
  k.mu_over_m = d.p.dynamic_viscosity / d.p.particle_mass;
  k.c_spiky = d.t.spiky;
  k.c_visc = d.t.viscosity;
  k.c_grad = d.t.poly_6_gradient;
  k.c_lap = d.t.poly_6_laplacian;
  const double inv_a = 1.0 / kAccScale, inv_v = 1.0 / kVelScale, h = d.p.h;
  const double m = d.p.particle_mass;
  k.kp = (float)(-m * d.t.spiky * inv_a);
  k.kv = (float)((double)d.p.dynamic_viscosity / m * d.t.viscosity * inv_a);
  k.kg = (float)((double)d.t.poly_6_gradient * h);
  k.kl = (float)((double)d.t.poly_6_laplacian * h * h);
  k.kr = (float)(-m * d.t.spiky * h * inv_v * inv_a);
  k.kd = (float)(m * d.t.poly_6_gradient * 1000.0 * h * inv_v / (double)d.p.fluid_density);
  k.kx = (float)(10.0 * inv_v / h);
  return k;
}

// Constants of the forces stage (forces.cl:45-112, sph.cl:53-58) for the
// fused inference, which sums the listed neighbours' pair terms itself.
struct ForceTail {
  float h2, spiky0, mu, sigma, thresh, gx, gy, gz;
};

inline ForceTail force_tail(const DevParams& d) {
  ForceTail t;
  t.h2 = d.p.h * d.p.h;
  const float h3 = t.h2 * d.p.h;
  t.spiky0 = -45.f / (3.14159274f * (h3 * h3));  // coincident particles (smoothing.cl:23-25)
  t.mu = d.p.dynamic_viscosity;
  t.sigma = d.p.surface_tension;
  t.thresh = d.p.surface_tension_threshold;
  t.gx = d.p.constant_acceleration.s[0];
  t.gy = d.p.constant_acceleration.s[1];
  t.gz = d.p.constant_acceleration.s[2];
  return t;
}

// Pair sums of the forces stage for particle i: pressure (without the
// -rho_i factor), viscosity (without mu), colour-field gradient and
// laplacian, as the forces kernel accumulates them (forces.cl:60-101).
struct PairSums {
  float px, py, pz, vx, vy, vz, nx, ny, nz, lap;
};

__device__ __attribute__((always_inline)) inline void pair_terms(PairSums& f, const EdgeConsts& k,
                                                                 const ForceTail& ft, float4 ai,
                                                                 float4 bi, float4 aj, float4 bj,
                                                                 float w) {
  float dx = ai.x - aj.x, dy = ai.y - aj.y, dz = ai.z - aj.z;
  float d2 = dx * dx + dy * dy + dz * dz;
  float r = __builtin_amdgcn_sqrtf(d2);
  float t = k.h2 - d2;
  float hr = k.h - r;
  float ps = (aj.w + ai.w) * k.m;
  const bool coincident = r < 1e-7f;
  float g = coincident ? ps * ft.spiky0 : ps * k.c_spiky * hr * hr * __builtin_amdgcn_rcpf(r);
  g *= w;
  f.px += g * (coincident ? 1.f : dx);
  f.py += g * (coincident ? 1.f : dy);
  f.pz += g * (coincident ? 1.f : dz);
  float vw = bj.w * k.c_visc * hr * w;
  f.vx += (bj.x - bi.x) * vw;
  f.vy += (bj.y - bi.y) * vw;
  f.vz += (bj.z - bi.z) * vw;
  float gw = bj.w * k.c_grad * t * t * w;
  f.nx += gw * dx;
  f.ny += gw * dy;
  f.nz += gw * dz;
  f.lap += bj.w * k.c_lap * t * (3.f * k.h2 - 7.f * d2) * w;
}

// The 32 edge inputs of edge (i <- j) in float32 (27 used, 5 zero), from
// the density stage's per-particle force inputs a = (x, p / rho^2) and
// b = (v, m / rho) and the node inputs nu. The pair terms are the ones the
// forces stage sums (kernels/forces.cl:60-101): pressure and viscosity
// accelerations in units of A, the colour-field gradient term times h and
// its laplacian term times h^2. Then three rates along the pair's motion
// (x = x_i - x_j, v = v_i - v_j): the time derivative of the pressure pair
// acceleration at fixed pressures, -ps c_spiky [(h - r)^2 / r v -
// (x.v) (h - r)(h + r) / r^3 x], times h / (V A); the density-rate pair term
// m c_grad (h^2 - r^2)^2 (x.v) times 1000 h / (rho0 V); and x.v times
// 10 / (h V).
__device__ inline void edge_features(float4 ai, float4 bi, float4 aj, float4 bj, float2 ni,
                                     float2 nj, const EdgeConsts& k, float f[kFeat]) {
  static_assert(kVelScale == 1.f, "velocity inputs are taken unscaled");
  float dx = ai.x - aj.x, dy = ai.y - aj.y, dz = ai.z - aj.z;
  float d2 = dx * dx + dy * dy + dz * dz;
  float r = __builtin_amdgcn_sqrtf(d2);  // the forces kernel's square root
  float q = r * k.inv_h;
  float w = 1.f - q * q;
  const float vx = bi.x - bj.x, vy = bi.y - bj.y, vz = bi.z - bj.z;
  f[0] = dx * k.inv_h, f[1] = dy * k.inv_h, f[2] = dz * k.inv_h;
  f[3] = vx, f[4] = vy, f[5] = vz;
  f[6] = q, f[7] = w * w * w;
  f[8] = ni.x, f[9] = ni.y, f[10] = nj.x, f[11] = nj.y;
  const float hr = k.h - r, t = k.h2 - d2, t2 = t * t;
  const float ws = ai.w + aj.w;  // p_i / rho_i^2 + p_j / rho_j^2
  const bool apart = r >= 1e-7f;
  const float ir = __builtin_amdgcn_rcpf(r);
  // pressure pair acceleration / A: -(ws m c_spiky (h - r)^2 / r) x / A
  const float g = apart ? ws * k.kp * hr * hr * ir : 0.f;
  f[12] = g * dx, f[13] = g * dy, f[14] = g * dz;
  // viscosity pair acceleration / A: (v_j - v_i) (m / rho_j) (mu / rho_i) c_visc (h - r) / A
  const float vw = bi.w * k.kv * bj.w * hr;
  f[15] = -vx * vw, f[16] = -vy * vw, f[17] = -vz * vw;
  // colour-field gradient term times h, laplacian term times h^2
  const float gw = bj.w * k.kg * t2;
  f[18] = gw * dx, f[19] = gw * dy, f[20] = gw * dz;
  f[21] = bj.w * k.kl * t * (3.f * k.h2 - 7.f * d2);
  const float xv = dx * vx + dy * vy + dz * vz;
  float ra = 0.f, rb = 0.f;
  if (apart) {
    ra = hr * hr * ir;
    rb = xv * hr * (k.h + r) * (ir * ir * ir);
  }
  const float cr = ws * k.kr;
  f[22] = cr * (ra * vx - rb * dx), f[23] = cr * (ra * vy - rb * dy);
  f[24] = cr * (ra * vz - rb * dz);
  f[25] = t2 * xv * k.kd;
  f[26] = xv * k.kx;
  for (int c = kFeatUsed; c < kFeat; ++c) f[c] = 0.f;
}

// nu_i = [rho_i / rho0 - 1, asinh(p_i / K) / 4] for every particle.
__global__ void k_node_inputs(const float* __restrict__ rho, const float* __restrict__ prs,
                              uint32_t n, float rho0, float K, float2* __restrict__ nu) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) nu[i] = node_in(rho[i], prs[i], rho0, K);
}

// Edge inputs e (32 bf16 per edge), after k_node_inputs.
__global__ __launch_bounds__(256) void k_edge_inputs(
    const float4* __restrict__ fab, const float2* __restrict__ nu,
    const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst, uint32_t e,
    EdgeConsts kc, uint16_t* __restrict__ E1) {
  for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < e; k += gridDim.x * 256) {
    uint32_t i = dst[k], j = src[k];
    float f[kFeat];
    edge_features(fab[2u * i], fab[2u * i + 1u], fab[2u * j], fab[2u * j + 1u], nu[i], nu[j],
                  kc, f);
    u32x4* o = (u32x4*)(E1 + (size_t)k * kFeat);
    for (int q = 0; q < kFeat / 8; ++q) {
      uint32_t packed[4];
      for (int t = 0; t < 4; ++t)
        packed[t] = (uint32_t)to_bf16(f[8 * q + 2 * t]) |
                    ((uint32_t)to_bf16(f[8 * q + 2 * t + 1]) << 16);
      o[q] = u32x4{packed[0], packed[1], packed[2], packed[3]};
    }
  }
}

// ---------------------------------------------------------------------------
// Fused inference: one kernel walks the density stage's neighbour lists and
// evaluates the whole network.
//
// A wave owns tiles of 16 consecutive sorted particles; lane l serves
// particle c = l % 16 of the tile in lane group g = l / 16. The edge layer
// runs transposed on 16x16x32 bf16 matrix cores, z^T = W1^T e^T, with the
// tile's particles as the 16 columns: at step s, column c holds particle c's
// s-th neighbour edge, so each lane's accumulator sums its own particle's
// edges in list order and the neighbour sum needs no cross-lane reduction.
// A lane holds z for hidden units 16 ob + 4 g + r (r = 0..3) of its column.
//
// Edge inputs are computed once per edge. In each round of 4 steps, lane
// (g, c) computes the inputs of particle c's edge 4 k + g and stores its 32
// inputs as bf16 in the wave's LDS block; the B operand of step 4 k + s for
// lane (g, c) is inputs 8 g .. 8 g + 7 of edge 4 k + s of particle c. Per
// particle column the block holds 4 edges x 64 bytes plus 16 bytes of
// padding: 272 bytes = 68 dwords, so the 16 columns of one read start on 16
// distinct multiples of 4 banks.
//
// The node MLP follows in registers: the neighbour sums are the B operand of
// node layer 1 in the permuted K order (slot t of lane group g is feature
// 16 (t / 4) + 4 g + t % 4 of a 32-wide block), node inputs 32..63 come in
// the natural order (slot t of group g is feature 32 + 8 g + t), and each
// later layer takes its B operand from the previous layer's registers in the
// permuted order. Weights are staged once per work-group in LDS in the
// matching orders.
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileP = 16;                 // particles per tile (MFMA columns)
constexpr int kSurWaves = 8;               // waves per work-group
constexpr int kColBytes = 4 * 64 + 16;     // LDS bytes per particle column
constexpr int kWaveLds = kTileP * kColBytes;

// Stages W (row-major, rows = inputs, ld = outputs) for k-steps
// [ks0, ks0 + nks) of a layer with `ks_total` k-steps and `nob` 16-wide
// output blocks: dst[(ob * ks_total + ks) * 64 + lane] holds the lane's 8 K
// slots of W^T row 16 ob + lane % 16, natural or permuted K order; input
// rows at or beyond `kvalid` are zero. `krow0` is the W row of k-step ks0.
__device__ __attribute__((always_inline)) inline void stage_layer(
    u32x4* dst, int ks_total, int ks0, int nks, int nob, const uint16_t* __restrict__ Wm, int ld,
    int krow0, int kvalid, bool perm) {
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
__device__ __attribute__((always_inline)) inline void mfma_layer(const u32x4* __restrict__ w,
                                                                 const bf16x8* bop,
                                                                 const float* __restrict__ bias,
                                                                 f32x4* y) {
  const int lane = threadIdx.x & 63, g = lane >> 4;
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob) {
    f32x4 a;
    for (int r = 0; r < 4; ++r) a[r] = bias[16 * ob + 4 * g + r];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, w[(ob * NKS + ks) * 64 + lane]), bop[ks], a, 0, 0, 0);
    y[ob] = a;
  }
}

// Permuted-order B operands (NOB / 2 k-steps) from a layer's registers,
// through SiLU.
template <int NOB>
__device__ __attribute__((always_inline)) inline void silu_operands(const f32x4* y, bf16x8* bop) {
#pragma unroll
  for (int ks = 0; ks < NOB / 2; ++ks) {
    float v8[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) v8[t] = silu(y[2 * ks + (t >> 2)][t & 3]);
    bop[ks] = __builtin_bit_cast(bf16x8, pack8(v8));
  }
}

// The neighbour of lane (g, c) in round k: edge 4 k + g of particle c (the
// particle itself when that edge is past its degree).
__device__ __attribute__((always_inline)) inline uint32_t edge_index(
    uint32_t k, uint32_t i, uint32_t n, uint32_t deg, const uint4* __restrict__ nbr) {
  const int g = (threadIdx.x & 63) >> 4;
  uint32_t j = i;
  if (4 * k + g < deg) {
    uint4 js = nbr[(size_t)k * n + i];
    j = g == 0 ? js.x : g == 1 ? js.y : g == 2 ? js.z : js.w;
  }
  return j;
}

struct EdgeFetch {
  float4 a, b;
  float2 nu;
  bool mine;
};

// The inputs of neighbour j, lane (g, c)'s edge of round k.
__device__ __attribute__((always_inline)) inline EdgeFetch fetch_edge(
    uint32_t k, uint32_t j, uint32_t deg, const float4* __restrict__ fab,
    const float2* __restrict__ nu) {
  const int g = (threadIdx.x & 63) >> 4;
  EdgeFetch e;
  e.mine = 4 * k + g < deg;
  e.a = fab[2u * j];
  e.b = fab[2u * j + 1u];
  e.nu = nu[j];
  return e;
}

// One round of 4 edge steps for the wave's tile (see above). MASKED rounds
// contain edges past some column's degree: those edges store zero inputs and
// their steps start from a zero accumulator, so they add relu(0) = 0.
template <bool MASKED, bool OWN>
__device__ __attribute__((always_inline)) inline void edge_round(
    uint32_t k, uint32_t deg, const float4& ai, const float4& bi, const float2& ni,
    const EdgeFetch& ej, const EdgeConsts& kc, const ForceTail& ft, uint8_t* wlds,
    const u32x4* __restrict__ w1s, const f32x4* zb, f32x4* s, PairSums& ps) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  if (OWN) pair_terms(ps, kc, ft, ai, bi, ej.a, ej.b, (MASKED && !ej.mine) ? 0.f : 1.f);
  float f[kFeat];
  edge_features(ai, bi, ej.a, ej.b, ni, ej.nu, kc, f);
  uint8_t* col = wlds + c * kColBytes;
  for (int q = 0; q < 4; ++q) {
    u32x4 v = pack8(f + 8 * q);
    if (MASKED && !ej.mine) v = u32x4{0u, 0u, 0u, 0u};
    *(u32x4*)(col + g * 64 + 16 * q) = v;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    const bf16x8 eb = __builtin_bit_cast(bf16x8, *(const u32x4*)(col + st * 64 + g * 16));
    const bool live = !MASKED || 4 * k + st < deg;
#pragma unroll
    for (int ob = 0; ob < kEdgeW / 16; ++ob) {
      f32x4 c0 = zb[ob];
      if (MASKED && !live) c0 = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, w1s[ob * 64 + lane]), eb, c0, 0, 0, 0);
      // s + relu(z) as max(s + z, s): the same value and rounding, and the
      // operands of the max are canonical (one instruction, not two)
      for (int r = 0; r < 4; ++r) s[ob][r] = fmaxf(s[ob][r] + z[r], s[ob][r]);
    }
  }
  // the next round's stores come after this round's reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// OWN: the forces stage's acceleration a0 is summed here from the listed
// neighbours (particles whose list overflowed take acc[i], which the
// forces kernel wrote for them); otherwise a0 = acc[i].
template <bool OWN>
__global__ __launch_bounds__(kSurWaves * 64) void k_surrogate(
    const float4* __restrict__ fab, const float2* __restrict__ nu,
    const float* __restrict__ rho, const uint4* __restrict__ nbr,
    const uint32_t* __restrict__ count, uint32_t n, EdgeConsts kc, ForceTail ft,
    const uint16_t* __restrict__ wb, const float* __restrict__ params, float4* __restrict__ acc,
    float* __restrict__ out) {
  const float gx = ft.gx, gy = ft.gy, gz = ft.gz;
  __shared__ u32x4 w1s[2 * 64];          // edge layer: 2 output blocks, 1 k-step
  __shared__ u32x4 wn1[4 * 2 * 64];      // node layer 1: k-step 0 permuted, 1 natural
  __shared__ u32x4 wn2[4 * 2 * 64];
  __shared__ u32x4 wn3[2 * 2 * 64];
  __shared__ float bias[kEdgeW + 2 * kNodeW + kOut];
  __shared__ __attribute__((aligned(16))) uint8_t tiles_lds[kSurWaves * kWaveLds];
  stage_layer(w1s, 1, 0, 1, 2, wb + param_offset(E_W1), kEdgeW, 0, kFeatUsed, false);
  stage_layer(wn1, 2, 0, 1, 4, wb + param_offset(N_W1), kNodeW, 0, kEdgeW, true);
  stage_layer(wn1, 2, 1, 1, 4, wb + param_offset(N_W1), kNodeW, kEdgeW, kEdgeW + 6, false);
  stage_layer(wn2, 2, 0, 2, 4, wb + param_offset(N_W2), kNodeW, 0, kNodeW, true);
  stage_layer(wn3, 2, 0, 2, 2, wb + param_offset(N_W3), kOut, 0, kNodeW, true);
  for (int k = threadIdx.x; k < kEdgeW + 2 * kNodeW + kOut; k += blockDim.x) {
    float v;
    if (k < kEdgeW) v = params[param_offset(E_B1) + k];
    else if (k < kEdgeW + kNodeW) v = params[param_offset(N_B1) + k - kEdgeW];
    else if (k < kEdgeW + 2 * kNodeW) v = params[param_offset(N_B2) + k - kEdgeW - kNodeW];
    else v = params[param_offset(N_B3) + k - kEdgeW - 2 * kNodeW];
    bias[k] = v;
  }
  __syncthreads();

  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, wave = threadIdx.x >> 6;
  uint8_t* wlds = tiles_lds + wave * kWaveLds;
  f32x4 zb[2];
  for (int ob = 0; ob < 2; ++ob)
    for (int r = 0; r < 4; ++r) zb[ob][r] = bias[16 * ob + 4 * g + r];
  const uint32_t waves = gridDim.x * kSurWaves;
  const uint32_t ntiles = (n + kTileP - 1) / kTileP;
  for (uint32_t tile = blockIdx.x * kSurWaves + wave; tile < ntiles; tile += waves) {
    const uint32_t ip = tile * kTileP + c;
    const bool valid = ip < n;
    const uint32_t i = valid ? ip : n - 1;
    const uint32_t deg = valid ? min(count[i], kMaxEdges) : 0u;
    uint32_t dmin = deg, dmax = deg;
    for (int o = 1; o < 16; o <<= 1) {
      dmin = min(dmin, (uint32_t)__shfl_xor((int)dmin, o, 64));
      dmax = max(dmax, (uint32_t)__shfl_xor((int)dmax, o, 64));
    }
    const uint32_t cnt = valid ? count[i] : 0u;
    const float4 ai = fab[2u * i], bi = fab[2u * i + 1u];
    const float2 ni = nu[i];
    f32x4 s[2];
    for (int ob = 0; ob < 2; ++ob) s[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
    PairSums ps = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // rounds inside every column's degree, then the masked tail; each
    // round's neighbour inputs are fetched one round ahead
    const uint32_t kfull = dmin >> 2, kend = (dmax + 3) >> 2;
    // neighbour indices are loaded two rounds ahead, so that a round's
    // gathers never wait for the index load that names them
    EdgeFetch cur;
    if (kend) cur = fetch_edge(0, edge_index(0, i, n, deg, nbr), deg, fab, nu);
    uint32_t jn = kend > 1 ? edge_index(1, i, n, deg, nbr) : i;
    for (uint32_t k = 0; k < kend; ++k) {
      EdgeFetch nxt = cur;
      if (k + 1 < kend) nxt = fetch_edge(k + 1, jn, deg, fab, nu);
      if (k + 2 < kend) jn = edge_index(k + 2, i, n, deg, nbr);
      if (k < kfull)
        edge_round<false, OWN>(k, deg, ai, bi, ni, cur, kc, ft, wlds, w1s, zb, s, ps);
      else
        edge_round<true, OWN>(k, deg, ai, bi, ni, cur, kc, ft, wlds, w1s, zb, s, ps);
      cur = nxt;
    }
    float4 a0;
    if (OWN) {
      // the four lane groups hold interleaved edges of the same particle
      auto group_sum = [](float& v) {
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
      };
      group_sum(ps.px), group_sum(ps.py), group_sum(ps.pz);
      group_sum(ps.vx), group_sum(ps.vy), group_sum(ps.vz);
      group_sum(ps.nx), group_sum(ps.ny), group_sum(ps.nz);
      group_sum(ps.lap);
      // the forces kernel's closing formula (forces.cl:95-111, sph.cl:53-58),
      // with the colour-field laplacian's self term
      const float rho_i = rho[i];
      const float lap = bi.w * kc.c_lap * ft.h2 * (3.f * ft.h2) + ps.lap;
      float fx = -rho_i * ps.px + ps.vx * ft.mu;
      float fy = -rho_i * ps.py + ps.vy * ft.mu;
      float fz = -rho_i * ps.pz + ps.vz * ft.mu;
      const float nl = sqrtf(ps.nx * ps.nx + ps.ny * ps.ny + ps.nz * ps.nz);
      if (nl > ft.thresh) {
        const float kk = -ft.sigma * lap / nl;
        fx += kk * ps.nx;
        fy += kk * ps.ny;
        fz += kk * ps.nz;
      }
      a0 = make_float4(fx / rho_i + gx, fy / rho_i + gy, fz / rho_i + gz, 0.f);
      if (cnt > kMaxEdges) a0 = acc[i];
    } else {
      a0 = acc[i];
    }

    // node layer 1: [S, nu, (a0 - g) / A, deg / C, 0...]
    bf16x8 bop[2];
    {
      float v8[8];
      for (int t = 0; t < 8; ++t) v8[t] = s[t >> 2][t & 3] * (1.f / kAggC);
      bop[0] = __builtin_bit_cast(bf16x8, pack8(v8));
      for (int t = 0; t < 8; ++t) v8[t] = 0.f;
      if (g == 0) {
        constexpr float inv_a = 1.f / kAccScale;
        v8[0] = ni.x, v8[1] = ni.y;
        v8[2] = (a0.x - gx) * inv_a, v8[3] = (a0.y - gy) * inv_a, v8[4] = (a0.z - gz) * inv_a;
        v8[5] = (float)deg * (1.f / kAggC);
      }
      bop[1] = __builtin_bit_cast(bf16x8, pack8(v8));
    }
    f32x4 y[4];
    mfma_layer<4, 2>(wn1, bop, bias + kEdgeW, y);
    silu_operands<4>(y, bop);
    mfma_layer<4, 2>(wn2, bop, bias + kEdgeW + kNodeW, y);
    silu_operands<4>(y, bop);
    f32x4 o[2];
    mfma_layer<2, 2>(wn3, bop, bias + kEdgeW + 2 * kNodeW, o);
    if (valid) {
      if (out) {
        float* orow = out + (size_t)i * kOut;
        for (int ob = 0; ob < 2; ++ob)
          *(float4*)(orow + 16 * ob + 4 * g) = make_float4(o[ob][0], o[ob][1], o[ob][2], o[ob][3]);
      }
      if (g == 0)
        acc[i] = make_float4(a0.x + kResScale * o[0][0], a0.y + kResScale * o[0][1],
                             a0.z + kResScale * o[0][2], a0.w);
    }
  }
}

// ---------------------------------------------------------------------------
// Training-path kernels (grid-stride loops unless noted).
// The edge layer of the training forward pass and its neighbour sum:
// z = e W1 + b1, S[i] = bf16(sum over i's edges of relu(z) / C), and for the
// backward pass one bit per (edge, feature), z > 0. A work-group takes
// kEdgeParts consecutive particles, whose edges are consecutive; 128 at a
// time pass through the matrix cores into LDS, where 32 threads per particle
// (one per feature) sum them in order. Reads the 64 bytes of each edge's
// inputs and writes 4 (storing z and summing it in a second pass had moved
// 64 + 128 + 128): 120 us for 5 million edges, 688 as the two passes.
constexpr uint32_t kEdgeParts = 32;
__global__ __launch_bounds__(256) void k_edge_layer(const uint16_t* __restrict__ E1,
                                                    const uint16_t* __restrict__ W1,
                                                    const float* __restrict__ b1,
                                                    const uint32_t* __restrict__ off, uint32_t n,
                                                    uint16_t* __restrict__ S,
                                                    uint32_t* __restrict__ mask) {
  static_assert(kEdgeW == 32 && kFeat == 32, "one 32x32 block per 32 edges");
  constexpr uint32_t kChunk = 128;
  __shared__ float zs[kChunk][kEdgeW + 1];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, col = lane & 31u, half = lane >> 5;
  const uint32_t i0 = blockIdx.x * kEdgeParts, i1 = min(n, i0 + kEdgeParts);
  const uint32_t e0 = off[i0], e1 = off[i1];
  // W1's operands (k-steps of 16, lane: column `col`, 8 inputs from 8 half)
  bf16x8 w[2];
  for (int ks = 0; ks < 2; ++ks) {
    uint32_t d[4];
    for (int q = 0; q < 4; ++q) {
      const uint32_t k = 16 * ks + 8 * half + 2 * q;
      d[q] = (uint32_t)W1[k * kEdgeW + col] | ((uint32_t)W1[(k + 1) * kEdgeW + col] << 16);
    }
    w[ks] = __builtin_bit_cast(bf16x8, u32x4{d[0], d[1], d[2], d[3]});
  }
  const float bias = b1[col];
  // particle i0 + p is summed by the threads of group p % 8
  const uint32_t grp = t >> 5, c = t & 31u;
  uint32_t pe0[kEdgeParts / 8], pe1[kEdgeParts / 8];
  float sum[kEdgeParts / 8];
#pragma unroll
  for (uint32_t q = 0; q < kEdgeParts / 8; ++q) {
    const uint32_t i = i0 + 8 * q + grp;
    pe0[q] = i < i1 ? off[i] : 0u;
    pe1[q] = i < i1 ? off[i + 1] : 0u;
    sum[q] = 0.f;
  }
  for (uint32_t c0 = e0; c0 < e1; c0 += kChunk) {
    const uint32_t er = c0 + 32 * wave + col;
    bf16x8 a[2];
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (er < e1) v = *(const u32x4*)(E1 + (size_t)er * kFeat + 16 * ks + 8 * half);
      a[ks] = __builtin_bit_cast(bf16x8, v);
    }
    f32x16 z;
    for (int r = 0; r < 16; ++r) z[r] = 0.f;
    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], w[0], z, 0, 0, 0);
    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], w[1], z, 0, 0, 0);
    // register r: edge 8 (r / 4) + 4 half + r % 4 of the wave's 32, feature col
    uint32_t bits = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t row = 8 * (r >> 2) + (r & 3);
      const float v = z[r] + bias;
      const uint64_t on = __ballot(v > 0.f);
      bits = col == row ? (uint32_t)on : (col == row + 4u ? (uint32_t)(on >> 32) : bits);
      zs[32 * wave + row + 4 * half][col] = fmaxf(v, 0.f);
    }
    if (half == 0u && er < e1) mask[er] = bits;
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kEdgeParts / 8; ++q) {
      const uint32_t k0 = max(pe0[q], c0), k1 = min(pe1[q], c0 + kChunk);
      for (uint32_t k = k0; k < k1; ++k) sum[q] += zs[k - c0][c];
    }
    __syncthreads();
  }
#pragma unroll
  for (uint32_t q = 0; q < kEdgeParts / 8; ++q) {
    const uint32_t i = i0 + 8 * q + grp;
    if (i < i1) S[(size_t)i * kEdgeW + c] = to_bf16(sum[q] * (1.f / kAggC));
  }
}

// The edge layer's gradients from d loss / d S (dY, row stride ldy):
// dz[e] = bf16(dY[dst[e]] / C) where the forward pass found z > 0, else 0;
// W += E1^T dz, b += the column sums of dz. A work-group takes `per`
// consecutive edges, 256 at a time: both operands are turned in registers
// into LDS rows of edges, and each wave multiplies a quarter of them. 193 us
// for 5 million edges; as three passes (dz, the product, the column sums) 945.
__global__ __launch_bounds__(256) void k_edge_grad(const uint16_t* __restrict__ E1,
                                                   const float* __restrict__ dY, int ldy,
                                                   const uint32_t* __restrict__ mask,
                                                   const uint32_t* __restrict__ dst, uint32_t e,
                                                   uint32_t per, float* __restrict__ W,
                                                   float* __restrict__ b) {
  static_assert(kEdgeW == 32 && kFeat == 32, "one 32x32 block");
  constexpr int kRow = 256 + 8;  // u16 per LDS row of edges
  __shared__ __attribute__((aligned(16))) uint16_t As[32 * kRow];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[32 * kRow];
  __shared__ float red[3][32][33];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t b0 = blockIdx.x * per, b1 = min(e, b0 + per);
  const uint32_t eq = (t >> 2) * 4u, f = (t & 3u) * 8u;  // 4 edges x 8 features per thread
  f32x16 acc;
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  float csum = 0.f;
  for (uint32_t c0 = b0; c0 < b1; c0 += 256u) {
    u32x4 va[4], vb[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t ed = c0 + eq + u;
      va[u] = vb[u] = u32x4{0u, 0u, 0u, 0u};
      if (ed < b1) {
        va[u] = *(const u32x4*)(E1 + (size_t)ed * kFeat + f);
        const float4* dp = (const float4*)(dY + (size_t)dst[ed] * ldy + f);
        const float4 x = dp[0], y = dp[1];
        const float d[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
        const uint32_t m = mask[ed] >> f;
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = (m >> q) & 1u ? d[q] * (1.f / kAggC) : 0.f;
        vb[u] = pack8(v);
      }
    }
    __syncthreads();  // the previous products have read LDS
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      uint16_t* ta = As + (f + 2 * p) * kRow + eq;
      uint16_t* tb = Bs + (f + 2 * p) * kRow + eq;
      *(uint2*)ta = make_uint2(__builtin_amdgcn_perm(va[1][p], va[0][p], 0x05040100u),
                               __builtin_amdgcn_perm(va[3][p], va[2][p], 0x05040100u));
      *(uint2*)(ta + kRow) = make_uint2(__builtin_amdgcn_perm(va[1][p], va[0][p], 0x07060302u),
                                        __builtin_amdgcn_perm(va[3][p], va[2][p], 0x07060302u));
      *(uint2*)tb = make_uint2(__builtin_amdgcn_perm(vb[1][p], vb[0][p], 0x05040100u),
                               __builtin_amdgcn_perm(vb[3][p], vb[2][p], 0x05040100u));
      *(uint2*)(tb + kRow) = make_uint2(__builtin_amdgcn_perm(vb[1][p], vb[0][p], 0x07060302u),
                                        __builtin_amdgcn_perm(vb[3][p], vb[2][p], 0x07060302u));
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 64; ks += 16) {
      const uint32_t at = (lane & 31u) * kRow + 64u * wave + ks + 8u * (lane >> 5);
      const bf16x8 a = __builtin_bit_cast(bf16x8, *(const u32x4*)(As + at));
      const bf16x8 bb = __builtin_bit_cast(bf16x8, *(const u32x4*)(Bs + at));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bb, acc, 0, 0, 0);
      const bf16x2 one = {(__bf16)1.f, (__bf16)1.f};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        csum = __builtin_amdgcn_fdot2_f32_bf16((bf16x2){bb[2 * q], bb[2 * q + 1]}, one, csum, false);
    }
  }
  csum += __shfl_xor(csum, 32, 64);
  if (lane < 32u) atomicAdd(b + lane, csum);
  if (wave)
    for (int r = 0; r < 16; ++r)
      red[wave - 1][8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)][lane & 31u] = acc[r];
  __syncthreads();
  if (wave == 0)
    for (int r = 0; r < 16; ++r) {
      const uint32_t row = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), cc = lane & 31u;
      atomicAdd(W + row * kEdgeW + cc, acc[r] + red[0][row][cc] + red[1][row][cc] + red[2][row][cc]);
    }
}

// u = bf16([S, nu, (a0 - g) / A, deg / C, 0...]) (64 wide), eight values per
// thread.
__global__ __launch_bounds__(256) void k_pack_u(const uint16_t* __restrict__ S,
                                                const float* __restrict__ nu,
                                                const float4* __restrict__ acc0,
                                                const float* __restrict__ degc, uint32_t n,
                                                float gx, float gy, float gz,
                                                uint16_t* __restrict__ u) {
  const size_t k = blockIdx.x * (size_t)256 + threadIdx.x;
  if (k >= (size_t)n * (kIn / 8)) return;
  const size_t i = k / (kIn / 8), c = 8 * (k % (kIn / 8));
  u32x4 v = {0u, 0u, 0u, 0u};
  if (c < kEdgeW) {
    v = *(const u32x4*)(S + i * kEdgeW + c);
  } else if (c == kEdgeW) {
    const float4 a = acc0[i];
    const float x[8] = {nu[2 * i], nu[2 * i + 1], (a.x - gx) * (1.f / kAccScale),
                        (a.y - gy) * (1.f / kAccScale), (a.z - gz) * (1.f / kAccScale), degc[i],
                        0.f, 0.f};
    v = pack8(x);
  }
  *(u32x4*)(u + i * kIn + c) = v;
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

// loc[ids[k]] = k
__global__ void k_invert(const uint32_t* __restrict__ ids, uint32_t n, uint32_t* __restrict__ loc) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) {
    uint32_t id = ids[k];
    if (id < n) loc[id] = k;
  }
}

// target[i] = ((vh_T - vh_S) / dt - a0_i) / R for the learner's sorted i.
__global__ void k_target(const uint32_t* __restrict__ perm, const float4* __restrict__ vh_s,
                         const uint32_t* __restrict__ loc, const float4* __restrict__ vh_t,
                         const float4* __restrict__ acc0, uint32_t n, float inv_dt,
                         float* __restrict__ target) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint32_t c = perm[i];
  float4 a = vh_s[c], b = vh_t[loc[c]], a0 = acc0[i];
  target[3 * i] = ((b.x - a.x) * inv_dt - a0.x) / kResScale;
  target[3 * i + 1] = ((b.y - a.y) * inv_dt - a0.y) / kResScale;
  target[3 * i + 2] = ((b.z - a.z) * inv_dt - a0.z) / kResScale;
}

// inv[perm[k]] = k
__global__ void k_invert_perm(const uint32_t* __restrict__ perm, uint32_t n,
                              uint32_t* __restrict__ inv) {
  uint32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < n) {
    uint32_t p = perm[k];
    if (p < n) inv[p] = k;
  }
}

// Density difference of particle (sorted position i of state a) against the
// same particle in state b: a's canonical index perm_a[i] carries identity
// ids_a[...]; b holds it at canonical loc_b[id], sorted inv_b[loc_b[id]].
// Grid-stride; each work-group writes its (max, sum) to part[2 blockIdx.x].
constexpr int kCmpBlocks = 1024;

__global__ __launch_bounds__(256) void k_compare(const uint32_t* __restrict__ perm_a,
                                                 const uint32_t* __restrict__ ids_a,
                                                 const float* __restrict__ rho_a,
                                                 const uint32_t* __restrict__ loc_b,
                                                 const uint32_t* __restrict__ inv_b,
                                                 const float* __restrict__ rho_b, uint32_t n,
                                                 float* __restrict__ part) {
  __shared__ float red[2][4];
  float mx = 0.f, sm = 0.f;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    uint32_t c = perm_a[i];
    uint32_t id = c < n ? ids_a[c] : 0u;
    uint32_t cb = id < n ? loc_b[id] : 0u;
    uint32_t ib = cb < n ? inv_b[cb] : 0u;
    float d = fabsf(rho_a[i] - rho_b[ib]);
    mx = fmaxf(mx, d);
    sm += d;
  }
  for (int o = 32; o > 0; o >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    sm += __shfl_xor(sm, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = mx;
    red[1][threadIdx.x >> 6] = sm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    part[2 * blockIdx.x + 1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  }
}

// res = (max, sum) over the `nparts` work-group partials; one work-group.
__global__ __launch_bounds__(256) void k_compare_final(const float* __restrict__ part,
                                                       uint32_t nparts, float* __restrict__ res) {
  __shared__ float red[2][4];
  float mx = 0.f, sm = 0.f;
  for (uint32_t k = threadIdx.x; k < nparts; k += 256) {
    mx = fmaxf(mx, part[2 * k]);
    sm += part[2 * k + 1];
  }
  for (int o = 32; o > 0; o >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    sm += __shfl_xor(sm, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = mx;
    red[1][threadIdx.x >> 6] = sm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    res[0] = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    res[1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
  }
}

// Adds the forces stage's acceleration of sorted particle j to its identity's
// running sum (each identity occurs once per substep).
__global__ void k_accum_acc(const float4* __restrict__ acc, const uint32_t* __restrict__ perm,
                            const uint32_t* __restrict__ ids, uint32_t n,
                            float* __restrict__ sum) {
  uint32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  uint32_t c = perm[j];
  uint32_t id = c < n ? ids[c] : n;
  if (id >= n) return;
  float4 a = acc[j];
  sum[3 * id] += a.x;
  sum[3 * id + 1] += a.y;
  sum[3 * id + 2] += a.z;
}

// target[i] = (sum[perm[i]] / nsub - a0_i) / R for the learner's sorted i.
__global__ void k_target_mean(const uint32_t* __restrict__ perm, const float* __restrict__ sum,
                              const float4* __restrict__ acc0, uint32_t n, float inv_nsub,
                              float* __restrict__ target) {
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint32_t c = perm[i];
  if (c >= n) c = 0;
  float4 a0 = acc0[i];
  target[3 * i] = (sum[3 * c] * inv_nsub - a0.x) / kResScale;
  target[3 * i + 1] = (sum[3 * c + 1] * inv_nsub - a0.y) / kResScale;
  target[3 * i + 2] = (sum[3 * c + 2] * inv_nsub - a0.z) / kResScale;
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

void launch_graph(clsph_nn* m, clsph_state* st) {
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

void launch_edge_inputs(clsph_nn* m, clsph_state* st) {
  hipStream_t s = st->ctx->stream;
  uint32_t n = m->n, e = m->e;
  const DevParams& d = st->host_dps[0];
  hipLaunchKernelGGL(k_graph, dim3(n ? (n + 255) / 256 : 1, 8), dim3(256), 0, s, st->nbr,
                     st->nbr_count, m->off, n, m->src, m->dst, m->degc);
  hipLaunchKernelGGL(k_node_inputs, grid_of_all(n), dim3(256), 0, s, st->rho_s, st->prs_s, n,
                     d.p.fluid_density, d.p.K, (float2*)m->nu);
  hipLaunchKernelGGL(k_edge_inputs, grid_for(e), dim3(256), 0, s, st->fab,
                     (const float2*)m->nu, m->src, m->dst, e, edge_consts(d), m->E1);
}

static inline const float* P(const clsph_nn* m, int id) { return m->params + param_offset(id); }
static inline const uint16_t* W(const clsph_nn* m, int id) { return m->wb + param_offset(id); }
static inline float* G(clsph_nn* m, int id) { return m->grad + param_offset(id); }

void forward(clsph_nn* m, const float4* acc0, float gx, float gy, float gz) {
  hipStream_t s = m->ctx->stream;
  const int n = (int)m->n;
  if (n) {
    hipLaunchKernelGGL(k_edge_layer, dim3((m->n + kEdgeParts - 1) / kEdgeParts), dim3(256), 0, s,
                       m->E1, W(m, E_W1), P(m, E_B1), m->off, m->n, m->S, m->mask);
    hipLaunchKernelGGL(k_pack_u, grid_of_all((size_t)n * (kIn / 8)), dim3(256), 0, s, m->S, m->nu,
                       acc0, m->degc, m->n, gx, gy, gz, m->u);
  }
  gemm_silu(s, m->u, kIn, W(m, N_W1), kNodeW, P(m, N_B1), m->p1, m->y1, n, kNodeW, kIn);
  gemm_silu(s, m->y1, kNodeW, W(m, N_W2), kNodeW, P(m, N_B2), m->p2, m->y2, n, kNodeW, kNodeW);
  gemm(s, false, false, false, m->y2, kNodeW, W(m, N_W3), kOut, m->out, kOut, n, kOut, kNodeW,
       1.f, P(m, N_B3));
}

void forward_fused(clsph_nn* m, clsph_state* st, float4* acc, float* out, bool own_forces,
                   hipEvent_t* ev, bool nu_ready) {
  hipStream_t s = m->ctx->stream;
  uint32_t n = st->n;
  m->n = n;
  const DevParams& d = st->host_dps[0];
  if (ev) (void)hipEventRecord(ev[0], s);
  if (!nu_ready)
    hipLaunchKernelGGL(k_node_inputs, grid_of_all(n), dim3(256), 0, s, st->rho_s, st->prs_s, n,
                       d.p.fluid_density, d.p.K, (float2*)m->nu);
  // persistent grid: the work-groups that fit on the device at once (the
  // kernel's registers and LDS allow two per compute unit) stage the weights
  // once each
  static int per_cu = 0;
  if (per_cu <= 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k_surrogate<true>,
                                                     kSurWaves * 64, 0) != hipSuccess ||
        per_cu <= 0)
      per_cu = 1;
  }
  uint32_t ntiles = (n + kTileP - 1) / kTileP;
  uint32_t blocks = (uint32_t)st->ctx->cus * (uint32_t)per_cu;
  if (blocks * kSurWaves > ntiles) blocks = (ntiles + kSurWaves - 1) / kSurWaves;
  if (blocks == 0) blocks = 1;
  if (own_forces)
    hipLaunchKernelGGL(k_surrogate<true>, dim3(blocks), dim3(kSurWaves * 64), 0, s, st->fab,
                       (const float2*)m->nu, st->rho_s, st->nbr, st->nbr_count, n,
                       edge_consts(d), force_tail(d), m->wb, m->params, acc, out);
  else
    hipLaunchKernelGGL(k_surrogate<false>, dim3(blocks), dim3(kSurWaves * 64), 0, s, st->fab,
                       (const float2*)m->nu, st->rho_s, st->nbr, st->nbr_count, n,
                       edge_consts(d), force_tail(d), m->wb, m->params, acc, out);
  if (ev) (void)hipEventRecord(ev[1], s);
}

// Backward of the node MLP and the edge layer.
void backward(clsph_nn* m) {
  hipStream_t s = m->ctx->stream;
  int n = (int)m->n, e = (int)m->e;
  fill(m->grad, kParamTotal, 0.f, s);
  fill(m->loss, 1, 0.f, s);
  hipLaunchKernelGGL(k_loss, grid_of_all(n), dim3(256), 0, s, m->out, m->target, m->n, m->dout,
                     m->loss);
  hipLaunchKernelGGL(k_cast, grid_for((size_t)n * kOut), dim3(256), 0, s, m->dout, m->dout_b,
                     (size_t)n * kOut);
  // layer 3
  gemm(s, true, false, true, m->y2, kNodeW, m->dout_b, kOut, G(m, N_W3), kOut, kNodeW, kOut, n,
       1.f);
  colsum(s, m->dout, kOut, n, kOut, nullptr, G(m, N_B3));
  gemm_dsilu(s, m->dout_b, kOut, W(m, N_W3), kOut, m->p2, m->dpb, n, kNodeW, kOut);
  // layer 2; each work-group's rows of dpb are its own input and output
  gemm_weight_grad(s, m->y1, kNodeW, m->dpb, kNodeW, G(m, N_W2), G(m, N_B2), kNodeW, kNodeW, n);
  gemm_dsilu(s, m->dpb, kNodeW, W(m, N_W2), kNodeW, m->p1, m->dpb, n, kNodeW, kNodeW);
  // layer 1, and d loss / d S (the first 32 inputs) into dY
  gemm_weight_grad(s, m->u, kIn, m->dpb, kNodeW, G(m, N_W1), G(m, N_B1), kIn, kNodeW, n);
  gemm(s, false, true, false, m->dpb, kNodeW, W(m, N_W1), kNodeW, m->dY, kNodeW, n, kEdgeW,
       kNodeW, 1.f);
  // edge layer
  if (e > 0) {
    // about two work-groups per compute unit, 1,024 edges each at least
    uint32_t per = ((uint32_t)e + 511u) / 512u;
    per = std::max(1024u, (per + 255u) & ~255u);
    hipLaunchKernelGGL(k_edge_grad, dim3(((uint32_t)e + per - 1u) / per), dim3(256), 0, s, m->E1,
                       m->dY, kNodeW, m->mask, m->dst, (uint32_t)e, per, G(m, E_W1), G(m, E_B1));
  }
}

void adam(clsph_nn* m, float lr, float beta1, float beta2, float eps) {
  m->adam_step += 1;
  float bc1 = 1.f - powf(beta1, (float)m->adam_step);
  float bc2 = 1.f - powf(beta2, (float)m->adam_step);
  hipLaunchKernelGGL(k_adam, grid_for(kParamTotal), dim3(256), 0, m->ctx->stream, m->params,
                     m->grad, m->adam_m, m->adam_v, (size_t)kParamTotal, lr, beta1, beta2, eps,
                     bc1, bc2, m->wb);
}

void cast_params(clsph_nn* m) {
  hipLaunchKernelGGL(k_cast, grid_for(kParamTotal), dim3(256), 0, m->ctx->stream, m->params,
                     m->wb, (size_t)kParamTotal);
}

void launch_target_mean(clsph_nn* m, clsph_state* learner, clsph_state* teacher, uint32_t nsub) {
  hipStream_t s = m->ctx->stream;
  uint32_t n = learner->n;
  fill(m->sum, 3 * (size_t)n, 0.f, s);
  for (uint32_t k = 0; k < nsub; ++k) {
    launch_grid_params(teacher);
    launch_hash(teacher);
    launch_sort(teacher);
    launch_density(teacher);
    launch_forces(teacher);
    hipLaunchKernelGGL(k_accum_acc, grid_of_all(n), dim3(256), 0, s, teacher->acc_s, teacher->val_b,
                       teacher->ids, n, m->sum);
    launch_advect(teacher);
    launch_track_ids(teacher);
  }
  hipLaunchKernelGGL(k_target_mean, grid_of_all(n), dim3(256), 0, s, learner->val_b, m->sum,
                     learner->acc_s, n, 1.f / (float)nsub, m->target);
}

void launch_target(clsph_nn* m, clsph_state* a, clsph_state* t, float dt) {
  hipStream_t s = m->ctx->stream;
  uint32_t n = a->n;
  hipLaunchKernelGGL(k_invert, grid_of_all(n), dim3(256), 0, s, t->ids, n, m->loc);
  hipLaunchKernelGGL(k_target, grid_of_all(n), dim3(256), 0, s, a->val_b, a->vh, m->loc, t->vh,
                     a->acc_s, n, 1.f / dt, m->target);
}

// Workspace of clsph_nn_gemm_noalloc: the device copies of its operands.
// Every GPU the library runs on holds one copy of this array until the
// process ends. Host code never passes the array's name to a kernel or a
// copy: the name is a host-side stand-in, and the device address comes from
// hipGetSymbolAddress below, per device.
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

hipError_t scratch_address(int device, void** ptr) {
  static std::mutex lock;
  static std::vector<void*> addr;  // per device, looked up once
  std::lock_guard<std::mutex> g(lock);
  if (device < 0) return hipErrorInvalidDevice;
  if ((size_t)device >= addr.size()) addr.resize((size_t)device + 1, nullptr);
  if (!addr[device]) {
    // the caller has made `device` current
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[device] = p;
  }
  *ptr = addr[device];
  return hipSuccess;
}

void launch_compare(clsph_nn* m, clsph_state* a, clsph_state* b, float res[2]) {
  hipStream_t s = m->ctx->stream;
  uint32_t n = a->n;
  hipLaunchKernelGGL(k_invert, grid_of_all(n), dim3(256), 0, s, b->ids, n, m->loc);
  hipLaunchKernelGGL(k_invert_perm, grid_of_all(n), dim3(256), 0, s, b->val_b, n, m->inv);
  uint32_t blocks = (n + 255) / 256;
  if (blocks > (uint32_t)kCmpBlocks) blocks = kCmpBlocks;
  if (blocks == 0) blocks = 1;
  // the partials go to m->sum: 2 ceil(n / 256) <= 2 n <= 3 n_cap floats
  hipLaunchKernelGGL(k_compare, dim3(blocks), dim3(256), 0, s, a->val_b, a->ids, a->rho_s, m->loc,
                     m->inv, b->rho_s, n, m->sum);
  hipLaunchKernelGGL(k_compare_final, dim3(1), dim3(256), 0, s, m->sum, blocks, m->cmp);
  (void)hipMemcpyAsync(res, m->cmp, 2 * sizeof(float), hipMemcpyDeviceToHost, s);
}

}  // namespace nn
}  // namespace clsph
