// The primal recomputation W = W0 + X A' (eval_recompute_primal,
// eval/core.h:148-182) on the matrix cores: with examples as rows,
//   W[j][l] = sum_i A[i][j] X[i][l]   (W: m x d, A: n x m, X: n x d),
// a contraction over the n examples with a small output.
//
// Both operands are contiguous across the output, so a slab of examples
// goes to LDS as it lies in memory ([example][class], [example][feature])
// and is read there by MFMA operand lanes: no transposed copies.  What
// bounds it is filling the chip: m = 137, d = 513 has 27 output tiles of
// 64 x 64 for 256 CUs, so the examples are split over enough workgroups
// for about four per CU, each split's tile goes to the workspace, and a
// second kernel adds the splits (and W0).  n = 20,011, m = 137, d = 513:
// fp64 1498 us as one split through transposed copies, 142 us here; fp32
// 2671 us, 77 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "eval_launch.hpp"

namespace sdca_gpu {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;   // output tile: 64 classes x 64 features, 4 waves of 32 x 32
// Examples per LDS slab: 16 KiB of the operands either way, about a
// microsecond of MFMAs for the next slab's loads to land in.
template <class D>
constexpr int kSlab = 128 / static_cast<int>(sizeof(D));
constexpr int kLd = kTile + 4;
// Workgroups wanted (four per CU), and the fewest examples worth a split.
constexpr int64_t kPrimalBlocks = 1024;
constexpr int64_t kPrimalMinChunk = 128;

// A wave's 32 x 32 block: one v_mfma_f32_32x32x2f32 accumulator, or 2 x 2
// of v_mfma_f64_16x16x4f64.
template <class D>
struct Block;
template <>
struct Block<float> {
  f32x16 acc;
  __device__ void clear() {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  }
  // Operand lanes: element l % 32 of example l / 32 of each pair.
  __device__ void slab(const float* as, const float* bs, int lane) {
    const float* a = as + (lane >> 5) * kLd + (lane & 31);
    const float* b = bs + (lane >> 5) * kLd + (lane & 31);
#pragma unroll
    for (int k = 0; k < kSlab<float>; k += 2)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k * kLd], b[k * kLd], acc, 0, 0, 0);
  }
  // Accumulator e of lane l: row 8 (e / 4) + 4 (l / 32) + e % 4, column l % 32.
  template <class F>
  __device__ void each(int lane, F f) const {
#pragma unroll
    for (int e = 0; e < 16; ++e) f(8 * (e >> 2) + 4 * (lane >> 5) + (e & 3), lane & 31, acc[e]);
  }
};
template <>
struct Block<double> {
  f64x4 acc[2][2];
  __device__ void clear() {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[q >> 1][q & 1][e] = 0.0;
  }
  // Operand lanes: element l % 16 of example l / 16 of each four.
  __device__ void slab(const double* as, const double* bs, int lane) {
    const double* a = as + (lane >> 4) * kLd + (lane & 15);
    const double* b = bs + (lane >> 4) * kLd + (lane & 15);
#pragma unroll
    for (int k = 0; k < kSlab<double>; k += 4) {
      const double a0 = a[k * kLd], a1 = a[k * kLd + 16];
      const double b0 = b[k * kLd], b1 = b[k * kLd + 16];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
  }
  // Accumulator e of lane l: row l / 16 + 4 e, column l % 16 of its block.
  template <class F>
  __device__ void each(int lane, F f) const {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        f(16 * (q >> 1) + (lane >> 4) + 4 * e, 16 * (q & 1) + (lane & 15), acc[q >> 1][q & 1][e]);
  }
};

// Slab [i0, i0 + kSlab) of a (rows x cols) matrix, columns [c0, c0 + 64).
// Columns past the matrix read its last one (their outputs are not stored),
// examples at or past `end` read as zero.
template <class D>
__device__ inline void slab_load(const D* __restrict__ src, int64_t cols, int64_t c0, int64_t i0,
                                 int64_t end, D (&r)[kSlab<D> / 4]) {
  const int64_t c = c0 + (threadIdx.x & 63);
  const D* p = src + (c < cols ? c : cols - 1);
#pragma unroll
  for (int h = 0; h < kSlab<D> / 4; ++h) {
    const int64_t i = i0 + (threadIdx.x >> 6) + 4 * h;
    const D x = p[(i < end ? i : end - 1) * cols];
    r[h] = i < end ? x : D(0);
  }
}
template <class D>
__device__ inline void slab_store(D* __restrict__ lds, const D (&r)[kSlab<D> / 4]) {
#pragma unroll
  for (int h = 0; h < kSlab<D> / 4; ++h)
    lds[((threadIdx.x >> 6) + 4 * h) * kLd + (threadIdx.x & 63)] = r[h];
}

// Grid: (feature tiles, class tiles, splits); split z takes the examples
// [z chunk, (z + 1) chunk) and writes P[z] (m x d).
template <class D>
__global__ void __launch_bounds__(256)
primal_gemm_kernel(const D* __restrict__ A, const D* __restrict__ X, D* __restrict__ P, int64_t n,
                   int64_t m, int64_t d, int64_t chunk, int64_t tiles_d, int64_t tiles_m) {
  __shared__ __align__(16) D As[2][kSlab<D> * kLd];
  __shared__ __align__(16) D Bs[2][kSlab<D> * kLd];
  const int64_t w = blockIdx.x;
  const int64_t z = w / (tiles_d * tiles_m);
  const int64_t j0 = (w / tiles_d) % tiles_m * kTile, l0 = w % tiles_d * kTile;
  const int64_t first = z * chunk, end = first + chunk < n ? first + chunk : n;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = static_cast<int>(threadIdx.x) >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  Block<D> blk;
  blk.clear();
  D ra[kSlab<D> / 4], rb[kSlab<D> / 4];
  slab_load(A, m, j0, first, end, ra);
  slab_load(X, d, l0, first, end, rb);
  slab_store(As[0], ra);
  slab_store(Bs[0], rb);
  __syncthreads();
  int cur = 0;
  for (int64_t i = first; i < end; i += kSlab<D>) {
    const bool more = i + kSlab<D> < end;
    if (more) {
      slab_load(A, m, j0, i + kSlab<D>, end, ra);
      slab_load(X, d, l0, i + kSlab<D>, end, rb);
    }
    blk.slab(As[cur] + 32 * wr, Bs[cur] + 32 * wc, lane);
    if (more) {
      slab_store(As[cur ^ 1], ra);
      slab_store(Bs[cur ^ 1], rb);
    }
    __syncthreads();
    cur ^= 1;
  }
  D* const out = P + z * m * d;
  blk.each(lane, [&](int r, int c, D v) {
    const int64_t j = j0 + 32 * wr + r, l = l0 + 32 * wc + c;
    if (j < m && l < d) out[j * d + l] = v;
  });
}

// W = sum of the splits + W0: 32 outputs per workgroup, eight threads each
// (every eighth split in order, then the eight sums in order), so that a
// small output over hundreds of splits is not one long chain of loads.
template <class D>
__global__ void __launch_bounds__(256)
primal_sum_kernel(const D* __restrict__ P, int splits, int64_t count, const D* W0, D* W) {
  __shared__ D part[8][32];
  const int c = static_cast<int>(threadIdx.x) & 31, g = static_cast<int>(threadIdx.x) >> 5;
  for (int64_t i0 = blockIdx.x * 32ll; i0 < count; i0 += gridDim.x * 32ll) {
    const int64_t i = i0 + c;
    D s = D(0);
    if (i < count) {
#pragma unroll 4
      for (int z = g; z < splits; z += 8) s += P[z * count + i];
    }
    part[g][c] = s;
    __syncthreads();
    if (g == 0 && i < count) {
#pragma unroll
      for (int h = 1; h < 8; ++h) s += part[h][c];
      W[i] = W0 ? s + W0[i] : s;
    }
    __syncthreads();
  }
}

int64_t primal_splits(int64_t d, int64_t m, int64_t n) {
  const int64_t tiles = ((d + kTile - 1) / kTile) * ((m + kTile - 1) / kTile);
  const int64_t want = (kPrimalBlocks + tiles - 1) / tiles;
  const int64_t most = (n + kPrimalMinChunk - 1) / kPrimalMinChunk;
  return std::max<int64_t>(1, std::min(want, most));
}

template <class D>
hipError_t launch_primal_t(const void* X, const void* A, const void* W0, void* W, void* ws,
                           int64_t d, int64_t m, int64_t n, hipStream_t stream) {
  const int64_t tiles_d = (d + kTile - 1) / kTile, tiles_m = (m + kTile - 1) / kTile;
  int64_t splits = primal_splits(d, m, n);
  int64_t chunk = (n + splits - 1) / splits;
  chunk = (chunk + kSlab<D> - 1) / kSlab<D> * kSlab<D>;
  splits = (n + chunk - 1) / chunk;
  // one split and no W0: straight to W
  D* const P = (splits == 1 && !W0) ? static_cast<D*>(W) : static_cast<D*>(ws);
  hipLaunchKernelGGL(primal_gemm_kernel<D>, dim3(static_cast<unsigned>(tiles_d * tiles_m * splits)),
                     dim3(256), 0, stream, static_cast<const D*>(A), static_cast<const D*>(X), P, n,
                     m, d, chunk, tiles_d, tiles_m);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || P == W) return e;
  const int64_t blocks = std::min<int64_t>(8192, (m * d + 31) / 32);
  hipLaunchKernelGGL(primal_sum_kernel<D>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,
                     P, static_cast<int>(splits), m * d, static_cast<const D*>(W0),
                     static_cast<D*>(W));
  return hipGetLastError();
}

}  // namespace

// Outputs of 512 tiles or more fill the chip with the score GEMM's own
// tiles (fp64 n = 50,000, m = 1000, d = 2000: 3.8 ms transposed, 4.5 ms
// here); where the fp32 product would go to the library, this kernel wins up
// to 256 classes, the library's transposed copies costing more than its
// GEMM gains (n = 100,000: m = 18, d = 3207 1150 -> 717 us; m = 200, d =
// 1024 1045 -> 738; m = 1000 stays).  fp64 sums over more than 65,536
// examples keep the one running sum of the score GEMM, for agreement with the
// W they always gave, which split sums would move by that sum's own error:
// more than 1e-14 of its norm.  Neither time nor accuracy asks for it (m =
// 137, d = 513, from long double in brackets: n = 65,536 split 452 us
// [1.2e-15]; 70,000 kept 2992 [8.2e-15], split 472 [1.8e-15]; 200,000 kept
// 8527 [1.6e-14], split 1334 [2.1e-15]).
bool primal_split(int data, int64_t d, int64_t m, int64_t n) {
  const int64_t tiles = ((d + kTile - 1) / kTile) * ((m + kTile - 1) / kTile);
  if (tiles >= 512) return false;
  if (data == SDCA_F64) return n <= 65536;
  return !blas_shape(m, d, n) || m <= 256;
}

int64_t primal_workspace_values(int64_t d, int64_t m, int64_t n) {
  return primal_splits(d, m, n) * m * d;
}

hipError_t launch_primal(int data, const void* X, const void* A, const void* W0, void* W, void* ws,
                         int64_t d, int64_t m, int64_t n, hipStream_t stream) {
  if (data == SDCA_F32) return launch_primal_t<float>(X, A, W0, W, ws, d, m, n, stream);
  return launch_primal_t<double>(X, A, W0, W, ws, d, m, n, stream);
}

}  // namespace sdca_gpu
