// Pieces shared by the fp32-precision kernels (ssa_f32.hip, ssa_d256.hip): a
// wave owns 32 rows, one per lane pair (l, l + 32), and streams blocks of 32
// rows of the other side through LDS.
#pragma once

#include "ssa_common.hpp"
#include "ssa_launch.hpp"
#include "ssa_tile.hpp"

namespace ssa {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Four consecutive elements of T as fp32 (16-byte or 8-byte aligned: columns
// are multiples of 4, rows 16-byte aligned), and back.
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
template <typename T>
__device__ __forceinline__ f32x4 ld4(const T* p) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  const t4 x = *reinterpret_cast<const t4*>(p);
  return f32x4{static_cast<float>(x[0]), static_cast<float>(x[1]), static_cast<float>(x[2]),
               static_cast<float>(x[3])};
}
template <typename T>
__device__ __forceinline__ void st4(T* p, f32x4 v) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<t4*>(p) = t4{static_cast<T>(v[0]), static_cast<T>(v[1]), static_cast<T>(v[2]),
                                 static_cast<T>(v[3])};
}

// sL = sign(x) log2(1 + c|x|) for a raw score x = q.k, c = scale b; u1 = 1 + c|x|
__device__ __forceinline__ float ssa_sl(float x, float u1) { return copysignf(fast_log2(u1), x); }

// A workgroup's place in a grid of nblk blocks of rows per (sequence, head):
// XCD-contiguous, the heaviest blocks (rank 0) of a pair of heads first, as
// FwdPlan and DkdvPlan.
struct Place {
  int rank, b, h;
  __device__ __forceinline__ Place(int block, int grid, int nblk, int B, bool packed) {
    int hb;
    dispatch_order(xcd_remap(block, grid), grid / nblk, nblk, packed ? 1 : kOrderGroup, hb, rank);
    b = hb % B;
    h = hb / B;
  }
};

// Sum of the accumulators of the waves that share owned rows, in the first of them (part == 0): the others leave theirs
// in LDS, element-major so that every access is contiguous.  Called by every
// wave; `lds` is free (all waves past their last read of the ring).
template <int ND, int KW>
__device__ __forceinline__ void merge_parts(f32x16* acc, float* lds, int group, int part, int lane) {
  if constexpr (KW > 1) {
    __syncthreads();
    float* mine = lds + static_cast<size_t>((group * (KW - 1) + part - 1) * ND * 16 * 64) + lane;
    if (part > 0) {
#pragma unroll
      for (int i = 0; i < ND * 16; ++i) mine[i * 64] = acc[i >> 4][i & 15];
    }
    __syncthreads();
    if (part == 0) {
#pragma unroll
      for (int w = 1; w < KW; ++w) {
        const float* src = lds + static_cast<size_t>((group * (KW - 1) + w - 1) * ND * 16 * 64) + lane;
#pragma unroll
        for (int i = 0; i < ND * 16; ++i) acc[i >> 4][i & 15] += src[i * 64];
      }
    }
  }
}

// The lane's share of its own row: columns 32 db + 8 g + 4 hh + (0..3).
template <typename T, int D>
__device__ __forceinline__ void store_own(const f32x16* acc, float scale, T* row, int hh) {
#pragma unroll
  for (int db = 0; db < (D + 31) / 32; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (32 * db + 8 * g >= D) break;  // head dim 16
      st4(row + 32 * db + 8 * g + 4 * hh,
          f32x4{acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]} * scale);
    }
  }
}

// A launch takes fewer than 2^32 threads along x: larger row grids (from 2^23
// workgroups) fold over y.
inline dim3 row_grid(int n) {
  const int y = (n + (1 << 23) - 1) >> 23;
  return dim3((n + y - 1) / y, y);
}

}  // namespace

}  // namespace ssa
