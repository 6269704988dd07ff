// Pieces shared by the fp32-precision kernels (ssa_f32.hip, ssa_d256.hip): a
// wave owns 32 rows, one per lane pair (l, l + 32), and streams blocks of 32
// rows of the other side through LDS.
#pragma once

#include "ssa_common.hpp"
#include "ssa_launch.hpp"
#include "ssa_rows_plan.hpp"
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

// Rows with non-finite results, once more.  The outer products give a masked
// pair the weight 0, which keeps it out of the sums only while the streamed row
// (and, in the backward, the pair's dP and score) is finite: 0 x inf is NaN.  A
// row that ends with an infinite or NaN element is therefore summed again over
// its valid pairs only, pair by pair from global memory, 32 columns at a time
// into its place in the output: the accumulators are free by then, and finite
// results, and the loops, pay one test of them.  RARE tells the compiler, which
// would take these nested loops for the hot ones and spill for them in the
// others (head dim 256 backward, 16 x 2048 causal in bf16: 286 us before, 312 with
// them, 289 so marked; small calls pay 0.3 to 0.7 us a kernel).
#define SSA_RARE(cond) __builtin_expect_with_probability(static_cast<bool>(cond), false, 1.0)
template <int ND>
__device__ __forceinline__ bool row_nonfinite(const f32x16* acc, float more = 0.f) {
  float t = more * 0.f;
#pragma unroll
  for (int i = 0; i < ND * 16; ++i) t = fmaf(acc[i >> 4][i & 15], 0.f, t);
  return pair_max(t == 0.f ? 0.f : 1.f) != 0.f;
}

// a . b of two rows, by the two lanes of a pair.
template <typename T, int D>
__device__ __forceinline__ float pair_dot(const T* a, const T* b, int hh) {
  float s = 0.f;
#pragma unroll 2
  for (int i = 4 * hh; i < D; i += 8) {
    const f32x4 x = ld4(a + i), y = ld4(b + i);
    s = fmaf(x.x, y.x, fmaf(x.y, y.y, fmaf(x.z, y.z, fmaf(x.w, y.w, s))));
  }
  return pair_sum(s);
}

// a += w (columns 8 g + 4 hh + (0..3) of 32 columns of a row), and their store.
template <typename T, int D>
__device__ __forceinline__ void add_cols(f32x16& a, float w, const T* row, int hh) {
#pragma unroll
  for (int g = 0; g < (D < 32 ? D / 8 : 4); ++g) {
    const f32x4 x = ld4(row + 8 * g + 4 * hh);
#pragma unroll
    for (int e = 0; e < 4; ++e) a[4 * g + e] = fmaf(w, x[e], a[4 * g + e]);
  }
}
template <typename T, int D>
__device__ __forceinline__ void store_cols(const f32x16& a, float scale, T* row, int hh) {
#pragma unroll
  for (int g = 0; g < (D < 32 ? D / 8 : 4); ++g)
    st4(row + 8 * g + 4 * hh, f32x4{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]} * scale);
}

// Forward: out = scale sum of exp2(t - base) v over keys 0 .. last.
template <typename T, int D>
__device__ __forceinline__ void row_fwd(T* out, float scale, const T* q, const T* k, int64_t kss, const T* v,
                                        int64_t vss, int last, float n, float c, float base, int hh) {
#pragma unroll 1
  for (int col = 0; col < D; col += 32) {
    f32x16 a = f32x16{};
#pragma unroll 1
    for (int j = 0; j <= last; ++j) {
      const float x = pair_dot<T, D>(q, k + j * kss, hh);
      add_cols<T, D>(a, fast_exp2(fmaf(n, ssa_sl(x, fmaf(c, fabsf(x), 1.f)), -base)), v + j * vss + col, hh);
    }
    store_cols<T, D>(a, scale, out + col, hh);
  }
}

// dQ: dq = scale sum of dS' k over keys 0 .. last.
template <typename T, int D>
__device__ __forceinline__ void row_dq(T* dq, float scale, const T* q, const T* dout, const T* k, int64_t kss,
                                       const T* v, int64_t vss, int last, float n, float c, float m, float delta,
                                       int hh) {
#pragma unroll 1
  for (int col = 0; col < D; col += 32) {
    f32x16 a = f32x16{};
#pragma unroll 1
    for (int j = 0; j <= last; ++j) {
      const float x = pair_dot<T, D>(q, k + j * kss, hh), dp = pair_dot<T, D>(dout, v + j * vss, hh);
      const float u1 = fmaf(c, fabsf(x), 1.f);
      const float w = fast_exp2(fmaf(n, ssa_sl(x, u1), -m));
      add_cols<T, D>(a, w * (dp - delta) * fast_rcp(u1), k + j * kss + col, hh);
    }
    store_cols<T, D>(a, scale, dq + col, hh);
  }
}

// dK, dV (null: not wanted) of key row `key` of (b, hk) over the queries that see
// it, and the sums of dT sL and dS' x of its pairs (in both lanes).
template <typename T, int D, bool CAUSAL>
__device__ __forceinline__ void row_dkdv(const BwdParams& p, const SeqView& sv, int b, int hk, int key, float n,
                                         float c, T* dk, float dk_scale, T* dv, float& dn, float& db, int hh) {
  const int G = p.Hq / p.Hkv;
  const T* k = static_cast<const T*>(p.k.ptr) + sv.off(p.k, b) + hk * p.k.sh + key * p.k.ss;
  const T* v = static_cast<const T*>(p.v.ptr) + sv.off(p.v, b) + hk * p.v.sh + key * p.v.ss;
#pragma unroll 1
  for (int col = 0; col < D; col += 32) {
    f32x16 ak = f32x16{}, av = f32x16{};
    float sn = 0.f, sb = 0.f;
#pragma unroll 1
    for (int h = hk * G; h < hk * G + G; ++h) {
      const T* q = static_cast<const T*>(p.q.ptr) + sv.off(p.q, b) + h * p.q.sh;
      const T* dout = static_cast<const T*>(p.dout.ptr) + sv.off(p.dout, b) + h * p.dout.sh;
      const int64_t mr = sv.mrow(b, h, p.Hq, p.T, p.N);
#pragma unroll 1
      for (int i = CAUSAL ? key : 0; i < sv.N; ++i) {
        const T *qi = q + i * p.q.ss, *di = dout + i * p.dout.ss;
        const float x = pair_dot<T, D>(qi, k, hh), dp = pair_dot<T, D>(di, v, hh);
        const float u1 = fmaf(c, fabsf(x), 1.f), sl = ssa_sl(x, u1);
        const float w = fast_exp2(fmaf(n, sl, -p.m[mr + i])), dt = w * (dp - p.delta[mr + i]);
        const float ds = dt * fast_rcp(u1);
        sn = fmaf(dt, sl, sn);
        sb = fmaf(ds, x, sb);
        add_cols<T, D>(ak, ds, qi + col, hh);
        add_cols<T, D>(av, w, di + col, hh);
      }
    }
    if (dk != nullptr) store_cols<T, D>(ak, dk_scale, dk + col, hh);
    if (dv != nullptr) store_cols<T, D>(av, 1.f, dv + col, hh);
    dn = sn;
    db = sb;
  }
}

}  // namespace

}  // namespace ssa
