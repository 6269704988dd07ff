// Fused element-wise operators of the SSA decoder layer around the attention
// path (gfx950): rotary position embedding (one HBM pass per call in the
// input dtype; the unfused PyTorch form makes six fp32 passes), RMSNorm
// (one pass forward, one backward, plus a fixed-order weight-gradient sum),
// the SwiGLU gate (one pass each way) and the output layer's cross-entropy
// (one pass over the logits each way, no fp32 copy of them).
//
// Rotate-half RoPE (Megatron's default, non-interleaved), per (s, b, h) row of
// D values, i < D / 2, with c = cos[s][i], t = sin[s][i]:
//   y[i]         = x[i] c - x[i + D/2] t
//   y[i + D/2]   = x[i + D/2] c + x[i] t
// The inverse (the backward: the transpose of a rotation) uses -t.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ssa_decoder_ops.h"

namespace {

template <typename T>
struct Pack4 {
  typedef T type __attribute__((ext_vector_type(4)));
};

// One thread: 4 frequencies (8 values) of one row.  Rows are (s, b, h) in
// that order; x has strides (ss, sb, sh) and stride 1 over D, y is
// contiguous [S, B, H, D].
template <typename T, int D>
__global__ __launch_bounds__(256) void rope_kernel(const T* __restrict__ x, int64_t ss, int64_t sb, int64_t sh,
                                                   T* __restrict__ y, const float* __restrict__ cs,
                                                   const float* __restrict__ sn, int S, int B, int H, float sign) {
  typedef typename Pack4<T>::type v4;
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr int TPR = D / 8;  // threads per row
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t row = gid / TPR;
  const int i = static_cast<int>(gid % TPR) * 4;
  if (row >= static_cast<int64_t>(S) * B * H) return;
  const int h = static_cast<int>(row % H);
  const int64_t sbi = row / H;
  const int b = static_cast<int>(sbi % B), s = static_cast<int>(sbi / B);
  const T* xr = x + s * ss + b * sb + h * sh;
  const v4 x1 = *reinterpret_cast<const v4*>(xr + i);
  const v4 x2 = *reinterpret_cast<const v4*>(xr + i + D / 2);
  const f4 c = *reinterpret_cast<const f4*>(cs + static_cast<int64_t>(s) * (D / 2) + i);
  const f4 t = *reinterpret_cast<const f4*>(sn + static_cast<int64_t>(s) * (D / 2) + i);
  v4 y1, y2;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = static_cast<float>(x1[e]), bb = static_cast<float>(x2[e]), te = sign * t[e];
    y1[e] = static_cast<T>(a * c[e] - bb * te);
    y2[e] = static_cast<T>(bb * c[e] + a * te);
  }
  T* yr = y + row * D;
  *reinterpret_cast<v4*>(yr + i) = y1;
  *reinterpret_cast<v4*>(yr + i + D / 2) = y2;
}

template <typename T>
hipError_t launch_rope(const ssa_rope_args* a, hipStream_t st) {
  const int64_t rows = static_cast<int64_t>(a->seqlen) * a->batch * a->heads;
  const int64_t threads = rows * (a->head_dim / 8);
  const int grid = static_cast<int>((threads + 255) / 256);
  const T* x = static_cast<const T*>(a->x);
  T* y = static_cast<T*>(a->y);
  const float sign = a->inverse ? -1.f : 1.f;
  switch (a->head_dim) {
    case 64:
      hipLaunchKernelGGL((rope_kernel<T, 64>), dim3(grid), dim3(256), 0, st, x, a->x_stride_s, a->x_stride_b,
                         a->x_stride_h, y, a->cos, a->sin, a->seqlen, a->batch, a->heads, sign);
      break;
    case 128:
      hipLaunchKernelGGL((rope_kernel<T, 128>), dim3(grid), dim3(256), 0, st, x, a->x_stride_s, a->x_stride_b,
                         a->x_stride_h, y, a->cos, a->sin, a->seqlen, a->batch, a->heads, sign);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; }

// ---------------------------------------------------------------------------
// RMSNorm over rows of H fp32 values: r = (mean(x^2) + eps)^-1/2,
// y = (x r) w in the output dtype.  Backward, with g = dy w and xh = x r:
//   dx = r (g - xh sum(g xh) / H),  dw = sum over rows of dy xh.
//
// Both directions are HBM streams.  Forward: one workgroup per row (2048 x 2048
// to bf16: 6.5 us; 25 MB, 5 us at the rate of a large copy).
constexpr int kNormThreads = 256;
constexpr int kNormMaxHidden = 4096;
constexpr int kNormBwdRows = 64;  // rows per dw partial

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();  // red is reused by consecutive calls
  if (lane == 0) red[wave] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

template <typename TO>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_fwd_kernel(const float* __restrict__ x,
                                                                   const float* __restrict__ w,
                                                                   TO* __restrict__ y, float* __restrict__ rstd,
                                                                   int H, float eps) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const float* xr = x + row * H;
  float ss = 0.f;
  for (int c = threadIdx.x * 4; c < H; c += kNormThreads * 4) {
    const f4 v = *reinterpret_cast<const f4*>(xr + c);
    ss += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
  }
  const float r = rsqrtf(block_sum(ss, red) / H + eps);
  TO* yr = y + row * H;
  for (int c = threadIdx.x * 4; c < H; c += kNormThreads * 4) {
    const f4 v = *reinterpret_cast<const f4*>(xr + c);
    const f4 wv = *reinterpret_cast<const f4*>(w + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) yr[c + e] = static_cast<TO>(v[e] * r * wv[e]);
  }
  if (threadIdx.x == 0) rstd[row] = r;
}

// Backward in two kernels.  dx: a wave holds a whole row (lane l: columns
// 4 (l + 64 k) .. + 3, k < K; K = 4, 8 or 16 covers hidden sizes up to 1024,
// 2048 and 4096), so a row needs wave reductions only.  dw: a workgroup sums 64
// rows of 256 columns (each wave 16 rows, all its loads in flight), one partial
// per 64 rows.  One kernel that walked 64 rows per workgroup for both, a row at
// a time with a block reduction between the halves of its work, filled 32 CUs
// at 2048 rows and waited at its barriers.  bf16 dy, hidden 2048, the whole
// backward: 2048 rows 89 -> 20 us (dx 11, dw partials 5, their sum 3.5; 42 MB
// are 8 us at the rate of a large copy), 16384 rows 193 -> 102 us.  At 16384
// rows one kernel for both that keeps a row per wave and the dw sums in
// registers measured 73 us, at 2048 rows 37.
// The row's dot product keeps the summation tree of 256 threads with columns
// 4 (t + 256 j): four partial sums per lane (k % 4), a butterfly each, then
// (d0 + d1) + (d2 + d3).
constexpr int kNormDxWaves = 4;

// Four elements of dy, which the interface asks to be 8-byte aligned in any dtype.
template <typename T>
struct GradPack4 {
  typedef T type __attribute__((ext_vector_type(4), aligned(8)));
};

template <typename TG, int K>
__global__ __launch_bounds__(kNormDxWaves * 64) void rmsnorm_dx_kernel(const float* __restrict__ x,
                                                                       const float* __restrict__ w,
                                                                       const TG* __restrict__ dy,
                                                                       const float* __restrict__ rstd,
                                                                       float* __restrict__ dx, int64_t row0, int T,
                                                                       int H) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef typename GradPack4<TG>::type g4;
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kNormDxWaves + (threadIdx.x >> 6) + row0;
  if (row >= T) return;
  const float r = rstd[row];
  const float* xr = x + row * H;
  const TG* gr = dy + row * H;
  f4 xv[K];
  g4 gv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = 4 * (lane + 64 * k);
    xv[k] = c < H ? *reinterpret_cast<const f4*>(xr + c) : f4{0.f, 0.f, 0.f, 0.f};
    gv[k] = c < H ? *reinterpret_cast<const g4*>(gr + c) : g4{};
  }
  float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = 4 * (lane + 64 * k);
    if (c < H) {
      const f4 wv = *reinterpret_cast<const f4*>(w + c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        dot[k & 3] = fmaf(static_cast<float>(gv[k][e]) * wv[e], xv[k][e] * r, dot[k & 3]);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) dot[i] += __shfl_xor(dot[i], off, 64);
  }
  const float m = ((dot[0] + dot[1]) + (dot[2] + dot[3])) / H;
  float* dxr = dx + row * H;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = 4 * (lane + 64 * k);
    if (c < H) {
      const f4 wv = *reinterpret_cast<const f4*>(w + c);
      f4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = r * fmaf(-(xv[k][e] * r), m, static_cast<float>(gv[k][e]) * wv[e]);
      *reinterpret_cast<f4*>(dxr + c) = o;
    }
  }
}

template <typename TG>
__global__ __launch_bounds__(256) void rmsnorm_dw_part_kernel(const float* __restrict__ x,
                                                              const TG* __restrict__ dy,
                                                              const float* __restrict__ rstd,
                                                              float* __restrict__ dw_part, int T, int H) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef typename GradPack4<TG>::type g4;
  __shared__ f4 part[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ncol = (H + 255) / 256, group = blockIdx.x / ncol;  // 64 rows; the column blocks of a group together
  const int c = 256 * (blockIdx.x % ncol) + 4 * lane;
  const int64_t r0 = static_cast<int64_t>(group) * kNormBwdRows + wave * 16;
  f4 acc = f4{0.f, 0.f, 0.f, 0.f};
  if (c < H) {
    f4 xv[16];
    g4 gv[16];
    float rs[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t row = r0 + i < T ? r0 + i : T - 1;
      xv[i] = *reinterpret_cast<const f4*>(x + row * H + c);
      gv[i] = *reinterpret_cast<const g4*>(dy + row * H + c);
      rs[i] = r0 + i < T ? rstd[row] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r0 + i < T) acc[e] = fmaf(static_cast<float>(gv[i][e]), xv[i][e] * rs[i], acc[e]);
    }
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && c < H) {
    f4 s = part[0][lane];
#pragma unroll
    for (int v = 1; v < 4; ++v) s += part[v][lane];
    *reinterpret_cast<f4*>(dw_part + static_cast<int64_t>(group) * H + c) = s;
  }
}

// dw[c] = sum over partials of dw_part[b][c]: 64 columns per workgroup, 16
// waves on every 16th partial, their sums added in order (one thread per
// column walked up to 256 partials one after another: 9 us at 32 of them).
__global__ __launch_bounds__(1024) void rmsnorm_dw_kernel(const float* __restrict__ dw_part, float* __restrict__ dw,
                                                          int nparts, int H) {
  __shared__ float sum[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (c < H)
    for (int b = wave; b < nparts; b += 16) s += dw_part[static_cast<int64_t>(b) * H + c];
  sum[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || c >= H) return;
  s = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) s += sum[v][lane];
  dw[c] = s;
}

template <typename TG, int K>
void launch_norm_dx(const ssa_rmsnorm_bwd_args* a, hipStream_t s) {
  constexpr int kMaxRows = 1 << 25;  // 2^31 threads a launch
  for (int64_t row0 = 0; row0 < a->rows; row0 += kMaxRows) {
    const int n = static_cast<int>(a->rows - row0 < kMaxRows ? a->rows - row0 : kMaxRows);
    hipLaunchKernelGGL((rmsnorm_dx_kernel<TG, K>), dim3((n + kNormDxWaves - 1) / kNormDxWaves),
                       dim3(kNormDxWaves * 64), 0, s, static_cast<const float*>(a->x),
                       static_cast<const float*>(a->weight), static_cast<const TG*>(a->dy), a->rstd, a->dx, row0,
                       a->rows, a->hidden);
  }
}

// dx, then the dw partials to `part` (their reads of x and dy find what dx's left
// in the caches: 16384 x 2048 bf16 98.6 us, the other way round 100.2); where dx
// takes the place of x or dy, the partials first.  K the smallest whose 256 K
// columns hold a row.
template <typename TG>
void launch_norm_bwd(const ssa_rmsnorm_bwd_args* a, float* part, int nparts, hipStream_t s) {
  auto dw_part = [&]() {
    hipLaunchKernelGGL((rmsnorm_dw_part_kernel<TG>), dim3((a->hidden + 255) / 256 * nparts), dim3(256), 0, s,
                       static_cast<const float*>(a->x), static_cast<const TG*>(a->dy), a->rstd, part, a->rows,
                       a->hidden);
  };
  const bool in_place = a->dx == a->x || a->dx == a->dy;
  if (in_place) dw_part();
  if (a->hidden <= 1024)
    launch_norm_dx<TG, 4>(a, s);
  else if (a->hidden <= 2048)
    launch_norm_dx<TG, 8>(a, s);
  else
    launch_norm_dx<TG, 16>(a, s);
  if (!in_place) dw_part();
}

// ---------------------------------------------------------------------------
// SwiGLU of the MLP: z = [gate | up] rows of 2F values (the fc1 output), h =
// silu(gate) up with silu(g) = g sigmoid(g), in fp32, rounded once.
// Backward from dh: with s = sigmoid(g), d_up = dh silu(g) and
// d_gate = dh up s (1 + g (1 - s)), written as the [d_gate | d_up] rows of dz.
template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* __restrict__ z, const T* __restrict__ dh,
                                                     T* __restrict__ out, int64_t T_rows, int F, int backward) {
  typedef typename Pack4<T>::type v4;
  const int q = F / 4;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (gid >= T_rows * q) return;
  const int64_t row = gid / q;
  const int c = static_cast<int>(gid % q) * 4;
  const T* zr = z + row * 2 * F;
  const v4 g = *reinterpret_cast<const v4*>(zr + c);
  const v4 u = *reinterpret_cast<const v4*>(zr + F + c);
  if (!backward) {
    v4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float gf = static_cast<float>(g[e]);
      h[e] = static_cast<T>(gf / (1.f + __expf(-gf)) * static_cast<float>(u[e]));
    }
    *reinterpret_cast<v4*>(out + row * F + c) = h;
  } else {
    const v4 d = *reinterpret_cast<const v4*>(dh + row * F + c);
    v4 dg, du;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float gf = static_cast<float>(g[e]), uf = static_cast<float>(u[e]), df = static_cast<float>(d[e]);
      const float sg = 1.f / (1.f + __expf(-gf));
      du[e] = static_cast<T>(df * gf * sg);
      dg[e] = static_cast<T>(df * uf * sg * (1.f + gf * (1.f - sg)));
    }
    T* orow = out + row * 2 * F;
    *reinterpret_cast<v4*>(orow + c) = dg;
    *reinterpret_cast<v4*>(orow + F + c) = du;
  }
}

// ---------------------------------------------------------------------------
// Cross-entropy over rows of V logits (bf16/fp16), one workgroup per row.
// Forward: lse = log sum exp (one pass, running max per thread, merged across
// the workgroup); loss = lse - logit[label] (0 for label < 0).  Backward:
// dlogit = (exp(logit - lse) - [v == label]) * scale, 0 for an ignored row.
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mm = fmaxf(m, m2);
  s = (m == -INFINITY ? 0.f : s * __expf(m - mm)) + (m2 == -INFINITY ? 0.f : s2 * __expf(m2 - mm));
  m = mm;
}

// lse_merge(m, s, x, 1) bit for bit with one exponential: of its two factors the
// larger side's is exp(0) = 1.  m starts at kLseFloor (below every finite 16-bit
// value) instead of -infinity, so that x = -infinity adds exp(-inf) = 0 without a
// test; x - x makes x = +infinity the NaN of exp(inf - inf).
constexpr float kLseFloor = -3.4028234663852886e38f;
constexpr int kXentStep = 256 * 4;  // logits of a row in one pass of the workgroup
__device__ __forceinline__ void lse_add(float& m, float& s, float x) {
  const float d = x - m;
  const float e = __expf(-fabsf(d));
  float se = s * e;
  asm("" : "+v"(se));  // rounded: lse_merge's product ends in a select and is not contracted with the sum either
  s = d > 0.f ? se + (1.f + (x - x)) : s + e;
  m = fmaxf(m, x);
}

// The forward reads the logits once.  With a load, a wait and four merges of two
// exponentials each per step it was bound by that chain: four loads in flight
// and one exponential per logit, 2048 x 65536 bf16 (268 MB) in
// 55 us for 80.
template <typename T>
__global__ __launch_bounds__(256) void xent_fwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                       float* __restrict__ loss, float* __restrict__ lse, int V) {
  typedef typename Pack4<T>::type v4;
  __shared__ float sm[4], ss[4];
  const int64_t row = blockIdx.x;
  const T* lr = logits + row * V;
  float m = kLseFloor, s = 0.f;
  int c = threadIdx.x * 4;
  for (; c + 3 * kXentStep < V; c += 4 * kXentStep) {
    v4 x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const v4*>(lr + c + i * kXentStep);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) lse_add(m, s, static_cast<float>(x[i][e]));
  }
  for (; c < V; c += kXentStep) {
    const v4 x = *reinterpret_cast<const v4*>(lr + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) lse_add(m, s, static_cast<float>(x[e]));
  }
  m = m == kLseFloor ? -INFINITY : m;  // no finite logit: as lse_merge has it
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lse_merge(m, s, __shfl_xor(m, off, 64), __shfl_xor(s, off, 64));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sm[wave] = m;
    ss[wave] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float M = sm[0], S = ss[0];
    for (int w = 1; w < 4; ++w) lse_merge(M, S, sm[w], ss[w]);
    const float l = M + __logf(S);
    lse[row] = l;
    const int64_t lab = labels[row];
    loss[row] = (lab >= 0 && lab < V) ? l - static_cast<float>(lr[lab]) : 0.f;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void xent_bwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                       const float* __restrict__ lse, const float* __restrict__ scale,
                                                       T* __restrict__ dlogits, int V) {
  typedef typename Pack4<T>::type v4;
  const int64_t row = blockIdx.x;
  const int64_t lab = labels[row];
  const bool valid = lab >= 0 && lab < V;
  const float l = lse[row], g = valid ? *scale : 0.f;
  const T* lr = logits + row * V;
  T* dr = dlogits + row * V;
  for (int c = threadIdx.x * 4; c < V; c += 256 * 4) {
    const v4 x = *reinterpret_cast<const v4*>(lr + c);
    v4 d;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float p = __expf(static_cast<float>(x[e]) - l) - (c + e == lab ? 1.f : 0.f);
      d[e] = static_cast<T>(p * g);
    }
    *reinterpret_cast<v4*>(dr + c) = d;
  }
}

// ---------------------------------------------------------------------------
// Gradient of an fp32 embedding table: one workgroup per 64 table rows and 256
// columns, one float4 of columns per lane.  It walks the token ids (L2 hits),
// keeps its own tokens in LDS in token order, sorts them by row (stable) and
// writes each of its rows once: the sum of the named dy rows, or zero.  The four
// waves share the sorted list evenly, sixteen loads in flight each whatever rows
// they belong to, so frequent tokens that sit together do not make a chain; a row
// cut by a wave's end is put together in LDS.  A list that may not hold another
// chunk is added to the rows and started again.  All sums in a fixed order.
// Bound by the table's write.  Against PyTorch's fill and add, us by tokens (drawn
// evenly; all the same): 65536 x 2048 table (537 MB) 2048: 254 -> 99; 300 -> 148,
// 3072: 338 -> 106; 410 -> 190; 32000 x 1024 1000: 80 -> 28; 116 -> 49.
typedef float emb4 __attribute__((ext_vector_type(4)));
constexpr int kEmbRows = 64, kEmbCols = 256, kEmbChunk = 1024, kEmbList = 2 * kEmbChunk, kEmbLoads = 16;
constexpr int kEmbMaxTokens = 1 << 26;  // a list entry: token << 6 | row

__global__ __launch_bounds__(256) void embedding_bwd_kernel(const int64_t* __restrict__ ids,
                                                            const float* __restrict__ dy, float* __restrict__ grad,
                                                            int T, int V, int H, int slabs) {
  __shared__ uint32_t list[kEmbList], sorted[kEmbList];
  __shared__ volatile int hist[4][kEmbRows];
  __shared__ int place[4][kEmbRows];
  __shared__ int wave_count[4], head_row[4];
  __shared__ emb4 part[4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t below = (1ull << lane) - 1;
  const int r0 = static_cast<int>(blockIdx.x / slabs) * kEmbRows;
  const int nrows = min(kEmbRows, V - r0);
  const int col = static_cast<int>(blockIdx.x % slabs) * kEmbCols + lane * 4;
  const bool on = col < H;

  constexpr int PER = kEmbChunk / 256;
  int64_t id[PER];
  auto load_ids = [&](int base) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int t = base + wave * (kEmbChunk / 4) + i * 64 + lane;
      id[i] = t < T ? ids[t] : -1;
    }
  };
  load_ids(0);
  int n = 0;
  bool first = true;
  for (int base = 0; base < T; base += kEmbChunk) {
    // this chunk's tokens of these rows, in token order
    bool hit[PER];
    uint32_t entry[PER];
    uint64_t mask[PER];
    int count = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      hit[i] = id[i] >= r0 && id[i] < r0 + nrows;
      entry[i] = static_cast<uint32_t>(base + wave * (kEmbChunk / 4) + i * 64 + lane) << 6 |
                 static_cast<uint32_t>(id[i] - r0);
      mask[i] = __ballot(hit[i]);
      count += __popcll(mask[i]);
    }
    load_ids(base + kEmbChunk);
    if (lane == 0) wave_count[wave] = count;
    __syncthreads();
    int pos = n;
    for (int w = 0; w < wave; ++w) pos += wave_count[w];
    n += (wave_count[0] + wave_count[1]) + (wave_count[2] + wave_count[3]);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (hit[i]) list[pos + __popcll(mask[i] & below)] = entry[i];
      pos += __popcll(mask[i]);
    }
    __syncthreads();
    if (n <= kEmbList - kEmbChunk && base + kEmbChunk < T) continue;

    // Stable sort by row: rank of each entry among its wave's earlier ones of the
    // row, then the row's and the wave's place.  (The next chunk writes `list`
    // after its first barrier, which every wave reaches after all of this.)
    hist[wave][lane] = 0;
    const int quarter = ((n + 255) / 256) * 64;
    constexpr int GR = kEmbList / 256;
    uint32_t ent[GR];
    int rank[GR];
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      if (i * 64 >= quarter) break;
      const int k = wave * quarter + i * 64 + lane;
      const bool have = k < n;
      ent[i] = have ? list[k] : 0u;
      const int r = ent[i] & 63;
      uint64_t same = __ballot(have);
#pragma unroll
      for (int b = 0; b < 6; ++b) {
        const uint64_t bit = __ballot(r >> b & 1);
        same &= r >> b & 1 ? bit : ~bit;
      }
      const int before = hist[wave][r];
      rank[i] = before + __popcll(same & below);
      if (have && (same >> lane) == 1) hist[wave][r] = rank[i] + 1;  // the group's last of the row
    }
    __syncthreads();
    const int h0 = hist[0][lane], h1 = hist[1][lane], h2 = hist[2][lane], h3 = hist[3][lane];
    int end = h0 + h1 + h2 + h3;  // of row `lane` in the sorted list
    const uint64_t has = __ballot(end != 0);
    const int total = end;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(end, off, 64);
      if (lane >= off) end += up;
    }
    const int start = end - total;
    place[wave][lane] = start + (wave > 0 ? h0 : 0) + (wave > 1 ? h1 : 0) + (wave > 2 ? h2 : 0);
    if (lane == 0) head_row[wave] = -1;
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      if (i * 64 >= quarter) break;
      if (wave * quarter + i * 64 + lane < n) sorted[place[wave][ent[i] & 63] + rank[i]] = ent[i];
    }
    __syncthreads();

    emb4* const row0 = reinterpret_cast<emb4*>(grad + static_cast<int64_t>(r0) * H + col);
    auto at = [&](int r) { return row0 + static_cast<int64_t>(r) * (H / 4); };
    if (first && on)
      for (int r = wave; r < nrows; r += 4)
        if (!(has >> r & 1)) *at(r) = emb4{};
    auto emit = [&](int r, emb4 g) {
      if (on) *at(r) = first ? g : *at(r) + g;
    };
    const int k0 = n * wave / 4, k1 = n * (wave + 1) / 4;
    int cur = -1;
    emb4 sum = {}, acc = {};  // of `cur`: whole batches, this batch (shorter chains round less)
    // `cur` ends: its sum to its row, or (begun in an earlier wave) to that wave
    auto close = [&]() {
      if (cur < 0) return;
      if (__builtin_amdgcn_readlane(start, cur) >= k0) {
        emit(cur, sum + acc);
      } else {
        part[wave][lane] = sum + acc;
        if (lane == 0) head_row[wave] = cur;
      }
    };
    for (int k = k0; k < k1; k += kEmbLoads) {
      const int cnt = min(kEmbLoads, k1 - k);
      const uint32_t mine = sorted[k + min(lane, cnt - 1)];
      emb4 v[kEmbLoads];
#pragma unroll
      for (int j = 0; j < kEmbLoads; ++j) {
        v[j] = emb4{};
        if (j < cnt) {
          const uint32_t e = __builtin_amdgcn_readlane(mine, j);
          if (on) v[j] = *reinterpret_cast<const emb4*>(dy + static_cast<int64_t>(e >> 6) * H + col);
        }
      }
#pragma unroll
      for (int j = 0; j < kEmbLoads; ++j) {
        if (j < cnt) {
          const int r = __builtin_amdgcn_readlane(mine, j) & 63;
          if (r != cur) {
            close();
            cur = r;
            sum = emb4{};
            acc = v[j];
          } else {
            acc += v[j];
          }
        }
      }
      sum += acc;
      acc = emb4{};
    }
    const bool open = cur >= 0 && __builtin_amdgcn_readlane(end, max(cur, 0)) > k1 &&
                      __builtin_amdgcn_readlane(start, max(cur, 0)) >= k0;
    if (!open) close();
    __syncthreads();
    if (open) {
      for (int w = wave + 1; w < 4; ++w)
        if (head_row[w] == cur) sum += part[w][lane];
      emit(cur, sum);
    }
    n = 0;
    first = false;
  }
}

int32_t check_norm(const void* x, const void* w, const void* a, const void* b, int32_t T, int32_t H, int32_t dtype) {
  if (x == nullptr || w == nullptr || a == nullptr || b == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  if (T <= 0 || H <= 0 || H % 4 != 0 || H > kNormMaxHidden) return SSA_OPS_ERR_SHAPE;
  if (dtype != 0 && dtype != 1 && dtype != 2) return SSA_OPS_ERR_DTYPE;
  if (!aligned(x, 16) || !aligned(w, 16)) return SSA_OPS_ERR_ALIGNMENT;
  return SSA_OPS_OK;
}

}  // namespace

extern "C" int32_t ssa_rope(const ssa_rope_args* a, void* stream) {
  if (a == nullptr || a->x == nullptr || a->y == nullptr || a->cos == nullptr || a->sin == nullptr)
    return SSA_OPS_ERR_NULL_POINTER;
  if (a->seqlen <= 0 || a->batch <= 0 || a->heads <= 0) return SSA_OPS_ERR_SHAPE;
  // (token, head) rows fit int32, so the grid of head_dim / 8 threads per row fits too
  const int64_t sb = static_cast<int64_t>(a->seqlen) * a->batch;
  if (sb > INT32_MAX || sb * a->heads > INT32_MAX) return SSA_OPS_ERR_SHAPE;
  if (a->head_dim != 64 && a->head_dim != 128) return SSA_OPS_ERR_SHAPE;
  if (a->dtype != 0 && a->dtype != 1) return SSA_OPS_ERR_DTYPE;
  if (a->x_stride_s < 0 || a->x_stride_b < 0 || a->x_stride_h < 0) return SSA_OPS_ERR_ALIGNMENT;
  // 8-byte vector accesses: every row start and the tables 4-element aligned
  if (!aligned(a->x, 8) || !aligned(a->y, 8) || !aligned(a->cos, 16) || !aligned(a->sin, 16) ||
      (a->x_stride_s % 4) != 0 || (a->x_stride_b % 4) != 0 || (a->x_stride_h % 4) != 0)
    return SSA_OPS_ERR_ALIGNMENT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const hipError_t e = a->dtype == 0 ? launch_rope<__bf16>(a, st) : launch_rope<_Float16>(a, st);
  return e == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}

extern "C" int64_t ssa_rmsnorm_workspace_floats(int32_t rows, int32_t hidden) {
  if (rows <= 0 || hidden <= 0) return 0;
  return (static_cast<int64_t>(rows) + kNormBwdRows - 1) / kNormBwdRows * hidden;
}

extern "C" int32_t ssa_rmsnorm_fwd(const ssa_rmsnorm_fwd_args* a, void* stream) {
  if (a == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  const int32_t st = check_norm(a->x, a->weight, a->y, a->rstd, a->rows, a->hidden, a->out_dtype);
  if (st != SSA_OPS_OK) return st;
  if (!aligned(a->y, 8)) return SSA_OPS_ERR_ALIGNMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float* x = static_cast<const float*>(a->x);
  const float* w = static_cast<const float*>(a->weight);
  switch (a->out_dtype) {
    case 0: hipLaunchKernelGGL(rmsnorm_fwd_kernel<__bf16>, dim3(a->rows), dim3(kNormThreads), 0, s, x, w,
                               static_cast<__bf16*>(a->y), a->rstd, a->hidden, a->eps); break;
    case 1: hipLaunchKernelGGL(rmsnorm_fwd_kernel<_Float16>, dim3(a->rows), dim3(kNormThreads), 0, s, x, w,
                               static_cast<_Float16*>(a->y), a->rstd, a->hidden, a->eps); break;
    default: hipLaunchKernelGGL(rmsnorm_fwd_kernel<float>, dim3(a->rows), dim3(kNormThreads), 0, s, x, w,
                                static_cast<float*>(a->y), a->rstd, a->hidden, a->eps); break;
  }
  return hipGetLastError() == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}

extern "C" int32_t ssa_rmsnorm_bwd(const ssa_rmsnorm_bwd_args* a, void* stream) {
  if (a == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  const int32_t st = check_norm(a->x, a->weight, a->dy, a->rstd, a->rows, a->hidden, a->dy_dtype);
  if (st != SSA_OPS_OK) return st;
  if (a->dx == nullptr || a->dweight == nullptr || a->workspace == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  if (!aligned(a->dx, 16) || !aligned(a->workspace, 16) || !aligned(a->dy, 8)) return SSA_OPS_ERR_ALIGNMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int nparts = static_cast<int>((static_cast<int64_t>(a->rows) + kNormBwdRows - 1) / kNormBwdRows);
  // up to 64 rows there is one partial, which is dw: no third launch (1 x 2048 9.5 -> 7.4 us, 64 x
  // 512 9.7 -> 6.7)
  const bool whole = nparts == 1 && aligned(a->dweight, 16);
  float* part = whole ? a->dweight : a->workspace;
  switch (a->dy_dtype) {
    case 0: launch_norm_bwd<__bf16>(a, part, nparts, s); break;
    case 1: launch_norm_bwd<_Float16>(a, part, nparts, s); break;
    default: launch_norm_bwd<float>(a, part, nparts, s); break;
  }
  if (hipGetLastError() != hipSuccess) return SSA_OPS_ERR_LAUNCH;
  if (whole) return SSA_OPS_OK;
  hipLaunchKernelGGL(rmsnorm_dw_kernel, dim3((a->hidden + 63) / 64), dim3(1024), 0, s, a->workspace, a->dweight,
                     nparts, a->hidden);
  return hipGetLastError() == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}

extern "C" int32_t ssa_swiglu(const ssa_swiglu_args* a, void* stream) {
  if (a == nullptr || a->z == nullptr || a->out == nullptr || (a->backward && a->dh == nullptr))
    return SSA_OPS_ERR_NULL_POINTER;
  if (a->rows <= 0 || a->ffn <= 0 || a->ffn % 4 != 0) return SSA_OPS_ERR_SHAPE;
  const int64_t threads = static_cast<int64_t>(a->rows) * (a->ffn / 4);  // one per 4 outputs
  if ((threads + 255) / 256 > INT32_MAX) return SSA_OPS_ERR_SHAPE;
  if (a->dtype != 0 && a->dtype != 1) return SSA_OPS_ERR_DTYPE;
  if (!aligned(a->z, 8) || !aligned(a->out, 8) || (a->backward && !aligned(a->dh, 8))) return SSA_OPS_ERR_ALIGNMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int grid = static_cast<int>((threads + 255) / 256);
  if (a->dtype == 0)
    hipLaunchKernelGGL(swiglu_kernel<__bf16>, dim3(grid), dim3(256), 0, s, static_cast<const __bf16*>(a->z),
                       static_cast<const __bf16*>(a->dh), static_cast<__bf16*>(a->out), static_cast<int64_t>(a->rows),
                       a->ffn, a->backward);
  else
    hipLaunchKernelGGL(swiglu_kernel<_Float16>, dim3(grid), dim3(256), 0, s, static_cast<const _Float16*>(a->z),
                       static_cast<const _Float16*>(a->dh), static_cast<_Float16*>(a->out),
                       static_cast<int64_t>(a->rows), a->ffn, a->backward);
  return hipGetLastError() == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}

extern "C" int32_t ssa_cross_entropy(const ssa_cross_entropy_args* a, void* stream) {
  if (a == nullptr || a->logits == nullptr || a->labels == nullptr || a->lse == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  if (!a->backward && a->loss == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  if (a->backward && (a->scale == nullptr || a->dlogits == nullptr)) return SSA_OPS_ERR_NULL_POINTER;
  if (a->rows <= 0 || a->vocab <= 0 || a->vocab % 4 != 0) return SSA_OPS_ERR_SHAPE;
  if (a->dtype != 0 && a->dtype != 1) return SSA_OPS_ERR_DTYPE;
  if (!aligned(a->logits, 8) || (a->backward && !aligned(a->dlogits, 8))) return SSA_OPS_ERR_ALIGNMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t* lab = static_cast<const int64_t*>(a->labels);
  if (!a->backward) {
    if (a->dtype == 0)
      hipLaunchKernelGGL(xent_fwd_kernel<__bf16>, dim3(a->rows), dim3(256), 0, s,
                         static_cast<const __bf16*>(a->logits), lab, a->loss, a->lse, a->vocab);
    else
      hipLaunchKernelGGL(xent_fwd_kernel<_Float16>, dim3(a->rows), dim3(256), 0, s,
                         static_cast<const _Float16*>(a->logits), lab, a->loss, a->lse, a->vocab);
  } else {
    if (a->dtype == 0)
      hipLaunchKernelGGL(xent_bwd_kernel<__bf16>, dim3(a->rows), dim3(256), 0, s,
                         static_cast<const __bf16*>(a->logits), lab, a->lse, a->scale,
                         static_cast<__bf16*>(a->dlogits), a->vocab);
    else
      hipLaunchKernelGGL(xent_bwd_kernel<_Float16>, dim3(a->rows), dim3(256), 0, s,
                         static_cast<const _Float16*>(a->logits), lab, a->lse, a->scale,
                         static_cast<_Float16*>(a->dlogits), a->vocab);
  }
  return hipGetLastError() == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}

extern "C" int32_t ssa_embedding_bwd(const ssa_embedding_bwd_args* a, void* stream) {
  if (a == nullptr || a->ids == nullptr || a->dy == nullptr || a->grad == nullptr) return SSA_OPS_ERR_NULL_POINTER;
  if (a->tokens <= 0 || a->tokens > kEmbMaxTokens || a->vocab <= 0 || a->hidden <= 0 || a->hidden % 4 != 0)
    return SSA_OPS_ERR_SHAPE;
  if (!aligned(a->ids, 8) || !aligned(a->dy, 16) || !aligned(a->grad, 16)) return SSA_OPS_ERR_ALIGNMENT;
  const int64_t slabs = (static_cast<int64_t>(a->hidden) + kEmbCols - 1) / kEmbCols;
  const int64_t grid = (static_cast<int64_t>(a->vocab) + kEmbRows - 1) / kEmbRows * slabs;
  if (grid > INT32_MAX) return SSA_OPS_ERR_SHAPE;
  hipLaunchKernelGGL(embedding_bwd_kernel, dim3(static_cast<uint32_t>(grid)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const int64_t*>(a->ids), a->dy, a->grad, a->tokens,
                     a->vocab, a->hidden, static_cast<int>(slabs));
  return hipGetLastError() == hipSuccess ? SSA_OPS_OK : SSA_OPS_ERR_LAUNCH;
}
