// SSA attention forward and backward of bf16 / fp16 at head dim 256 (the
// largest the reference's Triton tiles hold, training/train/train_ssa_triton/
// SSA/ssa_triton_kernel.py:761-764; the functions are those of ssa_fwd.hip and
// ssa_bwd.hip).
//
// Products.  As in ssa_f32.hip a wave owns 32 rows, one per lane pair, their
// operand fragments in registers, and streams blocks of 32 rows of the other
// side through LDS: scores S = X_streamed X_own^T and outer products acc^T +=
// X_streamed^T w on v_mfma_f32_32x32x16.  The scores take the 16-bit inputs as
// they are (exact in fp32).  The weights w (P or dS') are fp32 and go in as the
// sum of two 16-bit halves, hi + lo, each multiplied (relative error 2^-17 in
// bf16, 2^-22 of a row's largest weight in fp16): no probability is rounded to 16
// bits.
//
// Schedule.  A wave's fragments and accumulators take 200 to 330 registers, so
// a SIMD holds one wave, which has to hide its own latencies.  An iteration has
// two phases.  Phase 1 computes the scores of the next block, a matrix
// instruction or two per tick with their LDS operands read four ticks ahead,
// beside one element of the current block's vector work in three stages on
// different elements (ticks are fenced, so the compiler keeps the mix).  Phase
// 2 is the outer product of the current block, 32 matrix instructions with
// their transposed operands read a group ahead.
//
// Measured at B = 1, H = 16, N = 2048 causal in bf16 (us; the vector-ALU kernels
// these replace, the same loops without the overlap, these): forward 3792, 126,
// 101; dK/dV 4622, 252, 195; dQ 4332, 125, 120.  The vector work is hidden
// (without it dQ takes 114); what is left is the K / V stream of a 64-row
// workgroup (64 KB a stage: without the loads 92) and each workgroup's start
// and end (28 of the 120 over two rounds).  128 rows a workgroup halve the
// stream but leave no second round to balance the causal blocks (129).
#include <utility>

#include "ssa_rows.hpp"

namespace ssa {

namespace {

constexpr int kD = 256, kNF = kD / 16, kND = kD / 32, kBB = BlockLayout<kD>::BLOCK;  // 16 KB per block
constexpr int kAhead = 4;  // ticks between an operand's LDS read and its use
constexpr int kTicks = kNF;

template <int... I, typename F>
__device__ __forceinline__ void for_ticks(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <typename T>
struct Mat16 {
  static constexpr bool F16 = !__is_same(T, __bf16);
  // fp16 holds 2^-24 .. 65504: the forward's probabilities are scaled up so that
  // the halves of all that matter in a row stay normal (against the lazily moved
  // running max at most PSUM); bf16 has fp32's range.
  static constexpr float FWD_SHIFT = F16 ? 4.f : 0.f;
  static constexpr float PSUM = F16 ? 32768.f : kPsumLimit;
  typedef typename Vec8<T>::type frag;
  typedef T v4 __attribute__((ext_vector_type(4)));
  struct Halves {
    frag hi[2], lo[2];
    __device__ __forceinline__ void put(int e, float w) {
      const T h = static_cast<T>(w);
      hi[e >> 3][e & 7] = h;
      lo[e >> 3][e & 7] = static_cast<T>(w - static_cast<float>(h));
    }
  };
  RowBase<kD> rb;
  TrBase<kD> tb;
  __device__ __forceinline__ explicit Mat16(int lane) : rb(lane & 31, lane >> 5), tb(lane) {}
  // fragment f of the row at `row`: columns 16 f + 8 hh + (0..7)
  __device__ static __forceinline__ frag load(const T* row, int f, int hh) {
    return load16<frag>(row + 16 * f + 8 * hh);
  }
  // Phase 1: s0 = X(lds0) own0^T and, with TWO, s1 = X(lds1) own1^T, with
  // tick(t) (a std::integral_constant) beside step t of each.
  template <bool TWO, typename Tick>
  __device__ __forceinline__ void scores(uint32_t lds0, uint32_t lds1, const frag* own0, const frag* own1, f32x16& s0,
                                         f32x16& s1, Tick tick) const {
    const RowBase<kD> r0 = at_tile(rb, lds0), r1 = at_tile(rb, TWO ? lds1 : lds0);
    frag a0[kAhead], a1[kAhead];
    auto read = [&](auto fc) {
      constexpr int f = decltype(fc)::value;
      if constexpr (f < kNF) {
        a0[f % kAhead] = tile_read_row<kD, frag>(r0, 0, f);
        if constexpr (TWO) a1[f % kAhead] = tile_read_row<kD, frag>(r1, 0, f);
      }
    };
    for_ticks(std::make_integer_sequence<int, kAhead>{}, read);
    __builtin_amdgcn_sched_barrier(0);
    for_ticks(std::make_integer_sequence<int, kTicks>{}, [&](auto tc) {
      constexpr int t = decltype(tc)::value;
      s0 = mfma32(a0[t % kAhead], own0[t], t == 0 ? f32x16{} : s0);
      if constexpr (TWO) s1 = mfma32(a1[t % kAhead], own1[t], t == 0 ? f32x16{} : s1);
      read(std::integral_constant<int, t + kAhead>{});
      tick(tc);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // Phase 2: acc^T += X(lds)^T (hi + lo): groups of two 32-column blocks.
  __device__ __forceinline__ void outer(uint32_t lds, const Halves& w, f32x16* acc) const {
    const TrBase<kD> t = at_tile(tb, lds);
    frag a[2][2];
    auto read = [&](auto gc) {
      constexpr int g = decltype(gc)::value;
      if constexpr (g < kND) {
        constexpr int ks = g / (kND / 2), d0 = 2 * (g % (kND / 2));
#pragma unroll
        for (int i = 0; i < 2; ++i)
          a[g & 1][i] = __builtin_shufflevector(tile_read_tr<kD, v4>(t, 0, ks, 0, d0 + i),
                                                tile_read_tr<kD, v4>(t, 0, ks, 1, d0 + i), 0, 1, 2, 3, 4, 5, 6, 7);
      }
    };
    read(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    for_ticks(std::make_integer_sequence<int, kND>{}, [&](auto gc) {
      constexpr int g = decltype(gc)::value, ks = g / (kND / 2), d0 = 2 * (g % (kND / 2));
      read(std::integral_constant<int, g + 1>{});
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[d0 + i] = mfma32(a[g & 1][i], w.hi[ks], acc[d0 + i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[d0 + i] = mfma32(a[g & 1][i], w.lo[ks], acc[d0 + i]);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
};

// Weights of any size on the fp16 halves: a power of two per owned row (a lane
// pair), set by its first block with a nonzero weight and lowered (exactly)
// whenever a larger one comes, keeps the row's largest weight seen below 2^15;
// the accumulators hold the scaled sums.  Each row keeps 2^-22 of its own
// weights that way, however large its neighbours' are (one scale for the 32 rows
// of a wave left a row of 2^-28 of their size 2^-10; the wave-wide maximum
// also took a shuffle per step: fp16 backward of 2 x 8/2 x 2048 causal 895 ->
// 718 us).  bf16 has fp32's range and needs none.
template <typename T>
struct WeightScale {
  float s = 0.f;
  __device__ __forceinline__ void apply(float* w, f32x16* acc) {
    float a = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) a = fmaxf(a, fabsf(w[r]));
    a = fminf(pair_max(a), 3.0e38f);
    const bool move = a * s > 32768.f || (s == 0.f && a > 0.f);
    if (__any(move)) {
      int ex = 0;  // a = m 2^ex, m in [1/2, 1)
      (void)frexpf(a, &ex);
      const float sn = move ? ldexpf(1.f, min(15 - ex, 60)) : s;
      const float f = s != 0.f ? sn / s : 1.f;
#pragma unroll
      for (int d = 0; d < kND; ++d) acc[d] *= f;
      s = sn;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) w[r] *= s;
  }
  __device__ __forceinline__ float inverse() const { return s != 0.f ? 1.f / s : 0.f; }
};

// Rows per workgroup (forward, dQ): 64, two waves each on alternate 32-row
// blocks of a 64-row stage, so that one sequence fills the chip.
constexpr int kKW = 2, kQW = 2, kBM = 32 * kQW, kBN = 32 * kKW;

// ---------------------------------------------------------------------------
// Forward.  K in two slots and V in two, turned over separately: iteration st
// reads K of stage st + 1 and V of stage st.  The running max moves lazily, as
// in ssa_fwd.hip: P is computed against it, and one test of the lane's sum of
// p bounds them all (and catches inf and NaN); the rare block that fails it
// takes its true max and recomputes P from the scores.
template <typename T, bool CAUSAL>
__global__ __launch_bounds__(256) void ssa_fwd_d256_kernel(FwdParams p) {
  using M = Mat16<T>;
  typedef typename M::frag frag;
  using Plan = RowPlan<kD, 2, CAUSAL, kKW>;
  using Loads = RowLoads256<CAUSAL, kKW, 2, 2>;
  __shared__ __attribute__((aligned(1024))) char smem[Loads::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int kw = wave % kKW, qw = wave / kKW;
  const int block = folded_block();
  if (block >= Plan::grid(p)) return;
  const Plan pl(p, Plan::place(p, block));  // dispatch and K / V loads (ssa_rows_plan.hpp)
  const SeqView& sv = pl.sv;
  const int b = pl.b, h = pl.h, N = pl.N, nst = pl.nst;
  if (pl.empty()) return;  // packed: past the end of a shorter document
  const Loads ld(p, pl, lane, wave);
  const int wq0 = pl.q0 + 32 * qw, qrow = wq0 + l32;
  const T* qg = reinterpret_cast<const T*>(head_rows<2>(sv, p.q, b, h));
  const T* kg = reinterpret_cast<const T*>(ld.k.g);
  const T* vg = reinterpret_cast<const T*>(ld.v.g);
  const float n = *p.n_ptr, c = p.scale * *p.b_ptr;
  const uint32_t lds0 = lds_addr(smem);
  auto k_at = [&](int st) { return Loads::k_at(lds0, st & 1); };
  auto v_at = [&](int st) { return Loads::v_at(lds0, st & 1); };
  auto load_k = [&](int st) { ld.load_k(pl, st, st & 1, lds0, wave); };
  auto load_v = [&](int st) { ld.load_v(pl, st, st & 1, lds0, wave); };
  load_k(0);
  load_k(1);
  load_v(0);
  const M mat(lane);
  frag qf[kNF];
#pragma unroll
  for (int f = 0; f < kNF; ++f) qf[f] = qrow < N ? M::load(qg + qrow * p.q.ss, f, hh) : zero8<frag>();
  f32x16 acc[kND];
#pragma unroll
  for (int d = 0; d < kND; ++d) acc[d] = f32x16{};
  float m = -INFINITY, l = 0.f;
  f32x16 s = f32x16{}, sn = f32x16{}, unused;
  auto active = [&](int st) {  // a prefix of the stages
    const int k0 = st * kBN + 32 * kw;
    return st < nst && k0 < N && wq0 < N && (!CAUSAL || k0 <= wq0 + 31);
  };
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (active(0)) mat.template scores<false>(k_at(0) + kw * kBB, 0, qf, qf, s, unused, [](auto) {});
  for (int st = 0; st < nst; ++st) {
    if (st > 0) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // K(st + 1) and V(st) have landed; K(st) and V(st - 1) are consumed
    load_k(st + 2);
    load_v(st + 1);
    if (!active(st)) continue;
    const int k0 = st * kBN + 32 * kw;
    const int last = (CAUSAL ? min(qrow, N - 1) : N - 1) - k0 - 4 * hh;  // crow(r, 0) <= last: a valid key
    const float base = M::FWD_SHIFT - m;
    typename M::Halves w;
    float Lv[16], pv[16], sum = 0.f;
    auto elements = [&](int t, auto masked) {
      auto A = [&](int e) {
        Lv[e] = fast_log2(fmaf(c, fabsf(s[e]), 1.f));
        pin(Lv[e]);
      };
      auto B = [&](int e) {
        pv[e] = fast_exp2(fmaf(n, copysignf(Lv[e], s[e]), base));
        if constexpr (decltype(masked)::value) pv[e] = crow(e, 0) <= last ? pv[e] : 0.f;
        pin(pv[e]);
      };
      auto C = [&](int e) {
        sum += pv[e];
        w.put(e, pv[e]);
      };
      if (t < 16) A(t);
      if (t >= 1 && t < 17) B(t - 1);
      if (t >= 2) C(t - 2);
    };
    if (active(st + 1)) {  // then this block has no masked key
      mat.template scores<false>(k_at(st + 1) + kw * kBB, 0, qf, qf, sn, unused,
                                 [&](auto tc) { elements(decltype(tc)::value, std::false_type{}); });
      elements(16, std::false_type{});
      elements(17, std::false_type{});
    } else {
#pragma unroll
      for (int t = 0; t < 18; ++t) elements(t, std::true_type{});
    }
    if (__any(!(sum <= M::PSUM))) {  // rare: the running max moves
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float t2 = n * ssa_sl(s[e], fmaf(c, fabsf(s[e]), 1.f));
        mx = fmaxf(mx, crow(e, 0) <= last ? t2 : -INFINITY);
      }
      mx = fmaxf(m, pair_max(mx));
      const float ref = mx == -INFINITY ? 0.f : mx;
      const float alpha = fast_exp2(m - ref);
      l *= alpha;
#pragma unroll
      for (int d = 0; d < kND; ++d) acc[d] *= alpha;
      m = mx;
      sum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float t2 = n * ssa_sl(s[e], fmaf(c, fabsf(s[e]), 1.f));
        const float pe = crow(e, 0) <= last ? fast_exp2(t2 - ref + M::FWD_SHIFT) : 0.f;
        sum += pe;
        w.put(e, pe);
      }
    }
    l += sum;
    mat.outer(v_at(st) + kw * kBB, w, acc);
    s = sn;
  }
  l = pair_sum(l);
  __syncthreads();  // every wave is past the ring (no load in flight)
  float* ml = reinterpret_cast<float*>(smem);  // [4 waves][m, l][32]
  if (hh == 0) {
    ml[(2 * wave) * 32 + l32] = m;
    ml[(2 * wave + 1) * 32 + l32] = l;
  }
  __syncthreads();
  const float own = m;
  l = 0.f;
#pragma unroll
  for (int i = 0; i < kKW; ++i) m = fmaxf(m, ml[2 * (qw * kKW + i) * 32 + l32]);
  const float ref = m == -INFINITY ? 0.f : m;
#pragma unroll
  for (int i = 0; i < kKW; ++i)
    l += ml[(2 * (qw * kKW + i) + 1) * 32 + l32] * fast_exp2(ml[2 * (qw * kKW + i) * 32 + l32] - ref);
  const float alpha = fast_exp2(own - ref);
#pragma unroll
  for (int d = 0; d < kND; ++d) acc[d] *= alpha;
  merge_parts<kND, kKW>(acc, reinterpret_cast<float*>(smem), qw, kw, lane);
  __syncthreads();
  if (kw == 0 && wq0 < N) {
    const bool bad = row_nonfinite<kND>(acc);
    T* og = static_cast<T*>(const_cast<void*>(p.o.ptr)) + sv.off(p.o, b) + h * p.o.sh;
    store_rows_via_lds<T, kD>(acc, 1.f / l, [&](int r) { return lds0 + qw * (32 * kD * 2) + r * (kD * 2); },
                              og + static_cast<int64_t>(wq0) * p.o.ss, p.o.ss, N - wq0, lane);
    if (SSA_RARE(__any(bad)) && bad && qrow < N) {
      __builtin_amdgcn_s_waitcnt(0);  // after the row's first store
      row_fwd<T, kD>(og + qrow * p.o.ss, 1.f / l, qg + qrow * p.q.ss, kg, p.k.ss, vg, p.v.ss, CAUSAL ? qrow : N - 1, n,
                     c, ref - M::FWD_SHIFT, hh);
    }
    if (hh == 0 && qrow < N) p.m[sv.mrow(b, h, p.Hq, p.T, p.N) + qrow] = m + (log2f(l) - M::FWD_SHIFT);
  }
}

// ---------------------------------------------------------------------------
// dK (with dn and db) or dV of 128 keys of one (batch, kv-head): 4 waves of 32
// keys, Q / dO blocks of 32 queries with their M and Delta over every q-head of
// the group.  The accumulators of both do not fit one wave beside the K and V
// fragments, so half of the grid computes dK (three products a block) and half
// dV (two); the operand of the outer product is held for one block longer.
// Per valid pair, as in ssa_bwd.hip: P = exp2(n sL - M), dT = P (dP - Delta),
// dS' = dT / (1 + c|x|).
template <typename T, bool CAUSAL, bool DK>
__device__ __forceinline__ void dkdv_d256_body(const BwdParams& p, char* smem, float (*red)[4], int block) {
  using M = Mat16<T>;
  typedef typename M::frag frag;
  using Plan = KeyPlan<kD, 2, CAUSAL, 1, 4>;
  using Ring = KeyRing256<DK>;
  constexpr int RQ = Ring::RQ, RD = Ring::RD;  // ring slots of Q and of dO
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int nkb = dkdv_key_blocks(p.N);
  const Plan pl(p, Plan::place(p, block));  // dispatch and Q / dO loads (ssa_rows_plan.hpp)
  const SeqView& sv = pl.sv;
  const int kb = pl.kb, b = pl.b, hk = pl.hk, bhk = pl.bhk, N = pl.N, k0 = pl.k0;
  const int64_t PP = static_cast<int64_t>(p.B) * p.Hkv * nkb;
  if (pl.empty()) {  // packed: past the end of a shorter document
    if (DK && tid == 0) {
      p.partials[static_cast<int64_t>(bhk) * nkb + kb] = 0.f;
      p.partials[PP + static_cast<int64_t>(bhk) * nkb + kb] = 0.f;
    }
    return;
  }
  const int k0w = k0 + 32 * wave, key = k0w + l32;
  const T* kg = static_cast<const T*>(p.k.ptr) + sv.off(p.k, b) + hk * p.k.sh;
  const T* vg = static_cast<const T*>(p.v.ptr) + sv.off(p.v, b) + hk * p.v.sh;
  const float n = *p.n_ptr, bv = *p.b_ptr, c = p.scale * bv;
  const uint32_t lds0 = lds_addr(smem);
  const LoadLane llq(lane, wave, p.q.ss), lld(lane, wave, p.dout.ss);
  const int qstart = pl.qstart, nst = pl.nst;
  // ring slots of stage st: the slot indices of stages st, st + 1 and st + 2
  // are kept, not divided out
  auto q_at = [&](int slot) { return Ring::q_at(lds0, slot); };
  auto d_at = [&](int slot) { return Ring::d_at(lds0, slot); };
  auto md_at = [&](int slot) { return Ring::md_at(lds0, slot); };
  Ring ring(qstart);  // the next stage to load
  auto load_next = [&]() { ring.load_next(p, pl, lds0, llq, lld, wave, lane); };
  load_next();
  load_next();
  const M mat(lane);
  frag kf[kNF], vf[DK ? kNF : 1];
#pragma unroll
  for (int f = 0; f < kNF; ++f) {
    kf[f] = key < N ? M::load(kg + key * p.k.ss, f, hh) : zero8<frag>();
    if constexpr (DK) vf[f] = key < N ? M::load(vg + key * p.v.ss, f, hh) : zero8<frag>();
  }
  f32x16 acc[kND];
#pragma unroll
  for (int d = 0; d < kND; ++d) acc[d] = f32x16{};
  float dn_acc = 0.f, dn_c = 0.f, db_acc = 0.f, db_c = 0.f;  // Kahan sums over the blocks' sums
  WeightScale<T> ws;
  f32x16 s = f32x16{}, dp = f32x16{}, sn = f32x16{}, dpn = f32x16{};
  // a block whose queries all precede this wave's keys (or no keys) has no work
  auto active = [&](int q0) { return k0w < N && (!CAUSAL || q0 + 31 >= k0w); };
  int q0 = qstart, qs = 0, ds = 0, ms = 0;  // stage st: first query, slots
  auto next_scores = [&](int qslot, int dslot, auto tick) {
    if constexpr (DK)
      mat.template scores<true>(q_at(qslot), d_at(dslot), kf, vf, sn, dpn, tick);
    else
      mat.template scores<false>(q_at(qslot), 0, kf, kf, sn, dpn, tick);
  };
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (active(q0)) {
    next_scores(0, 0, [](auto) {});
    s = sn;
    dp = dpn;
  }
  for (int st = 0; st < nst; ++st) {
    if (st > 0) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // stage st + 1 has landed; what stage st + 2 overwrites is consumed
    load_next();
    const int q1 = q0 + 32 >= N ? qstart : q0 + 32;  // first query of stage st + 1
    const int qs1 = qs + 1 == RQ ? 0 : qs + 1, ds1 = ds + 1 == RD ? 0 : ds + 1;
    const bool now = active(q0), next = st + 1 < nst && active(q1);
    if (now) {
      f32x4_t mv[4], dl[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mv[j] = lds_read_f4(md_at(ms) + (8 * j + 4 * hh) * 4);
        if constexpr (DK) dl[j] = lds_read_f4(md_at(ms) + 128 + (8 * j + 4 * hh) * 4);
      }
      typename M::Halves w;
      float Lv[16], rv[16], pv[16], wv[16], tdn = 0.f, tdb = 0.f;
      auto elements = [&](int t, auto masked) {
        auto A = [&](int e) {
          const float u1 = fmaf(c, fabsf(s[e]), 1.f);
          Lv[e] = fast_log2(u1);
          pin(Lv[e]);
          if constexpr (DK) {
            rv[e] = fast_rcp(u1);
            pin(rv[e]);
          }
        };
        auto B = [&](int e) {
          Lv[e] = copysignf(Lv[e], s[e]);
          pv[e] = fast_exp2(fmaf(n, Lv[e], -mv[e >> 2][e & 3]));
          if constexpr (decltype(masked)::value) {
            const int qi = q0 + crow(e, hh);
            pv[e] = qi < N && key < N && (!CAUSAL || key <= qi) ? pv[e] : 0.f;
          }
          pin(pv[e]);
        };
        auto C = [&](int e) {
          if constexpr (DK) {
            const float dt = pv[e] * (dp[e] - dl[e >> 2][e & 3]);
            wv[e] = dt * rv[e];
            tdn = fmaf(dt, Lv[e], tdn);
            tdb = fmaf(wv[e], s[e], tdb);
          } else {
            wv[e] = pv[e];
          }
          if constexpr (!M::F16) w.put(e, wv[e]);
        };
        if (t < 16) A(t);
        if (t >= 1 && t < 17) B(t - 1);
        if (t >= 2) C(t - 2);
      };
      auto block_of = [&](auto masked) {
        if (next)
          next_scores(qs1, ds1, [&](auto tc) { elements(decltype(tc)::value, masked); });
        else
          for_ticks(std::make_integer_sequence<int, 16>{}, [&](auto tc) { elements(decltype(tc)::value, masked); });
        elements(16, masked);
        elements(17, masked);
      };
      if (q0 + 32 > N || k0w + 32 > N || (CAUSAL && k0w + 31 > q0))
        block_of(std::true_type{});
      else
        block_of(std::false_type{});
      if constexpr (DK) {
        const float y = tdn - dn_c, t = dn_acc + y;
        dn_c = (t - dn_acc) - y;
        dn_acc = t;
        const float y2 = tdb - db_c, t2 = db_acc + y2;
        db_c = (t2 - db_acc) - y2;
        db_acc = t2;
      }
      if constexpr (M::F16) {
        ws.apply(wv, acc);
#pragma unroll
        for (int e = 0; e < 16; ++e) w.put(e, wv[e]);
      }
      mat.outer(DK ? q_at(qs) : d_at(ds), w, acc);
    } else if (next) {
      next_scores(qs1, ds1, [](auto) {});
    }
    s = sn;
    dp = dpn;
    q0 = q1;
    qs = qs1;
    ds = ds1;
    ms = ms == 2 ? 0 : ms + 1;
  }
  if (key < N) {
    const Tensor4& o = DK ? p.dk : p.dv;
    T* row = static_cast<T*>(const_cast<void*>(o.ptr)) + sv.off(o, b) + hk * o.sh + key * o.ss;
    float scale = DK ? p.scale * n * bv : 1.f;
    const float whole = scale;
    if constexpr (M::F16) scale *= ws.inverse();
    const bool bad = row_nonfinite<kND>(acc, DK ? dn_acc + db_acc : 0.f);
    if (!bad) store_own<T, kD>(acc, scale, row, hh);
    if (SSA_RARE(__any(bad)) && bad) {
      dn_c = db_c = 0.f;
      row_dkdv<T, kD, CAUSAL>(p, sv, b, hk, key, n, c, DK ? row : nullptr, whole, DK ? nullptr : row, dn_acc, db_acc,
                              hh);
      if (hh != 0) dn_acc = db_acc = 0.f;  // both lanes of the pair have the whole sums
    }
  }
  if constexpr (DK) {
    // dn / db partial of this key block: lane butterfly, then the waves in order
    float pdn = dn_acc - dn_c, pdb = db_acc - db_c;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      pdn += __shfl_xor(pdn, off, 64);
      pdb += __shfl_xor(pdb, off, 64);
    }
    if (lane == 0) {
      red[0][wave] = pdn;
      red[1][wave] = pdb;
    }
    __syncthreads();
    if (tid == 0) {
      p.partials[static_cast<int64_t>(bhk) * nkb + kb] =
          kLn2 * ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3]));
      p.partials[PP + static_cast<int64_t>(bhk) * nkb + kb] =
          n * p.scale * ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
    }
  }
}

template <typename T, bool CAUSAL>
__global__ __launch_bounds__(256) void ssa_bwd_dkdv_d256_kernel(BwdParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[KeyRing256<true>::LDS_BYTES];
  __shared__ float red[2][4];
  // the dK workgroups (three products per block) before the lighter dV ones
  const int grid = dkdv_key_blocks(p.N) * p.B * p.Hkv, block = folded_block();
  if (block < grid)
    dkdv_d256_body<T, CAUSAL, true>(p, smem, red, block);
  else if (block < 2 * grid)
    dkdv_d256_body<T, CAUSAL, false>(p, smem, red, block - grid);
}

// ---------------------------------------------------------------------------
// dQ: the scores and dP are recomputed (dQ += scale n b dS' k).  K in three
// slots (read by the scores of its stage and, one iteration later, by the
// outer product), V in two: all 160 KB.
template <typename T, bool CAUSAL>
__global__ __launch_bounds__(256) void ssa_bwd_dq_d256_kernel(BwdParams p) {
  using M = Mat16<T>;
  typedef typename M::frag frag;
  using Plan = RowPlan<kD, 2, CAUSAL, kKW>;
  using Loads = RowLoads256<CAUSAL, kKW, 3, 2>;
  __shared__ __attribute__((aligned(1024))) char smem[Loads::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int kw = wave % kKW, qw = wave / kKW;
  const int block = folded_block();
  if (block >= Plan::grid(p)) return;
  if (p.fuse_reduce && block == 0) {  // the backward's dn / db sums, before the first load (reduce_partials_body)
    reduce_partials_body(p.partials, static_cast<int64_t>(p.B) * p.Hkv * dkdv_key_blocks(p.N), p.dn, p.db,
                         reinterpret_cast<float(*)[256]>(smem), threadIdx.x);
    __syncthreads();
  }
  const Plan pl(p, Plan::place(p, block));
  const SeqView& sv = pl.sv;
  const int b = pl.b, h = pl.h, N = pl.N, nst = pl.nst;
  if (pl.empty()) return;  // packed: past the end of a shorter document
  const Loads ld(p, pl, lane, wave);
  const int wq0 = pl.q0 + 32 * qw, qrow = wq0 + l32;
  const T* qg = reinterpret_cast<const T*>(head_rows<2>(sv, p.q, b, h));
  const T* dog = reinterpret_cast<const T*>(head_rows<2>(sv, p.dout, b, h));
  const T* kg = reinterpret_cast<const T*>(ld.k.g);
  const T* vg = reinterpret_cast<const T*>(ld.v.g);
  const int64_t mr = sv.mrow(b, h, p.Hq, p.T, p.N);
  const float n = *p.n_ptr, bv = *p.b_ptr, c = p.scale * bv;
  const uint32_t lds0 = lds_addr(smem);
  auto k_at = [&](int slot) { return Loads::k_at(lds0, slot) + kw * kBB; };
  auto v_at = [&](int st) { return Loads::v_at(lds0, st & 1) + kw * kBB; };
  int ls = 0, lk_slot = 0;  // the next stage to load
  auto load_next = [&]() {
    ld.load_k(pl, ls, lk_slot, lds0, wave);
    ld.load_v(pl, ls, ls & 1, lds0, wave);
    ++ls;
    lk_slot = lk_slot == 2 ? 0 : lk_slot + 1;
  };
  load_next();
  load_next();
  const M mat(lane);
  frag qf[kNF], dof[kNF];
#pragma unroll
  for (int f = 0; f < kNF; ++f) {
    qf[f] = qrow < N ? M::load(qg + qrow * p.q.ss, f, hh) : zero8<frag>();
    dof[f] = qrow < N ? M::load(dog + qrow * p.dout.ss, f, hh) : zero8<frag>();
  }
  const float mi = qrow < N ? p.m[mr + qrow] : 0.f, di = qrow < N ? p.delta[mr + qrow] : 0.f;
  f32x16 dq[kND];
#pragma unroll
  for (int d = 0; d < kND; ++d) dq[d] = f32x16{};
  WeightScale<T> ws;
  f32x16 s = f32x16{}, dp = f32x16{}, sn = f32x16{}, dpn = f32x16{};
  auto active = [&](int st) {  // a prefix of the stages
    const int k0 = st * kBN + 32 * kw;
    return st < nst && k0 < N && wq0 < N && (!CAUSAL || k0 <= wq0 + 31);
  };
  int ks = 0;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (active(0)) mat.template scores<true>(k_at(0), v_at(0), qf, dof, s, dp, [](auto) {});
  for (int st = 0; st < nst; ++st) {
    if (st > 0) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // stage st + 1 has landed; K(st - 1) and V(st) are consumed
    load_next();
    const int ks1 = ks == 2 ? 0 : ks + 1;
    if (active(st)) {
      const int k0 = st * kBN + 32 * kw;
      const int last = (CAUSAL ? min(qrow, N - 1) : N - 1) - k0 - 4 * hh;  // crow(r, 0) <= last: a valid key
      typename M::Halves w;
      float Lv[16], rv[16], pv[16], wv[16];
      auto elements = [&](int t, auto masked) {
        auto A = [&](int e) {
          const float u1 = fmaf(c, fabsf(s[e]), 1.f);
          Lv[e] = fast_log2(u1);
          rv[e] = fast_rcp(u1);
          pin(Lv[e]);
          pin(rv[e]);
        };
        auto B = [&](int e) {
          pv[e] = fast_exp2(fmaf(n, copysignf(Lv[e], s[e]), -mi));
          if constexpr (decltype(masked)::value) pv[e] = crow(e, 0) <= last ? pv[e] : 0.f;
          pin(pv[e]);
        };
        auto C = [&](int e) {
          wv[e] = pv[e] * (dp[e] - di) * rv[e];
          if constexpr (!M::F16) w.put(e, wv[e]);
        };
        if (t < 16) A(t);
        if (t >= 1 && t < 17) B(t - 1);
        if (t >= 2) C(t - 2);
      };
      if (active(st + 1)) {  // then this block has no masked key
        mat.template scores<true>(k_at(ks1), v_at(st + 1), qf, dof, sn, dpn,
                                  [&](auto tc) { elements(decltype(tc)::value, std::false_type{}); });
        elements(16, std::false_type{});
        elements(17, std::false_type{});
      } else {
#pragma unroll
        for (int t = 0; t < 18; ++t) elements(t, std::true_type{});
      }
      if constexpr (M::F16) {
        ws.apply(wv, dq);
#pragma unroll
        for (int e = 0; e < 16; ++e) w.put(e, wv[e]);
      }
      mat.outer(k_at(ks), w, dq);
      s = sn;
      dp = dpn;
    }
    ks = ks1;
  }
  if constexpr (M::F16) {  // bring the sharing waves' sums to true scale
    const float inv = ws.inverse();
#pragma unroll
    for (int d = 0; d < kND; ++d) dq[d] *= inv;
  }
  merge_parts<kND, kKW>(dq, reinterpret_cast<float*>(smem), qw, kw, lane);
  __syncthreads();
  if (kw == 0 && wq0 < N) {
    const bool bad = row_nonfinite<kND>(dq);
    T* dqg = static_cast<T*>(const_cast<void*>(p.dq.ptr)) + sv.off(p.dq, b) + h * p.dq.sh;
    store_rows_via_lds<T, kD>(dq, p.scale * n * bv, [&](int r) { return lds0 + qw * (32 * kD * 2) + r * (kD * 2); },
                              dqg + static_cast<int64_t>(wq0) * p.dq.ss, p.dq.ss, N - wq0, lane);
    if (SSA_RARE(__any(bad)) && bad && qrow < N) {
      __builtin_amdgcn_s_waitcnt(0);  // after the row's first store
      row_dq<T, kD>(dqg + qrow * p.dq.ss, p.scale * n * bv, qg + qrow * p.q.ss, dog + qrow * p.dout.ss, kg, p.k.ss, vg,
                    p.v.ss, CAUSAL ? qrow : N - 1, n, c, mi, di, hh);
    }
  }
}

}  // namespace

#define SSA_D256_LAUNCH(KERNEL, GRID)                                                                    \
  do {                                                                                                   \
    if (D != kD || (dtype != 0 && dtype != 1)) return hipErrorInvalidValue;                               \
    if (dtype == 0 && causal) hipLaunchKernelGGL((KERNEL<__bf16, true>), GRID, dim3(256), 0, s, p);       \
    else if (dtype == 0) hipLaunchKernelGGL((KERNEL<__bf16, false>), GRID, dim3(256), 0, s, p);           \
    else if (causal) hipLaunchKernelGGL((KERNEL<_Float16, true>), GRID, dim3(256), 0, s, p);              \
    else hipLaunchKernelGGL((KERNEL<_Float16, false>), GRID, dim3(256), 0, s, p);                         \
    return hipGetLastError();                                                                            \
  } while (0)

hipError_t launch_fwd_d256(const FwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  SSA_D256_LAUNCH(ssa_fwd_d256_kernel, folded_grid((p.N + kBM - 1) / kBM * p.B * p.Hq, 256));
}

hipError_t launch_bwd_dkdv_d256(const BwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  SSA_D256_LAUNCH(ssa_bwd_dkdv_d256_kernel, folded_grid(dkdv_key_blocks(p.N) * p.B * p.Hkv * 2, 256));
}

hipError_t launch_bwd_dq_d256(const BwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  SSA_D256_LAUNCH(ssa_bwd_dq_d256_kernel, folded_grid((p.N + kBM - 1) / kBM * p.B * p.Hq, 256));
}

}  // namespace ssa
