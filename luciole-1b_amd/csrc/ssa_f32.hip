// SSA attention forward and backward of fp32 inputs at every head dim, on the
// matrix cores, with every product and sum in fp32 (bf16 / fp16: ssa_fwd.hip,
// ssa_bwd*.hip and, at head dim 256, ssa_d256.hip).
//
// The reference runs its Triton kernels on fp32 tensors with fp32 operands in
// the dot products (MATMUL_PRECISION = tl.float32,
// training/train/train_ssa_triton/SSA/ssa_triton_kernel.py:766-772, 819-825)
// and checks them to atol 5e-4 / rtol 1e-3 and scalar 5e-5 + 1e-4 |ref|
// (check_ssa_triton_parity.py:1064-1069), a bar that no bf16 rounding of the
// operands meets.  Masks, GQA, packed sequences and the dn / db partials (one
// per 128-key block, the layout ssa_reduce_partials_kernel sums) are those of
// the other kernels; the reference accepts every power-of-two head dim
// (ssa_triton_kernel.py:761-764), and head dim 256 is the largest its Triton
// tiles hold.
//
// One structure for all three kernels.  A wave owns 32 rows (queries in the
// forward and dQ, keys in dK/dV), one per lane pair (l, l + 32), and holds
// their operand fragments in registers; the other side streams through LDS in
// blocks of 32 rows (direct-to-LDS loads, the next stage in flight under the
// current one).  Two operations do all the work (Mat below):
//   scores: S = X_streamed X_own^T, the streamed row on the accumulator's row
//           axis, so lane l holds the scores of its own row with streamed
//           rows crow(r, hh);
//   outer:  acc^T += X_streamed^T w, w the 16 weights (P or dS') of the lane's
//           own row, straight from the accumulator they were computed in.
// Both run on v_mfma_f32_32x32x2_f32, whose products and sums are fp32.
//
// What bounds it: an fp32 MFMA takes 64 cycles for 4096 FLOPs, so the fp32
// kernels run at the rate of the matrix cores' fp32 form (138 TFLOP/s in a
// large library product) and need little of LDS or the vector ALU.  The
// streamed rows are split over the waves of a workgroup (kw = 2 or 4 blocks
// at a time) up to head dim 128, so that a workgroup owns 32 or 64 rows: a
// grid of one sequence then fills the chip, and causal blocks balance.
// Measured (us, the earlier vector-ALU kernels -> these): fp32, B = 1, H = 16,
// N = 1024, D = 64 causal: forward 376 -> 43, dK/dV 498 -> 124, dQ 380 -> 53.
// Head dim 256 (K, V, Q or dO fragments and accumulators of 128 registers each):
// 16 x 2048 causal forward 3800 -> 614, backward 8920 -> 1950; 16 x 4096 14700 ->
// 1310 and 35500 -> 5440.  It fits one wave's registers with the scores in VGPRs
// (_build.py) and LDS reads kept near their use, but for 91 spills of the causal
// dQ; without either it spilled up to 340 (751 and 2350 at 2048).
#include "ssa_rows.hpp"

namespace ssa {

namespace {

// The two matrix operations on a streamed block of 32 rows x D in LDS, stored
// in the block-chunk-major layout of ssa_tile.hpp (LD: its width in 16-bit
// columns, so fp32 blocks are 2 D wide and the same loaders move them).
template <int D>
struct Mat {
  static constexpr int LD = 2 * D, BLOCK = BlockLayout<LD>::BLOCK, ND = D >= 32 ? D / 32 : 1, NF = D / 8;
  typedef f32x4 frag;
  RowBase<LD> rb;
  uint32_t ob[2];
  // ob: streamed row 8 a + 4 hh + e, column 32 db + l32 sits in chunk c = 8 db +
  // l32 / 4 at row position (row ^ 4 (c & 3)); the XOR splits into the lane's
  // part and the parity of a, so every fetch is ob[a & 1] plus an immediate.
  // Head dim 16 has four chunks: lanes 16-31 fetch copies, and the accumulator
  // rows they feed (columns 16-31) are never stored.
  __device__ __forceinline__ explicit Mat(int lane) : rb(lane & 31, lane >> 5) {
    const int l32 = lane & 31, hh = lane >> 5;
    const int c = (l32 >> 2) & (D / 4 >= 8 ? 7 : D / 4 - 1), x = c & 3;
#pragma unroll
    for (int par = 0; par < 2; ++par)
      ob[par] = static_cast<uint32_t>(c * 512 + (8 * (par ^ (x >> 1)) + 4 * (hh ^ (x & 1))) * 16 + (l32 & 3) * 4);
  }
  // fragment f: columns 8 f + 4 hh + (0..3), one MFMA step each
  __device__ static __forceinline__ frag load(const float* row, int f, int hh) { return ld4(row + 8 * f + 4 * hh); }
  // Chains of 32 columns added in a tree: one chain over the row was off by more
  // than the vector-ALU kernels' partial sums (against 64 bits, N = 64 causal, of
  // the norm: dq at head dim 128 3.4e-7 and 256 4.4e-7 in one chain, 2.5e-7 and
  // 2.7e-7 so, 2.6e-7 and 2.8e-7 there).
  template <int F0, int N>
  __device__ __forceinline__ f32x16 chain(const RowBase<LD>& r, const frag* own) const {
    if constexpr (N > 4) {
      const f32x16 a = chain<F0, N / 2>(r, own);
      // head dim 256 fills the registers: no LDS reads ahead over a chain or an outer step
      if constexpr (D >= 256) __builtin_amdgcn_sched_barrier(0);
      return a + chain<F0 + N / 2, N / 2>(r, own);
    } else {
      f32x16 s = f32x16{};
#pragma unroll
      for (int f = F0; f < F0 + N; ++f) {
        const f32x4 a = tile_read_row<LD, f32x4>(r, 0, f);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], own[f][e], s, 0, 0, 0);
      }
      return s;
    }
  }
  __device__ __forceinline__ f32x16 scores(uint32_t lds, const frag* own) const {
    return chain<0, NF>(at_tile(rb, lds), own);
  }
  __device__ __forceinline__ void outer(uint32_t lds, const float* w, f32x16* acc) const {
    const uint32_t b[2] = {opaque(ob[0] + lds), opaque(ob[1] + lds)};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (D >= 256) __builtin_amdgcn_sched_barrier(0);
      const uint32_t imm = (r >> 3) * 256 + (r & 3) * 16;
#pragma unroll
      for (int db = 0; db < ND; ++db) {
        const float a =
            *(const __attribute__((address_space(3))) float*)(uintptr_t)(b[(r >> 2) & 1] + imm + db * 4096);
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, w[r], acc[db], 0, 0, 0);
      }
    }
  }
};

template <int D>
struct Cfg : SplitF32<D> {
  static constexpr int QW = 4 / SplitF32<D>::KW;  // waves on different rows (forward, dQ): 32 QW rows per workgroup
  static constexpr int BM = 32 * QW, BN = 32 * SplitF32<D>::KW;
  static constexpr int DKDV_THREADS = 256 * SplitF32<D>::QS;  // workgroups own 128 keys, the unit of the partials
};

// ---------------------------------------------------------------------------
// Forward: BM queries of one (batch, q-head), K / V streamed BN keys a stage.
// Online softmax in base 2 with the running max moved lazily (kRescaleTau; of 32
// rows some exact max moves in most tiles; M is exact either way); the waves
// that share queries merge (m, l, acc) at the end.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) void ssa_fwd_f32_kernel(FwdParams p) {
  using M = Mat<D>;
  using C = Cfg<D>;
  using Plan = RowPlan<D, 4, CAUSAL, C::KW>;
  using Loads = RowLoadsF32<D, CAUSAL, C::KW>;
  constexpr int KW = C::KW, BN = C::BN, BB = C::BB, ND = M::ND;
  __shared__ __attribute__((aligned(1024))) char smem[Loads::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int kw = wave % KW, qw = wave / KW;
  const int block = folded_block();
  if (block >= Plan::grid(p)) return;
  const Plan pl(p, Plan::place(p, block));  // dispatch and K / V loads (ssa_rows_plan.hpp)
  const SeqView& sv = pl.sv;
  const int b = pl.b, h = pl.h, N = pl.N, nst = pl.nst;
  if (pl.empty()) return;  // packed: past the end of a shorter document
  const Loads ld(p, pl, lane, wave);
  const int wq0 = pl.q0 + 32 * qw, qrow = wq0 + l32;
  const float* qg = reinterpret_cast<const float*>(head_rows<4>(sv, p.q, b, h));
  const float* kg = reinterpret_cast<const float*>(ld.k.g);
  const float* vg = reinterpret_cast<const float*>(ld.v.g);
  const float n = *p.n_ptr, c = p.scale * *p.b_ptr;
  const uint32_t lds0 = lds_addr(smem);
  auto k_at = [&](int st, int i) { return Loads::k_at(lds0, st, i); };
  ld.load(pl, 0, lds0, wave);
  const M mat(lane);
  typename M::frag qf[M::NF];
#pragma unroll
  for (int f = 0; f < M::NF; ++f)
    qf[f] = qrow < N ? M::load(qg + qrow * p.q.ss, f, hh) : typename M::frag{};
  f32x16 acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = f32x16{};
  float m = -INFINITY, l = 0.f;
  for (int st = 0; st < nst; ++st) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // stage st has landed, stage st - 1 is consumed
    if (st + 1 < nst) ld.load(pl, st + 1, lds0, wave);
    const int k0 = st * BN + 32 * kw;
    if (k0 >= N || wq0 >= N || (CAUSAL && k0 > wq0 + 31)) continue;
    const f32x16 s = mat.scores(k_at(st, kw), qf);
    float t[16];
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = n * ssa_sl(s[r], fmaf(c, fabsf(s[r]), 1.f));
    if (k0 + 32 > N || (CAUSAL && k0 + 31 > wq0)) {
      const int last = CAUSAL ? min(qrow, N - 1) : N - 1;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + crow(r, hh) > last) t[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, t[r]);
    mx = fmaxf(m, pair_max(mx));
    if (__any(mx > m + kRescaleTau)) {  // rare: the running max moves, and with it what is summed so far
      const float alpha = fast_exp2(m - (mx == -INFINITY ? 0.f : mx));
      l *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[d] *= alpha;
      m = mx;
    }
    const float base = m == -INFINITY ? 0.f : m;  // no key of this row yet: p = 0
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      t[r] = fast_exp2(t[r] - base);
      sum += t[r];
    }
    l += sum;
    mat.outer(k_at(st, kw) + BB, t, acc);
  }
  l = pair_sum(l);
  if constexpr (KW > 1) {
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
    for (int i = 0; i < KW; ++i) m = fmaxf(m, ml[2 * (qw * KW + i) * 32 + l32]);
    const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int i = 0; i < KW; ++i)
      l += ml[(2 * (qw * KW + i) + 1) * 32 + l32] * fast_exp2(ml[2 * (qw * KW + i) * 32 + l32] - base);
    const float alpha = fast_exp2(own - base);
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[d] *= alpha;
    merge_parts<ND, KW>(acc, reinterpret_cast<float*>(smem), qw, kw, lane);
  }
  if (kw == 0 && qrow < N) {
    float* og = static_cast<float*>(const_cast<void*>(p.o.ptr)) + sv.off(p.o, b) + h * p.o.sh;
    const bool bad = row_nonfinite<ND>(acc);
    if (!bad)
      store_own<float, D>(acc, 1.f / l, og + qrow * p.o.ss, hh);  // every row has a key (causal: itself)
    if (SSA_RARE(__any(bad)) && bad)
      row_fwd<float, D>(og + qrow * p.o.ss, 1.f / l, qg + qrow * p.q.ss, kg, p.k.ss, vg, p.v.ss, CAUSAL ? qrow : N - 1,
                        n, c, m == -INFINITY ? 0.f : m, hh);
    if (hh == 0) p.m[sv.mrow(b, h, p.Hq, p.T, p.N) + qrow] = m + log2f(l);
  }
}

// Delta = rowsum(dO * O): D / 4 lanes per row, 4-element loads, butterfly.
template <typename T, int D>
__global__ __launch_bounds__(256) void ssa_bwd_preprocess_f32_kernel(BwdParams p) {
  constexpr int LPR = D / 4, RPB = 256 / LPR;
  const int tid = threadIdx.x;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * RPB + tid / LPR;
  const int sub = tid % LPR;
  const int64_t total = static_cast<int64_t>(p.B) * p.Hq * p.N;
  float acc = 0.f;
  if (row < total) {
    const int s = static_cast<int>(row % p.N);
    const int64_t bh = row / p.N;
    const int h = static_cast<int>(bh % p.Hq), b = static_cast<int>(bh / p.Hq);
    const f32x4 o = ld4(static_cast<const T*>(p.o.ptr) + b * p.o.sb + h * p.o.sh + s * p.o.ss + 4 * sub);
    const f32x4 g = ld4(static_cast<const T*>(p.dout.ptr) + b * p.dout.sb + h * p.dout.sh + s * p.dout.ss + 4 * sub);
    acc = fmaf(o.x, g.x, fmaf(o.y, g.y, fmaf(o.z, g.z, o.w * g.w)));
  }
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (row < total && sub == 0) p.delta[row] = acc;
}

// ---------------------------------------------------------------------------
// dK, dV (+ dn / db partials) for 128 keys of one (batch, kv-head): four
// groups of 32 keys, QS waves each on alternate 32-query blocks; Q / dO blocks
// with their M and Delta stream through LDS over every q-head of the GQA
// group.  Per valid pair, as in ssa_bwd.hip: P = exp2(n sL - M), dT = P (dP -
// Delta), dS' = dT / (1 + c|x|), dV += P dO, dK += dS' q (scaled by scale n b
// at the end), dn += ln2 dT sL, db += n scale dS' x.
template <int D, bool CAUSAL, bool DO_DK, bool DO_DV>
__device__ __forceinline__ void dkdv_f32_body(const BwdParams& p, char* smem, float (*red)[8], int block) {
  using M = Mat<D>;
  using C = Cfg<D>;
  constexpr int QS = C::QS, NWV = 4 * QS, BB = C::BB, ND = M::ND, STEP = 32 * QS;
  using Plan = KeyPlan<D, 4, CAUSAL, QS, NWV>;
  using Stage = KeyStageF32<D, QS>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int qs = wave % QS, kg4 = wave / QS;
  const int nkb = dkdv_key_blocks(p.N);
  const Plan pl(p, Plan::place(p, block));  // dispatch and Q / dO loads (ssa_rows_plan.hpp)
  const SeqView& sv = pl.sv;
  const int kb = pl.kb, b = pl.b, hk = pl.hk, bhk = pl.bhk, N = pl.N, k0 = pl.k0;
  const int64_t PP = static_cast<int64_t>(p.B) * p.Hkv * nkb;
  if (pl.empty()) {  // packed: past the end of a shorter document
    if (DO_DK && tid == 0) {
      p.partials[static_cast<int64_t>(bhk) * nkb + kb] = 0.f;
      p.partials[PP + static_cast<int64_t>(bhk) * nkb + kb] = 0.f;
    }
    return;
  }
  const int k0w = k0 + 32 * kg4, key = k0w + l32;
  const float* kg = static_cast<const float*>(p.k.ptr) + sv.off(p.k, b) + hk * p.k.sh;
  const float* vg = static_cast<const float*>(p.v.ptr) + sv.off(p.v, b) + hk * p.v.sh;
  const float n = *p.n_ptr, bv = *p.b_ptr, c = p.scale * bv;
  const uint32_t lds0 = lds_addr(smem);
  const LoadLane llq(lane, wave, p.q.ss * 2), lld(lane, wave, p.dout.ss * 2);
  const int qstart = pl.qstart, nst = pl.nst;
  auto blk_at = [&](int st, int i) { return Stage::blk_at(lds0, st, i); };
  auto load_stage = [&](int st, int g, int q0) { Stage::load(p, pl, st, g, q0, lds0, llq, lld, wave, lane); };
  load_stage(0, 0, qstart);
  const M mat(lane);
  typename M::frag kf[M::NF], vf[M::NF];
#pragma unroll
  for (int f = 0; f < M::NF; ++f) {
    kf[f] = key < N ? M::load(kg + key * p.k.ss, f, hh) : typename M::frag{};
    if constexpr (DO_DK) vf[f] = key < N ? M::load(vg + key * p.v.ss, f, hh) : typename M::frag{};
  }
  f32x16 dk[ND], dv[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) dk[d] = dv[d] = f32x16{};
  float dn_acc = 0.f, dn_c = 0.f, db_acc = 0.f, db_c = 0.f;  // Kahan sums over the blocks' sums
  int g = 0, q0 = qstart;  // of stage st
  for (int st = 0; st < nst; ++st) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // stage st has landed, stage st - 1 is consumed
    const int qi0 = q0 + 32 * qs;
    q0 += STEP;
    if (q0 >= N) {
      q0 = qstart;
      ++g;
    }
    if (st + 1 < nst) load_stage(st + 1, g, q0);
    if (qi0 >= N || k0w >= N || (CAUSAL && qi0 + 31 < k0w)) continue;
    const uint32_t at = blk_at(st, qs);
    const f32x16 s = mat.scores(at, kf);
    f32x16 dp = f32x16{};
    if constexpr (DO_DK) dp = mat.scores(at + BB, vf);
    float pv[16], ds[16];
    float tdn = 0.f, tdb = 0.f;
    const bool masked = qi0 + 32 > N || k0w + 32 > N || (CAUSAL && k0w + 31 > qi0);  // wave-uniform
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4_t mv = lds_read_f4(at + 2 * BB + (8 * j + 4 * hh) * 4);
      const f32x4_t dl = lds_read_f4(at + 2 * BB + 128 + (8 * j + 4 * hh) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * j + e;
        const float x = s[r];
        const float u1 = fmaf(c, fabsf(x), 1.f);
        const float sl = ssa_sl(x, u1);
        float w = fast_exp2(fmaf(n, sl, -mv[e]));
        if (masked) {
          const int qi = qi0 + crow(r, hh);
          if (qi >= N || key >= N || (CAUSAL && key > qi)) w = 0.f;
        }
        pv[r] = w;
        if constexpr (DO_DK) {
          const float dt = w * (dp[r] - dl[e]);
          ds[r] = dt * fast_rcp(u1);
          tdn = fmaf(dt, sl, tdn);
          tdb = fmaf(ds[r], x, tdb);
        }
      }
    }
    if constexpr (DO_DV) mat.outer(at + BB, pv, dv);
    if constexpr (DO_DK) {
      const float y = tdn - dn_c, t = dn_acc + y;
      dn_c = (t - dn_acc) - y;
      dn_acc = t;
      const float y2 = tdb - db_c, t2 = db_acc + y2;
      db_c = (t2 - db_acc) - y2;
      db_acc = t2;
      mat.outer(at, ds, dk);
    }
  }
  if constexpr (DO_DK) merge_parts<ND, QS>(dk, reinterpret_cast<float*>(smem), kg4, qs, lane);
  if constexpr (DO_DV) merge_parts<ND, QS>(dv, reinterpret_cast<float*>(smem), kg4, qs, lane);
  // keys with non-finite sums in any of their waves (ssa_rows.hpp): the first of these waves sums them again
  bool bad = DO_DK && row_nonfinite<ND>(dk, dn_acc + db_acc);
  if constexpr (DO_DV) bad = bad || row_nonfinite<ND>(dv);
  if (QS > 1) {
    if (lane == 0) red[2][wave] = __any(bad) ? 1.f : 0.f;
    __syncthreads();
    float any_bad = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) any_bad += red[2][w];
    if (SSA_RARE(any_bad != 0.f)) {
      int* rows = reinterpret_cast<int*>(smem);  // [QS][4][32]
      if (hh == 0) rows[(qs * 4 + kg4) * 32 + l32] = bad;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < QS; ++i) bad = bad || rows[(i * 4 + kg4) * 32 + l32] != 0;
    }
  }
  if (key < N) {
    float *dkr = nullptr, *dvr = nullptr;
    if constexpr (DO_DK)
      dkr = static_cast<float*>(const_cast<void*>(p.dk.ptr)) + sv.off(p.dk, b) + hk * p.dk.sh + key * p.dk.ss;
    if constexpr (DO_DV)
      dvr = static_cast<float*>(const_cast<void*>(p.dv.ptr)) + sv.off(p.dv, b) + hk * p.dv.sh + key * p.dv.ss;
    if (!bad) {
      if constexpr (DO_DK)
        if (qs == 0) store_own<float, D>(dk, p.scale * n * bv, dkr, hh);
      if constexpr (DO_DV)
        if (qs == 0) store_own<float, D>(dv, 1.f, dvr, hh);
    }
    if (SSA_RARE(__any(bad)) && bad) {
      dn_acc = dn_c = db_acc = db_c = 0.f;
      if (qs == 0)
        row_dkdv<float, D, CAUSAL>(p, sv, b, hk, key, n, c, dkr, p.scale * n * bv, dvr, dn_acc, db_acc, hh);
      if (hh != 0) dn_acc = db_acc = 0.f;  // both lanes of the pair have the whole sums
    }
  }
  if constexpr (DO_DK) {
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
      float sdn = 0.f, sdb = 0.f;
#pragma unroll
      for (int w = 0; w < NWV; ++w) {
        sdn += red[0][w];
        sdb += red[1][w];
      }
      p.partials[static_cast<int64_t>(bhk) * nkb + kb] = kLn2 * sdn;
      p.partials[PP + static_cast<int64_t>(bhk) * nkb + kb] = n * p.scale * sdb;
    }
  }
}

// ROLES: half of the grid computes dK (and dn, db; three products a block) and
// half dV (two).
template <int D, bool CAUSAL, bool ROLES>
__global__ __launch_bounds__((Cfg<D>::DKDV_THREADS)) void ssa_bwd_dkdv_f32_kernel(BwdParams p) {
  using C = Cfg<D>;
  __shared__ __attribute__((aligned(1024))) char smem[KeyStageF32<D, C::QS>::LDS_BYTES];
  __shared__ float red[3][8];
  const int block = folded_block(), grid = dkdv_key_blocks(p.N) * p.B * p.Hkv;
  if constexpr (ROLES) {
    // dK workgroups (three products per block) before the lighter dV ones
    if (block < grid)
      dkdv_f32_body<D, CAUSAL, true, false>(p, smem, red, block);
    else if (block < 2 * grid)
      dkdv_f32_body<D, CAUSAL, false, true>(p, smem, red, block - grid);
  } else if (block < grid) {
    dkdv_f32_body<D, CAUSAL, true, true>(p, smem, red, block);
  }
}

// ---------------------------------------------------------------------------
// dQ for BM query rows of one (batch, q-head): K / V streamed BN keys a stage;
// the scores and dP are recomputed (dQ += scale n b dS' k).
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) void ssa_bwd_dq_f32_kernel(BwdParams p) {
  using M = Mat<D>;
  using C = Cfg<D>;
  using Plan = RowPlan<D, 4, CAUSAL, C::KW>;
  using Loads = RowLoadsF32<D, CAUSAL, C::KW>;
  constexpr int KW = C::KW, BN = C::BN, BB = C::BB, ND = M::ND;
  __shared__ __attribute__((aligned(1024))) char smem[Loads::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int kw = wave % KW, qw = wave / KW;
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
  const float* qg = reinterpret_cast<const float*>(head_rows<4>(sv, p.q, b, h));
  const float* dog = reinterpret_cast<const float*>(head_rows<4>(sv, p.dout, b, h));
  const float* kg = reinterpret_cast<const float*>(ld.k.g);
  const float* vg = reinterpret_cast<const float*>(ld.v.g);
  const int64_t mr = sv.mrow(b, h, p.Hq, p.T, p.N);
  const float n = *p.n_ptr, bv = *p.b_ptr, c = p.scale * bv;
  const uint32_t lds0 = lds_addr(smem);
  auto k_at = [&](int st, int i) { return Loads::k_at(lds0, st, i); };
  ld.load(pl, 0, lds0, wave);
  const M mat(lane);
  typename M::frag qf[M::NF], dof[M::NF];
#pragma unroll
  for (int f = 0; f < M::NF; ++f) {
    qf[f] = qrow < N ? M::load(qg + qrow * p.q.ss, f, hh) : typename M::frag{};
    dof[f] = qrow < N ? M::load(dog + qrow * p.dout.ss, f, hh) : typename M::frag{};
  }
  const float mi = qrow < N ? p.m[mr + qrow] : 0.f, di = qrow < N ? p.delta[mr + qrow] : 0.f;
  f32x16 dq[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) dq[d] = f32x16{};
  for (int st = 0; st < nst; ++st) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // stage st has landed, stage st - 1 is consumed
    if (st + 1 < nst) ld.load(pl, st + 1, lds0, wave);
    const int k0 = st * BN + 32 * kw;
    if (k0 >= N || wq0 >= N || (CAUSAL && k0 > wq0 + 31)) continue;
    const uint32_t at = k_at(st, kw);
    const f32x16 s = mat.scores(at, qf), dp = mat.scores(at + BB, dof);
    float ds[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float x = s[r];
      const float u1 = fmaf(c, fabsf(x), 1.f);
      const float pv = fast_exp2(fmaf(n, ssa_sl(x, u1), -mi));
      ds[r] = pv * (dp[r] - di) * fast_rcp(u1);
    }
    if (k0 + 32 > N || wq0 + 32 > N || (CAUSAL && k0 + 31 > wq0)) {
      const int last = qrow >= N ? -1 : (CAUSAL ? min(qrow, N - 1) : N - 1);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + crow(r, hh) > last) ds[r] = 0.f;
    }
    mat.outer(at, ds, dq);
  }
  merge_parts<ND, KW>(dq, reinterpret_cast<float*>(smem), qw, kw, lane);
  if (kw == 0 && qrow < N) {
    float* dqr = static_cast<float*>(const_cast<void*>(p.dq.ptr)) + sv.off(p.dq, b) + h * p.dq.sh + qrow * p.dq.ss;
    const bool bad = row_nonfinite<ND>(dq);
    if (!bad)
      store_own<float, D>(dq, p.scale * n * bv, dqr, hh);
    if (SSA_RARE(__any(bad)) && bad)
      row_dq<float, D>(dqr, p.scale * n * bv, qg + qrow * p.q.ss, dog + qrow * p.dout.ss, kg, p.k.ss, vg, p.v.ss,
                       CAUSAL ? qrow : N - 1, n, c, mi, di, hh);
  }
}

// One launch of KERNEL<DD, CAUSAL>, and the head dims.
#define SSA_F32_LAUNCH(KERNEL, THREADS, DD, GRID, P, CAUSAL, S)                                     \
  do {                                                                                              \
    if (CAUSAL) hipLaunchKernelGGL((KERNEL<DD, true>), GRID(DD), dim3(THREADS(DD)), 0, S, P);        \
    else hipLaunchKernelGGL((KERNEL<DD, false>), GRID(DD), dim3(THREADS(DD)), 0, S, P);              \
  } while (0)
#define SSA_F32_DISPATCH(KERNEL, THREADS, GRID, P, D, CAUSAL, S)                 \
  switch (D) {                                                                   \
    case 16: SSA_F32_LAUNCH(KERNEL, THREADS, 16, GRID, P, CAUSAL, S); break;     \
    case 32: SSA_F32_LAUNCH(KERNEL, THREADS, 32, GRID, P, CAUSAL, S); break;     \
    case 64: SSA_F32_LAUNCH(KERNEL, THREADS, 64, GRID, P, CAUSAL, S); break;     \
    case 128: SSA_F32_LAUNCH(KERNEL, THREADS, 128, GRID, P, CAUSAL, S); break;   \
    case 256: SSA_F32_LAUNCH(KERNEL, THREADS, 256, GRID, P, CAUSAL, S); break;   \
    default: return hipErrorInvalidValue;                                        \
  }

template <typename T, int D>
static void launch_pre(const BwdParams& p, hipStream_t s) {
  const int64_t rows = static_cast<int64_t>(p.B) * p.Hq * p.N;
  const int rpb = 256 / (D / 4);
  const int grid = static_cast<int>((rows + rpb - 1) / rpb);
  hipLaunchKernelGGL((ssa_bwd_preprocess_f32_kernel<T, D>), dim3(grid), dim3(256), 0, s, p);
}

}  // namespace

#define SSA_F32_ROW_GRID(DD) folded_grid((p.N + Cfg<DD>::BM - 1) / Cfg<DD>::BM * p.B * p.Hq, 256)
#define SSA_F32_THREADS(DD) 256

// dK and dV in one workgroup (four products a block) or in two (three and two).
// Apart they have twice the workgroups, the longest of them three quarters as
// long: worth a quarter more work while the grid leaves CUs idle, that is up to
// 128 workgroups of 128 keys without the mask and, since half of a causal
// grid's work is in its first quarter, up to 256 with it (us, together -> apart:
// causal D = 64 1 x 16 x 1024 148 -> 124, 1 x 16 x 2048 (256) 290 -> 252, D = 128
// 1 x 16 x 1100 318 -> 252; full D = 64 1 x 16 x 1024 151 -> 131, 2 x 16 x 1100
// (288) 329 -> 327).  At head dim 256 the accumulators of both do not fit one
// wave beside the K and V fragments.
constexpr int kRolesGrid = 128;
template <int D, bool CAUSAL>
static hipError_t launch_dkdv(const BwdParams& p, hipStream_t s) {
  const int grid = dkdv_key_blocks(p.N) * p.B * p.Hkv;
  constexpr int threads = Cfg<D>::DKDV_THREADS;
  if (D >= 256 || grid <= (CAUSAL ? 2 : 1) * kRolesGrid) {
    hipLaunchKernelGGL((ssa_bwd_dkdv_f32_kernel<D, CAUSAL, true>), folded_grid(2 * grid, threads), dim3(threads), 0,
                       s, p);
    return hipGetLastError();
  }
  if constexpr (D < 256)
    hipLaunchKernelGGL((ssa_bwd_dkdv_f32_kernel<D, CAUSAL, false>), folded_grid(grid, threads), dim3(threads), 0,
                       s, p);
  return hipGetLastError();
}

hipError_t launch_fwd_f32(const FwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  if (dtype != kDtypeF32) return launch_fwd_d256(p, dtype, D, causal, s);
  SSA_F32_DISPATCH(ssa_fwd_f32_kernel, SSA_F32_THREADS, SSA_F32_ROW_GRID, p, D, causal, s)
  return hipGetLastError();
}

hipError_t launch_bwd_preprocess_f32(const BwdParams& p, int dtype, int D, hipStream_t s) {
  if (dtype == kDtypeF32) {
    switch (D) {
      case 16: launch_pre<float, 16>(p, s); break;
      case 32: launch_pre<float, 32>(p, s); break;
      case 64: launch_pre<float, 64>(p, s); break;
      case 128: launch_pre<float, 128>(p, s); break;
      case 256: launch_pre<float, 256>(p, s); break;
      default: return hipErrorInvalidValue;
    }
  } else if (D == 256) {
    if (dtype == 0)
      launch_pre<__bf16, 256>(p, s);
    else
      launch_pre<_Float16, 256>(p, s);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv_f32(const BwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  if (dtype != kDtypeF32) return launch_bwd_dkdv_d256(p, dtype, D, causal, s);
  switch (D) {
    case 16: return causal ? launch_dkdv<16, true>(p, s) : launch_dkdv<16, false>(p, s);
    case 32: return causal ? launch_dkdv<32, true>(p, s) : launch_dkdv<32, false>(p, s);
    case 64: return causal ? launch_dkdv<64, true>(p, s) : launch_dkdv<64, false>(p, s);
    case 128: return causal ? launch_dkdv<128, true>(p, s) : launch_dkdv<128, false>(p, s);
    case 256: return causal ? launch_dkdv<256, true>(p, s) : launch_dkdv<256, false>(p, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_bwd_dq_f32(const BwdParams& p, int dtype, int D, bool causal, hipStream_t s) {
  if (dtype != kDtypeF32) return launch_bwd_dq_d256(p, dtype, D, causal, s);
  SSA_F32_DISPATCH(ssa_bwd_dq_f32_kernel, SSA_F32_THREADS, SSA_F32_ROW_GRID, p, D, causal, s)
  return hipGetLastError();
}

}  // namespace ssa
