// Dispatch, stage rings and tile loads of the fp32-precision kernels (ssa_f32.hip,
// ssa_d256.hip), as ssa_plan.hpp holds those of the 16-bit ones: __host__
// __device__, so that tests/host_addr replays exactly this code.
//
// A 16-bit or fp32 row of D elements of E bytes is LD = D E / 2 columns of 16
// bits to the tile loaders, and its stride is counted in those.
#pragma once

#include "ssa_launch.hpp"
#include "ssa_tile.hpp"

namespace ssa {

// A workgroup's place in a grid of nblk blocks of rows per (sequence, head):
// XCD-contiguous, the heaviest blocks (rank 0) of a pair of heads first, as
// FwdPlan and DkdvPlan.
struct Place {
  int rank, b, h;
  __host__ __device__ __forceinline__ Place(int block, int grid, int nblk, int B, bool packed) {
    int hb;
    dispatch_order(xcd_remap(block, grid), grid / nblk, nblk, packed ? 1 : kOrderGroup, hb, rank);
    b = hb % B;
    h = hb / B;
  }
};

// The rows of one head of a tensor, streamed in blocks of 32 by NW waves.
template <int LD, int NW>
struct BlockStream {
  static constexpr int BB = BlockLayout<LD>::BLOCK;
  const char* g;
  int64_t ss;  // in 16-bit columns
  LoadLane ll;
  __host__ __device__ __forceinline__ BlockStream(const void* rows, int64_t ss16, int lane, int wave)
      : g(static_cast<const char*>(rows)), ss(ss16), ll(lane, wave, ss16) {}
  // blocks of rows row0 + 32 i (those at or past N clamped to the last) to lds + i * pitch
  template <int BLOCKS, typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load(int row0, int N, uint32_t lds, uint32_t pitch, int wave,
                                                const Mem& mem = Mem()) const {
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) tile_load_async<LD, 32, NW>(g, ss, row0 + 32 * i, N, lds + i * pitch, wave, ll, mem);
  }
};

// Head `head` of sequence b: the first row of a tensor of E-byte elements.
template <int E>
__host__ __device__ __forceinline__ const char* head_rows(const SeqView& sv, const Tensor4& t, int b, int head) {
  return static_cast<const char*>(t.ptr) + (sv.off(t, b) + head * t.sh) * E;
}

// ---------------------------------------------------------------------------
// Forward and dQ: 4 waves, KW of them on the same 32 queries and alternate blocks
// of a stage of KW blocks of 32 keys.
template <int D, int E, bool CAUSAL, int KW>
struct RowPlan {
  static constexpr int LD = D * E / 2, BB = BlockLayout<LD>::BLOCK;
  static constexpr int QW = 4 / KW, BM = 32 * QW, BN = 32 * KW, NW = 4;
  static_assert(BM >= 32, "grids of 2^28 units of 128 rows stay below 2^31 workgroups");
  int b, h, hk, N, q0, nst;
  SeqView sv;
  template <typename P>
  __host__ __device__ static __forceinline__ int blocks(const P& p) {
    return (p.N + BM - 1) / BM;
  }
  template <typename P>
  __host__ __device__ static __forceinline__ int grid(const P& p) {
    return blocks(p) * p.B * p.Hq;
  }
  template <typename P>
  __host__ __device__ __forceinline__ RowPlan(const P& p, const Place& pl)
      : b(pl.b), h(pl.h), hk(pl.h / (p.Hq / p.Hkv)), sv(p.cu_seqlens, p.T, p.N, pl.b) {
    N = sv.N;
    q0 = (blocks(p) - 1 - pl.rank) * BM;
    const int kv_end = CAUSAL ? (N < q0 + BM ? N : q0 + BM) : N;
    nst = (kv_end + BN - 1) / BN;
  }
  template <typename P>
  __host__ __device__ static __forceinline__ Place place(const P& p, int block) {
    return Place(block, grid(p), blocks(p), p.B, p.cu_seqlens != nullptr);
  }
  __host__ __device__ __forceinline__ bool empty() const { return q0 >= N; }  // packed: past a shorter document
};

// fp32: blocks a stage (= waves that share 32 owned rows) of the forward and dQ, and
// of dK/dV (two waves per 32 keys up to head dim 64).  A stage holds two blocks (K
// and V, or Q and dO) per wave, twice buffered, in at most 128 KB of LDS.
template <int D>
struct SplitF32 {
  static constexpr int BB = BlockLayout<2 * D>::BLOCK;
  static constexpr int KW = 4 * BB <= 32768 ? 4 : (BB <= 16384 ? 2 : 1), QS = D <= 64 ? 2 : 1;
};

// fp32: K and V of a stage together, two stages.  Block i of stage st: K at
// k_at(st, i), V behind it.
template <int D, bool CAUSAL, int KW>
struct RowLoadsF32 {
  using Plan = RowPlan<D, 4, CAUSAL, KW>;
  static constexpr int BB = Plan::BB, LDS_BYTES = 2 * KW * 2 * BB;
  BlockStream<Plan::LD, 4> k, v;
  template <typename P>
  __host__ __device__ __forceinline__ RowLoadsF32(const P& p, const Plan& pl, int lane, int wave)
      : k(head_rows<4>(pl.sv, p.k, pl.b, pl.hk), p.k.ss * 2, lane, wave),
        v(head_rows<4>(pl.sv, p.v, pl.b, pl.hk), p.v.ss * 2, lane, wave) {}
  __host__ __device__ static __forceinline__ uint32_t k_at(uint32_t lds0, int st, int i) {
    return lds0 + ((st & 1) * KW + i) * 2 * BB;
  }
  template <typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load(const Plan& pl, int st, uint32_t lds0, int wave,
                                                const Mem& mem = Mem()) const {
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      k.template load<1>(st * Plan::BN + 32 * i, pl.N, k_at(lds0, st, i), 0, wave, mem);
      v.template load<1>(st * Plan::BN + 32 * i, pl.N, k_at(lds0, st, i) + BB, 0, wave, mem);
    }
  }
};

// Head dim 256 in 16 bits: K and V in rings of their own (KS and VS slots), a
// stage of each loaded by itself.
template <bool CAUSAL, int KW, int KS, int VS>
struct RowLoads256 {
  using Plan = RowPlan<256, 2, CAUSAL, KW>;
  static constexpr int BB = Plan::BB, STAGE = KW * BB, LDS_BYTES = (KS + VS) * STAGE;
  BlockStream<Plan::LD, 4> k, v;
  template <typename P>
  __host__ __device__ __forceinline__ RowLoads256(const P& p, const Plan& pl, int lane, int wave)
      : k(head_rows<2>(pl.sv, p.k, pl.b, pl.hk), p.k.ss, lane, wave),
        v(head_rows<2>(pl.sv, p.v, pl.b, pl.hk), p.v.ss, lane, wave) {}
  __host__ __device__ static __forceinline__ uint32_t k_at(uint32_t lds0, int slot) { return lds0 + slot * STAGE; }
  __host__ __device__ static __forceinline__ uint32_t v_at(uint32_t lds0, int slot) {
    return lds0 + (KS + slot) * STAGE;
  }
  template <typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load_k(const Plan& pl, int st, int slot, uint32_t lds0, int wave,
                                                  const Mem& mem = Mem()) const {
    if (st < pl.nst) k.template load<KW>(st * Plan::BN, pl.N, k_at(lds0, slot), BB, wave, mem);
  }
  template <typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load_v(const Plan& pl, int st, int slot, uint32_t lds0, int wave,
                                                  const Mem& mem = Mem()) const {
    if (st < pl.nst) v.template load<KW>(st * Plan::BN, pl.N, v_at(lds0, slot), BB, wave, mem);
  }
};

// ---------------------------------------------------------------------------
// dK/dV: 128 keys, QS blocks of 32 queries a stage over every q-head of the
// group, NW waves.
template <int D, int E, bool CAUSAL, int QS, int NW>
struct KeyPlan {
  static constexpr int LD = D * E / 2, BB = BlockLayout<LD>::BLOCK, STEP = 32 * QS;
  int kb, b, hk, bhk, G, N, k0, qstart, nqs, nst;
  SeqView sv;
  template <typename P>
  __host__ __device__ static __forceinline__ int grid(const P& p) {
    return dkdv_key_blocks(p.N) * p.B * p.Hkv;
  }
  template <typename P>
  __host__ __device__ static __forceinline__ Place place(const P& p, int block) {
    return Place(block, grid(p), dkdv_key_blocks(p.N), p.B, p.cu_seqlens != nullptr);
  }
  template <typename P>
  __host__ __device__ __forceinline__ KeyPlan(const P& p, const Place& pl)
      : kb(pl.rank), b(pl.b), hk(pl.h), bhk(pl.h * p.B + pl.b), G(p.Hq / p.Hkv), sv(p.cu_seqlens, p.T, p.N, pl.b) {
    N = sv.N;
    k0 = kb * 128;
    qstart = CAUSAL ? k0 : 0;
    nqs = (N - qstart + STEP - 1) / STEP;
    nst = G * nqs;
  }
  __host__ __device__ __forceinline__ bool empty() const { return k0 >= N; }
  // Q, dO and M, Delta of BLOCKS blocks from query q0 of q-head g of the group;
  // block i of each at its address + i * pitch.  M and Delta of block i come from
  // wave NW - 1 - i.
  template <int BLOCKS, typename P, typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load(const P& p, int g, int q0, uint32_t q_lds, uint32_t d_lds,
                                                uint32_t md_lds, uint32_t pitch, const LoadLane& llq,
                                                const LoadLane& lld, int wave, int lane, const Mem& mem = Mem()) const {
    const int h = hk * G + g;
    const char* qg = head_rows<E>(sv, p.q, b, h);
    const char* dog = head_rows<E>(sv, p.dout, b, h);
    const int64_t mr = sv.mrow(b, h, p.Hq, p.T, p.N);
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) {
      tile_load_async<LD, 32, NW>(qg, p.q.ss * (E / 2), q0 + 32 * i, N, q_lds + i * pitch, wave, llq, mem);
      tile_load_async<LD, 32, NW>(dog, p.dout.ss * (E / 2), q0 + 32 * i, N, d_lds + i * pitch, wave, lld, mem);
      if (wave == NW - 1 - i) pair32_load_async(p.m + mr, p.delta + mr, q0 + 32 * i, N, md_lds + i * pitch, lane, mem);
    }
  }
};

// fp32: QS blocks a stage, each Q, dO, M[32], Delta[32], two stages.
template <int D, int QS>
struct KeyStageF32 {
  static constexpr int BB = BlockLayout<2 * D>::BLOCK, BLK = 2 * BB + 256, LDS_BYTES = 2 * QS * BLK;
  __host__ __device__ static __forceinline__ uint32_t blk_at(uint32_t lds0, int st, int i) {
    return lds0 + (st & 1) * QS * BLK + i * BLK;
  }
  template <typename P, typename Plan, typename Mem = DeviceMem>
  __host__ __device__ static __forceinline__ void load(const P& p, const Plan& pl, int st, int g, int q0, uint32_t lds0,
                                                       const LoadLane& llq, const LoadLane& lld, int wave, int lane,
                                                       const Mem& mem = Mem()) {
    const uint32_t at = blk_at(lds0, st, 0);
    pl.template load<QS>(p, g, q0, at, at + BB, at + 2 * BB, BLK, llq, lld, wave, lane, mem);
  }
};

// Head dim 256 in 16 bits: a block of Q and of dO a stage, in rings of three and two
// slots (the operand of dK's outer product, Q, or of dV's, dO, is held for one stage
// longer), M and Delta in one of three.  Holds the next stage to load; slots are
// kept, not divided out.
template <bool DK>
struct KeyRing256 {
  static constexpr int RQ = DK ? 3 : 2, RD = DK ? 2 : 3, BB = BlockLayout<256>::BLOCK;
  static constexpr int LDS_BYTES = 5 * BB + 3 * 256;
  int g = 0, q0, st = 0, q_slot = 0, d_slot = 0, m_slot = 0;
  __host__ __device__ __forceinline__ explicit KeyRing256(int qstart) : q0(qstart) {}
  __host__ __device__ static __forceinline__ uint32_t q_at(uint32_t lds0, int slot) { return lds0 + slot * BB; }
  __host__ __device__ static __forceinline__ uint32_t d_at(uint32_t lds0, int slot) { return lds0 + (RQ + slot) * BB; }
  __host__ __device__ static __forceinline__ uint32_t md_at(uint32_t lds0, int slot) {
    return lds0 + 5 * BB + slot * 256;
  }
  template <typename P, typename Plan, typename Mem = DeviceMem>
  __host__ __device__ __forceinline__ void load_next(const P& p, const Plan& pl, uint32_t lds0, const LoadLane& llq,
                                                     const LoadLane& lld, int wave, int lane, const Mem& mem = Mem()) {
    if (st >= pl.nst) return;
    pl.template load<1>(p, g, q0, q_at(lds0, q_slot), d_at(lds0, d_slot), md_at(lds0, m_slot), 0, llq, lld, wave, lane,
                        mem);
    ++st;
    q_slot = q_slot + 1 == RQ ? 0 : q_slot + 1;
    d_slot = d_slot + 1 == RD ? 0 : d_slot + 1;
    m_slot = m_slot == 2 ? 0 : m_slot + 1;
    q0 += 32;
    if (q0 >= pl.N) {
      q0 = pl.qstart;
      ++g;
    }
  }
};

}  // namespace ssa
