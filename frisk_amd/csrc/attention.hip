// Fused attention forward for gfx950: O = softmax(scale * Q K^T) V, one pass over the keys with a running
// maximum and denominator, the program of the reference's sketch tmp/ir.mlir:87-157 (copy Q; for each key tile:
// copy K, gemm, reduce max, exp2, reduce sum, rescale, copy V, gemm; copy O) executed as one kernel.
//
// A work-group of 8 waves owns 256 queries of one (batch, head); a wave owns 32 of them for the whole kernel, two
// waves share a SIMD.  Key / value tiles of 64 keys stream HBM/L2 -> LDS with global_load_lds_dwordx4 through rings
// of three (K) and four (V) tiles.  The two waves of a SIMD alternate between an MFMA phase and a softmax (VALU)
// phase in opposite order, so the matrix pipe and the vector pipe of the SIMD are busy at the same time.
// Both products are computed transposed so that a lane owns one query:
//   S^T[key][q] = sum_d K[key][d] Q[q][d]     MFMA A = K fragment (LDS), B = Q fragment (registers, loaded once)
//   O^T[d][q]   = sum_key V[key][d] P[q][key] MFMA A = V fragment (LDS, transpose read), B = P fragment
// In the 32x32 result layout lane l holds column l % 32 (a query) and rows 4*(l/32) + (r%4) + 8*(r/4): the maximum
// and the sum over keys are 16 in-register operations per atom plus one exchange with lane l ^ 32, and the
// probabilities of S^T are already the B operand of the second product if its K slots are read in the same
// permuted key order (slot 8g+e of a 16-key step is key 4g + e%4 + 8*(e/4)) -- the transpose reads of V fetch
// their 4-row groups in that order, so P never goes through LDS.
// Where that leaves CUs idle the waves of a work-group split its keys instead of sharing them: 2, 4 or 8 shares of 4, 2 or 1
// waves, 128, 64 or 32 queries, each share with its own rings, merged through LDS at the end (attention_key_shares).
#include "gemm_kernel.hip.inc"
#include "attention.h"

namespace frisk {

template <int DT_, bool KT_, int KS_, int KB_ = 64, int NSK_ = 3> struct AttnCfg {
  static constexpr int DT = DT_;
  static constexpr bool KT = KT_;  // K stored [head_dim][seq_k]
  static constexpr int KS = KS_;   // shares of the keys inside a work-group, SW waves each
  static constexpr int NW = 8, SW = NW / KS, QW = 32;
  static constexpr int D = kAttnHeadDim, QB = QW * SW, KB = KB_;
  static constexpr int KA = KB / 32, DA = D / 32;
  // LDS ring depths of a share: K is consumed one tile ahead of V.  Iteration kt stages K tile kt + NSK and V tile kt + NSV - 1
  // during its M phase; with single buffers (NSK = 1) K tile kt + 1 and V tile kt during its V phase
  static constexpr int NSK = NSK_, NSV = NSK == 1 ? 1 : NSK + 1;
  typedef Mma<DT> M;
  typedef TileLayout<2, !KT, KB, D> LK;    // first product contracts over head_dim
  typedef TileLayout<2, false, D, KB> LV;  // second product contracts over keys; head_dim runs along the row
  static constexpr int RING_BYTES = NSK * LK::BYTES + NSV * LV::BYTES;  // of one share
  static constexpr int OUT_BYTES_PER_WAVE = 32 * (64 * 2 + 16);  // output staging: 32 queries x 64 columns, rows padded by 16 B
  // merging the shares (over the rings, when they are done with): 32 queries x 128 fp32 per wave, rows padded by 16 B, then a
  // (reference, denominator) pair per wave and query
  static constexpr int MERGE_ROW = D * 4 + 16, MERGE_STATS = NW * QW * MERGE_ROW, MERGE_BYTES = MERGE_STATS + NW * QW * 8;
  static constexpr int LDS_BYTES = KS == 1 ? RING_BYTES + NW * OUT_BYTES_PER_WAVE : (KS * RING_BYTES > MERGE_BYTES ? KS * RING_BYTES : MERGE_BYTES);
  static_assert(M::ES == 2 && M::KA == 16, "16-bit operands");
  static_assert(LV::SH == 0 && LV::MK <= 3, "the V swizzle may only depend on the key row modulo 4");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget of one CU");
};

// Address of the transpose read that serves head_dim atom `da` (32 columns of V) with K slots in the permuted key
// order: the lane's register holds key row 4g + (l%16)/4 of the tile, instruction q of step t adds 16t + 8q rows.
template <class LV> struct PermutedKeyReader {
  FRISK_DEV unsigned lane_reg(int lane, int da) {
    const int blk = lane >> 4, l16 = lane & 15, g = blk >> 1;
    return (unsigned)LV::offset(4 * g + (l16 >> 2), (32 * da + 16 * (blk & 1) + 4 * (l16 & 3)) * 2);
  }
  static constexpr int delta(int t, int q) { return (16 * t + 8 * q) * LV::ROWB; }
  FRISK_DEV void read(unsigned reg, int t, int* out) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      FRISK_LDS const char* p = (FRISK_LDS const char*)(uintptr_t)reg + delta(t, q);
      v2i w = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((FRISK_LDS v4s*)p));
      out[2 * q] = w[0];
      out[2 * q + 1] = w[1];
    }
  }
};

// two fp32 -> one packed 16-bit pair, and sum of a packed pair added to an fp32 (one v_dot2 with a pair of ones)
template <int DT> struct Pack16;
template <> struct Pack16<FRISK_F16> {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  FRISK_DEV int two(float a, float b) {
    h2 v = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(int, v);
  }
  FRISK_DEV float add_pair(int pair, float acc) { return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, pair), h2{(_Float16)1, (_Float16)1}, acc, false); }
};
template <> struct Pack16<FRISK_BF16> {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  FRISK_DEV int two(float a, float b) {
    b2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(int, v);
  }
  FRISK_DEV float add_pair(int pair, float acc) { return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, pair), b2{(__bf16)1.f, (__bf16)1.f}, acc, false); }
};

// The exponent reference of a query row is only raised when the row maximum has grown by more than this many powers
// of two since it was last set: the accumulators are then rescaled (rarely), and probabilities stay below 2^8.
// The final division by the denominator makes the result independent of the reference.
constexpr float kAttnRescaleSlack = 8.f;

constexpr int kAttnPrefetch = 4;  // MFMA units between a fragment's LDS read and its use

template <class C>
__global__ void __launch_bounds__(C::NW * 64) attention_kernel(AttentionParams p) {
  typedef typename C::M M;
  typedef typename C::LK LK;
  typedef typename C::LV LV;
  typedef TileStager<LK, C::SW> SK;
  typedef TileStager<LV, C::SW> SV;
  typedef FragReader<LK, 16, C::KA, C::D / 16> RK;
  typedef PermutedKeyReader<LV> RV;
  typedef Pack16<C::DT> PK;
  constexpr int D = C::D, KB = C::KB, KA = C::KA, DA = C::DA, DSTEPS = D / 16, KSTEPS = KB / 16;
  constexpr int N1 = DSTEPS * KA;   // MFMAs of the first product per tile
  constexpr int N2 = KSTEPS * DA;   // MFMAs of the second product per tile
  constexpr int NE = KA * 16;       // scores per lane per tile
  static_assert(N1 == N2 && NE == 2 * N1, "the interleaving below is written for 32 or 64 keys x 128 head_dim");

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const unsigned smem_u = (unsigned)(uintptr_t)(FRISK_LDS char*)smem;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int share = wave / C::SW, swave = wave % C::SW;  // which keys, and which of the waves that walk them
  const unsigned k_ring = smem_u + share * C::RING_BYTES, v_ring = k_ring + C::NSK * LK::BYTES;
  const int lq = lane & 31, lh = lane >> 5;

  // consecutive work-group ids go to the 8 XCDs round-robin: give each XCD whole heads
  int cid = blockIdx.x;
  if (p.xcd_remap) {
    const int per = gridDim.x >> 3;
    if (cid < per * 8) cid = (cid & 7) * per + (cid >> 3);
  }
  const int bh = cid / p.q_blocks, qb = cid % p.q_blocks;
  const int64_t q0 = (int64_t)qb * C::QB + swave * C::QW;

  // the share's key tiles: `nkt` of them from `first` on; the work-group walks as many steps as its longest share has tiles
  const int tiles = p.seq_k / KB;
  const int nkt = C::KS == 1 ? tiles : tiles / C::KS + (share < tiles % C::KS ? 1 : 0), steps = C::KS == 1 ? tiles : (tiles + C::KS - 1) / C::KS;
  const int64_t first = C::KS == 1 ? 0 : (int64_t)share * (tiles / C::KS) + (share < tiles % C::KS ? share : tiles % C::KS);

  // Q fragments for the whole kernel: lane (q, g) holds Q[q][16 ks + 8 g .. + 7]
  v4i qf[DSTEPS];
  {
    const char* qbase = (const char*)p.Q + (((int64_t)bh * p.seq_q + q0 + lq) * D + 8 * lh) * 2;
#pragma unroll
    for (int ks = 0; ks < DSTEPS; ++ks) qf[ks] = *(const v4i*)(qbase + 32 * ks);
  }

  // staging: wave-uniform tile pointers plus one lane offset per operand
  const int64_t k_ld = C::KT ? (int64_t)p.seq_k * 2 : (int64_t)D * 2;
  const int64_t k_step = C::KT ? (int64_t)KB * 2 : (int64_t)KB * D * 2;
  const char* srcK = (const char*)p.K + (int64_t)bh * p.seq_k * D * 2 + first * k_step + SK::wave_src_offset(swave, k_ld);
  const char* srcV = (const char*)p.V + ((int64_t)bh * p.seq_k + first * KB) * D * 2 + SV::wave_src_offset(swave, D * 2);
  unsigned voffK[SK::PER_WAVE], voffV[SV::PER_WAVE];
#pragma unroll
  for (int i = 0; i < SK::PER_WAVE; ++i) voffK[i] = SK::transfer_src_offset(i, lane, swave, k_ld);
#pragma unroll
  for (int i = 0; i < SV::PER_WAVE; ++i) voffV[i] = SV::transfer_src_offset(i, lane, swave, D * 2);
  constexpr int PER_TILE = SK::PER_WAVE + SV::PER_WAVE;
  int k_slot_issue = 0, v_slot_issue = 0;
  auto stage_k = [&]() {
    const unsigned dst = k_ring + k_slot_issue * LK::BYTES + (unsigned)swave * 1024u;
#pragma unroll
    for (int i = 0; i < SK::PER_WAVE; ++i) SK::issue_one(i, srcK, voffK, dst);
    srcK += k_step;
    k_slot_issue = k_slot_issue == C::NSK - 1 ? 0 : k_slot_issue + 1;
  };
  auto stage_v = [&]() {
    const unsigned dst = v_ring + v_slot_issue * LV::BYTES + (unsigned)swave * 1024u;
#pragma unroll
    for (int i = 0; i < SV::PER_WAVE; ++i) SV::issue_one(i, srcV, voffV, dst);
    srcV += (int64_t)KB * D * 2;
    v_slot_issue = v_slot_issue == C::NSV - 1 ? 0 : v_slot_issue + 1;
  };

  unsigned rk[RK::NREG], rv[DA];
  RK::init(lane, 0, 0, rk);
#pragma unroll
  for (int da = 0; da < DA; ++da) rv[da] = RV::lane_reg(lane, da);

  v16f o[DA];
#pragma unroll
  for (int da = 0; da < DA; ++da)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[da][r] = 0.f;
  float l_run = 0.f;  // this lane's part of the denominator (its half of the keys of every tile)

  const float c = p.scale_log2;
  // One tile of work is an M phase (32 MFMAs: second product of tile j, then scores of tile j+1) and a V phase
  // (probabilities of a tile: maximum, exp2, rounding, denominator).  The two waves that share a SIMD run them in
  // opposite order -- waves 0-3 do V then M between two barriers, waves 4-7 M then V, half a tile behind -- so one
  // wave's MFMAs always run beside the other wave's VALU work.
  v16f s[KA];
  v4i pf[KSTEPS];
  // exponent reference of this lane's query.  A share whose scores are all -inf must come out as zeros beside the others, so
  // it starts from a finite number there (2^(-inf - m) is 0)
  float m_run = C::KS == 1 ? -INFINITY : -3e38f;
  auto k_read = [&](const unsigned* ck, int u, int* f) { RK::read(ck, u % KA, u / KA, f); };
  auto v_read = [&](unsigned vbase, int u, int* f) { RV::read(rv[u % DA] + vbase, u / DA, f); };
  // M phase of tile j: o += V_j^T P_j^T (unit u: key step u / DA, head_dim atom u % DA), then, if `scores`,
  // s = K_{j+1} Q^T (unit u: head_dim step u / KA, key atom u % KA).  Fragments are read two units ahead.
  auto m_phase = [&](unsigned vbase, unsigned kbase, bool scores) {
    // the MFMAs of this wave go before the vector instructions of the wave it shares the SIMD with, which fill the slots between them
    // (us without / with: f16 32 x 4096 x 4096 248.1 / 245.8, bf16 with K stored [128][seq_k] 237.8 / 232.2, f16 16 x 2048 x 2048 38.9 / 37.8; the
    // softmax phase first instead: 250.8, 236.8, 39.9)
    __builtin_amdgcn_s_setprio(1);
    unsigned ck[RK::NREG];
#pragma unroll
    for (int r = 0; r < RK::NREG; ++r) ck[r] = rk[r] + kbase;
    // fragment of unit x (0 .. N2-1: V, N2 .. N2+N1-1: K) goes to f[x % NB], read PF units ahead of its MFMA
    constexpr int PF = kAttnPrefetch, NB = PF + 1;
    int f[NB][4];
    const int last = scores ? N2 + N1 : N2;
    auto fetch = [&](int x) {
      if (x < N2) v_read(vbase, x, f[x % NB]);
      else if (x < last) k_read(ck, x - N2, f[x % NB]);
    };
#pragma unroll
    for (int x = 0; x < PF; ++x) fetch(x);
#pragma unroll
    for (int u = 0; u < N2; ++u) {
      const v4i vfrag = {f[u % NB][0], f[u % NB][1], f[u % NB][2], f[u % NB][3]};
      M::run(vfrag, pf[u / DA], o[u % DA]);
      fetch(u + PF);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (scores) {
#pragma unroll
      for (int u = 0; u < N1; ++u) {
        const int x = u + N2;
        const v4i kfrag = {f[x % NB][0], f[x % NB][1], f[x % NB][2], f[x % NB][3]};
        if (u < KA) s[u % KA] = v16f{};  // folds into the MFMA's C operand: no registers are cleared
        M::run(kfrag, qf[u / KA], s[u % KA]);
        fetch(x + PF);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // V phase: probabilities of the tile whose scores are in s.  Score e of the lane, e = 16 ka + r, belongs to
  // 16-key step e / 8.
  auto v_phase = [&]() {
    float mx = s[0][0];
#pragma unroll
    for (int ka = 0; ka < KA; ++ka)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[ka][r]);
    {
      // lanes l and l ^ 32 hold the two halves of a query's keys.  One v_permlane32_swap of two copies of the value leaves
      // the lower half's maximum in every lane of one result and the upper half's in the other; unlike a shuffle it
      // does not go through the LDS queue (291 against 300 us at 32 x 4096 x 4096)
      const int mine = __builtin_bit_cast(int, mx);
      const auto both = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
      mx = fmaxf(__builtin_bit_cast(float, (int)both[0]), __builtin_bit_cast(float, (int)both[1])) * c;
    }
    if (__builtin_amdgcn_ballot_w64(mx > m_run + kAttnRescaleSlack) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int da = 0; da < DA; ++da)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[da][r] *= alpha;
    }
    float l_part[4] = {l_run, 0.f, 0.f, 0.f};  // four chains instead of one of 16 dependent additions
#pragma unroll
    for (int e = 0; e < NE; e += 2) {
      const float x0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e / 16][e % 16], c, -m_run));
      const float x1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e / 16][e % 16 + 1], c, -m_run));
      const int pair = PK::two(x0, x1);
      pf[e / 8][(e % 8) / 2] = pair;
      l_part[(e / 2) % 4] = PK::add_pair(pair, l_part[(e / 2) % 4]);
      if (e % 8 == 6) __builtin_amdgcn_sched_barrier(0);  // keeps the scheduler from holding all 32 exponentials in flight
    }
    // The probabilities are only used by the MFMAs of the M phase, two barriers away: left alone, the compiler sinks
    // the whole computation there.  Pin the values to this phase.
#pragma unroll
    for (int t = 0; t < KSTEPS; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(pf[t][j]));
    l_run = (l_part[0] + l_part[1]) + (l_part[2] + l_part[3]);
    asm volatile("" : "+v"(l_run));
  };

  // prologue: the first AHEAD tiles in flight, scores of tile 0
  constexpr int AHEAD = C::NSK;
  static_assert(AHEAD >= 1 && AHEAD <= 3, "the waits below");
  static_for<0, AHEAD>([&](auto t) FRISK_LAMBDA_INLINE {
    if (decltype(t)::value < nkt) {
      stage_k();
      if (AHEAD > 1) stage_v();
    }
  });
  if (AHEAD > 2 && nkt > 2) wait_vmcnt<2 * PER_TILE>(); else if (AHEAD > 1 && nkt > 1) wait_vmcnt<PER_TILE>(); else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  {
    unsigned ck[RK::NREG];
#pragma unroll
    for (int r = 0; r < RK::NREG; ++r) ck[r] = rk[r] + k_ring;
#pragma unroll
    for (int ka = 0; ka < KA; ++ka)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[ka][r] = 0.f;
#pragma unroll
    for (int u = 0; u < N1; ++u) {
      int f[4];
      k_read(ck, u, f);
      const v4i kfrag = {f[0], f[1], f[2], f[3]};
      M::run(kfrag, qf[u / KA], s[u % KA]);
    }
  }
  asm volatile("" ::: "memory");  // the reads above stay in front of the barriers below
  __builtin_amdgcn_sched_barrier(0);

  // Every wave runs the same loop -- barrier, V(kt), barrier, M(kt) -- but waves 4-7 pass one extra barrier first,
  // which puts them half an iteration behind waves 0-3 for the whole kernel (waves 0-3 pass the matching barrier at
  // the end).  Before either barrier of iteration kt a wave's share of tile kt+1 has landed (at most tile kt+2 is
  // outstanding), so tile kt+1 is complete in LDS before any wave's M(kt); when a wave stages tile kt+3, every wave
  // has passed the barrier that follows its M(kt-1), the last reader of K tile kt and V tile kt-1.
  // With several shares the waves of a share run in step (they are all among 0-3 or among 4-7), so only the barrier before M
  // publishes their tiles, and the same holds with tiles staged two ahead instead of three: tile kt+1 is then all that is
  // outstanding there.  With single buffers the barrier before V(kt) follows M(kt-1), the last reader of what is overwritten.
  // A share with a tile less than the longest idles through the last step.
  const bool trails = wave >= C::NW / 2;
  if (trails) __builtin_amdgcn_s_barrier();
  int k_slot = C::NSK > 1, v_slot = 0;  // ring slots M(kt) reads: K tile kt+1 and V tile kt
  for (int kt = 0; kt < steps; ++kt) {
    if constexpr (C::KS == 1) {
      if (kt + 2 < nkt) wait_vmcnt<PER_TILE>(); else wait_vmcnt<0>();
    } else {
      asm volatile("" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);  // the phases are register-only work: without these the compiler moves it across the barriers
    if (AHEAD == 1) {
      if (kt + 1 < nkt) stage_k();
      if (kt < nkt) stage_v();
    }
    if (C::KS == 1 || kt < nkt) v_phase();
    __builtin_amdgcn_sched_barrier(0);
    if (AHEAD > 2 && kt + 2 < nkt) wait_vmcnt<PER_TILE>(); else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (AHEAD > 1 && kt + AHEAD < nkt) {
      stage_k();
      stage_v();
    }
    if (C::KS == 1 || kt < nkt) m_phase(v_ring + v_slot * LV::BYTES, k_ring + k_slot * LK::BYTES, kt + 1 < nkt);
    __builtin_amdgcn_sched_barrier(0);
    k_slot = k_slot == C::NSK - 1 ? 0 : k_slot + 1;
    v_slot = v_slot == C::NSV - 1 ? 0 : v_slot + 1;
  }
  if (!trails) __builtin_amdgcn_s_barrier();

  if constexpr (C::KS > 1) {
    // Every wave leaves its unscaled O and its (reference, denominator) pairs in LDS; then the waves of the KS shares of a
    // 32-query atom take 32 / KS of its queries each: O = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s, M the largest m_s.
    __syncthreads();  // the rings are done with
    typedef float v2f __attribute__((ext_vector_type(2)));
    const float l = l_run + __shfl_xor(l_run, 32);
    const unsigned mine = smem_u + (wave * 32 + lq) * C::MERGE_ROW;
#pragma unroll
    for (int da = 0; da < DA; ++da)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *(FRISK_LDS v4f*)(uintptr_t)(mine + (32 * da + 8 * r4 + 4 * lh) * 4) = v4f{o[da][4 * r4], o[da][4 * r4 + 1], o[da][4 * r4 + 2], o[da][4 * r4 + 3]};
    if (lh == 0) *(FRISK_LDS v2f*)(uintptr_t)(smem_u + C::MERGE_STATS + (wave * 32 + lq) * 8) = v2f{m_run, l};
    __syncthreads();
    char* obase = (char*)p.O + ((int64_t)bh * p.seq_q + q0) * D * 2;
#pragma unroll
    for (int j = 0; j < 32 / C::KS / 4; ++j) {
      const int q = share * (32 / C::KS) + 4 * j + (lane >> 4), col = 8 * (lane & 15);
      float m[C::KS], den[C::KS], top = -INFINITY, total = 0.f, out[8] = {};
#pragma unroll
      for (int s2 = 0; s2 < C::KS; ++s2) {
        const v2f st = *(const FRISK_LDS v2f*)(uintptr_t)(smem_u + C::MERGE_STATS + ((s2 * C::SW + swave) * 32 + q) * 8);
        m[s2] = st[0];
        den[s2] = st[1];
        top = fmaxf(top, m[s2]);
      }
#pragma unroll
      for (int s2 = 0; s2 < C::KS; ++s2) {
        m[s2] = __builtin_amdgcn_exp2f(m[s2] - top);
        total += m[s2] * den[s2];
      }
      const float inv = 1.f / total;
#pragma unroll
      for (int s2 = 0; s2 < C::KS; ++s2) {
        const unsigned from = smem_u + ((s2 * C::SW + swave) * 32 + q) * C::MERGE_ROW + col * 4;
        const v4f a = *(const FRISK_LDS v4f*)(uintptr_t)from, b = *(const FRISK_LDS v4f*)(uintptr_t)(from + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[e] += m[s2] * a[e];
          out[4 + e] += m[s2] * b[e];
        }
      }
      v4i w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = PK::two(out[2 * e] * inv, out[2 * e + 1] * inv);
      FRISK_STORE_C((v4i*)(obase + (int64_t)q * D * 2 + col * 2), w);
      if (p.lse && col == 0) p.lse[(int64_t)bh * p.seq_q + q0 + q] = (top + __builtin_amdgcn_logf(total)) * 0.6931471805599453f;
    }
    return;
  }

  // O = O^T / l.  Lane (q, h) holds head_dim columns 32 da + 8 (r/4) + 4 h + r%4 of its query: 8-byte pieces.  They
  // go through a wave-private LDS region (64 columns at a time, rows padded by 16 B) and come back as 16-byte
  // pieces, 8 lanes per row, so that every global store covers whole 128-byte lines of O.  LDS operations of one
  // wave execute in order and the region lies behind the rings, which other waves may still be reading.
  {
    const float l = l_run + __shfl_xor(l_run, 32);
    const float inv = 1.f / l;
    const int64_t row = (int64_t)bh * p.seq_q + q0 + lq;
    constexpr int OROW = 64 * 2 + 16;
    const unsigned region = smem_u + C::RING_BYTES + wave * C::OUT_BYTES_PER_WAVE;
    char* obase = (char*)p.O + ((int64_t)bh * p.seq_q + q0) * D * 2;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int d2 = 0; d2 < 2; ++d2)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int da = 2 * half + d2;
          v2i w;
          w[0] = PK::two(o[da][4 * r4] * inv, o[da][4 * r4 + 1] * inv);
          w[1] = PK::two(o[da][4 * r4 + 2] * inv, o[da][4 * r4 + 3] * inv);
          *(FRISK_LDS v2i*)(uintptr_t)(region + lq * OROW + (32 * d2 + 8 * r4 + 4 * lh) * 2) = w;
        }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int orow = (lane >> 3) + 8 * j, chunk = lane & 7;
        const v4i w = *(const FRISK_LDS v4i*)(uintptr_t)(region + orow * OROW + chunk * 16);
        FRISK_STORE_C((v4i*)(obase + (int64_t)orow * D * 2 + (64 * half + 8 * chunk) * 2), w);
      }
    }
    if (p.lse && lh == 0) p.lse[row] = (m_run + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
  }
}

// A group of 256 queries takes one CU, so few heads or short query sequences leave most of the chip idle: 8 heads x 256 queries are
// 8 work-groups.  With the keys dealt to `shares` sets of waves inside a work-group it owns 256 / shares queries and walks 1 / shares
// of the key tiles, and shares times as many work-groups exist; nothing but the merge in LDS at the end is added, no second launch
// and no scratch memory.  Each K and V tile then feeds fewer queries, so on a full chip fewer shares are better.  The line is drawn
// by a time model: per round of 256 work-groups 3.5 us (prologue, merge, stores) and per step `part` us while the chip is nearly
// empty up to `full` when every CU is busy (power and L2).  Measured, us, 1 / 2 / 4 / 8 shares (heads x seq_q x seq_k, f16):
//   8 x 256 x 256    10.8 /  9.5 /  8.0 /  7.3      8 x 256 x 4096   90.6 / 58.1 / 30.7 / 26.5    32 x 256 x 960   25.5 / 18.8 / 13.1 / 12.1
//   32 x 512 x 1600  39.6 / 28.1 / 19.6 / 29.1      16 x 2048 x 2048 50.0 / 39.0 / 42.8 / 62.3    32 x 2048 x 512  20.8 / 26.0 / 34.2 / 56.9
//   36 x 2048 x 2048 (288 groups of 256) 113.0 / 106.7 / 100.5 / 146.9
int attention_key_shares(int64_t groups, int64_t seq_k) {
  static constexpr struct { int shares, keys; double part, full; } kinds[] = {{1, 64, 1.33, 1.9}, {2, 64, 1.6, 2.1}, {4, 64, 1.5, 2.1}, {8, 32, 1.27, 1.85}};
  if (groups > 1024) return 1;
  int best = 1;
  double best_time = 0;
  for (const auto& k : kinds) {
    const int64_t tiles = seq_k / k.keys, steps = (tiles + k.shares - 1) / k.shares, wgs = groups * k.shares;
    if (tiles < k.shares) break;  // every share has a tile
    const double rounds = (double)(wgs / 256), rest = (double)(wgs % 256) / 256;
    const double time = rounds * (3.5 + (double)steps * k.full) + (rest > 0 ? 3.5 + (double)steps * (k.part + (k.full - k.part) * rest) : 0.0);
    if (k.shares == 1 || time < 0.97 * best_time) {
      best = k.shares;
      best_time = time;
    }
  }
  return best;
}

template <class C> static hipError_t prepare_one() {
  return hipFuncSetAttribute((const void*)attention_kernel<C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
}
// the configurations a launch chooses from, by number of shares
template <int DT, bool KT, class F> static hipError_t with_shares(int shares, F&& f) {
  if (shares == 8) return f(AttnCfg<DT, KT, 8, 32, 1>{});
  if (shares == 4) return f(AttnCfg<DT, KT, 4, 64, 1>{});
  if (shares == 2) return f(AttnCfg<DT, KT, 2, 64, 2>{});
  return f(AttnCfg<DT, KT, 1, 64, 3>{});
}
template <class F> static hipError_t with_config(int dtype, int k_transposed, int shares, F&& f) {
  if (dtype == FRISK_F16) return k_transposed ? with_shares<FRISK_F16, true>(shares, f) : with_shares<FRISK_F16, false>(shares, f);
  return k_transposed ? with_shares<FRISK_BF16, true>(shares, f) : with_shares<FRISK_BF16, false>(shares, f);
}

// Raising the dynamic-LDS cap is not a stream operation and must precede a captured launch; done once per process.
hipError_t prepare_attention() {
  static std::atomic<bool> done{false};
  if (done.load(std::memory_order_acquire)) return hipSuccess;
  for (const int dtype : {FRISK_F16, FRISK_BF16})
    for (const int k_transposed : {0, 1})
      for (const int shares : {1, 2, 4, 8})
        if (hipError_t e = with_config(dtype, k_transposed, shares, [](auto c) { return prepare_one<decltype(c)>(); }); e != hipSuccess) return e;
  done.store(true, std::memory_order_release);
  return hipSuccess;
}

template <class C> static hipError_t launch_one(AttentionParams p, hipStream_t stream) {
  p.q_blocks = p.seq_q / C::QB;
  const int64_t groups = (int64_t)p.batch_heads * p.q_blocks;
  p.xcd_remap = groups % 8 == 0 ? 1 : 0;
  hipLaunchKernelGGL(attention_kernel<C>, dim3((unsigned)groups), dim3(C::NW * 64), C::LDS_BYTES, stream, p);
  return hipGetLastError();
}

hipError_t launch_attention(int dtype, int k_transposed, const AttentionParams& p, hipStream_t stream) {
  if (hipError_t e = prepare_attention(); e != hipSuccess) return e;
  const int shares = attention_key_shares((int64_t)p.batch_heads * (p.seq_q / kAttnQueriesPerGroup), p.seq_k);
  return with_config(dtype, k_transposed, shares, [&](auto c) { return launch_one<decltype(c)>(p, stream); });
}

}  // namespace frisk
