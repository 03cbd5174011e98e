// dK/dV (and with it, in one launch, dQ) of problems that leave CUs idle, 16-bit elements, D = 64 and 128.
//
// What such a launch waits for is the chain of one key tile: every query row that sees it, of every query head of its group.  So
// the four waves of a workgroup own the SAME 32 keys, and each takes every fourth block of 32 rows -- counted through the
// heads of the group -- through a buffer of LDS of its own: no barrier until the waves' sums are added up at the end, in
// their order.  (The forms of fa_bwd_dkdv.hip give every wave, or pair of waves, keys of its own and walk all rows with each:
// 32 on 8 heads x 1339 rows, D = 64: 120 us for one long chain per 128 keys on 88 CUs, 75 here.)  A block of 32 x 32 pairs costs about
// 1.4 us at D = 128, one wave to a SIMD, against 0.5 of its MFMAs: the reads of both operands from LDS count as much, and at
// D = 128 a workgroup holds the whole LDS.  Hence for few workgroups only: see bwd_small.
#include "fa_tile.h"
#ifdef FA_TRACE
namespace fa { namespace { FA_TRACE_ARRAY(g_trace_dq); } }   // stamps of dq workgroups that share a launch: not read
// words as in fa_bwd_dkdv.hip, of the first wave; its tiles are blocks of 32 rows
namespace fa { FA_TRACE_ARRAY(g_trace_small); }
#endif
#include "fa_dq_body.h"

namespace fa {
namespace {

constexpr int kWaves = 4;
constexpr int kRb = 32;        // rows of a block, keys of a workgroup
constexpr int dkdv_small_sub(int D) { return (D > 64 ? kSeqKeyTile : 128) / kRb; }   // workgroups to a key tile of the packed plan

template <int D> constexpr int rows_bytes() { return kRb * D * 2; }
template <int D> constexpr int stage_bytes() { return 2 * rows_bytes<D>() + 512; }   // Q, dO, [LSE, delta, id, name of a row]
template <int D> constexpr size_t small_lds() {
  constexpr size_t stages = size_t(2 * kWaves) * stage_bytes<D>(), sums = size_t(kWaves) * 2 * kRb * D * 4;
  return stages > sums ? stages : sums;
}

// 32 gathered rows on their way into a wave's buffer
template <int D>
struct RowStream {
  static constexpr int CPR = D / 8, RPI = 64 / CPR, NI = kRb / RPI;
  // rel(r): the row that goes to place r, or -1 (reads as zero, like any beyond the matrix)
  template <class F>
  FA_DEV static void issue(const buf_rsrc_t rsrc, const int row_bytes, char* lds, const F& rel) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = i * RPI + lane / CPR, row = rel(r);
      const int c = (lane % CPR) ^ swz<D, SWZ_ROW>(r);
      buf_load_lds16(rsrc, lds + i * 1024, row >= 0 ? row * row_bytes + c * 16 : kOobOffset, 0);
    }
  }
};

// Number k * kWaves + wave of the blocks that may hold a kept pair, through the heads of the group; all of it wave-uniform.
// Blocks are named by their 32 rows' place in the natural order, or (ids) in the order of the mask plan.
template <bool CAUSAL, bool DOC>
struct BlockIter {
  int gi, base, t_last, cnt;
  unsigned long long mask, full;   // candidates of 64 rows from `base` on; those with more than 32 rows
  int half;                        // 0, 1: which half of the lowest candidate is next
  int ek, k_lo, k_hi;              // this lane's key id under head gi, and the span of the workgroup's
  int r_lo, r_hi;                  // (no ids) rows that may see a key of the workgroup

  template <class Head, class Chunk>
  FA_DEV void init(const Head& head, const Chunk& chunk, int lo, int hi) {
    r_lo = lo; r_hi = hi; cnt = 0; gi = 0; half = 0;
    head(*this);
    start(chunk);
  }
  template <class Chunk>
  FA_DEV void start(const Chunk& chunk) {
    base = DOC ? 0 : (r_lo / 64) / 64 * 64;
    mask = 0;
    if (base < t_last) chunk(*this);
  }
  // next block of this wave: its number of 32 rows, or -1; `gi` is its head
  template <class Head, class Chunk>
  FA_DEV int next(const int G, const int wave, const Head& head, const Chunk& chunk) {
    for (;;) {
      while (mask == 0) {
        base += 64;
        if (base < t_last) { chunk(*this); continue; }
        if (++gi >= G) { mask = 0; gi = G; base = t_last; return -1; }
        head(*this);
        start(chunk);
      }
      const int j = __builtin_ctzll(mask), blk = 2 * (base + j) + half;
      const bool there = DOC ? (half == 0 || ((full >> j) & 1) != 0) : (32 * blk <= r_hi && 32 * blk + 31 >= r_lo);
      if (half == 1) mask &= mask - 1;
      half ^= 1;
      if (!there) continue;
      if ((cnt++ & (kWaves - 1)) == wave) return blk;
    }
  }
};

template <typename Tag, int D, bool CAUSAL, bool DOC, bool OWN_DELTA>
FA_DEV void dkdv_small_body(const KArgs& a, const int bid, char* smem) {
  using E = Elem<Tag>;
  using T = typename E::scalar;
  using vec8 = typename E::vec8;
  constexpr int KS = D / 16, DBN = D / 32, RB = rows_bytes<D>();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lq = lane & 31, g = lane >> 5;
  const bool packed = !DOC && a.ktab != nullptr;
  constexpr int SUB = dkdv_small_sub(D);
  FA_STAMP(g_trace_small, 0, FA_CLOCK()); FA_STAMP(g_trace_small, 1, 0); FA_STAMP(g_trace_small, 5, 0); FA_STAMP(g_trace_small, 7, -1);
  FA_TRACE_ONLY(int tr_tiles = 0;)
  int slot, bhk;
  if (!block_to_tile(packed ? a.nKent * SUB : (a.N + kRb - 1) / kRb, a.B * a.Hk, true, slot, bhk, bid)) return;
  const int b = bhk / a.Hk, hk = bhk % a.Hk;
  int M = a.M, N = a.N, gap = a.gap, n0 = slot * kRb;
  int64_t q0 = 0, k0 = 0;
  if (packed) {
    if (slot / SUB >= a.shdr->nk) return;
    const SeqTile* __restrict__ e = a.ktab + slot / SUB;
    M = __builtin_amdgcn_readfirstlane(e->M); N = __builtin_amdgcn_readfirstlane(e->N); gap = __builtin_amdgcn_readfirstlane(e->gap);
    q0 = __builtin_amdgcn_readfirstlane(e->q0); k0 = __builtin_amdgcn_readfirstlane(e->k0);
    n0 = (__builtin_amdgcn_readfirstlane(e->tile) * SUB + slot % SUB) * kRb;
    if (n0 >= N) return;
  }
  const int key = n0 + lq, keyc = min(key, N - 1);
  FA_STAMP(g_trace_small, 7, (long long)(n0 / kRb) | ((long long)bhk << 16));
  vec8 kf[KS], vf[KS];
  {
    const T* kp = reinterpret_cast<const T*>(a.k) + b * a.k_bs + hk * a.k_hs + (k0 + keyc) * a.k_rs;
    const T* vp = reinterpret_cast<const T*>(a.v) + b * a.v_bs + hk * a.v_hs + (k0 + keyc) * a.v_rs;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = *reinterpret_cast<const vec8*>(kp + ks * 16 + g * 8);
      vf[ks] = *reinterpret_cast<const vec8*>(vp + ks * 16 + g * 8);
    }
  }
  // rows that may see this lane's key, by name (index, or with ids the diagonal position of the plan): [row_lo, row_lo + row_span)
  const int gk = DOC ? 0 : gap, rcap = DOC ? kPosMax : M - 1;
  const int row_lo = CAUSAL ? (key <= a.pfx_m1 ? 0 : max(0, key - gk)) : 0;
  const int row_hi = CAUSAL ? min(rcap, key - gk + a.win - 1) : rcap;
  const unsigned row_span = (key < N && row_hi >= row_lo) ? (unsigned)(row_hi - row_lo + 1) : 0u;
  const int wg_rlo = CAUSAL ? (n0 <= a.pfx_m1 ? 0 : max(0, n0 - gk)) : 0;
  const int wg_rhi = CAUSAL ? min(rcap, n0 + kRb - 1 - gk + a.win - 1) : rcap;

  f32x16 dv[DBN], dk[DBN];
#pragma unroll
  for (int db = 0; db < DBN; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dv[db][r] = dk[db][r] = 0.f;
  LdsOffsets<D> lo;
  lo.init();

  using Iter = BlockIter<CAUSAL, DOC>;
  auto head = [&](Iter& it) __attribute__((always_inline)) {   // what the blocks of head it.gi depend on
    it.t_last = DOC ? a.nQs : (wg_rhi < wg_rlo ? 0 : wg_rhi / 64 + 1);
    it.ek = 0;
    if (DOC) {
      it.ek = a.ek32[b * a.ek_bs + (hk * a.G + it.gi) * a.ek_hs + keyc];
      int lo_ = key < N ? it.ek : 0x7fffffff, hi_ = key < N ? it.ek : (int)0x80000000;
#pragma unroll
      for (int off = 16; off >= 1; off >>= 1) { lo_ = min(lo_, __shfl_xor(lo_, off)); hi_ = max(hi_, __shfl_xor(hi_, off)); }
      it.k_lo = lo_; it.k_hi = hi_;
    }
  };
  auto chunk = [&](Iter& it) __attribute__((always_inline)) {   // 64 candidates, one per lane
    const int t = it.base + lane, h = hk * a.G + it.gi;
    bool v = t < it.t_last, f = true;
    if (DOC) {
      if (v) {
        const IdSummary qs = a.qsum[b * a.qs_bs + h * a.qs_hs + t];
        v = qs.nvalid > 0 && doc_may_keep(qs.lo, qs.hi, qs.glob, it.k_lo, it.k_hi) &&
            !(CAUSAL && ((qs.rmax < n0 && n0 > a.pfx_m1) || qs.rmin > wg_rhi));
        f = qs.nvalid > 32;
      }
    } else {
      v = v && 64 * t + 63 >= wg_rlo;
      if (v && a.bmask != nullptr) v = a.bmask[b * a.bm_bs + h * a.bm_hs + int64_t(t) * a.bm_rs + n0 / FA_MASK_BLOCK] != 0;
    }
    it.mask = __builtin_amdgcn_ballot_w64(v);
    it.full = __builtin_amdgcn_ballot_w64(f);
  };

  char* const mine = smem + wave * (2 * stage_bytes<D>());
  // With ids: this lane's row (place lane % 32 of a block), fetched a block ahead of the loads that need it.
  auto place = [&](const int blk, const int gi) __attribute__((always_inline)) -> int {
    return a.perm[b * a.pm_bs + (hk * a.G + gi) * a.pm_hs + 32 * blk + lq];
  };
  vec8 of[KS] = {}, of_n[KS] = {};   // (OWN_DELTA) the lane's part of its row of O: of the block at hand, and of the next
  auto load = [&](const int blk, const int gi, int idx, char* st) __attribute__((always_inline)) {
    const int h = hk * a.G + gi;
    if (DOC) settle(idx);   // (it has arrived: the caller waited)
    const T* qp = reinterpret_cast<const T*>(a.q) + b * a.q_bs + h * a.q_hs + q0 * a.q_rs;
    const T* dop = reinterpret_cast<const T*>(a.dout) + b * a.do_bs + h * a.do_hs + q0 * a.do_rs;
    const int own = DOC ? max(idx, 0) : min(32 * blk + lq, M - 1);
    const int64_t row_l = (int64_t(b) * a.H + h) * a.M + q0 + own;
    if (OWN_DELTA) {
      const T* op = reinterpret_cast<const T*>(a.o) + b * a.o_bs + h * a.o_hs + (q0 + own) * a.o_rs + g * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) of_n[ks] = *reinterpret_cast<const vec8*>(op + ks * 16);
    }
    auto rel = [&](const int r) __attribute__((always_inline)) { return DOC ? __shfl(idx, r) : 32 * blk + r; };
    auto rsrc = [&](const T* p, const int64_t rs) { return make_rsrc(p, M > 0 ? (unsigned)((int64_t(M - 1) * rs + D) * 2) : 0u); };
    RowStream<D>::issue(rsrc(qp, a.q_rs), int(a.q_rs) * 2, st, rel);
    RowStream<D>::issue(rsrc(dop, a.do_rs), int(a.do_rs) * 2, st + RB, rel);
    glb_load_lds4((!OWN_DELTA && g == 1 ? a.delta : a.lse) + row_l, st + 2 * RB);
    if (DOC) glb_load_lds4((g == 0 ? a.peq : a.ppos) + (b * a.pm_bs + h * a.pm_hs + 32 * blk + lq), st + 2 * RB + 256);
  };

  auto compute = [&](const int blk, const int ek, char* st) __attribute__((always_inline)) {
    const char* lds_q = st;
    const char* lds_do = st + RB;
    const char* aux = st + 2 * RB;
    // Operands are requested in batches ahead of the products that take them (left to itself the compiler puts a read, a full wait
    // and its MFMA back to back, and there is one wave or two to a SIMD to hide that).
    vec8 qa[KS], da[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) { qa[ks] = lds_row8<E>(lds_q + lo.row[ks]); da[ks] = lds_row8<E>(lds_do + lo.row[ks]); }
    __builtin_amdgcn_sched_barrier(0);
    f32x16 x, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = dp[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      x = E::mfma32(qa[ks], kf[ks], x);
      dp = E::mfma32(da[ks], vf[ks], dp);
    }
    // delta = rowsum(O * dO): of row l % 32, then, through LDS, of the rows of this lane's scores; in the order of delta_kernel, so that
    // the separate launches give the same bits
    if (OWN_DELTA) {
      const float part = row_delta<KS>(of, da);
      if (g == 0) *reinterpret_cast<float*>(st + 2 * RB + 128 + 4 * lq) = part;
      asm volatile("" ::: "memory");   // (LDS operations of a wave execute in order)
    }
    vec8 dt[2 * DBN], qt[2 * DBN];
    auto transposed = [&](const int i) __attribute__((always_inline)) {
      const int at = (i / DBN) * 16 * D * 2;
      dt[i] = lds_tr8<E>(lds_do + lo.tr[i % DBN][0] + at, lds_do + lo.tr[i % DBN][1] + at);
      qt[i] = lds_tr8<E>(lds_q + lo.tr[i % DBN][0] + at, lds_q + lo.tr[i % DBN][1] + at);
    };
    constexpr bool EARLY = D > 64;   // (two waves to a SIMD have no registers for that)
    if (EARLY) {
#pragma unroll
      for (int i = 0; i < 2 * DBN; ++i) transposed(i);
    }
    f32x4 Lv[4], dl[4];
    i32x4 eqv[4], nm[4];
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int i0 = 8 * q4 + 4 * g;
      Lv[q4] = *reinterpret_cast<const f32x4*>(aux + 4 * i0);
      dl[q4] = *reinterpret_cast<const f32x4*>(aux + 128 + 4 * i0);
      if (DOC) { eqv[q4] = *reinterpret_cast<const i32x4*>(aux + 256 + 4 * i0); nm[q4] = *reinterpret_cast<const i32x4*>(aux + 384 + 4 * i0); }
      else { eqv[q4] = i32x4{0, 0, 0, 0}; nm[q4] = i32x4{32 * blk + i0, 32 * blk + i0 + 1, 32 * blk + i0 + 2, 32 * blk + i0 + 3}; }
    }
    __builtin_amdgcn_sched_barrier(0);
    vec8 pf[2], sf[2];
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      float p[4], ds[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        bool keep = (unsigned)(nm[q4][t] - row_lo) < row_span;
        if (DOC) keep = keep && (eqv[q4][t] >= 0 || eqv[q4][t] == ek);
        const float e = fast_exp2(__builtin_fmaf(x[4 * q4 + t], a.scale_log2e, -Lv[q4][t]));
        p[t] = keep ? e : 0.f;
        ds[t] = keep ? e * (dp[4 * q4 + t] - dl[q4][t]) : 0.f;
      }
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        const typename E::vec2 pr = E::cvt2(p[t], p[t + 1]), sr = E::cvt2(ds[t], ds[t + 1]);
        const int i = 4 * (q4 & 1) + t;
        pf[q4 >> 1][i] = pr[0]; pf[q4 >> 1][i + 1] = pr[1];
        sf[q4 >> 1][i] = sr[0]; sf[q4 >> 1][i + 1] = sr[1];
      }
    }
#pragma unroll
    for (int i = 0; i < 2 * DBN; ++i) {
      if (!EARLY) transposed(i);
      dv[i % DBN] = E::mfma32(dt[i], pf[i / DBN], dv[i % DBN]);
      dk[i % DBN] = E::mfma32(qt[i], sf[i / DBN], dk[i % DBN]);
    }
    // Every read of this block ends up in a product above, so its wait stands above this line, and the loads that fill the buffer
    // again stand below it.  (A wait of its own there, or behind the reads, cost 3 - 14 % of a long chain through the schedule
    // around it.)
    __builtin_amdgcn_sched_barrier(0);
  };

  FA_STAMP(g_trace_small, 2, FA_CLOCK());
  Iter it;
  it.init(head, chunk, wg_rlo, wg_rhi);
  int cur = it.next(a.G, wave, head, chunk), ek = it.ek, gi = it.gi, idx = 0;
  if (cur >= 0) {
    if (DOC) idx = place(cur, gi);
    wait_async_loads();
    load(cur, gi, idx, mine);
  }
  int nxt = cur >= 0 ? it.next(a.G, wave, head, chunk) : -1, ek_n = it.ek, gi_n = it.gi, idx_n = 0;
  if (DOC && nxt >= 0) idx_n = place(nxt, gi_n);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) { settle(kf[ks]); settle(vf[ks]); }
  int buf = 0;
  while (cur >= 0) {
    wait_async_loads();
    FA_TRACE_ONLY(if (tr_tiles++ == 0) FA_STAMP(g_trace_small, 3, FA_CLOCK());)
    if (OWN_DELTA) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) { settle(of_n[ks]); of[ks] = of_n[ks]; }
    }
    int nx2 = -1, ek2 = 0, gi2 = 0, idx2 = 0;
    if (nxt >= 0) {
      load(nxt, gi_n, idx_n, mine + (buf ^ 1) * stage_bytes<D>());
      nx2 = it.next(a.G, wave, head, chunk); ek2 = it.ek; gi2 = it.gi;
      if (DOC && nx2 >= 0) idx2 = place(nx2, gi2);
    }
    compute(cur, ek, mine + buf * stage_bytes<D>());
    buf ^= 1;
    cur = nxt; ek = ek_n;
    nxt = nx2; ek_n = ek2; gi_n = gi2; idx_n = idx2;
  }

  FA_STAMP(g_trace_small, 4, FA_CLOCK()); FA_STAMP(g_trace_small, 6, tr_tiles);
  // the waves' sums, in their order: wave w adds up 32-column blocks w, w + 4, ... of dV and dK
  __syncthreads();
  f32x4* sums = reinterpret_cast<f32x4*>(smem) + lane;   // [wave][dV, dK blocks][quads of a lane's registers][lane]
  auto at = [&](const int w, const int blk, const int q4) { return ((w * 2 * DBN + blk) * 4 + q4) * 64; };
#pragma unroll
  for (int db = 0; db < DBN; ++db)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      sums[at(wave, db, q4)] = f32x4{dv[db][4 * q4], dv[db][4 * q4 + 1], dv[db][4 * q4 + 2], dv[db][4 * q4 + 3]};
      sums[at(wave, DBN + db, q4)] = f32x4{dk[db][4 * q4], dk[db][4 * q4 + 1], dk[db][4 * q4 + 2], dk[db][4 * q4 + 3]};
    }
  __syncthreads();
  if (key >= N) return;
#pragma unroll
  for (int i = 0; i < 2 * DBN / kWaves; ++i) {
    const int blk = i * kWaves + wave, db = blk % DBN;
    T* p = blk < DBN ? reinterpret_cast<T*>(a.dv) + b * a.dv_bs + hk * a.dv_hs + (k0 + key) * a.dv_rs
                     : reinterpret_cast<T*>(a.dk) + b * a.dk_bs + hk * a.dk_hs + (k0 + key) * a.dk_rs;
    const float sc = blk < DBN ? 1.f : a.scale;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      f32x4 v = sums[at(0, blk, q4)];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) v += sums[at(w, blk, q4)];
      const typename E::vec2 x0 = E::cvt2(v[0] * sc, v[1] * sc), x1 = E::cvt2(v[2] * sc, v[3] * sc);
      typename E::vec4 x = {x0[0], x0[1], x1[0], x1[1]};
      *reinterpret_cast<typename E::vec4*>(p + 32 * db + 8 * q4 + 4 * g) = x;
    }
  }
  FA_STAMP(g_trace_small, 5, FA_CLOCK());
}

template <int D> constexpr int kPerSimd = D > 64 ? 1 : 2;

template <typename Tag, int D, bool CAUSAL, bool DOC>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kPerSimd<D>, kPerSimd<D>)))
void dkdv_small_kernel(const KArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  dkdv_small_body<Tag, D, CAUSAL, DOC, false>(a, (int)blockIdx.x, smem);
}
template <typename Tag, int D, bool CAUSAL, int MODE>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kPerSimd<D>, kPerSimd<D>)))
void bwd_small_kernel(const KArgs a, const int n_dkdv) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int bid = (int)blockIdx.x;
  if (bid < n_dkdv) dkdv_small_body<Tag, D, CAUSAL, MODE == GEO_DOC, true>(a, bid, smem);   // the longer ones first
  else dq_body<Tag, D, CAUSAL, MODE>(a, bid - n_dkdv, smem);
}

int dkdv_blocks(const KArgs& a, int D, bool doc) {
  const int slots = !doc && a.ktab != nullptr ? a.nKent * dkdv_small_sub(D) : (a.N + kRb - 1) / kRb;
  return grid_blocks(slots, a.B * a.Hk);
}

template <typename Tag, int D, bool CAUSAL, bool DOC>
int launch_dkdv(const KArgs& a, hipStream_t s) {
  auto kern = dkdv_small_kernel<Tag, D, CAUSAL, DOC>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, small_lds<D>(), lds_allowed)) return e;
  hipLaunchKernelGGL(kern, dim3(dkdv_blocks(a, D, DOC)), dim3(64 * kWaves), small_lds<D>(), s, a);
  return (int)hipGetLastError();
}
template <typename Tag, int D, bool CAUSAL, int MODE>
int launch_both(const KArgs& a, hipStream_t s) {
  constexpr size_t lds = small_lds<D>() > dq_lds<D>() ? small_lds<D>() : dq_lds<D>();
  auto kern = bwd_small_kernel<Tag, D, CAUSAL, MODE>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, lds, lds_allowed)) return e;
  const int n_dkdv = dkdv_blocks(a, D, MODE == GEO_DOC), n_dq = grid_blocks(launch_slots<MODE>(a), launch_groups<MODE>(a));
  hipLaunchKernelGGL(kern, dim3(n_dkdv + n_dq), dim3(64 * kWaves), lds, s, a, n_dkdv);
  return (int)hipGetLastError();
}
template <typename Tag, int D>
int launch_cd(const KArgs& a, bool causal, bool doc, bool both, hipStream_t s) {
  if (!both) {
    if (doc) return causal ? launch_dkdv<Tag, D, true, true>(a, s) : launch_dkdv<Tag, D, false, true>(a, s);
    return causal ? launch_dkdv<Tag, D, true, false>(a, s) : launch_dkdv<Tag, D, false, false>(a, s);
  }
  if (doc) return causal ? launch_both<Tag, D, true, GEO_DOC>(a, s) : launch_both<Tag, D, false, GEO_DOC>(a, s);
  if (geo_general(a)) return causal ? launch_both<Tag, D, true, GEO_GENERAL>(a, s) : launch_both<Tag, D, false, GEO_GENERAL>(a, s);
  return causal ? launch_both<Tag, D, true, GEO_PLAIN>(a, s) : launch_both<Tag, D, false, GEO_PLAIN>(a, s);
}

}  // namespace

// Which problems: by the workgroups of 32 keys that they have (kv; packed sequences: as many as the plan's table holds) and by the
// blocks of 32 rows that one of them walks, over the heads of a group (half of them under a causal mask): its chain.  The whole
// backward in this form : in the others, geometric mean over random problems [smallest, largest]:
//   D = 64, two workgroups to a CU.  Up to one to a CU: 0.79 [0.68, 1.03] to kv 128, 0.88 [0.71, 1.07] to 192, 0.94 [0.59, 1.09] to 256.
//     Beyond, short chains lose what the four waves add up at their end and what a second workgroup on the CU costs
//       chain                      to 4               to 8               to 12              to 16              to 24
//       causal, kv 320 - 384  1.07 [1.01, 1.24]  1.00 [0.80, 1.15]  0.84 [0.76, 1.12]  0.78 [0.63, 0.94]  0.73 [0.64, 0.83]
//       kv 384 - 448          1.05 [1.03, 1.07]  1.20 [0.93, 1.54]  1.02 [0.95, 1.20]  0.93 [0.81, 1.19]  0.80 [0.73, 0.87]
//       kv 448 - 512          1.28 [1.05, 1.39]  1.17 [0.98, 1.50]  1.04 [1.00, 1.18]  0.95 [0.85, 1.07]  0.92 [0.80, 1.11]
//     (windows, with the keys that are seen, and block maps alike), but keys that are twice the rows or more have equally long chains: one head to a
//     key head, kv from 320 on, 1.18 [1.00, 1.41] for chains of 11 to 61 (4 heads x 425 rows on 3031 keys 18 us in the others, 25 here); without a mask, kv 352 - 512, 1.1 [0.92, 1.50] up to 32 blocks and 0.93 beyond; with the same ids on both
//     sides 1.13 [1.01, 1.40] from kv 384 and up to 1.43 below for few rows, but 0.90 where the column form is the other one; packed
//     sequences 0.81 [0.61, 1.27] throughout.
//   D = 128, one workgroup to a CU, for its LDS.  One query head to a key head: kv to 64 0.91 [0.62, 1.09], to 96 0.95 [0.77, 1.06], to 128
//     0.96 [0.60, 1.33], to 160 1.10 [0.78, 1.57].  Several, whose chains are longer, and then dq's workgroups of a group count as one:
//     sum to 128 0.80 [0.49, 1.05], to 216 0.81 [0.55, 1.20], to 256 0.84 [0.70, 1.03], to 300 0.98 [0.65, 1.46].  Without a mask all
//     chains are equally long, and short ones do not make up for the second round of the workgroups that exceed the CUs: 8 key heads x 151
//     rows on 614 keys (kv 160, chain 20) 27 us in the others, 32 here, 32 x 38 on 149 (160, 8) 15.5 : 19.5; 4 x 64/8 x 147 (160, 40) 48.7 : 40.4.
bool bwd_small(const KArgs& a, int D, bool causal, bool doc) {
  if (D < 64) return false;
  const int64_t kv = dkdv_blocks(a, D, doc);
  const bool packed = !doc && a.ktab != nullptr, full = !causal && !doc && a.bmask == nullptr;
  int chain = (a.M + kRb - 1) / kRb;
  if (causal && !doc) chain = a.win < 0x3fffffff ? std::min(chain, a.win / kRb + 3) : (chain + 1) / 2;
  const int64_t walked = int64_t(chain) * a.G;
  if (D <= 64) {
    if (kv > 2 * kCUs) return false;
    if (kv <= kCUs || packed) return true;
    if (doc) return !causal || a.qpos != nullptr || a.gap >= 128 || (kv <= kCUs * 3 / 2 && a.M > 150);   // (the first ones: next to the column form otherwise)
    if (causal && a.G == 1 && a.N >= 2 * a.M && kv > 312 && a.win >= 0x3fffffff && a.bmask == nullptr) return false;
    return full ? kv <= 352 || walked > 32 : 16 * walked >= kv * seen_keys(a, causal) / std::max(1, a.N) - 320;
  }
  if (a.G == 1) return kv <= 96;
  if (full && !packed && kv > kCUs / 2 && walked <= 24) return false;
  const int64_t dq = doc ? grid_blocks(launch_slots<GEO_DOC>(a), launch_groups<GEO_DOC>(a))
                         : geo_general(a) ? grid_blocks(launch_slots<GEO_GENERAL>(a), launch_groups<GEO_GENERAL>(a))
                                          : grid_blocks(launch_slots<GEO_PLAIN>(a), launch_groups<GEO_PLAIN>(a));
  return kv + dq / a.G <= 216;
}

int launch_bwd_small(const KArgs& a, int dtype, int D, bool causal, bool doc, bool both, hipStream_t s) {
  if (D == 128) return dtype == FA_DTYPE_BF16 ? launch_cd<bf16_t, 128>(a, causal, doc, both, s) : launch_cd<fp16_t, 128>(a, causal, doc, both, s);
  if (D == 64) return dtype == FA_DTYPE_BF16 ? launch_cd<bf16_t, 64>(a, causal, doc, both, s) : launch_cd<fp16_t, 64>(a, causal, doc, both, s);
  return -1;
}

#ifdef FA_TRACE
int trace_read_small(long long* host, int n) { return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(g_trace_small), size_t(n) * 8); }
#endif

}  // namespace fa
