// The operator for fp32 tensors: forward, delta, dk/dv and dq with `v_mfma_f32_16x16x4_f32`
// (products and accumulation in fp32 throughout).  The reference accepts fp32 tensors like any
// other float type (flash_triton.py:508-564 has no dtype check; its score and probability
// matrices then stay fp32, :88,126) -- this is that case, at full fp32 precision.
//
//   forward  S^T = K Q^T | online softmax (exp2 domain) | O^T += V^T P^T          flash_triton.py:26-172
//   dq       S^T = K Q^T, dP^T = V dO^T | dS = P (dP - delta) | dQ^T += K^T dS^T  flash_triton.py:325-433
//   dk/dv    S = Q K^T, dP = dO V^T | P, dS | dV^T += dO^T P, dK^T += Q^T dS      flash_triton.py:175-321
//
// The SW waves of a workgroup own the SAME RB * 16 rows (or keys), and each takes every SW-th block of 16 of the other side.
// Nothing is shared on the way: operands go from memory straight into the registers of the wave that uses them (a block's
// rows are used by one wave only, so LDS would not save a load), the next block's while this one is computed, with no
// barrier until the waves' sums are added up at the end.  An fp32 MFMA is slow against its operands (32 clocks for 4
// registers), so what counts is that no wave waits and that the longest row range is cut into enough pieces.  Four waves with
// 32 rows each around tiles in LDS, as this was before, against these kernels, us (forward, dq, dk/dv):
//   D = 64    2 x 4 heads x 512, documents    23.8 34.0 38.0 (dq and dk/dv in one launch: 44)  ->  12.5  29.6 (one launch)
//             2 x 4 x 3000, documents         311 387 108     ->  45.6 65.9 78.1
//             8 x 16 x 4096, documents        874 1183 1409   ->  422 640 1181
//             8 x 16 x 4096, causal           3071 4050 5025  ->  2385 3302 4528
//   D = 128   2 x 4 x 512, documents          45.6 66.9 133   ->  17.6 51.0 (one launch)
//             8 x 16 x 2048, causal           1504 2092 2537  ->  1187 2008 2540
//
// A 16x16x4 product takes one element per lane: A[row l % 16][k = l / 16], B[k = l / 16][column l % 16], C/D register r of a
// lane is row 4 * (l / 16) + r of column l % 16.  The contraction index may be walked in any order that both sides share, so
//   score products   k-step (j, e): d = 16 j + 4 (l / 16) + e     -- a lane reads 16 bytes of its row for four MFMAs
//   second products  k-step r: row 4 (l / 16) + r of the block, whose P (dS) the lane holds in register r; output column block
//                    db of lane l: d = VW * (l % 16) + db (VW = 4 from D = 64 on) -- 16 bytes of that row for four MFMAs,
//                    whole rows per load instruction, and the sums come out 16 bytes at a time as well.
//
// Masks: a wave passes over a block of which no pair is kept.  With ids the query side is walked in the permuted order of the
// mask plan (local rows first, then global rows), rows are gathered through the permutation, causal terms use the diagonal
// positions that the plan stored, and 64 rows or keys that the plan's summaries rule out are not looked at; a block mask's
// bytes stand for 64 x 64 pairs and are tested in the same place.
#include "fa_tile.h"

namespace fa {
namespace {

FA_DEV f32x4 mfma16(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int kSB = 16;   // rows (keys) of a block, on either side
static_assert(kSumRows == FA_MASK_BLOCK && kSumRows % (2 * kSB) == 0, "summaries and mask blocks are walked alike");
enum { kPlain, kDoc, kBlock };   // masks besides the causal ones: none, document ids, a block mask

// largest / smallest over the 16 lanes that hold a block's rows (the four groups of 16 hold the same ones)
FA_DEV int min16(int x) {
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) x = min(x, __shfl_xor(x, off));
  return x;
}
FA_DEV int max16(int x) {
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) x = max(x, __shfl_xor(x, off));
  return x;
}
// over the lanes l ^ 16, l ^ 32, l ^ 48 (same column)
FA_DEV float col_max(float x) { x = xhalf_max(x); return fmaxf(x, __shfl_xor(x, 16)); }
FA_DEV float col_sum(float x) { x = xhalf_sum(x); return x + __shfl_xor(x, 16); }

FA_DEV const char* slice(const void* p, int64_t elems) { return reinterpret_cast<const char*>(p) + elems * 4; }

template <int D> struct Dims {
  static constexpr int KJ = D / 16;                 // 16-byte reads of a row by a lane (score products)
  static constexpr int DB = D / 16;                 // output blocks of 16 columns
  static constexpr int VW = DB < 4 ? DB : 4;        // floats a lane reads at a time (second products)
  static constexpr int NR = DB / VW;
  static constexpr int PITCH = D + 4;               // floats of a row in the merge buffer
};

// a row's part that this lane holds for the score products
template <int D> struct RowFrag {
  f32x4 v[Dims<D>::KJ];
  // off: byte offset of the row plus 16 * (l / 16)   (a slice spans less than 2 GiB: 32-bit offsets on a wave-uniform base)
  FA_DEV void load(const char* base, unsigned off) {
#pragma unroll
    for (int j = 0; j < Dims<D>::KJ; ++j) v[j] = *reinterpret_cast<const f32x4*>(base + (off + 64u * j));
  }
};
// one row's columns that this lane holds for the second products
template <int D> struct ColFrag {
  float v[Dims<D>::DB];
  // off: byte offset of the row plus 4 * VW * (l % 16)
  FA_DEV void load(const char* base, unsigned off) {
    constexpr int VW = Dims<D>::VW;
    typedef float vw __attribute__((ext_vector_type(VW < 2 ? 2 : VW)));
#pragma unroll
    for (int i = 0; i < Dims<D>::NR; ++i) {
      const char* p = base + (off + 64u * VW * i);
      if constexpr (VW == 1) v[i] = *reinterpret_cast<const float*>(p);
      else {
        const vw x = *reinterpret_cast<const vw*>(p);
#pragma unroll
        for (int e = 0; e < VW; ++e) v[i * VW + e] = x[e];
      }
    }
  }
};

// C^T (rows of A x columns of B) over the whole row length for RB column blocks.  One chain per block in every shape: the backward's
// scores then round as the forward's did, and a score's error cancels against its share of the LSE.  (With two chains where RB
// is 1 and one where it is 2, dk and dv of a forward in the one shape and a backward in the other were off by 2.1 times as much.)
template <int D, int RB> FA_DEV void score(f32x4 (&x)[RB], const RowFrag<D>& a, const RowFrag<D> (&b)[RB]) {
#pragma unroll
  for (int u = 0; u < RB; ++u) x[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < Dims<D>::KJ; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int u = 0; u < RB; ++u) x[u] = mfma16(a.v[j][e], b[u].v[j][e], x[u]);
}
// Rows that are not there were read from some row that is; zeroed, since 0 times an infinity of that row is not 0.
template <int D> FA_DEV void zero_dead(ColFrag<D> (&t)[4], const bool (&dead)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int db = 0; db < Dims<D>::DB; ++db) t[r].v[db] = dead[r] ? 0.f : t[r].v[db];
}
template <int D, int RB> FA_DEV void second(f32x4 (&acc)[RB][Dims<D>::DB], const ColFrag<D> (&t)[4], const f32x4 (&p)[RB]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int db = 0; db < Dims<D>::DB; ++db)
#pragma unroll
      for (int u = 0; u < RB; ++u) acc[u][db] = mfma16(t[r].v[db], p[u][r], acc[u][db]);
}

// Blocks of 16 of the streamed side for one wave: every SW-th of [b0, b1), where TEST only those whose 64-entry summary (or byte
// of the block mask) passes `test` (64 of them tested at a time, one per lane).
template <bool TEST, int SW> struct Blocks {
  unsigned long long mask = 0;
  int base = -0x40000000, end = 0;
  // first block >= t of this wave, or -1
  template <class Test> FA_DEV int next(int t, int n, const Test& test) {
    for (; t < end; t += SW) {
      if (!TEST) return t;
      const int e = t / (kSumRows / kSB);
      if (e - base >= 64 || e < base) {
        base = e;
        const int i = base + (threadIdx.x & 63);
        bool ok = false;
        if (i < n) ok = test(i);
        mask = __builtin_amdgcn_ballot_w64(ok);
      }
      if ((mask >> (e - base)) & 1) return t;
    }
    return -1;
  }
};

// The accumulators of a wave (lane: row or key l % 16; DB x 4 columns) as [16][PITCH] arrays of the merge buffer, one per block.
template <int D, int RB> FA_DEV void put_rows(float* buf, const f32x4 (&acc)[RB][Dims<D>::DB], int lc, int g4) {
  constexpr int VW = Dims<D>::VW;
#pragma unroll
  for (int u = 0; u < RB; ++u)
#pragma unroll
    for (int i = 0; i < Dims<D>::NR; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < VW; ++e) buf[(u * kSB + lc) * Dims<D>::PITCH + i * 16 * VW + VW * (4 * g4 + r) + e] = acc[u][i * VW + e][r];
}

template <int D, int RB, int SW> constexpr size_t merge_floats() { return size_t(SW) * RB * kSB * Dims<D>::PITCH; }
template <int D, int RB, int SW> constexpr size_t merge_lds(int sets) { return (sets * merge_floats<D, RB, SW>() + (2 * SW + 1) * RB * kSB) * 4; }

// Query side of the forward and dq: this lane's rows (l % 16 of every block) and what the workgroup's rows can see.
template <bool CAUSAL, bool DOC, int RB> struct QSide16 {
  int row[RB], rowc[RB], eq_i[RB], lim_i[RB], low_i[RB];
  int w_lo, w_hi, w_glob;
  int kb0, kb1;    // key blocks of 16 to look at
  FA_DEV bool init(const KArgs& a, int b, int h, int tile, int lc) {
    int kfirst = 0, klast = 0x3fffff, w_lim = -1, w_low = 0x7fffffff;
    if (DOC) {
      const IdSummary qs = a.qsum[b * a.qs_bs + h * a.qs_hs + tile * (RB * kSB) / kSumRows];
      kfirst = qs.kfirst; klast = qs.klast;
    }
    w_lo = 0x7fffffff; w_hi = (int)0x80000000; w_glob = 0;
    int pos[RB];
#pragma unroll
    for (int u = 0; u < RB; ++u) {
      if (!DOC) {
        const int r = (tile * RB + u) * kSB + lc;
        row[u] = r < a.M ? r : -1;
        pos[u] = a.gap + r;
        eq_i[u] = 0;
      } else {
        const int64_t pi = b * a.pm_bs + h * a.pm_hs + (tile * RB + u) * kSB + lc;
        row[u] = a.perm[pi]; eq_i[u] = a.peq[pi]; pos[u] = a.ppos[pi];
      }
    }
    bool some = false;
#pragma unroll
    for (int u = 0; u < RB; ++u) {
      const bool live = row[u] >= 0;
      some = some || live;
      rowc[u] = live ? row[u] : 0;
      if (!live) pos[u] = -1;
      lim_i[u] = !live ? -1 : CAUSAL ? min(max(pos[u], a.pfx_m1), a.N - 1) : a.N - 1;
      low_i[u] = CAUSAL ? pos[u] - a.win + 1 : 0;
      w_lim = max(w_lim, lim_i[u]);
      w_low = min(w_low, live ? low_i[u] : 0x7fffffff);
      if (DOC) {
        w_lo = min(w_lo, live && eq_i[u] < 0 ? eq_i[u] : 0x7fffffff);
        w_hi = max(w_hi, live && eq_i[u] < 0 ? eq_i[u] : (int)0x80000000);
        w_glob |= live && eq_i[u] >= 0;
      }
    }
    if (__builtin_amdgcn_ballot_w64(some) == 0) return false;
    w_lim = max16(w_lim); w_low = max(0, min16(w_low));
    if (DOC) { w_lo = min16(w_lo); w_hi = max16(w_hi); w_glob = __builtin_amdgcn_ballot_w64(w_glob != 0) != 0; }
    kb0 = w_low / kSB;
    kb1 = w_lim < w_low ? kb0 : w_lim / kSB + 1;
    if (DOC && klast < kfirst) kb1 = kb0;
    else if (DOC) {
      kb0 = max(kb0, kfirst * (kSumRows / kSB));
      kb1 = min(kb1, (klast + 1) * (kSumRows / kSB));
    }
    kb0 = __builtin_amdgcn_readfirstlane(kb0);
    kb1 = __builtin_amdgcn_readfirstlane(kb1);
    return true;
  }
  // which of the keys key0 .. + 3 this lane's row of block u may see
  FA_DEV void keep(int u, int key0, const i32x4& ids, bool (&k)[4]) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = key0 + r;
      k[r] = key <= lim_i[u] && key >= low_i[u] && (!DOC || eq_i[u] >= 0 || ids[r] == eq_i[u]);
    }
  }
};
FA_DEV bool any_lane(const bool (&k)[4]) { return __builtin_amdgcn_ballot_w64(k[0] || k[1] || k[2] || k[3]) != 0; }

template <int D, bool CAUSAL, int MODE, int RB, int SW>
FA_DEV void fwd16_body(const KArgs& a, const int bid, float* lds) {
  constexpr bool DOC = MODE == kDoc, BM = MODE == kBlock;
  constexpr int DB = Dims<D>::DB, PITCH = Dims<D>::PITCH, ROWS = RB * kSB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, g4 = lane >> 4;
  const int BH = a.B * a.H;
  const int nQt = DOC ? a.Pp / ROWS : (a.M + ROWS - 1) / ROWS;
  const int tile = nQt - 1 - bid / BH;   // the last rows see the most keys (with ids: the global rows): first
  const int bh = bid % BH, b = bh / a.H, h = bh % a.H, hk = h / a.G;
  QSide16<CAUSAL, DOC, RB> qc;
  if (!qc.init(a, b, h, tile, lc)) return;
  const char* kp = slice(a.k, b * a.k_bs + hk * a.k_hs);
  const char* vp = slice(a.v, b * a.v_bs + hk * a.v_hs);
  const unsigned k_rb = 4u * (unsigned)a.k_rs, v_rb = 4u * (unsigned)a.v_rs, rof = 16u * g4, cof = 4u * Dims<D>::VW * lc;
  const int* ekp = DOC ? a.ek32 + b * a.ek_bs + h * a.ek_hs : nullptr;
  const IdSummary* ksum = DOC ? a.ksum + b * a.ks_bs + h * a.ks_hs : nullptr;
  const unsigned char* bmr = BM ? a.bmask + b * a.bm_bs + h * a.bm_hs + int64_t(tile * ROWS / FA_MASK_BLOCK) * a.bm_rs : nullptr;

  RowFrag<D> q[RB];
#pragma unroll
  for (int u = 0; u < RB; ++u) q[u].load(slice(a.q, b * a.q_bs + h * a.q_hs), 4u * (unsigned)a.q_rs * qc.rowc[u] + rof);
  float c = a.scale_log2e;
  const float sgn = c < 0.f ? -1.f : 1.f;   // keep max(raw score) == max(scaled score): move the sign into Q
  c *= sgn;

  f32x4 o[RB][DB];
  float m_run[RB], l_run[RB];
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    m_run[u] = -INFINITY; l_run[u] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[u][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  RowFrag<D> kr;
  ColFrag<D> vc[4];
  i32x4 ids = {0, 0, 0, 0}, ids_n = ids;
  const int last = a.N - 1;
  auto load_rows = [&](const int kb) __attribute__((always_inline)) {
    kr.load(kp, k_rb * min(kb * kSB + lc, last) + rof);
    if (DOC) ids_n = *reinterpret_cast<const i32x4*>(ekp + kb * kSB + 4 * g4);   // (padded to whole tiles of 64)
  };
  auto load_cols = [&](const int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) vc[r].load(vp, v_rb * min(kb * kSB + 4 * g4 + r, last) + cof);
  };
  Blocks<DOC || BM, SW> bl;
  bl.end = qc.kb1;
  auto next = [&](int t) {
    if (BM) return bl.next(t, a.nBc, [&](int i) { return bmr[i] != 0; });
    return bl.next(t, a.nKs, [&](int i) { return doc_may_keep(qc.w_lo, qc.w_hi, qc.w_glob, ksum[i].lo, ksum[i].hi); });
  };
  int kb = next(qc.kb0 + wave);
  if (kb >= 0) { load_rows(kb); load_cols(kb); }
#pragma unroll
  for (int u = 0; u < RB; ++u)
#pragma unroll
    for (int j = 0; j < Dims<D>::KJ; ++j) q[u].v[j] *= sgn;
  while (kb >= 0) {
    const int nx = next(kb + SW);
    ids = ids_n;
    bool keep[RB][4], any = false;
#pragma unroll
    for (int u = 0; u < RB; ++u) { qc.keep(u, kb * kSB + 4 * g4, ids, keep[u]); any = any || any_lane(keep[u]); }
    f32x4 x[RB];
    if (any) score<D, RB>(x, kr, q);
    __builtin_amdgcn_sched_barrier(0);
    if (nx >= 0) load_rows(nx);   // the next block's operands travel behind the half of this one that still computes
    __builtin_amdgcn_sched_barrier(0);
    if (any) {
#pragma unroll
      for (int u = 0; u < RB; ++u) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[u][r] = keep[u][r] ? x[u][r] : -INFINITY;
        const float mx = col_max(fmaxf(fmaxf(x[u][0], x[u][1]), fmaxf(x[u][2], x[u][3]))) * c;
        const float m_new = fmaxf(m_run[u], mx);
        const float alpha = m_run[u] == -INFINITY ? 0.f : fast_exp2(m_run[u] - m_new);
        const float msub = m_new == -INFINITY ? 0.f : m_new;
        m_run[u] = m_new;
        float ps = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) { x[u][r] = fast_exp2(__builtin_fmaf(x[u][r], c, -msub)); ps += x[u][r]; }
        l_run[u] = l_run[u] * alpha + ps;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[u][db] *= alpha;
      }
      if ((kb + 1) * kSB > a.N) {
        const int n = a.N - kb * kSB - 4 * g4;
        const bool dead[4] = {n < 1, n < 2, n < 3, n < 4};
        zero_dead<D>(vc, dead);
      }
      second<D, RB>(o, vc, x);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (nx >= 0) load_cols(nx);
    __builtin_amdgcn_sched_barrier(0);
    kb = nx;
  }

  // the waves' partial states to one
  float* ml = lds + merge_floats<D, RB, SW>();            // [2][SW][ROWS]: reference points, sums
  int* rows = reinterpret_cast<int*>(ml + 2 * SW * ROWS);
  put_rows<D, RB>(lds + wave * ROWS * PITCH, o, lc, g4);
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const float l_tot = col_sum(l_run[u]);
    if (g4 == 0) { ml[wave * ROWS + u * kSB + lc] = m_run[u]; ml[(SW + wave) * ROWS + u * kSB + lc] = l_tot; }
    if (wave == 0 && g4 == 0) rows[u * kSB + lc] = qc.row[u];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ROWS * (D / 4); i += 64 * SW) {
    const int r = i / (D / 4), c4 = i % (D / 4), row = rows[r];
    if (row < 0) continue;
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < SW; ++w) m = fmaxf(m, ml[w * ROWS + r]);
    float l = 0.f;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SW; ++w) {
      const float mw = ml[w * ROWS + r], wt = mw == -INFINITY ? 0.f : fast_exp2(mw - m);
      l += wt * ml[(SW + w) * ROWS + r];
      x += wt * *reinterpret_cast<const f32x4*>(lds + (w * ROWS + r) * PITCH + 4 * c4);
    }
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.o) + b * a.o_bs + h * a.o_hs + int64_t(row) * a.o_rs + 4 * c4) = x * inv;
    if (c4 == 0) a.lse[(int64_t(b) * a.H + h) * a.M + row] = l > 0.f ? m + fast_log2(l) : -INFINITY;
  }
}

template <int D, bool CAUSAL, int MODE, int RB, int SW>
FA_DEV void dq16_body(const KArgs& a, const int bid, float* lds) {
  constexpr bool DOC = MODE == kDoc, BM = MODE == kBlock;
  constexpr int DB = Dims<D>::DB, PITCH = Dims<D>::PITCH, ROWS = RB * kSB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, g4 = lane >> 4;
  const int BH = a.B * a.H;
  const int nQt = DOC ? a.Pp / ROWS : (a.M + ROWS - 1) / ROWS;
  const int tile = nQt - 1 - bid / BH;
  const int bh = bid % BH, b = bh / a.H, h = bh % a.H, hk = h / a.G;
  QSide16<CAUSAL, DOC, RB> qc;
  if (!qc.init(a, b, h, tile, lc)) return;
  const char* kp = slice(a.k, b * a.k_bs + hk * a.k_hs);
  const char* vp = slice(a.v, b * a.v_bs + hk * a.v_hs);
  const unsigned k_rb = 4u * (unsigned)a.k_rs, v_rb = 4u * (unsigned)a.v_rs, rof = 16u * g4, cof = 4u * Dims<D>::VW * lc;
  const int* ekp = DOC ? a.ek32 + b * a.ek_bs + h * a.ek_hs : nullptr;
  const IdSummary* ksum = DOC ? a.ksum + b * a.ks_bs + h * a.ks_hs : nullptr;
  const unsigned char* bmr = BM ? a.bmask + b * a.bm_bs + h * a.bm_hs + int64_t(tile * ROWS / FA_MASK_BLOCK) * a.bm_rs : nullptr;

  const float c = a.scale_log2e;
  RowFrag<D> q[RB], dout[RB];
  float L_i[RB], delta_i[RB];
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const int64_t row_l = (int64_t(b) * a.H + h) * a.M + qc.rowc[u];
    q[u].load(slice(a.q, b * a.q_bs + h * a.q_hs), 4u * (unsigned)a.q_rs * qc.rowc[u] + rof);
    dout[u].load(slice(a.dout, b * a.do_bs + h * a.do_hs), 4u * (unsigned)a.do_rs * qc.rowc[u] + rof);
    L_i[u] = a.lse[row_l];
    if (a.dq_delta) {   // delta = rowsum(O * dO) formed here and left for dk/dv
      RowFrag<D> of;
      of.load(slice(a.o, b * a.o_bs + h * a.o_hs), 4u * (unsigned)a.o_rs * qc.rowc[u] + rof);
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < Dims<D>::KJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) part += of.v[j][e] * dout[u].v[j][e];
      delta_i[u] = col_sum(part);
      if (wave == 0 && g4 == 0 && qc.row[u] >= 0) a.delta[row_l] = delta_i[u];
    } else {
      delta_i[u] = a.delta[row_l];
    }
    if (L_i[u] == -INFINITY) L_i[u] = INFINITY;   // row without any kept key: P = exp2(-inf) = 0
  }

  f32x4 acc[RB][DB];
#pragma unroll
  for (int u = 0; u < RB; ++u)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[u][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int last = a.N - 1;
  RowFrag<D> kr, vr;
  ColFrag<D> kc[4];
  i32x4 ids = {0, 0, 0, 0}, ids_n = ids;
  auto load_rows = [&](const int kb) __attribute__((always_inline)) {
    const int key = min(kb * kSB + lc, last);
    kr.load(kp, k_rb * key + rof);
    vr.load(vp, v_rb * key + rof);
    if (DOC) ids_n = *reinterpret_cast<const i32x4*>(ekp + kb * kSB + 4 * g4);
  };
  auto load_cols = [&](const int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) kc[r].load(kp, k_rb * min(kb * kSB + 4 * g4 + r, last) + cof);
  };
  Blocks<DOC || BM, SW> bl;
  bl.end = qc.kb1;
  auto next = [&](int t) {
    if (BM) return bl.next(t, a.nBc, [&](int i) { return bmr[i] != 0; });
    return bl.next(t, a.nKs, [&](int i) { return doc_may_keep(qc.w_lo, qc.w_hi, qc.w_glob, ksum[i].lo, ksum[i].hi); });
  };
  int kb = next(qc.kb0 + wave);
  if (kb >= 0) { load_rows(kb); load_cols(kb); }
  while (kb >= 0) {
    const int nx = next(kb + SW);
    ids = ids_n;
    bool keep[RB][4], any = false;
#pragma unroll
    for (int u = 0; u < RB; ++u) { qc.keep(u, kb * kSB + 4 * g4, ids, keep[u]); any = any || any_lane(keep[u]); }
    f32x4 x[RB], dp[RB];
    if (any) { score<D, RB>(x, kr, q); score<D, RB>(dp, vr, dout); }
    __builtin_amdgcn_sched_barrier(0);
    if (nx >= 0) load_rows(nx);
    __builtin_amdgcn_sched_barrier(0);
    if (any) {
#pragma unroll
      for (int u = 0; u < RB; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float ds = fast_exp2(__builtin_fmaf(x[u][r], c, -L_i[u])) * (dp[u][r] - delta_i[u]);
          x[u][r] = keep[u][r] ? ds : 0.f;
        }
      if ((kb + 1) * kSB > a.N) {
        const int n = a.N - kb * kSB - 4 * g4;
        const bool dead[4] = {n < 1, n < 2, n < 3, n < 4};
        zero_dead<D>(kc, dead);
      }
      second<D, RB>(acc, kc, x);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (nx >= 0) load_cols(nx);
    __builtin_amdgcn_sched_barrier(0);
    kb = nx;
  }
  int* rows = reinterpret_cast<int*>(lds + merge_floats<D, RB, SW>());
  put_rows<D, RB>(lds + wave * ROWS * PITCH, acc, lc, g4);
#pragma unroll
  for (int u = 0; u < RB; ++u)
    if (wave == 0 && g4 == 0) rows[u * kSB + lc] = qc.row[u];
  __syncthreads();
  for (int i = threadIdx.x; i < ROWS * (D / 4); i += 64 * SW) {
    const int r = i / (D / 4), c4 = i % (D / 4), row = rows[r];
    if (row < 0) continue;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SW; ++w) x += *reinterpret_cast<const f32x4*>(lds + (w * ROWS + r) * PITCH + 4 * c4);
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.dq) + b * a.dq_bs + h * a.dq_hs + int64_t(row) * a.dq_rs + 4 * c4) = x * a.scale;
  }
}

template <int D, bool CAUSAL, int MODE, int RB, int SW, bool OWN_DELTA>
FA_DEV void dkdv16_body(const KArgs& a, const int bid, float* lds) {
  constexpr bool DOC = MODE == kDoc, BM = MODE == kBlock;
  constexpr int DB = Dims<D>::DB, PITCH = Dims<D>::PITCH, ROWS = RB * kSB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, g4 = lane >> 4;
  const int BHk = a.B * a.Hk;
  const int n0 = (bid / BHk) * ROWS;   // causal: the first keys are seen by the most rows: first
  const int bhk = bid % BHk, b = bhk / a.Hk, hk = bhk % a.Hk;
  RowFrag<D> k[RB], v[RB];
  const unsigned q_rb = 4u * (unsigned)a.q_rs, do_rb = 4u * (unsigned)a.do_rs, o_rb = 4u * (unsigned)a.o_rs, rof = 16u * g4, cof = 4u * Dims<D>::VW * lc;
  // Rows that may see this lane's keys, by name (index, or with ids the diagonal position of the plan): [row_lo, row_lo + row_span)
  const int gk = DOC ? 0 : a.gap, rcap = DOC ? kPosMax : a.M - 1;
  int row_lo[RB];
  unsigned row_span[RB];
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const int key = n0 + u * kSB + lc, keyc = min(key, a.N - 1);
    k[u].load(slice(a.k, b * a.k_bs + hk * a.k_hs), 4u * (unsigned)a.k_rs * keyc + rof);
    v[u].load(slice(a.v, b * a.v_bs + hk * a.v_hs), 4u * (unsigned)a.v_rs * keyc + rof);
    row_lo[u] = CAUSAL ? (key <= a.pfx_m1 ? 0 : max(0, key - gk)) : 0;
    const int row_hi = CAUSAL ? min(rcap, key - gk + a.win - 1) : rcap;
    row_span[u] = (key < a.N && row_hi >= row_lo[u]) ? (unsigned)(row_hi - row_lo[u] + 1) : 0u;
  }
  const float c = a.scale_log2e;
  const int wg_rhi = CAUSAL ? min(rcap, n0 + ROWS - 1 - gk + a.win - 1) : rcap;
  const int mb0 = DOC ? 0 : (CAUSAL ? (n0 <= a.pfx_m1 ? 0 : max(0, n0 - gk) / kSB) : 0);
  const int mb1 = DOC ? a.Pp / kSB : (wg_rhi < 0 ? 0 : wg_rhi / kSB + 1);

  f32x4 dv[RB][DB], dk[RB][DB];
#pragma unroll
  for (int u = 0; u < RB; ++u)
#pragma unroll
    for (int db = 0; db < DB; ++db) dv[u][db] = dk[u][db] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int gi = 0; gi < a.G; ++gi) {
    const int h = hk * a.G + gi;
    const char* qp = slice(a.q, b * a.q_bs + h * a.q_hs);
    const char* dop = slice(a.dout, b * a.do_bs + h * a.do_hs);
    const char* op = slice(a.o, b * a.o_bs + h * a.o_hs);
    const char* lsep = slice(a.lse, (int64_t(b) * a.H + h) * a.M);
    const char* delp = slice(a.delta, (int64_t(b) * a.H + h) * a.M);
    const char* pmp = slice(a.perm, b * a.pm_bs + h * a.pm_hs);
    const char* pqp = slice(a.peq, b * a.pm_bs + h * a.pm_hs);
    const char* ppp = slice(a.ppos, b * a.pm_bs + h * a.pm_hs);
    const IdSummary* qsum = DOC ? a.qsum + b * a.qs_bs + h * a.qs_hs : nullptr;
    const unsigned char* bmc = BM ? a.bmask + b * a.bm_bs + h * a.bm_hs + n0 / FA_MASK_BLOCK : nullptr;
    int ek_j[RB], k_lo = 0x7fffffff, k_hi = (int)0x80000000;
#pragma unroll
    for (int u = 0; u < RB; ++u) {
      ek_j[u] = 0;
      if (DOC) {
        const int key = n0 + u * kSB + lc;
        ek_j[u] = a.ek32[b * a.ek_bs + h * a.ek_hs + min(key, a.N - 1)];
        k_lo = min(k_lo, key < a.N ? ek_j[u] : 0x7fffffff);
        k_hi = max(k_hi, key < a.N ? ek_j[u] : (int)0x80000000);
      }
    }
    if (DOC) { k_lo = min16(k_lo); k_hi = max16(k_hi); }
    // With ids: the row this lane reads for the score products, and rows 4 g4 .. + 3 of the block with their ids and names.  The
    // indices travel a block ahead of the rows they name.
    struct Rows { int own; i32x4 r, eq, nm; } ix = {}, cur = {};
    auto load_idx = [&](const int mb) __attribute__((always_inline)) {
      if (!DOC) return;
      const unsigned at = 4u * kSB * mb;
      ix.own = max(*reinterpret_cast<const int*>(pmp + (at + 4u * lc)), 0);
      ix.r = *reinterpret_cast<const i32x4*>(pmp + (at + rof));
      ix.eq = *reinterpret_cast<const i32x4*>(pqp + (at + rof));
      ix.nm = *reinterpret_cast<const i32x4*>(ppp + (at + rof));
    };
    RowFrag<D> qr, dr, orow;
    ColFrag<D> qc[4], dc[4];
    float L[4], del[4];
    auto load_rows = [&](const int mb) __attribute__((always_inline)) {
      const int own = DOC ? ix.own : min(mb * kSB + lc, a.M - 1);
      qr.load(qp, q_rb * own + rof);
      dr.load(dop, do_rb * own + rof);
      if (OWN_DELTA) orow.load(op, o_rb * own + rof);
    };
    auto load_cols = [&](const Rows& x, const int mb) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = DOC ? max(x.r[r], 0) : min(mb * kSB + 4 * g4 + r, a.M - 1);
        L[r] = *reinterpret_cast<const float*>(lsep + 4u * row);
        if (!OWN_DELTA) del[r] = *reinterpret_cast<const float*>(delp + 4u * row);
        dc[r].load(dop, do_rb * row + cof);
        qc[r].load(qp, q_rb * row + cof);
      }
    };
    Blocks<DOC || BM, SW> bl;
    bl.end = mb1;
    auto next = [&](int t) {
      if (BM) return bl.next(t, a.nBr, [&](int i) { return bmc[int64_t(i) * a.bm_rs] != 0; });
      return bl.next(t, a.nQs, [&](int i) {
        const IdSummary qs = qsum[i];
        return qs.nvalid > 0 && doc_may_keep(qs.lo, qs.hi, qs.glob, k_lo, k_hi) && !(CAUSAL && ((qs.rmax < n0 && n0 > a.pfx_m1) || qs.rmin > wg_rhi));
      });
    };
    int mb = next(mb0 + wave), nx = -1;
    if (mb >= 0) {
      load_idx(mb);
      nx = next(mb + SW);
      cur = ix;
      load_rows(mb);
      load_cols(cur, mb);
      if (nx >= 0) load_idx(nx);
    }
    while (mb >= 0) {
      const int nx2 = nx >= 0 ? next(nx + SW) : -1;
      bool keep[RB][4], any = false;
#pragma unroll
      for (int u = 0; u < RB; ++u) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int nm = DOC ? cur.nm[r] : mb * kSB + 4 * g4 + r;   // (rows past the end lie beyond every span)
          keep[u][r] = (unsigned)(nm - row_lo[u]) < row_span[u] && (!DOC || cur.eq[r] >= 0 || cur.eq[r] == ek_j[u]);
        }
        any = any || any_lane(keep[u]);
      }
      bool dead[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) dead[r] = DOC ? cur.r[r] < 0 : mb * kSB + 4 * g4 + r >= a.M;
      f32x4 x[RB], dp[RB];
      if (any) {
        score<D, RB>(x, qr, k);
        score<D, RB>(dp, dr, v);
        if (OWN_DELTA) {   // delta = rowsum(O * dO): of row l % 16 in every lane, then of the four rows of this lane's scores
          float part = 0.f;
#pragma unroll
          for (int j = 0; j < Dims<D>::KJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) part += orow.v[j][e] * dr.v[j][e];
          part = col_sum(part);
#pragma unroll
          for (int r = 0; r < 4; ++r) del[r] = __shfl(part, 4 * g4 + r);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (nx >= 0) {   // the next block's operands travel behind the half of this one that still computes
        load_rows(nx);
        cur = ix;
        if (nx2 >= 0) load_idx(nx2);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (any) {
#pragma unroll
        for (int u = 0; u < RB; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float p = fast_exp2(__builtin_fmaf(x[u][r], c, -L[r]));
            x[u][r] = keep[u][r] ? p : 0.f;
            dp[u][r] = keep[u][r] ? p * (dp[u][r] - del[r]) : 0.f;
          }
        if (__builtin_amdgcn_ballot_w64(dead[3]) != 0) {   // (a group's last rows are the missing ones)
          zero_dead<D>(dc, dead);
          zero_dead<D>(qc, dead);
        }
        second<D, RB>(dv, dc, x);
        second<D, RB>(dk, qc, dp);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (nx >= 0) load_cols(cur, nx);
      __builtin_amdgcn_sched_barrier(0);
      mb = nx; nx = nx2;
    }
  }

  put_rows<D, RB>(lds + wave * ROWS * PITCH, dv, lc, g4);
  put_rows<D, RB>(lds + (SW + wave) * ROWS * PITCH, dk, lc, g4);
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * ROWS * (D / 4); i += 64 * SW) {
    const int set = i / (ROWS * (D / 4)), r = i / (D / 4) % ROWS, c4 = i % (D / 4);
    if (n0 + r >= a.N) continue;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SW; ++w) x += *reinterpret_cast<const f32x4*>(lds + ((set * SW + w) * ROWS + r) * PITCH + 4 * c4);
    float* p = set == 0 ? reinterpret_cast<float*>(a.dv) + b * a.dv_bs + hk * a.dv_hs + int64_t(n0 + r) * a.dv_rs
                        : reinterpret_cast<float*>(a.dk) + b * a.dk_bs + hk * a.dk_hs + int64_t(n0 + r) * a.dk_rs;
    *reinterpret_cast<f32x4*>(p + 4 * c4) = set == 0 ? x : x * a.scale;
  }
}

enum { kFwd, kDq, kDkdv, kBoth };

// Two waves to a SIMD, or the registers of one where 256 do not hold the operands and sums.  (D = 128, 8 x 16 heads x 2048,
// causal, RB 2: dq 3.67 -> 2.01 ms, dk/dv 10.0 -> 2.54 ms.  At D = 64 dk/dv with RB 2 lacks a few, 52 bytes of a lane in scratch
// memory, 140 with ids, and is still the fastest there.)
template <int WHICH, int D, int RB> constexpr int kWavesPerSimd = D == 128 && WHICH != kFwd && !(WHICH == kDq && RB == 1) ? 1 : 2;
template <int WHICH, int D, bool CAUSAL, int MODE, int RB, int SW>
__global__ __launch_bounds__(64 * SW) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd<WHICH, D, RB>)))
void f32_kernel(const KArgs a, const int n_dkdv, const int n_all) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* lds = reinterpret_cast<float*>(smem);
  const int bid = (int)(blockIdx.y * gridDim.x + blockIdx.x);
  if (bid >= n_all) return;
  if constexpr (WHICH == kFwd) fwd16_body<D, CAUSAL, MODE, RB, SW>(a, bid, lds);
  else if constexpr (WHICH == kDq) dq16_body<D, CAUSAL, MODE, RB, SW>(a, bid, lds);
  else if constexpr (WHICH == kDkdv) dkdv16_body<D, CAUSAL, MODE, RB, SW, false>(a, bid, lds);
  else if (bid < n_dkdv) dkdv16_body<D, CAUSAL, MODE, RB, SW, true>(a, bid, lds);   // the longer ones first
  else dq16_body<D, CAUSAL, MODE, RB, SW>(a, bid - n_dkdv, lds);
}

template <int WHICH, int D, bool CAUSAL, int MODE, int RB, int SW>
int launch(const KArgs& a, hipStream_t s) {
  constexpr int ROWS = RB * kSB;
  const int n_q = (MODE == kDoc ? a.Pp / ROWS : (a.M + ROWS - 1) / ROWS) * a.B * a.H, n_k = (a.N + ROWS - 1) / ROWS * a.B * a.Hk;
  constexpr size_t lds = merge_lds<D, RB, SW>(WHICH == kDkdv || WHICH == kBoth ? 2 : 1);
  auto kern = f32_kernel<WHICH, D, CAUSAL, MODE, RB, SW>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, lds, lds_allowed)) return e;
  const int blocks = WHICH == kFwd || WHICH == kDq ? n_q : WHICH == kDkdv ? n_k : n_k + n_q;
  constexpr int kMaxX = 1 << 22;      // (a grid dimension stops at 2^32 threads)
  hipLaunchKernelGGL(kern, dim3(blocks < kMaxX ? blocks : kMaxX, (blocks + kMaxX - 1) / kMaxX), dim3(64 * SW), lds, s, a, n_k, blocks);
  return (int)hipGetLastError();
}

// Which of three shapes a launch takes, by the blocks of 16 rows (keys) that it has.  us (forward, dq, dk/dv):
//                                          RB 1, SW 8 *       RB 2, SW 4         RB 2, SW 2
//   D = 64  2 x 4 heads x 1024, causal (512)    22.6 35.6 37.2     28.2 36.9 46.1     48.9 63.5 79.8
//           2 x 4 x 2048, documents  (1024)     33.6 43.4 54.6     61.1 79.0 46.2     108 140 60
//           8 x 8 x 256, causal      (1024)     16.5 26.0 33.5     14.0 21.7 25.6     20.4 26.8 34.3
//           2 x 4 x 3000, documents  (1504)     45.6 65.6 85.2     84.6 114 74        156 201 75
//           8 x 16 x 512, causal     (4096)     70.6 119 170       55.5 89.2 112      57.1 73.8 104
//           8 x 8 x 1241, documents  (4992)     87.4 190 228       66.1 111 168       88.2 114 148
//           3 x 16 x 3490, documents (10512)    194 407 541        151 239 383        257 315 327
//           8 x 16 x 4096, documents (32768)    681 1390 2021      459 773 1367       422 640 1155
//           8 x 16 x 4096, causal    (32768)    2886 4643 6466     2439 3438 4784     2395 3335 4643
//   D = 128 2 x 4 x 512, causal      (256)      17.7 27.3 31.8     26.1 37.7 46.4     43.4 61.2 76.7
//           2 x 4 x 2048, causal     (1024)     108 176 220        116 144 178        209 237 287
//           8 x 8 x 1241, documents  (4992)     209 334 406        126 251 305        140 195 246
//           8 x 16 x 2048, causal    (16384)    1749 2763 3556     1232 2199 2728     1187 2008 2540
//   * dk/dv at D = 128: SW 4, since one wave to a SIMD is all that its registers allow
// Few blocks: the chain of one of them counts, so all waves share it.  Many: the work counts, and a block of 32 reads the
// other side half as often; then also what a workgroup adds up at its end.  (Rows with ids: the global ones among them walk
// all keys, the others a few blocks: the chain counts longer.)  Where a block walks few blocks of the other side, its chain, what a
// workgroup adds up at its end counts earlier, and with ids every empty place of the plan's order costs a workgroup: exceptions below.
// Many short rows without them, against tiles in LDS as before these kernels: 8 x 32 heads x 32 with ids, dq 10.6 -> 26.6; 4 x 64 x 92,
// D = 128, with ids, forward 30 -> 59 (27 now); 2 x 64 x 209, D = 128, no mask, dk/dv 83 -> 108.  Of the launches of 2000 random problems 151
// were slower than before these kernels without the exceptions, 50 with them, and 5 are slower than without (up to 1.16, launches of 10 us).
template <int WHICH, int D> constexpr int kFewWaves = D == 128 && (WHICH == kDkdv || WHICH == kBoth) ? 4 : 8;
// 0, 1, 2: the columns of the table
template <int WHICH, int MODE> int shape(const KArgs& a, int D, bool causal) {
  static_assert(WHICH != kBoth, "dq and dk/dv in one launch have one shape");
  constexpr bool IDS = WHICH != kDkdv && MODE == kDoc;
  const int64_t n = WHICH == kDkdv ? int64_t((a.N + kSB - 1) / kSB) * a.B * a.Hk : int64_t((a.M + kSB - 1) / kSB) * a.B * a.H;
  const int64_t chain = WHICH == kDkdv ? int64_t((a.M + kSB - 1) / kSB) * a.G : (a.N + kSB - 1) / kSB;
  constexpr int kFew = IDS ? 2048 : 768;
  const int many = WHICH == kFwd || (IDS && D <= 64) ? 16384 : 4096;
  if (IDS) {
    const int64_t places = int64_t(a.Pp / kSB) * a.B * a.H;
    if (chain <= 6 && places >= 2048) return 2;
    if (n <= kFew && places >= std::max<int64_t>(WHICH == kFwd ? 4096 : 2048, 128 * chain)) return 1;
  } else if (WHICH != kFwd && MODE != kBlock) {
    if ((chain <= 3 && n >= 512) || (chain <= 8 && n >= 1024)) return 2;
    if (MODE == kPlain && !causal) {   // workgroups of equal length
      if (chain < 16 && n >= 1280) return 2;
      if (D == 128 && a.G == 1 && n > kFew && n < many) {
        // One (the second shape) or two (the third) to a CU: whichever's rounds take less, two side by side 1.9 times as long as
        // one (dq: 16 heads x 1810 437 : 415 us, four rounds or two; 24 x 1500 460 : 515, five or three).
        const int64_t wgs = (n + 1) / 2, one = (wgs + kCUs - 1) / kCUs, two = (wgs + 2 * kCUs - 1) / (2 * kCUs);
        return 19 * two < 10 * one ? 2 : 1;
      }
    }
  }
  return n <= kFew ? 0 : n < many ? 1 : 2;
}
template <int WHICH, int D, bool CAUSAL, int MODE>
int launch_shape(const KArgs& a, hipStream_t s) {
  if constexpr (WHICH == kBoth) {
    return launch<WHICH, D, CAUSAL, MODE, 1, kFewWaves<WHICH, D>>(a, s);
  } else {
    const int sh = shape<WHICH, MODE>(a, D, CAUSAL);
    if (sh == 0) return launch<WHICH, D, CAUSAL, MODE, 1, kFewWaves<WHICH, D>>(a, s);
    if (sh == 1) return launch<WHICH, D, CAUSAL, MODE, 2, 4>(a, s);
    return launch<WHICH, D, CAUSAL, MODE, 2, 2>(a, s);
  }
}
template <int WHICH, int D, bool CAUSAL>
int launch_mode(const KArgs& a, bool doc, hipStream_t s) {
  if (doc) return launch_shape<WHICH, D, CAUSAL, kDoc>(a, s);
  return a.bmask != nullptr ? launch_shape<WHICH, D, CAUSAL, kBlock>(a, s) : launch_shape<WHICH, D, CAUSAL, kPlain>(a, s);
}
template <int WHICH, int D>
int launch_c(const KArgs& a, bool causal, bool doc, hipStream_t s) {
  return causal ? launch_mode<WHICH, D, true>(a, doc, s) : launch_mode<WHICH, D, false>(a, doc, s);
}
template <int WHICH>
int launch_d(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) {
  switch (D) {
    case 128: return launch_c<WHICH, 128>(a, causal, doc, s);
    case 64: return launch_c<WHICH, 64>(a, causal, doc, s);
    case 32: return launch_c<WHICH, 32>(a, causal, doc, s);
    case 16: return launch_c<WHICH, 16>(a, causal, doc, s);
    default: return -1;
  }
}

constexpr int kDeltaThreads = 256;
// delta[b,h,m] = sum_d O[b,h,m,d] * dO[b,h,m,d]; D/4 lanes per row, 16-byte loads.
template <int D>
__global__ __launch_bounds__(kDeltaThreads) void delta_f32_kernel(const KArgs a) {
  constexpr int LPR = D / 4, RPB = kDeltaThreads / LPR;
  const int row = blockIdx.x * RPB + threadIdx.x / LPR;
  const int cc = threadIdx.x % LPR;
  // (batch, head) pairs are walked with the grid's stride: grid dimension y stops at 65535
  for (int bh = blockIdx.y; bh < a.B * a.H; bh += gridDim.y) {
    const int b = bh / a.H, h = bh % a.H;
    float acc = 0.f;
    if (row < a.M) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.o) + b * a.o_bs + h * a.o_hs +
                                                      int64_t(row) * a.o_rs + cc * 4);
      const f32x4 y = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.dout) + b * a.do_bs + h * a.do_hs +
                                                      int64_t(row) * a.do_rs + cc * 4);
      acc = x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
    }
#pragma unroll
    for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
    if (cc == 0 && row < a.M) a.delta[(int64_t(b) * a.H + h) * a.M + row] = acc;
  }
}

}  // namespace

int launch_fwd_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) { return launch_d<kFwd>(a, D, causal, doc, s); }
int launch_bwd_dq_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) { return launch_d<kDq>(a, D, causal, doc, s); }
int launch_bwd_dkdv_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) { return launch_d<kDkdv>(a, D, causal, doc, s); }

// dq and dk/dv side by side in one launch, each forming delta itself: where the workgroups of both (32 rows or keys counted as
// one) are about as many as the CUs can hold.  2 x 4 heads x 512 rows with documents, D = 64, forward and backward: 64.9 us against
// 69.0 with two launches.  At the line, 8 x 8 heads x 128, causal: 28.1 us against 26.2 and the gap between two launches.  Not
// with ids where the empty places of the plan's order are more workgroups than that (8 x 32 x 29, 8192 of them, 1.5 times as long), nor
// without a mask where all chains are long and alike, as many rows as keys, and leave a last round half empty (4 x 1754, D = 64, 440
// workgroups 174 : 149; 17 random problems 0.89 [0.85, 0.97]).  Where dk/dv's are the longer ones or the shorter, for heads that share keys or other numbers of
// rows, the two fill each other's gaps (2 x 4/1 x 1219, D = 128 312 : 395, 1 x 2 x 4240 on 2436 538 : 671).
bool bwd_f32_in_one(const KArgs& a, int D, bool causal) {
  const int64_t keys = int64_t((a.N + 31) / 32) * a.B * a.Hk, wgs = int64_t((a.M + 31) / 32) * a.B * a.H + keys;
  if (wgs > 2 * kCUs || int64_t(a.Pp / 32) * a.B * a.H + keys > 8 * kCUs) return false;
  const int longer = std::max(a.M, a.N), shorter = std::min(a.M, a.N);
  return causal || wgs <= kCUs * 3 / 2 || a.G > 1 || D < 32 || shorter <= 63 * kSB || 4 * longer > 5 * shorter;
}
int bwd_f32_shapes(const KArgs& a, int D, bool causal, bool doc) {
  auto both = [&](auto mode) { return 0x10 * shape<kDq, decltype(mode)::value>(a, D, causal) + 0x40 * shape<kDkdv, decltype(mode)::value>(a, D, causal); };
  return doc ? both(IntC<kDoc>{}) : a.bmask != nullptr ? both(IntC<kBlock>{}) : both(IntC<kPlain>{});
}
int launch_bwd_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s) { return launch_d<kBoth>(a, D, causal, doc, s); }

int launch_bwd_delta_f32(const KArgs& a, int D, hipStream_t s) {
  const int BH = a.B * a.H < 65535 ? a.B * a.H : 65535;
  switch (D) {
    case 128: hipLaunchKernelGGL((delta_f32_kernel<128>), dim3((a.M + 7) / 8, BH), dim3(kDeltaThreads), 0, s, a); break;
    case 64: hipLaunchKernelGGL((delta_f32_kernel<64>), dim3((a.M + 15) / 16, BH), dim3(kDeltaThreads), 0, s, a); break;
    case 32: hipLaunchKernelGGL((delta_f32_kernel<32>), dim3((a.M + 31) / 32, BH), dim3(kDeltaThreads), 0, s, a); break;
    case 16: hipLaunchKernelGGL((delta_f32_kernel<16>), dim3((a.M + 63) / 64, BH), dim3(kDeltaThreads), 0, s, a); break;
    default: return -1;
  }
  return (int)hipGetLastError();
}

}  // namespace fa
