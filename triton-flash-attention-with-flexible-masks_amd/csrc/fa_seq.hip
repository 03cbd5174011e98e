// Tile tables of a packed batch of sequences (FA_SCORE_MODE3_PACKED), and the arrival counters of the launches that
// split key ranges without a mask plan.
//
// The boundaries of the sequences are known on the device only, so the kernels are launched for as many tiles as the
// totals can give and look their tile up here: a sequence starts a tile of its own, and its rows and keys are named by
// pointer and length, so the kernels run the code of the unmasked problem on it -- no ids, no gather, no tile that two
// sequences share.  One kernel, one workgroup per table; it takes the place of the dozen small kernels (ids, positions,
// mask plan) that a packed batch needed when it was given to the kernels as a document mask.
#include <stddef.h>

#include "fa_tile.h"

namespace fa {
namespace {

static_assert(offsetof(SeqTile, gap) == 16 && offsetof(SeqTile, nchunk) == 28 && offsetof(SeqTile, part) == 36, "the plan writes entries in pieces of 16 bytes");

constexpr int kThreads = 1024;
constexpr int kBuckets = 128;     // classes of tile lengths the table is sorted by, longest first
constexpr int kLdsSeqs = 8192;    // sequences whose tile offsets fit LDS (more: they are kept in the table's own memory)
constexpr int kLdsCu = 2048;      // sequences whose boundaries are kept in LDS too (more: read again where they are needed)

struct SeqPlanArgs {
  const void* cu_q;
  const void* cu_k;
  int i64, nseq, Tq, Tk, pack, bm, bk, causal, win;
  int spare, min_chunk, heads;    // extra entries a split may use, key tiles per chunk at least, head groups of the launch
  SeqHdr* hdr;
  SeqTile* qtab;
  SeqTile* ktab;
  int nQ, nK;                     // capacities
  int* cnt;
  int n_cnt;
};

struct Seq { int q0, M, k0, N, gap; };

FA_DEV int cu_at(const void* p, int i64, int i, int total) {
  const long long v = i64 ? reinterpret_cast<const long long*>(p)[i] : (long long)reinterpret_cast<const int*>(p)[i];
  return v < 0 ? 0 : (v > total ? total : (int)v);
}
// sequence s of nseq; number nseq is what lies behind the last boundary
FA_DEV int bound_at(const void* cu, int i64, int nseq, int total, int s) { return s == 0 ? 0 : (s > nseq ? total : cu_at(cu, i64, s, total)); }
FA_DEV Seq seq_of_bounds(int nseq, int s, int q0, int q1, int k0, int k1) {
  Seq r;
  r.q0 = q0; r.k0 = k0; r.M = max(0, q1 - q0); r.N = max(0, k1 - k0);
  r.gap = s < nseq ? r.N - r.M : 0;
  return r;
}

// v and what stands `CTRL` lanes before it; lanes that CTRL or ROWS leave without such a lane get `none`.  (Every lane of the wave is active where
// these are called.  A step costs some ten clocks; through ds_bpermute, as __shfl, it was 130.)
template <int CTRL, int ROWS = 0xf>
FA_DEV int lanes_before(int v, int none) { return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false); }
constexpr int kShr1 = 0x111, kShr2 = 0x112, kShr4 = 0x114, kShr8 = 0x118, kBcast15 = 0x142, kBcast31 = 0x143;   // within rows of 16 lanes; last lane of a row, of two rows, to the next
template <typename F>
FA_DEV int wave_fold(int v, int none, F&& f) {   // inclusive, over the lanes of a wave
  v = f(v, lanes_before<kShr1>(v, none));
  v = f(v, lanes_before<kShr2>(v, none));
  v = f(v, lanes_before<kShr4>(v, none));
  v = f(v, lanes_before<kShr8>(v, none));
  v = f(v, lanes_before<kBcast15, 0xa>(v, none));
  v = f(v, lanes_before<kBcast31, 0xc>(v, none));
  return v;
}
FA_DEV int wave_scan(int v) { return wave_fold(v, 0, [](int a, int b) { return a + b; }); }
FA_DEV int wave_max(int v) { return __builtin_amdgcn_readlane(wave_fold(v, (int)0x80000000, [](int a, int b) { return max(a, b); }), 63); }
FA_DEV float wave_sum(float v) {
  const int r = wave_fold(__float_as_int(v), 0, [](int a, int b) { return __float_as_int(__int_as_float(a) + __int_as_float(b)); });
  return __int_as_float(__builtin_amdgcn_readlane(r, 63));
}

// Block 0 writes the query tiles, block 1 the key tiles.  What bounds it: a chain of short phases in one workgroup, each the latency of a few LDS
// accesses and a barrier.  32 sequences with 91 query and 998 key tiles 8.6 -> 5.7 us (a chunked prefill of them 104.2 -> 101.8), 24 with 466 and
// 240 tiles 9.9 -> 7.4, against waves' scans through ds_bpermute, flat look-ups, two passes of atomics and whole entries of 64 bytes.
// BIG: more than kLdsSeqs sequences, their offsets in global memory (a kernel of its own: through a pointer to either, every access is a flat one).
template <bool BIG>
__global__ __launch_bounds__(kThreads) void seq_plan_kernel(const SeqPlanArgs p, int* __restrict__ spill) {
  constexpr int kWaves = kThreads / 64;
  __shared__ int s_off[BIG ? 1 : kLdsSeqs + 1];
  __shared__ int s_cuq[kLdsCu + 2], s_cuk[kLdsCu + 2];
  __shared__ int s_wave[2][kWaves], s_max[kWaves];
  __shared__ float s_work[kWaves];
  __shared__ int s_bucket[kBuckets];
  __shared__ int s_tot, s_cnt, s_part;
  const bool keys = blockIdx.x == 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ns = p.nseq + 1;
  int* const far = spill + (keys ? ns + 1 : 0);
  auto off = [&](int s) -> int { if constexpr (BIG) return far[s]; else return s_off[s]; };
  auto put_off = [&](int s, int v) { if constexpr (BIG) far[s] = v; else s_off[s] = v; };
  if (!keys)
    for (int i = tid; i < p.n_cnt; i += kThreads) p.cnt[i] = 0;
  const bool in_lds = ns <= kLdsCu;
  if (in_lds)
    for (int i = tid; i <= ns; i += kThreads) {
      s_cuq[i] = bound_at(p.cu_q, p.i64, p.nseq, p.Tq, i);
      s_cuk[i] = bound_at(p.cu_k, p.i64, p.nseq, p.Tk, i);
    }
  auto seq_at = [&](int s) {
    if (in_lds) return seq_of_bounds(p.nseq, s, s_cuq[s], s_cuq[s + 1], s_cuk[s], s_cuk[s + 1]);
    return seq_of_bounds(p.nseq, s, bound_at(p.cu_q, p.i64, p.nseq, p.Tq, s), bound_at(p.cu_q, p.i64, p.nseq, p.Tq, s + 1),
                         bound_at(p.cu_k, p.i64, p.nseq, p.Tk, s), bound_at(p.cu_k, p.i64, p.nseq, p.Tk, s + 1));
  };
  if (tid == 0) { s_cnt = 0; s_part = 0; }
  for (int i = tid; i < kBuckets; i += kThreads) s_bucket[i] = 0;
  __syncthreads();

  // (packed rows stay below 2^31; tile heights are powers of two, and mostly the heads that share a tile: no 64-bit or general division by them)
  const int pack_sh = (p.pack & (p.pack - 1)) == 0 ? __builtin_ctz(p.pack) : -1;
  auto query_of = [&](unsigned r) { return int(pack_sh >= 0 ? r >> pack_sh : r / unsigned(p.pack)); };
  const int sh = __builtin_ctz(keys ? p.bk : p.bm);
  const unsigned pack = p.pack, bm = p.bm;
  auto tiles_of = [&](const Seq& q) { return keys ? (q.N + p.bk - 1) >> sh : int((unsigned(q.M) * pack + bm - 1) >> sh); };
  // length of a tile: 64-key tiles its rows see, or 64-row tiles that see its keys
  auto length_of = [&](const Seq& q, int t) {
    if (keys) {
      const int n0 = t * p.bk, n1 = min(q.N, n0 + p.bk) - 1;
      const int lo = p.causal ? max(0, n0 - q.gap) : 0;
      const int hi = p.causal ? min(q.M - 1, n1 - q.gap + p.win - 1) : q.M - 1;
      return hi >= lo ? hi / 64 - lo / 64 + 1 : 0;
    }
    const int r0 = query_of(unsigned(t) << sh), r1 = query_of(min(unsigned(q.M) * pack, unsigned(t + 1) << sh) - 1);
    const int lo = p.causal ? max(0, q.gap + r0 - p.win + 1) : 0;
    const int hi = p.causal ? min(q.N - 1, q.gap + r1) : q.N - 1;
    return hi >= lo ? hi / 64 - lo / 64 + 1 : 0;
  };

  // tile offsets of the sequences
  int longest = 1, n_tiles = 0;
  for (int s0 = 0, buf = 0; s0 < ns; s0 += kThreads, buf ^= 1) {   // (two buffers: one barrier a round)
    const int s = s0 + tid;
    int n = 0;
    if (s < ns) {
      const Seq q = seq_at(s);
      n = tiles_of(q);
      longest = max(longest, (keys ? q.M : q.N) / 64 + 2);
    }
    const int inc = wave_scan(n);
    if (lane == 63) s_wave[buf][wave] = inc;
    __syncthreads();
    const int before = wave_scan(lane < kWaves ? s_wave[buf][lane] : 0);   // the waves' totals
    if (s < ns) put_off(s, n_tiles + (wave > 0 ? __builtin_amdgcn_readlane(before, wave - 1) : 0) + inc - n);
    n_tiles += __builtin_amdgcn_readlane(before, kWaves - 1);
  }
  if (tid == 0) put_off(ns, n_tiles);
  longest = wave_max(longest);
  if (lane == 0) s_max[wave] = longest;
  if constexpr (BIG) __threadfence_block();
  __syncthreads();
  longest = wave_max(lane < kWaves ? s_max[lane] : 1);
  const int nt = min(n_tiles, keys ? p.nK : p.nQ);
  auto seq_of = [&](int t) {   // last sequence whose offset is not past t (empty sequences share their offset with the next)
    int a = 0, b = ns - 1;
    while (a < b) {
      const int m = (a + b + 1) / 2;
      if (off(m) <= t) a = m; else b = m - 1;
    }
    return a;
  };

  // sequence and length of tile t; the thread's first one is looked up once for the three passes below
  int my_seq = -1, my_len = 0;
  if (tid < nt) { my_seq = seq_of(tid); my_len = length_of(seq_at(my_seq), tid - off(my_seq)); }
  auto look = [&](int t, int& s, int& len) {
    if (t == tid) { s = my_seq; len = my_len; return; }
    s = seq_of(t);
    len = length_of(seq_at(s), t - off(s));
  };

  // chunks: the work of all tiles over the entries a split launch aims at
  int chunk = 0x7fffffff;
  if (!keys) {
    const int spare = int64_t(nt) * p.heads >= kSeqFullWgs ? min(p.spare, kSeqTargetFull / p.heads + 1) : p.spare;
    float work = 0.f;
    for (int t = tid; t < nt; t += kThreads) {
      int s, len;
      look(t, s, len);
      work += float(len);
    }
    work = wave_sum(work);
    if (lane == 0) s_work[wave] = work;
    __syncthreads();
    work = wave_sum(lane < kWaves ? s_work[lane] : 0.f);
    chunk = max(p.min_chunk, int(work / spare) + 1);
  }
  const int longest_all = min(longest, chunk);
  const float to_bucket = float(kBuckets) / float(longest_all + 1);
  auto chunks_of = [&](int len) { return len <= chunk ? 1 : min(kSplitKMaxFew, (len + chunk - 1) / chunk); };
  auto bucket_of = [&](int len, int nc) {   // 0: the longest
    const int l = nc == 1 ? len : (len + nc - 1) / nc;
    return kBuckets - 1 - min(kBuckets - 1, int(float(l) * to_bucket));
  };
  int my_bucket = 0, my_place = 0;   // of the thread's first tile
  for (int t = tid; t < nt; t += kThreads) {
    int s, len;
    look(t, s, len);
    const int nc = chunks_of(len), bucket = bucket_of(len, nc), place = atomicAdd(&s_bucket[bucket], nc);
    if (t == tid) { my_bucket = bucket; my_place = place; }
  }
  __syncthreads();
  if (wave == 0) {   // exclusive offsets of the buckets
    int carry = 0;
    for (int b0 = 0; b0 < kBuckets; b0 += 64) {
      const int n = s_bucket[b0 + lane], inc = wave_scan(n);
      s_bucket[b0 + lane] = carry + inc - n;
      carry += __builtin_amdgcn_readlane(inc, 63);
    }
    if (lane == 0) s_tot = carry;
  }
  __syncthreads();
  SeqTile* tab = keys ? p.ktab : p.qtab;
  const int cap = keys ? p.nK : p.nQ;
  for (int t = tid; t < nt; t += kThreads) {
    int s, len;
    look(t, s, len);
    const Seq q = seq_at(s);
    const int nc = chunks_of(len);
    const int at = nt <= kThreads ? s_bucket[my_bucket] + my_place : atomicAdd(&s_bucket[bucket_of(len, nc)], nc);
    int cnt = 0, part = 0;
    if (nc > 1) { cnt = atomicAdd(&s_cnt, 1); part = atomicAdd(&s_part, nc); }
    for (int c = 0; c < nc && at + c < cap; ++c) {
      // (whole entries would be written in four pieces a thread, 64 bytes apart; what is read of them lies in the first three, of key tiles in two)
      i32x4* e = reinterpret_cast<i32x4*>(tab + at + c);
      e[0] = i32x4{q.q0, q.M, q.k0, q.N};
      e[1] = i32x4{q.gap, t - off(s), c, nc};
      if (!keys) e[2] = i32x4{cnt, part, 0, 0};
    }
  }
  if (tid == 0) {
    if (keys) p.hdr->nk = min(s_tot, cap);
    else p.hdr->nq = min(s_tot, cap);
  }
}

__global__ __launch_bounds__(256) void zero_kernel(int* __restrict__ p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

int launch_zero_counters(int* cnt, int n, hipStream_t s) {
  hipLaunchKernelGGL(zero_kernel, dim3((n + 255) / 256), dim3(256), 0, s, cnt, n);
  return (int)hipGetLastError();
}

int launch_seq_plan(const fa_params* p, const FwdCfg& c, const TabLayout& w, hipStream_t s) {
  char* ws = reinterpret_cast<char*>(p->workspace);
  const int nh = p->H / c.pack;
  SeqPlanArgs a;
  a.cu_q = p->eq; a.cu_k = p->ek; a.i64 = p->id_dtype == FA_IDTYPE_I64; a.nseq = p->nseq;
  a.Tq = p->M; a.Tk = p->N; a.pack = c.pack; a.bm = c.bm; a.bk = seq_key_tile(p->D);
  a.causal = p->causal != 0;
  a.win = p->window > 0 && p->window < 0x3fffffff ? p->window : 0x3fffffff;
  a.spare = w.nCnt; a.min_chunk = c.dec ? 4 : 8; a.heads = nh;
  a.hdr = reinterpret_cast<SeqHdr*>(ws + w.off_hdr);
  a.qtab = reinterpret_cast<SeqTile*>(ws + w.off_q);
  a.ktab = reinterpret_cast<SeqTile*>(ws + w.off_k);
  a.nQ = w.nQ; a.nK = w.nK;
  a.cnt = reinterpret_cast<int*>(ws + w.off_cnt);
  a.n_cnt = w.nCnt * nh;
  int* spill = reinterpret_cast<int*>(ws + w.off_spill);
  if (p->nseq + 1 <= kLdsSeqs) hipLaunchKernelGGL(seq_plan_kernel<false>, dim3(2), dim3(kThreads), 0, s, a, spill);
  else hipLaunchKernelGGL(seq_plan_kernel<true>, dim3(2), dim3(kThreads), 0, s, a, spill);
  return (int)hipGetLastError();
}

}  // namespace fa
