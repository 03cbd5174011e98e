// Forward for a handful of query rows against many keys (16-bit types, no ids): decoding, the last tokens of a prompt.
//
// Bound by memory: every K / V row is needed once per key head, 4 * D bytes for 4 * D * rows FLOPs, and the card reads
// at 4-5 TB/s.  What the layout is chosen for:
//   * all query heads of a key head share a workgroup: a tile is up to 32 (query, head of the group) pairs, so K and V
//     are read once per key head and not once per query head (the 128-row form read them G times);
//   * every wave streams key blocks of its own (32 keys: K and V, global -> LDS, kStages deep) and keeps a softmax state
//     of its own.  No barrier sits in the loop, 16 KB per wave and stage are in flight at D = 128, one workgroup of
//     four waves takes 128 KB of a CU's LDS; the four states are merged once, through LDS;
//   * the key range is cut into chunks until the chip is full (pick_split, fa_common.h); the last chunk to arrive
//     merges the partial results, rows x D fp32 each.
// Measured (16 sequences x 8 key heads x 6001 keys, G = 4, D = 128, bf16, 394 MB): 228 us in the 128-row form, 77 here, 5.1 TB/s
// with launch and merge.  Where short ranges leave more workgroups than CUs, two of them share one (half the LDS, the register file
// halved too): see kDecTiles2 and kDecShort in fa_common.h.  Starting the workgroups at different places of their ranges changed nothing (77.3).
#include "fa_tile.h"

namespace fa {
namespace {

// LDS of a wave: stages x (K + V) x 32 keys x D x 2 bytes.  One workgroup to a CU, or two (short ranges, see kDecTiles).
template <int WPC> constexpr int dec_stage_bytes() { return 32 * 1024 / WPC; }
template <int WPC, int D> constexpr size_t dec_lds() {
  const size_t merge = (512 + 4 * ((D + 31) / 32) * 16 * 64) * 4, tiles = 4 * dec_stage_bytes<WPC>();
  return merge > tiles ? merge : tiles;
}

// One wave's tile stream: 32 rows of D elements, global -> LDS, in the swizzled layout of fa_tile.h.
template <int DL, int GD>
struct WaveLoader {
  static constexpr int CPR = DL / 8, RPI = 64 / CPR, NI = 32 / RPI, NV = 16 / RPI < 1 ? 1 : 16 / RPI;
  buf_rsrc_t rsrc;
  int voff[NV];   // the swizzle has a period of 16 rows: NV instructions, then the same offsets again
  int row_bytes;
  FA_DEV void init(const void* base, int64_t rs, int nrows) {
    const int lane = threadIdx.x & 63;
    rsrc = make_rsrc(base, nrows > 0 ? (unsigned)((int64_t(nrows - 1) * rs + GD) * 2) : 0u);
    row_bytes = int(rs) * 2;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int r = lane / CPR, c = (lane % CPR) ^ swz<DL, SWZ_ROW>(v * RPI + r);
      voff[v] = c < GD / 8 ? r * row_bytes + c * 16 : kOobOffset;
    }
  }
  FA_DEV void issue(int row0, const char* lds) const {
#pragma unroll
    for (int i = 0; i < NI; ++i) buf_load_lds16(rsrc, lds + i * 1024, voff[i % NV], (row0 + i * RPI) * row_bytes);
  }
};

template <int N> FA_DEV void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }

template <typename Tag, int D, bool CAUSAL, int WPC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPC, WPC)))
void decode_kernel(const KArgs a) {
  using E = Elem<Tag>;
  using T = typename E::scalar;
  using vec8 = typename E::vec8;
  constexpr int KS = D / 16, DL = D < 32 ? 32 : D, DBN = DL / 32;
  constexpr int TB = 32 * DL * 2;                          // bytes of a 32-key tile
  constexpr int NST = dec_stage_bytes<WPC>() / (2 * TB);   // stages per wave: 2 (1) at D = 128, 4 (2) at 64, 8 (4) below
  using Loader = WaveLoader<DL, D>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lq = lane & 31, g = lane >> 5;

  const TileGeo ge = tile_geo(a, (int)blockIdx.x);
  if (ge.M < 0) return;   // a slot the plan did not use
  const int Mr = ge.M * a.pack, r0 = ge.tile * 32;
  const int pr = r0 + lq;
  const bool live = pr < Mr;
  const int qi = live ? pr / a.pack : 0, hg = live ? pr - qi * a.pack : 0;
  const int rmin = r0 / a.pack, rmax = min(r0 + 31, Mr - 1) / a.pack;
  const int lim_i = CAUSAL ? min(max(ge.gap + qi, a.pfx_m1), ge.N - 1) : ge.N - 1;
  const int low_i = CAUSAL ? ge.gap + qi - a.win + 1 : -0x3fffffff;
  const int limmin = CAUSAL ? min(max(ge.gap + rmin, a.pfx_m1), ge.N - 1) : ge.N - 1;
  const int limmax = CAUSAL ? min(max(ge.gap + rmax, a.pfx_m1), ge.N - 1) : ge.N - 1;
  const int lowmax = CAUSAL ? ge.gap + rmax - a.win + 1 : -0x3fffffff;
  // key blocks (of 32) the tile sees, and this chunk's share of them (a multiple of the four waves)
  const int b0 = CAUSAL ? max(0, ge.gap + rmin - a.win + 1) / 32 : 0;
  const int b1 = (limmax + 32) / 32;
  const int per = (max(0, b1 - b0) + 4 * ge.nchunk - 1) / (4 * ge.nchunk) * 4;
  const int cb0 = b0 + ge.chunk * per, cb1 = min(b1, cb0 + per);

  const T* qp = reinterpret_cast<const T*>(a.q) + ge.b * a.q_bs + int64_t(ge.h0 + hg) * a.q_hs + (ge.q0 + qi) * a.q_rs;
  const T* kp = reinterpret_cast<const T*>(a.k) + ge.b * a.k_bs + ge.hk * a.k_hs + ge.k0 * a.k_rs;
  const T* vp = reinterpret_cast<const T*>(a.v) + ge.b * a.v_bs + ge.hk * a.v_hs + ge.k0 * a.v_rs;
  Loader ldK, ldV;
  ldK.init(kp, a.k_rs, ge.N);
  ldV.init(vp, a.v_rs, ge.N);
  char* my = smem + wave * dec_stage_bytes<WPC>();
  vec8 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const vec8*>(qp + ks * 16 + g * 8);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) settle(qf[ks]);
  float c = a.scale_log2e;
  if (c < 0.f) {   // keep max(raw score) == max(scaled score): move the sign into Q
    c = -c;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = neg8<E>(qf[ks]);
  }
  LdsOffsets<DL> lo;
  lo.init();

  constexpr float kUnset = -1e30f, kSumLimit = 4096.f;   // the lazily moved reference point of fa_fwd.hip
  float m_ref = kUnset, l_run = 0.f;
  f32x16 o[DBN];
#pragma unroll
  for (int db = 0; db < DBN; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  auto issue = [&](const int st, const int blk) __attribute__((always_inline)) {
    ldK.issue(blk * 32, my + st * (2 * TB));
    ldV.issue(blk * 32, my + st * (2 * TB) + TB);
  };
  auto compute = [&](const int st, const int blk) __attribute__((always_inline)) {
    const char* lk = my + st * (2 * TB);
    const char* lv = lk + TB;
    const int n0 = blk * 32;
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 s[2] = {zero, zero};
    vec8 kf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = lds_row8<E>(lk + lo.row[ks]);
    vec8 vf[2 * DBN];
#pragma unroll
    for (int i = 0; i < 2 * DBN; ++i)
      vf[i] = lds_tr8<E>(lv + lo.tr[i % DBN][0] + (i / DBN) * 16 * DL * 2, lv + lo.tr[i % DBN][1] + (i / DBN) * 16 * DL * 2);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s[ks & 1] = E::mfma32(kf[ks], qf[ks], s[ks & 1]);
    if (KS > 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[0][r] += s[1][r];
    }
    if (n0 + 31 > limmin || n0 < lowmax) {
      asm volatile("" ::: "memory");   // keep this a real (wave-uniform) branch
      mask_lim(s[0], lim_i - n0 - 4 * g, low_i - n0 - 4 * g, -INFINITY);
    }
    f32x16 p;
    float ps = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) { p[r] = fast_exp2(__builtin_fmaf(s[0][r], c, -m_ref)); ps += p[r]; }
    if (__builtin_amdgcn_ballot_w64(!(ps <= kSumLimit)) != 0) {
      float mx = s[0][0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[0][r]);
      mx = xhalf_max(mx) * c;
      const float m_new = fmaxf(m_ref, mx), alpha = fast_exp2(m_ref - m_new);
      m_ref = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DBN; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      ps = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) { p[r] = fast_exp2(__builtin_fmaf(s[0][r], c, -m_ref)); ps += p[r]; }
    }
    l_run += ps;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      vec8 pf;
#pragma unroll
      for (int t = 0; t < 8; t += 2) {
        const typename E::vec2 x = E::cvt2(p[8 * half + t], p[8 * half + t + 1]);
        pf[t] = x[0]; pf[t + 1] = x[1];
      }
#pragma unroll
      for (int db = 0; db < DBN; ++db) o[db] = E::mfma32(vf[half * DBN + db], pf, o[db]);
    }
  };

  // the wave's blocks: cb0 + wave, + 4, + 8, ...; stage j % NST holds the j-th of them
  constexpr int PER_STAGE = 2 * Loader::NI;
  const int nmine = cb1 - cb0 > wave ? (cb1 - cb0 - wave + 3) / 4 : 0;
  const int first = cb0 + wave;
#pragma unroll
  for (int st = 0; st < NST; ++st)
    if (st < nmine) issue(st, first + 4 * st);
  for (int j = 0; j < nmine; j += NST) {
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      if (j + st >= nmine) break;
      // the loads of the NST - 1 blocks behind this one may stay in flight; at the end of the range fewer were issued
      if (j + st + NST - 1 < nmine) wait_loads<(NST - 1) * PER_STAGE>(); else wait_loads<0>();
      compute(st, first + 4 * (j + st));
      if (j + st + NST < nmine) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this stage's reads are done before it is filled again
        issue(st, first + 4 * (j + st + NST));
      }
    }
  }

  // the four waves' states become one: wave `db` adds up columns 32 * db .. of every wave's O
  const float l_w = xhalf_sum(l_run);
  __syncthreads();   // nobody reads tiles any more
  float* mb = reinterpret_cast<float*>(smem);
  mb[wave * 64 + lane] = m_ref;
  mb[256 + wave * 64 + lane] = l_w;
#pragma unroll
  for (int db = 0; db < DBN; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) mb[512 + ((wave * DBN + db) * 16 + r) * 64 + lane] = o[db][r];
  __syncthreads();
  float wgt[4], m_tot = kUnset, l_tot = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) m_tot = fmaxf(m_tot, mb[w * 64 + lane]);
#pragma unroll
  for (int w = 0; w < 4; ++w) { wgt[w] = fast_exp2(mb[w * 64 + lane] - m_tot); l_tot += wgt[w] * mb[256 + w * 64 + lane]; }
  f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (wave < DBN) {
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += wgt[w] * mb[512 + ((w * DBN + wave) * 16 + r) * 64 + lane];
  }
  T* op = reinterpret_cast<T*>(a.o) + ge.b * a.o_bs + ge.h0 * a.o_hs + ge.q0 * a.o_rs;
  float* lsep = a.lse + (int64_t(ge.b) * a.H + ge.h0) * a.M + ge.q0;
  if (ge.nchunk == 1) {
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if (live && wave == 0 && g == 0) lsep[int64_t(hg) * a.M + qi] = l_tot > 0.f ? m_tot + fast_log2(l_tot) : -INFINITY;
    if (live && wave < DBN) {
      T* orow = op + hg * a.o_hs + qi * a.o_rs;
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int col = 32 * wave + 8 * q4 + 4 * g;
        if (col >= D) continue;
        const typename E::vec2 x0 = E::cvt2(acc[4 * q4] * inv, acc[4 * q4 + 1] * inv), x1 = E::cvt2(acc[4 * q4 + 2] * inv, acc[4 * q4 + 3] * inv);
        typename E::vec4 x = {x0[0], x0[1], x1[0], x1[1]};
        *reinterpret_cast<typename E::vec4*>(orow + col) = x;
      }
    }
    return;
  }
  // one chunk of several: the un-normalised sums leave as fp32, row by row, and the last chunk to arrive merges
  const int64_t pi = int64_t(ge.part) + int64_t(ge.chunk) * ge.pstride;
  float* po = a.sk_o + pi * (32 * D);
  float* pml = a.sk_ml + pi * (32 * 2);
  if (live && wave == 0 && g == 0) store_dev(pml + lq * 2, m_tot, l_tot);
  if (live && wave < DBN) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int col = 32 * wave + 8 * q4 + 4 * g;
      if (col >= D) continue;
      f32x4 x = {acc[4 * q4], acc[4 * q4 + 1], acc[4 * q4 + 2], acc[4 * q4 + 3]};
      store_dev(po + lq * D + col, x);
    }
  }
  if (!split_arrive(a.sk_cnt + ge.cnt, ge.nchunk)) return;
  constexpr int C4 = D / 4, NS = 8;
  const int nrow = min(32, Mr - r0);
  for (int i = threadIdx.x; i < nrow * C4; i += 256) {
    const int r = i / C4, c4 = i % C4;
    float mm = kUnset, ll = 0.f;
    f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < ge.nchunk; c0 += NS) {   // NS chunks side by side: every device-scope load is a round trip
      float m_[NS], l_[NS];
      f32x4 x_[NS];
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const int64_t pc = int64_t(ge.part) + int64_t(min(c0 + u, ge.nchunk - 1)) * ge.pstride;
        load_dev(a.sk_ml + pc * 64 + r * 2, m_[u], l_[u]);
        x_[u] = load_dev4(a.sk_o + pc * (32 * D) + r * D + 4 * c4);
      }
      float mn = mm;
#pragma unroll
      for (int u = 0; u < NS; ++u) mn = fmaxf(mn, m_[u]);
      const float al = fast_exp2(mm - mn);
      mm = mn; ll *= al; s4 *= al;
#pragma unroll
      for (int u = 0; u < NS; ++u) {
        const float w = c0 + u < ge.nchunk ? fast_exp2(m_[u] - mm) : 0.f;
        ll += w * l_[u];
        s4 += w * x_[u];
      }
    }
    const int pq = r0 + r, q_ = pq / a.pack, h_ = pq - q_ * a.pack;
    const float inv = ll > 0.f ? 1.0f / ll : 0.f;
    if (c4 == 0) lsep[int64_t(h_) * a.M + q_] = ll > 0.f ? mm + fast_log2(ll) : -INFINITY;
    const typename E::vec2 x0 = E::cvt2(s4[0] * inv, s4[1] * inv), x1 = E::cvt2(s4[2] * inv, s4[3] * inv);
    typename E::vec4 x = {x0[0], x0[1], x1[0], x1[1]};
    *reinterpret_cast<typename E::vec4*>(op + h_ * a.o_hs + q_ * a.o_rs + 4 * c4) = x;
  }
}

template <typename Tag, int D, bool CAUSAL, int WPC>
int launch_wpc(const KArgs& a, hipStream_t s) {
  auto kern = decode_kernel<Tag, D, CAUSAL, WPC>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, dec_lds<WPC, D>(), lds_allowed)) return e;
  hipLaunchKernelGGL(kern, dim3(tile_geo_blocks(a)), dim3(256), (dec_lds<WPC, D>()), s, a);
  return (int)hipGetLastError();
}
template <typename Tag, int D, bool CAUSAL>
int launch_one(const KArgs& a, hipStream_t s) {
  if (a.wpc > 1) return launch_wpc<Tag, D, CAUSAL, 2>(a, s);
  return launch_wpc<Tag, D, CAUSAL, 1>(a, s);
}
template <typename Tag>
int launch_d(const KArgs& a, int D, bool causal, hipStream_t s) {
  switch (D) {
    case 128: return causal ? launch_one<Tag, 128, true>(a, s) : launch_one<Tag, 128, false>(a, s);
    case 64: return causal ? launch_one<Tag, 64, true>(a, s) : launch_one<Tag, 64, false>(a, s);
    case 32: return causal ? launch_one<Tag, 32, true>(a, s) : launch_one<Tag, 32, false>(a, s);
    case 16: return causal ? launch_one<Tag, 16, true>(a, s) : launch_one<Tag, 16, false>(a, s);
    default: return -1;
  }
}

}  // namespace

int launch_decode(const KArgs& a, int dtype, int D, bool causal, hipStream_t s) {
  return dtype == FA_DTYPE_BF16 ? launch_d<bf16_t>(a, D, causal, s) : launch_d<fp16_t>(a, D, causal, s);
}

}  // namespace fa
