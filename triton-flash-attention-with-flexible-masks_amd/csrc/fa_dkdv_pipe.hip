// dK/dV at D = 128 without ids as a pipeline of two kinds of waves, for long streams of query tiles.
//
// A workgroup holds 128 keys in 8 waves, two to each block of 32 keys.  One wave of a pair ("score") computes S -> P -> dV, the
// other ("gradient") dP -> dS -> dK, so that each needs one operand set and one accumulator set and two waves fit on a SIMD.
// Query tiles (Q, dO, LSE, delta; 64 rows) are streamed through three stages of LDS, and the gradient wave runs behind:
// between two barriers
//   score wave     S(t) = Q K^T  |  P(t) -> LDS (fp16)         |  dV += dO(t)^T P(t)
//   gradient wave  -dS(t-1) = P(t-1) * (delta - dP(t-1))       |  -dK += Q(t-1)^T -dS(t-1),  delta - dP(t) (from delta, with -V)
// Neither waits for what the other does in the same step (P crosses behind the barrier of the tile stream: no flag, no polling),
// and the stream goes on through the query heads of a group without draining.
//
// What bounds it: the power limit first.  On random operands the clock settles at 2.10 GHz with the matrix pipes 51 % busy (counters,
// causal, 32 heads x 16384 rows; 3 stages x 32 KB, 32 KB of P: one workgroup to a CU); on zeros the same launch takes 3.4 ms instead of 4.2.  Causal, 32 heads x 16384
// rows, against the form in which the gradient wave polls for the P of its own tile: 4.51 -> 4.26, 4.42 -> 4.20, 4.84 -> 4.60 ms
// on three cards; with the subtraction of delta in the accumulators (see fa_bwd_dkdv.hip) another 4.20 -> 3.95.
// Steps of 32 rows (four stages) in workgroups of 128 or 64 keys: 4.60 ms against 4.26, and slower than the polling form with 64
// keys on short streams too (window of 1024 717 : 692 us, documents 702 : 689, packed sequences 293 : 288).
#include "fa_tile.h"

namespace fa {
#ifdef FA_TRACE
FA_TRACE_ARRAY(g_trace_pipe);   // words as in fa_bwd_dkdv.hip, of the first score wave (word 1 is 0: nothing is polled)
#endif

constexpr int kPipePre = 4;    // row-wise operand fragments requested ahead of their MFMA
constexpr int kPipePre2 = 3;   // transposed ones

template <int D>
constexpr size_t dkdv_pipe_lds() { return 3 * (2 * 64 * D * 2 + 512) + 2 * 4 * 4096; }

template <typename Tag, bool CAUSAL>
FA_DEV void dkdv_pipe_body(const KArgs& a, const int bid, char* smem) {
  using E = Elem<Tag>;
  using T = typename E::scalar;
  using vec8 = typename E::vec8;
  constexpr int D = 128, NKB = 4, BK = 32 * NKB, BQ = 64, KS = D / 16, DBN = D / 32, NW = 2 * NKB, NST = 3;
  constexpr int TILE_BYTES = BQ * D * 2, STAGE = 2 * TILE_BYTES;   // Q, dO
  constexpr int AUX_OFF = NST * STAGE, AUX_BYTES = 512;            // per stage: LSE, delta
  constexpr int P_OFF = AUX_OFF + NST * AUX_BYTES, P_BYTES = 4096; // [2 (tile parity)][NKB]: P of 64 rows x 32 keys as fp16
  using Loader = TileLoader<D, BQ, D, NW>;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // waves of a kind share a SIMD (waves go round the four of them): 4.19 ms against 4.30 for one of each kind, which both want the
  // matrix pipe when a step begins
  const int role = wave & 1, kb = wave >> 1;
  const int lq = lane & 31, g = lane >> 5;
  const int nKt = (a.N + BK - 1) / BK;
  FA_STAMP(g_trace_pipe, 0, FA_CLOCK()); FA_STAMP(g_trace_pipe, 1, 0); FA_STAMP(g_trace_pipe, 5, 0); FA_STAMP(g_trace_pipe, 7, -1);
  FA_TRACE_ONLY(int tr_tiles = 0; bool tr_first = false;)
  int kt, bhk;
  if (!block_to_tile(nKt, a.B * a.Hk, false, kt, bhk, bid)) return;  // causal: the first key tiles see the most rows
  FA_STAMP(g_trace_pipe, 7, (long long)kt | ((long long)bhk << 16));
  const int b = bhk / a.Hk, hk = bhk % a.Hk;
  const int M = a.M, N = a.N, gap = a.gap, G = a.G, win = a.win, pfx_m1 = a.pfx_m1;
  const int n0 = kt * BK, nw = n0 + kb * 32, key = nw + lq, keyc = key < N ? key : N - 1;

  // B operand held for the whole kernel: K^T for the score wave, V^T for the gradient wave
  const T* srcp = role == 0 ? reinterpret_cast<const T*>(a.k) + b * a.k_bs + hk * a.k_hs + keyc * a.k_rs
                            : reinterpret_cast<const T*>(a.v) + b * a.v_bs + hk * a.v_hs + keyc * a.v_rs;
  vec8 frag[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) frag[ks] = *reinterpret_cast<const vec8*>(srcp + ks * 16 + g * 8);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) settle(frag[ks]);
  // (the gradient's first product starts from delta and runs on -V: its accumulators hold delta - dP, dS comes out with the sign
  // turned, put right by the scale at the end, and the subtraction costs no instruction of its own)
  if (role == 1) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) frag[ks] = neg8<E>(frag[ks]);
  }
  const float c = a.scale_log2e;
  // rows that may see this lane's key: [row_lo, row_lo + row_span)
  const int row_lo = CAUSAL ? (key <= pfx_m1 ? 0 : max(0, key - gap)) : 0;
  const int row_hi = CAUSAL ? min(M - 1, key - gap + win - 1) : M - 1;
  const unsigned row_span = (key < N && row_hi >= row_lo) ? (unsigned)(row_hi - row_lo + 1) : 0u;

  LdsOffsets<D> lo;
  lo.init();
  f32x16 acc[DBN];   // dV^T (score wave) or dK^T (gradient wave): lane = key column, registers = d rows
#pragma unroll
  for (int db = 0; db < DBN; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;

  // the stream: every query tile this workgroup can need, of one query head of the group after the other
  const int first = CAUSAL ? (n0 <= pfx_m1 ? 0 : max(0, n0 - gap) / BQ) : 0;
  const int wg_rhi = CAUSAL ? min(M - 1, n0 + BK - 1 - gap + win - 1) : M - 1;   // the last row that sees a key of this workgroup
  const int last = CAUSAL ? min((M + BQ - 1) / BQ, max(0, wg_rhi + BQ) / BQ) : (M + BQ - 1) / BQ;
  int gi = 0;
  const int* auxp = nullptr;
  Loader ldQ, ldO;
  auto open_head = [&]() __attribute__((always_inline)) {
    LateArgs& ga = late_args();
    const int h = hk * G + gi;
    auxp = reinterpret_cast<const int*>(wave == 0 ? ga.lse : ga.delta) + (int64_t(b) * ga.H + h) * M;
    ldQ.init(reinterpret_cast<const T*>(ga.q) + b * ga.q_bs + h * ga.q_hs, ga.q_rs, M);
    ldO.init(reinterpret_cast<const T*>(ga.dout) + b * ga.do_bs + h * ga.do_hs, ga.do_rs, M);
  };
  constexpr int NPART = 2 * Loader::PER;
  auto load_part = [&](const int tile, const int stage, const int j) __attribute__((always_inline)) {
    const int i = j >> 1;
    const Loader& ld = (j & 1) ? ldO : ldQ;
    buf_load_lds16(ld.rsrc, smem + stage * STAGE + (j & 1) * TILE_BYTES + (i * NW + wave) * 1024, ld.voff, (tile * BQ + i * NW * Loader::RPI) * ld.row_bytes);
  };
  auto load_aux = [&](const int tile, const int stage) __attribute__((always_inline)) {
    const int r = min(tile * BQ + lane, M - 1);
    if (wave < 2) glb_load_lds4(auxp + r, smem + AUX_OFF + stage * AUX_BYTES + wave * 256);
  };
  // decisions of this wave pair for a query tile
  auto decide = [&](const int t) __attribute__((always_inline)) {
    const int m0 = t * BQ, rmin = m0, rmax = min(m0 + BQ - 1, M - 1);
    const bool skip = (nw >= N) || (CAUSAL && ((gap + rmax < nw && nw > pfx_m1) || gap + rmin - win + 1 > nw + 31));
    const bool lim = (m0 + BQ > M) || (nw + 32 > N) ||
                     (CAUSAL && ((gap + rmin < nw + 31 && nw + 31 > pfx_m1) || gap + rmax - win + 1 > nw));
    return (skip ? TF_SKIP : 0) | (lim ? TF_LIM : 0);
  };
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  // two row blocks of first products, fed alternately (see fa_bwd_dkdv.hip)
  auto first_products = [&](const char* rows, f32x16 (&x)[2]) __attribute__((always_inline)) {
    mfma_phase();
    __builtin_amdgcn_sched_barrier(0);
    constexpr int NF = 2 * KS, PF = kPipePre;
    auto fetch = [&](const int i) __attribute__((always_inline)) { return lds_row8<E>(rows + lo.row[i / 2] + (i & 1) * 32 * D * 2); };
    vec8 rf[NF];
#pragma unroll
    for (int i = 0; i < PF; ++i) rf[i] = fetch(i);
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      if (i + PF < NF) rf[i + PF] = fetch(i + PF);
      __builtin_amdgcn_sched_barrier(0);
      x[i & 1] = E::mfma32(rf[i], frag[i / 2], x[i & 1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    vector_phase();
  };
  auto second_products = [&](const char* tr, const vec8 (&yf)[4]) __attribute__((always_inline)) {
    mfma_phase();
    constexpr int NM = 4 * DBN, PRE = kPipePre2;
    auto fetch = [&](const int i) __attribute__((always_inline)) {
      const int c16 = i / DBN, db = i % DBN;
      return lds_tr8<E>(tr + lo.tr[db][0] + c16 * 16 * D * 2, tr + lo.tr[db][1] + c16 * 16 * D * 2);
    };
    __builtin_amdgcn_sched_barrier(0);
    vec8 tf[NM];
#pragma unroll
    for (int i = 0; i < PRE; ++i) tf[i] = fetch(i);
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      if (i + PRE < NM) tf[i + PRE] = fetch(i + PRE);
      __builtin_amdgcn_sched_barrier(0);
      acc[i % DBN] = E::mfma32(tf[i], yf[i / DBN], acc[i % DBN]);
    }
    __builtin_amdgcn_sched_barrier(0);
    vector_phase();
  };

  auto stream = [&](auto role_c) __attribute__((always_inline)) {
    constexpr int ROLE = decltype(role_c)::value;
    f32x16 x[2];   // gradient wave: delta - dP of the tile before, kept from step to step
    int prev_fl = TF_SKIP;
    int t = first, stage = 0, par = 0;
    bool more = first < last, prev = false;
    if (more) {
      open_head();
      FA_STAMP(g_trace_pipe, 2, FA_CLOCK());
#pragma unroll
      for (int j = 0; j < NPART; ++j) load_part(t, 0, j);
      load_aux(t, 0);
    }
    while (more || prev) {
      const int cur = t, cur_fl = more ? decide(t) : TF_SKIP;
      const int m0 = cur * BQ;
      const int pst = stage == 0 ? NST - 1 : stage - 1, nst = stage == NST - 1 ? 0 : stage + 1;
      wait_async_loads();
      __syncthreads();
      FA_TRACE_ONLY(if (!tr_first) { FA_STAMP(g_trace_pipe, 3, FA_CLOCK()); tr_first = true; } tr_tiles += more;)
      // the tile after this one
      bool nmore = false;
      if (more) {
        nmore = true;
        if (++t >= last) {
          t = first;
          if (++gi < G) open_head(); else nmore = false;
        }
        if (nmore) {
          load_part(t, nst, 0); load_part(t, nst, 1);
          load_aux(t, nst);
        }
      }
      auto load_rest = [&]() __attribute__((always_inline)) {
        if (!nmore) return;
#pragma unroll
        for (int j = 2; j < NPART; ++j) load_part(t, nst, j);
      };
      const char* lqt = smem + stage * STAGE;
      const char* ldo = lqt + TILE_BYTES;
      if constexpr (ROLE == 0) {
        if (cur_fl & TF_SKIP) { load_rest(); }
        else {
          const char* aux = smem + AUX_OFF + stage * AUX_BYTES;
          f32x4 Lv[2][4];
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) Lv[0][q4] = *reinterpret_cast<const f32x4*>(aux + (8 * q4 + 4 * g) * 4);
          x[0] = zero; x[1] = zero;
          first_products(lqt, x);
          load_rest();
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) Lv[1][q4] = *reinterpret_cast<const f32x4*>(aux + (32 + 8 * q4 + 4 * g) * 4);
          vec8 yf[4];
          char* pbuf = smem + P_OFF + (par * NKB + kb) * P_BYTES + lane * 16;
#pragma unroll
          for (int qb = 0; qb < 2; ++qb) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
#pragma unroll
              for (int e = 0; e < 4; ++e) x[qb][4 * q4 + e] = fast_exp2(__builtin_fmaf(x[qb][4 * q4 + e], c, -Lv[qb][q4][e]));
            if (cur_fl & TF_LIM) {
              asm volatile("" ::: "memory");  // keep this a real (wave-uniform) branch: never if-converted
#pragma unroll
              for (int q4 = 0; q4 < 4; ++q4)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  x[qb][4 * q4 + e] = (unsigned)(m0 + 32 * qb + 8 * q4 + 4 * g + e - row_lo) < row_span ? x[qb][4 * q4 + e] : 0.f;
            }
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              vec8& y = yf[2 * qb + half];
#pragma unroll
              for (int e = 0; e < 8; e += 2) {
                const typename E::vec2 pr = E::cvt2(x[qb][8 * half + e], x[qb][8 * half + e + 1]);
                y[e] = pr[0]; y[e + 1] = pr[1];
              }
              f16x8 ph;
#pragma unroll
              for (int e = 0; e < 8; e += 2) {
                const f32x2 pp = {x[qb][8 * half + e], x[qb][8 * half + e + 1]};
                const f16x2 hh = __builtin_convertvector(pp, f16x2);
                ph[e] = hh[0]; ph[e + 1] = hh[1];
              }
              *reinterpret_cast<f16x8*>(pbuf + (2 * qb + half) * 1024) = ph;
            }
          }
          second_products(ldo, yf);
        }
      } else {
        if (!(prev_fl & TF_SKIP)) {
          const char* pbuf = smem + P_OFF + ((par ^ 1) * NKB + kb) * P_BYTES + lane * 16;
          vec8 yf[4];
          f16x8 ph[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) ph[i] = *reinterpret_cast<const f16x8*>(pbuf + i * 1024);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
              float s0, s1;
              mul_f16_f32(ph[i], e, x[i >> 1][8 * (i & 1) + e], x[i >> 1][8 * (i & 1) + e + 1], s0, s1);
              const typename E::vec2 pr = E::cvt2(s0, s1);
              yf[i][e] = pr[0]; yf[i][e + 1] = pr[1];
            }
          load_rest();
          second_products(smem + pst * STAGE, yf);
        } else load_rest();
        if (!(cur_fl & TF_SKIP)) {
          const char* aux = smem + AUX_OFF + stage * AUX_BYTES + 256;
#pragma unroll
          for (int qb = 0; qb < 2; ++qb)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
              const f32x4 dl = *reinterpret_cast<const f32x4*>(aux + (32 * qb + 8 * q4 + 4 * g) * 4);
#pragma unroll
              for (int e = 0; e < 4; ++e) x[qb][4 * q4 + e] = dl[e];
            }
          first_products(ldo, x);
        }
      }
      prev = more; prev_fl = cur_fl; more = nmore;
      stage = nst; par ^= 1;
    }
  };
  if (role == 0) stream(IntC<0>{}); else stream(IntC<1>{});
  FA_STAMP(g_trace_pipe, 4, FA_CLOCK()); FA_STAMP(g_trace_pipe, 6, tr_tiles);

  // dK / dV rows leave through LDS (store_rows_through_lds), once every wave is done with the last query tile
  LateArgs& la = late_args();
  __syncthreads();
  char* patch = smem + wave * row_patch_bytes<D>();
  T* base = role == 0 ? reinterpret_cast<T*>(la.dv) + b * la.dv_bs + hk * la.dv_hs : reinterpret_cast<T*>(la.dk) + b * la.dk_bs + hk * la.dk_hs;
  const int64_t rs = role == 0 ? la.dv_rs : la.dk_rs;
  store_rows_through_lds<E, D, DBN>(patch, acc, role == 0 ? 1.0f : -la.scale, [&](const int r) -> T* {
    return nw + r < N ? base + int64_t(nw + r) * rs : nullptr;
  });
  FA_STAMP(g_trace_pipe, 5, FA_CLOCK());
}

template <typename Tag, bool CAUSAL>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bwd_dkdv_pipe_kernel(const KArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  dkdv_pipe_body<Tag, CAUSAL>(a, (int)blockIdx.x, smem);
}
template <typename Tag, bool CAUSAL>
static int launch_pipe(const KArgs& a, hipStream_t s) {
  constexpr size_t lds = dkdv_pipe_lds<128>();
  auto kern = bwd_dkdv_pipe_kernel<Tag, CAUSAL>;
  static bool lds_allowed[64] = {};   // per kernel instantiation and device
  if (int e = allow_lds(kern, lds, lds_allowed)) return e;
  hipLaunchKernelGGL(kern, dim3(grid_blocks((a.N + 127) / 128, a.B * a.Hk)), dim3(512), lds, s, a);
  return (int)hipGetLastError();
}

int launch_dkdv_pipe(const KArgs& a, int dtype, bool causal, hipStream_t s) {
  if (dtype == FA_DTYPE_BF16) return causal ? launch_pipe<bf16_t, true>(a, s) : launch_pipe<bf16_t, false>(a, s);
  return causal ? launch_pipe<fp16_t, true>(a, s) : launch_pipe<fp16_t, false>(a, s);
}
#ifdef FA_TRACE
int trace_read_pipe(long long* host, int n) { return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(g_trace_pipe), size_t(n) * 8); }
#endif

}  // namespace fa
