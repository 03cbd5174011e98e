// Shared device/host definitions for the gfx950 flash-attention kernels.
//
// Register-level conventions used by every compute kernel in this directory
// (CDNA4 v_mfma_f32_32x32x16_{bf16,f16}, wave64):
//   A operand (32 x 16): lane l holds row  (l & 31), k = 8*(l >> 5) .. +7
//   B operand (16 x 32): lane l holds col  (l & 31), k = 8*(l >> 5) .. +7
//   C/D       (32 x 32): lane l holds col  (l & 31), register r (0..15) is
//                        row 8*(r >> 2) + 4*(l >> 5) + (r & 3)
// ds_read_b64_tr_b16: inside each group of 16 lanes, result lane i, element e is
// taken from source lane 4*e + (i >> 2), element (i & 3) of its 8-byte read.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/flash_mi355.h"

namespace fa {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

#define FA_LDS(p) ((__attribute__((address_space(3))) void*)(p))
#define FA_GLB(p) ((const __attribute__((address_space(1))) void*)(p))
#define FA_DEV __device__ __forceinline__
#define FA_HD __host__ __device__ inline

constexpr float kLog2e = 1.4426950408889634f;

// Rows covered by one entry of the id summaries written by the mask plan.
constexpr int kSumRows = 64;
// The local-row part of the permuted order is padded to this many entries, so that a
// workgroup of up to 256 query rows never mixes local and global rows.
constexpr int kPermAlign = 256;
// Tiles of global rows (eq >= 0) see every key up to their own position, i.e. up to the whole
// sequence: a single workgroup walking 16K keys is the critical path of the kernel.  The key range
// of the first `tiles` such tiles of a (batch, head) is therefore cut into up to `k` chunks handled
// by different workgroups; each writes an fp32 partial result and the last one to arrive (an atomic
// counter per tile) merges them.  The merge order is fixed, results stay reproducible.
constexpr int kSplitMinTiles = 16;   // key tiles (of 64) per chunk below which splitting does not pay
constexpr int kSplitKMax = 4;        // more chunks did not pay on any shape with enough query tiles to fill the chip
constexpr int kSplitKMaxFew = 16;    // ... but they do when the whole launch is short of workgroups (few query rows)
constexpr int kSplitFewWgs = 1024;   // query tiles in the launch (all heads) below which it counts as short of workgroups
constexpr int kCUs = 256;
// Forward and dq of masked problems with few query tiles take tiles of 64 rows, whose waves split every key tile in two
// (QTileCtx::halved): twice the workgroups, each half as long, at about 1.3 times the instructions per pair.  By the workgroups that
// tiles of 128 rows would make, all heads counted, 64-row tiles : 128, geometric mean over random problems [smallest, largest]:
//   block map, kernels of a forward and backward [forward alone]
//                                    to 128                    to 256                    to 384                    to 512
//     D = 128, bands of 2 - 16     0.88, 0.83 - 0.92         1.02, 0.88 - 1.23         1.07, 0.90 - 1.18         1.13, 1.08 - 1.17 [1.25 - 1.41]
//              128 x 128 pieces    0.89, 0.82 - 0.94         0.93, 0.85 - 0.99         0.99, 0.83 - 1.10         1.06, 1.03 - 1.11
//              full                0.86, 0.83 - 0.90         0.89, 0.87 - 0.90         0.95, 0.90 - 1.02         0.99, 0.93 - 1.03
//              random, 10 - 30 %   0.87, 0.84 - 0.90         0.88, 0.70 - 0.95                          [0.74, 0.56 - 1.04]
//     D = 64,  bands               0.84, 0.79 - 0.90         0.98, 0.89 - 1.06         0.95, 0.88 - 1.05         1.10, 1.00 - 1.17 [1.06 - 1.29]
//              128 x 128 pieces    0.88, 0.86 - 0.89         0.94, 0.90 - 0.99         0.94, 0.89 - 1.00         0.99, 0.93 - 1.05
//              full                0.80, 0.79 - 0.81         0.92, 0.90 - 0.95         0.94, 0.91 - 0.98         0.94, 0.88 - 0.99
//              random                                        0.94, 0.92 - 0.96         0.91, 0.87 - 0.98         0.95, 0.94 - 0.95
//     The lines lie where narrow bands, whose workgroups are mostly set-up, begin to lose; the host cannot tell them from the others.  At D = 128 they do as soon
//     as two 64-row tiles share a CU (18 heads x 1024 rows, bands of 2 blocks, forward 9.8 -> 11.4 us, backward 13.8 -> 18.7), at D = 64 when a fourth would.
//   documents, kernels of a forward and backward [forward alone]
//                     512 to 1279 rows, to 256               to 128                  to 256                  to 384                  to 512
//     D = 128   0.94, 0.84 - 1.00 [.74 - 1.03]  0.91, 0.80 - 1.01       0.87, 0.76 - 0.94       0.95, 0.83 - 1.12       0.97, 0.80 - 1.06 [.68 - 1.24]
//     D = 64    0.97, 0.93 - 1.04 [.78 - 1.04]  0.91, 0.82 - 0.98       0.93, 0.81 - 1.01       0.92, 0.77 - 1.09       0.89, 0.79 - 1.00 [.65 - 1.18]
//     The line lies where tiles of 64 rows are all resident at once, two (D = 128) or three to a CU: beyond it documents without global rows, whose
//     workgroups are mostly set-up, take a second round for nothing (8 heads x 7109 rows, D = 128, forward and backward 114 -> 121 us, 4 x 8 x 1289 on 4235
//     keys 158 -> 176), which the host cannot tell from those that gain (12 x 5178 with a tenth of the rows global 164 -> 131).  Rows below
//     kLowLongRows gain nothing from the third: D = 64 to 384 1.00 - 1.02.
// Fewer than kLowMinRows rows keep tiles of 128: up to one workgroup to a CU they would gain 0.95 (D = 64) and 0.97 (D = 128) [0.82, 1.03] in the
// kernels of a forward and backward, whose passes wait for the host there, and a row whose softmax is kept in two states is rounded
// otherwise: dQ of 2 heads x 384 rows at a scale of 0.25, D = 128, comes out at 1.05 of the largest error that is allowed for (0.0595), with one
// state at 0.72, at the same 2-norm.  Neither do rows with positions of their own (packed sequences with ids) take them: D = 128 0.94 - 1.17, D = 64
// 0.88 - 1.05.
constexpr int kLowLongRows = 1280, kLowMinRows = 512;
inline int doc_rows(int B, int H, int M, int D, bool own_pos = false) {
  const int64_t wgs = int64_t(B) * H * ((M + 127) / 128);
  return !own_pos && M >= kLowMinRows && (wgs <= kCUs || (D <= 64 && M >= kLowLongRows && wgs <= kCUs * 3 / 2)) ? 64 : 128;
}
// dq of long rows at D = 128 would gain under random maps (16 heads x 16384 rows, a quarter on, 479 -> 425 us), whose tiles of 128 rows visit the columns of
// two unlike rows of blocks, and loses where neighbouring rows are alike: bands of 4 / 16 blocks 1.14 - 1.31 / 1.05 - 1.20, maps in pieces of 128 x 128
// 1.00 - 1.15, full ones 1.02 - 1.09 (16 - 32 heads x 6016 - 16384 rows, causal and not, as many keys and twice as many).
inline int block_rows(int B, int H, int M, int D) { return int64_t(B) * H * ((M + 127) / 128) <= (D > 64 ? kCUs / 2 : kCUs * 3 / 2) ? 64 : 128; }
struct SplitCfg {
  int k;      // chunks per tile (1: nothing is ever split)
  int tiles;  // global-row tiles per (batch, head) that can be split
  int rows;   // rows of a query tile, 128 or 64
};
// Chunks of at least 32 key tiles (2 .. kSplitKMax of them), and as many splittable tiles as the
// scratch budget allows (at most 64): long sequences with few heads have many global-row tiles, each
// of them long.  The budget is a hard bound on the scratch part of the workspace: with many (batch,
// head) pairs it buys fewer tiles per pair, down to none (such launches have workgroups to spare and
// short key ranges per tile; with fewer than two tiles in the budget at 4 chunks, 2 chunks are tried).
// With fewer than kSplitFewWgs query tiles in the whole launch (decoding, the tail of a long prompt, a short
// query block against a long packed key sequence) the chunks go down to kSplitMinTiles key tiles, up to
// kSplitKMaxFew of them.  Never more splittable tiles than M rows can fill.
constexpr uint64_t kSplitScratchBudget = uint64_t(128) << 20;   // bytes of sk_ml + sk_o
inline SplitCfg split_config(int B, int H, int M, int N, int D, bool own_pos, uint64_t budget = kSplitScratchBudget) {
  SplitCfg c = {1, 0, doc_rows(B, H, M, D, own_pos)};
  const int nKs = (N + kSumRows - 1) / kSumRows;
  if (nKs < 2 * kSplitMinTiles) return c;   // no key range can be long enough to be cut
  const int qtiles = (M + 127) / 128 + 1;   // 128-row tiles of global rows a (batch, head) can have
  const uint64_t wgs = uint64_t(B) * H * qtiles;
  if (wgs < kSplitFewWgs) {
    // Short of workgroups: the chunks of the global-row tiles are what fills the chip.  About 256 workgroups
    // that each stream their own K / V chunk keep the memory system busy (more of them only add merge work),
    // and every (batch, head) has at least one such tile.
    const uint64_t bh = uint64_t(B) * H;
    const int fill = int(256 / bh);
    const int kmax = fill < kSplitKMax ? kSplitKMax : (fill > kSplitKMaxFew ? kSplitKMaxFew : fill);
    const int want = nKs / kSplitMinTiles;
    c.k = want < 2 ? 2 : (want > kmax ? kmax : want);
  } else {
    c.k = nKs / 32 < 2 ? 2 : (nKs / 32 > kSplitKMax ? kSplitKMax : nKs / 32);
  }
  auto tiles_for = [&](int k) {
    const uint64_t per_tile = uint64_t(k) * 128 * (D + 2) * 4;
    const uint64_t t = budget / (uint64_t(B) * H * per_tile);
    return t > 64 ? 64 : int(t);
  };
  c.tiles = tiles_for(c.k);
  if (c.tiles < 2 && c.k > 2) { c.k = 2; c.tiles = tiles_for(2); }
  if (c.tiles > qtiles) c.tiles = qtiles;
  if (c.tiles <= 0) { c.tiles = 0; c.k = 1; }
  c.tiles *= 128 / c.rows;   // (the same rows, and the same scratch)
  return c;
}

// ---------------------------------------------------------------------------
// Shape of the launches without ids (and without a block map): how many query heads share a tile, how many rows a
// tile has, whether the key range of a tile is cut.
//   pack : the G query heads of one key head share their tiles: packed row r is query r / G of head r % G.  A tile
//          then meets the diagonal with 128 / G queries instead of 128 (less of it is masked), all the heads that
//          read the same K / V sit on one XCD, and a short query block fills tiles instead of padding them.  For long
//          blocks too, although the general set-up costs more: causal, 32 heads of D = 128, G = 4, forward and backward
//          273 -> 268 us at 2K rows, 9427 -> 9292 at 16K, forward alone 2029 -> 1978; window of 1024 1399 -> 1364;
//          4 x 16 heads of D = 64, G = 2, 2K rows, forward 60 -> 53, 4K rows without a mask 1253 -> 1251.
//   bm   : 128 rows, or 64 when 128-row tiles would leave CUs without a workgroup (the 64-row form splits every key
//          tile between two waves, see QTileCtx::halved).
//   dec  : few rows in all (packed sequences: in an average one): the form of fa_decode.hip, tiles of 32 packed rows.
//   split: chunks of the key range; only with FA_FLAG_SPLIT_KEYS, which gives the launch a workspace for them.
// ---------------------------------------------------------------------------
// The decode form also takes problems of at most this many 32-row tiles (one workgroup to a CU) whose rows see at most
// kDecKeys keys on average: four waves on different key blocks are a shorter chain than four on the same tile.  1 x 8
// heads x 1000 rows, causal 17.8 -> 15.3 us, 4 x 2 x 4 heads x 64 rows on 1000 keys 18.3 -> 14.8; with more tiles it takes a
// second round (336 of them: 11.2 -> 14.9), on longer ranges the 64-row form reads K and V half as often (32 heads x 128
// rows on 2000 keys 21.7 -> 24.2).  The backward's dq takes the same tiles, half of its waves without rows: a little slower
// where they are many, faster where they are few, and the sum of the kernels gains (64-row tiles : these, us: 8 heads x 1000
// rows 52.8 : 52.4, the backward of it 30.2 : 32.3; 8 heads x 512 33.3 : 31.2; 16 x 500 34.8 : 35.0; 64 rows on 1000 keys
// 44.3 : 40.0; 40 rows on 900 39.7 : 32.0).
// From there to two such tiles to a CU the forward takes the decode form with two workgroups to a CU, half the stages each,
// and the backward the tiles it would have without (us, 64-row form : this one): 32 heads on 8 x 333 rows 10.9 : 9.3, x 512
// 12.9 : 11.2, without a causal mask 11.0 : 10.4; 32 heads x 500 12.4 : 10.8; 16 x 1000 18.7 : 16.8, without a causal mask 20.6 :
// 21.2 (hence kDecKeys2); D = 64: 16 on 4 heads x 900 12.9 : 9.6, 4 x 16 x 256 7.0 : 6.6.  With more tiles a second round begins:
// 32 on 8 x 700 (704 tiles) 16.4 : 19.2.
constexpr int kDecTiles = kCUs, kDecTiles2 = 2 * kCUs, kDecKeys = 1024, kDecKeys2 = 768;
// A single tile to a head and more heads than CUs: two workgroups to a CU up to this many keys x D (us, one : two to a CU; 512
// tiles on 100 keys 12.0 : 7.2, 400 24.8 : 20.0, 900 41.6 : 37.9, D = 64 on 1000 28.5 : 24.4, 2048 tiles on 700 136 : 128; on 3000
// 136 : 139).  Packed sequences take the 64-row form there (256 on 128 keys 37 : 53).
constexpr int kDecShort = 1536 * 128;
// With packed sequences of at most 32 rows on average the decode form, one workgroup to a CU, is the better one for few
// tiles (a split key range adds to them) and, whatever their number, for long key ranges: 4 sequences x 8 key heads on 8192
// keys 44 us against 70 of 64-row tiles; 64 on 1100 keys 63 : 68, on 2048 112 : 122, on 8192 434 : 471, 256 on 2048 423 : 420
// (D = 64: 64 on 2048 129 : 124, 16 on 2048 44 : 37, on 8192 128 : 135).  Many short ranges want several workgroups to a CU:
// 64 on 512 keys 36 : 33, 4 key heads 37 : 27, 256 on 128 62 : 45, 1024 on 128 236 : 163; 600 sequences of 3 - 48 tokens, 8
// heads 165 : 69, 32 heads of D = 64 460 : 126.
constexpr int kDecSeqTiles = kCUs / 2, kDecSeqKeys = 1024;   // keys at D = 128; four times as many at 64
struct FwdCfg { int pack, bm, tiles, split; bool dec; int wpc; };
// Chunks for `wgs` tiles of `steps` steps each: the cheapest total by a model of rounds x (set-up + steps of a chunk)
// + merging, in units of one step; `slots` workgroups run at a time.  A chunk keeps at least `min_steps` steps.
inline int pick_split(int64_t wgs, int steps, int slots, float setup, float merge, int min_steps) {
  int best = 1;
  float best_t = 1e30f;
  for (int s = 1; s <= kSplitKMaxFew && (s == 1 || steps / s >= min_steps); ++s) {
    const int64_t rounds = (wgs * s + slots - 1) / slots;
    // a launch that does not fill the chip streams faster per workgroup, but not without bound
    const float fill = rounds > 1 ? 1.f : float(wgs * s) / slots;
    const float step = fill > 0.4f ? fill : 0.4f;
    const float t = rounds * (setup + float((steps + s - 1) / s) * step) + (s > 1 ? merge : 0.f);
    if (t < best_t * 0.97f) { best_t = t; best = s; }
  }
  return best;
}
// Query heads that share a tile.  The kernels count packed rows in int, up to the end of the last tile: none share where
// that would not hold.  (A little further, at 2^31 rows of all heads, a launch has more work-items than a grid can: an error.)
inline int shared_heads(const fa_params* p) {
  const int G = p->H / p->Hk;
  return int64_t(p->M) * G <= 0x7fffffff - 256 ? G : 1;
}
inline FwdCfg fwd_config(const fa_params* p, bool fwd = true) {   // fwd: for the forward (the backward may take other tiles)
  FwdCfg c = {1, 128, 0, 1, false, 1};
  if (p->score_mode == FA_SCORE_MODE3_PACKED) {
    // the host knows the totals only: 32-row tiles when an average sequence fills no more
    c.pack = shared_heads(p);
    const int64_t nseq = p->nseq > 0 ? p->nseq : 1, rows = int64_t(p->M) * c.pack, avg = rows / nseq;
    c.dec = avg <= 32 && (nseq * (p->H / c.pack) <= kDecSeqTiles || p->N / nseq * p->D * p->D >= int64_t(kDecSeqKeys) * 128 * 128);
    c.bm = c.dec ? 32 : (avg <= 64 || (rows / 128 + p->nseq) * (p->H / c.pack) < kCUs ? 64 : 128);
    return c;
  }
  if (p->score_mode == FA_SCORE_MODE2_BLOCK && p->dtype != FA_DTYPE_FP32) {
    c.bm = block_rows(p->B, p->H, p->M, p->D);
    c.tiles = (p->M + c.bm - 1) / c.bm;
    return c;
  }
  if (p->score_mode != FA_SCORE_MODE0_NOPE || p->dtype == FA_DTYPE_FP32) { c.tiles = (p->M + 127) / 128; return c; }
  c.pack = shared_heads(p);
  const int64_t rows = int64_t(p->M) * c.pack, bh = int64_t(p->B) * (p->H / c.pack);
  const int nk = p->window > 0 && p->causal && p->window < p->N - p->M ? p->window + p->M : p->N;   // keys a tile can see
  const int seen = p->causal && p->N >= p->M ? nk - (nk == p->N ? p->M / 2 : 0) : nk;   // keys a row sees on average
  if (rows <= 32 || (bh * ((rows + 31) / 32) <= kDecTiles && seen <= kDecKeys)) {
    c.dec = true; c.bm = 32; c.tiles = int((rows + 31) / 32);
    // a step: four waves x 32 keys.  64 KB at D = 128 take a CU 3 us at the rate the whole card reads; setting a
    // workgroup up takes about as long, handing the result over and merging one and a half steps
    const float rel = 128.f / p->D;
    if (p->flags & FA_FLAG_SPLIT_KEYS) c.split = pick_split(bh * c.tiles, (nk + 127) / 128, kCUs, 1.2f * rel, 1.5f * rel, 2);
    if (c.split == 1 && bh * c.tiles > kCUs && int64_t(nk) * p->D <= kDecShort) c.wpc = 2;
    return c;
  }
  c.tiles = int((rows + 127) / 128);
  // 64-row tiles where 128-row ones leave CUs idle, and up to nearly two of those to a CU where a causal mask makes them unequal: all are resident
  // at once, and the launch waits for the longest.  64 rows : 128 by the tiles of 128 rows, geometric mean [smallest, largest]:
  //                                                    to 320             to 384             to 448             to 512
  //   D = 128, 2500 rows and more, forward     0.87 [0.85, 0.89]  0.89 [0.86, 0.91]  0.91 [0.88, 0.95]  0.97 [0.83, 1.12]
  //                   forward and backward     0.90 [0.87, 0.93]  0.93 [0.90, 0.96]  0.95 [0.94, 0.98]  0.98 [0.89, 1.04]
  //            1024 to 2048 rows, forward      0.96 [0.88, 1.01]  1.07 [1.05, 1.11]  1.14 [1.02, 1.20]  1.06 [1.05, 1.07]
  //                   forward and backward     0.94 [0.91, 0.97]  1.01 [1.00, 1.01]  1.03 [1.01, 1.04]  0.99 [0.99, 1.00]
  //   D = 64,  2500 rows and more, forward     0.85 [0.82, 0.89]  0.87 [0.84, 0.90]  0.88 [0.82, 0.90]  0.87 [0.81, 0.92], to 576 0.87
  //              backward, as many keys        0.95 [0.82, 1.04]  0.92 [0.84, 1.03]  0.97 [0.91, 1.07]  0.92 [0.90, 0.95]
  //              backward, up to a quarter more 1.00 [0.98, 1.01] 0.98 [0.93, 1.03]  1.05 [1.04, 1.07]  1.03 [0.92, 1.10]
  //            1024 to 2048 rows, forward      0.92 [0.89, 0.96]  0.85 [0.83, 0.88]  0.95 [0.91, 1.02]  0.95 [0.95, 0.95]
  //                             backward       1.03 [0.94, 1.14]  0.96 [0.91, 1.09]  1.00 [0.94, 1.11]  0.97 [0.97, 0.97]
  // (1 x 4 x 12000, D = 128, forward and backward 747 -> 680 us.)  What loses to 512 at D = 128 are heads that the XCDs do not share evenly (5 x 12000 rows on
  // 13200 keys 1044 -> 1087, 7 x 9000 682 -> 702).  Equal tiles
  // lose what a 64-row tile costs more: no mask, D = 128 1.20 - 1.31; windows of up to half of the keys, D = 128 1.06 - 1.43, D = 64 from 448 on 0.94 - 1.24;
  // prefixes, forward and backward, of a quarter of the keys 0.87 - 0.97 (D = 64 to 1.01), of half 1.00 - 1.08 (0.92 - 1.05), of three quarters 1.03 - 1.14;
  // half as many keys again as rows 0.94 - 0.99, forward alone 0.87 - 1.03.
  const int64_t wgs = c.tiles * bh;
  int64_t low = kCUs - 1;
  if (p->causal && (p->window <= 0 || p->window >= p->N) && p->prefix <= p->N / 4 && p->N - p->M <= p->M / 4) {
    if (p->M >= 2500) low = p->D > 64 ? kCUs * 7 / 4 : fwd || p->N - p->M <= p->M / 16 ? kCUs * 9 / 4 : kCUs * 3 / 2;
    else if (p->M >= 1024 && p->D > 64) low = kCUs * 5 / 4;
    else if (p->M >= 1024 && fwd) low = kCUs * 7 / 4;
  }
  if (wgs <= low) { c.bm = 64; c.tiles = int((rows + 63) / 64); }
  // a step: one 64-key tile; two workgroups to a CU
  if ((p->flags & FA_FLAG_SPLIT_KEYS) && c.tiles * bh < 2 * kCUs)
    c.split = pick_split(c.tiles * bh, (nk + 63) / 64, 2 * kCUs, 3.f, 4.f, 8);
  if (fwd && c.split == 1 && bh * ((rows + 31) / 32) <= kDecTiles2 && seen <= kDecKeys2) { c.dec = true; c.bm = 32; c.tiles = int((rows + 31) / 32); c.wpc = 2; }
  return c;
}

// Packed sequences (FA_SCORE_MODE3_PACKED): one entry of the tile tables the plan kernel writes (fa_seq.hip).
struct SeqTile {
  int q0, M, k0, N;      // the sequence's first query row and its rows, its first key and its keys
  int gap;               // row i of the sequence has its diagonal at key gap + i
  int tile;              // query tile (of bm packed rows) or key tile of the sequence
  int chunk, nchunk;     // share of the key range (query tiles only)
  int cnt, part;         // arrival counter and first partial result of a split tile, per head: times nHp, plus the head
  int pad[6];
};
struct SeqHdr { int nq, nk, pad[2]; };   // entries in use

// Compile-time integer handed to a generic lambda.
template <int V> struct IntC { static constexpr int value = V; };

constexpr int kPairSpinDefault = 1 << 14;

// Clock stamps per workgroup, for the measurement build only (compiled with -DFA_TRACE into a library of its
// own, libflash_mi355_trace.so, read by `bench.py --wg-trace`).  A traced kernel keeps eight 64-bit words per
// workgroup in a device array (wall clock, 100 MHz) that fa_trace_read copies out.  In the product build the
// macros expand to nothing.
#ifdef FA_TRACE
constexpr int kTraceWgs = 65536;
#define FA_TRACE_ARRAY(name) __device__ long long name[8 * fa::kTraceWgs]
#define FA_STAMP(buf, i, v) do { if (threadIdx.x == 0 && blockIdx.x < fa::kTraceWgs) buf[blockIdx.x * 8 + (i)] = (long long)(v); } while (0)
#define FA_CLOCK() wall_clock64()
#define FA_TRACE_ONLY(...) __VA_ARGS__
#else
#define FA_STAMP(buf, i, v) do {} while (0)
#define FA_CLOCK() 0
#define FA_TRACE_ONLY(...)
#endif

// Key position of a row's diagonal as the kernels use it: at least -1 (the row sees nothing), and
// small enough that position + window never overflows.
constexpr int kPosMax = 0x3fffffff;
FA_HD int clamp_pos(int v) { return v < -1 ? -1 : (v > kPosMax ? kPosMax : v); }

struct bf16_t {};
struct fp16_t {};

template <typename Tag> struct Elem;

template <> struct Elem<bf16_t> {
  typedef __bf16 scalar;
  typedef bf16x8 vec8;
  typedef bf16x4 vec4;
  typedef bf16x2 vec2;
  static FA_DEV f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static FA_DEV vec4 lds_tr(const void* p) {
    return __builtin_bit_cast(vec4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p)));
  }
  static FA_DEV vec2 cvt2(float x, float y) {
    f32x2 t = {x, y};
    return __builtin_convertvector(t, vec2);
  }
};

template <> struct Elem<fp16_t> {
  typedef _Float16 scalar;
  typedef f16x8 vec8;
  typedef f16x4 vec4;
  typedef f16x2 vec2;
  static FA_DEV f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static FA_DEV vec4 lds_tr(const void* p) {
    return __builtin_bit_cast(vec4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p)));
  }
  static FA_DEV vec2 cvt2(float x, float y) {
    f32x2 t = {x, y};
    return __builtin_convertvector(t, vec2);
  }
};

// Sign flip of 8 packed 16-bit floats (exact for both bf16 and fp16).
template <typename E>
FA_DEV typename E::vec8 neg8(typename E::vec8 x) {
  i32x4 u = __builtin_bit_cast(i32x4, x);
  u ^= (int)0x80008000;
  return __builtin_bit_cast(typename E::vec8, u);
}

// Exchange between lane l and lane l ^ 32: returns the partner's value.
FA_DEV float xhalf(float x) {
  unsigned u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  // r[0] = {lo, lo}, r[1] = {hi, hi}: the partner of a low lane is r[1], of a high lane r[0]
  unsigned lo = r[0], hi = r[1];
  return __uint_as_float((threadIdx.x & 32) ? lo : hi);
}
FA_DEV float xhalf_max(float x) {
  unsigned u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
FA_DEV float xhalf_sum(float x) {
  unsigned u = __float_as_uint(x);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Elements e, e + 1 of packed fp16 values times fp32 ones: a multiply-add with zero is one instruction that converts on the way
// (v_fma_mix_f32; a product alone is two).  Left to the compiler, since the fp32 operands are accumulators of a matrix product: it
// waits until that product can be read, which it does not do for inline assembly.
FA_DEV void mul_f16_f32(f16x8 p, const int e, float x0, float x1, float& y0, float& y1) {
  y0 = __builtin_fmaf(float(p[e]), x0, 0.f);
  y1 = __builtin_fmaf(float(p[e + 1]), x1, 0.f);
}

// Eight products of 16-bit elements, added up in order.  Not to be contracted: for fp16 the compiler makes two-element dot
// products of some such sums and not of others, which round differently, and a delta is to have the same bits wherever it is formed.
template <typename V>
FA_DEV float dot8(const V& x, const V& y) {
#pragma clang fp contract(off)
  float s = 0.f;
#pragma unroll
  for (int t = 0; t < 8; ++t) s = __builtin_fmaf(float(x[t]), float(y[t]), s);
  return s;
}

// Make a 16-byte value loaded from global memory "used" right here.  The compiler waits for a
// load at the first use of its result; for operands that are loaded once and first used inside
// the tile loop that wait (s_waitcnt vmcnt) would sit in the loop, where it also waits for the
// asynchronous tile loads issued just before it -- the loads it is meant to overlap with.
template <typename V>
FA_DEV void settle(V& x) {
  i32x4 u = __builtin_bit_cast(i32x4, x);
  asm volatile("" : "+v"(u));
  x = __builtin_bit_cast(V, u);
}
FA_DEV void settle(float& x) { asm volatile("" : "+v"(x)); }
FA_DEV void settle(int& x) { asm volatile("" : "+v"(x)); }

// Issue priority of a wave while it feeds the matrix pipe.  Two waves share a SIMD; the one that has MFMAs to issue goes
// first, and the other's softmax fills the slots in between: 0.5 - 3 % of the kernels' times.
FA_DEV void mfma_phase() { __builtin_amdgcn_s_setprio(1); }
FA_DEV void vector_phase() { __builtin_amdgcn_s_setprio(0); }

FA_DEV float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
FA_DEV float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// ---------------------------------------------------------------------------
// Mask engine, element level.  keep(i, j) of the reference:
//   tail   : j < N (and i < M at the store)             flash_triton.py:103-105
//   causal : gap + i >= j, gap = max(0, N - M)          flash_triton.py:107
//   doc    : eq_i >= 0 || eq_i == ek_j                  flash_triton.py:114
// ---------------------------------------------------------------------------
//   window : j > gap + i - win (win = 0x3fffffff: off)    sliding window, causal only
//   prefix : the causal term also holds for j <= pfx_m1   prefix-LM (pfx_m1 = -1: off)
//   pos_i  : key position of row i's diagonal: gap + i, or the caller's per-row position (fa_params.qpos)
template <bool CAUSAL, bool DOC>
FA_DEV bool keep_elem(int pos_i, int j, int N, int eq_i, int ek_j, int win, int pfx_m1) {
  bool keep = j < N;
  if (CAUSAL) keep = keep && ((pos_i >= j) || (j <= pfx_m1)) && (j > pos_i - win);
  if (DOC) keep = keep && ((eq_i >= 0) || (eq_i == ek_j));
  return keep;
}

// ---------------------------------------------------------------------------
// Mask plan.  With document ids the query rows of one (batch, head) are split
// into LOCAL rows (eq < 0: see only keys with the same id) and GLOBAL rows
// (eq >= 0: see every key), each group kept in ascending row order:
//   perm[0 .. nL)            local rows            (padded with -1 up to nLp,
//   perm[nLp .. nLp + nG)    global rows            nLp = nL rounded up to kPermAlign)
// Query-side tiles are tiles of this permuted order, so a tile is either all
// local (it only needs the key tiles whose id interval meets its own) or all
// global (no doc test at all, plain causal structure).  Keys stay in natural
// order.  One IdSummary describes 64 consecutive entries of either side.
// ---------------------------------------------------------------------------
struct IdSummary {
  int lo, hi;      // min / max id: query side over local rows (lo > hi if none), key side over all keys
  int glob;        // query side: 1 if the tile holds global rows
  int rmin, rmax;  // query side: smallest / largest diagonal position (ppos) of the tile's rows (rmax = -1 if empty);
                   // key side: first / last key of the tile
  int nvalid;      // query side: rows of the tile that exist
  int kfirst, klast;  // query side: first / last key tile (of 64 keys) the rows can need (klast < kfirst: none)
};

struct QHeader {
  int nL, nG, nLp, nT128;  // nT128: 128-row tiles of the permuted order that hold rows
  int k0;                  // first key tile (of 64) that a local row can need (0x7fffffff: none can need any):
                           // the keys before it are seen by global rows only
  int pad[3];
};

// A tile pair can hold a kept element only if a global query row exists or the
// local-id interval of the query rows meets the id interval of the keys.
FA_DEV bool doc_may_keep(int q_lo, int q_hi, int q_glob, int k_lo, int k_hi) {
  return q_glob || (q_lo <= k_hi && k_lo <= q_hi);
}
// Every (row, key) pair of the tile pair passes the doc test.
FA_DEV bool doc_all_keep(int q_lo, int q_hi, int k_lo, int k_hi) {
  // no local row at all, or one local id shared by every key
  return (q_lo > q_hi) || (q_lo == q_hi && k_lo == k_hi && q_lo == k_lo);
}

// Key columns that no local row can need (QHeader::k0) are seen by the global rows only.  When those rows
// are few -- at most kGcolTilesMax tiles of 64, over all query heads of a group -- a kernel of its own takes
// these columns: it keeps the rows' Q / dO tiles in LDS and streams the keys (fa_dkdv_cols.h), instead
// of one workgroup per 64 keys that sets up a tile stream for one or two tiles.
constexpr int kGcolTilesMax = 2;
constexpr int kGcolMinGap = 512;   // keys without a diagonal of their own from which the form is put into the launch

// Kernel-side view of the operands (built on the host from fa_params).
struct KArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  float* lse;
  const void* dout;
  void* dq;
  void* dk;
  void* dv;
  float* delta;
  const int* eq32;        // [B, Hq', Mp]   ids in natural row order
  const int* ek32;        // [B, Hk', Np]
  const int* perm;        // [B, Hq', Pp]   permuted order -> original row (or -1)
  const int* peq;         // [B, Hq', Pp]   id of that row
  const int* ppos;        // [B, Hq', Pp]   key position of that row's diagonal (gap + row, or the caller's qpos), -1 for padding
  const int* qpos;        // the caller's per-row positions [B, M] in natural order, or null (mask dump)
  int64_t qp_bs;
  const QHeader* qhdr;    // [B, Hq']
  const IdSummary* qsum;  // [B, Hq', nQs]  per 64 entries of the permuted order
  const IdSummary* ksum;  // [B, Hk', nKs]  per 64 keys
  // split-key scratch of the global-row tiles, see SplitCfg: per (b, h, global tile g)
  int split_k, split_tiles;
  int* sk_cnt;            // [B, H, split_tiles]                  arrival counters (zero between kernels)
  float* sk_ml;           // [B, H, split_tiles, split_k, bm, 2]  per row: reference point, row sum
  float* sk_o;            // [B, H, split_tiles, split_k, bm, D]  per row: unnormalised partial result
  int64_t q_bs, q_hs, q_rs;
  int64_t k_bs, k_hs, k_rs;
  int64_t v_bs, v_hs, v_rs;
  int64_t o_bs, o_hs, o_rs;
  int64_t do_bs, do_hs, do_rs;
  int64_t dq_bs, dq_hs, dq_rs;
  int64_t dk_bs, dk_hs, dk_rs;
  int64_t dv_bs, dv_hs, dv_rs;
  int64_t eq_bs, eq_hs;   // strides of eq32 (head stride 0 when shared)
  int64_t ek_bs, ek_hs;
  int64_t pm_bs, pm_hs;   // strides of perm
  int64_t qh_bs, qh_hs;   // strides of qhdr in entries
  int64_t qs_bs, qs_hs;   // strides of qsum in entries
  int64_t ks_bs, ks_hs;
  int B, H, Hk, G, M, N, gap;
  int win;      // sliding window: a row sees keys j > gap + i - win (0x3fffffff: no window)
  int pfx_m1;   // prefix-LM: keys j <= pfx_m1 are seen by every row (-1: no prefix)
  int Pp;                 // entries of the permuted order per (b, h)
  int nQs, nKs;           // summary entries per (b, h)
  // the launches without ids: see FwdCfg
  int pack, nHp;          // query heads per tile, H / pack
  int bm, nTiles;         // rows per query tile (also with ids), tiles per (batch, head group)
  int dsplit;             // chunks of the key range of every tile
  int wpc;                // the decode form: workgroups to a CU
  // packed sequences: tables of the plan (null otherwise) and their capacities
  const SeqHdr* shdr;
  const SeqTile* qtab;
  const SeqTile* ktab;
  int nQent, nKent;
  int dq_delta;           // the dq kernel computes delta from O and dO itself and stores it
  int pair_spin;          // dk/dv, role-split form: polls of the pair flag before the gradient wave gives up
  // block mask (FA_SCORE_MODE2_BLOCK): bytes [B, H, nBr, nBc] per 64 x 64 block of (row, key) pairs, or null
  const unsigned char* bmask;
  int64_t bm_bs, bm_hs, bm_rs;
  int nBr, nBc;
  float scale;            // sm_scale
  float scale_log2e;      // sm_scale * log2(e)
};

// The kernel arguments read again, where they are needed late: left alone, the compiler loads every argument at the
// top of the kernel, and the ones only the end uses fill scalar registers (and, spilled, vector lanes that the tile loop
// reads back) all the way through.
typedef const __attribute__((address_space(4))) KArgs LateArgs;
FA_DEV LateArgs& late_args() {
  LateArgs* p = (LateArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}

// Workspace layout shared by host and device code.
struct WsLayout {
  int Hq1, Hk1;           // heads stored for eq / ek (1 when the head stride is 0)
  int Mp, Np;             // M, N rounded up to kSumRows
  int Pp;                 // length of the permuted order
  int nQs, nKs;
  int nCh;                // row chunks of the partition kernels
  int nSk;                // arrival counters
  uint64_t low_bytes;     // what they take more than one to 128 rows would
  uint64_t off_eq32, off_ek32, off_perm, off_peq, off_ppos, off_cnt, off_qhdr, off_qsum, off_ksum;  // bytes
  uint64_t off_sk_cnt, off_sk_ml, off_sk_o, total;
  uint64_t plan_bytes;   // leading part that carries state from the plan to the kernels; the rest is scratch
  SplitCfg split;        // split of long key ranges this layout has scratch for
};

// split_budget: bytes the scratch of the split key ranges (sk_ml, sk_o) may take
inline WsLayout ws_layout(const fa_params* p, uint64_t split_budget = kSplitScratchBudget) {
  WsLayout w;
  w.Hq1 = (p->eq_stride[1] == 0) ? 1 : p->H;
  w.Hk1 = (p->ek_stride[1] == 0) ? 1 : p->H;
  w.Mp = (p->M + kSumRows - 1) / kSumRows * kSumRows;
  w.nKs = (p->N + kSumRows - 1) / kSumRows;
  w.Np = w.nKs * kSumRows;
  w.Pp = (p->M + kPermAlign - 1) / kPermAlign * kPermAlign + kPermAlign;
  w.nQs = w.Pp / kSumRows;
  uint64_t o = 0;
  auto take = [&](uint64_t bytes) { uint64_t r = o; o += (bytes + 255) & ~uint64_t(255); return r; };
  w.off_eq32 = take(uint64_t(p->B) * w.Hq1 * w.Mp * 4);
  w.off_ek32 = take(uint64_t(p->B) * w.Hk1 * w.Np * 4);
  w.off_perm = take(uint64_t(p->B) * w.Hq1 * w.Pp * 4);
  w.off_peq = take(uint64_t(p->B) * w.Hq1 * w.Pp * 4);
  w.off_ppos = take(uint64_t(p->B) * w.Hq1 * w.Pp * 4);
  w.nCh = (w.Mp + 1023) / 1024;
  w.off_cnt = take(uint64_t(p->B) * w.Hq1 * w.nCh * 4);
  w.off_qhdr = take(uint64_t(p->B) * w.Hq1 * sizeof(QHeader));
  w.off_qsum = take(uint64_t(p->B) * w.Hq1 * w.nQs * sizeof(IdSummary));
  w.off_ksum = take(uint64_t(p->B) * w.Hk1 * w.nKs * sizeof(IdSummary));
  // scratch of the split tiles: only when a key range can be long enough to be cut
  const SplitCfg sc = split_config(p->B, p->H, p->M, p->N, p->D, p->qpos != nullptr, split_budget);
  w.split = sc;
  const uint64_t nsk = uint64_t(p->B) * p->H * sc.tiles;
  w.nSk = int(nsk) * (sc.rows / doc_rows(p->B, p->H, p->M, p->D));   // as many with qpos as without: the layout does not depend on it
  w.off_sk_cnt = take(uint64_t(w.nSk) * 4);
  w.low_bytes = (o - w.off_sk_cnt) - ((nsk * sc.rows / 128 * 4 + 255) & ~uint64_t(255));
  w.plan_bytes = o;      // the counters (zeroed by the plan, left at zero by every kernel) are state
  w.off_sk_ml = take(nsk * sc.k * sc.rows * 2 * 4);
  w.off_sk_o = take(nsk * sc.k * sc.rows * uint64_t(p->D) * 4);
  w.total = o;
  return w;
}

// fa_fwd_static takes the problems whose layout fits FA_STATIC_WS_BYTES with one arrival counter to 128 rows; 64-row tiles have two, which lie in a margin of
// the array (doc_rows: at most 384 tiles of 128 rows and one more to each of 96 (batch, head) pairs).
constexpr uint64_t kStaticMargin = 4096;
inline bool fits_static(const WsLayout& w) { return w.total - w.low_bytes <= FA_STATIC_WS_BYTES && w.low_bytes <= kStaticMargin; }

// Layouts without a mask plan.  Mode 0 with FA_FLAG_SPLIT_KEYS: arrival counters (the part called plan) and partial
// results.  Packed sequences: header, tile tables, counters, and partial results.
struct TabLayout {
  uint64_t off_hdr, off_q, off_k, off_spill, off_cnt, plan_bytes, off_ml, off_o, total;
  int nQ, nK, nCnt, nPart;   // entries per head group
};
// Keys per entry of the key-tile table: the 64-key role-split form at D = 128 (sequences are short), 128 keys below.
constexpr int kSeqKeyTile = 64;
FA_HD int seq_key_tile(int D) { return D > 64 ? kSeqKeyTile : 128; }
// Workgroups the split key ranges of a packed batch aim at.  A split tile pays for its partial results (64 KB per chunk
// of 128 rows at D = 128, written and read again), so they are cut to fill the chip (two workgroups to a CU) and,
// once there are tiles enough for that, only where one is several times as long as the rest.  Swept over 64 .. 2048:
// 32 sequences of up to 128 queries on 500 - 3500 keys (720 tiles) 105 / 107 / 118 / 130 / 163 us at 64 / 128 / 448 /
// 768 / 1536, one of 256 queries on 8000 keys (64 tiles) 105 / 68 / 59 / 78 / 137.
constexpr int kSeqTargetWgs = 448, kSeqFullWgs = 400, kSeqTargetFull = 128;
inline TabLayout tab_layout(const fa_params* p, const FwdCfg& c) {
  TabLayout w = {};
  uint64_t o = 0;
  auto take = [&](uint64_t bytes) { uint64_t r = o; o += (bytes + 255) & ~uint64_t(255); return r; };
  const int nh = p->H / c.pack;
  if (p->score_mode == FA_SCORE_MODE0_NOPE) {
    if (c.split <= 1) return w;
    w.nCnt = p->B * c.tiles; w.nPart = w.nCnt * c.split;
    w.off_cnt = take(uint64_t(w.nCnt) * nh * 4);
  } else {
    w.off_hdr = take(sizeof(SeqHdr));
    const int spare = kSeqTargetWgs / nh + 1;
    w.nQ = int((int64_t(p->M) * c.pack) / c.bm) + p->nseq + 1 + spare;
    w.nK = p->N / seq_key_tile(p->D) + p->nseq + 1;
    w.nCnt = spare; w.nPart = 2 * spare;
    w.off_q = take(uint64_t(w.nQ) * sizeof(SeqTile));
    w.off_k = take(uint64_t(w.nK) * sizeof(SeqTile));
    w.off_spill = take(p->nseq < 8000 ? 0 : uint64_t(p->nseq + 2) * 2 * 4);   // tile offsets of very many sequences (fa_seq.hip)
    w.off_cnt = take(uint64_t(w.nCnt) * nh * 4);
  }
  w.plan_bytes = o;
  w.off_ml = take(uint64_t(w.nPart) * nh * c.bm * 2 * 4);
  w.off_o = take(uint64_t(w.nPart) * nh * c.bm * uint64_t(p->D) * 4);
  w.total = o;
  return w;
}

// Raise the dynamic LDS limit of a kernel once per device (the attribute is per device and per
// kernel; a process may drive several GPUs).  `done` is the caller's per-kernel record.
template <typename K>
static int allow_lds(K kern, size_t lds, bool (&done)[64]) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64 || !done[dev]) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    if (dev >= 0 && dev < 64) done[dev] = true;
  }
  return 0;
}

// Launchers implemented one per translation unit; each returns a hipError_t as int.
int launch_fwd(const KArgs& a, int dtype, int D, bool causal, bool doc, hipStream_t s);
int launch_decode(const KArgs& a, int dtype, int D, bool causal, hipStream_t s);   // at most 32 packed rows, or packed sequences with 32-row tiles
int launch_zero_counters(int* cnt, int n, hipStream_t s);
int launch_seq_plan(const fa_params* p, const FwdCfg& c, const TabLayout& w, hipStream_t s);
int launch_bwd_delta(const KArgs& a, int dtype, int D, hipStream_t s);
int launch_bwd_dq(const KArgs& a, int dtype, int D, bool causal, bool doc, hipStream_t s);
int launch_bwd_dkdv(const KArgs& a, int dtype, int D, bool causal, bool doc, hipStream_t s);
int launch_dkdv_pipe(const KArgs& a, int dtype, bool causal, hipStream_t s);   // long tile streams without ids at D = 128 (fa_dkdv_pipe.hip)
bool bwd_in_one(const KArgs& a, int D, bool causal, bool doc);
int dkdv_form(const KArgs& a, int D, bool causal, bool doc, bool both);   // FA_FORM_* of fa_bwd_dkdv.hip (the problems that fa_bwd_small.hip leaves), 16-bit elements
int launch_bwd_both(const KArgs& a, int dtype, int D, bool causal, bool doc, hipStream_t s);   // dq and dk/dv, delta read by both
int read_pair_wait_expired(unsigned long long* n);   // expired pair waits of the dk/dv kernel on the current device (synchronises)
#ifdef FA_TRACE
int trace_read_fwd(long long* host, int n);
int trace_read_dq(long long* host, int n);
int trace_read_dkdv(long long* host, int n);
int trace_read_pipe(long long* host, int n);
int trace_read_small(long long* host, int n);
#endif
// the same four for fp32 tensors (fa_f32.hip)
int launch_fwd_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s);
int launch_bwd_delta_f32(const KArgs& a, int D, hipStream_t s);
int launch_bwd_dq_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s);
int launch_bwd_dkdv_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s);
bool bwd_f32_in_one(const KArgs& a, int D, bool causal);
int bwd_f32_shapes(const KArgs& a, int D, bool causal, bool doc);   // of dq's and dk/dv's workgroups, as FA_FORM_FP32 carries them
int launch_bwd_f32(const KArgs& a, int D, bool causal, bool doc, hipStream_t s);
// keys that a row sees at all: workgroups of the others end at once
inline int seen_keys(const KArgs& a, bool causal) { return causal && a.win < 0x3fffffff ? int(std::min<int64_t>(a.N, int64_t(a.M) + a.win + a.pfx_m1 + 1)) : a.N; }
// problems that leave CUs idle (fa_bwd_small.hip): whether dk/dv takes its form there, and with dq in one launch or by itself
bool bwd_small(const KArgs& a, int D, bool causal, bool doc);
int launch_bwd_small(const KArgs& a, int dtype, int D, bool causal, bool doc, bool both, hipStream_t s);
int launch_mask_plan(const fa_params* p, const WsLayout& w, hipStream_t s);
int launch_mask_dump(const KArgs& a, bool causal, bool doc, uint8_t* out, hipStream_t s);

}  // namespace fa
