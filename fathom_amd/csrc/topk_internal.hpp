// Selection machinery shared by the standalone top-k and the fused scan+top-k.
//
// Exact top-kk of a row in four steps:
//   select    from a sample of the row (tiles of 2048 tokens, every S-th
//             tile): T_lo, a lower bound of the sample's kk-th largest key,
//             and T_hi, a lower bound of its r-th largest, r = about
//             kAlphaX2 / 2 * kk * (sample size / n).  A sample is a subset of the
//             row, so T_lo never exceeds the row's kk-th largest key; T_hi is
//             a guess that about kAlphaX2 / 2 * kk elements of the row reach;
//   filter    elements with key >= T_hi become the row's candidates.  If there
//             are at least kk, T_hi <= the row's kk-th largest key and they
//             hold the whole top kk;
//   fallback  rows with fewer than kk candidates (a sample that was not
//             representative) are filtered again with T_lo, into the same
//             buffer under a second count; other rows skip the pass (the
//             fused scan's finalize workgroup rescans such a row itself);
//   finalize  one workgroup per row selects the exact kk largest candidates by
//             K64 = key << 32 | (0xFFFFFFFF - index) and writes them sorted.
// Exactness never depends on the sample: a poor sample only costs a fallback
// pass or more candidates (the buffer holds a whole row, so it cannot overflow).
//
// Candidates are kept in one of two layouts:
//   list      (score-row filter) appended at a row counter: cand[0, count);
//   regions   (fused scan) region r of a row holds the candidates of tokens
//             [r * kRegTok, (r + 1) * kRegTok) -- one wave's blocks -- at
//             cand[r * kRegTok, r * kRegTok + rc[r]), written with the count
//             rc[r] by that wave alone: no atomics.  A pass writes every
//             region of a row it does not skip.
#pragma once
#include "common.hpp"

namespace fathom {

constexpr int64_t kTileTok = 2048;  // tokens per sample tile of the score-row top-k
constexpr int64_t kRegTok = 1024;   // tokens per candidate region and sample tile of the fused scan (one wave-tile)
constexpr int64_t kMaxSample = 65536; // sampled keys per row (held in registers by select)

// Largest kk of the sampled chains (sample -> select -> filter -> finalize, the
// fused scan's), and of the selections that sort once.
constexpr int64_t kSelMaxK = 2048;
constexpr int64_t kRankListMax = 8192;

// expected first-pass candidates per row, in units of kk: kAlphaX2 / 2
constexpr int64_t kAlphaX2 = 5;

// Rows up to this length have their group maxima held two per thread (longer ones,
// up to kGmaxSelectMax, eight), and are kept in the drop-in order by the fused scan.
constexpr int64_t kRowSelectMax = 32768;

// Longest rows that the fused scan + top-k selects from its scores' 16-token group
// maxima, in two launches (the plan, where asked for, made in the scan) instead of
// the sampled chain's four: the scores cost 4.25 bytes per token and head of
// stores, the chain its latency-bound launches.  Scan + top-k, us, chain against
// group maxima: 8 x 4 heads of 40000 tokens 34.5; 23.0, of 131072 35.7; 30.4, of
// 262144 36.3; 43.1; 32 x 4 heads of 65536 57.5; 43.1; 8 x 7 heads of 131072 63; 51;
// 16 x 8 heads of 131072 65; 52; 2 x 4 heads of 262144 31.6; 30.4.
constexpr int64_t kGmaxSelectMax = 131072;
constexpr int64_t kGmaxWideMax = 524288;  // and of the wide selection (kk above kSelMaxK)

// Tokens per group of the group maxima that the fused scan's short-row pass
// writes beside its scores (one lane's 16 tokens of a block).
constexpr int64_t kGroupTok = 16;

// The rows selected by one workgroup each: from the group maxima, or (up to
// kRowSelectMax tokens, few groups per selected key) read whole.  Above kSelMaxK
// the groups must number at least 5/4 kk and their list must fit; the others take
// the chain and the wide selection.  sink_local_topk of 32 rows, us, chain and wide
// selection against this one: n = 8192, k = 4096 107; 17.5, 30000, 4096 104; 29, 32768,
// 8000 136; 37, 100000, 4096 82; 47, 300007, 4096 104; 71, 524288, 4096 91; 72; beyond
// the limits 1048576, 4096 98; 97 and 300007, 8192 121; 116 (198 on rows whose list
// does not fit).  Those are independent scores; neighbours that score alike (correlation
// lengths of 16 and 256 tokens) cost both sides more: 100000, 4096 88; 74 and 126; 72,
// 300007, 4096 99; 94 and 146; 87, 500000, 5000 96; 110 and 157; 102, 500000, 6136 102; 123
// and 190; 116.
inline bool group_select_takes(int64_t n, int64_t kk) {
  if (kk <= kSelMaxK) return n <= kGmaxSelectMax;
  if (n <= kRowSelectMax) return kk <= kRankListMax;
  return n <= kGmaxWideMax && kk <= 6144 && 4 * cdiv(n, kGroupTok) >= 5 * kk;
}

// The fused scan's own score order, rows held in whole blocks (so no store is
// split or unaligned, whatever n is): [bh][head][token], the drop-in order
// padded, or -- more than four heads, long rows -- per bh and tile of 16 blocks
// [16 token quads of a block][head][block][4].  A store instruction of the scan is
// one quad of every block; the drop-in order leaves 16-byte pieces 256 bytes
// apart, the quad order runs of 256 bytes per head, but a group's 64 bytes then
// lie in four lines when the selection reads them.  The last tile's runs are as
// long as its blocks.  Scan + selection, us (drop-in; quad): 8 x 7 heads of 131072
// tokens 54; 51, 16 x 8 heads 71; 53, 8 x 7 heads of 20000 tokens 26.1; 28.0.  Up to
// four heads store 8-byte pairs per lane: 8 x 4 heads of 131072 tokens 30.3; 32.8,
// and of 131071 tokens 30.3 padded against 37.1 unpadded.
__host__ __device__ inline int64_t tile_score_floats(int64_t n) { return cdiv(n, kBlk) * kBlk; }
__host__ __device__ inline bool quad_order(int64_t G, int64_t n) { return G > 4 && n > kRowSelectMax; }
// Where the quad of token tt of the tile of blocks beta0 .. is, from the tile's first score.
__device__ __forceinline__ uint32_t quad_off(uint32_t nblk, uint32_t G, uint32_t h, uint32_t beta0, uint32_t tt) {
  constexpr uint32_t kTile = (uint32_t)(kRegTok / kBlk);
  const uint32_t nbt = min(nblk - beta0, kTile);
  return (((tt % kBlk) / 4u * G + h) * nbt + tt / kBlk) * 4u;
}

// Candidate counters of a row, one per 256 bytes: every workgroup of a pass
// adds to its row's counter, and atomics to one cache line serialise.
constexpr int64_t kCntStride = 64;

struct TopkSel {
  uint32_t *thr;        // [rows] first-pass threshold key T_hi
  uint32_t *thr_lo;     // [rows] safe threshold key T_lo
  uint32_t *cand_cnt;   // [rows * kCntStride] candidates of the first pass
  uint32_t *cand2_cnt;  // [rows * kCntStride] candidates of the fallback pass
  uint64_t *cand;       // [rows, cand_cap] K64 candidates (of the pass in effect)
  int64_t cand_cap;
  uint32_t *rc1;        // region layout: [rows, nreg] counts of the first pass (null: list layout)
  uint32_t *rc2;        // region layout: [rows, nreg] counts of the fallback pass
  int64_t nreg;         // regions per row (cand_cap / kRegTok)
  uint32_t kk;
  __host__ __device__ uint32_t *cnt1(int64_t row) const { return cand_cnt + row * kCntStride; }
  __host__ __device__ uint32_t *cnt2(int64_t row) const { return cand2_cnt + row * kCntStride; }
};

// Sample stride in tiles of `tile` tokens: about 16384 sampled tokens per row
// (32768 for the fused scan's wave-tiles, whose first-pass threshold then sits
// at about 40 sampled keys for 1M-token rows: a fallback rescan of a row, the
// price of a threshold above the row's kk-th key, stays below 1e-6 per row),
// more where the sample must hold 2 kk keys or where about 16 sampled keys must
// reach the first-pass threshold (kAlphaX2 / 2 * kk * sample / n >= 16), at
// most kMaxSample keys.  The stride rounds up, so the sample never exceeds
// that many tiles.
inline int64_t topk_tile_stride(int64_t n, int64_t kk, int64_t tile) {
  const int64_t ntiles = cdiv(n, tile);
  int64_t want = tile == kRegTok ? 32 : cdiv(8 * kTileTok, tile);
  // the fused scan's sample keeps 64 group maxima per tile: at least 2 kk of them
  if (tile == kRegTok && kk > 0) {
    const int64_t g = cdiv(2 * kk, kRegTok / kGroupTok);
    want = g > want ? g : want;
  }
  if (kk > 0) {
    const int64_t a = cdiv(2 * kk, tile), b = cdiv(32 * n, kAlphaX2 * kk * tile);
    want = a > want ? a : want;
    want = b > want ? b : want;
  }
  const int64_t cap = kMaxSample / tile;
  if (want > cap) want = cap;
  const int64_t S = cdiv(ntiles, want);
  return S < 1 ? 1 : S;
}

inline int64_t topk_sample_tiles(int64_t n, int64_t S, int64_t tile) { return cdiv(cdiv(n, tile), S); }

// Rank in the sample of the first-pass threshold: about kAlphaX2 / 2 * kk of the row's
// n elements are expected at or above it (kk when the sample is the row).
inline int64_t topk_hi_rank(int64_t n, int64_t S, int64_t kk, int64_t tile) {
  int64_t sampled = 0;
  for (int64_t t = 0, nt = topk_sample_tiles(n, S, tile); t < nt; ++t) {
    const int64_t left = n - t * S * tile;
    sampled += left < tile ? (left > 0 ? left : 0) : tile;
  }
  const int64_t r = (kAlphaX2 * kk * sampled + 2 * n - 1) / (2 * n);
  return r < 1 ? 1 : (r > kk ? kk : r);
}

// 256-byte section alignment inside workspaces
inline size_t ws_align(size_t x) { return (x + 255) & ~(size_t)255; }

// Layout of the selection state inside a workspace; returns bytes used.
// nreg > 0: region layout with nreg regions per row (cand_cap = nreg * kRegTok).
size_t topk_sel_layout(int64_t rows, int64_t cand_cap, int64_t nreg, char *base, TopkSel *s);

// Whole top-k workspace: sampled keys [rows, samp_cap] + selection state with
// candidate room for a full row (regions: whole groups of four regions, the
// list layout otherwise).  Samples are tiles of kRegTok tokens with regions,
// kTileTok otherwise.  S is sized for kk = k (an upper bound on k - sink - local; a
// larger kk only means a denser sample).
size_t topk_layout(int64_t rows, int64_t n, int64_t k, bool regions, char *base, uint32_t **samp, int64_t *samp_cap,
                   TopkSel *sel, int64_t *S_out);

// The attention over each row's k <= 512 selected positions that a selection goes on
// to: q [rows, D] query heads (row = bh * G + g), K, V bf16 rows [BH, cap, D = 128] in
// device memory, out [rows, D] fp32, equal to gather_attention's output for the
// selected indices.
struct AttnArgs {
  const float *q;
  int64_t G;
  const void *K, *V;
  int64_t cap;
  float scale;
  float *out;
};
constexpr int64_t kAttnFusedMax = 512;

// T_lo (rank kk) and T_hi (rank r_hi <= kk) of every row's sample; clears the counters.
int launch_select_keys(const uint32_t *samp, int64_t rows, int64_t samp_cap, int64_t kk, int64_t r_hi, TopkSel s,
                       hipStream_t st);
// Thresholds of the fused scan's rows from their sample's group maxima
// (ng <= 4096 per row).
int launch_select_groups(const uint32_t *gmax, int64_t rows, int64_t ng, int64_t kk, int64_t r_hi, TopkSel s,
                         hipStream_t st);
int launch_sample_scores(const float *scores, int64_t rows, int64_t n, int64_t S, int64_t sink, int64_t lstart,
                         uint32_t *samp, int64_t samp_cap, hipStream_t st);
// First pass (fallback = false) or fallback pass (rows whose first pass found fewer than kk).
int launch_filter_scores(const float *scores, int64_t rows, int64_t n, int64_t sink, int64_t lstart, TopkSel s,
                         bool fallback, hipStream_t st);
// Either layout (s.rc1 set: regions).
int launch_finalize(int64_t rows, int64_t m, int64_t k, int64_t sink, int64_t local, TopkSel s, int64_t *idx,
                    hipStream_t st);
// Exact top kk of score rows from their 16-token group maxima (gmax [rows, ceil(n / 16)]
// largest masked keys; scores in the fused scan's order): only the groups that
// can hold a top-kk key are read.
// att (k <= 512): the same workgroups go on to their query heads' attention.
int launch_rowselect_gmax(const float *scores, const uint32_t *gmax, int64_t rows, int64_t G, int64_t n, int64_t m,
                          int64_t k, int64_t sink, int64_t local, int64_t *idx, const AttnArgs *att, hipStream_t st);
// kk == 0: only the sink and local positions are written.
int launch_fixed_only(int64_t rows, int64_t m, int64_t k, int64_t sink, int64_t local, int64_t *idx, hipStream_t st);
// State of the wide selection (exact top kk of candidate lists for any kk by a
// 64-bit radix select, then a counting or bitonic sort; launches of
// data-independent shape).
size_t wide_select_bytes(int64_t rows, int64_t kk);
// Ranks of the kk <= kRankListMax distinct values of each row of sel [rows, P]
// by one counting sort, written as idx [rows, k] (then the fixed positions).
int launch_rank_list(const uint64_t *sel, int64_t P, int64_t rows, int64_t kk, int64_t m, int64_t k, int64_t sink,
                     int64_t local, int64_t *idx, hipStream_t st);
// The wide selection over the candidate lists (list layout) of the chain's filter passes.
int wide_select_list(const TopkSel &s, int64_t rows, int64_t m, int64_t k, int64_t sink, int64_t local, int64_t *idx,
                     void *workspace, size_t workspace_bytes, hipStream_t st);
// Top-k of score rows with kk above kSelMaxK: sample -> select -> filter (and
// the fallback pass), then the wide selection over each row's candidate list;
// workspace of wide_topk_bytes(rows, n, k) (k bounds kk from above).
size_t wide_topk_bytes(int64_t rows, int64_t n, int64_t k);
int wide_topk_run(const float *scores, int64_t rows, int64_t n, int64_t m, int64_t k, int64_t sink, int64_t local,
                  int64_t *idx, void *workspace, size_t workspace_bytes, hipStream_t st);
// Shape checks shared by the top-k entry points (FATHOM_OK or an error status).
int check_topk_args(int64_t rows, int64_t n, int64_t m, int64_t k, int64_t sink, int64_t local, const char *who);

// Wave-aggregated append of K64 values whose predicate holds to a row's list.
__device__ __forceinline__ void wave_append(bool pred, uint64_t val, uint32_t *counter, uint64_t *buf, uint64_t cap,
                                            int lane) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
  base = __builtin_amdgcn_readlane(base, leader);
  const uint64_t slot = (uint64_t)base + __popcll(m & ((1ull << lane) - 1ull));
  if (pred && slot < cap) buf[slot] = val;
}

// Wave-aggregated append into a workgroup-local LDS list; entries past lcap go
// straight to the global list (one atomic each: only hit by adversarial rows).
__device__ __forceinline__ void wave_append_local(bool pred, uint64_t val, uint32_t *lcnt, uint64_t *lbuf,
                                                  uint32_t lcap, uint32_t *gcnt, uint64_t *gbuf, uint64_t gcap,
                                                  int lane) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(lcnt, (uint32_t)__popcll(m));
  base = __builtin_amdgcn_readlane(base, leader);
  const uint32_t slot = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  if (pred) {
    if (slot < lcap) {
      lbuf[slot] = val;
    } else {
      const uint32_t p = atomicAdd(gcnt, 1u);
      if ((uint64_t)p < gcap) gbuf[p] = val;
    }
  }
}

// Copies a workgroup's LDS list to the global list with one reservation.
// Call from all threads after a barrier that completes the appends.
__device__ __forceinline__ void flush_local(const uint32_t *lcnt, const uint64_t *lbuf, uint32_t lcap,
                                            uint32_t *gcnt, uint64_t *gbuf, uint64_t gcap, uint32_t *s_base) {
  const uint32_t nloc = min(*lcnt, lcap);
  if (threadIdx.x == 0) *s_base = nloc ? atomicAdd(gcnt, nloc) : 0u;
  __syncthreads();
  const uint32_t base = *s_base;
  for (uint32_t i = threadIdx.x; i < nloc; i += blockDim.x)
    if ((uint64_t)base + i < gcap) gbuf[base + i] = lbuf[i];
}

__device__ __forceinline__ uint64_t k64_of(uint32_t key, int64_t i) {
  return ((uint64_t)key << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)i);
}

}  // namespace fathom
