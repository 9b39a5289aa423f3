// Sink/local-masked exact top-k over score rows.
//
// Orderable keys: score_key maps a float to a uint32 whose unsigned order is
// torch.topk's value order; K64 = key << 32 | (0xFFFFFFFF - index) makes every
// element of a row distinct and orders equal scores by ascending index.
// Rows of up to 131072 tokens (wide selections: 524288) are selected by one
// workgroup each, from their 16-token group maxima or read whole; longer ones run
// select -> filter -> finalize (topk_internal.hpp), where the fused scan+top-k
// replaces `filter` by the scan kernel's own emission.
//
// Selection of the need-th largest value of a set (range_select): the active
// values lie in [lo, hi]; a 2048-bin LDS histogram of (v - lo) >> s, with s
// chosen so the bins span exactly that range, locates the bin holding the
// need-th largest; the range shrinks to that bin (by >= 11 bits) and the
// search repeats until the bin holds exactly the values still needed.  Bins
// follow the values' actual spread, so a row's candidates -- all packed just
// above a threshold -- still spread over many bins (few atomic collisions),
// and a 64-bit K64 needs at most six rounds.
#include <type_traits>

#include "topk_internal.hpp"
#include "scan_core.hpp"
#include "attn_core.hpp"

namespace fathom {
namespace {

constexpr int kSelThreads = 1024;
constexpr int kSelPer = (int)(kMaxSample / kSelThreads);  // keys per thread in select
constexpr int kFinThreads = 1024;
constexpr int kFilterThreads = 256;
constexpr uint32_t kFilterLocal = 2048;  // LDS candidates per filter workgroup
constexpr int kCandLds = 16384;          // candidates selected in LDS (128 KB)
constexpr int kMaxK = (int)kSelMaxK;      // largest kk of these selections
constexpr int kBins = 2048;
constexpr int kMaxWaves = 16;            // waves of a 1024-thread workgroup

struct RangeShared {
  uint32_t hist[kBins];
  uint64_t wmin[kMaxWaves], wmax[kMaxWaves];
  uint32_t wsum[kMaxWaves];
  uint64_t fin[kWave];  // the last few values of a range, selected by one wave
  uint64_t lo, hi, thr;
  uint32_t need, done, hsel, fcnt, hcnt;
};

// The two values of lane pair {i & ~J, i | J} (in some order) for a compare-
// exchange at distance J, on the VALU: DPP quad permutes (J = 1, 2), a quad
// reversal then a half-row mirror (J = 4: i ^ 3 ^ 7), a row rotation by 8
// (J = 8), and the gfx950 row swaps v_permlane16/32_swap (J = 16, 32: the
// values of lanes i & ~J and i | J).
template <int J>
__device__ __forceinline__ void lane_pair(uint64_t v, uint64_t &x, uint64_t &y) {
  const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
  uint32_t l0, l1, h0, h1;
  if constexpr (J == 16 || J == 32) {
    const auto pl = J == 16 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                            : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto ph = J == 16 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                            : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    l0 = pl[0];
    l1 = pl[1];
    h0 = ph[0];
    h1 = ph[1];
  } else {
    l0 = lo;
    h0 = hi;
    if constexpr (J == 1) {
      l1 = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
      h1 = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, false);
    } else if constexpr (J == 2) {
      l1 = __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
      h1 = __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xF, 0xF, false);
    } else if constexpr (J == 4) {  // quad_perm [3,2,1,0], then row_half_mirror
      l1 = __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(lo, 0x1B, 0xF, 0xF, false), 0x141, 0xF, 0xF, false);
      h1 = __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(hi, 0x1B, 0xF, 0xF, false), 0x141, 0xF, 0xF, false);
    } else {
      static_assert(J == 8, "compare-exchange distance");
      l1 = __builtin_amdgcn_mov_dpp(lo, 0x128, 0xF, 0xF, false);  // row_ror:8
      h1 = __builtin_amdgcn_mov_dpp(hi, 0x128, 0xF, 0xF, false);
    }
  }
  x = ((uint64_t)h0 << 32) | l0;
  y = ((uint64_t)h1 << 32) | l1;
}

template <int KB, int J>
__device__ __forceinline__ uint64_t bitonic_merge(uint64_t v, int lane) {
  uint64_t x, y;
  lane_pair<J>(v, x, y);
  const bool keep_max = ((lane & J) == 0) == ((lane & KB) == 0);
  const uint64_t mx = x > y ? x : y, mn = x > y ? y : x;
  v = keep_max ? mx : mn;
  if constexpr (J > 1) v = bitonic_merge<KB, J / 2>(v, lane);
  return v;
}

// Descending bitonic sort of the 64 values of a wave (one per lane), in
// registers: 21 compare-exchange stages of a few VALU instructions each.
__device__ __forceinline__ uint64_t wave_sort_desc(uint64_t v, int lane) {
  v = bitonic_merge<2, 1>(v, lane);
  v = bitonic_merge<4, 2>(v, lane);
  v = bitonic_merge<8, 4>(v, lane);
  v = bitonic_merge<16, 8>(v, lane);
  v = bitonic_merge<32, 16>(v, lane);
  v = bitonic_merge<64, 32>(v, lane);
  return v;
}

// Wave-wide minimum and maximum of 64-bit values (every lane gets both):
// butterfly over the same lane pairs as the sort.
template <int J>
__device__ __forceinline__ void minmax_step(uint64_t &mn, uint64_t &mx) {
  uint64_t a, b, c, d;
  lane_pair<J>(mn, a, b);
  lane_pair<J>(mx, c, d);
  mn = a < b ? a : b;
  mx = c > d ? c : d;
}
__device__ __forceinline__ void wave_minmax_u64(uint64_t &mn, uint64_t &mx) {
  minmax_step<1>(mn, mx);
  minmax_step<2>(mn, mx);
  minmax_step<4>(mn, mx);
  minmax_step<8>(mn, mx);
  minmax_step<16>(mn, mx);
  minmax_step<32>(mn, mx);
}

// Descending ranks of the first nlim slots (a power of two, 64 <= nlim <= E *
// 1024) of E * 1024 values, thread t holding slots t + 1024 e (the whole
// workgroup calls it; slots from nlim on take no part).  Each wave sorts its
// 64-value runs in registers; merge levels in LDS double the runs until at
// most 8 remain; then a value's rank is the number of greater values over all
// runs (binary searches), and put(rank, value) is called for every slot below
// nlim.  Distinct values get distinct ranks; equal values share one.  a and b:
// LDS buffers of nlim values.
template <int E, typename Put>
__device__ __forceinline__ void block_rank_desc(const uint64_t (&v)[E], uint64_t *a, uint64_t *b, int nlim, Put put) {
  const int t = threadIdx.x, lane = t & 63;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (t + 1024 * e < nlim) a[t + 1024 * e] = wave_sort_desc(v[e], lane);  // uniform per wave
  __syncthreads();
  int w = kWave;
  for (; nlim > 8 * w; w <<= 1) {
    // merge: an element's new place is its index in its own run plus the
    // partner run's elements ahead of it (strictly greater for the left run,
    // greater or equal for the right one: equal values keep run order)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = t + 1024 * e;
      if (i >= nlim) continue;
      const uint64_t x = a[i];
      const int r = i / w, p = i - r * w;
      const bool left = (r & 1) == 0;
      const uint64_t *part = a + (r ^ 1) * w;
      int c = 0;
      for (int step = w; step > 0; step >>= 1) {
        if (c + step <= w) {
          const uint64_t y = part[c + step - 1];
          if (left ? (y > x) : (y >= x)) c += step;
        }
      }
      b[(r >> 1) * 2 * w + p + c] = x;
    }
    __syncthreads();
    uint64_t *tmp = a;
    a = b;
    b = tmp;
  }
  const int nr = nlim / w;  // at most 8 runs
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = t + 1024 * e;
    if (i >= nlim) continue;
    const uint64_t x = a[i];
    // greater values per run, by binary searches in all runs at once (eight
    // independent LDS reads per step); x's own run counts the values before it
    int c[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) c[q] = 0;
    for (int step = w; step > 0; step >>= 1) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int j = min(c[q] + step, w) - 1;
        const uint64_t y = a[(q < nr ? q * w : 0) + j];  // in bounds for every q
        if (q < nr && c[q] + step <= w && y > x) c[q] += step;
      }
    }
    int rank = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) rank += c[q];
    put(rank, x);
  }
}

__device__ __forceinline__ bool finite_key(uint32_t key) { return key > kKeyNegInf && key < 0xFF800000u; }

// Linear bins of scores over the finite range [lo, hi] of keys: -inf in the
// bottom bin, NaN and +inf in the top one.  Every step of the map is monotone.
struct LinearBins {
  float flo, scale;
  __device__ __forceinline__ LinearBins(uint32_t lo, uint32_t hi)
      : flo(key_value(lo)), scale((float)kBins / (key_value(hi) - flo)) {}
  __device__ __forceinline__ uint32_t of(uint32_t key) const {
    const float x = fminf(fmaxf((key_value(key) - flo) * scale, 0.0f), (float)(kBins - 1));  // NaN (equal scores): 0
    return finite_key(key) ? (uint32_t)x : key > kKeyNegInf ? (uint32_t)(kBins - 1) : 0u;
  }
  __device__ __forceinline__ bool positive(uint32_t bin) const { return flo + (float)bin / scale > 0.0f; }
};
// Bins of keys over the finite range [lo, hi], NaN and +inf in the top one.
struct KeyBins {
  uint32_t lo;
  int sft;
  __device__ __forceinline__ KeyBins(uint32_t lo_, uint32_t hi) : lo(lo_) {
    const uint32_t R = hi > lo_ ? hi - lo_ : 0u;
    const int bl = R ? 32 - __clz((int)R) : 0;
    sft = bl > 11 ? bl - 11 : 0;
  }
  __device__ __forceinline__ uint32_t of(uint32_t key) const {
    return finite_key(key) ? (key - lo) >> sft : key > kKeyNegInf ? (uint32_t)(kBins - 1) : 0u;
  }
};

// Descending ranks of the cnt valid values of E * 1024 (thread t holding slots
// t + 1024 e; the valid ones are the slots below cnt -- LINEAR: the nonzero ones --
// all distinct) by a
// counting sort: 2048 bins of (v - min) >> s over the values' range (LINEAR: of
// the scores themselves over the finite ones' range, -inf in the bottom bin, NaN
// and +inf in the top one), each
// value's place in its bin from a returning LDS atomic, the bins' offsets by a
// prefix sum from the top bin down, then every value's rank = the values in
// higher bins + the greater values of its own bin (a few, read from the
// values placed in bin order).  Bins whose values all rank at or past limit are
// left out.  Values crowd a bin only where their range is
// dominated by a few outliers: then (more than kCrowd in one bin) the ranks
// come from block_rank_desc over the first nlim slots instead (LINEAR: nothing is
// ranked and the call returns false).  put(rank, v)
// is called for every valid value of rank below limit (and some past it).  scratch: LDS of max(E * 1024 + 2048,
// 2 * nlim) values.
// The bits of a key grow with the logarithm of the score's magnitude: right for the
// tail above a threshold, with its outliers, but a whole row's scores, of both
// signs, crowd into a few dozen bins; those take LINEAR (n = 1000, the selection:
// 13.8 -> 4.8 us).
// The sort of 8192 allows its bins more before it falls back, to about 80 us of merges
// (32 rows of 500000 tokens, correlation length 4, k = 6136: 177 -> 102 us).
template <int E, bool LINEAR = false, typename Put>
__device__ __forceinline__ bool bin_rank_desc(const uint64_t (&v)[E], int cnt, int limit, uint64_t *scratch,
                                              RangeShared &sh, int nlim, Put put) {
  static_assert(kBins == 2 * kFinThreads, "two bins per thread");
  constexpr uint32_t kCrowd = E > 4 ? 192 : 48;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = kFinThreads >> 6;
  uint64_t *placed = scratch;                                           // [E * 1024] values in bin order
  uint32_t *hist = reinterpret_cast<uint32_t *>(scratch + E * 1024);    // [2048] values per bin
  uint32_t *above = hist + kBins;                                       // [2048] values in higher bins
  const auto valid = [&](int e) { return LINEAR ? v[e] != 0ull : t + 1024 * e < cnt; };
  uint64_t mn = ~0ull, mx = 0ull;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (valid(e) && (!LINEAR || finite_key((uint32_t)(v[e] >> 32)))) {
      mn = v[e] < mn ? v[e] : mn;
      mx = v[e] > mx ? v[e] : mx;
    }
  wave_minmax_u64(mn, mx);
  if (lane == 0) {
    sh.wmin[wave] = mn;
    sh.wmax[wave] = mx;
  }
  hist[t] = hist[t + kFinThreads] = 0u;
  if (t == 0) sh.fcnt = 0u;
  __syncthreads();
  uint64_t lo = ~0ull, hi = 0ull;
  for (int w = 0; w < nw; ++w) {
    lo = sh.wmin[w] < lo ? sh.wmin[w] : lo;
    hi = sh.wmax[w] > hi ? sh.wmax[w] : hi;
  }
  const uint64_t R = cnt > 0 ? hi - lo : 0ull;
  const int bl = R ? 64 - __clzll((long long)R) : 0;
  const int sft = bl > 11 ? bl - 11 : 0;  // (v - lo) >> sft < 2048
  const LinearBins lin((uint32_t)(lo >> 32), (uint32_t)(hi >> 32));
  uint32_t bin[E], slot[E];
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (valid(e)) {
      bin[e] = LINEAR ? lin.of((uint32_t)(v[e] >> 32)) : (uint32_t)((v[e] - lo) >> sft);
      slot[e] = atomicAdd(&hist[bin[e]], 1u);
    }
  __syncthreads();
  // values in higher bins: thread t holds bins 2047 - 2t, 2046 - 2t
  const uint32_t c0 = hist[kBins - 1 - 2 * t], c1 = hist[kBins - 2 - 2 * t], c = c0 + c1;
  const uint32_t wi = wave_incl_scan_u32(c);
  if (lane == kWave - 1) sh.wsum[wave] = wi;
  __syncthreads();
  uint32_t ab = wi - c;
  for (int w = 0; w < wave; ++w) ab += sh.wsum[w];
  const uint32_t lim = (uint32_t)limit;
  if ((c0 > kCrowd && ab < lim) || (c1 > kCrowd && ab + c0 < lim)) sh.fcnt = 1u;  // any thread: the same value
  above[kBins - 1 - 2 * t] = ab;
  above[kBins - 2 - 2 * t] = ab + c0;
  __syncthreads();
  if (sh.fcnt) {  // uniform
    if constexpr (LINEAR) return false;
    __syncthreads();  // scratch is rewritten
    block_rank_desc<E>(v, scratch, scratch + nlim, nlim, [&](int rank, uint64_t x) {
      if (rank < cnt) put(rank, x);
    });
    return true;
  }
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (valid(e) && above[bin[e]] < lim) placed[above[bin[e]] + slot[e]] = v[e];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (valid(e) && above[bin[e]] < lim) {
      const uint32_t base = above[bin[e]], n = hist[bin[e]];
      uint32_t rank = base;
      for (uint32_t j = 0; j < n; ++j) rank += placed[base + j] > v[e] ? 1u : 0u;
      put((int)rank, v[e]);
    }
  return true;
}

// Value sources of the selections.  for_each(f) calls f(ok, v) for every value
// v of the set, each thread of the workgroup for its share, in loops that are
// uniform over the workgroup (all threads call it; f runs with every lane
// active, v meaningful where ok).  The selections never depend on the order.
struct ArraySrc {  // values p[0, cnt) (LDS or global memory)
  const uint64_t *p;
  int64_t cnt;
  template <typename F>
  __device__ __forceinline__ void for_each(F f) const {
    for (int64_t i0 = 0; i0 < cnt; i0 += blockDim.x) {
      const int64_t i = i0 + threadIdx.x;
      const bool ok = i < cnt;
      f(ok, ok ? p[i] : 0ull);
    }
  }
};

// A row's candidates in the region layout: region r holds rc[r] values at
// cand[r * kRegTok, ...).  Each wave takes batches of 64 regions (the next
// batch's counts load while the current one is read); lane e of a step reads
// the batch's e-th value, found by a binary search over the lanes' exclusive
// prefix sums of the counts.
static_assert(kRegTok < (1 << 11), "region counts fit the 11-bit wave sums of RegionSrc");
struct RegionSrc {
  const uint32_t *rc;
  const uint64_t *cand;
  int64_t nreg;
  template <typename F>
  __device__ __forceinline__ void for_each(F f) const {
    const int lane = threadIdx.x & 63;
    const int64_t step = (int64_t)(blockDim.x >> 6) * kWave;
    int64_t r0 = (int64_t)(threadIdx.x >> 6) * kWave;
    uint32_t c = r0 + lane < nreg ? min(rc[r0 + lane], (uint32_t)kRegTok) : 0u;
    while (r0 < nreg) {  // uniform per wave
      const int64_t r1 = r0 + step;
      const uint32_t cn = r1 + lane < nreg ? min(rc[r1 + lane], (uint32_t)kRegTok) : 0u;
      const uint32_t pre = (uint32_t)wave_excl_scan_small<11>((int)c, lane);  // counts <= kRegTok = 1024
      const uint32_t tot = (uint32_t)wave_sum_small<11>((int)c);
      for (uint32_t e0 = 0; e0 < tot; e0 += kWave) {
        const uint32_t e = e0 + lane;
        int j = 0;  // the last lane whose prefix is <= e: its region holds value e
#pragma unroll
        for (int sft = 32; sft > 0; sft >>= 1)
          if (__shfl(pre, j + sft, kWave) <= e) j += sft;
        const uint32_t pj = __shfl(pre, j, kWave);
        const bool ok = e < tot;
        f(ok, ok ? cand[(r0 + j) * kRegTok + (e - pj)] : 0ull);
      }
      r0 = r1;
      c = cn;
    }
  }
};

// Wave-aggregated append of the values whose ok holds to an LDS list (one LDS
// atomic per wave); the counter keeps counting past cap, values past it are
// dropped.  Call with every lane of the wave active.
__device__ __forceinline__ void lds_append(bool ok, uint64_t v, uint32_t *cnt, uint64_t *buf, uint32_t cap, int lane) {
  const uint64_t m = __ballot(ok);
  if (m == 0ull) return;
  const int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0u;
  if (lane == leader) base = atomicAdd(cnt, (uint32_t)__popcll(m));
  base = __builtin_amdgcn_readlane(base, leader);
  const uint32_t slot = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
  if (ok && slot < cap) buf[slot] = v;
}

// Copies a source's values to LDS (at most cap of them); returns how many the
// source holds.  All threads call it; s_cnt is free again on return.
template <typename Src>
__device__ __forceinline__ uint32_t stage_lds(const Src &src, uint64_t *buf, uint32_t cap, uint32_t &s_cnt) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x == 0) s_cnt = 0u;
  __syncthreads();
  src.for_each([&](bool ok, uint64_t v) { lds_append(ok, v, &s_cnt, buf, cap, lane); });
  __syncthreads();
  const uint32_t tot = s_cnt;
  __syncthreads();
  return tot;
}

// Copies a row's candidates in the region layout to LDS (at most cap of them)
// and returns how many it holds.  Per chunk of up to 4 * kFinThreads regions:
// each thread loads 4 counts at once, a workgroup prefix sum turns them into
// the regions' first slots (in pre: 4 * kFinThreads words of LDS), then value
// e of the chunk is read by thread e mod kFinThreads after a binary search in
// pre -- every load of a chunk is in flight at once, however unevenly the
// candidates spread.  nreg: a multiple of 4.  All threads call it.
__device__ __forceinline__ uint32_t stage_regions(const uint32_t *rc, const uint64_t *cand, int64_t nreg, uint64_t *buf, uint32_t cap,
                                  uint32_t *pre, RangeShared &sh) {
  constexpr int kR = 4 * kFinThreads;  // regions per chunk
  constexpr int kU = 4;                // values per thread read together
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  uint32_t base = 0u;
  for (int64_t c0 = 0; c0 < nreg; c0 += kR) {
    const int nr = (int)min((int64_t)kR, nreg - c0);
    uint4 c = make_uint4(0u, 0u, 0u, 0u);
    if (4 * tid < nr) c = *reinterpret_cast<const uint4 *>(rc + c0 + 4 * tid);
    c.x = min(c.x, (uint32_t)kRegTok);
    c.y = min(c.y, (uint32_t)kRegTok);
    c.z = min(c.z, (uint32_t)kRegTok);
    c.w = min(c.w, (uint32_t)kRegTok);
    const uint32_t t = c.x + c.y + c.z + c.w;
    const uint32_t wi = wave_incl_scan_u32(t), wx = wi - t;
    if (lane == kWave - 1) sh.wsum[wave] = wi;
    __syncthreads();
    uint32_t off = wx, tot = 0u;
    for (int w = 0; w < nw; ++w) {
      const uint32_t ws = sh.wsum[w];
      off += w < wave ? ws : 0u;
      tot += ws;
    }
    if (4 * tid < nr) {
      pre[4 * tid] = off;
      pre[4 * tid + 1] = off + c.x;
      pre[4 * tid + 2] = off + c.x + c.y;
      pre[4 * tid + 3] = off + c.x + c.y + c.z;
    }
    __syncthreads();
    for (uint32_t e0 = 0; e0 < tot; e0 += kU * kFinThreads) {
      uint64_t v[kU];
      uint32_t slot[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t e = e0 + u * kFinThreads + tid;
        slot[u] = ~0u;
        v[u] = 0ull;
        if (e < tot) {
          int lo = 0, hi = nr - 1;  // the last region whose first slot is <= e
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (pre[mid] <= e) lo = mid;
            else hi = mid - 1;
          }
          v[u] = cand[(c0 + lo) * kRegTok + (e - pre[lo])];
          slot[u] = base + e;
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (slot[u] < cap) buf[slot[u]] = v[u];
    }
    base += tot;
    __syncthreads();  // pre and wsum are rewritten by the next chunk
  }
  return base;
}

// Smallest value >= lo of the need-th largest element among the cnt values of
// src (all threads of the workgroup call it).  Returns thr with #{v >= thr} >=
// need, equality when the values are distinct; thr = 0 when there are fewer
// than need values.
template <typename Src>
__device__ __forceinline__ uint64_t range_select(const Src &src, int64_t cnt, uint32_t need, RangeShared &sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  if (cnt < (int64_t)need || need == 0) return 0ull;
  // value range
  uint64_t mn = ~0ull, mx = 0ull;
  src.for_each([&](bool ok, uint64_t v) {
    if (ok) {
      mn = v < mn ? v : mn;
      mx = v > mx ? v : mx;
    }
  });
  wave_minmax_u64(mn, mx);
  if (lane == 0) {
    sh.wmin[wave] = mn;
    sh.wmax[wave] = mx;
  }
  __syncthreads();
  if (tid == 0) {
    uint64_t a = ~0ull, b = 0ull;
    for (int w = 0; w < nw; ++w) {
      a = sh.wmin[w] < a ? sh.wmin[w] : a;
      b = sh.wmax[w] > b ? sh.wmax[w] : b;
    }
    sh.lo = a;
    sh.hi = b;
    sh.need = need;
    sh.done = 0u;
    sh.hsel = ~0u;
    sh.thr = a;
  }
  __syncthreads();
  // each round narrows the range of distinct 64-bit values by at least 11
  // bits, so six rounds end it; the bound keeps a source that yields fewer
  // values than cnt from looping
  for (int round = 0; round < 8; ++round) {
    const uint64_t lo = sh.lo, hi = sh.hi;
    const uint32_t nd = sh.need;
    const uint64_t R = hi - lo;
    const int bl = R ? 64 - __clzll((long long)R) : 0;
    const int s = bl > 11 ? bl - 11 : 0;
    const int nb = (int)(R >> s) + 1;
    for (int b = tid; b < nb; b += blockDim.x) sh.hist[b] = 0u;
    __syncthreads();
    src.for_each([&](bool ok, uint64_t v) {
      if (ok && v >= lo && v <= hi) atomicAdd(&sh.hist[(v - lo) >> s], 1u);
    });
    __syncthreads();
    // values in the bins above each thread's pair (thread t owns bins 2t, 2t + 1)
    const int b0 = 2 * tid;
    const uint32_t h0 = b0 < nb ? sh.hist[b0] : 0u, h1 = b0 + 1 < nb ? sh.hist[b0 + 1] : 0u;
    const uint32_t x = h0 + h1;
    const uint32_t incl = wave_incl_scan_u32(x);
    const uint32_t wtot = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (lane == 0) sh.wsum[wave] = wtot;
    __syncthreads();
    uint32_t later = 0u;
    for (int w = wave + 1; w < nw; ++w) later += sh.wsum[w];
    const uint32_t above = wtot - incl + later;  // values in bins above b0 + 1
    int bsel = -1;
    uint32_t nsel = 0u, hsel = 0u;
    if (above < nd && above + h1 >= nd) {
      bsel = b0 + 1;
      nsel = nd - above;
      hsel = h1;
    } else if (above + h1 < nd && above + h1 + h0 >= nd) {
      bsel = b0;
      nsel = nd - above - h1;
      hsel = h0;
    }
    __syncthreads();  // every thread has read lo/hi/need
    if (bsel >= 0) {
      const uint64_t nlo = lo + ((uint64_t)bsel << s);
      const uint64_t width = s ? (((uint64_t)1 << s) - 1ull) : 0ull;
      sh.lo = nlo;
      sh.hi = (hi - nlo) > width ? nlo + width : hi;
      sh.need = nsel;
      sh.thr = nlo;
      sh.hsel = hsel;
      sh.done = (hsel == nsel || s == 0) ? 1u : 0u;
    }
    __syncthreads();
    if (sh.done) break;
    if (sh.hsel <= (uint32_t)kWave) {
      // at most 64 values left in the range: gather them, one wave sorts them
      // and the need-th largest is the threshold
      const uint64_t flo = sh.lo, fhi = sh.hi;
      const uint32_t fneed = sh.need;
      if (tid == 0) sh.fcnt = 0u;
      __syncthreads();
      src.for_each([&](bool ok, uint64_t v) {
        lds_append(ok && v >= flo && v <= fhi, v, &sh.fcnt, sh.fin, (uint32_t)kWave, lane);
      });
      __syncthreads();
      if (wave == 0) {
        const uint32_t fc = min(sh.fcnt, (uint32_t)kWave);
        const uint64_t y = wave_sort_desc((uint32_t)lane < fc ? sh.fin[lane] : 0ull, lane);
        if ((uint32_t)lane == fneed - 1u) sh.thr = y;
      }
      __syncthreads();
      break;
    }
  }
  return sh.thr;
}

template <typename Scores>
__device__ __forceinline__ uint32_t masked_key(const Scores &row, int64_t i, int64_t sink, int64_t lstart) {
  return (i < sink || i >= lstart) ? kKeyNegInf : score_key(row[i]);
}

__global__ __launch_bounds__(256) void sample_scores_kernel(const float *__restrict__ scores, int64_t n, int64_t S,
                                                            int64_t sink, int64_t lstart, uint32_t *__restrict__ samp,
                                                            int64_t samp_cap) {
  const int64_t row = blockIdx.y;
  const float *rs = scores + row * n;
  const int64_t ti = blockIdx.x;
  for (int o = threadIdx.x; o < kTileTok; o += 256) {
    const int64_t pos = ti * S * kTileTok + o;
    samp[row * samp_cap + ti * kTileTok + o] = pos < n ? masked_key(rs, pos, sink, lstart) : 0u;
  }
}

// Largest masked key of each 16-token group of score rows (gmax [rows, ceil(n /
// 16)]).  A workgroup takes 4096 tokens, every load in flight at once; a group is
// the 16 lanes of a DPP row, and lane u of a row writes the row's u-th group.
// Rows need no alignment.  Bound: HBM, 4.25 bytes per score.  sink_local_topk of
// 32 rows, k = 512, with it and the selection below against the sample -> select ->
// filter -> finalize chain: n = 32768 46 -> 17.2 us, 50021 48.8 -> 17.7, 131072 42.8 ->
// 19.8.
constexpr int kGmaxPer = 16;
__global__ __launch_bounds__(256) void group_max_kernel(const float *__restrict__ scores, int64_t n, int64_t sink,
                                                        int64_t lstart, uint32_t *__restrict__ gmax) {
  const int64_t row = blockIdx.y, i0 = (int64_t)blockIdx.x * (256 * kGmaxPer) + threadIdx.x;
  const float *rs = scores + row * n;
  float v[kGmaxPer];
#pragma unroll
  for (int u = 0; u < kGmaxPer; ++u) v[u] = i0 + u * 256 < n ? rs[i0 + u * 256] : 0.0f;
  uint32_t mine = 0u;
#pragma unroll
  for (int u = 0; u < kGmaxPer; ++u) {
    const int64_t i = i0 + u * 256;
    uint32_t key = i < n ? ((i < sink || i >= lstart) ? kKeyNegInf : score_key(v[u])) : 0u;
    key = max(key, (uint32_t)__builtin_amdgcn_mov_dpp((int)key, 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
    key = max(key, (uint32_t)__builtin_amdgcn_mov_dpp((int)key, 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
    key = max(key, (uint32_t)__builtin_amdgcn_mov_dpp((int)key, 0x141, 0xF, 0xF, false));  // row_half_mirror
    key = max(key, (uint32_t)__builtin_amdgcn_mov_dpp((int)key, 0x140, 0xF, 0xF, false));  // row_mirror
    if (u == (int)(threadIdx.x & 15)) mine = key;
  }
  const int64_t ngrp = cdiv(n, kGroupTok);
  const int64_t g = (int64_t)blockIdx.x * (256 * kGmaxPer / kGroupTok) + (threadIdx.x & 15) * 16 + (threadIdx.x >> 4);
  if (g < ngrp) gmax[row * ngrp + g] = mine;
}

// Candidates of score rows (keys >= the row's threshold): kPer scores per thread
// and step, their loads in flight at once, 16-byte loads when rows are 16-byte aligned.
// Bound: HBM, 4 bytes per score (sink_local_topk: see launch_filter_scores).
template <bool VEC, int kPer>
__global__ __launch_bounds__(kFilterThreads) void filter_scores_kernel(const float *__restrict__ scores, int64_t n,
                                                                       int64_t sink, int64_t lstart, TopkSel s,
                                                                       bool fallback, int steps) {
  __shared__ uint64_t lbuf[kFilterLocal];
  __shared__ uint32_t lcnt, lbase;
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t row = blockIdx.y;
  if (fallback && *s.cnt1(row) >= s.kk) return;  // the first pass holds the row's top kk
  const float *rs = scores + row * n;
  const uint32_t thr = fallback ? s.thr_lo[row] : s.thr[row];
  uint32_t *cnt = fallback ? s.cnt2(row) : s.cnt1(row);
  uint64_t *cand = s.cand + row * s.cand_cap;
  if (tid == 0) lcnt = 0u;
  __syncthreads();
  constexpr int64_t kFilterStep = kPer * kFilterThreads;
  const int64_t end = min((int64_t)(blockIdx.x + 1) * steps * kFilterStep, n);
  for (int64_t start = (int64_t)blockIdx.x * steps * kFilterStep; start < end; start += kFilterStep) {  // uniform
    const auto at = [&](int u) { return start + (VEC ? 4 * (tid + kFilterThreads * (u >> 2)) + (u & 3) : tid + kFilterThreads * u); };
    float v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u += VEC ? 4 : 1) {
      const int64_t i = at(u);
      if constexpr (VEC) {  // n is a multiple of 4
        float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n) f = *reinterpret_cast<const float4 *>(rs + i);
        v[u] = f.x;
        v[u + 1] = f.y;
        v[u + 2] = f.z;
        v[u + 3] = f.w;
      } else {
        v[u] = i < n ? rs[i] : 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int64_t i = at(u);
      const bool in = i < n;
      const uint32_t key = in ? ((i < sink || i >= lstart) ? kKeyNegInf : score_key(v[u])) : 0u;
      wave_append_local(in && key >= thr, k64_of(key, i), &lcnt, lbuf, kFilterLocal, cnt, cand, (uint64_t)s.cand_cap, lane);
    }
  }
  __syncthreads();
  flush_local(&lcnt, lbuf, kFilterLocal, cnt, cand, (uint64_t)s.cand_cap, &lbase);
}

// Writes the tail of a row's output: zeros after the got selected positions
// (fewer candidates than kk), then the sink and local positions.
__device__ __forceinline__ void write_fixed(int64_t *out, int got, int64_t kk, int64_t m, int64_t sink, int64_t local) {
  for (int i = got + (int)threadIdx.x; i < (int)kk; i += kFinThreads) out[i] = 0;
  for (int i = threadIdx.x; i < (int)(sink + local); i += kFinThreads)
    out[kk + i] = (i < sink) ? (int64_t)i : (int64_t)(m - local + (i - sink));
}

// Exact top kk of the cnt distinct K64 values of src, sorted descending (score
// descending, index ascending), written to out, followed by the sink and local
// positions (the whole workgroup calls it).  cl: LDS scratch of kCandLds
// values; with stage set and cnt <= kCandLds the values are copied there first
// (src must not read cl then).
template <typename Src>
__device__ __forceinline__ void select_sorted(const Src &src, int64_t cnt, int64_t kk, int64_t m, int64_t sink,
                                              int64_t local, int64_t *out, uint64_t *cl, uint64_t *ss,
                                              RangeShared &sh, uint32_t &s_cnt, bool stage) {
  const int tid = threadIdx.x, lane = tid & 63;
  // the exact kk largest first (range selection), then sorted
  auto survivors = [&](const auto &sr) {
    const uint64_t thr = range_select(sr, cnt, (uint32_t)kk, sh);
    if (tid == 0) s_cnt = 0u;
    __syncthreads();
    sr.for_each([&](bool ok, uint64_t v) { lds_append(ok && v >= thr, v, &s_cnt, ss, (uint32_t)kMaxK, lane); });
  };
  if (stage && cnt <= kCandLds) {
    stage_lds(src, cl, (uint32_t)kCandLds, s_cnt);
    survivors(ArraySrc{cl, cnt});
  } else {
    survivors(src);
  }
  __syncthreads();
  const int nv = (int)min(min(s_cnt, (uint32_t)kMaxK), (uint32_t)kk);
  uint64_t v2[2];  // zero: padding (below every K64)
  v2[0] = tid < nv ? ss[tid] : 0ull;
  v2[1] = tid + kFinThreads < nv ? ss[tid + kFinThreads] : 0ull;
  __syncthreads();  // cl is the sort scratch from here
  int nlim = kWave;
  while (nlim < nv) nlim <<= 1;  // the survivors fill the first nv <= 2048 slots
  const int got = nv < (int)kk ? nv : (int)kk;
  // only the survivors are ranked and written
  bin_rank_desc<2>(v2, nv, got, cl, sh, nlim, [&](int rank, uint64_t x) {
    if (rank < got) out[rank] = (int64_t)(0xFFFFFFFFu - (uint32_t)x);
  });
  write_fixed(out, got, kk, m, sink, local);
}

// Exact top kk of a row's candidates (list layout): those of the first pass,
// or, where it found fewer than kk, those of the fallback pass (which ran for
// exactly such rows); counts in the row counters.
__global__ __launch_bounds__(kFinThreads) void finalize_kernel(int64_t m, int64_t k, int64_t sink, int64_t local,
                                                               TopkSel s, int64_t *__restrict__ idx) {
  __shared__ uint64_t cl[kCandLds];
  __shared__ uint64_t ss[kMaxK];
  __shared__ RangeShared sh;
  __shared__ uint32_t s_cnt;
  const int64_t row = blockIdx.x;
  const int64_t kk = k - sink - local;
  const uint64_t *gc = s.cand + row * s.cand_cap;
  int64_t *out = idx + row * k;
  const uint32_t c1 = *s.cnt1(row);
  const int64_t cnt = min((int64_t)(c1 >= s.kk ? c1 : *s.cnt2(row)), s.cand_cap);
  select_sorted(ArraySrc{gc, cnt}, cnt, kk, m, sink, local, out, cl, ss, sh, s_cnt, true);
}

// A row's output: ranked values below got are written (their tokens also to
// `ranked`, LDS of k int32, if non-null), then the fixed positions.
struct RowOut {
  int64_t *p;
  int64_t kk, m, sink, local;
  int32_t *ranked;
  int got;
  __device__ __forceinline__ void put(int rank, uint64_t x) const {
    if (rank >= got) return;
    const uint32_t tok = 0xFFFFFFFFu - (uint32_t)x;
    p[rank] = (int64_t)tok;
    if (ranked) ranked[rank] = (int32_t)tok;
  }
  // true where the tokens are in `ranked` too
  __device__ __forceinline__ bool finish() const {
    write_fixed(p, got, kk, m, sink, local);
    if (ranked) {  // the same tokens as write_fixed's
      for (int i = got + (int)threadIdx.x; i < (int)kk; i += kFinThreads) ranked[i] = 0;
      for (int i = threadIdx.x; i < (int)(sink + local); i += kFinThreads)
        ranked[kk + i] = (int32_t)((i < sink) ? (int64_t)i : (m - local + (i - sink)));
    }
    return ranked != nullptr;
  }
};

// The attention that follows a row's selection (k <= 512, rows in device memory):
// the workgroup's 16 waves take the row's k positions, exactly as gather_attention's
// attn_stream_kernel does for one split (empty waves add nothing), so out equals
// gather_attention's output.  The ranked tokens stay in LDS, in cl's upper half, past
// the sort's scratch and the attention's triples.
struct RowAttn {
  const float *q;  // [rows, D] fp32 query heads (row = bh * G + g)
  int64_t G;
  attn::RowSrc rs;
  float scale;
  float *out;      // [rows, D] fp32
};
__device__ __forceinline__ int32_t *ranked_lds(uint64_t *cl) {
  static_assert(kCandLds / 2 >= 4 * kFinThreads + kBins && kCandLds / 2 >= 2 * 4 * kFinThreads &&
                    2 * (kCandLds / 2) >= kMaxK + kFinThreads,
                "the ranked tokens lie past the sort's scratch and hold k of them");
  return reinterpret_cast<int32_t *>(cl + kCandLds / 2);
}
__device__ __forceinline__ void row_attention(const RowAttn &ra, const int64_t *ig, int64_t k, bool in_lds,
                                              const int32_t *ranked, uint64_t *cl) {
  constexpr int NW = kFinThreads / kWave;
  static_assert(NW == 16, "one attention split of 16 waves");
  static_assert(sizeof(float) * (2 * NW + NW * attn::kAttnD) <= sizeof(uint64_t) * (kCandLds / 2),
                "the attention's LDS in cl's lower half");
  __syncthreads();  // the row's indices are written (and cl's lower half is free)
  const int64_t row = blockIdx.x, bh = row / ra.G;
  float *wm = reinterpret_cast<float *>(cl), *wl = wm + NW;
  auto wo = reinterpret_cast<float(*)[attn::kAttnD]>(wl + NW);
  const float *qr = ra.q + row * attn::kAttnD;
  float *orow = ra.out + row * attn::kAttnD;
  if (in_lds)  // uniform: the tokens from LDS, else from the index list just written
    attn::attn_stream_block<NW, false>(qr, [&](int64_t j) { return (int64_t)ranked[j]; }, k, 0, bh, ra.rs, ra.scale, wm,
                                       wl, wo, orow, nullptr, true);
  else
    attn::attn_stream_block<NW, false>(qr, [&](int64_t j) { return ig[j]; }, k, 0, bh, ra.rs, ra.scale, wm, wl, wo, orow,
                                       nullptr, true);
}

// The fallback of the fused scan + top-k, run by the finalize workgroup of a
// row whose candidate pass found fewer than kk candidates: the row (head h of
// bh) is rescanned with T_lo into the regions under the second count array by
// the workgroup's first waves, with the scan's plan tables in tsh (LDS that the
// caller frees for it).  The rescan computes the scores of the candidate pass
// bit for bit (the same chain of matrix instructions per token).
__device__ __forceinline__ void rescan_row(const sc::ScanArgs &a, const sc::Emit &em, int64_t bh, int h,
                                           sc::Shared &tsh) {
  sc::plan_tables(tsh, a, bh, sc::kGS * sc::kSlice);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (wave < sc::kWaves) {
    const int64_t nlist = em.sel.nreg > a.nwt ? em.sel.nreg : a.nwt;
    const uint32_t skipm = ((1u << a.G) - 1u) & ~(1u << h);
    sc::tile_pass<sc::kEmitFilter, 1, true, sc::kGS>(a, em, tsh, bh, lane, wave, sc::kWaves, nlist, 0, sc::kQS, skipm);
    __builtin_amdgcn_s_setprio(0);
  }
  // the rescan's region counts and candidates are read back by other waves of
  // the workgroup, and their old values may sit in the CU's L1: write back and
  // invalidate before the barrier
  __threadfence();
  __syncthreads();
}

// Exact top kk of a row of the fused scan + top-k from its candidate regions
// (row = bh * G + h), copied to LDS while they are counted; a row with more
// than kCandLds candidates is selected from its regions in place.  A row with
// fewer than kk first-pass candidates is rescanned first (rescan_row).
template <bool ATTN>
__global__ __launch_bounds__(kFinThreads) void finalize_fused_kernel(int64_t m, int64_t k, int64_t sink, int64_t local,
                                                                     sc::ScanArgs a, sc::Emit em,
                                                                     int64_t *__restrict__ idx, RowAttn ra) {
  __shared__ uint64_t cl[kCandLds];
  __shared__ uint64_t ss[kMaxK];
  __shared__ RangeShared sh;
  __shared__ uint32_t s_cnt;
  static_assert(sizeof(sc::Shared) <= sizeof(cl), "the rescan's plan tables fit the candidate buffer");
  const TopkSel &s = em.sel;
  const int64_t row = blockIdx.x;
  const int64_t kk = k - sink - local;
  const uint64_t *gc = s.cand + row * s.cand_cap;
  int64_t *out = idx + row * k;
  int32_t *ranked = ATTN ? ranked_lds(cl) : nullptr;
  bool in_lds = false;
  uint32_t *pre = reinterpret_cast<uint32_t *>(ss);  // free until the survivors are collected
  RegionSrc src{s.rc1 + row * s.nreg, gc, s.nreg};
  uint32_t cnt = stage_regions(src.rc, gc, s.nreg, cl, (uint32_t)kCandLds, pre, sh);
  if (cnt < s.kk) {  // uniform
    __syncthreads();  // cl holds the plan tables from here
    rescan_row(a, em, row / a.G, (int)(row % a.G), *reinterpret_cast<sc::Shared *>(cl));
    src.rc = s.rc2 + row * s.nreg;
    cnt = stage_regions(src.rc, gc, s.nreg, cl, (uint32_t)kCandLds, pre, sh);
  }
  if (cnt <= (uint32_t)(4 * kFinThreads)) {  // uniform
    // every candidate ranked at once (a few times kk of them): the top kk by
    // rank, written in order
    uint64_t v4[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t i = threadIdx.x + (uint32_t)e * kFinThreads;
      v4[e] = i < cnt ? cl[i] : 0ull;
    }
    __syncthreads();  // cl is the ranking scratch from here
    int nlim = kWave;
    while (nlim < (int)cnt) nlim <<= 1;
    const RowOut ro{out, kk, m, sink, local, ranked, (int64_t)cnt < kk ? (int)cnt : (int)kk};
    bin_rank_desc<4>(v4, (int)cnt, ro.got, cl, sh, nlim, [&](int rank, uint64_t x) { ro.put(rank, x); });
    in_lds = ro.finish();
  } else if (cnt <= (uint32_t)kCandLds) {
    select_sorted(ArraySrc{cl, (int64_t)cnt}, cnt, kk, m, sink, local, out, cl, ss, sh, s_cnt, false);
  } else {
    select_sorted(src, cnt, kk, m, sink, local, out, cl, ss, sh, s_cnt, false);
  }
  if constexpr (ATTN) row_attention(ra, out, k, in_lds, ranked, cl);
}

// Wave-wide minimum and maximum of 32-bit values (in every lane): DPP row
// reductions, then the four rows' results read out.
template <int CTL>
__device__ __forceinline__ void minmax_dpp(uint32_t &mn, uint32_t &mx) {
  mn = min(mn, (uint32_t)__builtin_amdgcn_mov_dpp((int)mn, CTL, 0xF, 0xF, false));
  mx = max(mx, (uint32_t)__builtin_amdgcn_mov_dpp((int)mx, CTL, 0xF, 0xF, false));
}
__device__ __forceinline__ void wave_minmax_u32(uint32_t &mn, uint32_t &mx) {
  minmax_dpp<0xB1>(mn, mx);   // quad_perm [1,0,3,2]
  minmax_dpp<0x4E>(mn, mx);   // quad_perm [2,3,0,1]
  minmax_dpp<0x141>(mn, mx);  // row_half_mirror
  minmax_dpp<0x140>(mn, mx);  // row_mirror
  mn = min(min((uint32_t)__builtin_amdgcn_readlane((int)mn, 0), (uint32_t)__builtin_amdgcn_readlane((int)mn, 16)),
           min((uint32_t)__builtin_amdgcn_readlane((int)mn, 32), (uint32_t)__builtin_amdgcn_readlane((int)mn, 48)));
  mx = max(max((uint32_t)__builtin_amdgcn_readlane((int)mx, 0), (uint32_t)__builtin_amdgcn_readlane((int)mx, 16)),
           max((uint32_t)__builtin_amdgcn_readlane((int)mx, 32), (uint32_t)__builtin_amdgcn_readlane((int)mx, 48)));
}

// Histogram round of kth_bound: the values v with (v - base) >> sh_in == bin_in
// (all when sh_in < 0) counted into 2048 bins of (v - base) >> sft; sets
// sh.hsel to the bin holding the need-th largest of them and sh.need to the
// count of those above it.
template <int PER>
__device__ __forceinline__ void bound_round(const uint32_t (&v)[PER], int cnt, uint32_t need, uint32_t base, int sft,
                                            int sh_in, uint32_t bin_in, RangeShared &sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (tid + u * kFinThreads < cnt && v[u] >= base && (sh_in < 0 || ((v[u] - base) >> sh_in) == bin_in))
      atomicAdd(&sh.hist[(v[u] - base) >> sft], 1u);
  __syncthreads();
  // running counts from the top bin down: thread t holds bins 2047 - 2t, 2046 - 2t
  const uint32_t c0 = sh.hist[kBins - 1 - 2 * tid], c1 = sh.hist[kBins - 2 - 2 * tid], c = c0 + c1;
  const uint32_t wi = wave_incl_scan_u32(c);
  if (lane == kWave - 1) sh.wsum[wave] = wi;
  __syncthreads();
  uint32_t above = wi - c;
  for (int w = 0; w < wave; ++w) above += sh.wsum[w];
  if (above < need && above + c0 >= need) {
    sh.hsel = (uint32_t)(kBins - 1 - 2 * tid);
    sh.need = above;
    sh.hcnt = c0;
  }
  if (above + c0 < need && above + c >= need) {
    sh.hsel = (uint32_t)(kBins - 2 - 2 * tid);
    sh.need = above + c0;
    sh.hcnt = c1;
  }
  sh.hist[tid] = 0u;  // for the next round
  sh.hist[tid + kFinThreads] = 0u;
  __syncthreads();
}

// A lower bound of the need-th largest of the cnt values v (thread t holds
// values t + 1024 u; need <= cnt).  The values at or below kKeyNegInf (group
// maxima of masked positions) are left out of the range: with fewer than need
// values above it the bound is 0.  A 2048-bin histogram over [min, max] of the
// others gives the bin that holds the need-th largest; its lower edge is the
// bound when at most kBoundFine values share the bin (a few extra candidates),
// else one more round over that bin refines it to within (max - min) / 2^22.
constexpr uint32_t kBoundFine = 32;
template <int PER>
__device__ __forceinline__ uint32_t kth_bound(const uint32_t (&v)[PER], int cnt, uint32_t need, RangeShared &sh) {
  static_assert(kBins == 2 * kFinThreads, "two bins per thread");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = kFinThreads >> 6;
  uint32_t mn = ~0u, mx = 0u, nv = 0u;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const bool on = tid + u * kFinThreads < cnt && v[u] > kKeyNegInf;
    if (on) {
      mn = min(mn, v[u]);
      mx = max(mx, v[u]);
    }
    nv += (uint32_t)__popcll(__ballot(on));
  }
  wave_minmax_u32(mn, mx);
  if (lane == 0) {
    sh.wmin[wave] = mn;
    sh.wmax[wave] = ((uint64_t)nv << 32) | mx;  // the wave's count beside its maximum
  }
  sh.hist[tid] = 0u;
  sh.hist[tid + kFinThreads] = 0u;
  __syncthreads();
  uint32_t lo = ~0u, hi = 0u, nvalid = 0u;
  for (int w = 0; w < nw; ++w) {
    lo = min(lo, (uint32_t)sh.wmin[w]);
    hi = max(hi, (uint32_t)sh.wmax[w]);
    nvalid += (uint32_t)(sh.wmax[w] >> 32);
  }
  if (nvalid < need) return 0u;  // uniform
  const uint32_t R = hi - lo;
  const int bl = R ? 32 - __clz((int)R) : 0;
  const int sft = bl > 11 ? bl - 11 : 0;  // (v - lo) >> sft < 2048
  bound_round<PER>(v, cnt, need, lo, sft, -1, 0u, sh);
  const uint32_t b = sh.hsel, base = lo + (b << sft);
  if (sft == 0 || sh.hcnt <= kBoundFine) return base;  // uniform
  const int sft2 = sft > 11 ? sft - 11 : 0;
  const uint32_t need2 = need - sh.need;
  __syncthreads();  // every thread has read sh.hsel, sh.need and sh.hcnt
  bound_round<PER>(v, cnt, need2, base, sft2, sft, 0u, sh);
  return base + (sh.hsel << sft2);
}

// Histogram scan of a round of two_bounds: bins counted from the top; for
// each of the two ranks, the bin that holds it and the count above that bin.
__device__ __forceinline__ void two_bins(const uint32_t *hist, uint32_t na, uint32_t nb, RangeShared &sh,
                                         uint32_t (&sel)[2], uint32_t (&above_sel)[2], uint32_t *s_sel) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t c0 = hist[kBins - 1 - 2 * tid], c1 = hist[kBins - 2 - 2 * tid], c = c0 + c1;
  const uint32_t wi = wave_incl_scan_u32(c);
  if (lane == kWave - 1) sh.wsum[wave] = wi;
  __syncthreads();
  uint32_t above = wi - c;
  for (int w = 0; w < wave; ++w) above += sh.wsum[w];
  const uint32_t need[2] = {na, nb};
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (above < need[r] && above + c0 >= need[r]) {
      s_sel[2 * r] = (uint32_t)(kBins - 1 - 2 * tid);
      s_sel[2 * r + 1] = above;
    }
    if (above + c0 < need[r] && above + c >= need[r]) {
      s_sel[2 * r] = (uint32_t)(kBins - 2 - 2 * tid);
      s_sel[2 * r + 1] = above + c0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    sel[r] = s_sel[2 * r];
    above_sel[r] = s_sel[2 * r + 1];
  }
}

// Lower bounds of the na-th and the nb-th largest of the cnt values v (thread
// t holds values t + 1024 u; nb, na <= cnt) in two histogram rounds shared by
// both ranks: 2048 bins over [min, max], then 2048 bins over each rank's bin
// (the second histogram in hist2).  Each bound is the lower edge of the final
// bin that holds its rank: at least that many values reach it, and it lies
// within (max - min) / 2^22 of the value of that rank.  Only values >= floor
// take part (floor must not exceed the na-th largest value: the ranks are the
// same among them), so a floor near the ranks keeps the bins narrow and the
// histogram atomics few.
template <int PER>
__device__ __forceinline__ void two_bounds(const uint32_t (&v)[PER], int cnt, uint32_t na, uint32_t nb,
                                           RangeShared &sh, uint32_t *hist2, uint32_t *s_sel, uint32_t &ta,
                                           uint32_t &tb, uint32_t floor = 0u, bool coarse_ok = false) {
  static_assert(kBins == 2 * kFinThreads, "two bins per thread");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = kFinThreads >> 6;
  uint32_t mn = ~0u, mx = 0u, nv = 0u;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const bool on = tid + u * kFinThreads < cnt && v[u] >= floor;
    if (on) {
      mn = min(mn, v[u]);
      mx = max(mx, v[u]);
    }
    nv += (uint32_t)__popcll(__ballot(on));
  }
  wave_minmax_u32(mn, mx);
  if (lane == 0) {
    sh.wmin[wave] = mn;
    sh.wmax[wave] = ((uint64_t)nv << 32) | mx;  // the wave's count beside its maximum
  }
  sh.hist[tid] = sh.hist[tid + kFinThreads] = 0u;
  hist2[tid] = hist2[tid + kFinThreads] = 0u;
  __syncthreads();
  uint32_t lo = ~0u, hi = 0u, nvalid = 0u;
  for (int w = 0; w < nw; ++w) {
    lo = min(lo, (uint32_t)sh.wmin[w]);
    hi = max(hi, (uint32_t)sh.wmax[w]);
    nvalid += (uint32_t)(sh.wmax[w] >> 32);
  }
  if (nvalid < na || nvalid < nb) {  // uniform: fewer values at or above floor than a rank
    ta = tb = 0u;
    return;
  }
  const uint32_t R = hi - lo;
  const int bl = R ? 32 - __clz((int)R) : 0;
  const int sft = bl > 11 ? bl - 11 : 0;  // (v - lo) >> sft < 2048
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (tid + u * kFinThreads < cnt && v[u] >= floor) atomicAdd(&sh.hist[(v[u] - lo) >> sft], 1u);
  __syncthreads();
  uint32_t sel[2], above[2];
  two_bins(sh.hist, na, nb, sh, sel, above, s_sel);
  const uint32_t base_a = lo + (sel[0] << sft), base_b = lo + (sel[1] << sft);
  bool coarse = false;
  if (coarse_ok) {  // uniform: both bins hold at most kBoundFine values
    coarse = sh.hist[sel[0]] <= kBoundFine && sh.hist[sel[1]] <= kBoundFine;
    __syncthreads();  // every thread has read the counts before the clear below
  }
  // one value per bin: the bins' values are the ranks' values; coarse: the
  // bins' lower edges
  if (sft == 0 || coarse) {  // uniform
    ta = base_a;
    tb = base_b;
    return;
  }
  const int sft2 = sft > 11 ? sft - 11 : 0;
  sh.hist[tid] = sh.hist[tid + kFinThreads] = 0u;  // every thread has read both histograms (two_bins' barriers)
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u)
    if (tid + u * kFinThreads < cnt && v[u] >= floor) {
      const uint32_t b = (v[u] - lo) >> sft;
      if (b == sel[0]) atomicAdd(&sh.hist[(v[u] - base_a) >> sft2], 1u);
      if (b == sel[1]) atomicAdd(&hist2[(v[u] - base_b) >> sft2], 1u);
    }
  __syncthreads();
  uint32_t sa[2], aa[2], sb[2], ab[2];
  two_bins(sh.hist, na - above[0], na - above[0], sh, sa, aa, s_sel);
  two_bins(hist2, nb - above[1], nb - above[1], sh, sb, ab, s_sel);
  ta = base_a + (sa[0] << sft2);
  tb = base_b + (sb[0] << sft2);
}

// Thresholds of a row from its sampled keys (the row's samp_cap keys, PER per
// thread): T_lo a lower bound of the sample's kk-th largest key, T_hi one of
// its r_hi-th largest (r_hi <= kk, so T_hi >= T_lo up to the bounds' bins).
// The sample is a subset of the row, so T_lo never exceeds the row's kk-th
// largest: every element of the row's top kk has key >= T_lo.  Also clears
// the row's candidate counters (list layout; the region layout has none).
template <int PER>
__global__ __launch_bounds__(kSelThreads) void select_keys_kernel(const uint32_t *__restrict__ samp,
                                                                  int64_t samp_cap, uint32_t kk, uint32_t r_hi,
                                                                  TopkSel s) {
  static_assert(kSelThreads == kFinThreads, "the bounds use the finalize block size");
  __shared__ RangeShared sh;
  __shared__ uint32_t hist2[kBins];
  __shared__ uint32_t s_sel[4];
  const int64_t row = blockIdx.x;
  const uint32_t *src = samp + row * samp_cap;
  uint32_t v[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int64_t i = threadIdx.x + (int64_t)u * kSelThreads;
    v[u] = i < samp_cap ? src[i] : 0u;
  }
  uint32_t t_lo = 0u, t_hi = 0u;  // fewer samples than kk: every element is a candidate
  if (samp_cap >= (int64_t)kk) two_bounds<PER>(v, (int)samp_cap, kk, r_hi < kk ? r_hi : kk, sh, hist2, s_sel, t_lo, t_hi);
  if (threadIdx.x == 0) {
    s.thr[row] = r_hi < kk ? t_hi : t_lo;
    s.thr_lo[row] = t_lo;
    if (!s.rc1) {  // the list layout's filter passes append at these counters
      *s.cnt1(row) = 0u;
      *s.cnt2(row) = 0u;
    }
  }
}

// The same thresholds from the maxima of the sample's 16-key groups (thread t
// holds groups t + 1024 u): each maximum is a sampled key, so the kk-th
// largest maximum bounds the sample's kk-th largest key from below (T_lo stays
// safe), and T_hi only falls (more candidates) where a group holds several of
// the top r_hi keys -- rare when kk is at most a quarter of the groups, the
// launch's condition.  Ranks 16 times fewer values than select_keys_kernel.
// DIRECT: samp already holds group maxima (the fused scan's sample, samp_cap
// of them per row), ranked as they are.
template <int PER, bool DIRECT>
__global__ __launch_bounds__(kSelThreads) void select_groups_kernel(const uint32_t *__restrict__ samp,
                                                                    int64_t samp_cap, uint32_t kk, uint32_t r_hi,
                                                                    TopkSel s) {
  __shared__ RangeShared sh;
  __shared__ uint32_t hist2[kBins];
  __shared__ uint32_t s_sel[4];
  const int64_t row = blockIdx.x;
  const int ng = (int)(DIRECT ? samp_cap : samp_cap / 16);
  uint32_t g[PER];
  if constexpr (DIRECT) {
    const uint32_t *src = samp + row * samp_cap;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = (int)threadIdx.x + u * kSelThreads;
      g[u] = i < ng ? src[i] : 0u;
    }
  } else {
    const uint4 *src = reinterpret_cast<const uint4 *>(samp + row * samp_cap);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = (int)threadIdx.x + u * kSelThreads;
      uint4 q[4] = {};
      if (i < ng) {
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = src[4 * i + j];
      }
      uint32_t m = 0u;
#pragma unroll
      for (int j = 0; j < 4; ++j) m = max(m, max(max(q[j].x, q[j].y), max(q[j].z, q[j].w)));
      g[u] = m;
    }
  }
  uint32_t t_lo = 0u, t_hi = 0u;  // fewer values than kk: every element is a candidate
  // the range leaves out the groups of masked positions (keys at or below
  // -inf); lower bounds from one round where the ranks' bins are sparse
  if (ng >= (int)kk && kk > 0)
    two_bounds<PER>(g, ng, kk, r_hi < kk ? r_hi : kk, sh, hist2, s_sel, t_lo, t_hi, kKeyNegInf + 1u, true);
  if (threadIdx.x == 0) {
    s.thr[row] = r_hi < kk ? t_hi : t_lo;
    s.thr_lo[row] = t_lo;
    if (!s.rc1) {
      *s.cnt1(row) = 0u;
      *s.cnt2(row) = 0u;
    }
  }
}

// A group's 16 scores from four quads `step` apart.
__device__ __forceinline__ void load_quads(const float *q, int64_t step, float (&v)[kGroupTok]) {
  float4 f[kGroupTok / 4];
#pragma unroll
  for (int r = 0; r < kGroupTok / 4; ++r) f[r] = *reinterpret_cast<const float4 *>(q + r * step);
#pragma unroll
  for (int r = 0; r < kGroupTok / 4; ++r) {
    v[4 * r] = f[r].x;
    v[4 * r + 1] = f[r].y;
    v[4 * r + 2] = f[r].z;
    v[4 * r + 3] = f[r].w;
  }
}

// Where a row's scores are: RowScores in the drop-in order, TileScores and
// QuadScores in the fused scan's.  group: the 16 scores of the
// group at t0 (past n: anything, and none where t0 is).
struct RowScores {
  const float *p;
  int64_t n;
  __device__ __forceinline__ RowScores(const float *scores, int64_t n_, int64_t) : p(scores + blockIdx.x * n_), n(n_) {}
  __device__ __forceinline__ float operator[](int64_t i) const { return p[i]; }
  __device__ __forceinline__ void group(int64_t t0, float (&v)[kGroupTok]) const {
#pragma unroll
    for (int r = 0; r < kGroupTok; ++r) v[r] = t0 + r < n ? p[t0 + r] : 0.0f;
  }
};
struct TileScores {  // quad_order(G, n) false
  const float *p;
  int64_t n;
  __device__ __forceinline__ TileScores(const float *scores, int64_t n_, int64_t)
      : p(scores + blockIdx.x * tile_score_floats(n_)), n(n_) {}
  __device__ __forceinline__ float operator[](int64_t i) const { return p[i]; }
  __device__ __forceinline__ void group(int64_t t0, float (&v)[kGroupTok]) const {
    if (t0 < n) load_quads(p + t0, 4, v);  // rows end on a whole block
  }
};
struct QuadScores {  // quad_order(G, n) true
  const float *p;    // the (batch, KV head) row's tiles
  int64_t n;
  int G, h;
  __device__ __forceinline__ QuadScores(const float *scores, int64_t n_, int64_t G_)
      : p(scores + (int64_t)(blockIdx.x / (uint32_t)G_) * G_ * tile_score_floats(n_)),
        n(n_), G((int)G_), h((int)(blockIdx.x % (uint32_t)G_)) {}
  __device__ __forceinline__ int64_t quad_at(int64_t i) const {  // the quad that holds token i
    const int64_t beta0 = i / kRegTok * (kRegTok / kBlk);
    return beta0 * (int64_t)(kBlk * G) + quad_off((uint32_t)cdiv(n, kBlk), (uint32_t)G, (uint32_t)h, (uint32_t)beta0, (uint32_t)(i - beta0 * kBlk));
  }
  __device__ __forceinline__ float operator[](int64_t i) const { return p[quad_at(i) + (i & 3)]; }
  __device__ __forceinline__ void group(int64_t t0, float (&v)[kGroupTok]) const {
    if (t0 >= n) return;
    const int64_t q0 = quad_at(t0);
    load_quads(p + q0, quad_at(t0 + 4) - q0, v);
  }
};

// Ranks the cnt <= 4096 (WIDE: 8192) candidates in cl (also the sort's scratch)
// into out.
template <bool LINEAR, bool WIDE>
__device__ __forceinline__ void rank_cands(uint64_t *cl, uint32_t cnt, RowOut &out, RangeShared &sh) {
  int nlim = kWave;
  while (nlim < (int)cnt) nlim <<= 1;
  out.got = (int64_t)cnt < out.kk ? (int)cnt : (int)out.kk;
  const auto rank_all = [&](auto per) {
    constexpr int E = decltype(per)::value;
    uint64_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint32_t i = threadIdx.x + (uint32_t)e * kFinThreads;
      v[e] = i < cnt ? cl[i] : 0ull;
    }
    __syncthreads();
    const auto put = [&](int rank, uint64_t x) { out.put(rank, x); };
    if (!bin_rank_desc<E, LINEAR>(v, (int)cnt, out.got, cl, sh, nlim, put)) {
      __syncthreads();  // scratch is rewritten
      bin_rank_desc<E>(v, (int)cnt, out.got, cl, sh, nlim, put);
    }
  };
  if (WIDE && cnt > (uint32_t)(4 * kFinThreads)) rank_all(std::integral_constant<int, 8>{});
  else if (!WIDE && cnt <= (uint32_t)(2 * kFinThreads)) rank_all(std::integral_constant<int, 2>{});
  else rank_all(std::integral_constant<int, 4>{});
}

// The range of the finite keys of E per thread (0: no key), and sh.hist cleared.
template <int E>
__device__ __forceinline__ void key_range(const uint32_t (&key)[E], uint32_t &lo, uint32_t &hi, RangeShared &sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = kFinThreads >> 6;
  uint32_t mn = ~0u, mx = 0u;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (finite_key(key[e])) {
      mn = min(mn, key[e]);
      mx = max(mx, key[e]);
    }
  wave_minmax_u32(mn, mx);
  if (lane == 0) {
    sh.wmin[wave] = mn;
    sh.wmax[wave] = mx;
  }
  sh.hist[tid] = sh.hist[tid + kFinThreads] = 0u;
  __syncthreads();
  lo = ~0u;
  hi = 0u;
  for (int w = 0; w < nw; ++w) {
    lo = min(lo, (uint32_t)sh.wmin[w]);
    hi = max(hi, (uint32_t)sh.wmax[w]);
  }
}

// The bin that holds the need-th largest of the keys (at least need of them),
// after key_range.
template <int E, typename Bins>
__device__ __forceinline__ uint32_t rank_bin(const uint32_t (&key)[E], uint32_t need, const Bins &bins, RangeShared &sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (key[e]) atomicAdd(&sh.hist[bins.of(key[e])], 1u);
  __syncthreads();
  // running counts from the top bin down: thread t holds bins 2047 - 2t, 2046 - 2t
  const uint32_t c0 = sh.hist[kBins - 1 - 2 * tid], c1 = sh.hist[kBins - 2 - 2 * tid], c = c0 + c1;
  const uint32_t wi = wave_incl_scan_u32(c);
  if (lane == kWave - 1) sh.wsum[wave] = wi;
  __syncthreads();
  uint32_t above = wi - c;
  for (int w = 0; w < wave; ++w) above += sh.wsum[w];
  if (above < need && above + c0 >= need) sh.hsel = (uint32_t)(kBins - 1 - 2 * tid);
  if (above + c0 < need && above + c >= need) sh.hsel = (uint32_t)(kBins - 2 - 2 * tid);
  __syncthreads();
  return sh.hsel;
}

// The keys in bin b and above: their count, and the place of the thread's first.
template <int E, typename Bins>
__device__ __forceinline__ uint32_t place_from_bin(const uint32_t (&key)[E], uint32_t b, const Bins &bins, uint32_t &off,
                                                   RangeShared &sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = kFinThreads >> 6;
  uint32_t own = 0u, cnt = 0u;
#pragma unroll
  for (int e = 0; e < E; ++e) own += key[e] && bins.of(key[e]) >= b ? 1u : 0u;
  const uint32_t wi = wave_incl_scan_u32(own);
  if (lane == kWave - 1) sh.wsum[wave] = wi;
  __syncthreads();
  off = wi - own;
  for (int w = 0; w < nw; ++w) {
    const uint32_t s = sh.wsum[w];
    off += w < wave ? s : 0u;
    cnt += s;
  }
  return cnt;
}

// Value sources of the narrowed selection: for_each(f) calls f(ok, key, token) for
// every value, in loops that are uniform per wave.
// Keys held in registers, thread t those of tokens t + 1024 e (0: none).
template <int E>
struct RegSrc {
  const uint32_t (&key)[E];
  template <typename F>
  __device__ __forceinline__ void for_each(F f) const {
#pragma unroll
    for (int e = 0; e < E; ++e) f(key[e] != 0u, key[e], threadIdx.x + (uint32_t)e * kFinThreads);
  }
};
// The unmasked tokens [sink, sink + len) of a row of n.
struct Unmasked {
  uint32_t sink, len;
  __device__ __forceinline__ Unmasked(int64_t n, int64_t s, int64_t lstart)
      : sink((uint32_t)min(s, n)), len((uint32_t)max(min(lstart, n) - min(s, n), (int64_t)0)) {}
  __device__ __forceinline__ uint32_t key(float v, uint32_t tok) const {
    return tok - sink < len ? score_key(v) : kKeyNegInf;
  }
};
// A row's scores, read anew on each pass.
template <typename Scores>
struct RowSrc {
  const Scores &rs;
  uint32_t n;
  Unmasked um;
  template <typename F>
  __device__ __forceinline__ void for_each(F f) const {
    constexpr int kU = 8;
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t w0 = threadIdx.x - lane; w0 < n; w0 += kU * kFinThreads) {  // uniform per wave
      float v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t i = w0 + lane + u * kFinThreads;
        v[u] = i < n ? rs[i] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t i = w0 + lane + u * kFinThreads;
        f(i < n, um.key(v[u], i), i);
      }
    }
  }
};
// The listed groups of a row: a wave takes 64 of them, 16 lanes each.
template <typename Scores>
struct GroupSrc {
  const Scores &rs;
  const uint16_t *list;
  uint32_t ngr, n;
  Unmasked um;
  template <typename F>
  __device__ __forceinline__ void for_each(F f) const {
    constexpr int kU = 8;
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t e0 = threadIdx.x - lane; e0 < ngr; e0 += kFinThreads) {  // uniform per wave
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t tok[kU];
        float v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const uint32_t e = e0 + (uint32_t)(4 * (kU * h + u)) + lane / kGroupTok;
          tok[u] = e < ngr ? (uint32_t)list[e] * (uint32_t)kGroupTok + lane % kGroupTok : n;
          v[u] = tok[u] < n ? rs[tok[u]] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) f(tok[u] < n, um.key(v[u], tok[u]), tok[u]);
      }
    }
  }
};

// A value into a bin of sh.hist: the lanes of a wave that share the first one's
// bin are added at once (equal scores would serialise on one LDS counter).
__device__ __forceinline__ void count_bin(bool in, uint32_t b, RangeShared &sh) {
  const uint64_t m = __ballot(in);
  if (m == 0ull) return;  // uniform per wave
  const int first = __ffsll((unsigned long long)m) - 1;
  const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)b, first);
  const uint32_t same = (uint32_t)__popcll(__ballot(in && b == b0));
  const bool lead = (threadIdx.x & 63) == (uint32_t)first;
  if (in && (lead || b != b0)) atomicAdd(&sh.hist[b], lead ? same : 1u);
}

// Where more of src's values with keys in [klo, khi] reach the first bound than one
// sort takes (ties, groups that hold several top keys): the top kk of them (at least
// kk, none of a higher key).  Each round counts the range in 2048 bins and keeps the
// bin that holds the kk-th: of keys, then, once the range is one key, of its tokens;
// as soon as at most cap >= kk values lie in that bin and above they are gathered in
// cl (which src does not read below cap) and sorted.  One workgroup works its way
// through the values at about 25 instructions each and pass, so there are as few
// passes as can be: two for a row of equal scores.
template <bool WIDE, typename Src>
__device__ __forceinline__ bool select_narrowed(const Src &src, uint32_t klo, uint32_t khi, int64_t n, uint32_t cap,
                                                RowOut &out, uint64_t *cl, RangeShared &sh, uint32_t &s_cnt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t kk = (uint32_t)out.kk;
  uint32_t above = 0u, tlo = 0u, thi = (uint32_t)(n - 1);  // values above the range; tokens of a range of one key
  for (;;) {  // uniform; a round takes 11 bits off the range or ends on one key
    const bool one = klo == khi;
    const uint32_t R = one ? thi - tlo : khi - klo;
    const int bl = R ? 32 - __clz((int)R) : 0, s = bl > 11 ? bl - 11 : 0;
    __syncthreads();  // hist, hsel and hcnt are read
    sh.hist[tid] = sh.hist[tid + kFinThreads] = 0u;
    if (tid == 0) sh.hsel = sh.hcnt = sh.need = 0u;
    __syncthreads();
    if (one) src.for_each([&](bool ok, uint32_t key, uint32_t tok) {
      count_bin(ok && key == klo && tok - tlo <= R, kBins - 1 - ((tok - tlo) >> s), sh);
    });
    else src.for_each([&](bool ok, uint32_t key, uint32_t) { count_bin(ok && key - klo <= R, (key - klo) >> s, sh); });
    __syncthreads();
    // running counts from the top bin down: thread t holds bins 2047 - 2t, 2046 - 2t
    const uint32_t c0 = sh.hist[kBins - 1 - 2 * tid], c1 = sh.hist[kBins - 2 - 2 * tid], c = c0 + c1;
    const uint32_t wi = wave_incl_scan_u32(c);
    if (lane == kWave - 1) sh.wsum[wave] = wi;
    __syncthreads();
    uint32_t ab = above + wi - c;
    for (int w = 0; w < wave; ++w) ab += sh.wsum[w];
    if (ab < kk && ab + c0 >= kk) {
      sh.hsel = (uint32_t)(kBins - 1 - 2 * tid);
      sh.need = ab;
      sh.hcnt = ab + c0;
    } else if (ab + c0 < kk && ab + c >= kk) {
      sh.hsel = (uint32_t)(kBins - 2 - 2 * tid);
      sh.need = ab + c0;
      sh.hcnt = ab + c;
    }
    __syncthreads();
    const uint32_t width = (1u << s) - 1u;
    if (one) {
      tlo += (uint32_t)(kBins - 1 - sh.hsel) << s;
      thi = min(thi, tlo + width);
    } else {
      klo += sh.hsel << s;
      khi = khi - klo > width ? klo + width : khi;
    }
    if (sh.hcnt <= cap || (one && s == 0)) break;
    above = sh.need;
  }
  if (tid == 0) s_cnt = 0u;
  __syncthreads();
  src.for_each([&](bool ok, uint32_t key, uint32_t tok) {
    lds_append(ok && (key > klo || (key == klo && tok <= thi)), k64_of(key, tok), &s_cnt, cl, cap, lane);
  });
  __syncthreads();
  rank_cands<false, WIDE>(cl, min(s_cnt, cap), out, sh);
  return out.finish();
}
// The range of src's keys.
template <typename Src>
__device__ __forceinline__ void key_span(const Src &src, uint32_t &mn, uint32_t &mx, RangeShared &sh) {
  mn = ~0u;
  mx = 0u;
  src.for_each([&](bool ok, uint32_t key, uint32_t) {
    mn = ok ? min(mn, key) : mn;
    mx = ok ? max(mx, key) : mx;
  });
  wave_minmax_u32(mn, mx);
  __syncthreads();  // wmin and wmax are read
  if ((threadIdx.x & 63) == 0) {
    sh.wmin[threadIdx.x >> 6] = mn;
    sh.wmax[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  for (int w = 0; w < kFinThreads / kWave; ++w) {
    mn = min(mn, (uint32_t)sh.wmin[w]);
    mx = max(mx, (uint32_t)sh.wmax[w]);
  }
}

// Exact top kk of a short row, read whole: up to 4096 tokens are ranked at once
// (E values per thread); longer rows first keep the scores of the bin that
// holds the kk-th largest and above, 2048 linear bins over the finite scores'
// range (kk and a few of them for spread scores; where they outgrow the sort, or the
// bins of a row of up to 4096 crowd, the bound is narrowed).
template <int E, bool WIDE, typename Scores>
__device__ __forceinline__ bool rowrank_row(const Scores &rs, int64_t n, RowOut &out, uint64_t *cl, RangeShared &sh,
                                            uint32_t &s_cnt) {
  const int tid = threadIdx.x;
  const int64_t kk = out.kk, sink = out.sink;
  const int64_t lstart = (out.m - out.local) > 0 ? (out.m - out.local) : 0;
  uint32_t key[E];  // 0: no candidate (below every score's key)
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t i = tid + (int64_t)e * kFinThreads;
    key[e] = i < n ? masked_key(rs, i, sink, lstart) : 0u;
  }
  const auto k64 = [&](int e) { return key[e] ? k64_of(key[e], tid + (int64_t)e * kFinThreads) : 0ull; };
  if constexpr (E <= 4) {
    uint64_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = k64(e);
    int nlim = kWave;
    while (nlim < (int)n) nlim <<= 1;
    out.got = (int)kk;
    if (!bin_rank_desc<E, true>(v, (int)n, out.got, cl, sh, nlim, [&](int rank, uint64_t x) { out.put(rank, x); })) {
      uint32_t cap = kFinThreads / 2;  // many equal scores: the fewer are sorted the better
      while (cap < (uint32_t)kk) cap <<= 1;
      uint32_t klo, khi;
      key_span(RegSrc<E>{key}, klo, khi, sh);
      return select_narrowed<false>(RegSrc<E>{key}, klo, khi, n, cap, out, cl, sh, s_cnt);
    }
    return out.finish();
  }
  uint32_t lo, hi;
  key_range<E>(key, lo, hi, sh);
  const LinearBins bins(lo, hi);
  const uint32_t b = rank_bin<E>(key, (uint32_t)kk, bins, sh);  // n >= kk keys are counted
  uint32_t off;
  const uint32_t cnt = place_from_bin<E>(key, b, bins, off, sh);
  constexpr uint32_t kSort = (WIDE ? 8 : 4) * kFinThreads;
  if (cnt > kSort) {  // uniform: ties, or a range that outliers stretch
    const RowSrc<Scores> src{rs, (uint32_t)n, Unmasked(n, sink, lstart)};
    uint32_t klo, khi;
    key_span(src, klo, khi, sh);
    return select_narrowed<WIDE>(src, klo, khi, n, kSort, out, cl, sh, s_cnt);
  }
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (key[e] && bins.of(key[e]) >= b) cl[off++] = k64(e);
  __syncthreads();
  // scores of both signs: linear bins again; a tail of positive ones: the keys'
  if (bins.positive(b)) rank_cands<false, WIDE>(cl, cnt, out, sh);
  else rank_cands<true, WIDE>(cl, cnt, out, sh);
  return out.finish();
}
// The rows that rowrank_row takes: short ones, and those with few groups per
// selected key, whose maxima bound little.  sink_local_topk of 32 rows, us, by
// group maxima (with their pass) and read whole: n = 1000, kk = 92 17.2; 4.9, 4096,
// 476 20; 7.8, 8192, 264 13.9; 11.2, 8192, 476 15.9; 11.3, 14000, 476 15.2; 17.4, 16384,
// 988 21.5; 18.7, 32768, 1064 21.6; 26.0, 32768, 2012 38.0; 26.7.
inline bool rowrank_takes(int64_t n, int64_t kk) {
  const int64_t ngrp = cdiv(n, kGroupTok);
  return n <= 4 * kFinThreads || (n <= 8 * kFinThreads && ngrp <= 2 * kk) || (n <= kRowSelectMax && 4 * ngrp <= 5 * kk);
}

// Exact top kk of short score rows whose 16-token group maxima the scan
// wrote beside them (gmax [rows, ceil(n / 16)]: the largest masked key of each
// group).  T, a lower bound of the kk-th largest group maximum, bounds the
// row's kk-th largest key from below (kk groups each hold a key >= T), and
// every key >= T lies in a group whose maximum is >= T: only those groups'
// scores are read, and their keys >= T are the candidates (a little over kk
// for spread scores).  Up to 4096 (WIDE: 8192) candidates are ranked by one sort;
// more are first cut to those of the key bin that holds the kk-th and above.  Where
// neighbouring tokens score alike a group holds several top keys and T falls, to
// 16 kk candidates at worst, and ties reach T in any number: more than the LDS list
// holds narrow T over the listed groups, a few passes over them; where no key is
// past T, the first kk tokens of that key are the answer.  sink_local_topk of 32
// rows, us, with the whole row selected in those cases and now: scores of
// correlation length 64 tokens, n = 131072, k = 2048 191; 51, 300007, 4096 734; 90, all
// equal, 131072, 512 489; 24.  Scan + top-k of 8 x 4 heads of 131072 with one query
// row of zeros, k = 512: 485; 33.
constexpr int kGroupList = (int)(sizeof(uint64_t) * kMaxK / sizeof(uint16_t));  // groups listed in ss
constexpr int kGroupListAll = kCandLds / 2 * (int)(sizeof(uint64_t) / sizeof(uint16_t));  // in cl's upper half
static_assert(kGmaxSelectMax / kGroupTok <= kGroupList && kGmaxWideMax / kGroupTok <= kGroupListAll &&
                  kGmaxWideMax / kGroupTok <= 65536,
              "every group can be listed, in 16 bits");
// The top kk of a row whose largest key is T and whose groups reach it at least kk
// times: the first kk tokens of that key, from the row's start on until they are found.
template <typename Scores>
__device__ __forceinline__ bool take_first(const Scores &rs, const uint32_t *__restrict__ gm, uint32_t n, const Unmasked &um,
                                           uint32_t T, RowOut &out, RangeShared &sh) {
  constexpr int kU = 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = kFinThreads >> 6;
  const uint32_t kk = (uint32_t)out.kk, ngrp = (uint32_t)cdiv(n, kGroupTok);
  out.got = (int)kk;
  uint32_t got = 0u;
  for (uint32_t c0 = 0; c0 < n && got < kk; c0 += kU * kFinThreads) {  // uniform
    const uint32_t w0 = c0 + (uint32_t)wave * (kU * kWave), g = w0 / kGroupTok + lane;
    uint64_t m[kU] = {};
    uint32_t hits = 0u;
    if (__ballot(g < ngrp && gm[min(g, ngrp - 1u)] >= T) != 0ull) {  // uniform per wave
      float v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = w0 + u * kWave + lane < n ? rs[w0 + u * kWave + lane] : 0.0f;
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t tok = w0 + u * kWave + lane;
        m[u] = __ballot(tok < n && um.key(v[u], tok) == T);
        hits += (uint32_t)__popcll(m[u]);
      }
    }
    if (lane == 0) sh.wsum[wave] = hits;
    __syncthreads();
    uint32_t off = got;
    for (int w = 0; w < nw; ++w) {
      const uint32_t ws = sh.wsum[w];
      off += w < wave ? ws : 0u;
      got += ws;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t tok = w0 + u * kWave + lane;
      if ((m[u] >> lane) & 1ull) out.put((int)min(off + (uint32_t)__popcll(m[u] & ((1ull << lane) - 1ull)), kk), k64_of(T, tok));
      off += (uint32_t)__popcll(m[u]);
    }
    __syncthreads();  // sh.wsum is rewritten
  }
  out.got = (int)min(got, kk);
  return out.finish();
}

// The row's k output tokens are left in out.ranked too, where it is given.
template <int kPer, bool WIDE, typename Scores>
__device__ __forceinline__ bool rowselect_gmax_row(const Scores &rs, const uint32_t *__restrict__ gmax, int64_t n,
                                                   RowOut &out, uint64_t *cl, uint64_t *ss, RangeShared &sh,
                                                   uint32_t &s_cnt) {
  uint16_t *glist = reinterpret_cast<uint16_t *>(ss), *glist_all = reinterpret_cast<uint16_t *>(cl + kCandLds / 2);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = kFinThreads >> 6;
  const int64_t row = blockIdx.x;
  const int64_t kk = out.kk, sink = out.sink;
  const int64_t lstart = (out.m - out.local) > 0 ? (out.m - out.local) : 0;
  const int ngrp = (int)cdiv(n, kGroupTok);
  uint32_t gm[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int g = tid + u * kFinThreads;
    gm[u] = g < ngrp ? gmax[row * ngrp + g] : 0u;
  }
  const uint32_t T = ngrp > kk ? kth_bound<kPer>(gm, ngrp, (uint32_t)kk, sh) : 0u;
  // the groups reaching T, listed by thread (groups tid + 1024 u)
  uint32_t ngr = 0u;
  {
    uint32_t c = 0u;
#pragma unroll
    for (int u = 0; u < kPer; ++u) c += (tid + u * kFinThreads < ngrp && gm[u] >= T) ? 1u : 0u;
    const uint32_t wi = wave_incl_scan_u32(c);
    if (lane == kWave - 1) sh.wsum[wave] = wi;
    __syncthreads();
    uint32_t off = wi - c;
    for (int w = 0; w < nw; ++w) {
      const uint32_t ws = sh.wsum[w];
      off += w < wave ? ws : 0u;
      ngr += ws;
    }
    uint16_t *list = WIDE && ngr > (uint32_t)kGroupList ? glist_all : glist;  // uniform
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int g = tid + u * kFinThreads;
      if (g < ngrp && gm[u] >= T) list[off++] = (uint16_t)g;
    }
    __syncthreads();
  }
  constexpr uint32_t kSort = (WIDE ? 8 : 4) * kFinThreads;
  static_assert(kSort <= kCandLds / 2 && kSort <= kGroupList, "gathered below the list in cl");
  static_assert(((int64_t)kCandLds + kGroupTok * 2 * kFinThreads) * kGroupListAll < ((int64_t)1 << 32) &&
                    (int64_t)kCandLds * (kGroupList + 2 * kFinThreads) < ((int64_t)1 << 32),
                "the estimate of the candidates in 32 bits");
  // their keys >= T, kU groups per thread and round, placed by a workgroup prefix sum
  constexpr int kU = WIDE ? 2 : 1;
  uint32_t cnt = ngr <= kSort ? 0u : kCandLds + 1;  // each group has one: more groups than the sort takes are narrowed
  uint32_t e0 = 0;  // read on while the candidates seem to fit (a thread's groups lie 1024 apart: a round is a fair sample)
  for (; e0 < ngr && cnt * ngr <= (uint32_t)kCandLds * e0; e0 += kU * kFinThreads) {  // uniform
    int64_t t0[kU];
    float v[kU][kGroupTok] = {};
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t e = e0 + u * kFinThreads + tid;
      t0[u] = e < ngr ? (int64_t)glist[e] * kGroupTok : n;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) rs.group(t0[u], v[u]);
    uint32_t key[kU][kGroupTok], c = 0u;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int r = 0; r < kGroupTok; ++r) {
        const int64_t i = t0[u] + r;
        key[u][r] = (i < sink || i >= lstart) ? kKeyNegInf : score_key(v[u][r]);
        c += (i < n && key[u][r] >= T) ? 1u : 0u;
      }
    const uint32_t wi = wave_incl_scan_u32(c);
    if (lane == kWave - 1) sh.wsum[wave] = wi;
    __syncthreads();
    uint32_t off = cnt + wi - c;
    for (int w = 0; w < nw; ++w) {
      const uint32_t ws = sh.wsum[w];
      off += w < wave ? ws : 0u;
      cnt += ws;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int r = 0; r < kGroupTok; ++r) {
        const int64_t i = t0[u] + r;
        if (i < n && key[u][r] >= T) {
          if (off < (uint32_t)kCandLds) cl[off] = k64_of(key[u][r], i);
          ++off;
        }
      }
    __syncthreads();  // sh.wsum is rewritten by the next step
  }
  if (e0 < ngr) cnt = kCandLds + 1;
  if (cnt > kSort && cnt <= (uint32_t)kCandLds) {  // uniform: the candidates in registers, cut by key bins
    constexpr int kHold = kCandLds / kFinThreads;
    static_assert(kHold * kFinThreads == kCandLds, "cl held in registers");
    uint64_t v[kHold];
    uint32_t key[kHold], lo, hi, off;
#pragma unroll
    for (int e = 0; e < kHold; ++e) {
      const uint32_t i = tid + (uint32_t)e * kFinThreads;
      v[e] = i < cnt ? cl[i] : 0ull;
      key[e] = (uint32_t)(v[e] >> 32);
    }
    key_range<kHold>(key, lo, hi, sh);
    const KeyBins bins(lo, hi);
    const uint32_t b = rank_bin<kHold>(key, (uint32_t)kk, bins, sh);
    const uint32_t kept = place_from_bin<kHold>(key, b, bins, off, sh);
    cnt = kept <= kSort ? kept : kCandLds + 1;
    if (kept <= kSort) {  // uniform; every thread has read cl
#pragma unroll
      for (int e = 0; e < kHold; ++e)
        if (key[e] && bins.of(key[e]) >= b) cl[off++] = v[e];
    }
    __syncthreads();
  }
  if (cnt > kSort) {  // uniform: keys from T to the largest group maximum
    uint32_t bot = ~0u, top = 0u;
    for (int g = tid; g < ngrp; g += kFinThreads) top = max(top, gmax[row * ngrp + g]);
    wave_minmax_u32(bot, top);
    if (lane == 0) sh.wmax[wave] = top;
    __syncthreads();
    for (int w = 0; w < nw; ++w) top = max(top, (uint32_t)sh.wmax[w]);
    if (top == T) return take_first(rs, gmax + row * ngrp, (uint32_t)n, Unmasked(n, sink, lstart), T, out, sh);
    const GroupSrc<Scores> src{rs, WIDE && ngr > (uint32_t)kGroupList ? glist_all : glist, ngr, (uint32_t)n,
                               Unmasked(n, sink, lstart)};
    return select_narrowed<WIDE>(src, T, top, n, kSort, out, cl, sh, s_cnt);
  }
  rank_cands<false, WIDE>(cl, cnt, out, sh);  // one sort ranks them
  return out.finish();
}

// A row's selection, one workgroup per row: rowrank_row with E tokens per thread,
// or (E = 0) rowselect_gmax_row with kPer groups per thread.  ATTN (the decode
// step's selection + attention, k <= 512, rows in device memory): the
// workgroup then runs the attention of its query head over the k indices it
// wrote, exactly as gather_attention's attn_stream_kernel does for one split
// (16 waves of 32 positions), so out equals gather_attention's output.
template <typename Scores, bool ATTN, bool WIDE, int kPer, int E>
__global__ __launch_bounds__(kFinThreads) void rowselect_kernel(const float *__restrict__ scores, int64_t G,
                                                                const uint32_t *__restrict__ gmax, int64_t n, int64_t m,
                                                                int64_t k, int64_t sink, int64_t local,
                                                                int64_t *__restrict__ idx, RowAttn ra) {
  __shared__ uint64_t cl[kCandLds];
  __shared__ uint64_t ss[kMaxK];
  __shared__ RangeShared sh;
  __shared__ uint32_t s_cnt;
  static_assert(!ATTN || !WIDE, "the attention's tokens lie past a sort of 4096");
  int32_t *ranked = ATTN ? ranked_lds(cl) : nullptr;
  RowOut ro{idx + blockIdx.x * k, k - sink - local, m, sink, local, ranked, 0};
  const Scores rs(scores, n, G);
  bool in_lds;
  if constexpr (E > 0) in_lds = rowrank_row<E, WIDE>(rs, n, ro, cl, sh, s_cnt);
  else in_lds = rowselect_gmax_row<kPer, WIDE>(rs, gmax, n, ro, cl, ss, sh, s_cnt);
  if constexpr (ATTN) row_attention(ra, idx + blockIdx.x * k, k, in_lds, ranked, cl);
}

// The wide selection's kk <= 8192 values of a row (sel [rows, P], all
// distinct) ranked by one counting sort and written as the row's indices, then
// the sink and local positions.
template <int E>
__global__ __launch_bounds__(kFinThreads) void rank_list_kernel(const uint64_t *__restrict__ sel, int64_t P, int64_t kk,
                                                               int64_t m, int64_t k, int64_t sink, int64_t local,
                                                               int64_t *__restrict__ idx) {
  __shared__ uint64_t cl[kCandLds];
  __shared__ RangeShared sh;
  static_assert(E * kFinThreads + kBins <= kCandLds, "the sort's scratch");
  const int64_t row = blockIdx.x;
  const uint64_t *src = sel + row * P;
  uint64_t v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int64_t i = threadIdx.x + e * kFinThreads;
    v[e] = i < kk ? src[i] : 0ull;
  }
  int nlim = kWave;
  while (nlim < (int)kk) nlim <<= 1;
  int64_t *out = idx + row * k;
  bin_rank_desc<E>(v, (int)kk, (int)kk, cl, sh, nlim,
                   [&](int rank, uint64_t x) { out[rank] = (int64_t)(0xFFFFFFFFu - (uint32_t)x); });
  write_fixed(out, (int)kk, kk, m, sink, local);
}

__global__ __launch_bounds__(256) void fixed_only_kernel(int64_t rows, int64_t m, int64_t k, int64_t sink,
                                                         int64_t local, int64_t *__restrict__ idx) {
  const int64_t total = rows * k;
  for (int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x; o < total; o += (int64_t)gridDim.x * 256) {
    const int64_t i = o % k;
    idx[o] = (i < sink) ? i : (m - local + (i - sink));
  }
}

}  // namespace

size_t topk_sel_layout(int64_t rows, int64_t cand_cap, int64_t nreg, char *base, TopkSel *s) {
  const size_t row_b = ws_align((size_t)rows * 4);                // thr, thr_lo
  const size_t cnt_b = ws_align((size_t)rows * 4 * kCntStride);  // cand_cnt, cand2_cnt
  const size_t reg_b = nreg > 0 ? ws_align((size_t)rows * (size_t)nreg * 4) : 0;  // rc1, rc2
  const size_t cand_b = ws_align((size_t)rows * (size_t)cand_cap * 8);
  if (s) {
    char *p = base;
    s->thr = reinterpret_cast<uint32_t *>(p);
    s->thr_lo = reinterpret_cast<uint32_t *>(p += row_b);
    s->cand_cnt = reinterpret_cast<uint32_t *>(p += row_b);
    s->cand2_cnt = reinterpret_cast<uint32_t *>(p += cnt_b);
    s->rc1 = nreg > 0 ? reinterpret_cast<uint32_t *>(p + cnt_b) : nullptr;
    s->rc2 = nreg > 0 ? reinterpret_cast<uint32_t *>(p + cnt_b + reg_b) : nullptr;
    s->nreg = nreg > 0 ? nreg : 0;
    s->cand = reinterpret_cast<uint64_t *>(p + cnt_b + 2 * reg_b);
    s->cand_cap = cand_cap;
    s->kk = 0u;
  }
  return 2 * row_b + 2 * cnt_b + 2 * reg_b + cand_b;
}

size_t topk_layout(int64_t rows, int64_t n, int64_t k, bool regions, char *base, uint32_t **samp, int64_t *samp_cap,
                   TopkSel *sel, int64_t *S_out) {
  const int64_t kk = k > 0 ? k : 0;
  const int64_t tile = regions ? kRegTok : kTileTok;
  const int64_t S = topk_tile_stride(n, kk, tile);
  // the fused scan's sample holds each tile's 64 group maxima, the score-row
  // top-k's every sampled key
  const int64_t cap = topk_sample_tiles(n, S, tile) * (regions ? kRegTok / kGroupTok : tile);
  const size_t samp_b = ws_align((size_t)rows * (size_t)cap * 4);
  if (samp) *samp = reinterpret_cast<uint32_t *>(base);
  if (samp_cap) *samp_cap = cap;
  if (S_out) *S_out = S;
  const int64_t cand_cap = regions ? cdiv(n, 4 * kRegTok) * 4 * kRegTok : n;
  return samp_b + topk_sel_layout(rows, cand_cap, regions ? cand_cap / kRegTok : 0, base ? base + samp_b : nullptr, sel);
}

int launch_select_keys(const uint32_t *samp, int64_t rows, int64_t samp_cap, int64_t kk, int64_t r_hi, TopkSel s,
                       hipStream_t st) {
  if (samp_cap > kMaxSample) return fail(FATHOM_ERR_INVALID, "select: %lld sampled keys exceed %lld", (long long)samp_cap, (long long)kMaxSample);
  const unsigned g = (unsigned)rows;
  const uint32_t ukk = (uint32_t)kk, urh = (uint32_t)r_hi;
  const int64_t ng = samp_cap / 16;
  if (samp_cap % 16 == 0 && ng >= 4 * kk && kk > 0) {  // 16-key group maxima (see select_groups_kernel)
    if (ng <= kSelThreads)
      select_groups_kernel<1, false><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
    else if (ng <= 2 * kSelThreads)
      select_groups_kernel<2, false><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
    else
      select_groups_kernel<4, false><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
    return launch_status("select_groups_kernel");
  }
  if (samp_cap <= 16 * kSelThreads)  // the chains' rows sample 10240 keys or more
    select_keys_kernel<16><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
  else if (samp_cap <= 32 * kSelThreads)
    select_keys_kernel<32><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
  else
    select_keys_kernel<kSelPer><<<g, kSelThreads, 0, st>>>(samp, samp_cap, ukk, urh, s);
  return launch_status("select_keys_kernel");
}

int launch_select_groups(const uint32_t *gmax, int64_t rows, int64_t ng, int64_t kk, int64_t r_hi, TopkSel s,
                         hipStream_t st) {
  if (ng > 4 * kSelThreads) return fail(FATHOM_ERR_INVALID, "select: %lld group maxima exceed %d", (long long)ng, 4 * kSelThreads);
  const unsigned g = (unsigned)rows;
  const uint32_t ukk = (uint32_t)kk, urh = (uint32_t)r_hi;
  if (ng <= 2 * kSelThreads)  // the chain's rows have 1664 sampled maxima or more
    select_groups_kernel<2, true><<<g, kSelThreads, 0, st>>>(gmax, ng, ukk, urh, s);
  else
    select_groups_kernel<4, true><<<g, kSelThreads, 0, st>>>(gmax, ng, ukk, urh, s);
  return launch_status("select_groups_kernel");
}

int launch_sample_scores(const float *scores, int64_t rows, int64_t n, int64_t S, int64_t sink, int64_t lstart,
                         uint32_t *samp, int64_t samp_cap, hipStream_t st) {
  sample_scores_kernel<<<dim3((unsigned)(samp_cap / kTileTok), (unsigned)rows), 256, 0, st>>>(scores, n, S, sink,
                                                                                            lstart, samp, samp_cap);
  return launch_status("sample_scores_kernel");
}

// One step of 4096 scores per workgroup (16 loads of a thread in flight); launches of
// 2^24 scores and more take 16 steps of 1024 (4 loads in flight, a quarter of the
// counter atomics).  sink_local_topk, k = 512, us, 16384 scores per workgroup with a
// load per step, and now: 32 rows of 200001 tokens 55.2; 37.7, 4 of 140000 40.6; 31.5, 32
// of 300007 57.8; 40.4, 16 of 1048577 56.3; 43.9, 32 of 1048576 49.9; 49.9 (54.6 in single
// steps of 4096).
int launch_filter_scores(const float *scores, int64_t rows, int64_t n, int64_t sink, int64_t lstart, TopkSel s,
                         bool fallback, hipStream_t st) {
  const bool large = rows * n >= (int64_t)1 << 24;
  const int steps = large ? 16 : 1;
  const dim3 grid((unsigned)cdiv(n, 16 * kFilterThreads * (large ? 4 : 1)), (unsigned)rows);
  const bool vec = n % 4 == 0 && reinterpret_cast<uintptr_t>(scores) % 16 == 0;
  const auto run = [&](auto kernel) { kernel<<<grid, kFilterThreads, 0, st>>>(scores, n, sink, lstart, s, fallback, steps); };
  if (large) vec ? run(filter_scores_kernel<true, 4>) : run(filter_scores_kernel<false, 4>);
  else vec ? run(filter_scores_kernel<true, 16>) : run(filter_scores_kernel<false, 16>);
  return launch_status("filter_scores_kernel");
}

namespace {
RowAttn row_attn(const AttnArgs &t, int64_t n) {
  return RowAttn{t.q, t.G, attn::RowSrc{(const char *)t.K, (const char *)t.V, nullptr, nullptr, t.cap, 0, n, 2 * attn::kAttnD},
                 t.scale, t.out};
}
}  // namespace

int launch_finalize(int64_t rows, int64_t m, int64_t k, int64_t sink, int64_t local, TopkSel s, int64_t *idx,
                    hipStream_t st) {
  finalize_kernel<<<(unsigned)rows, kFinThreads, 0, st>>>(m, k, sink, local, s, idx);
  return launch_status("finalize_kernel");
}

int launch_finalize_fused(const sc::ScanArgs &a, const sc::Emit &em, int64_t rows, int64_t m, int64_t k, int64_t sink,
                          int64_t local, int64_t *idx, const AttnArgs *att, hipStream_t st) {
  if (att)
    finalize_fused_kernel<true><<<(unsigned)rows, kFinThreads, 0, st>>>(m, k, sink, local, a, em, idx, row_attn(*att, a.n));
  else
    finalize_fused_kernel<false><<<(unsigned)rows, kFinThreads, 0, st>>>(m, k, sink, local, a, em, idx, RowAttn{});
  return launch_status("finalize_fused_kernel");
}

namespace {
template <typename Scores, bool ATTN>
int launch_row_select(const float *scores, int64_t G, const uint32_t *gmax, int64_t rows, int64_t n, int64_t m, int64_t k,
                      int64_t sink, int64_t local, int64_t *idx, const RowAttn &ra, hipStream_t st) {
  static_assert(kRowSelectMax == 2 * kFinThreads * kGroupTok && kGmaxSelectMax == 8 * kFinThreads * kGroupTok &&
                    kGmaxWideMax == 32 * kFinThreads * kGroupTok,
                "groups per thread");
  const int64_t kk = k - sink - local;
  if (!group_select_takes(n, kk) || (ATTN && kk > kSelMaxK))
    return fail(FATHOM_ERR_INVALID, "row selection: n=%lld kk=%lld not taken", (long long)n, (long long)kk);
  const unsigned g = (unsigned)rows;
  const auto run = [&](auto kernel) { kernel<<<g, kFinThreads, 0, st>>>(scores, G, gmax, n, m, k, sink, local, idx, ra); };
  const bool wide = kk > kSelMaxK && n > 4 * kFinThreads;
  if (n <= kRowSelectMax) {
    if constexpr (!std::is_same<Scores, QuadScores>::value) {  // quad order: longer rows only
      const bool whole = rowrank_takes(n, kk);
      if (wide) {
        if constexpr (!ATTN) {
          if (whole && n <= 8 * kFinThreads) run(rowselect_kernel<Scores, false, true, 0, 8>);
          else if (whole) run(rowselect_kernel<Scores, false, true, 0, 32>);
          else run(rowselect_kernel<Scores, false, true, 8, 0>);
        }
      } else if (!whole) {
        run(rowselect_kernel<Scores, ATTN, false, 2, 0>);
      } else if (n <= kFinThreads) {
        run(rowselect_kernel<Scores, ATTN, false, 0, 1>);
      } else if (n <= 4 * kFinThreads) {
        run(rowselect_kernel<Scores, ATTN, false, 0, 4>);
      } else if (n <= 8 * kFinThreads) {
        run(rowselect_kernel<Scores, ATTN, false, 0, 8>);
      } else {
        run(rowselect_kernel<Scores, ATTN, false, 0, 32>);
      }
    }
  } else if (wide) {
    if constexpr (!ATTN) {
      if (n <= kGmaxSelectMax) run(rowselect_kernel<Scores, false, true, 8, 0>);
      else run(rowselect_kernel<Scores, false, true, 32, 0>);
    }
  } else {
    run(rowselect_kernel<Scores, ATTN, false, 8, 0>);
  }
  return launch_status("rowselect_kernel");
}
}  // namespace

int launch_rowselect_gmax(const float *scores, const uint32_t *gmax, int64_t rows, int64_t G, int64_t n, int64_t m,
                          int64_t k, int64_t sink, int64_t local, int64_t *idx, const AttnArgs *att, hipStream_t st) {
  const RowAttn ra = att ? row_attn(*att, n) : RowAttn{};
  if (att)
    return quad_order(G, n) ? launch_row_select<QuadScores, true>(scores, G, gmax, rows, n, m, k, sink, local, idx, ra, st)
                            : launch_row_select<TileScores, true>(scores, G, gmax, rows, n, m, k, sink, local, idx, ra, st);
  return quad_order(G, n) ? launch_row_select<QuadScores, false>(scores, G, gmax, rows, n, m, k, sink, local, idx, ra, st)
                          : launch_row_select<TileScores, false>(scores, G, gmax, rows, n, m, k, sink, local, idx, ra, st);
}

int launch_rank_list(const uint64_t *sel, int64_t P, int64_t rows, int64_t kk, int64_t m, int64_t k, int64_t sink,
                     int64_t local, int64_t *idx, hipStream_t st) {
  if (kk > kRankListMax) return fail(FATHOM_ERR_INVALID, "rank_list: kk=%lld exceeds %lld", (long long)kk, (long long)kRankListMax);
  if (kk <= 4 * kFinThreads)
    rank_list_kernel<4><<<(unsigned)rows, kFinThreads, 0, st>>>(sel, P, kk, m, k, sink, local, idx);
  else
    rank_list_kernel<8><<<(unsigned)rows, kFinThreads, 0, st>>>(sel, P, kk, m, k, sink, local, idx);
  return launch_status("rank_list_kernel");
}

int launch_fixed_only(int64_t rows, int64_t m, int64_t k, int64_t sink, int64_t local, int64_t *idx, hipStream_t st) {
  if (k == 0) return FATHOM_OK;
  fixed_only_kernel<<<(unsigned)min(cdiv(rows * k, 256), (int64_t)65535), 256, 0, st>>>(rows, m, k, sink, local, idx);
  return launch_status("fixed_only_kernel");
}

size_t wide_topk_bytes(int64_t rows, int64_t n, int64_t k) {
  return topk_layout(rows, n, k, false, nullptr, nullptr, nullptr, nullptr, nullptr) +
         wide_select_bytes(rows, k < n ? k : n);
}

int wide_topk_run(const float *scores, int64_t rows, int64_t n, int64_t m, int64_t k, int64_t sink, int64_t local,
                  int64_t *idx, void *workspace, size_t workspace_bytes, hipStream_t st) {
  const int64_t kk = k - sink - local;
  const size_t chain = topk_layout(rows, n, k, false, nullptr, nullptr, nullptr, nullptr, nullptr);
  const size_t need = chain + wide_select_bytes(rows, kk);
  if (!workspace || workspace_bytes < need)
    return fail(FATHOM_ERR_WORKSPACE, "top-k (kk=%lld): workspace %zu bytes, need %zu", (long long)kk, workspace_bytes,
                need);
  TopkSel s;
  uint32_t *samp = nullptr;
  int64_t samp_cap = 0, S = 1;
  topk_layout(rows, n, k, false, static_cast<char *>(workspace), &samp, &samp_cap, &s, &S);
  s.kk = (uint32_t)kk;
  const int64_t lstart = (m - local) > 0 ? (m - local) : 0;
  const int64_t r_hi = topk_hi_rank(n, S, kk, kTileTok);
  int rc = launch_sample_scores(scores, rows, n, S, sink, lstart, samp, samp_cap, st);
  if (rc) return rc;
  rc = launch_select_keys(samp, rows, samp_cap, kk, r_hi, s, st);
  if (rc) return rc;
  rc = launch_filter_scores(scores, rows, n, sink, lstart, s, false, st);
  if (rc) return rc;
  if (r_hi < kk) {  // rows whose first pass found fewer than kk take T_lo
    rc = launch_filter_scores(scores, rows, n, sink, lstart, s, true, st);
    if (rc) return rc;
  }
  return wide_select_list(s, rows, m, k, sink, local, idx, static_cast<char *>(workspace) + chain,
                          workspace_bytes - chain, st);
}

int check_topk_args(int64_t rows, int64_t n, int64_t m, int64_t k, int64_t sink, int64_t local, const char *who) {
  if (rows < 1 || rows > 65535) return fail(FATHOM_ERR_INVALID, "%s: rows=%lld outside [1, 65535]", who, (long long)rows);
  if (n < 1 || n > 0x7FFFFFFFLL) return fail(FATHOM_ERR_INVALID, "%s: n=%lld unsupported", who, (long long)n);
  if (sink < 0 || local < 0 || k < 0) return fail(FATHOM_ERR_INVALID, "%s: negative k/sink/local", who);
  const int64_t kk = k - sink - local;
  if (kk < 0) return fail(FATHOM_ERR_INVALID, "%s: k=%lld < sink+local=%lld", who, (long long)k, (long long)(sink + local));
  if (kk > n) return fail(FATHOM_ERR_INVALID, "%s: k - sink - local = %lld exceeds n=%lld", who, (long long)kk, (long long)n);
  if (sink > n || m < n || local > m)
    return fail(FATHOM_ERR_INVALID, "%s: need sink <= n <= m and local <= m (sink=%lld n=%lld m=%lld local=%lld)", who,
                (long long)sink, (long long)n, (long long)m, (long long)local);
  return FATHOM_OK;
}

}  // namespace fathom

using namespace fathom;

namespace fathom {
namespace {
// k bounds kk = k - sink - local from above: where kk may exceed kSelMaxK the
// chain's layout is followed by the wide selection's state.
size_t topk_ws(int64_t rows, int64_t n, int64_t k) {
  return k <= kSelMaxK ? topk_layout(rows, n, k, false, nullptr, nullptr, nullptr, nullptr, nullptr)
                       : wide_topk_bytes(rows, n, k);
}
}  // namespace
}  // namespace fathom

extern "C" size_t fathom_topk_workspace_bytes(int64_t rows, int64_t n, int64_t k) {
  if (rows < 1 || n < 1 || k < 0) return 0;
  return topk_ws(rows, n, k);
}

extern "C" int fathom_sink_local_topk(const float *scores, int64_t rows, int64_t n, int64_t m, int64_t k,
                                      int64_t sink, int64_t local, int64_t *idx, void *workspace,
                                      size_t workspace_bytes, void *stream) {
  if (!scores || !idx) return fail(FATHOM_ERR_INVALID, "sink_local_topk: null pointer");
  int rc = check_topk_args(rows, n, m, k, sink, local, "sink_local_topk");
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  const int64_t kk = k - sink - local;
  if (kk == 0) return launch_fixed_only(rows, m, k, sink, local, idx, st);
  const size_t need = kk > kSelMaxK ? wide_topk_bytes(rows, n, k)
                                    : topk_layout(rows, n, k, false, nullptr, nullptr, nullptr, nullptr, nullptr);
  if (!workspace || workspace_bytes < need)
    return fail(FATHOM_ERR_WORKSPACE, "sink_local_topk: workspace %zu bytes, need %zu", workspace_bytes, need);
  const int64_t lstart = (m - local) > 0 ? (m - local) : 0;
  if (group_select_takes(n, kk)) {
    uint32_t *gmax = static_cast<uint32_t *>(workspace);  // 4 bytes per 16 scores, the layout has 8 per score
    if (!rowrank_takes(n, kk)) {
      group_max_kernel<<<dim3((unsigned)cdiv(n, 256 * kGmaxPer), (unsigned)rows), 256, 0, st>>>(scores, n, sink, lstart, gmax);
      rc = launch_status("group_max_kernel");
    }
    return rc ? rc
              : launch_row_select<RowScores, false>(scores, 1, gmax, rows, n, m, k, sink, local, idx, RowAttn{}, st);
  }
  if (kk > kSelMaxK) return wide_topk_run(scores, rows, n, m, k, sink, local, idx, workspace, workspace_bytes, st);
  TopkSel s;
  uint32_t *samp = nullptr;
  int64_t samp_cap = 0, S = 1;
  topk_layout(rows, n, k, false, static_cast<char *>(workspace), &samp, &samp_cap, &s, &S);
  s.kk = (uint32_t)kk;
  const int64_t r_hi = topk_hi_rank(n, S, kk, kTileTok);
  rc = launch_sample_scores(scores, rows, n, S, sink, lstart, samp, samp_cap, st);
  if (rc) return rc;
  rc = launch_select_keys(samp, rows, samp_cap, kk, r_hi, s, st);
  if (rc) return rc;
  rc = launch_filter_scores(scores, rows, n, sink, lstart, s, false, st);
  if (rc) return rc;
  if (r_hi < kk) {  // T_hi may exceed a row's kk-th largest key
    rc = launch_filter_scores(scores, rows, n, sink, lstart, s, true, st);
    if (rc) return rc;
  }
  return launch_finalize(rows, m, k, sink, local, s, idx, st);
}
