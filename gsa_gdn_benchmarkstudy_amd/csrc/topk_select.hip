// Exact per-row top-k of an fp32 score matrix (the AdaptiveTopKSelector API).
//
// Scores map to order-preserving uint32 keys (score_key: -inf -> -1e9, NaN
// above +inf); ties at the k-th value go to the lowest indices.  One block per
// row, in one of two ways:
//
// topk_sorted_kernel, for GSA_ORDER_SCORE_DESC (by score descending, index
// ascending): a counting sort by value.  The row is read once (into registers
// up to 16384 keys), its valid scores are counted into value-linear bins
// between their minimum and maximum, a suffix scan turns the counts into
// output positions and finds the bin that holds the k-th, the entries of the
// bins above and of that bin are scattered to their bins' places in LDS, and
// each takes its place within its bin by comparing itself with the bin's other
// entries (about two per bin on scores of the indexer).  Invalid (-inf)
// entries follow by index.
//
// topk_general_row, for GSA_ORDER_INDEX_ASC and for the rows the first way
// leaves (bins overfull with ties, an infinite range, NaN, scores at or below
// -1e9): four 8-bit radix passes over the row find the k-th largest key theta
// and how many entries equal to it are taken, then ordered block-wide
// compaction (valid ascending, then invalid), or a bitonic sort in LDS by
// (key desc, index asc).  Such a row pays for the first way's passes too: T = 8192,
// k = 2048, 2048 rows, 37 us on scores of the indexer, 270 with one far outlier or of
// two values, 170 rounded to 50 levels (radix passes for every row: 420 - 540).
//
// What bounds it: the VALU (91 % busy: the bin and the place of every key; LDS 43 %).
// Reading the matrix and writing 9 bytes per selected entry would take 79 us at T =
// 8192, k = 2048 at the rate of a large copy; this takes 110, radix passes and a
// bitonic sort for every row took 1775.
#include "gsa_common.h"

namespace gsa {

template <int kThreads>
struct SelShared {
  uint32_t hist[256];
  uint32_t wave_cnt[2][kThreads / 64];
  uint32_t prefix;
  int need;
};

// Exclusive block-wide prefix count of two predicates over one kThreads-entry
// chunk; returns this thread's ranks and the chunk totals.
template <int kThreads>
__device__ __forceinline__ void block_rank2(SelShared<kThreads>& sm, bool p0, bool p1, int& r0, int& r1,
                                            int& tot0, int& tot1) {
  const int wave = threadIdx.x >> 6;
  const uint64_t m0 = ballot64(p0), m1 = ballot64(p1);
  if ((threadIdx.x & 63) == 0) {
    sm.wave_cnt[0][wave] = (uint32_t)__popcll(m0);
    sm.wave_cnt[1][wave] = (uint32_t)__popcll(m1);
  }
  __syncthreads();
  int b0 = 0, b1 = 0, t0 = 0, t1 = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    const int c0 = (int)sm.wave_cnt[0][w], c1 = (int)sm.wave_cnt[1][w];
    if (w < wave) { b0 += c0; b1 += c1; }
    t0 += c0; t1 += c1;
  }
  r0 = b0 + count_below(m0);
  r1 = b1 + count_below(m1);
  tot0 = t0; tot1 = t1;
  __syncthreads();   // wave_cnt is reused by the next chunk
}

// One row's outputs: `width` entries of which the first k are selected.
template <typename IdxT>
struct TopkOut {
  IdxT* idx;             // the row's indices
  uint8_t* mask;         // the row's mask, or null
  int32_t* count;        // the row's count, or null
};

// Radix select, then compaction or a bitonic sort in sort_buf (the power of
// two above k entries; GSA_ORDER_SCORE_DESC only).
template <int kThreads, typename IdxT>
__device__ void topk_general_row(const float* __restrict__ srow, int Tkv, int k, int order, SelShared<kThreads>& sm,
                                 uint64_t* sort_buf, const TopkOut<IdxT>& out) {
  const int tid = threadIdx.x;
  // ---- radix select: 4 passes of 8 bits, MSB first ----
  if (tid == 0) { sm.prefix = 0u; sm.need = k; }
  for (int level = 0; level < 4; ++level) {
    for (int i = tid; i < 256; i += kThreads) sm.hist[i] = 0u;
    __syncthreads();
    const uint32_t pre = sm.prefix;
    const int hi_shift = 32 - 8 * level, lo_shift = 24 - 8 * level;
    for (int j = tid; j < Tkv; j += kThreads) {
      const uint32_t key = score_key(srow[j]);
      if (level == 0 || (key >> hi_shift) == pre) atomicAdd(&sm.hist[(key >> lo_shift) & 255u], 1u);
    }
    __syncthreads();
    if (tid < 64) {      // one wave: the highest digit d with count(digits >= d) >= need, four digits a lane
      const int need = sm.need;
      int cb[4], own = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) { cb[i] = (int)sm.hist[4 * tid + i]; own += cb[i]; }
      int c = own;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_down(c, o, 64);
        if (tid + o < 64) c += y;
      }
      c -= own;                                  // entries in the digits of the lanes above
#pragma unroll
      for (int i = 3; i >= 0; --i) {
        if (c < need && c + cb[i] >= need) {     // one lane, one digit
          sm.need = need - c;
          sm.prefix = (pre << 8) | (uint32_t)(4 * tid + i);
        }
        c += cb[i];
      }
    }
    __syncthreads();
  }
  const uint32_t theta = sm.prefix;
  const int tie_need = sm.need;

  if (order == GSA_ORDER_INDEX_ASC) {
    // Sweep 1 writes valid selected entries, sweep 2 the invalid ones after them.
    int n_valid = 0;
    for (int sweep = 0; sweep < 2; ++sweep) {
      int ties = 0, written = 0;
      for (int j0 = 0; j0 < Tkv; j0 += kThreads) {
        const int j = j0 + tid;
        float s = 0.f;
        uint32_t key = 0u;
        if (j < Tkv) { s = srow[j]; key = score_key(s); }
        const bool in = j < Tkv;
        const bool tie = in && key == theta;
        int trank, dummy, ttot, dtot;
        block_rank2(sm, tie, false, trank, dummy, ttot, dtot);
        const bool sel = in && (key > theta || (tie && ties + trank < tie_need));
        const bool valid = s != -__builtin_inff();
        const bool mine = sel && (sweep == 0 ? valid : !valid);
        int pos, dummy2, ptot, dtot2;
        block_rank2(sm, mine, false, pos, dummy2, ptot, dtot2);
        const int o = n_valid * sweep + written + pos;
        if (mine && o < k) {
          out.idx[o] = (IdxT)j;
          if (out.mask) out.mask[o] = (uint8_t)(sweep == 0);
        }
        ties += ttot;
        written += ptot;
      }
      if (sweep == 0) n_valid = written;
    }
    if (tid == 0 && out.count) *out.count = n_valid;
    return;
  }
  // Gather the selection into LDS as (key << 32 | ~index), sort descending.
  int kp = 1;
  while (kp < k) kp <<= 1;
  int ties = 0, written = 0;
  for (int j0 = 0; j0 < Tkv; j0 += kThreads) {
    const int j = j0 + tid;
    uint32_t key = 0u;
    if (j < Tkv) key = score_key(srow[j]);
    const bool in = j < Tkv;
    const bool tie = in && key == theta;
    int trank, dummy, ttot, dtot;
    block_rank2(sm, tie, false, trank, dummy, ttot, dtot);
    const bool sel = in && (key > theta || (tie && ties + trank < tie_need));
    int pos, d2, ptot, dt2;
    block_rank2(sm, sel, false, pos, d2, ptot, dt2);
    if (sel && written + pos < kp) sort_buf[written + pos] = ((uint64_t)key << 32) | (uint64_t)(~(uint32_t)j);
    ties += ttot;
    written += ptot;
  }
  for (int i = written + tid; i < kp; i += kThreads) sort_buf[i] = 0ull;  // sorts last
  __syncthreads();
  // bitonic sort, descending
  for (int size = 2; size <= kp; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int q = tid; q < kp / 2; q += kThreads) {           // pair q: entries i and i + stride
        const int i = 2 * q - (q & (stride - 1)), jx = i + stride;
        const uint64_t a = sort_buf[i], c = sort_buf[jx];
        const bool desc = (i & size) == 0;
        if (desc ? (a < c) : (a > c)) { sort_buf[i] = c; sort_buf[jx] = a; }
      }
      __syncthreads();
    }
  }
  int nv_local = 0;
  for (int i = tid; i < k; i += kThreads) {
    // padding entries (key 0) never reach the first k once k are selected;
    // clamp anyway so a short selection cannot index outside the row
    const int j = max(0, min((int)(~(uint32_t)(sort_buf[i] & 0xffffffffull)), Tkv - 1));
    out.idx[i] = (IdxT)j;
    const bool valid = srow[j] != -__builtin_inff();
    if (out.mask) out.mask[i] = (uint8_t)valid;
    nv_local += valid ? 1 : 0;
  }
  if (out.count) {
    if (tid == 0) sm.need = 0;   // reused as the valid-entry total
    __syncthreads();
    if (nv_local) atomicAdd(&sm.need, nv_local);
    __syncthreads();
    if (tid == 0) *out.count = sm.need;
  }
}

// Output rows are `width` entries wide.  Row r selects k = width entries, or
// k = min(k_rows[r], width) when k_rows is given; entries k .. width-1 of a
// row are then index 0 with mask 0.
struct TopkArgs {
  const float* S; int64_t s_sb, s_st;
  int T, Tkv, width;
  const int32_t* k_rows;
  int32_t* count_out;
  uint8_t* mask_out;
};

template <typename IdxT>
__device__ __forceinline__ TopkOut<IdxT> topk_row_out(const TopkArgs& p, IdxT* idx_out, int row, int k, int threads) {
  TopkOut<IdxT> out;
  out.idx = idx_out + (int64_t)row * p.width;
  out.mask = p.mask_out ? p.mask_out + (int64_t)row * p.width : nullptr;
  out.count = p.count_out ? p.count_out + row : nullptr;
  for (int i = k + (int)threadIdx.x; i < p.width; i += threads) {
    out.idx[i] = 0;
    if (out.mask) out.mask[i] = 0;
  }
  return out;
}

constexpr int kAscThreads = 1024;

// Every row by the general way: rows longer than kMaxSorted, whose validity
// words do not fit the 64 KiB of LDS beside the entry buffer and the bins.  Bound by
// the latency of its passes, so it needs two blocks per CU: one kernel for both orders
// and index types has 68 VGPRs and one block, T = 70000, k = 2048, 512 rows 530 us.
constexpr int kMaxSorted = 65536;

template <int kOrder, typename IdxT>
__global__ __launch_bounds__(kAscThreads, 8) void topk_general_kernel(TopkArgs p, IdxT* __restrict__ idx) {
  __shared__ SelShared<kAscThreads> sm;
  extern __shared__ uint64_t dyn[];          // GSA_ORDER_SCORE_DESC: a power of two above k entries
  const int row = blockIdx.x;
  const float* srow = p.S + (row / p.T) * p.s_sb + (int64_t)(row % p.T) * p.s_st;
  const int k = p.k_rows ? min(p.k_rows[row], p.width) : p.width;
  topk_general_row<kAscThreads>(srow, p.Tkv, k, kOrder, sm, dyn, topk_row_out(p, idx, row, k, kAscThreads));
}

// ---------------------------------------------------------------------------
// Counting sort by value.  kThreads threads; thread tid holds the row's keys
// c * kThreads + tid, c < kPer, in registers, or (kPer = 0) reads them again
// in each of the three passes; kBpt bins per thread.  Shared memory: the bins,
// the entry buffer (`slots` entries of 8 bytes), one bit per key of the row.
// ---------------------------------------------------------------------------
constexpr int kMaxBin = 192;      // entries of one bin that are placed by comparison; a fuller one: general row
constexpr int kSlack = 256;       // slots past k for the rest of the bin that holds the k-th entry

// Slots of the entry buffer: the general row sorts a power of two above k there.
constexpr int sort_slots(int k) {
  int kp = 1;
  while (kp < k) kp <<= 1;
  return kp > k + kSlack ? kp : k + kSlack;
}

template <int kThreads, int kPer, int kBpt, typename IdxT>
__global__ __launch_bounds__(kThreads, kThreads == 1024 ? 8 : 1) void topk_sorted_kernel(TopkArgs p, IdxT* __restrict__ idx_out, int slots) {
  constexpr int kBins = kBpt * kThreads;
  constexpr int kWaves = kThreads / 64;
  extern __shared__ uint64_t dyn[];          // entry buffer [slots], then the validity words
  __shared__ __align__(16) uint32_t bins[kBins + 4];   // bins[kBins] = 0: where the highest bin's entries start
  __shared__ SelShared<kThreads> sm;
  __shared__ float wmin[kWaves], wmax[kWaves];
  __shared__ uint32_t wsum[kWaves];
  __shared__ int st_bad, st_bin;
  uint64_t* buf = dyn;
  uint64_t* vbits = dyn + slots;             // bit j % 64 of word j / 64: key j is invalid (-inf)

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = blockIdx.x;
  const float* srow = p.S + (row / p.T) * p.s_sb + (int64_t)(row % p.T) * p.s_st;
  const int Tkv = p.Tkv;
  const int k = p.k_rows ? min(p.k_rows[row], p.width) : p.width;
  const auto out = topk_row_out(p, idx_out, row, k, kThreads);
  const int nchunk = (Tkv + kThreads - 1) / kThreads;

  // f(c, j, s) for each of the thread's keys j = c * kThreads + tid; the whole
  // wave takes every chunk (ballots), so s of a j past the row is -inf.
  float sv[kPer > 0 ? kPer : 1];
  auto each = [&](auto&& f) {
    if constexpr (kPer > 0) {
#pragma unroll
      for (int c = 0; c < kPer; ++c)
        if (c < nchunk) f(c * kThreads + tid, sv[c]);
    } else {
      for (int c = 0; c < nchunk; ++c) {
        const int j = c * kThreads + tid;
        f(j, j < Tkv ? srow[j] : -__builtin_inff());
      }
    }
  };
  if constexpr (kPer > 0) {
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const int j = c * kThreads + tid;
      sv[c] = j < Tkv ? srow[j] : -__builtin_inff();
    }
  }
#pragma unroll
  for (int i = 0; i < kBpt; i += 4) *reinterpret_cast<u32x4*>(&bins[kBpt * tid + i]) = u32x4{0u, 0u, 0u, 0u};
  if (tid == 0) { bins[kBins] = 0u; st_bad = 0; st_bin = 0; }

  // ---- range of the valid scores, validity words ----
  float mn = __builtin_inff(), mx = -__builtin_inff();
  bool odd = false;
  each([&](int j, float s) {
    const bool inv = s == -__builtin_inff();
    const uint64_t m = ballot64(inv && j < Tkv);
    if (lane == 0 && j < Tkv) vbits[j >> 6] = m;
    odd |= !(s < __builtin_inff());            // +inf or NaN
    mn = fminf(mn, inv ? __builtin_inff() : s);
    mx = fmaxf(mx, s);
  });
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  odd = ballot64(odd) != 0;
  if (lane == 0) { wmin[wave] = mn; wmax[wave] = mx; }
  __syncthreads();
  if (odd && lane == 0) st_bad = 1;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) { mn = fminf(mn, wmin[w]); mx = fmaxf(mx, wmax[w]); }
  // value-linear bins; monotone in s (each step rounds monotonically), so the
  // order between bins is the order of the scores
  // (one value, or a single valid entry: all in bin 0)
  const float scale = mx > mn ? (float)kBins / (mx - mn) : 0.f;
  const bool none = !(mn < __builtin_inff());              // no valid score at all
  // the invalid entries rank as -1e9: below every valid one only while mn is above that
  const bool fine = none || (mn > -1e9f && mx - mn < __builtin_inff() && scale < 1e30f);
  auto bin_of_score = [&](float s) { return min((int)((s - mn) * scale), kBins - 1); };

  if (fine)
    each([&](int, float s) {
      const bool valid = s != -__builtin_inff() && s < __builtin_inff();
      if constexpr (kPer > 0) {
        if (valid) atomicAdd(&bins[bin_of_score(s)], 1u);
      } else {
        // one addition for a wave whose keys share a bin: 64 on one word one after
        // another are much of what a row with a far outlier pays for nothing (T = 40000,
        // k = 64, 512 rows 276 us, 230 with it; rows of the indexer 54 and 56.  Where the
        // keys are in registers it takes 11 - 25 % of the time of such rows.)
        const int bin = valid ? bin_of_score(s) : -1, first = __builtin_amdgcn_readfirstlane(bin);
        if (ballot64(bin != first) == 0) {
          if (first >= 0 && lane == 0) atomicAdd(&bins[first], 64u);
        } else if (valid) {
          atomicAdd(&bins[bin], 1u);
        }
      }
    });
  __syncthreads();
  bool general = st_bad || !fine;                            // uniform: shared flag, block-wide range

  // ---- bins -> first output position of each (entries of all higher bins) ----
  uint32_t want = 0;                                         // valid entries selected
  if (!general) {
    uint32_t cnt[kBpt], own = 0;
#pragma unroll
    for (int i = 0; i < kBpt; i += 4) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(&bins[kBpt * tid + i]);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        cnt[i + u] = v[u];
        own += v[u];
      }
    }
    uint32_t suf = own;                                      // inclusive suffix sum over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = (uint32_t)__shfl_down((int)suf, o, 64);
      if (lane + o < 64) suf += y;
    }
    if (lane == 0) wsum[wave] = suf;
    __syncthreads();
    uint32_t a = suf - own, total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w > wave) a += wsum[w];
      total += wsum[w];
    }
    want = min((uint32_t)k, total);
#pragma unroll
    for (int i = kBpt - 1; i >= 0; --i) {
      // the bin that holds the last wanted entry; fuller bins than can be
      // placed by comparison, or a last bin that does not fit the buffer
      if (a < want) {
        if (cnt[i] > (uint32_t)kMaxBin || a + cnt[i] > (uint32_t)slots) st_bad = 1;
        if (a + cnt[i] >= want) st_bin = kBpt * tid + i;
      }
      const uint32_t c = cnt[i];
      cnt[i] = a;
      a += c;
    }
#pragma unroll
    for (int i = 0; i < kBpt; i += 4)
      *reinterpret_cast<u32x4*>(&bins[kBpt * tid + i]) = u32x4{cnt[i], cnt[i + 1], cnt[i + 2], cnt[i + 3]};
    __syncthreads();
    general = st_bad != 0;
  }
  if (general) {
    topk_general_row<kThreads>(srow, Tkv, k, GSA_ORDER_SCORE_DESC, sm, buf, out);
    return;
  }

  // ---- scatter: (key, ~index) of every entry from the k-th's bin up ----
  const int last_bin = st_bin;
  if (want > 0)
    each([&](int j, float s) {
      if (s != -__builtin_inff()) {
        const int bin = bin_of_score(s);
        if (bin >= last_bin) {
          const uint32_t at = atomicAdd(&bins[bin], 1u);     // afterwards bins[b] = end of bin b = start of bin b-1
          buf[at] = ((uint64_t)score_key(s) << 32) | (uint64_t)(~(uint32_t)j);
        }
      }
    });
  __syncthreads();
  // ---- place each entry within its bin ----
  const int placed = want > 0 ? (int)bins[last_bin] : 0;
  for (int i = tid; i < placed; i += kThreads) {
    const uint64_t e = buf[i];
    const uint32_t key = (uint32_t)(e >> 32);
    const float s = __uint_as_float((key & 0x80000000u) ? key & 0x7fffffffu : ~key);
    const int bin = bin_of_score(s);
    const int lo = (int)bins[bin + 1], hi = (int)bins[bin];
    int at = lo;
    for (int q = lo; q < hi; ++q) at += buf[q] > e ? 1 : 0;
    if (at < (int)want) {
      out.idx[at] = (IdxT)(~(uint32_t)e);
      if (out.mask) out.mask[at] = 1;
    }
  }
  // ---- then the invalid entries of lowest index ----
  const int rest = k - (int)want;
  if (rest > 0) {
    const int nw = (Tkv + 63) >> 6;
    int base = 0;                                            // invalid entries in the words before this turn's
    for (int w0 = 0; w0 < nw && base < rest; w0 += 64) {     // every wave walks the words; they share the writes
      const uint64_t m = w0 + lane < nw ? vbits[w0 + lane] : 0ull;
      const int n = __popcll(m);
      int incl = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
      }
      const int first = base + incl - n;
      for (int l = wave; l < 64 && w0 + l < nw; l += kWaves) {
        const uint64_t ml = (uint64_t)__shfl((long long)m, l, 64);
        const int at = __shfl(first, l, 64) + count_below(ml);
        if (((ml >> lane) & 1ull) && at < rest) {
          out.idx[want + at] = (IdxT)(64 * (w0 + l) + lane);
          if (out.mask) out.mask[want + at] = 0;
        }
      }
      base += __shfl(incl, 63, 64);
    }
  }
  if (tid == 0 && out.count) *out.count = (int)want;
}

// Population variance of each row's finite (not -inf) scores, two passes
// (mean, then squared deviations) as the variance rule states it
// (gsa_explained.ipynb:577-592); a row without finite scores gets 0.
__global__ __launch_bounds__(256) void row_var_kernel(const float* __restrict__ S, int64_t s_sb, int64_t s_st,
                                                      int T, int Tkv, float* __restrict__ var) {
  __shared__ float part[4];
  __shared__ int cpart[4];
  const int row = blockIdx.x;
  const int b = row / T, t = row % T;
  const float* srow = S + b * s_sb + (int64_t)t * s_st;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float sum = 0.f;
  int cnt = 0;
  for (int j = tid; j < Tkv; j += 256) {
    const float v = srow[j];
    if (v != -__builtin_inff()) { sum += v; ++cnt; }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o, 64);
    cnt += __shfl_xor(cnt, o, 64);
  }
  if (lane == 0) { part[wave] = sum; cpart[wave] = cnt; }
  __syncthreads();
  const float n = (float)max(1, cpart[0] + cpart[1] + cpart[2] + cpart[3]);
  const float mean = (((part[0] + part[1]) + part[2]) + part[3]) / n;
  __syncthreads();
  float sq = 0.f;
  for (int j = tid; j < Tkv; j += 256) {
    const float v = srow[j];
    if (v != -__builtin_inff()) {
      const float d = v - mean;
      sq = __builtin_fmaf(d, d, sq);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
  if (lane == 0) part[wave] = sq;
  __syncthreads();
  if (tid == 0) var[row] = (((part[0] + part[1]) + part[2]) + part[3]) / n;
}

}  // namespace gsa

using namespace gsa_host;

namespace {

// LDS of topk_sorted_kernel beside its static arrays: the entry buffer and one
// bit per key.  At k = 4096: 34 KiB, and 32 bytes per 256 keys.
size_t sorted_lds(int k, int Tkv) {
  return (size_t)(gsa::sort_slots(k) + (Tkv + 63) / 64) * sizeof(uint64_t);
}

template <int kThreads, int kPer, int kBpt, typename IdxT>
int launch_sorted(const gsa::TopkArgs& a, int B, IdxT* idx, hipStream_t s) {
  const int slots = gsa::sort_slots(a.width);
  hipLaunchKernelGGL((gsa::topk_sorted_kernel<kThreads, kPer, kBpt, IdxT>), dim3(B * a.T), dim3(kThreads),
                     sorted_lds(a.width, a.Tkv), s, a, idx, slots);
  return launch_status();
}

template <int kOrder, typename IdxT>
int launch_general(const gsa::TopkArgs& a, int B, IdxT* idx, hipStream_t s) {
  const size_t lds = kOrder == GSA_ORDER_SCORE_DESC ? (size_t)gsa::sort_slots(a.width) * sizeof(uint64_t) : 0;
  hipLaunchKernelGGL((gsa::topk_general_kernel<kOrder, IdxT>), dim3(B * a.T), dim3(gsa::kAscThreads), lds, s, a, idx);
  return launch_status();
}

// Threads and keys per thread by the row's length: a block's barriers cost more
// with more waves, so a thread takes 16 keys (32 past 8192) before the block
// grows.  A causal T x T matrix of indexer scores, k = min(T, 2048), us with 256 / 512 /
// 1024 threads: T = 2048 23 / 24 / 35, T = 4096 48 / 48 / 68, T = 8192 125 / 117 / 152,
// T = 16384 499 / 350 / 396.  Rows past 16384 keys are read again in each pass, whose
// latency 1024 threads hide better (T = 40000, k = 2048, 512 rows 99 us with 512, 60).
template <typename IdxT>
int launch_by_length(const gsa::TopkArgs& a, int B, IdxT* idx, hipStream_t s) {
  if (a.Tkv <= 2048) return launch_sorted<256, 8, 4>(a, B, idx, s);
  if (a.Tkv <= 4096) return launch_sorted<256, 16, 4>(a, B, idx, s);
  if (a.Tkv <= 8192) return launch_sorted<512, 16, 4>(a, B, idx, s);
  if (a.Tkv <= 16384) return launch_sorted<512, 32, 8>(a, B, idx, s);
  if (a.Tkv <= gsa::kMaxSorted) return launch_sorted<1024, 0, 4>(a, B, idx, s);
  return launch_general<GSA_ORDER_SCORE_DESC>(a, B, idx, s);
}

int launch_topk(const gsa::TopkArgs& a, int B, int order, int32_t* idx, hipStream_t s) {
  if (order == GSA_ORDER_SCORE_DESC) return launch_by_length(a, B, idx, s);
  return launch_general<GSA_ORDER_INDEX_ASC>(a, B, idx, s);
}

// Checks shared by the entry points.
int topk_checks(const float* scores, const void* idx_out, int idx_align, const int32_t* count_out, int B, int T,
                int Tkv) {
  if (!scores || !idx_out) return GSA_ERR_NULL;
  if (B < 1 || T < 1 || Tkv < 1 || (int64_t)B * T > 0x7fffffffLL) return GSA_ERR_SHAPE;
  if (!aligned(scores, 4) || !aligned(idx_out, idx_align) || (count_out && !aligned(count_out, 4)))
    return GSA_ERR_ALIGN;
  return GSA_OK;
}

}  // namespace

extern "C" int gsa_topk_select(const float* scores, int64_t s_sb, int64_t s_st,
                               int B, int T, int Tkv, int k_eff, int order,
                               int32_t* idx_out, int32_t* count_out, uint8_t* mask_out,
                               void* stream) {
  const int st = topk_checks(scores, idx_out, 4, count_out, B, T, Tkv);
  if (st == GSA_ERR_NULL || st == GSA_ERR_SHAPE) return st;
  if (order != GSA_ORDER_INDEX_ASC && order != GSA_ORDER_SCORE_DESC) return GSA_ERR_FLAGS;
  if (k_eff < 1 || k_eff > Tkv) return GSA_ERR_K;
  if (order == GSA_ORDER_SCORE_DESC && k_eff > GSA_TOPK_DESC_MAX_K) return GSA_ERR_K;
  if (st) return st;
  const gsa::TopkArgs a{scores, s_sb, s_st, T, Tkv, k_eff, nullptr, count_out, mask_out};
  return launch_topk(a, B, order, idx_out, static_cast<hipStream_t>(stream));
}

extern "C" int gsa_topk_select_i64(const float* scores, int64_t s_sb, int64_t s_st, int B, int T, int Tkv,
                                   int k_eff, int64_t* idx_out, uint8_t* mask_out, void* stream) {
  const int st = topk_checks(scores, idx_out, 8, nullptr, B, T, Tkv);
  if (st == GSA_ERR_NULL || st == GSA_ERR_SHAPE) return st;
  if (k_eff < 1 || k_eff > Tkv || k_eff > GSA_TOPK_DESC_MAX_K) return GSA_ERR_K;
  if (st) return st;
  const gsa::TopkArgs a{scores, s_sb, s_st, T, Tkv, k_eff, nullptr, nullptr, mask_out};
  return launch_by_length(a, B, idx_out, static_cast<hipStream_t>(stream));
}

extern "C" int gsa_topk_select_adaptive(const float* scores, int64_t s_sb, int64_t s_st,
                                        int B, int T, int Tkv, int k_base, int k_min, int k_max, int order,
                                        int32_t* idx_out, int32_t* count_out, uint8_t* mask_out,
                                        int32_t* k_out, float* var_out, void* stream) {
  if (!k_out || !var_out) return GSA_ERR_NULL;
  int st = topk_checks(scores, idx_out, 4, count_out, B, T, Tkv);
  if (st == GSA_ERR_NULL || st == GSA_ERR_SHAPE) return st;
  if (order != GSA_ORDER_INDEX_ASC && order != GSA_ORDER_SCORE_DESC) return GSA_ERR_FLAGS;
  if (k_base < 1 || k_min < 1 || k_max < k_min) return GSA_ERR_K;
  const int width = k_max < Tkv ? k_max : Tkv;
  if (order == GSA_ORDER_SCORE_DESC && width > GSA_TOPK_DESC_MAX_K) return GSA_ERR_K;
  if (st || !aligned(k_out, 4) || !aligned(var_out, 4)) return GSA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(gsa::row_var_kernel, dim3(B * T), dim3(256), 0, s, scores, s_sb, s_st, T, Tkv, var_out);
  if ((st = launch_status())) return st;
  if ((st = launch_adaptive_k(var_out, B * T, k_base, k_min, k_max, width, k_out, s))) return st;
  const gsa::TopkArgs a{scores, s_sb, s_st, T, Tkv, width, k_out, count_out, mask_out};
  return launch_topk(a, B, order, idx_out, s);
}
