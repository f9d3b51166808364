// Attention over per-row index lists on the matrix cores (the
// fused_sparse_attention launcher).
//
// The gather kernel (sparse_attn.hip) reads K and V of every selected key once
// per query row -- 8 KiB per selected key in bf16 at 16 heads, 16 KiB in fp32
// -- and takes 12.8 ms at T = 8192, k = 2048, where the arithmetic needs 0.1.
// Here the lists become a bitmask, and the block-dense kernels compute every
// 64-key tile that holds a selected key of a query block on MFMA, with the
// bitmask applied to the scores: K and V are read once per 256 query rows
// (0.50 ms there).
//
// Both give the softmax over the selected keys, except where a row's list
// names a key twice (the lists weigh it twice, a bitmask once) or a value is
// not finite (a masked tile multiplies it by zero).  Such rows are marked --
// the first kind here, the second by the attention kernel -- and the gather
// kernel computes them in a last launch; unmarked rows' blocks end at once.
#include "gsa_common.h"

#include <algorithm>
#include <climits>
#include <cmath>

namespace gsa {

// Index lists -> bitmask, tile range and repeat mark of each row: one block per row.
struct SelRowsArgs {
  const void* idx; int idx64; int64_t i_sb, i_st; int k_sel;
  const int32_t* count; const uint8_t* mask;
  int T, Tkv, W;
  uint32_t* bits; int2* range; uint8_t* twice;   // range of a row that names a key twice: empty
};

template <typename IdxT>
__global__ __launch_bounds__(256) void selected_rows_kernel(SelRowsArgs p) {
  extern __shared__ uint32_t sw[];           // the row's W words
  __shared__ int st_lo, st_hi, st_twice;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int b = row / p.T, t = row % p.T;
  for (int i = tid; i < p.W; i += 256) sw[i] = 0u;
  if (tid == 0) { st_lo = INT_MAX; st_hi = 0; st_twice = 0; }
  __syncthreads();
  int n = p.k_sel;
  if (p.count) n = min(n, p.count[row]);
  const int64_t base = b * p.i_sb + (int64_t)t * p.i_st;
  const IdxT* irow = static_cast<const IdxT*>(p.idx) + base;
  const uint8_t* mrow = p.mask ? p.mask + base : nullptr;
  bool twice = false;
  for (int m = tid; m < n; m += 256) {
    if (mrow == nullptr || mrow[m] != 0) {
      const int j = min(max((int)irow[m], 0), p.Tkv - 1);
      const uint32_t bit = 1u << (j & 31);
      twice |= (atomicOr(&sw[j >> 5], bit) & bit) != 0u;
    }
  }
  if (ballot64(twice) && lane == 0) st_twice = 1;
  __syncthreads();
  uint32_t* brow = p.bits + (int64_t)row * p.W;
  int lo = INT_MAX, hi = 0;
  for (int i = tid; i < p.W; i += 256) {
    const uint32_t w = sw[i];
    brow[i] = w;
    if (w) { lo = min(lo, i >> 1); hi = (i >> 1) + 1; }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  if (lane == 0 && hi) { atomicMin(&st_lo, lo); atomicMax(&st_hi, hi); }
  __syncthreads();
  if (tid == 0) {
    // no tile for a row that the gather computes in any case: blocks of such rows
    // end after one (T = 4096, k = 64, every list with a repeat 359 us -> 254; gather alone 223)
    p.range[row] = st_twice ? int2{INT_MAX, 0} : int2{st_lo, st_hi};
    p.twice[row] = (uint8_t)st_twice;
  }
}

}  // namespace gsa

using namespace gsa_host;

namespace {

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t bits_bytes(int B, int T, int Tkv) { return align256((size_t)B * T * ((Tkv + 63) / 64) * 8); }

// Bitmask, tile ranges, repeat marks, redo marks, then the attention kernel's own.
size_t workspace(int B, int T, int Tkv, int H, int dtype) {
  return bits_bytes(B, T, Tkv) + align256((size_t)B * T * 8) + align256((size_t)B * T) + align256((size_t)B * T * H) +
         (dtype == GSA_DTYPE_BF16 ? dense_selected_bytes(B, T, Tkv, H) : dense_f32_bytes(B, T, Tkv, H));
}

constexpr size_t kMaxWorkspace = (size_t)4 << 30;

// Whether the matrix-core way is the faster one, from the time each takes (us; fitted
// to both, whole calls, at 1400 random sizes: 1 - 64 heads, B = 1 - 8, T <= 4096, Tkv <=
// 20000, k <= 2048; the pick is 0.5 % above the better one on average).
// The gather: 8 (5 in fp32), and the larger of its chain of loads within a row's
// block, 0.355 + 0.004 H per key (0.387 + 0.0082 H), and what it reads, 820 (1160) per
// million rows x keys x 16 heads; at least 20.5, the host's pace.  T = 512, k = 128,
// H = 16 74; T = 8192, k = 2048 13002; T = 27, Tkv = 12402, k = 126, H = 8 49.
// The matrix cores: 11 (10) for the launches, 3.6 (9.9) for each 64-key tile that a CU
// takes one after another -- its mean share, or a block's tiles, or where blocks are
// split a part of one: 1.4 times the mean, 8 at least (0.6 or 0.33 times, 2 at least)
// -- 1.55 (1.15) for each part that the last one adds, and 10.5 per million list
// entries; at least 26.  The same three calls: 37, 502, 84; fp32 T = 50, Tkv = 13628,
// k = 182, H = 4 146 where the gather takes 92.  (Query and key length alike are taken
// for causal, else all Tkv tiles are counted: what a selection leaves out is known
// on the device only.)
// The masks reach -8e36 times the scale, which has to stay far below every
// score: a scale outside [1e-10, 1e10] takes the gather.  A row's bits fit the
// LDS of a block, and the workspace (2 bytes per element of V, 5 bits per row
// and key) is kept to 4 GiB.
bool dense_serves(int B, int T, int Tkv, int H, int k_sel, float scale, int dtype) {
  const bool bf16 = dtype == GSA_DTYPE_BF16;
  if (!bf16 && dtype != GSA_DTYPE_F32) return false;
  if (!(scale >= 1e-10f && scale <= 1e10f)) return false;
  if ((size_t)((Tkv + 63) / 64) * 8 > 65536 - 64) return false;
  const int64_t NT = (Tkv + 63) / 64, groups = ((int64_t)T + 255) / 256 * 8;
  const double entries = 1e-6 * B * T * (double)k_sel, reads = entries * H / 16;
  const double gather = bf16 ? 8.0 + std::max((0.355 + 0.004 * H) * k_sel, 820.0 * reads)
                             : 5.0 + std::max((0.387 + 0.0082 * H) * k_sel, 1160.0 * reads);
  const double nqb = bf16 ? groups / 8 : (T + 127) / 128;
  const double mean = NT * (B * (double)H * nqb) / 256 * (T == Tkv ? (nqb + 1) / (2 * nqb) : 1.0);
  const double part = bf16 ? std::max(8.0, 1.4 * mean) : std::max(2.0, (2 * mean < 40 ? 0.6 : 0.33) * mean);
  const double serial = std::max(mean, std::min((double)NT, part)), parts = part < NT ? std::ceil(NT / part) : 0.0;
  const double dense = (bf16 ? 11.0 : 10.0) + (bf16 ? 3.6 : 9.9) * serial + (bf16 ? 1.55 : 1.15) * parts + 10.5 * entries;
  if (std::max(26.0, dense) > std::max(20.5, gather)) return false;
  if (B * groups * NT > 0x3fffffffLL / 32 || (int64_t)B * H * NT > 0x3fffffffLL) return false;
  return workspace(B, T, Tkv, H, dtype) <= kMaxWorkspace;
}

}  // namespace

extern "C" size_t gsa_selected_attn_workspace_bytes(int B, int T, int Tkv, int H, int k_sel, float scale, int dtype) {
  if (B < 1 || T < 1 || Tkv < 1 || H < 1 || H > 64 || !dense_serves(B, T, Tkv, H, k_sel, scale, dtype)) return 0;
  return workspace(B, T, Tkv, H, dtype);
}

extern "C" int gsa_selected_attn(const void* q, int64_t q_sb, int64_t q_st,
                                 const void* k, int64_t k_sb, int64_t k_st,
                                 const void* v, int64_t v_sb, int64_t v_st,
                                 const void* idx, int idx_bytes, int64_t i_sb, int64_t i_st, int k_sel,
                                 const int32_t* count, const uint8_t* mask,
                                 void* out, int64_t out_sb, int64_t out_st,
                                 int B, int T, int Tkv, int H, int d, float scale, int dtype,
                                 void* ws, size_t ws_bytes, void* stream) {
  if (!q || !k || !v || !idx || !out || !ws) return GSA_ERR_NULL;
  if (dtype_size(dtype) == 0) return GSA_ERR_DTYPE;
  if (B < 1 || T < 1 || Tkv < 1 || d != 128 || H < 1 || H > 64) return GSA_ERR_SHAPE;
  if ((int64_t)B * T > 0x7fffffffLL) return GSA_ERR_SHAPE;
  if (k_sel < 0) return GSA_ERR_K;
  if (idx_bytes != 4 && idx_bytes != 8) return GSA_ERR_DTYPE;
  const size_t need = gsa_selected_attn_workspace_bytes(B, T, Tkv, H, k_sel, scale, dtype);
  if (need == 0 || ws_bytes < need) return GSA_ERR_SHAPE;
  // per-lane load offsets within a tile are 32-bit byte offsets
  for (const int64_t st : {q_st, k_st, v_st, out_st})
    if (st < 0 || st > (1 << 24)) return GSA_ERR_SHAPE;
  if (!vec_ok(q, q_sb, q_st, dtype) || !vec_ok(k, k_sb, k_st, dtype) || !vec_ok(v, v_sb, v_st, dtype) ||
      !vec_ok(out, out_sb, out_st, dtype) || !aligned(idx, idx_bytes) || (count && !aligned(count, 4)) ||
      !aligned(ws, 256))
    return GSA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* base = static_cast<char*>(ws);
  uint32_t* bits = reinterpret_cast<uint32_t*>(base);
  base += bits_bytes(B, T, Tkv);
  int2* range = reinterpret_cast<int2*>(base);
  base += align256((size_t)B * T * 8);
  uint8_t* twice = reinterpret_cast<uint8_t*>(base);
  base += align256((size_t)B * T);
  uint8_t* redo = reinterpret_cast<uint8_t*>(base);
  base += align256((size_t)B * T * H);
  const int W = 2 * ((Tkv + 63) / 64);
  const gsa::SelRowsArgs r{idx, idx_bytes == 8, i_sb, i_st, k_sel, count, mask, T, Tkv, W, bits, range, twice};
  if (idx_bytes == 8)
    hipLaunchKernelGGL(gsa::selected_rows_kernel<int64_t>, dim3(B * T), dim3(256), (size_t)W * 4, s, r);
  else
    hipLaunchKernelGGL(gsa::selected_rows_kernel<int32_t>, dim3(B * T), dim3(256), (size_t)W * 4, s, r);
  int st = launch_status();
  if (st) return st;
  AttnShape a{q, q_sb, q_st, k, k_sb, k_st, v, v_sb, v_st, out, out_sb, out_st, B, T, Tkv, H, scale};
  const gsa::Selection sel{bits, range, twice, redo};
  st = dtype == GSA_DTYPE_BF16 ? launch_dense_selected(a, sel, base, s) : launch_dense_f32(a, sel, base, s);
  if (st) return st;
  return launch_gather_rows(a, IndexLists{idx, idx_bytes == 8, i_sb, i_st, k_sel, count, mask}, sel, dtype, s);
}

// ---------------------------------------------------------------------------
// The layer's fp32 attention: the selection is there as a causal bitmask.
// ---------------------------------------------------------------------------

// Workspace of gsa_masked_attn: the redo marks, the index lists and counts of
// marked rows, then the attention kernel's own.
static size_t masked_workspace(int B, int T, int H, int k_sel) {
  return align256((size_t)B * T * H) + align256((size_t)B * T * k_sel * 4) + align256((size_t)B * T * 4) +
         dense_f32_bytes(B, T, T, H);
}

// From the time each way takes (us, 16 heads): the gather 20 and the larger of 0.5 per
// key of a row and 1.8 per 1000 pairs of a row and a key (and the index lists, left
// out), the matrix cores 30 for the launches and 4.9 for each 32-key tile of a
// 128-row block per CU (T = 2048, k = 256: 191 against 485 and 52 for the lists).
extern "C" size_t gsa_masked_attn_workspace_bytes(int B, int T, int H, int k_sel, int dtype) {
  if (B < 1 || T < 1 || H < 1 || H > 64 || k_sel < 1 || k_sel > T || dtype != GSA_DTYPE_F32) return 0;
  if ((int64_t)B * T > 0x7fffffffLL) return 0;
  const double k = k_sel, pairs = B * (k * (k + 1) / 2 + (T - k) * k);
  const double gather = 20.0 + std::max(0.5 * k, 0.0018 * pairs * H / 16);
  const double tiles = (T + 31) / 32 * (((T + 127) / 128 + 1) / 2.0) * B * H;
  if (30.0 + 4.9 * tiles / 256 > gather) return 0;
  return masked_workspace(B, T, H, k_sel);
}

extern "C" int gsa_masked_attn(const void* q, int64_t q_sb, int64_t q_st,
                               const void* k, int64_t k_sb, int64_t k_st,
                               const void* v, int64_t v_sb, int64_t v_st,
                               const uint32_t* bits, int k_sel,
                               const void* og, int64_t o_sb, int64_t o_st,
                               const void* cos, const void* sin, int64_t cs_st,
                               void* out, int64_t out_sb, int64_t out_st,
                               int B, int T, int H, int d, float scale, int dtype, int flags,
                               void* ws, size_t ws_bytes, void* stream) {
  if (!q || !k || !v || !bits || !out || !ws) return GSA_ERR_NULL;
  if (flags & ~(GSA_ATTN_ROPE_Q | GSA_ATTN_OUT_GATE)) return GSA_ERR_FLAGS;
  if ((flags & GSA_ATTN_ROPE_Q) && (!cos || !sin)) return GSA_ERR_NULL;
  if ((flags & GSA_ATTN_OUT_GATE) && !og) return GSA_ERR_NULL;
  if (dtype != GSA_DTYPE_F32) return GSA_ERR_DTYPE;
  if (B < 1 || T < 1 || d != 128 || H < 1 || H > 64) return GSA_ERR_SHAPE;
  if ((int64_t)B * T > 0x7fffffffLL || (int64_t)B * H * ((T + 127) / 128) > 0x7fffffffLL) return GSA_ERR_SHAPE;
  if (k_sel < 1 || k_sel > T) return GSA_ERR_K;
  if (!(scale > 0.f)) return GSA_ERR_SHAPE;             // a row's largest score is found before the scale
  if (ws_bytes < masked_workspace(B, T, H, k_sel)) return GSA_ERR_SHAPE;
  for (const int64_t st : {k_st, v_st})                 // 32-bit byte offsets within a tile
    if (st < 0 || st > (1 << 24)) return GSA_ERR_SHAPE;
  if (!vec_ok(q, q_sb, q_st, dtype) || !vec_ok(k, k_sb, k_st, dtype) || !vec_ok(v, v_sb, v_st, dtype) ||
      !vec_ok(out, out_sb, out_st, dtype) || !aligned(bits, 8) || !aligned(ws, 256))
    return GSA_ERR_ALIGN;
  if ((flags & GSA_ATTN_OUT_GATE) && !vec_ok(og, o_sb, o_st, dtype)) return GSA_ERR_ALIGN;
  if ((flags & GSA_ATTN_ROPE_Q) && (!vec_ok(cos, 0, cs_st, dtype) || !vec_ok(sin, 0, cs_st, dtype)))
    return GSA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* base = static_cast<char*>(ws);
  uint8_t* redo = reinterpret_cast<uint8_t*>(base);
  base += align256((size_t)B * T * H);
  int32_t* idx = reinterpret_cast<int32_t*>(base);
  base += align256((size_t)B * T * k_sel * 4);
  int32_t* count = reinterpret_cast<int32_t*>(base);
  base += align256((size_t)B * T * 4);
  const AttnShape a{q, q_sb, q_st, k, k_sb, k_st, v, v_sb, v_st, out, out_sb, out_st, B, T, T, H, scale,
                    og, o_sb, o_st, cos, sin, cs_st, flags};
  const gsa::Selection sel{bits, nullptr, nullptr, redo};
  int st = launch_dense_f32(a, sel, base, s);
  if (st) return st;
  if ((st = launch_marked_indices(bits, B, T, k_sel, redo, H, idx, count, s))) return st;
  return launch_gather_rows(a, IndexLists{idx, 0, (int64_t)T * k_sel, k_sel, k_sel, count, nullptr}, sel, dtype, s);
}
