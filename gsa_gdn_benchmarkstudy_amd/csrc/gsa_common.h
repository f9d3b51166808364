// Shared device helpers and host-side argument checks for the gfx950 GSA
// kernels.  Wave64 throughout: a "row group" is one DPP row of 16 lanes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/gsa_hip.h"

// Every product and sum rounds on its own (torch's rounding points); fused
// multiply-adds are written explicitly where wanted.
#pragma clang fp contract(off)

namespace gsa {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Never apply __builtin_bit_cast to one element of a vector (`v[i]` of a
// u32x4): this compiler reads element 0 for every i -- for a loop over
// `__builtin_bit_cast(bf16x2, v[i])` it loads a single dword.  Copy the
// element into a scalar first, or bit-cast whole vectors and arrays.

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------
// bf16 <-> fp32.  Rounding is round-to-nearest-even, the rounding torch uses
// when an fp32 intermediate is stored as bf16, done by the hardware convert
// (v_cvt_pk_bf16_f32; two values per instruction in pack_bf16); NaN stays
// NaN.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bf16lo(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16hi(uint32_t packed) { return __uint_as_float(packed & 0xffff0000u); }

__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ float round_bf16(float f) {
  return __uint_as_float(f32_to_bf16_bits(f) << 16);
}
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Storage-type traits: how one 16-lane head slice of 8 elements is held.
template <typename T> struct Elem;
template <> struct Elem<uint16_t> {          // bf16 storage
  static constexpr bool kBf16 = true;
  __device__ static float rnd(float f) { return round_bf16(f); }
};
template <> struct Elem<float> {
  static constexpr bool kBf16 = false;
  __device__ static float rnd(float f) { return f; }
};

// Load / store 8 consecutive elements as fp32.
__device__ __forceinline__ void load8(const uint16_t* p, float (&x)[8]) {
  u32x4 r = *reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) { x[2 * i] = bf16lo(r[i]); x[2 * i + 1] = bf16hi(r[i]); }
}
__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
  floatx4 a = *reinterpret_cast<const floatx4*>(p);
  floatx4 b = *reinterpret_cast<const floatx4*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) { x[i] = a[i]; x[4 + i] = b[i]; }
}
__device__ __forceinline__ void store8(uint16_t* p, const float (&x)[8]) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
  *reinterpret_cast<u32x4*>(p) = r;
}
__device__ __forceinline__ void store8(float* p, const float (&x)[8]) {
  floatx4 a, b;
#pragma unroll
  for (int i = 0; i < 4; ++i) { a[i] = x[i]; b[i] = x[4 + i]; }
  *reinterpret_cast<floatx4*>(p) = a;
  *reinterpret_cast<floatx4*>(p + 4) = b;
}

// sigmoid(x) = 1 / (1 + 2^(-x*log2 e)), hardware exp2 and reciprocal
// (about 1 ulp each).  exp2 overflow gives +inf and the reciprocal 0, the
// correct limit.
__device__ __forceinline__ float sigmoidf_fast(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
}

// ---------------------------------------------------------------------------
// Cross-lane helpers (DPP within a 16-lane row; ballots over the wave).
// ---------------------------------------------------------------------------
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}
// row_ror:n is DPP control 0x120 + n.  Rotations make every lane of the row
// hold the full reduction.
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp<0x128>(v);
  v += dpp<0x124>(v);
  v += dpp<0x122>(v);
  v += dpp<0x121>(v);
  return v;
}
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp<0x128>(v));
  v = fmaxf(v, dpp<0x124>(v));
  v = fmaxf(v, dpp<0x122>(v));
  v = fmaxf(v, dpp<0x121>(v));
  return v;
}
// Value of lane (i + 8) mod 16 within the row.
__device__ __forceinline__ float row16_swap8(float v) { return dpp<0x128>(v); }

__device__ __forceinline__ int lane_id() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}
__device__ __forceinline__ uint64_t ballot64(bool p) { return __ballot(p); }
// Number of set bits of `mask` below the calling lane.
__device__ __forceinline__ int count_below(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// RoPE on one lane's 8 elements: x*cos + rotate_half(x)*sin, where
// rotate_half takes element i+64 (negated) for i < 64 and element i-64 for
// i >= 64 -- the value held by lane (li +/- 8) of the same 16-lane row.
template <typename T>
__device__ __forceinline__ void rope8(float (&x)[8], const float (&c)[8], const float (&s)[8], int li) {
  float partner[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) partner[i] = row16_swap8(x[i]);
  const float sign = li < 8 ? -1.f : 1.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float a = Elem<T>::rnd(x[i] * c[i]);
    const float r = Elem<T>::rnd((sign * partner[i]) * s[i]);
    x[i] = Elem<T>::rnd(a + r);
  }
}

// ---------------------------------------------------------------------------
// Query blocks split along their keys (the block-dense attention kernels).
// With few query blocks, or causal ones of very different length, one block
// per CU leaves most of the chip idle while the longest runs; a unit is then one
// of `parts` equal pieces of a query block's key tiles.  Each unit writes its
// sums and softmax state to its slot and counts itself; the last one to arrive
// adds all parts in their order (so the result does not depend on which was
// last) and goes on to the epilogue.  No unit waits for another.
//
// Query block qb has min(nt, step * (qb + 1)) tiles (causal) or nt (step 0).
// Blocks qs and up are split into parts of at most `chunk` tiles.  The order is
// longest first, roughly: the unsplit blocks above 3/4 of chunk (qa .. qs-1), the
// parts, the shorter blocks.  (A sorted table in the kernel arguments cost every
// block 3 us to look its unit up.)
// ---------------------------------------------------------------------------
struct UnitPlan {
  int n;                                  // units per (batch, head); 0: no plan, the kernel's own order
  int slots;                              // partial slots per (batch, head)
  int nqb, nt, step, chunk, qs, qa;
  uint32_t inv;                           // ceil(2^32 / chunk)
  __host__ __device__ int tiles(int qb) const {
    const int t = step * (qb + 1);
    return step && t < nt ? t : nt;
  }
};
struct Unit { int qb, part, parts, slot; };
__device__ __forceinline__ Unit plan_unit(const UnitPlan& p, int u) {
  if (u < p.qs - p.qa) return Unit{p.qs - 1 - u, 0, 1, 0};
  u -= p.qs - p.qa;
  int slot = 0;
  for (int qb = p.nqb - 1; qb >= p.qs; --qb) {
    const int parts = (int)__umulhi((uint32_t)(p.tiles(qb) + p.chunk - 1), p.inv);
    if (u < parts) return Unit{qb, u, parts, slot};
    u -= parts;
    slot += parts;
  }
  return Unit{p.qa - 1 - u, 0, 1, 0};
}
// Floats of one slot: per wave 64 accumulator registers, m and l of 64 lanes.
constexpr int kPartWave = 66 * 64;

// Publishes this unit's O^T accumulators, reference m and sum l (whole row, in
// both lanes) and, in the last unit to arrive, replaces them by the sums over
// all parts; false in the other units, which have nothing left to do.
// slots: the query block's first slot; `flag`: one word of LDS that no wave
// uses any more.  The units may run on different XCDs, whose L2 caches are not
// coherent: every value goes out and comes back by agent-scope accesses (written
// through and read past L2), complete (vmcnt(0)) before the workgroup counts
// itself.  (Plain stores with an agent-scope release write a whole L2 back for
// each unit: T = 2048, bf16,
// 63 us, 53 this way.)
__device__ __forceinline__ void part_store(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float part_load(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool merge_parts(floatx16 (&o)[4], float& m, float& l, float* slots, int part, int parts,
                                            int waves, int wave, int lane, uint32_t* counter, uint32_t* flag) {
  float* const mine = slots + ((int64_t)part * waves + wave) * kPartWave + lane;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) part_store(mine + (16 * dt + r) * 64, o[dt][r]);
  part_store(mine + 64 * 64, m);
  part_store(mine + 65 * 64, l);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*flag != (uint32_t)(parts - 1)) return false;
  const float* const all = slots + (int64_t)wave * kPartWave + lane;
  float top = -__builtin_inff();
  for (int s = 0; s < parts; ++s) top = fmaxf(top, part_load(all + (int64_t)s * waves * kPartWave + 64 * 64));
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  l = 0.f;
  for (int s = 0; s < parts; ++s) {
    const float* const at = all + (int64_t)s * waves * kPartWave;
    const float ms = part_load(at + 64 * 64);
    const float w = ms == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(ms - top);
    l = __builtin_fmaf(part_load(at + 65 * 64), w, l);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = __builtin_fmaf(part_load(at + (16 * dt + r) * 64), w, o[dt][r]);
  }
  m = top;
  return true;
}

// Monotone map of an fp32 score to uint32: a > b  <=>  key(a) > key(b).
// -inf is first replaced by -1e9 (the selector's fill value) and every NaN
// ranks above +inf, as torch.topk orders them.
__device__ __forceinline__ uint32_t score_key(float s) {
  if (s == -__builtin_inff()) s = -1e9f;
  uint32_t u = __float_as_uint(s);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ---------------------------------------------------------------------------
// Helpers of the block-dense attention kernels (lane l and l^32: one query row)
// ---------------------------------------------------------------------------
// Value of lane l^32 combined with the own value: permlane32_swap of (v, v)
// leaves {v[l], v[l^32]} in the two results on every lane.  max_halves takes
// values that are never NaN (maxima seeded with -inf), so a compare-select
// is enough (fmaxf would first quiet both operands).
__device__ __forceinline__ float max_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const float a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
  return a > b ? a : b;
}
__device__ __forceinline__ float sum_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// 32-bit LDS address of a shared-memory pointer.
__device__ __forceinline__ uint32_t lds_addr(const void* ptr) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)ptr;
}

// Direct global -> LDS load: every lane's 16 bytes at base + voff land at
// lds + 16 * lane (base and lds uniform).  Issued as inline asm so that the
// compiler's own bookkeeping does not make each LDS read wait for every such
// load in flight; completion is awaited explicitly (vmcnt) before the
// barrier that publishes a tile.  m0 holds the LDS address; nothing else in
// this kernel uses m0.  An LDS DMA reads m0 one wait state after the SALU
// write at the earliest (the s_nop; the compiler pads its own LDS DMA the
// same way on gfx950).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_lds16(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// s_waitcnt immediate (gfx9 encoding): vmcnt(0), expcnt and lgkmcnt not waited
constexpr int kWaitVmcnt0 = (0x7 << 4) | (0xf << 8);

// ---------------------------------------------------------------------------
// A selection in the form that the MFMA attention kernels take, and the marks
// of what the gather kernel has to compute after them.
// ---------------------------------------------------------------------------
struct Selection {
  const uint32_t* bits;   // [B*T][W] bitmask, W = 2*ceil(Tkv/64): bit j of a row: key j is selected
  const int2* range;      // [B*T] first and past-last 64-key tile of the row's keys (none, or named twice: INT_MAX, 0)
  const uint8_t* twice;   // [B*T] nonzero: the row's list names a key twice, so the bitmask cannot stand for it (or null)
  uint8_t* redo;          // [B*T*H] written by the attention kernel: nonzero: that head of the row has to come from the gather kernel
};

// The two lanes of a row agree on its redo mark and write it.
__device__ __forceinline__ void mark_row(uint8_t* mark, bool good) {
  const uint32_t g = good ? 1u : 0u;
  const auto r = __builtin_amdgcn_permlane32_swap(g, g, false, false);
  *mark = (uint8_t)((r[0] & r[1]) ^ 1u);
}

// 64-key tiles [x, y) that hold a selected key of rows r0 .. r1-1 of sequence b
// (at least one tile), agreed on by the kLanes lanes of an aligned group.
template <int kLanes>
__device__ __forceinline__ int2 tile_range(const int2* range, int64_t row_base, int r0, int r1) {
  int lo = 0x7fffffff, hi = 0;
  for (int r = r0 + (int)(threadIdx.x & (kLanes - 1)); r < r1; r += kLanes) {
    const int2 v = range[row_base + r];
    lo = min(lo, v.x);
    hi = max(hi, v.y);
  }
#pragma unroll
  for (int o = 1; o < kLanes; o <<= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  return hi > lo ? int2{lo, hi} : int2{0, 1};
}

}  // namespace gsa

// ---------------------------------------------------------------------------
// Host-side checks shared by the entry points.
// ---------------------------------------------------------------------------
namespace gsa_host {

// The plan for nqb query blocks (UnitPlan) with parts of at most `chunk` >= 4
// tiles; n = 0 where nothing is split.
inline gsa::UnitPlan split_plan(int nqb, int nt, int step, int chunk) {
  gsa::UnitPlan p{};
  p.nqb = nqb; p.nt = nt; p.step = step; p.chunk = chunk;
  p.inv = (uint32_t)((((uint64_t)1 << 32) + chunk - 1) / chunk);
  while (p.qs < nqb && p.tiles(p.qs) <= chunk) ++p.qs;
  while (p.qa < p.qs && 4 * p.tiles(p.qa) <= 3 * chunk) ++p.qa;
  for (int qb = p.qs; qb < nqb; ++qb) p.slots += (p.tiles(qb) + chunk - 1) / chunk;
  if (p.slots) p.n = p.qs + p.slots;
  return p;
}

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline int dtype_size(int dtype) {
  return dtype == GSA_DTYPE_BF16 ? 2 : (dtype == GSA_DTYPE_F32 ? 4 : 0);
}
// A [.., T, H*d] tensor read 16 bytes at a time: base and strides must keep
// every 8-element (bf16) or 4-element (fp32) group 16-byte aligned.
inline bool vec_ok(const void* p, int64_t sb, int64_t st, int dtype) {
  const int64_t grp = dtype == GSA_DTYPE_BF16 ? 8 : 4;
  return aligned(p, 16) && (sb % grp) == 0 && (st % grp) == 0;
}
inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? GSA_OK : -static_cast<int>(e);
}

// Variance-based per-row k from per-row variances var[0..n) (indexer.hip):
// k = min(clamp(floor(k_base * max(mean(var),1e-6) / max(var,1e-6)), k_min, k_max), k_cap).
// One launch on `stream`; returns launch_status().
int launch_adaptive_k(const float* var, int n, int k_base, int k_min, int k_max, int k_cap, int32_t* k_rows,
                      hipStream_t stream);

// Zeroes n words (a kernel, so that a graph may record it; dense_attn_f32.hip).
int launch_clear(uint32_t* p, int n, hipStream_t stream);

// Attention over a selection of Tkv keys per row: q, out [B,T,H,128], k, v
// [B,Tkv,H,128], innermost dimensions contiguous, 16-byte aligned rows.
struct AttnShape {
  const void* q; int64_t q_sb, q_st;
  const void* k; int64_t k_sb, k_st;
  const void* v; int64_t v_sb, v_st;
  void* out; int64_t out_sb, out_st;
  int B, T, Tkv, H;
  float scale;
  // RoPE of q and the output gate, by GSA_ATTN_ROPE_Q and GSA_ATTN_OUT_GATE
  const void* og; int64_t o_sb, o_st;
  const void* cos; const void* sin; int64_t cs_st;
  int flags;
};
// The index lists a selection came from (idx64: 64-bit indices; count and mask nullable).
struct IndexLists {
  const void* idx; int idx64; int64_t i_sb, i_st; int k_sel;
  const int32_t* count; const uint8_t* mask;
};
// bf16 on MFMA (dense_attn.hip), without RoPE and gate; ws:
// dense_selected_bytes bytes, 256-byte aligned.
size_t dense_selected_bytes(int B, int T, int Tkv, int H);
int launch_dense_selected(const AttnShape& a, const gsa::Selection& sel, void* ws, hipStream_t stream);
// fp32 on MFMA (dense_attn_f32.hip); sel.range null: a causal selection.
// ws: dense_f32_bytes bytes, 256-byte aligned.
size_t dense_f32_bytes(int B, int T, int Tkv, int H);
int launch_dense_f32(const AttnShape& a, const gsa::Selection& sel, void* ws, hipStream_t stream);
// The gather kernel on what sel.twice and sel.redo mark (sparse_attn.hip).
int launch_gather_rows(const AttnShape& a, const IndexLists& l, const gsa::Selection& sel, int dtype,
                       hipStream_t stream);
// Ascending indices [B*T][k_sel] and counts of the rows of a causal bitmask
// [B*T][2*ceil(T/64)] that `redo` ([B*T*H]) marks (indexer.hip).
int launch_marked_indices(const uint32_t* bits, int B, int T, int k_sel, const uint8_t* redo, int H, int32_t* idx,
                          int32_t* count, hipStream_t stream);

}  // namespace gsa_host
