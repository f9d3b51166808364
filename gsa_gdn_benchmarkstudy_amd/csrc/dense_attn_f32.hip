// Block-dense attention over a selection bitmask in fp32, on the fp32 matrix
// instruction.  Same function as the gather kernel (softmax over each row's
// selected keys), with K and V read once per query block instead of once per
// query row.
//
// Block: one head, 128 query rows (4 waves of 32), 32-key tiles of K and V in
// LDS, two slots each, filled by direct global->LDS loads one tile ahead; two
// blocks per CU (66 KiB of LDS each), so that one block's softmax runs beside
// the other's products.  Both products are taken transposed with
// v_mfma_f32_32x32x2_f32,
//   S^T = K Q^T   (A = K tile, B = q in registers)
//   O^T = V^T P^T (A = V tile, B = P in registers)
// so that lane l = 32h + i holds query row i: its softmax state is in two
// lanes and P never moves.  An fp32 operand is one register (2 k positions, one
// per lane half), which leaves the order of the contracted index free:
//   S^T, step (j, e): d = 8j + 4h + e, so that one 16-byte read of a key's row
//     feeds four steps, and RoPE's partner d + 64 is register j + 8 of the lane;
//   O^T, step r: key 8(r/4) + 4h + r%4, the key that score register r holds, so
//     that P is used where it was computed and V needs no transposition; MFMA
//     row rho of block dt is dim 4 rho + dt, so that one 16-byte read of V feeds
//     the four blocks and a lane's outputs are 16-byte pieces.
// K rows are padded to 33 16-byte units (an odd stride: operand reads of 32
// rows do not collide); V is read by whole rows and needs no padding.
//
// What bounds it: the fp32 matrix instruction, 128 of 64 cycles per wave and
// 32-key tile (157 TFLOP/s nominal; a large fp32 matrix product of the library
// reaches 133 here); the softmax is about 200 VALU instructions beside them.  At
// T = 8192, H = 16 a causal call executes 0.279 TFLOP in 2.3 ms: 121 TFLOP/s,
// where the gather of k = 2048 keys took 25.8 ms.
#include "gsa_common.h"

#include <cmath>

namespace gsa {

constexpr int kFRows = 128;               // query rows per block
constexpr int kFKeys = 32;                // keys per tile
constexpr int kFKRow = 33;                // K row: 32 units of 16 bytes and one of padding
constexpr int kFKInstr = 17;              // load instructions (64 units) per K tile: 1056 units
constexpr int kFVInstr = 16;              // and per V tile: 1024 units
constexpr int kFSlot = (kFKInstr + kFVInstr) * 64;   // units of one K + V slot pair

struct DenseF32Args {
  const float* q; int64_t q_sb, q_st;
  const float* k; int64_t k_sb, k_st;
  const float* v; int64_t v_sb, v_st;
  const uint32_t* bits; int W;            // [B*T][W]
  const int2* range;                      // Selection::range, or null: causal
  uint8_t* redo;
  const float* og; int64_t o_sb, o_st;
  const float* cos; const float* sin; int64_t cs_st;
  float* out; int64_t out_sb, out_st;
  int B, T, Tkv, H, nqb;
  float scale_l2;
  int flags;
  float* parts; uint32_t* counters;       // plan.n > 0: slots [B*H][plan.slots], arrivals [B*H][nqb]
};

__global__ __launch_bounds__(256, 2) void dense_attn_f32_kernel(DenseF32Args p, UnitPlan plan) {
  extern __shared__ __align__(16) u32x4 dsm[];       // slot s: K units, then V units
  const int tid = threadIdx.x, lane = tid & 63;
  const int wu = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i32 = lane & 31, h = lane >> 5;
  // heads fastest (a head's blocks share an XCD's L2), heaviest query blocks first
  int b, qb, hd;
  Unit unit{0, 0, 1, 0};
  if (plan.n) {
    hd = blockIdx.x % p.H;
    b = blockIdx.x / p.H % p.B;
    unit = plan_unit(plan, blockIdx.x / (p.H * p.B));
    qb = unit.qb;
  } else {
    const int per_b = p.nqb * p.H, r2 = blockIdx.x % per_b;
    b = blockIdx.x / per_b;
    qb = p.nqb - 1 - r2 / p.H;
    hd = r2 % p.H;
  }
  const int q0 = qb * kFRows;
  const int row = q0 + 32 * wu + i32, rowc = min(row, p.T - 1);

  // the block's 32-key tiles [kt0, kt0 + nkt)
  int kt0 = 0, nkt = (min(p.Tkv, q0 + kFRows) + kFKeys - 1) / kFKeys;
  if (p.range) {
    const int2 tr = tile_range<64>(p.range, (int64_t)b * p.T, q0, min(q0 + kFRows, p.T));
    kt0 = 2 * __builtin_amdgcn_readfirstlane(tr.x);
    nkt = min(2 * __builtin_amdgcn_readfirstlane(tr.y), (p.Tkv + kFKeys - 1) / kFKeys) - kt0;
  }
  const int parts = min(unit.parts, nkt);
  if (parts > 1) {                         // this unit's share of them (a part past the tiles has none)
    if (unit.part >= parts) return;
    const int t0 = nkt * unit.part / parts, t1 = nkt * (unit.part + 1) / parts;
    kt0 += t0;
    nkt = t1 - t0;
  } else if (unit.part) {
    return;
  }

  // ---- tile loads: wave w issues instructions w, w + 4, ... of a tile's 17 (K)
  // and 16 (V).  K instruction i fills units 64i .. 64i+63 (key u/33, unit
  // u%33; units past the row or the tile re-read a valid one), V instruction i
  // keys 2i and 2i+1.  Keys past Tkv-1 re-read key Tkv-1 (never selected).
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(dsm));
  const float* kbase = p.k + b * p.k_sb + hd * 128;
  const float* vbase = p.v + b * p.v_sb + hd * 128;
  const uint32_t kst = (uint32_t)p.k_st * 4u, vst = (uint32_t)p.v_st * 4u;
  constexpr int kNK = (kFKInstr + 3) / 4, kNV = kFVInstr / 4;
  int kkey[kNK];
  uint32_t kcol[kNK];
#pragma unroll
  for (int n = 0; n < kNK; ++n) {
    const int u = min((4 * n + wu) * 64 + lane, kFKeys * kFKRow - 1);
    kkey[n] = u / kFKRow;
    kcol[n] = (uint32_t)min(u - kkey[n] * kFKRow, 31) * 16u;
  }
  const uint32_t vcol = (uint32_t)i32 * 16u;
  auto issue = [&](int t) __attribute__((always_inline)) {   // tile kt0 + t into slot t & 1
    const int j0 = (kt0 + t) * kFKeys, last = p.Tkv - 1 - j0;
    const float* kb = kbase + j0 * p.k_st;
    const float* vb = vbase + j0 * p.v_st;
    const uint32_t dst = lds0 + (uint32_t)((t & 1) * kFSlot * 16 + wu * 1024);
#pragma unroll
    for (int n = 0; n < kNK; ++n)
      if (4 * n + wu < kFKInstr) load_lds16(kb, (uint32_t)min(kkey[n], last) * kst + kcol[n], dst + n * 4096u);
#pragma unroll
    for (int n = 0; n < kNV; ++n)
      load_lds16(vb, (uint32_t)min(2 * (4 * n + wu) + h, last) * vst + vcol, dst + (uint32_t)(kFKInstr * 1024) + n * 4096u);
  };
  const uint32_t* wrow = p.bits + ((int64_t)b * p.T + rowc) * p.W + kt0;
  issue(0);
  uint32_t word = row < p.T ? wrow[0] : 0u;

  // ---- q: step (j, e) of S^T: d = 8j + 4h + e ----
  floatx4 q[16];
  {
    const float* qp = p.q + b * p.q_sb + (int64_t)rowc * p.q_st + hd * 128 + 4 * h;
#pragma unroll
    for (int j = 0; j < 16; ++j) q[j] = *reinterpret_cast<const floatx4*>(qp + 8 * j);
    if (p.flags & GSA_ATTN_ROPE_Q) {
      const float* cp = p.cos + (int64_t)rowc * p.cs_st + 4 * h;
      const float* sp = p.sin + (int64_t)rowc * p.cs_st + 4 * h;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const floatx4 c0 = *reinterpret_cast<const floatx4*>(cp + 8 * j);
        const floatx4 c1 = *reinterpret_cast<const floatx4*>(cp + 8 * j + 64);
        const floatx4 s0 = *reinterpret_cast<const floatx4*>(sp + 8 * j);
        const floatx4 s1 = *reinterpret_cast<const floatx4*>(sp + 8 * j + 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = q[j][e], hi = q[j + 8][e];
          const float a = lo * c0[e], r = -hi * s0[e], c = hi * c1[e], z = lo * s1[e];
          q[j][e] = a + r;
          q[j + 8][e] = c + z;
        }
      }
    }
  }

  floatx16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  // softmax state of the lane's row, log2 domain: the reference m moves only when
  // a tile's maximum exceeds it by more than kLazyF (as in dense_attn.hip)
  constexpr float kLazyF = 8.f;
  float m = -__builtin_inff(), mlz = -__builtin_inff(), nm = 0.f, l = 0.f;
  const int kread = i32 * kFKRow + h;                            // + 2j units: d = 8j + 4h
  const int vread = kFKInstr * 64 + 4 * h * 32 + i32;            // + (8(r/4) + r%4) rows of 32 units

  for (int t = 0; t < nkt; ++t) {
    // this wave's loads of tile t have landed (the compiler's own wait, so that
    // it also knows its bitmask word to be there); the barrier publishes every
    // wave's and frees the other slot
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint32_t w = word >> (4 * h);
    if (t + 1 < nkt) {
      word = row < p.T ? wrow[t + 1] : 0u;
      issue(t + 1);
    }
    const u32x4* slot = dsm + (t & 1) * kFSlot;
    // four sums of 32 products each, then their tree: the rounding of one chain
    // of 128 would be the largest error of the output
    floatx16 sp[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int r = 0; r < 16; ++r) sp[e][r] = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const floatx4 f = __builtin_bit_cast(floatx4, slot[kread + 2 * j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) sp[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[e], q[j][e], sp[e], 0, 0, 0);
    }
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = (sp[0][r] + sp[1][r]) + (sp[2][r] + sp[3][r]);
    float mx = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = (w & (1u << (8 * (r >> 2) + (r & 3)))) ? s[r] : -__builtin_inff();
      mx = fmaxf(mx, s[r]);
    }
    mx = max_halves(mx) * p.scale_l2;
    if (ballot64(mx > mlz)) {                                    // some row's reference moves
      const bool bump = mx > mlz;
      const float alpha = bump ? __builtin_amdgcn_exp2f(m - mx) : 1.f;   // m = -inf -> 0
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      l *= alpha;
      m = bump ? mx : m;
      mlz = m + kLazyF;
      nm = m == -__builtin_inff() ? 0.f : -m;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], p.scale_l2, nm));
      l += s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const floatx4 f = __builtin_bit_cast(floatx4, slot[vread + (8 * (r >> 2) + (r & 3)) * 32]);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[dt], s[r], o[dt], 0, 0, 0);
    }
  }

  // ---- epilogue: normalise, optional output gate; dims 4(8(r/4) + 4h + r%4) + dt ----
  l = sum_halves(l);
  if (parts > 1) {
    const int64_t bh = (int64_t)b * p.H + hd;
    __syncthreads();                       // the tile slots are free: dsm[0] carries the arrival count
    if (!merge_parts(o, m, l, p.parts + (bh * plan.slots + unit.slot) * (4 * kPartWave), unit.part, parts, 4, wu, lane,
                     p.counters + bh * p.nqb + qb, reinterpret_cast<uint32_t*>(dsm)))
      return;
  }
  float z = 0.f;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) z = __builtin_fmaf(o[dt][r], 0.f, z);
  if (row >= p.T) return;
  // a row whose sums are not positive finite numbers goes to the gather kernel
  // (no valid key, or infinities or NaN in its tiles, which a zero weight does not stop)
  mark_row(p.redo + ((int64_t)b * p.T + row) * p.H + hd, l > 0.f && l < __builtin_inff() && z == 0.f);
  float* op = p.out + b * p.out_sb + (int64_t)row * p.out_st + hd * 128;
  const float* gp = p.og + b * p.o_sb + (int64_t)row * p.o_st + hd * 128;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int d = 4 * (8 * (r >> 2) + 4 * h + (r & 3));
    floatx4 y;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) y[dt] = l > 0.f ? o[dt][r] / l : 0.f;
    if (p.flags & GSA_ATTN_OUT_GATE) {
      const floatx4 gl = *reinterpret_cast<const floatx4*>(gp + d);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) y[dt] *= sigmoidf_fast(gl[dt]);
    }
    *reinterpret_cast<floatx4*>(op + d) = y;
  }
}

}  // namespace gsa

using namespace gsa_host;

namespace {

__global__ __launch_bounds__(256) void clear_kernel(uint32_t* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// How the query blocks are split, by sizes alone (query and key length alike are
// taken for causal): into parts of 0.6 of a CU's mean share of the tiles while
// that is small (fewer parts, less to add up), 0.33 beyond (finer parts, a shorter
// tail), 4 tiles at least.  16 heads, causal, us without / with (parts of 0.33
// and 0.6 of the share): T = 512 96 / 60 60, T = 1537 230 / 166 147, T = 2048
// 298 / 226 191, B = 2 T = 1537 382 / 250 275, T = 3000 537 / 378 426, T = 4096
// 815 / 611 725, B = 2 T = 4096 1225 / 1160 1224.
gsa::UnitPlan f32_plan(int B, int T, int Tkv, int H) {
  const int nqb = (T + gsa::kFRows - 1) / gsa::kFRows, nt = (Tkv + gsa::kFKeys - 1) / gsa::kFKeys;
  const int step = T == Tkv ? gsa::kFRows / gsa::kFKeys : 0;
  const double tiles = step ? 0.5 * step * nqb * (nqb + 1) : (double)nt * nqb;
  const double share = tiles * B * H / 256;
  return split_plan(nqb, nt, step, (int)std::max(4.0, std::ceil(share * (share < 40 ? 0.6 : 0.33))));
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t counter_bytes(int B, int T, int H) {
  return align256((size_t)B * H * ((T + gsa::kFRows - 1) / gsa::kFRows) * sizeof(uint32_t));
}

}  // namespace

int gsa_host::launch_clear(uint32_t* p, int n, hipStream_t stream) {
  hipLaunchKernelGGL(clear_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, p, n);
  return launch_status();
}

size_t gsa_host::dense_f32_bytes(int B, int T, int Tkv, int H) {
  const gsa::UnitPlan plan = f32_plan(B, T, Tkv, H);
  if (!plan.n) return 0;
  return counter_bytes(B, T, H) + (size_t)B * H * plan.slots * 4 * gsa::kPartWave * sizeof(float);
}

int gsa_host::launch_dense_f32(const AttnShape& s, const gsa::Selection& sel, void* ws, hipStream_t stream) {
  constexpr int kMaxDevices = 64;
  constexpr size_t kLds = (size_t)2 * gsa::kFSlot * 16;
  static bool done[kMaxDevices] = {};        // (a benign race: concurrent first calls set the same attribute)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return GSA_ERR_SHAPE;
  if (!done[dev]) {                          // more than the default 64 KiB of LDS per block
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gsa::dense_attn_f32_kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    if (e != hipSuccess) return -static_cast<int>(e);
    done[dev] = true;
  }
  const int nqb = (s.T + gsa::kFRows - 1) / gsa::kFRows;
  const gsa::UnitPlan plan = f32_plan(s.B, s.T, s.Tkv, s.H);
  uint32_t* counters = static_cast<uint32_t*>(ws);
  float* parts = reinterpret_cast<float*>(static_cast<char*>(ws) + counter_bytes(s.B, s.T, s.H));
  if (plan.n) {
    const int st = launch_clear(counters, s.B * s.H * nqb, stream);
    if (st) return st;
  }
  const gsa::DenseF32Args a{
      static_cast<const float*>(s.q), s.q_sb, s.q_st, static_cast<const float*>(s.k), s.k_sb, s.k_st,
      static_cast<const float*>(s.v), s.v_sb, s.v_st, sel.bits, 2 * ((s.Tkv + 63) / 64), sel.range, sel.redo,
      static_cast<const float*>(s.og), s.o_sb, s.o_st, static_cast<const float*>(s.cos),
      static_cast<const float*>(s.sin), s.cs_st, static_cast<float*>(s.out), s.out_sb, s.out_st,
      s.B, s.T, s.Tkv, s.H, nqb, s.scale * gsa::kLog2e, s.flags, parts, counters};
  hipLaunchKernelGGL(gsa::dense_attn_f32_kernel, dim3(s.B * s.H * (plan.n ? plan.n : nqb)), dim3(256), kLds, stream, a,
                     plan);
  return launch_status();
}
