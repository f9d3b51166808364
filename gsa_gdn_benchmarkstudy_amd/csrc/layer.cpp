// The layer between its two GEMMs in one call: the fused select, the producer with
// the mask operands, and the dense attention, enqueued on one stream.
//
// For short sequences the host sets the pace: with one Python call, a set of
// tensor views and an event pair per step, a forward of 512 tokens took 260 us
// of which the GPU worked 91.  The steps' own entry points do the checks.
#include "../../include/gsa_hip.h"
#include "layer_steps.h"

namespace {

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Workspace: [selection bitmask][select][RoPE(k)][V^T][mask operands, split blocks].
struct Layout {
  size_t select, k_rope, vt, masks, total;
  Layout(int B, int T, int H, bool adaptive) {
    const size_t W = 2 * (size_t)((T + 63) / 64), rows = (size_t)B * T;
    select = align256(rows * W * 4);
    k_rope = select + align256(adaptive ? gsa_indexer_select_adaptive_workspace_bytes(B, T)
                                        : gsa_indexer_select_workspace_bytes(B, T));
    vt = k_rope + align256(rows * H * 128 * 2);
    masks = vt + align256((size_t)B * H * 128 * ((T + 63) / 64 * 64) * 2);
    total = masks + gsa_dense_attn_workspace_bytes(B, T, T) + gsa_dense_attn_split_bytes(B, T, T, H, 1);
  }
};

}  // namespace

extern "C" size_t gsa_layer_workspace_bytes(int B, int T, int H, int adaptive) {
  if (B < 1 || T < 1 || H < 1 || H > 64) return 0;
  return Layout(B, T, H, adaptive != 0).total;
}

extern "C" int gsa_layer_attn(const void* proj, int64_t p_sb, int64_t p_st, const int64_t* offsets,
                              const float* idx_bias, float idx_scale,
                              const void* cos, const void* sin, int64_t cs_st, const void* halves, int64_t h_st,
                              int B, int T, int H, int d, int Hi, int di, float scale,
                              int k_eff, int k_base, int k_min, int k_max, int32_t* k_out,
                              void* out, int64_t out_sb, int64_t out_st,
                              void* ws, size_t ws_bytes, void* stream) {
  if (!proj || !offsets || !idx_bias || !cos || !sin || !halves || !out || !ws) return GSA_ERR_NULL;
  if (B < 1 || T < 1 || d != 128 || H < 1 || H > 64) return GSA_ERR_SHAPE;
  const bool adaptive = k_eff == 0;
  const Layout at(B, T, H, adaptive);
  if (ws_bytes < at.total) return GSA_ERR_SHAPE;
  if (reinterpret_cast<uintptr_t>(ws) % 256) return GSA_ERR_ALIGN;
  const uint16_t* p = static_cast<const uint16_t*>(proj);
  const uint16_t *q = p + offsets[0], *k = p + offsets[1], *v = p + offsets[2], *vg = p + offsets[3],
                 *og = p + offsets[4], *iq = p + offsets[5], *ik = p + offsets[6], *iw = p + offsets[7];
  char* base = static_cast<char*>(ws);
  uint32_t* bits = reinterpret_cast<uint32_t*>(base);
  const int ntiles = (T + 63) / 64, W = 2 * ntiles, ldv = 64 * ntiles;
  const int64_t b_sb = (int64_t)T * W;
  int st;
  if (adaptive)
    st = gsa_indexer_select_adaptive(iq, p_sb, p_st, ik, p_sb, p_st, iw, p_sb, p_st, idx_bias, idx_scale, B, T, Hi, di,
                                     k_base, k_min, k_max, GSA_DTYPE_BF16, bits, b_sb, W, nullptr, nullptr, k_out,
                                     nullptr, base + at.select, at.k_rope - at.select, stream);
  else
    st = gsa_indexer_select(iq, p_sb, p_st, ik, p_sb, p_st, iw, p_sb, p_st, idx_bias, idx_scale, B, T, Hi, di, k_eff,
                            GSA_DTYPE_BF16, bits, b_sb, W, nullptr, nullptr, base + at.select, at.k_rope - at.select,
                            stream);
  if (st) return st;
  void* k_rope = base + at.k_rope;
  void* vt = base + at.vt;
  const size_t mask_bytes = at.total - at.masks;
  const bool split = gsa_dense_attn_split_bytes(B, T, T, H, 1) != 0;
  st = gsa_host::prologue_vt_lane_masks(k, p_sb, p_st, v, p_sb, p_st, vg, p_sb, p_st, cos, sin, cs_st, B, T, H, d,
                                        GSA_DTYPE_BF16, k_rope, vt, ldv, bits, b_sb, W, T, 1, base + at.masks,
                                        mask_bytes, split, stream);
  if (st) return st;
  const int64_t hd = (int64_t)H * d;
  return gsa_host::dense_attn(
      q, p_sb, p_st, k_rope, T * hd, hd, vt, hd * ldv, (int64_t)d * ldv, ldv, bits, b_sb, W, og, p_sb, p_st, halves,
      nullptr, h_st, out, out_sb, out_st, B, T, T, H, d, scale, GSA_DTYPE_BF16,
      GSA_ATTN_ROPE_Q | GSA_ATTN_OUT_GATE | GSA_ATTN_ROPE_HALVES | GSA_ATTN_MASKS_READY |
          (split ? GSA_ATTN_SPLIT : 0),
      1, base + at.masks, mask_bytes, true, stream);
}
