// Steps of gsa_layer_attn (layer.cpp) that take more than their public entry points.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace gsa_host {

// gsa_prologue_vt_lane_masks; clear: the arrival counters of split query blocks
// behind the masks are cleared too (ws as gsa_dense_attn takes it with
// GSA_ATTN_SPLIT; without the flag nothing past the masks is written).
int prologue_vt_lane_masks(const void* k, int64_t k_sb, int64_t k_st,
                           const void* v, int64_t v_sb, int64_t v_st,
                           const void* vg, int64_t g_sb, int64_t g_st,
                           const void* cos, const void* sin, int64_t cs_st,
                           int B, int T, int H, int d, int dtype,
                           void* k_out, void* vt, int ldv,
                           const uint32_t* bits, int64_t b_sb, int64_t b_st, int Tkv,
                           int causal, void* ws, size_t ws_bytes, bool clear, void* stream);

// gsa_dense_attn; cleared: with GSA_ATTN_MASKS_READY, the mask step has cleared
// the arrival counters of split query blocks too (else a launch here does).
int dense_attn(const void* q, int64_t q_sb, int64_t q_st,
               const void* k, int64_t k_sb, int64_t k_st,
               const void* vt, int64_t vt_sb, int64_t vt_sh, int ldv,
               const uint32_t* bits, int64_t b_sb, int64_t b_st,
               const void* og, int64_t o_sb, int64_t o_st,
               const void* cos, const void* sin, int64_t cs_st,
               void* out, int64_t out_sb, int64_t out_st,
               int B, int T, int Tkv, int H, int d, float scale,
               int dtype, int flags, int causal,
               void* ws, size_t ws_bytes, bool cleared,
               void* stream);

}  // namespace gsa_host
