// Parameter block of the FP16 prefill kernels (device-side headers only).
#pragma once

#include "fa_common.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

namespace rdna_amd {

struct PrefillParams {
    const _Float16* q;
    const _Float16* k;
    const _Float16* v;
    _Float16* o;
    const float* rot_cos;
    const float* rot_sin;
    int64_t q_sb, q_sh, q_ss;
    int64_t k_sb, k_sh, k_ss;
    int64_t v_sb, v_sh, v_ss;
    int64_t o_sb, o_sh, o_ss;
    int32_t Sq, Hkv, ratio;
    int32_t G;             // query heads per workgroup
    int32_t rows_per_wg;   // query rows per head per workgroup (32 * waves / G)
    int32_t n_row_tiles;   // ceil(Sq / rows_per_wg)
    int32_t n_head_groups; // B * Hkv * groups_per_kv
    int32_t groups_per_kv; // ratio / G
    int32_t hg_chunk;      // head groups per XCD at a time (0 = head groups fastest)
    int32_t n_items;       // n_row_tiles * n_head_groups (persistent kernels)
    float c;               // max(|scale| * log2(e), 1e-30)
    float q_sign;          // sign of scale, folded into Q (exact in fp16)
    float qmul;            // q_sign * c: Q pre-scaled into log2 units (kernels that do so, when c <= 1)
    MaskSpec mask;
    int32_t rope_q;        // rotate Q with rot_cos / rot_sin while loading it
    // key splits of every row tile (the split instantiations): the grid has
    // splits * n_row_tiles "row tiles", and each writes its rows' partials
    int32_t splits;
    float* part_o;  // [splits][B * Hq * Sq][D] (SplitRows)
    float* part_ml; // [splits][B * Hq * Sq][2]
    int64_t n_rows; // B * Hq * Sq
};

// Splits row tile index rt of a split grid into row tile and split, and the
// tile's n key tiles from t_begin on into the split's share of them.
__device__ __forceinline__ void split_row_tile(const PrefillParams& p, int& rt, int& split) {
    split = rt / p.n_row_tiles;
    rt -= split * p.n_row_tiles;
}
__device__ __forceinline__ void split_key_tiles(int splits, int split, int& t_begin, int& n) {
    const int per = (n + splits - 1) / splits;
    const int first = min(split * per, n);
    t_begin += first;
    n = min(per, n - first);
}

// Partial of one wave's 32 rows q0 .. q0 + 31 (those < sq) of head h: O^T
// accumulators for columns c0 .. c0 + 32 NDT - 1, unnormalised, relative to m
// with row sum l.  A lane's 16 bytes of a row meet the rest of their cache
// line in the L2 within the next three stores.
template <int NDT>
__device__ __forceinline__ void store_partial(const f16x (&oacc)[NDT], float m, float l, bool write_ml, float* part_o,
                                              float* part_ml, int64_t row, int D, int c0, int g) {
    float* const o = part_o + row * D + c0 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
        for (int qq = 0; qq < 4; qq++) {
            *reinterpret_cast<f4*>(o + 32 * dt + 8 * qq) = f4{oacc[dt][4 * qq], oacc[dt][4 * qq + 1],
                                                             oacc[dt][4 * qq + 2], oacc[dt][4 * qq + 3]};
        }
    }
    if (write_ml) {
        *reinterpret_cast<float2*>(part_ml + row * 2) = float2{m, l};
    }
}

// Head groups an XCD should work through at a time so that their K/V
// (kv_bytes each) fit its L2; 0 when the grid cannot be dealt evenly.
int xcd_head_group_chunk(int n_head_groups, int64_t kv_bytes);

// Prefill for head_dim 160..256 (fa_fwd_f16_kpair.hip): 8 waves, each pair of
// waves 32 rows of one head, so a workgroup holds kKPairRows / G rows of G
// heads (the launcher's PrefillParams must be set up that way).
constexpr int kKPairRows = 128;
int launch_kpair(const PrefillParams& p, int head_dim, int64_t n_wg, hipStream_t stream, std::string& err);

// Prefill for head_dim 288..512 (fa_fwd_f16_dpair.hip): 8 waves, each pair of
// waves 32 rows of one head with the head dimension split between them, so a
// workgroup holds kDPairRows / G rows of G heads (the launcher's
// PrefillParams must be set up that way).
constexpr int kDPairRows = 128;
int launch_dpair(const PrefillParams& p, int head_dim, int64_t n_wg, hipStream_t stream, std::string& err);

} // namespace rdna_amd
