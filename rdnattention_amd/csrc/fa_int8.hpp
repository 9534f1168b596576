// Parameter block and launch helpers shared by the INT8 attention kernels
// (fa_fwd_int8.hip: head_dim 64 with both GEMMs on int8 MFMA;
// fa_fwd_int8_f16pv.hip: head_dim 128 and the per-token V scale extension,
// with P V on fp16 MFMA).
#pragma once

#include "fa_common.hpp"
#include "fa_host.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

namespace rdna_amd {

constexpr int kI8Waves = 8;
constexpr int kI8Threads = 64 * kI8Waves;
constexpr int kI8BN = 64; // keys per tile = the reference's max-update block (Bc)

constexpr float kLog2Of127 = 6.98868468677f; // log2(127)

// c0 of the scheme's y = 127 p = 2^(s - m + log2 127), evaluated as
// fma(t, qeff, c0) with c0 = log2(127) - m (m = the running max, 0 while it
// is -inf).  The reference clamps pq = min(127, lroundf(127 p))
// (src/rdna/fa2_forward_int8qk.hip:335-339); here the bound comes from c0.
// The block maximum gives y <= 127 * 2^(e), e the rounding of m (from its
// product) and of c0, each within ulp(m): below |m| = 2^15, e <= 2^-8 and
// y <= 127.35 rounds to 127.  Above, c0 is lowered by |m| 2^-21 (at least
// four ulp(m)), so y < 127 there too; those rows' scores carry less than 8
// fractional bits in fp32 anyway.
__device__ __forceinline__ float int8_exp_offset(float m) {
    const float mc = m == -INFINITY ? 0.0f : m;
    const float a = fabsf(mc);
    return (kLog2Of127 - mc) - (a >= 32768.0f ? a * 0x1p-21f : 0.0f);
}

typedef int i2 __attribute__((ext_vector_type(2)));

// ds_read_b64_tr_b8 (gfx950 LDS transpose read).  Within each 16-lane group,
// lane i receives as byte k the byte (i % 8) of the 8-byte word whose address
// lane 2k + i / 8 supplies: if lane j points at row j / 2, bytes 8 (j % 2) ..
// +7 of an 8-row x 16-byte block, lane i gets column i of the block, the
// eight rows' bytes in order.
__device__ __forceinline__ i2 lds_read_tr8(uint32_t lds_byte_addr) {
    typedef __attribute__((address_space(3))) i2 lds_i2;
    const auto* lp = reinterpret_cast<const __attribute__((address_space(3))) char*>(
        lds_byte_addr);
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i2*)lp);
}
__device__ __forceinline__ i2 lds_read_tr8(const int8_t* p) {
    return lds_read_tr8((uint32_t)reinterpret_cast<uintptr_t>(p));
}

// 8 signed bytes -> fp16 (exact: every int8 is an fp16 integer).  Flipping the
// sign bit gives u = v + 128 as an unsigned byte; a byte permute pairs each u with
// the high byte 0x64, i.e. the fp16 value 1024 + u (exact: the ulp in [1024, 2048)
// is 1), and one packed subtract of 1152 leaves v.  Five VALU instructions per 4
// values.
__device__ __forceinline__ h8 widen8(i2 w) {
    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    h2 r[4];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const uint32_t u = (uint32_t)w[c] ^ 0x80808080u;
        // byte selects: 0-3 pick bytes of u, 4 picks byte 0 of 0x64646464
        r[2 * c] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - off;
        r[2 * c + 1] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - off;
    }
    return h8{r[0][0], r[0][1], r[1][0], r[1][1], r[2][0], r[2][1], r[3][0], r[3][1]};
}

struct Int8Params {
    const int8_t* q;
    const int8_t* k;
    const int8_t* v;
    _Float16* o;
    const float* qsv;  // [B, Hq, Sq] or null
    const float* ksv;  // [B, Hkv, Sk] or null
    const float* vch;  // [B, Hkv, D] per-channel V scale or null
    const float* vtok; // [B, Hkv, Sk] per-token V scale (the per-token kernel) or null
    int32_t* scores;   // [B, Hq, Sq, Sk] int32 (the score-export instantiations only)
    float q_scale, k_scale;
    float v_scale;
    float scale_log2e;
    int64_t q_sb, q_sh, q_ss;
    int64_t k_sb, k_sh, k_ss;
    int64_t v_sb, v_sh, v_ss;
    int64_t o_sb, o_sh, o_ss;
    int32_t Hq, Sq, Hkv, ratio, G, rows_per_wg, n_row_tiles, n_head_groups, groups_per_kv;
    int32_t hg_chunk; // head groups per XCD at a time (0 = head groups fastest)
    int32_t n_items;  // n_row_tiles * n_head_groups (* splits)
    MaskSpec mask;
    // key splits of every row tile (see PrefillParams and Int8Mode)
    int32_t splits;
    float* part_o;
    float* part_ml;
    float* row_max; // [splits][n_rows] largest score of each row in each split, log2 units
    int64_t n_rows;
};

// What a prefill kernel instantiation computes.  kWhole: the output of whole
// rows.  The scheme quantises P against the running maximum over all earlier
// keys, so the keys of a row tile are split in two launches: kRowMax finds
// every row's largest score in each split (no softmax, no P V), and kSplit
// starts each split's running maximum at the largest of the earlier ones and
// writes partials for the combine kernel.  kAlternate, for launches of few row
// tiles: both wave groups hold the same 128 rows and take the key tiles in turn
// (PPMode::kAlternate of the FP16 kernel), handing the running maximum to each
// other through LDS from softmax phase to softmax phase, which follow the key
// order; so P is quantised as without it.
enum class Int8Mode { kWhole, kRowMax, kSplit, kAlternate };

// The running maximum that split `split` of a row starts from.
__device__ __forceinline__ float earlier_max(const Int8Params& p, int split, int64_t row) {
    float m = -INFINITY;
    for (int s = 0; s < split; s++) {
        m = fmaxf(m, p.row_max[s * p.n_rows + row]);
    }
    return m;
}

// Kernel parameters and grid size of an INT8 launch.  Returns the number of
// row tiles (workgroups of a one-tile-per-workgroup grid), or -1 with `err`.
int64_t int8_params(const AttnArgs& a, Int8Params& p, std::string& err);

// The kernel with P V on fp16 MFMA (fa_fwd_int8_f16pv.hip): head_dim 128
// (forward and, with `scores`, the score export) and the per-token V scale at
// head_dim 64 or 128.
int launch_int8_f16pv(const Int8Params& p, int head_dim, bool scores, Int8Mode mode, int64_t n_wg,
                      hipStream_t stream, std::string& err);

// Split-K decode (fa_fwd_int8_decode.hip): (Hq / Hkv) * Sq <= 32, head_dim 64
// or 128; and whether a call takes it.
bool int8_splitk_supported(const AttnArgs& a);
bool int8_prefer_splitk(const AttnArgs& a);
int fwd_int8_splitk(const AttnArgs& a, const Int8Params& p, hipStream_t stream, std::string& err);
struct CallPlan;
int int8_decode_plan(const AttnArgs& a, CallPlan& plan, std::string& err);

} // namespace rdna_amd
