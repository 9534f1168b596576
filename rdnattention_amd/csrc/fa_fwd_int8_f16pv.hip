// INT8 FlashAttention forward for gfx950 with P V on fp16 MFMA: the kernel for
// head_dim 128 and for the per-token V scale extension (fa_fwd_int8.hip runs
// head_dim 64 with both GEMMs on int8 MFMA).
//
// Q K^T and the softmax follow the reference's scheme (forwardKernelInt8QK,
// src/rdna/fa2_forward_int8qk.hip:229-495):
//
//   S_ij  = sum_d q_i8 k_i8                          (exact int32)
//   s_ij  = S_ij * qs_i * ks_j * scale * log2(e)      (fp32, log2 domain)
//   per 64-key block, aligned to key 0 (the reference's Bc = 64):
//     m'  = max(m, max_j s_ij);  O *= 2^(m - m'),  l *= 2^(m - m')
//     p   = 2^(s - m'),  l += sum p                  (unquantised p)
//     pq  = min(127, round(p * 127))                 (P as integers 0..127)
//     O  += sum_j pq_j v_j
//   out = O * v_scale / (127 l)  (0 when no key is visible)
//
// Why P V runs on fp16 MFMA here: pq (0..127) and v (-127..127) are exact fp16
// integers and their products exact in fp32, and with O and l kept relative
// to a lagging reference m_ref <= m (raised only when m exceeds it by more
// than 2^8) each block's P enters the product as pq * fp16(2^(m - m_ref)), so
// O needs one fp32 accumulator per element and no per-block fold.  Summing
// the blocks in int32 on int8 MFMA instead needs an int32 and an fp32
// accumulator per element and a fold whenever a row maximum moves; at
// head_dim 128 that is 128 registers per 32-row tile, which forces wave pairs
// per tile (128 query rows per workgroup) and measured 1.6x slower than this
// kernel on the causal GQA S = 8192 shape.  At head_dim 64 it is 9 % faster,
// so fa_fwd_int8.hip serves that head dim.
//
// The running max m is exact per block, as the scheme requires (pq depends
// on it).  The P V products pq * fp16(f) are rounded once to fp16 (relative
// 2^-11, values <= 127 * 256) and the row sum uses sum p * the same factor, so
// O / l is the scheme's ratio.
//
// Deliberate differences, all far below the INT8 tolerance: round() is
// round-half-to-even (v_rndne_f32) where the reference calls lroundf (half
// away from zero), 127 p is evaluated as 2^(s - m' + log2 127), the per-block
// v_scale/127 factor is applied once at the end, and P is scaled by the
// reference factor above.
//
// Kernel structure is the FP16 ping-pong design (fa_fwd_f16.hip): 8 waves in
// two groups alternating MFMA and VALU phases, S^T = K Q^T so a lane owns one
// query column, and P^T going from the S accumulator straight into the B
// operand of O^T = V^T P^T.  An MFMA phase issues the Q K^T MFMAs first and
// the P V MFMAs after them, with the dequantisation of the scores riding on
// the P V MFMAs.  Per score the softmax side costs one dequantisation fma
// (the Q K^T chains start at the bit pattern of 1.5 2^23, so the int32 sum
// read as fp32 is 1.5 2^23 + S), half a max3, the exponent fma, the
// exponent, the row-sum add, one v_fma_mix (fp16(1 + 127 p 2^-10) rounds
// 127 p to an integer) and half a packed fma (times the reference factor).  V is converted to fp16 while it is staged into
// LDS (a byte permute against the fp16 exponent of 1024, then one packed
// subtract; with a per-token V scale, fp16(sat(v * vs)) per row) and its V^T
// operands come from ds_read_b64_tr_b16 transpose reads.  The grid is
// persistent (persistent_item), and O leaves through an LDS buffer as
// whole-row non-temporal stores (store_o_tile).
//
// VTOK (an extension; the reference lists a per-token V scale as missing
// because the scale sits inside the P V sum, FEATURES.md:191, :201-202): V
// row j is dequantised by its own scale vs_j while it is staged,
// v'_j = fp16(sat(v_j * vs_j)), and P V runs on these fp16 values.
//
// SCORES (a test instantiation): the same kernel with the softmax, P V and
// output compiled out; every S^T accumulator block its first GEMM produces is
// written to an int32 score buffer, so the tests can check the production
// GEMM's scores bit for bit.
#include "fa_common.hpp"
#include "fa_host.hpp"
#include "fa_internal.hpp"
#include "fa_int8.hpp"
#include "fa_prefill.hpp"
#include "fa_splitk.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace rdna_amd {

#if !defined(RDNATTENTION_NO_INT8)

namespace {

typedef int8_t i8x8 __attribute__((ext_vector_type(8)));

template <int D>
struct I8Cfg {
    // K: int8 rows of D bytes at a D+16 byte stride (16 rows read with
    // ds_read_b128 land in distinct banks); V: converted to fp16 while staged,
    // rows at D+32 halves (conflict-free 4-row transpose reads)
    static constexpr int LDK = D + 16;         // bytes
    static constexpr int LDV = D + 32;         // halves
    static constexpr int TILE_K = kI8BN * LDK; // bytes
    static constexpr int TILE_V = kI8BN * LDV; // halves
    static constexpr int NS = D / 32;          // int8 QK^T reduction steps (32 per MFMA)
    static constexpr int NDT = D / 32;         // O^T row tiles
    static constexpr int KCH = D / 16;         // 16-byte int8 chunks per row
    static constexpr int HALF_TASK = 32 * KCH; // one group's chunks of one K (or V) tile
    static constexpr int CT = (HALF_TASK + 255) / 256;
    static constexpr int LDO = D + 8; // halves; output staging rows (conflict-free like K rows)
};

constexpr int kI8OpDepth = 6;                // MFMA operands in flight in the MFMA phase (4: +1 %)
constexpr float kI8RefThreshold = 8.0f;      // log2 units: P is scaled by at most 2^8 (127 * 256 < 65504)
// Start of the Q K^T chains: the int32 bit pattern of this float (1.5 2^23),
// so the accumulator read as fp32 is kI8Bias + S, exact for |S| < 2^22
constexpr float kI8Bias = 12582912.0f;
// P enters P V as pq f 2^-10 (the quantisation's fp16 step, see phase_v);
// the output factor multiplies the 2^10 back
constexpr float kI8PScale = 0x1p-10f;

__device__ __forceinline__ i4 buffer_load_i4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff = 0) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    u4 x = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return __builtin_bit_cast(i4, x);
}

// 16 signed bytes -> two h8
__device__ __forceinline__ void i8x16_to_h8x2(i4 w, h8& lo, h8& hi) {
    lo = widen8(i2{w[0], w[1]});
    hi = widen8(i2{w[2], w[3]});
}

// 16 signed bytes of one V row -> two h8 of fp16(sat(v * vs)): the product in
// fp32 (v exact, vs as given), saturated to the fp16 range so that no V value
// becomes infinite (a zero P times an infinite V would be NaN for every row
// sharing the tile), then rounded once to fp16
__device__ __forceinline__ void i8x16_to_h8x2_scaled(i4 w, float vs, h8& lo, h8& hi) {
    const i8x8 a = __builtin_bit_cast(i8x8, i2{w[0], w[1]});
    const i8x8 b = __builtin_bit_cast(i8x8, i2{w[2], w[3]});
#pragma unroll
    for (int e = 0; e < 8; e++) {
        lo[e] = (_Float16)__builtin_amdgcn_fmed3f((float)a[e] * vs, -65504.0f, 65504.0f);
        hi[e] = (_Float16)__builtin_amdgcn_fmed3f((float)b[e] * vs, -65504.0f, 65504.0f);
    }
}

// Scheme (the reference's, fa2_forward_int8qk.hip:281-382), per 64-key block b
// aligned to key 0, with s_j = S_j * qs * ks_j * scale * log2(e):
//   m_b  = max(m_{b-1}, max_j s_j)     (exact: pq below depends on it)
//   y_j  = 127 * 2^(s_j - m_b)         (computed as 2^(s_j - m_b + log2 127))
//   pq_j = round(y_j) in [0, 127]
//   f_b  = fp16(2^(m_b - m_ref))       (m_ref <= m_b: raised, with O and l
//                                       rescaled, only when m_b - m_ref > 8)
//   l   += f_b * sum_j y_j              (unquantised p, in units of 1/127)
//   O   += sum_j fp16(pq_j * f_b) v_j
//   out  = O * v_scale / l
// S runs on int8 MFMA (exact int32).  P V runs on fp16 MFMA and accumulates
// straight into fp32, so O needs no per-block int32 -> fp32 conversion.
//
// VTOK (an extension; the reference has no per-token V scale): V row j is
// dequantised by its own scale vs_j while it is staged,
// v'_j = fp16(sat(v_j * vs_j)), and P V runs on these fp16 values.
//
// SCORES: the S^T accumulators of every computed key tile are written to
// p.scores and nothing else is computed (test instantiation).
//
// MODE: see Int8Mode.
template <int D, bool VTOK, bool SCORES>
__global__ __launch_bounds__(kI8Threads, 1) void fa_fwd_int8_f16pv(Int8Params p) {
    constexpr Int8Mode MODE = Int8Mode::kWhole;
#include "fa_int8_f16pv_body.inl"
}

template <int D, bool VTOK, Int8Mode MODE>
__global__ __launch_bounds__(kI8Threads, 1) void fa_fwd_int8_f16pv_split(Int8Params p) {
    constexpr bool SCORES = false;
#include "fa_int8_f16pv_body.inl"
}

template <int D, bool VTOK, bool SCORES>
int launch_f16pv(const Int8Params& p, Int8Mode mode, int64_t n_wg, hipStream_t stream, std::string& err) {
    // persistent: as many workgroups as the device holds at once, each
    // walking its share of the n_wg row tiles
    void (*kernel)(Int8Params) = &fa_fwd_int8_f16pv<D, VTOK, SCORES>;
    if constexpr (!SCORES) {
        if (mode == Int8Mode::kRowMax) {
            kernel = &fa_fwd_int8_f16pv_split<D, VTOK, Int8Mode::kRowMax>;
        } else if (mode == Int8Mode::kSplit) {
            kernel = &fa_fwd_int8_f16pv_split<D, VTOK, Int8Mode::kSplit>;
        } else if (mode == Int8Mode::kAlternate) {
            kernel = &fa_fwd_int8_f16pv_split<D, VTOK, Int8Mode::kAlternate>;
        }
    }
    const int64_t resident = resident_workgroups(reinterpret_cast<const void*>(kernel), kI8Threads, err);
    if (resident <= 0) {
        return -1;
    }
    const int64_t grid = std::min(n_wg, resident);
    KernelTimerGuard timer(stream);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(kI8Threads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = hipGetErrorString(e);
        return -1;
    }
    return 0;
}

} // namespace

int launch_int8_f16pv(const Int8Params& p, int head_dim, bool scores, Int8Mode mode, int64_t n_wg,
                      hipStream_t stream, std::string& err) {
    const bool vtok = p.vtok != nullptr;
    switch (head_dim) {
    case 64:
        if (vtok && !scores) {
            return launch_f16pv<64, true, false>(p, mode, n_wg, stream, err);
        }
        break;
    case 128:
        if (scores) {
            return launch_f16pv<128, false, true>(p, mode, n_wg, stream, err);
        }
        return vtok ? launch_f16pv<128, true, false>(p, mode, n_wg, stream, err)
                    : launch_f16pv<128, false, false>(p, mode, n_wg, stream, err);
    default: break;
    }
    err = "unsupported head_dim for the fp16 P V int8 kernel";
    return -1;
}

#endif

} // namespace rdna_amd
