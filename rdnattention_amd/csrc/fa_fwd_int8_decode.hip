// INT8 split-K decode for gfx950: few query rows per kv head.  The prefill
// kernels put 256 query rows in a workgroup, so one decode row per head left
// 255 of them and most CUs idle.
//
// The scheme is the prefill kernels' (fa_fwd_int8_f16pv.hip): exact int32 S,
// the running max per 64-key block in key order, P quantised to integers 0..127
// against it, l from the unquantised p, P V on fp16 MFMA (both factors are
// exact fp16 integers).  P's step follows the largest score of ALL earlier
// keys, which a workgroup that takes the keys of one split does not see; with
// its own maximum instead the result is another one (1.6e-2 max-abs from the
// scheme on a causal S = 600 prompt of N(0, 1), more than the INT8 bar, although
// no further from float64).  So two launches:
//
//   fa_int8_decode_scores  K once: t = S ks per (column, key) and the maximum
//                          per (column, 64-key block) into scratch
//   fa_int8_decode_pv      V once: the running maximum at each block from the
//                          block maxima, P, P V, and the merge of
//                          fa_fwd_decode.hip
//
// What bounds both is the cache's bytes (t adds M / D of K's four times over:
// an eighth for 4 rows at D = 128).  Grid (splits, B * Hkv), the M = ratio *
// Sq <= 32 rows of a kv head as the 32 columns of the MFMAs, eight waves on
// interleaved 64-key tiles, one slot each, filled by non-temporal HBM -> LDS
// DMA; two workgroups fit a CU (of TC = 4), and where a launch has as many some
// waves' tiles are in flight while others compute.  V stays int8 in LDS; its
// operands come from ds_read_b64_tr_b8 transpose reads and are widened to fp16 in
// registers.
//
// B = 8 Hq = 32 Hkv = 8 Sk = 8192 D = 128 (136 MB): 16.9 us (scores),
// 18.6 us (P V) and 4.2 us (merge), 43 us a call; on the prefill kernel 205.  One
// launch with each wave's own maximum: 27.4 + 4.2, 32 us a call.
#include "fa_common.hpp"
#include "fa_host.hpp"
#include "fa_int8.hpp"
#include "fa_internal.hpp"
#include "fa_splitk.hpp"

#include <algorithm>
#include <type_traits>

namespace rdna_amd {

#if !defined(RDNATTENTION_NO_INT8)

namespace {

constexpr int kI8DecWaves = 8;
constexpr int kI8DecThreads = 64 * kI8DecWaves;

struct Int8DecodeParams {
    Int8Params a;
    SplitRows out;
    int32_t keys_per_split, key0;
    int32_t blocks; // 64-key blocks from key0 on
    float* t;       // [B*Hkv][blocks][16][TC][4] scores (see t_index)
    float* bmax;    // [B*Hkv][blocks][TC] block maxima, log2 units
};

// Columns kept in the scratch: the M <= 32 rows rounded up to 4 or 32.
// Scores of a block: key 8 i + 4 g + e of column c at ((2 i + g) TC + c) 4 + e,
// so that a half-wave's accesses of 16 bytes per column are contiguous.
template <int TC>
struct TCfg {
    static constexpr int BLOCK_FLOATS = kI8BN * TC;
    static constexpr int DMAS = BLOCK_FLOATS * 4 / 1024;
    static constexpr int MAX_TILES = TC == 4 ? 256 : 128; // of one split, whose block maxima are in LDS
};

template <int D>
struct I8DecCfg {
    static constexpr int RB = D;                  // row bytes (unpadded)
    static constexpr int TILE_BYTES = kI8BN * RB; // one K (or V) tile
    static constexpr int SCALE_BYTES = 4 * kI8BN; // one scale per key
    static constexpr int NS = D / 32;  // int8 Q K^T steps
    static constexpr int NDT = D / 32; // O^T row tiles
};

// XOR swizzle of the 16-byte chunk index of row r.  Rows r and r + 2 (D = 128,
// 8 chunks) or r + 4 (D = 64, 4 chunks) start in the same bank.  The K read
// takes one chunk of 16 consecutive rows, a transpose read of V one pair of
// chunks of rows {0..3, 8..11} (+ 4): the first wants all of a residue's
// rows apart, the second rows r and r + 8 in different pairs, hence row bit 3
// above row bit 2 at D = 128 (at D = 64 it is the upper of the two already).
template <int D>
__device__ __forceinline__ int i8dec_swz(int r) {
    if constexpr (D == 128) {
        return (((r >> 1) & 1) << 2) | (((r >> 3) & 1) << 1) | ((r >> 2) & 1);
    } else {
        return (r >> 2) & 3;
    }
}

// DMA source offsets of a tile with row stride `ss`: lane i of DMA j writes LDS
// bytes 1024 j + 16 i of the tile, i.e. stored chunk n % KCH of row r = n / KCH
// with n = 64 j + i, which holds logical chunk (n % KCH) ^ swz(r).  A DMA moves
// 1024 / D rows; of j the swizzle depends on j % 2 at most (row bit 3), so two
// vector offsets and the DMA's rows as the scalar offset do.
template <int D>
struct TileOffsets {
    uint32_t v[2];
    uint32_t rows_b; // bytes from one DMA's rows to the next

    __device__ __forceinline__ TileOffsets(int64_t ss, int lane) {
        constexpr int KCH = D / 16;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = 64 * j + lane;
            const int r = n / KCH;
            v[j] = (uint32_t)((int64_t)(lane / KCH) * ss + 16 * ((n - r * KCH) ^ i8dec_swz<D>(r)));
        }
        rows_b = (uint32_t)(1024 / D * ss);
    }
    __device__ __forceinline__ void issue(i32x4_t rsrc, uint32_t lds) const {
#pragma unroll
        for (int j = 0; j < kI8BN * D / 1024; j++) {
            dma_load16_nt_s(rsrc, v[j & 1], j * rows_b, lds + 1024 * j);
        }
    }
};

// 8 signed bytes of 8 keys with the scales lo (keys 0..3) and hi (4..7):
// fp16(sat(v * vs)), as the prefill kernel stages a per-token-scaled V row
__device__ __forceinline__ h8 widen8_scaled(i2 w, f4 lo, f4 hi) {
    typedef int8_t i8x8 __attribute__((ext_vector_type(8)));
    const i8x8 a = __builtin_bit_cast(i8x8, w);
    h8 r;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        r[e] = (_Float16)__builtin_amdgcn_fmed3f((float)a[e] * lo[e], -65504.0f, 65504.0f);
        r[e + 4] = (_Float16)__builtin_amdgcn_fmed3f((float)a[e + 4] * hi[e], -65504.0f, 65504.0f);
    }
    return r;
}

// What both kernels start from: this workgroup's (b, kv head), its columns and
// its 64-key tiles.
struct DecWork {
    int b, kvh, q, h;       // of this lane's column
    bool col_valid;
    int blk0;               // first tile, as a block from key0 on
    int nt;                 // tiles
    int kt_first;           // first key of that tile
};

__device__ __forceinline__ DecWork dec_work(const Int8DecodeParams& pp, int l32) {
    const Int8Params& p = pp.a;
    DecWork w;
    const int bkv = blockIdx.y;
    w.b = bkv / p.Hkv;
    w.kvh = bkv - w.b * p.Hkv;
    // column l32 <-> (query head, query row)
    w.col_valid = l32 < p.ratio * p.Sq;
    const int hoff = w.col_valid ? l32 / p.Sq : 0;
    w.q = w.col_valid ? l32 - hoff * p.Sq : 0;
    w.h = w.kvh * p.ratio + hoff;
    // this split's tiles, restricted to what any of the M rows can see
    const int k_begin = pp.key0 + blockIdx.x * pp.keys_per_split;
    const int k_end = min(k_begin + pp.keys_per_split, p.mask.sk);
    int vis_lo, vis_hi;
    visible_key_range(p.mask, 0, p.Sq - 1, vis_lo, vis_hi);
    const int lo = max(k_begin, vis_lo);
    const int hi = min(k_end - 1, vis_hi);
    w.nt = 0;
    w.kt_first = k_begin;
    if (hi >= lo) {
        w.kt_first = lo / kI8BN * kI8BN;
        w.nt = hi / kI8BN + 1 - lo / kI8BN;
    }
    w.blk0 = (w.kt_first - pp.key0) / kI8BN;
    return w;
}

// qeff of a column: its scores are t qeff in log2 units, qeff > 0 (t carries the
// factor itself where that is not positive)
__device__ __forceinline__ float dec_qc(const Int8Params& p, const DecWork& w) {
    const float qs =
        p.qsv != nullptr && w.col_valid ? p.qsv[((int64_t)w.b * p.Hq + w.h) * p.Sq + w.q] : p.q_scale;
    return qs * p.scale_log2e;
}

template <int D, int TC>
__global__ __launch_bounds__(kI8DecThreads, 4) void fa_int8_decode_scores(Int8DecodeParams pp) {
    using C = I8DecCfg<D>;
    constexpr int WAVE_BYTES = C::TILE_BYTES + 2 * C::SCALE_BYTES; // K, its scales (two slots)
    __shared__ __attribute__((aligned(16))) char dsm[kI8DecWaves * WAVE_BYTES];
    const Int8Params& p = pp.a;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // wave-uniform
    const int lane = threadIdx.x & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const DecWork w = dec_work(pp, l32);
    const int my_tiles = w.nt > wave ? (w.nt - wave + kI8DecWaves - 1) / kI8DecWaves : 0;

    const int8_t* kbase = p.k + w.b * p.k_sb + w.kvh * p.k_sh;
    const float* ksrow = p.ksv != nullptr ? p.ksv + ((int64_t)w.b * p.Hkv + w.kvh) * p.mask.sk : nullptr;
    const char* wsm = dsm + wave * WAVE_BYTES;
    const uint32_t lds_k = (uint32_t)reinterpret_cast<uintptr_t>(wsm);
    const TileOffsets<D> kto(p.k_ss, lane);
    auto issue_k = [&](int j_tile) {
        const int kt0 = w.kt_first + (wave + kI8DecWaves * j_tile) * kI8BN;
        const i32x4_t r = make_rsrc_v(kbase + (int64_t)kt0 * p.k_ss,
                                      tile_bytes<kI8BN>(p.mask.sk - kt0, (uint32_t)p.k_ss, D));
        kto.issue(r, lds_k);
        // its scales, a dword per lane (those past Sk read as 0)
        if (ksrow != nullptr) {
            const int left = min(p.mask.sk - kt0, kI8BN);
            dma_load4(make_rsrc_v(ksrow + kt0, left > 0 ? 4u * (uint32_t)left : 0u), 4u * lane,
                      lds_k + C::TILE_BYTES + (j_tile & 1) * C::SCALE_BYTES);
        }
    };
    // the first tile leaves before the Q loads: one memory round trip, not two
    if (my_tiles > 0) {
        issue_k(0);
    }
    // Q^T operand: lane holds Q[q][32 s + 16 g .. +15]
    i4 qreg[C::NS];
    const int8_t* qrow = p.q + w.b * p.q_sb + w.h * p.q_sh + (int64_t)w.q * p.q_ss;
#pragma unroll
    for (int s = 0; s < C::NS; s++) {
        qreg[s] = w.col_valid ? *reinterpret_cast<const i4*>(qrow + 32 * s + 16 * g) : i4{};
    }
    const float qc = dec_qc(p, w);
    const float qeff = qc > 0.0f ? qc : 1.0f;
    const float tmul = qc > 0.0f ? 1.0f : qc;
    int row_lo = 1, row_hi = 0; // an unused column sees nothing
    if (w.col_valid) {
        row_key_bounds(p.mask, w.q, row_lo, row_hi);
    }

    for (int j = 0; j < my_tiles; j++) {
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // K(j) and its scales landed
        const int kt0 = w.kt_first + (wave + kI8DecWaves * j) * kI8BN;
        // S^T[key][col] = K Q^T, two blocks of 32 keys
        i16x sacc[2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
            const int r = 32 * kt + l32;
            const char* krow = wsm + r * C::RB;
            const int sw = i8dec_swz<D>(r);
            sacc[kt] = i16x{};
#pragma unroll
            for (int s = 0; s < C::NS; s++) {
                const i4 a = *reinterpret_cast<const i4*>(krow + (((2 * s + g) ^ sw) << 4));
                sacc[kt] = mfma_32x32x32_i8(a, qreg[s], sacc[kt]);
            }
        }
        if (j + 1 < my_tiles) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of K(j) has returned
            issue_k(j + 1);
        }
        const int64_t blk = (int64_t)blockIdx.y * pp.blocks + w.blk0 + wave + kI8DecWaves * j;
        float* const tb = pp.t + blk * TCfg<TC>::BLOCK_FLOATS + (g * TC + l32) * 4;
        const float* ksl = reinterpret_cast<const float*>(wsm + C::TILE_BYTES + (j & 1) * C::SCALE_BYTES) + 4 * g;
        const int a = row_lo - kt0 - 4 * g;
        const int bnd = row_hi - kt0 - 4 * g;
        float mx[8];
#pragma unroll
        for (int i = 0; i < 8; i++) { // keys 8 i + 4 g .. +3
            f4 ks = {p.k_scale, p.k_scale, p.k_scale, p.k_scale};
            if (ksrow != nullptr) {
                ks = *reinterpret_cast<const f4*>(ksl + 8 * i);
            }
            f4 t;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = (float)sacc[i >> 2][4 * (i & 3) + e] * ks[e];
                t[e] = (8 * i + e < a || 8 * i + e > bnd) ? -INFINITY : x * tmul;
            }
            mx[i] = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
            if (l32 < TC) {
                *reinterpret_cast<f4*>(tb + 2 * i * TC * 4) = t;
            }
        }
        const float m = pair_max(max_tree<8>([&](int e) { return mx[e]; })) * qeff; // -inf stays -inf
        if (g == 0 && l32 < TC) {
            pp.bmax[blk * TC + l32] = m;
        }
    }
}

template <int D, bool VTOK, int TC>
__global__ __launch_bounds__(kI8DecThreads, TC == 4 && !(VTOK && D == 128) ? 4 : 2) void fa_int8_decode_pv(Int8DecodeParams pp) {
    using C = I8DecCfg<D>;
    using T = TCfg<TC>;
    constexpr int T_BYTES = T::BLOCK_FLOATS * 4;
    constexpr int WAVE_BYTES = C::TILE_BYTES + T_BYTES + (VTOK ? C::SCALE_BYTES : 0); // V, t, V scales
    constexpr int BM_FLOATS = T::MAX_TILES * TC;
    constexpr int TILES = kI8DecWaves * WAVE_BYTES;
    constexpr int FINISH = finish_lds_bytes(D, kI8DecWaves);
    static_assert(TILES + BM_FLOATS * 4 <= (TC == 4 ? 80 : 160) * 1024, "LDS");
    // the tiles, then the split's block maxima; the merge reuses both
    __shared__ __attribute__((aligned(16))) char dsm[TILES + BM_FLOATS * 4 > FINISH ? TILES + BM_FLOATS * 4 : FINISH];
    float* const sm_bm = reinterpret_cast<float*>(dsm + TILES);
    const Int8Params& p = pp.a;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // wave-uniform
    const int lane = tid & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int c = l32 < TC ? l32 : TC - 1; // column in the scratch
    const DecWork w = dec_work(pp, l32);
    const int my_tiles = w.nt > wave ? (w.nt - wave + kI8DecWaves - 1) / kI8DecWaves : 0;

    const int8_t* vbase = p.v + w.b * p.v_sb + w.kvh * p.v_sh;
    const float* vsrow = VTOK ? p.vtok + ((int64_t)w.b * p.Hkv + w.kvh) * p.mask.sk : nullptr;
    const char* wsm = dsm + wave * WAVE_BYTES;
    const uint32_t lds_v = (uint32_t)reinterpret_cast<uintptr_t>(wsm);
    const uint32_t lds_t = lds_v + C::TILE_BYTES;
    const float* const group_t = pp.t + (int64_t)blockIdx.y * pp.blocks * T::BLOCK_FLOATS;
    const TileOffsets<D> vto(p.v_ss, lane);
    auto issue = [&](int j_tile) {
        const int n = wave + kI8DecWaves * j_tile;
        const int kt0 = w.kt_first + n * kI8BN;
        const i32x4_t rt = make_rsrc_v(group_t + (int64_t)(w.blk0 + n) * T::BLOCK_FLOATS, T_BYTES);
#pragma unroll
        for (int j = 0; j < T::DMAS; j++) {
            dma_load16(rt, 1024 * j + 16 * lane, lds_t + 1024 * j);
        }
        const i32x4_t r = make_rsrc_v(vbase + (int64_t)kt0 * p.v_ss,
                                      tile_bytes<kI8BN>(p.mask.sk - kt0, (uint32_t)p.v_ss, D));
        vto.issue(r, lds_v);
        if constexpr (VTOK) {
            const int left = min(p.mask.sk - kt0, kI8BN);
            dma_load4(make_rsrc_v(vsrow + kt0, left > 0 ? 4u * (uint32_t)left : 0u), 4u * lane, lds_t + T_BYTES);
        }
    };
    if (my_tiles > 0) {
        issue(0);
    }
    const float qc = dec_qc(p, w);
    const float qeff = qc > 0.0f ? qc : 1.0f;

    // this split's block maxima to LDS, and the maximum over all earlier blocks:
    // every thread over its column's blocks, then over the threads
    const float* const bm = pp.bmax + (int64_t)blockIdx.y * pp.blocks * TC;
    float before = -INFINITY;
    for (int i = tid; i < w.blk0 * TC; i += kI8DecThreads) { // column i % TC = tid % TC
        before = fmaxf(before, bm[i]);
    }
    for (int i = tid; i < w.nt * TC; i += kI8DecThreads) {
        sm_bm[i] = bm[w.blk0 * TC + i];
    }
#pragma unroll
    for (int off = 32; off >= TC; off >>= 1) {
        before = fmaxf(before, __shfl_xor(before, off));
    }
    __shared__ float sm_before[kI8DecWaves * TC]; // [wave][column]
    if (lane < TC) {
        sm_before[wave * TC + lane] = before;
    }
    __syncthreads();
    float m_run = -INFINITY;
#pragma unroll
    for (int i = 0; i < kI8DecWaves; i++) {
        m_run = fmaxf(m_run, sm_before[i * TC + c]);
    }

    f16x oacc[C::NDT];
#pragma unroll
    for (int dt = 0; dt < C::NDT; dt++) {
        oacc[dt] = f16x{};
    }
    float l_run = 0.0f;
    int seen = 0; // blocks of the split up to this wave's last
    for (int j = 0; j < my_tiles; j++) {
        // the running maximum at this block
        float m_new = m_run;
        for (; seen <= wave + kI8DecWaves * j; seen++) {
            m_new = fmaxf(m_new, sm_bm[seen * TC + c]);
        }
        if (wave_any(m_new > m_run)) {
            const float alpha = m_new > m_run ? fast_exp2(m_run - m_new) : 1.0f; // m_run = -inf -> 0
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < C::NDT; dt++) {
                oacc[dt] *= alpha;
            }
        }
        const float c0 = int8_exp_offset(m_run);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // t(j), V(j) and its scales landed
        const float* const tl = reinterpret_cast<const float*>(wsm + C::TILE_BYTES) + (g * TC + c) * 4;
        h8 pb[4];
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f}; // four independent chains
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const f4 t = *reinterpret_cast<const f4*>(tl + 2 * i * TC * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                // y = 127 p; its integer as fp16 exactly
                const float y = fast_exp2(fmaf(t[e], qeff, c0));
                ps[e] += y;
                pb[i >> 1][4 * (i & 1) + e] = (_Float16)rintf(y);
            }
        }
        l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);
        // O^T += V^T P^T: slot k of the lane's operand is key 16 u + 4 g + k % 4
        // + 8 (k / 4), as in pb[u]
        {
            const int j16 = lane & 15;
            const int k = j16 >> 1; // the row this lane addresses
            const float* vsl = reinterpret_cast<const float*>(wsm + C::TILE_BYTES + T_BYTES) + 4 * g;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = 16 * u + 4 * g + (k & 3) + 8 * (k >> 2);
                const uint32_t row = lds_v + r * C::RB + 8 * (j16 & 1);
                f4 vlo = {}, vhi = {};
                if constexpr (VTOK) {
                    vlo = *reinterpret_cast<const f4*>(vsl + 16 * u);
                    vhi = *reinterpret_cast<const f4*>(vsl + 16 * u + 8);
                }
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
                    const int ch = 2 * dt + ((lane >> 4) & 1);
                    const i2 x = lds_read_tr8(row + ((ch ^ i8dec_swz<D>(r)) << 4));
                    const h8 v8 = VTOK ? widen8_scaled(x, vlo, vhi) : widen8(x);
                    oacc[dt] = mfma_32x32x16_f16(v8, pb[u], oacc[dt]);
                }
            }
        }
        if (j + 1 < my_tiles) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of the slot has returned
            issue(j + 1);
        }
    }
    __builtin_amdgcn_s_waitcnt(0); // all DMAs and LDS traffic of this wave done
    // O in units of pq v, l in units of 1/127
    const float* vch = p.vch != nullptr ? p.vch + ((int64_t)w.b * p.Hkv + w.kvh) * D : nullptr;
    finish_rows<D, kI8DecWaves>(oacc, m_run, l_run, dsm, pp.out, w.b, w.kvh, blockIdx.x, [&](f4 x, int d) {
        x *= p.v_scale;
        return vch != nullptr ? x * *reinterpret_cast<const f4*>(vch + d) : x;
    });
}

// Columns in the scratch (TC) of a call with up to 32 rows per kv head.
int scratch_columns(const AttnArgs& a) {
    return (int64_t)(a.Hq / a.Hkv) * a.Sq <= 4 ? 4 : 32;
}

// 64-key blocks from the first to the last key that some row sees.
int64_t visible_blocks(const AttnArgs& a) {
    const MaskSpec mask{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    int lo, hi;
    visible_key_range(mask, 0, a.Sq - 1, lo, hi);
    return hi < lo ? 0 : hi / kI8BN + 1 - lo / kI8BN;
}

// Scores and block maxima of a call.
int64_t score_bytes(const AttnArgs& a) {
    return (int64_t)a.B * a.Hkv * visible_blocks(a) * (kI8BN + 1) * scratch_columns(a) * (int64_t)sizeof(float);
}

template <int D, bool VTOK, int TC>
int int8_decode_splits(const AttnArgs& a, SplitKPlan& plan, std::string& err) {
    const int64_t resident =
        resident_workgroups(reinterpret_cast<const void*>(&fa_int8_decode_pv<D, VTOK, TC>), kI8DecThreads, err);
    if (resident <= 0) {
        return -1;
    }
    // rounds of `resident` workgroups, each 2 us and its keys at 40 KB/us, all
    // together 6.8 TB/s; 5 us for the merge
    const int64_t n_bkv = (int64_t)a.B * a.Hkv;
    plan = splitk_plan_for(
        a, kI8BN, kI8DecWaves * kI8BN, TCfg<TC>::MAX_TILES * kI8BN, SIZE_MAX, [&](int s, int64_t keys) {
            const int64_t wgs = n_bkv * s;
            const double rate = std::min(40e3, 6.8e6 / (double)std::min(wgs, resident));
            return (double)((wgs + resident - 1) / resident) * (2.0 + (double)(keys * 2 * D) / rate) +
                   (s > 1 ? 5.0 : 0.0);
        });
    return 0;
}

template <int D, bool VTOK, int TC>
int launch_int8_decode(const AttnArgs& a, const Int8Params& ip, hipStream_t stream, std::string& err) {
    SplitKPlan plan;
    if (int8_decode_splits<D, VTOK, TC>(a, plan, err) != 0) {
        return -1;
    }
    Int8DecodeParams p{};
    p.a = ip;
    p.keys_per_split = plan.keys_per_split;
    p.key0 = plan.key0;
    p.blocks = (int32_t)visible_blocks(a); // key0 begins the first of them
    const size_t blocks = (size_t)a.B * a.Hkv * p.blocks;
    StreamScratch ws(ScratchUse::SplitKPartials), scores(ScratchUse::Int8Scores);
    int rc = splitk_begin(a, plan.splits, ws, stream, p.out, err);
    if (rc == 0) {
        rc = scores.alloc((size_t)score_bytes(a), stream, err);
    }
    if (rc != 0) {
        return rc;
    }
    p.t = static_cast<float*>(scores.ptr);
    p.bmax = p.t + blocks * TCfg<TC>::BLOCK_FLOATS;
    const dim3 grid(plan.splits, a.B * a.Hkv);
    {
        KernelTimerGuard timer(stream);
        hipLaunchKernelGGL((fa_int8_decode_scores<D, TC>), grid, dim3(kI8DecThreads), 0, stream, p);
        hipLaunchKernelGGL((fa_int8_decode_pv<D, VTOK, TC>), grid, dim3(kI8DecThreads), 0, stream, p);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = hipGetErrorString(e);
        return -1;
    }
    return splitk_finish(a, p.out, stream, err);
}

template <int D, bool VTOK>
int launch_int8_decode_as(const AttnArgs& a, const Int8Params& p, hipStream_t stream, std::string& err) {
    return scratch_columns(a) == 4 ? launch_int8_decode<D, VTOK, 4>(a, p, stream, err)
                                   : launch_int8_decode<D, VTOK, 32>(a, p, stream, err);
}

template <int D>
int decode_splits_as(const AttnArgs& a, SplitKPlan& plan, std::string& err) {
    return scratch_columns(a) == 4 ? int8_decode_splits<D, false, 4>(a, plan, err)
                                   : int8_decode_splits<D, false, 32>(a, plan, err);
}

} // namespace

bool int8_splitk_supported(const AttnArgs& a) {
    // one block of MFMA columns, few enough keys for kMaxSplits splits, at most 1
    // GiB of scores and block maxima, a grid (y = kv heads) within HIP's limit
    const int64_t M = (int64_t)(a.Hq / a.Hkv) * a.Sq;
    const int64_t max_blocks =
        (int64_t)kMaxSplits * (scratch_columns(a) == 4 ? TCfg<4>::MAX_TILES : TCfg<32>::MAX_TILES);
    return M <= 32 && (int64_t)a.B * a.Hkv <= kMaxGridY && visible_blocks(a) <= max_blocks &&
           score_bytes(a) <= (int64_t)1 << 30;
}

// The decode kernels or, where they are supported too, the prefill kernels (whose
// workgroup holds all rows of up to four query heads of a kv head, and of up to
// 512 workgroups may alternate).  Time prefill / decode, each over caches that
// together exceed the last-level cache, by prefill workgroups:
//   * up to 256 the two launches and the merge cost about 5 us (a cache of 64 keys
//     9.2 / 12.9 us): even at about 576 keys at D = 64 (8 kv heads of 512 keys
//     0.95 to 1.03, of 640 1.03 to 1.16), 448 at D = 128 (1.07 to 1.15)
//   * beyond, prefill runs in rounds: up to 512 from 192 keys (512 kv heads with
//     one row 1.15, of 128 keys 0.9 to 0.98), from 128 at D = 128 (384 heads 0.99 to
//     1.04) or with several workgroups per kv head (1.0 to 1.25); above from 128
//     (768 heads 1.09 to 1.14), and always with several workgroups per kv head
//     (320 heads of eight rows, 1 key 1.08) or from 1024 workgroups on (4096 heads
//     of one key 1.2)
//   * rows of one workgroup that take the 32-column scratch, whose scores are
//     more bytes than K: prefill that fills its rounds is quicker (256 kv heads
//     with 8 to 32 rows, 512 to 8192 keys 0.82 to 1.03, 512 of them 0.84 to 0.98;
//     but 128 1.0 to 1.8, and 320 and 384 from 256 keys 1.07 to 1.17 at D = 64), and
//     more often so with 32 rows of one head, in one wave, at D = 128 (192 heads
//     0.94 to 0.97, of 8192 keys 1.12, 384 0.92 to 1.0); and where its one round leaves CUs idle but
//     the scores leave the last-level cache (192 heads of 16384 keys, 408 MB: 0.8;
//     128 heads, 272 MB: 1.5).  Above 512 workgroups they do not alternate
//     (1024 heads with 16 rows, 192 keys 1.07 at D = 64; at D = 128 4096 of 320 1.05,
//     768, whole rounds, of 384 to 576 0.93 to 0.96; with 32 rows of one head 1.06
//     from 256 and 1.1 from 1024)
bool int8_prefer_splitk(const AttnArgs& a) {
    if (!int8_splitk_supported(a)) {
        return false;
    }
    const int ratio = a.Hq / a.Hkv;
    const int groups = ratio % 4 == 0 ? ratio / 4 : ratio % 2 == 0 ? ratio / 2 : ratio; // per kv head
    const bool one_wave = ratio == groups;
    const int64_t n_wg = (int64_t)a.B * a.Hkv * groups;
    const int64_t keys = visible_blocks(a) * kI8BN;
    const bool d64 = a.D == 64;
    const int64_t even = d64 ? 576 : 448;
    if (groups > 1 || scratch_columns(a) == 4) {
        if (n_wg > 512) {
            return n_wg >= 1024 || groups > 1 || keys >= 128;
        }
        return keys >= (n_wg <= 256 ? even : groups > 1 || !d64 ? 128 : 192);
    }
    const int64_t rounds = (n_wg + 255) / 256;
    const bool filled = 10 * n_wg > (one_wave && !d64 && keys < 4096 ? 7 : 9) * 256 * rounds;
    if (n_wg > 512) {
        const int64_t d128 = one_wave ? 1024 : n_wg >= 2048 ? 256 : filled && n_wg < 1024 ? 768 : 384;
        return keys >= (d64 ? (one_wave ? 256 : 192) : d128);
    }
    if (filled) {
        return false;
    }
    return rounds > 1 ? keys >= (d64 ? 256 : 320) : keys >= even && score_bytes(a) <= (int64_t)320 << 20;
}

int int8_decode_plan(const AttnArgs& a, CallPlan& plan, std::string& err) {
    plan = CallPlan{CallForm::kDecode, 0, (size_t)score_bytes(a)};
    SplitKPlan splits;
    if ((a.D == 64 ? decode_splits_as<64>(a, splits, err) : decode_splits_as<128>(a, splits, err)) != 0) {
        return -1;
    }
    plan.splits = splits.splits;
    plan.scratch += splitk_partial_bytes(a, splits.splits);
    return 0;
}

int fwd_int8_splitk(const AttnArgs& a, const Int8Params& p, hipStream_t stream, std::string& err) {
    const bool vtok = p.vtok != nullptr;
    if (a.D == 64) {
        return vtok ? launch_int8_decode_as<64, true>(a, p, stream, err)
                    : launch_int8_decode_as<64, false>(a, p, stream, err);
    }
    return vtok ? launch_int8_decode_as<128, true>(a, p, stream, err)
                : launch_int8_decode_as<128, false>(a, p, stream, err);
}

#endif

} // namespace rdna_amd
