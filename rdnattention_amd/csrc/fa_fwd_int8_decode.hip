// INT8 split-K decode for gfx950: few query rows per kv head.  The prefill
// kernels put 256 query rows in a workgroup, so one decode row per head left
// 255 of them and most CUs idle.
//
// The scheme is the prefill kernels' (fa_fwd_int8_f16pv.hip): exact int32 S,
// the running max per 64-key block, P quantised to integers 0..127 against it,
// l from the unquantised p, P V on fp16 MFMA (both factors are exact fp16
// integers).  Each wave keeps its own running max over the blocks it takes, so
// a block's step of 1/127 refers to the largest score of that wave's keys so
// far: at most the sequential scheme's, i.e. P is quantised at least as finely.
//
// What bounds it is the cache's bytes.  The structure is the FP16 split-K
// kernel's (fa_fwd_decode.hip): grid (splits, B * Hkv), the M = ratio * Sq <=
// 32 rows of a kv head as the 32 columns of the MFMAs, eight waves on
// interleaved 64-key tiles with one K and one V slot each, filled by
// non-temporal HBM -> LDS DMA: K(j + 1) (with its scales) leaves when S(j) has
// read K(j), V(j + 1) after P V(j).  V stays int8 in LDS; its operands come
// from ds_read_b64_tr_b8 transpose reads and are widened to fp16 in registers.
//
// B = 8 Hq = 32 Hkv = 8 Sk = 8192 D = 128 (136 MB): 27.4 us (5.0 TB/s) and 4.2
// us for the merge; the prefill kernel 201 us.
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
};

template <int D>
struct I8DecCfg {
    static constexpr int RB = D;                  // row bytes (unpadded)
    static constexpr int KCH = D / 16;            // 16-byte chunks per row
    static constexpr int TILE_BYTES = kI8BN * RB; // one K (or V) tile
    static constexpr int DMA_PER_TILE = TILE_BYTES / 1024;
    static constexpr int SCALE_BYTES = 4 * kI8BN; // one scale per key
    static constexpr int WAVE_BYTES = 2 * TILE_BYTES + 3 * SCALE_BYTES; // K, V, K scales (two slots), V scales
    static constexpr int NS = D / 32;  // int8 Q K^T steps
    static constexpr int NDT = D / 32; // O^T row tiles
    static_assert(kI8DecWaves * WAVE_BYTES <= 160 * 1024, "tiles fit the LDS");
    static_assert(finish_lds_bytes(D, kI8DecWaves) <= kI8DecWaves * WAVE_BYTES, "the merge reuses the tile area");
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

// ds_read_b64_tr_b8: within each 16-lane group, lane i receives as byte k
// byte i % 8 of the 8-byte word that lane 2k + i / 8 addresses; with lane j at
// row j / 2, columns 8 (j % 2) .. +7 of an 8 x 16 block, lane i gets column i.
typedef int i2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ i2 lds_read_tr8(uint32_t lds_byte_addr) {
    typedef int i2_raw __attribute__((__vector_size__(2 * sizeof(int))));
    typedef __attribute__((address_space(3))) i2_raw lds_i2;
    i2_raw r = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
        (lds_i2*)reinterpret_cast<const __attribute__((address_space(3))) char*>(lds_byte_addr));
    return __builtin_bit_cast(i2, r);
}

// 8 signed bytes -> fp16 (exact): flipping the sign bit gives u = v + 128, a
// byte permute against 0x64 makes the fp16 number 1024 + u, minus 1152 is v
__device__ __forceinline__ h8 widen8(i2 w) {
    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    h2 r[4];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const uint32_t u = (uint32_t)w[c] ^ 0x80808080u;
        r[2 * c] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - off;
        r[2 * c + 1] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - off;
    }
    return h8{r[0][0], r[0][1], r[1][0], r[1][1], r[2][0], r[2][1], r[3][0], r[3][1]};
}

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

// four waves per SIMD at D = 64: two workgroups share a CU's LDS (with per-token
// V scales the 128 registers would not do without spills)
template <int D, bool VTOK>
__global__ __launch_bounds__(kI8DecThreads, D == 64 && !VTOK ? 4 : 2) void fa_fwd_int8_decode(Int8DecodeParams pp) {
    using C = I8DecCfg<D>;
    const Int8Params& p = pp.a;
    __shared__ __attribute__((aligned(16))) char dsm[kI8DecWaves * C::WAVE_BYTES];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // wave-uniform
    const int lane = tid & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int split = blockIdx.x;
    const int bkv = blockIdx.y;
    const int b = bkv / p.Hkv;
    const int kvh = bkv - b * p.Hkv;

    // column l32 <-> (query head, query row)
    const bool col_valid = l32 < p.ratio * p.Sq;
    const int hoff = col_valid ? l32 / p.Sq : 0;
    const int q = col_valid ? l32 - hoff * p.Sq : 0;
    const int h = kvh * p.ratio + hoff;

    // this split's 64-key tiles, restricted to what any of the M rows can see
    const int k_begin = pp.key0 + split * pp.keys_per_split;
    const int k_end = min(k_begin + pp.keys_per_split, p.mask.sk);
    int vis_lo, vis_hi;
    visible_key_range(p.mask, 0, p.Sq - 1, vis_lo, vis_hi);
    const int lo = max(k_begin, vis_lo);
    const int hi = min(k_end - 1, vis_hi);
    int t0 = 0, nt = 0; // tiles of this wave: kt = t0 + wave + kI8DecWaves * j
    if (hi >= lo) {
        t0 = lo / kI8BN;
        nt = hi / kI8BN + 1 - t0;
    }
    const int my_tiles = nt > wave ? (nt - wave + kI8DecWaves - 1) / kI8DecWaves : 0;

    const int8_t* kbase = p.k + b * p.k_sb + kvh * p.k_sh;
    const int8_t* vbase = p.v + b * p.v_sb + kvh * p.v_sh;
    const int64_t tok = ((int64_t)b * p.Hkv + kvh) * p.mask.sk; // per-token scale rows
    const char* wsm = dsm + wave * C::WAVE_BYTES;
    const uint32_t lds_k = (uint32_t)reinterpret_cast<uintptr_t>(wsm);
    const uint32_t lds_v = lds_k + C::TILE_BYTES;
    const uint32_t lds_ks = lds_v + C::TILE_BYTES;
    const uint32_t lds_vs = lds_ks + 2 * C::SCALE_BYTES;

    // DMA source offsets: lane i of DMA j writes LDS bytes 1024 j + 16 i of the
    // tile, i.e. stored chunk n % KCH of row r = n / KCH with n = 64 j + i,
    // which holds logical chunk (n % KCH) ^ swz(r)
    uint32_t kdo[C::DMA_PER_TILE], vdo[C::DMA_PER_TILE];
#pragma unroll
    for (int j = 0; j < C::DMA_PER_TILE; j++) {
        const int n = 64 * j + lane;
        const int r = n / C::KCH;
        const int cl = (n - r * C::KCH) ^ i8dec_swz<D>(r);
        kdo[j] = (uint32_t)((int64_t)r * p.k_ss + 16 * cl);
        vdo[j] = (uint32_t)((int64_t)r * p.v_ss + 16 * cl);
    }
    // a tile's scales: a dword per lane, always issued (from an empty buffer
    // where there are none), so that the number in flight is fixed
    auto issue_scales = [&](const float* s, int kt0, uint32_t lds) {
        const int left = min(p.mask.sk - kt0, kI8BN);
        dma_load4(make_rsrc_v(s + kt0, s != nullptr && left > 0 ? 4u * (uint32_t)left : 0u), 4u * lane, lds);
    };
    const float* ksrow = p.ksv != nullptr ? p.ksv + tok : nullptr;
    auto issue_k = [&](int j_tile) {
        const int kt0 = (t0 + wave + kI8DecWaves * j_tile) * kI8BN;
        const i32x4_t r = make_rsrc_v(kbase + (int64_t)kt0 * p.k_ss,
                                      tile_bytes<kI8BN>(p.mask.sk - kt0, (uint32_t)p.k_ss, D));
#pragma unroll
        for (int j = 0; j < C::DMA_PER_TILE; j++) {
            dma_load16_nt(r, kdo[j], lds_k + 1024 * j);
        }
        issue_scales(ksrow, kt0, lds_ks + (j_tile & 1) * C::SCALE_BYTES);
    };
    auto issue_v = [&](int j_tile) {
        const int kt0 = (t0 + wave + kI8DecWaves * j_tile) * kI8BN;
        const i32x4_t r = make_rsrc_v(vbase + (int64_t)kt0 * p.v_ss,
                                      tile_bytes<kI8BN>(p.mask.sk - kt0, (uint32_t)p.v_ss, D));
#pragma unroll
        for (int j = 0; j < C::DMA_PER_TILE; j++) {
            dma_load16_nt(r, vdo[j], lds_v + 1024 * j);
        }
        if constexpr (VTOK) {
            issue_scales(p.vtok + tok, kt0, lds_vs);
        }
    };
    constexpr int K_DMAS = C::DMA_PER_TILE + 1;
    constexpr int V_DMAS = C::DMA_PER_TILE + (VTOK ? 1 : 0);

    // the first tiles leave before the Q loads: one memory round trip, not two
    if (my_tiles > 0) {
        issue_k(0);
        issue_v(0);
    }
    // Q^T operand: lane holds Q[q][32 s + 16 g .. +15]
    i4 qreg[C::NS];
    float qs = p.q_scale;
    {
        const int8_t* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)q * p.q_ss;
#pragma unroll
        for (int s = 0; s < C::NS; s++) {
            qreg[s] = col_valid ? *reinterpret_cast<const i4*>(qrow + 32 * s + 16 * g) : i4{};
        }
        if (p.qsv != nullptr && col_valid) {
            qs = p.qsv[((int64_t)b * p.Hq + h) * p.Sq + q];
        }
    }
    // the row max is taken over t = S ks when every lane's qc is positive;
    // otherwise t is scaled by qc first
    const float qc = qs * p.scale_log2e;
    const bool qpos = !wave_any(!(qc > 0.0f));
    const float qeff = qpos ? qc : 1.0f;
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    int row_lo, row_hi;
    row_key_bounds(p.mask, q, row_lo, row_hi);
    if (!col_valid) {
        row_lo = 1;
        row_hi = 0; // sees nothing
    }

    f16x oacc[C::NDT];
#pragma unroll
    for (int dt = 0; dt < C::NDT; dt++) {
        oacc[dt] = f16x{};
    }
    float m_run = -INFINITY, l_run = 0.0f;

    for (int j = 0; j < my_tiles; j++) {
        // K(j) landed: only V(j)'s DMAs, issued after it, may be outstanding
        // (the first tiles were awaited with Q)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(V_DMAS));
        const int kt0 = (t0 + wave + kI8DecWaves * j) * kI8BN;

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
        const bool more = j + 1 < my_tiles;
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of K(j) has returned
            issue_k(j + 1);
        }
        // t = S ks, masked; the scores are t qeff in log2 units
        float t[32];
        const int a = row_lo - kt0 - 4 * g;
        const int bnd = row_hi - kt0 - 4 * g;
        const float* ksl =
            reinterpret_cast<const float*>(wsm + 2 * C::TILE_BYTES + (j & 1) * C::SCALE_BYTES) + 4 * g;
#pragma unroll
        for (int i = 0; i < 8; i++) { // keys 8 i + 4 g .. +3
            f4 ks = *reinterpret_cast<const f4*>(ksl + 8 * i);
            if (p.ksv == nullptr) {
                ks = f4{p.k_scale, p.k_scale, p.k_scale, p.k_scale};
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                t[4 * i + e] = (float)sacc[i >> 2][4 * (i & 3) + e] * ks[e];
            }
        }
        if (!qpos) {
#pragma unroll
            for (int e = 0; e < 32; e++) {
                t[e] *= qc;
            }
        }
#pragma unroll
        for (int e = 0; e < 32; e++) {
            const int off = 32 * (e >> 4) + 8 * ((e >> 2) & 3) + (e & 3);
            t[e] = (off < a || off > bnd) ? -INFINITY : t[e];
        }
        const float mx = pair_max(max_tree<32>([&](int e) { return t[e]; })) * qeff; // qeff > 0: -inf stays -inf
        const float m_new = fmaxf(m_run, mx);
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
        h8 pb[4];
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f}; // four independent chains
#pragma unroll
        for (int e = 0; e < 32; e++) {
            // y = 127 p; its integer as fp16 exactly
            const float y = fast_exp2(fmaf(t[e], qeff, c0));
            ps[e & 3] += y;
            pb[e >> 3][e & 7] = (_Float16)rintf(y);
        }
        l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);

        // V(j) landed: only K(j + 1)'s DMAs are younger
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(K_DMAS));
        } else {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        }
        // O^T += V^T P^T: slot k of the lane's operand is key 16 u + 4 g + k % 4
        // + 8 (k / 4), as in pb[u]
        {
            const int j16 = lane & 15;
            const int k = j16 >> 1; // the row this lane addresses
            const float* vsl = reinterpret_cast<const float*>(wsm + 2 * C::TILE_BYTES + 2 * C::SCALE_BYTES) + 4 * g;
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
                    const int c = 2 * dt + ((lane >> 4) & 1);
                    const i2 w = lds_read_tr8(row + ((c ^ i8dec_swz<D>(r)) << 4));
                    const h8 v8 = VTOK ? widen8_scaled(w, vlo, vhi) : widen8(w);
                    oacc[dt] = mfma_32x32x16_f16(v8, pb[u], oacc[dt]);
                }
            }
        }
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of V(j) has returned
            issue_v(j + 1);
        }
    }
    __builtin_amdgcn_s_waitcnt(0); // all DMAs and LDS traffic of this wave done
    // O in units of pq v, l in units of 1/127
    const float* vch = p.vch != nullptr ? p.vch + ((int64_t)b * p.Hkv + kvh) * D : nullptr;
    finish_rows<D, kI8DecWaves>(oacc, m_run, l_run, dsm, pp.out, b, kvh, split, [&](f4 x, int d) {
        x *= p.v_scale;
        return vch != nullptr ? x * *reinterpret_cast<const f4*>(vch + d) : x;
    });
}

template <int D, bool VTOK>
int launch_int8_decode_as(const AttnArgs& a, const Int8Params& ip, hipStream_t stream, std::string& err) {
    const int64_t resident =
        resident_workgroups(reinterpret_cast<const void*>(&fa_fwd_int8_decode<D, VTOK>), kI8DecThreads, err);
    if (resident <= 0) {
        return -1;
    }
    const SplitKPlan plan = splitk_plan_for(a, kI8BN, kI8DecWaves * kI8BN, 2 * D, resident, SIZE_MAX);
    Int8DecodeParams p{};
    p.a = ip;
    p.keys_per_split = plan.keys_per_split;
    p.key0 = plan.key0;
    StreamScratch ws(ScratchUse::SplitKPartials);
    if (splitk_begin(a, plan.splits, ws, stream, p.out, err) != 0) {
        return -1;
    }
    {
        KernelTimerGuard timer(stream);
        hipLaunchKernelGGL((fa_fwd_int8_decode<D, VTOK>), dim3(plan.splits, a.B * a.Hkv), dim3(kI8DecThreads), 0,
                           stream, p);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            err = hipGetErrorString(e);
            return -1;
        }
    }
    return splitk_finish(a, p.out, stream, err);
}

} // namespace

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
