// FP16 split-K ("flash-decoding") forward for gfx950: few query rows per kv
// head against a long key sequence.  No counterpart in the reference, whose
// decode rows run one workgroup per (batch, head) over the whole cache
// (docs/api.md:203-204); same results, same masking rules.
//
// The shape is HBM-bound (each K/V byte is used by only ratio * Sq query
// rows), so the design goal is bytes in flight, not MFMA rate:
//
//   * grid = (splits, B * Hkv); a workgroup owns one contiguous key range of
//     one kv head and all M = (Hq/Hkv) * Sq query rows of that head group,
//     packed as the 32 columns of one MFMA block (M <= 32)
//   * its waves (eight up to D = 160) work independently on interleaved
//     32-key tiles: each streams K and V with buffer_load ... lds (HBM -> LDS,
//     no VGPR staging), non-temporal since every byte is read once, into its
//     own K and V slots; K(j + 1) leaves as soon as S(j) has read K(j), V(j +
//     1) after P V(j), so one of the two is always in flight; no workgroup
//     barriers in the loop
//     (B = 8 Hq = 16 Hkv = 8 Sk = 6001 D = 256, 393 MB: 65 us, 6.1 TB/s; the
//     prefill kernel, one row of 128 in use, 183 us; two waves with two slots
//     each of K and V, 111 us: a wave spends ~80 cycles issuing each 1 KB DMA,
//     so more waves, not deeper slots, keep the bytes coming)
//   * LDS rows are stored with an XOR swizzle of their 16-byte chunks so the
//     ds_read_b128 of K (16 rows) and the ds_read_b64_tr_b16 of V (4 rows x
//     32 B) both hit distinct banks although the DMA writes rows unpadded
//   * the waves' (max, sum, O) are merged in LDS; one partial per workgroup
//     goes to a stream-ordered scratch buffer; a combine kernel merges the
//     splits (the same log-sum-exp merge a cross-GPU sequence split would use)
#include "fa_common.hpp"
#include "fa_host.hpp"
#include "fa_internal.hpp"
#include "fa_splitk.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace rdna_amd {

float softmax_log2_scale(float scale);

namespace {

constexpr int kDecTile = 32; // keys per wave tile
constexpr float kDecRescaleThreshold = 8.0f;

struct DecodeParams {
    const _Float16* q;
    const _Float16* k;
    const _Float16* v;
    const float* rot_cos;
    const float* rot_sin;
    int64_t q_sb, q_sh, q_ss;
    int64_t k_sb, k_sh, k_ss;
    int64_t v_sb, v_sh, v_ss;
    SplitRows out;
    int32_t Hkv, keys_per_split;
    int32_t key0; // first key of split 0
    float c;
    float q_sign;
    MaskSpec mask;
    int32_t rope_q;
    int32_t pair_heads; // pairs of kv heads to one XCD (D % 64 == 32)
};

template <int D>
struct DecCfg {
    // LDS holds one K and one V tile per wave, 128 D bytes: eight waves up to
    // D = 160 (160 KB there), six at 192 (144 KB), four above (128 KB at 256;
    // one wave per SIMD, whose O alone takes 128 registers)
    static constexpr int WAVES = D <= 160 ? 8 : (D <= 192 ? 6 : 4);
    static constexpr int THREADS = 64 * WAVES;
    // waves per SIMD: two workgroups share a CU's LDS at D = 64, four at 32
    static constexpr int WAVES_PER_SIMD = D <= 32 ? 7 : (D <= 64 ? 4 : 1);
    static constexpr int RB = 2 * D;                 // row bytes (unpadded)
    static constexpr int KCH = D / 8;                // 16-byte chunks per row
    static constexpr int TILE_BYTES = kDecTile * RB; // one K (or V) tile
    static constexpr int WAVE_BYTES = 2 * TILE_BYTES;
    static constexpr int NS = D / 16;
    static constexpr int NDT = D / 32;
    static constexpr int DMA_PER_TILE = TILE_BYTES / 1024; // 1 KB per wave-wide DMA
    static_assert(WAVES * WAVE_BYTES <= 160 * 1024, "K/V tiles fit the LDS");
    static_assert(finish_lds_bytes(D, WAVES) <= WAVES * WAVE_BYTES, "the merge reuses the tile area");
};

// XOR swizzle of the 16-byte chunk index of row r (see the file comment).
// Rows are 2 D bytes and the 64 banks 256 B: rows r and r + 4 (D % 64 = 32),
// r + 2 (D % 128 = 64) or r + 1 (D % 128 = 0) start in the same bank, so that
// many chunk positions spread them: XOR within groups of 4, 8 or 16 chunks
// (each divides D / 8).
template <int D>
__device__ __forceinline__ int dec_swz(int r) {
    if constexpr (D % 64 == 32) {
        return (r >> 2) & 3;
    } else if constexpr (D % 128 == 64) {
        return (((r >> 1) & 3) << 1) | ((r >> 3) & 1);
    } else {
        return ((r & 7) << 1) | ((r >> 3) & 1);
    }
}

template <int D>
__global__ __launch_bounds__(DecCfg<D>::THREADS, DecCfg<D>::WAVES_PER_SIMD) void fa_fwd_f16_decode(DecodeParams p) {
    using C = DecCfg<D>;
    __shared__ __attribute__((aligned(16))) char dsm[C::WAVES * C::WAVE_BYTES];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6); // wave-uniform
    const int lane = tid & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    int split = blockIdx.x;
    int bkv = blockIdx.y;
    if constexpr (D % 64 == 32) {
        // Rows of 64, 192, ... bytes: in a [B, S, 2, H, D] cache two heads share every
        // (or every third, ...) 128-byte line.  Pairs of heads go to one XCD, whose
        // L2 then fetches it once: workgroup `id` runs on XCD id % 8, and its slot
        // there is one head of pair slot / 2.
        if (p.pair_heads != 0) {
            const int id = bkv * (int)gridDim.x + split;
            const int pair = (id & 7) + 8 * (id >> 4);
            split = pair % (int)gridDim.x;
            bkv = 2 * (pair / (int)gridDim.x) + ((id >> 3) & 1);
        }
    }
    const int b = bkv / p.Hkv;
    const int kvh = bkv - b * p.Hkv;

    // column l32 <-> (query head, query row)
    const bool col_valid = l32 < p.out.ratio * p.out.Sq;
    const int hoff = col_valid ? l32 / p.out.Sq : 0;
    const int q = col_valid ? l32 - hoff * p.out.Sq : 0;
    const int h = kvh * p.out.ratio + hoff;

    // this split's key range, restricted to what any of the M rows can see
    const int k_begin = p.key0 + split * p.keys_per_split;
    const int k_end = min(k_begin + p.keys_per_split, p.mask.sk);
    int vis_lo, vis_hi;
    visible_key_range(p.mask, 0, p.out.Sq - 1, vis_lo, vis_hi);
    const int lo = max(k_begin, vis_lo);
    const int hi = min(k_end - 1, vis_hi);
    int t0 = 0, nt = 0; // tiles of this wave: kt = t0 + wave + WAVES * j
    if (hi >= lo) {
        t0 = lo / kDecTile;
        nt = hi / kDecTile + 1 - t0;
    }
    const int my_tiles = nt > wave ? (nt - wave + C::WAVES - 1) / C::WAVES : 0;

    const _Float16* kbase = p.k + b * p.k_sb + kvh * p.k_sh;
    const _Float16* vbase = p.v + b * p.v_sb + kvh * p.v_sh;
    char* wsm = dsm + wave * C::WAVE_BYTES;

    // DMA source offsets: lane i of DMA j writes LDS bytes 1024 j + 16 i of the
    // tile, i.e. stored chunk n % KCH of row r = n / KCH with n = 64 j + i,
    // which holds logical chunk (n % KCH) ^ swz(r)
    uint32_t kdo[C::DMA_PER_TILE], vdo[C::DMA_PER_TILE];
#pragma unroll
    for (int j = 0; j < C::DMA_PER_TILE; j++) {
        const int n = 64 * j + lane;
        const int r = n / C::KCH;
        const int cl = (n - r * C::KCH) ^ dec_swz<D>(r);
        kdo[j] = (uint32_t)(((int64_t)r * p.k_ss + 8 * cl) * 2);
        vdo[j] = (uint32_t)(((int64_t)r * p.v_ss + 8 * cl) * 2);
    }
    const uint32_t lds_k = (uint32_t)reinterpret_cast<uintptr_t>(wsm);
    const uint32_t lds_v = lds_k + C::TILE_BYTES;
    auto issue_k = [&](int j_tile) {
        const int kt0 = (t0 + wave + C::WAVES * j_tile) * kDecTile;
        const i32x4_t r = make_rsrc_v(kbase + (int64_t)kt0 * p.k_ss,
                                      tile_bytes<kDecTile>(p.mask.sk - kt0, (uint32_t)(p.k_ss * 2), D * 2));
#pragma unroll
        for (int j = 0; j < C::DMA_PER_TILE; j++) {
            dma_load16_nt(r, kdo[j], lds_k + 1024 * j);
        }
    };
    auto issue_v = [&](int j_tile) {
        const int kt0 = (t0 + wave + C::WAVES * j_tile) * kDecTile;
        const i32x4_t r = make_rsrc_v(vbase + (int64_t)kt0 * p.v_ss,
                                      tile_bytes<kDecTile>(p.mask.sk - kt0, (uint32_t)(p.v_ss * 2), D * 2));
#pragma unroll
        for (int j = 0; j < C::DMA_PER_TILE; j++) {
            dma_load16_nt(r, vdo[j], lds_v + 1024 * j);
        }
    };

    // The first tiles leave before the Q loads, so that a short key range
    // costs one memory round trip and not two; the wait for Q drains them too
    // (the compiler's vmcnt waits do not count the DMAs), once.
    if (my_tiles > 0) {
        issue_k(0);
        issue_v(0);
    }
    h8 qreg[C::NS];
    {
        const int qr = q; // 0 for an unused column
        const _Float16* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qr * p.q_ss;
        load_q_operand(qreg, qrow, p.rot_cos + (int64_t)qr * (D / 2), p.rot_sin + (int64_t)qr * (D / 2), g, col_valid,
                       p.rope_q != 0, p.q_sign < 0.0f);
    }
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
        // (the first two tiles were awaited with Q)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(C::DMA_PER_TILE));
        const int kt0 = (t0 + wave + C::WAVES * j) * kDecTile;
        const char* sk = wsm;
        const char* sv = wsm + C::TILE_BYTES;

        // S^T[key][col] = K Q^T over one 32-key tile
        f16x sacc = {};
        {
            const int r = l32;
            const char* krow = sk + r * C::RB;
            const int sw = dec_swz<D>(r);
#pragma unroll
            for (int s = 0; s < C::NS; s++) {
                const int cl = 2 * s + g;
                h8 a = *reinterpret_cast<const h8*>(krow + ((cl ^ sw) << 4));
                sacc = mfma_32x32x16_f16(a, qreg[s], sacc);
            }
        }
        const bool more = j + 1 < my_tiles;
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of K(j) has returned
            issue_k(j + 1);
        }
        // mask (only where a tile crosses a row's visible range; cheap anyway)
        {
            const int a = row_lo - kt0 - 4 * g;
            const int bnd = row_hi - kt0 - 4 * g;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int off = 8 * (e >> 2) + (e & 3);
                sacc[e] = (off < a || off > bnd) ? -INFINITY : sacc[e];
            }
        }
        float mx = max_tree<16>([&](int e) { return sacc[e]; });
        mx = pair_max(mx);
        const float m_new = fmaxf(m_run, mx * p.c);
        const bool grow = m_new > m_run + kDecRescaleThreshold;
        if (wave_any(grow)) {
            const float alpha = grow ? fast_exp2(m_run - m_new) : 1.0f;
            if (grow) {
                m_run = m_new;
            }
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < C::NDT; dt++) {
                oacc[dt] *= alpha;
            }
        }
        const float m_use = (m_run == -INFINITY) ? 0.0f : m_run;
        h8 pb[2];
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f}; // four independent chains
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float pv = fast_exp2(fmaf(sacc[e], p.c, -m_use));
            ps[e & 3] += pv;
            pb[e >> 3][e & 7] = (_Float16)pv;
        }
        l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);

        // V(j) landed: only K(j + 1)'s DMAs are younger
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(C::DMA_PER_TILE));
        } else {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        }
        // O^T += V^T P^T; V^T operand through transpose reads
        {
            const int j16 = lane & 15;
#pragma unroll
            for (int u = 0; u < 2; u++) {
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
                    h4 half4[2];
#pragma unroll
                    for (int hh = 0; hh < 2; hh++) {
                        const int r = 16 * u + 8 * hh + 4 * g + (j16 >> 2);
                        const int d = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (j16 & 3);
                        const int cl = d >> 3;
                        const char* addr = sv + r * C::RB + ((cl ^ dec_swz<D>(r)) << 4) + ((d & 7) << 1);
                        half4[hh] = lds_read_tr16(reinterpret_cast<const _Float16*>(addr));
                    }
                    h8 a = __builtin_shufflevector(half4[0], half4[1], 0, 1, 2, 3, 4, 5, 6, 7);
                    oacc[dt] = mfma_32x32x16_f16(a, pb[u], oacc[dt]);
                }
            }
        }
        if (more) {
            __builtin_amdgcn_s_waitcnt(waitcnt_lgkm(0)); // every read of V(j) has returned
            issue_v(j + 1);
        }
    }
    __builtin_amdgcn_s_waitcnt(0); // all DMAs and LDS traffic of this wave done
    finish_rows<D, C::WAVES>(oacc, m_run, l_run, dsm, p.out, b, kvh, split, [](f4 x, int) { return x; });
}

// One workgroup per output row: log-sum-exp merge of the
// splits, normalised in fp32, rounded once to fp16.  Merging inside the split
// kernel instead, by the last workgroup of each group to arrive, measured
// slower although it saves this launch (B = 4 Hq = 32 Hkv = 8 Sk = 4096 D =
// 128: 31.6 against 19.2 us a call; B = 16 Sk = 32768: 330 against 317): the
// device-scope release and acquire it needs write back and invalidate whole
// L2s.
template <int T>
__global__ __launch_bounds__(T) void fa_decode_combine(SplitRows r, int32_t D) {
    __shared__ __attribute__((aligned(16))) float lds[merge_lds_floats(kMaxSplits, T)];
    const int row = blockIdx.x; // (b * Hq + h) * Sq + q
    const int bh = row / r.Sq;
    const int b = bh / r.Hq;
    _Float16* orow = r.row(b, bh - b * r.Hq, row - bh * r.Sq);
    const SplitParts parts{r.part_o + (int64_t)row * D, r.part_ml + (int64_t)row * 2, r.n_rows * D, 2 * r.n_rows,
                           r.splits, D};
    merge_splits<T>(parts, lds, [&](int d, f4 x) {
        *reinterpret_cast<h4*>(orow + d) = __builtin_convertvector(x, h4);
    });
}

template <int D>
int launch_decode(const DecodeParams& p, int n_bkv, hipStream_t stream, std::string& err) {
    KernelTimerGuard timer(stream);
    hipLaunchKernelGGL(fa_fwd_f16_decode<D>, dim3(p.out.splits, n_bkv), dim3(DecCfg<D>::THREADS), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = hipGetErrorString(e);
        return -1;
    }
    return 0;
}

// f(std::integral_constant<int, D>) for the head dims the kernel is built for
template <class F>
auto for_dim(int d, F&& f) -> decltype(f(std::integral_constant<int, 32>{})) {
    switch (d) {
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 96: return f(std::integral_constant<int, 96>{});
    case 128: return f(std::integral_constant<int, 128>{});
    case 160: return f(std::integral_constant<int, 160>{});
    case 192: return f(std::integral_constant<int, 192>{});
    case 224: return f(std::integral_constant<int, 224>{});
    default: return f(std::integral_constant<int, 256>{});
    }
}

} // namespace

bool splitk_supported(const AttnArgs& a) {
    const int M = (a.Hq / a.Hkv) * a.Sq;
    return (a.D == 32 || a.D == 64 || a.D == 128) && M <= 32;
}

bool splitk_built(const AttnArgs& a) {
    return a.D <= 256 && (int64_t)(a.Hq / a.Hkv) * a.Sq <= 32 && (int64_t)a.B * a.Hkv <= kMaxGridY;
}

size_t splitk_partial_bytes(const AttnArgs& a, int splits) {
    return splits <= 1 ? 0 : (size_t)a.B * a.Hq * a.Sq * splits * (a.D + 2) * sizeof(float);
}

SplitKPlan splitk_plan_for(const AttnArgs& a, int tile, int round, int64_t max_keys, size_t max_partials,
                           const std::function<double(int, int64_t)>& time_us) {
    // The keys that some row sees, from a tile boundary on, are dealt to the
    // splits in multiples of `round` keys.
    const MaskSpec mask{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    int lo, hi;
    visible_key_range(mask, 0, a.Sq - 1, lo, hi);
    SplitKPlan plan;
    if (hi < lo) {
        plan.keys_per_split = tile;
        return plan; // one split, which writes zeros
    }
    plan.key0 = lo / tile * tile;
    const int keys = hi + 1 - plan.key0;
    const int units = (keys + round - 1) / round;
    double best = INFINITY;
    // over 1 .. kMaxSplits, the smallest count of each size (another one has an
    // empty split)
    for (int s = 1; s <= std::min(units, kMaxSplits);) {
        const int per = (units + s - 1) / s;
        const int64_t kps = (int64_t)per * round;
        if (kps <= max_keys && region_bytes(splitk_partial_bytes(a, s)) <= max_partials) {
            const double t = time_us(s, std::min<int64_t>(kps, keys));
            if (t < best) {
                best = t;
                plan.splits = s;
                plan.keys_per_split = (int)kps;
            }
        }
        if (per == 1) {
            break;
        }
        s = (units + per - 2) / (per - 1);
    }
    return plan;
}

int splitk_plan(const AttnArgs& a, size_t max_partials, SplitKPlan& plan, std::string& err) {
    return for_dim(a.D, [&](auto d) {
        using C = DecCfg<decltype(d)::value>;
        int cus = 0;
        const int64_t resident = resident_workgroups(
            reinterpret_cast<const void*>(&fa_fwd_f16_decode<decltype(d)::value>), C::THREADS, err, &cus);
        if (resident <= 0) {
            return -1;
        }
        // A launch runs in rounds of `resident` workgroups, the last with what is
        // left.  A round takes 3 us and its bytes: those of the CU with the most
        // workgroups at 34 KB/us (24 at D = 32, 30 at 64, 36 above 192), and of all at 6.8
        // TB/s.  So 192 workgroups (64 heads of 8198 keys, D = 128, 3 splits: 54.3 us)
        // are no match for 256 (4: 50.8), and at D = 64, where two share a CU, 160
        // heads of 7166 keys take 66 us with one split, 77 with two, 55 with three
        // and 65 with four.  The merge, a second launch, adds about 9 us, 15 ns per
        // split and the partials, written and read, at 2.5 MB/us.  Fitted to 520
        // calls (8 to 512 kv heads, 512 to 16384 keys, one and four rows, caches
        // beyond the last-level cache) over all splits: 1.1 % above the best of them
        // on average with a head's rows in one block (36 KB/us would fit best), 2.6
        // % with the rows apart, as in a [B, S, 2, H, D] cache (26 to 31); the bits do
        // not depend on the strides.  A rate of 40 KB/us per workgroup and no CUs: 2.3
        // and 4.8 %.  Splits of single tiles: rounds of the waves leave the last one
        // short.
        const double cu_rate = a.D <= 32 ? 24e3 : a.D <= 64 ? 30e3 : a.D <= 192 ? 34e3 : 36e3;
        const int64_t n_bkv = (int64_t)a.B * a.Hkv;
        plan = splitk_plan_for(a, kDecTile, kDecTile, INT32_MAX, max_partials, [&](int s, int64_t keys) {
            const double bytes = (double)(keys * 2 * C::RB);
            auto round_us = [&](int64_t n) {
                return 3.0 + std::max((double)((n + cus - 1) / cus) * bytes / cu_rate, (double)n * bytes / 6.8e6);
            };
            const int64_t rounds = n_bkv * s / resident, rest = n_bkv * s % resident;
            return (double)rounds * round_us(resident) + (rest > 0 ? round_us(rest) : 0.0) +
                   (s > 1 ? 9.0 + 0.015 * s + 2.0 * (double)splitk_partial_bytes(a, s) / 2.5e6 : 0.0);
        });
        return 0;
    });
}

int splitk_begin(const AttnArgs& a, int splits, StreamScratch& ws, hipStream_t stream, SplitRows& r,
                 std::string& err) {
    r.o = static_cast<_Float16*>(a.o);
    r.o_sb = a.os[0];
    r.o_sh = a.os[1];
    r.o_ss = a.os[2];
    r.n_rows = (int64_t)a.B * a.Hq * a.Sq;
    r.Sq = a.Sq;
    r.Hq = a.Hq;
    r.ratio = a.Hq / a.Hkv;
    r.splits = splits;
    // every partial is written by its split's workgroup before the combine
    // reads it, so the buffer needs no clearing
    if (const int rc = ws.alloc(splitk_partial_bytes(a, splits), stream, err)) {
        return rc;
    }
    r.part_o = static_cast<float*>(ws.ptr);
    r.part_ml = splits > 1 ? r.part_o + (size_t)splits * r.n_rows * a.D : nullptr;
    return 0;
}

int splitk_finish(const AttnArgs& a, const SplitRows& r, hipStream_t stream, std::string& err) {
    if (r.splits == 1) {
        return 0;
    }
    // four waves per row where few rows have many splits
    const dim3 grid((uint32_t)r.n_rows);
    if (r.splits >= 8 && r.n_rows < 2048) {
        hipLaunchKernelGGL(fa_decode_combine<256>, grid, dim3(256), 0, stream, r, a.D);
    } else {
        hipLaunchKernelGGL(fa_decode_combine<64>, grid, dim3(64), 0, stream, r, a.D);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = hipGetErrorString(e);
        return -1;
    }
    return 0;
}

int fwd_f16_splitk(const AttnArgs& a, bool rope_q, hipStream_t stream, std::string& err, ScratchRegion* region) {
    DecodeParams p{};
    p.q = static_cast<const _Float16*>(a.q);
    p.k = static_cast<const _Float16*>(a.k);
    p.v = static_cast<const _Float16*>(a.v);
    p.rot_cos = a.rot_cos;
    p.rot_sin = a.rot_sin;
    p.q_sb = a.qs[0];
    p.q_sh = a.qs[1];
    p.q_ss = a.qs[2];
    p.k_sb = a.ks[0];
    p.k_sh = a.ks[1];
    p.k_ss = a.ks[2];
    p.v_sb = a.vs[0];
    p.v_sh = a.vs[1];
    p.v_ss = a.vs[2];
    p.Hkv = a.Hkv;
    p.c = softmax_log2_scale(a.scale);
    p.q_sign = a.scale < 0.0f ? -1.0f : 1.0f;
    p.mask = MaskSpec{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    p.rope_q = rope_q ? 1 : 0;

    SplitKPlan plan;
    const size_t room = region != nullptr ? region->bytes - region->used : SIZE_MAX;
    if (splitk_plan(a, room, plan, err) != 0) {
        return -1;
    }
    StreamScratch ws(ScratchUse::SplitKPartials, region);
    int rc = splitk_begin(a, plan.splits, ws, stream, p.out, err);
    if (rc == kScratchFull && splitk_plan(a, 0, plan, err) == 0) { // one split
        rc = splitk_begin(a, plan.splits, ws, stream, p.out, err);
    }
    p.keys_per_split = plan.keys_per_split;
    p.key0 = plan.key0;
    // rows of neighbouring heads next to each other, an even number of heads, whole
    // rounds of pairs over the 8 XCDs.  us a call without / with, one row per head:
    // D = 32, 128 heads of 9027 keys 54.7 / 37.9, 64 of 13925 45.5 / 31.3; D = 96, 512
    // of 4122 172 / 161; D = 160, 128 of 3000 51.8 / 47.9
    p.pair_heads = (a.ks[1] == a.D || a.vs[1] == a.D) && a.Hkv % 2 == 0 &&
                   (int64_t)a.B * a.Hkv * plan.splits % 16 == 0;
    if (rc != 0 ||
        for_dim(a.D, [&](auto d) { return launch_decode<decltype(d)::value>(p, a.B * a.Hkv, stream, err); }) != 0) {
        return -1;
    }
    return splitk_finish(a, p.out, stream, err);
}

} // namespace rdna_amd
