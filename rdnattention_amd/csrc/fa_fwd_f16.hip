// FP16 FlashAttention-2 forward for gfx950 (MI355X): the prefill kernel for
// head_dim <= 128 and the FP16 dispatcher (D 160..256: fa_fwd_f16_kpair.hip,
// D 288..512: fa_fwd_f16_dpair.hip, decode: fa_fwd_decode.hip).
//
// Replaces the reference's forwardKernel / forwardKernelGqa
// (src/rdna/fa2_forward_f16.hip:633-877) with a CDNA4 MFMA design:
//
//   * fa_fwd_f16_pp<D> (D <= 128): 8 waves in two groups that alternate an
//     MFMA phase and a softmax + staging phase (ping-pong, described above
//     the kernel); persistent grid from D = 64 up; Q staged through LDS with
//     row-contiguous loads; output stored through LDS as whole rows,
//     non-temporal
//   * every wave owns 32 query rows of one head and a workgroup holds G query
//     heads of one kv head (G | Hq/Hkv, G <= 4), so each K/V tile staged in
//     LDS serves all of them
//   * S^T = K Q^T on v_mfma_f32_32x32x16_f16: a lane owns one query column,
//     so the row max/sum are lane-local plus one exchange across half-waves
//   * P^T leaves the S^T accumulator in exactly the B-operand layout of the
//     O^T = V^T P^T MFMA, so P never touches LDS; V^T operands come from
//     row-major V tiles through ds_read_b64_tr_b16 transpose reads
//   * key tiles outside the causal/window band are skipped, tiles inside it
//     run a mask-free path, only boundary tiles evaluate the mask
//   * the running max is only raised when it grows by more than 2^8 (the
//     result is the same softmax; P stays <= 256, exact in fp16's range), so
//     the O accumulator is rarely rescaled
//   * RoPE: Q is rotated once when loaded, K once up front (fa_rope.hip)
//   * calls too small for the chip split their keys over workgroups
//     (prefill_splits) or let the two groups take the key tiles in turn
//     (prefill_alternate)
#include "fa_common.hpp"
#include "fa_host.hpp"
#include "fa_internal.hpp"
#include "fa_prefill.hpp"
#include "fa_splitk.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace rdna_amd {
namespace {

constexpr int kBN = 64;                 // keys per tile
constexpr float kRescaleThreshold = 8.0f; // log2 units

// ---------------------------------------------------------------------------
// Ping-pong prefill (D <= 128): 8 waves in two groups that alternate between
// an MFMA phase and a VALU phase, barrier to barrier, so every SIMD always has
// one wave feeding the matrix core while its partner runs the softmax:
//
//   group A:  M(0) V(0) M(1) V(1) ... M(n-1) V(n-1) M(n)  -
//   group B:  -    M(0) V(0) M(1) ...        M(n-1) V(n-1) M(n)
//
//   M(i): S(i) = K(i) Q^T and O += V(i-1)^T P(i-1)     (32 MFMAs at D=128)
//   V(i): online softmax of S(i) -> P(i), rescale of O, and staging of the
//         group's half of the next K/V tiles (registers -> LDS, HBM -> regs)
//
// K(i) and V(i-1) are read in global phases 2i and 2i+1 and live in LDS slot
// i % 2 and (i - 1) % 2.  Group A stages pair (K(i+1), V(i)) in its V(i)
// (phase 2i+1), group B stages pair (K(i+2), V(i+1)) in its V(i) (phase 2i+2);
// both write slots whose last readers finished before the preceding barrier.
// At D = 128 the tiles move by HBM -> LDS DMA instead (one 1 KB instruction
// per 4-row group): the loads' issue and the LDS stores left the softmax side,
// which is the longer one (0.4 % faster on causal GQA B4 Hq32 Hkv8 S4096 D128
// in same-box A/B runs, 16 fewer registers, 7.7 KB less LDS).  Group B issues
// K(i+2) at the start of its V(i) and awaits it at the end of its M(i+1), two
// phases of latency.  Group A issues V(i) at the start of its own V(i) and
// awaits it at the end of that phase: V(i-2)'s slot was last read in phase
// 2i-1, and V(i) is first read in phase 2i+2.  Each group's softmax side then
// carries four DMAs per wave per tile instead of zero and eight (-0.8 % on the
// causal GQA shape above, -1.1 % on causal GQA B2 Hq32 Hkv8 S8192 D128).
// ---------------------------------------------------------------------------
constexpr int kPPWaves = 8;
constexpr int kOpDepth = 4; // MFMA operands in flight in the MFMA phase
constexpr int kPPThreads = 64 * kPPWaves;

template <int D>
struct PPCfg {
    // LDS row strides (64 banks x 4 B): K rows are read 16 at a time with
    // ds_read_b128 -> a 16 B step mod 256 B keeps them in distinct banks; V rows
    // are read 4 at a time, 64 B each, by the transpose read -> a 64 B step
    static constexpr int LDK = D + 8;
    static constexpr int LDV = D + 32;
    // D = 128: K/V tiles staged by HBM -> LDS DMA, one instruction per 4-row
    // group (1 KB).  Row 4j + b of a tile sits at byte 256 b of group j, its
    // 16-byte chunk c at position c ^ 4b; groups lie PSK (PSV) halves apart,
    // 16 (64) bytes more than 1 KB.  The 16-row b128 K reads then hit 16
    // distinct 16-byte bank groups (group j at 16 j mod 256, row b's chunk
    // moved by 64 b), and the 8-row transpose reads of V fall twice on each
    // 64-byte quarter (group j at 64 j, row b's chunk quad moved by b).
    static constexpr bool DMA = D == 128;
    static constexpr int PSK = 520;
    static constexpr int PSV = 544;
    static constexpr int TILE_K = DMA ? (kBN / 4) * PSK : kBN * LDK;
    static constexpr int TILE_V = DMA ? (kBN / 4) * PSV : kBN * LDV;
    static constexpr int NS = D / 16;
    static constexpr int NDT = D / 32;
    static constexpr int KCH = D / 8;
    static constexpr int HALF_TASK = 32 * KCH;         // one group's chunks of one K (or V) tile
    static constexpr int CT = (HALF_TASK + 255) / 256; // K (and V) chunks per thread
    // Q of the row tile, RoPE applied: [wave][32 rows][LDQ], read like K rows
    static constexpr int LDQ = D + 8;
    static constexpr int TILE_Q = kPPWaves * 32 * LDQ;
    static constexpr int QCT = kPPWaves * 32 * KCH / kPPThreads; // Q chunks per thread (= NS)
    // One resident workgroup per CU from D = 64 up (VGPRs): a persistent grid
    // then saves the workgroup switches and balances the row tiles. At D = 32
    // two workgroups share a CU and hide each other's prologue instead, which
    // the persistent loop's extra registers would prevent.
    static constexpr bool PERSIST = D >= 64;
};

// PRE (used when c = |scale| log2(e) <= 1, which covers 1/sqrt(D) for every
// head dim): Q is staged pre-multiplied by q_sign * c, so the QK^T MFMAs
// produce scores in log2 units, and each S^T accumulator chain starts from
// -m (m the lane's running max, 0 while no key is visible) instead of 0, so
// the MFMA output is the exponent itself: p = 2^acc with no per-score
// multiply-add.  The accumulators are shifted only when the running max
// moves.  Without PRE, Q carries only the sign and p = 2^(acc c - m).
//
// MODE: kWhole as described; kSplit, every row tile's key tiles are dealt to
// p.splits workgroups, which write partials for the combine kernel; kAlternate,
// for launches whose few row tiles are long serial chains: both groups hold
// the same 128 rows and take the key tiles in turn, group A tiles 0, 2, 4, ...
// and group B tiles 1, 3, 5, ..., each staging its own tiles into one K and one
// V slot (pair (K(i+1), V(i)) of its sequence at the start of its V(i), when
// its M(i) has read their predecessors), and group B's O is merged into group
// A's through LDS at the end.  A row tile then takes half as many steps.
enum class PPMode { kWhole, kSplit, kAlternate };

template <int D, bool PRE, PPMode MODE>
__device__ __forceinline__ void pp_body(PrefillParams p) {
    using C = PPCfg<D>;
    constexpr bool SPLIT = MODE == PPMode::kSplit;
    constexpr bool ALT = MODE == PPMode::kAlternate;
    constexpr int ROW_WAVES = ALT ? kPPWaves / 2 : kPPWaves; // waves with rows of their own
    // K (and V) chunks that one group stages, and per thread of it
    constexpr int TASK = ALT ? 2 * C::HALF_TASK : C::HALF_TASK;
    constexpr int CT = (TASK + 255) / 256;
    constexpr int QCT = ROW_WAVES * 32 * C::KCH / kPPThreads; // Q chunks per thread
    // sK[slot], sV[slot], sQ
    __shared__ __attribute__((aligned(16))) _Float16 smem[2 * C::TILE_K + 2 * C::TILE_V + C::TILE_Q];
    _Float16* const sKs = smem;
    _Float16* const sVs = smem + 2 * C::TILE_K;
    _Float16* const sQ = smem + 2 * C::TILE_K + 2 * C::TILE_V;

    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int grp = wave >> 2;       // 0 = group A, 1 = group B
    const int gtid = tid & 255;      // thread index inside the group
    const int rw = ALT ? wave & 3 : wave; // wave by its rows
    const int ugrp = ALT ? __builtin_amdgcn_readfirstlane(grp) : 0;

    // ---- staging: this group's half (rows 32*grp .. +31) of K(x) and V(x-1)
    uint32_t coff_k[CT], coff_v[CT];
    int clk[CT], clv[CT]; // LDS element offsets inside a tile, -1 = no chunk
#pragma unroll
    for (int it = 0; it < CT; it++) {
        const int e = gtid + it * 256;
        const bool ok = TASK % 256 == 0 || e < TASK;
        const int row = (ALT ? 0 : 32 * grp) + (ok ? e / C::KCH : 0);
        const int ch = ok ? e - (e / C::KCH) * C::KCH : 0;
        coff_k[it] = (uint32_t)(((int64_t)row * p.k_ss + 8 * ch) * 2);
        coff_v[it] = (uint32_t)(((int64_t)row * p.v_ss + 8 * ch) * 2);
        clk[it] = ok ? row * C::LDK + 8 * ch : -1;
        clv[it] = ok ? row * C::LDV + 8 * ch : -1;
    }
    // DMA staging (PPCfg::DMA): wave w of group B (K) or A (V) moves 4-row
    // groups 4w .. 4w + 3 of each tile, lane i global chunk (i % 16) ^ 4 (i /
    // 16) of row 4j + i / 16 to LDS byte 16 i of group j; the group's row
    // offset is the instruction's scalar offset, its LDS address M0.
    const uint32_t dma_j0 = (uint32_t)__builtin_amdgcn_readfirstlane((wave & 3) * 4);
    const uint32_t dma_c = (uint32_t)((lane & 15) ^ (4 * (lane >> 4)));
    const uint32_t dma_vk = (uint32_t)(lane >> 4) * (uint32_t)(p.k_ss * 2) + 16u * dma_c;
    const uint32_t dma_vv = (uint32_t)(lane >> 4) * (uint32_t)(p.v_ss * 2) + 16u * dma_c;
    const uint32_t lds_k = (uint32_t)reinterpret_cast<uintptr_t>(sKs);
    const uint32_t lds_v = (uint32_t)reinterpret_cast<uintptr_t>(sVs);
    // Persistent (PPCfg::PERSIST): this workgroup walks its share of the row
    // tiles (one per workgroup of a one-tile-per-workgroup grid, see
    // persistent_item). Every group passes the same barriers per item and
    // leaves an item only after its last LDS read, so the next item's
    // prologue may overwrite LDS. Otherwise the grid has one workgroup per
    // row tile.
    auto run_tile = [&](const int wg) {
        int hg, rt, split = 0;
        wg_tile(wg, p.n_head_groups, SPLIT ? p.n_row_tiles * p.splits : p.n_row_tiles, p.hg_chunk, hg, rt);
        if constexpr (SPLIT) {
            split_row_tile(p.n_row_tiles, rt, split);
        }
        const int per_b = p.Hkv * p.groups_per_kv;
        const int b = hg / per_b;
        const int rem = hg - b * per_b;
        const int kvh = rem / p.groups_per_kv;
        const int sub = rem - kvh * p.groups_per_kv;
        const int h = kvh * p.ratio + sub * p.G + (rw % p.G);
        const int wg_q0 = rt * p.rows_per_wg;
        const int q0 = wg_q0 + (rw / p.G) * 32;
        const int q = q0 + l32;
        const bool wave_active = q0 < p.Sq;
        const int q_hi = min(q0 + 31, p.Sq - 1);

        const _Float16* qbase = p.q + b * p.q_sb + h * p.q_sh;
        const _Float16* kbase = p.k + b * p.k_sb + kvh * p.k_sh;
        const _Float16* vbase = p.v + b * p.v_sb + kvh * p.v_sh;
        _Float16* obase = p.o + b * p.o_sb + h * p.o_sh;

        // Q^T operand (lane holds Q[q][16s + 8g .. +7], RoPE applied), staged
        // through sQ: in the operand layout each lane reads 16 B of its own row,
        // so every load instruction touches 32 rows (cache lines) and the
        // prologue waited on L1 lookups. All threads instead load the tile's Q
        // (and RoPE table) chunks row-contiguously, 16 lanes per 256 B, rotate
        // them and write sQ; after the prologue barrier each wave reads its
        // operand from sQ with conflict-free b128 reads (the K-row layout).
        h8 qreg[C::NS];
        auto stage_q = [&]() {
            const _Float16* qb = p.q + b * p.q_sb + (int64_t)(kvh * p.ratio + sub * p.G) * p.q_sh;
            // chunk c of this thread: (head j, row r, 16-byte column ch), ch
            // fastest; row r of head j is row r % 32 of wave j + G * (r / 32).
            // A tile holds rows_per_wg = 256 / G rows of each of G heads, G in
            // {1, 2, 4}: head and row are a shift and a mask of the slot row
            // (a division by rows_per_wg cost ~30 instructions per chunk).
            // Recomputed from an opaque copy of the thread id at each use so
            // that no index stays live across the loads' latency.
            const uint32_t rsh = (ALT ? 7u : 8u) - (uint32_t)(p.G >> 1); // log2 rows_per_wg
            struct Chunk {
                uint32_t j, r, ch;
            };
            auto chunk = [&](uint32_t t, int c) {
                const uint32_t idx = t + kPPThreads * c;
                const uint32_t rj = idx / C::KCH;
                return Chunk{rj >> rsh, rj & ((1u << rsh) - 1u), idx - rj * C::KCH};
            };
            auto src_row = [&](const Chunk& k) { return wg_q0 + (int)k.r < p.Sq ? (uint32_t)wg_q0 + k.r : 0u; };
            h8 x[QCT];
            f4 cs[QCT], sn[QCT];
            uint32_t t = tid;
            asm volatile("" : "+v"(t));
            // The table loads are issued first, so that they and the Q loads
            // are in flight together: issued after the Q loads, they waited
            // for all of them (the conversions that both the rotation and the
            // plain scaling start with were hoisted above the branch).
            if (p.rope_q) {
#pragma unroll
                for (int c = 0; c < QCT; c++) {
                    const Chunk k = chunk(t, c);
                    const uint64_t off = (uint64_t)src_row(k) * (D / 2) + 4 * k.ch;
                    cs[c] = *reinterpret_cast<const f4*>(p.rot_cos + off);
                    sn[c] = *reinterpret_cast<const f4*>(p.rot_sin + off);
                }
            }
#pragma unroll
            for (int c = 0; c < QCT; c++) {
                const Chunk k = chunk(t, c);
                x[c] = *reinterpret_cast<const h8*>(qb + (int64_t)k.j * p.q_sh + (int64_t)src_row(k) * p.q_ss +
                                                    8 * k.ch);
            }
            if (p.rope_q) {
#pragma unroll
                for (int c = 0; c < QCT; c++) {
                    x[c] = PRE ? rope8_cs_mul(x[c], cs[c], sn[c], p.qmul) : rope8_cs(x[c], cs[c], sn[c]);
                }
            } else if constexpr (PRE) {
#pragma unroll
                for (int c = 0; c < QCT; c++) {
                    x[c] = scale8(x[c], p.qmul);
                }
            }
            const bool neg = !PRE && p.q_sign < 0.0f; // PRE: the sign is in qmul
            asm volatile("" : "+v"(t));
#pragma unroll
            for (int c = 0; c < QCT; c++) {
                const Chunk k = chunk(t, c);
                const uint32_t dst = ((k.j + p.G * (k.r >> 5)) * 32 + (k.r & 31)) * C::LDQ + 8 * k.ch;
                *reinterpret_cast<h8*>(&sQ[dst]) = wg_q0 + (int)k.r < p.Sq ? (neg ? -x[c] : x[c]) : h8{};
            }
        };
        auto read_q = [&]() {
            const _Float16* src = sQ + (rw * 32 + l32) * C::LDQ + 8 * g;
#pragma unroll
            for (int st = 0; st < C::NS; st++) {
                qreg[st] = *reinterpret_cast<const h8*>(src + 16 * st);
            }
        };

        const int wg_q_hi = min(wg_q0 + p.rows_per_wg, p.Sq) - 1;
        int klo, khi;
        visible_key_range(p.mask, wg_q0, wg_q_hi, klo, khi);
        int t_begin = 0, n = 0;
        if (khi >= klo) {
            t_begin = klo / kBN;
            n = khi / kBN + 1 - t_begin;
        }
        if constexpr (SPLIT) {
            split_key_tiles(p.splits, split, t_begin, n);
        }
        // key tile i of this wave's sequence of ng tiles
        const int ng = ALT ? (n + 1 - ugrp) / 2 : n;
        auto tile_at = [&](int i) { return ALT ? t_begin + 2 * i + ugrp : t_begin + i; };
        const int Sk = p.mask.sk;
        const uint32_t k_row_b = (uint32_t)(p.k_ss * 2), v_row_b = (uint32_t)(p.v_ss * 2);
        int row_lo, row_hi;
        row_key_bounds(p.mask, q, row_lo, row_hi);
        // class of key tile t_begin + i for this wave's rows (0 skip, 1 no mask, 2 masked)
        const TileClasses tcls = wave_active ? tile_classes<kBN>(p.mask, q0, q_hi) : TileClasses{1, 0, 1, 0};

        f16x oacc[C::NDT];
#pragma unroll
        for (int dt = 0; dt < C::NDT; dt++) {
            oacc[dt] = f16x{};
        }
        float m_run = -INFINITY;
        float m_use = 0.0f; // m_run, or 0 while it is -inf (PRE: the S^T accumulators start at -m_use)
        f16x minit = f16x{};
        float l_run = 0.0f;
        f16x sacc[2];
        sacc[0] = f16x{};
        sacc[1] = f16x{};
        h8 pb[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            pb[u] = h8{};
        }
        int cls_prev = 0; // classification of the tile whose P is held in pb

        h8 kreg[CT], vreg[CT];
        // registers <- HBM for pair x (K tile x if x < n, V tile x-1 if 1 <= x <= n);
        // a missing tile gets num_records 0, so its loads return 0 and touch nothing.
        // A tile spans at most kBN rows at a seq stride <= 2^24 elements, so its
        // byte range fits 32 bits (tile_bytes); this keeps the per-tile
        // descriptor set-up to a few scalar instructions.
        // Each group calls load_pair with x = 0, 1, 2, ... in order, so the tile
        // addresses advance by one tile stride per call (unsigned arithmetic:
        // V tile -1 of the first call is never read, its num_records is 0).
        uint64_t k_addr = reinterpret_cast<uint64_t>(kbase) + (uint64_t)((int64_t)tile_at(0) * kBN * p.k_ss * 2);
        uint64_t v_addr = reinterpret_cast<uint64_t>(vbase) + (uint64_t)((int64_t)tile_at(-1) * kBN * p.v_ss * 2);
        constexpr int STEP = ALT ? 2 * kBN : kBN;
        const uint64_t k_step = (uint64_t)(STEP * p.k_ss * 2), v_step = (uint64_t)(STEP * p.v_ss * 2);
        auto load_pair = [&](int x) {
            const int tk = tile_at(x), tv = ALT ? tile_at(x - 1) : t_begin + x - 1;
            const auto rk = make_rsrc(reinterpret_cast<const void*>(k_addr),
                                      x < ng ? tile_bytes<kBN>(Sk - tk * kBN, k_row_b, D * 2) : 0u);
            const auto rv = make_rsrc(reinterpret_cast<const void*>(v_addr),
                                      (x >= 1 && x <= ng) ? tile_bytes<kBN>(Sk - tv * kBN, v_row_b, D * 2) : 0u);
            k_addr += k_step;
            v_addr += v_step;
#pragma unroll
            for (int it = 0; it < CT; it++) {
                kreg[it] = buffer_load_h8(rk, coff_k[it], 0);
                vreg[it] = buffer_load_h8(rv, coff_v[it], 0);
            }
        };
        // LDS <- registers for pair x.  Written whether or not the tiles exist:
        // a missing tile was loaded as zeros into a slot that no phase reads
        // (K(x) for x >= n, V(x - 1) for x < 1 or x > n), and every slot is
        // written on the same schedule as for an existing tile, after the last
        // read of its previous contents.  No branches in the VALU phase.
        auto store_pair = [&](int x) {
            _Float16* sK = sKs + (ALT ? ugrp : x & 1) * C::TILE_K;
            _Float16* sV = sVs + (ALT ? ugrp : (x - 1) & 1) * C::TILE_V;
#pragma unroll
            for (int it = 0; it < CT; it++) {
                if (TASK % 256 == 0 || clk[it] >= 0) {
                    *reinterpret_cast<h8*>(&sK[clk[it]]) = kreg[it];
                    *reinterpret_cast<h8*>(&sV[clv[it]]) = vreg[it];
                }
            }
        };

        // DMA staging: each group sets up pair x = 0, 1, 2, ... in order (the
        // same address stepping as load_pair) and issues its half of the 8
        // DMAs: K group dma_j0 + k / 2 for even k (group B), V group dma_j0 +
        // k / 2 for odd k (group A).
        struct DmaPair {
            i32x4_t rk, rv;
            uint32_t mk, mv;
        };
        auto uniform = [](i32x4_t r) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                r[e] = __builtin_amdgcn_readfirstlane(r[e]);
            }
            return r;
        };
        auto dma_pair = [&](int x) {
            const int tk = tile_at(x), tv = ALT ? tile_at(x - 1) : t_begin + x - 1;
            DmaPair d;
            d.rk = uniform(make_rsrc_v(reinterpret_cast<const void*>(k_addr),
                                       x < ng ? tile_bytes<kBN>(Sk - tk * kBN, k_row_b, D * 2) : 0u));
            d.rv = uniform(make_rsrc_v(reinterpret_cast<const void*>(v_addr),
                                       (x >= 1 && x <= ng) ? tile_bytes<kBN>(Sk - tv * kBN, v_row_b, D * 2) : 0u));
            d.mk = (uint32_t)__builtin_amdgcn_readfirstlane(
                (int)(lds_k + (uint32_t)(((ALT ? ugrp : x & 1) * C::TILE_K + (int)dma_j0 * C::PSK) * 2)));
            d.mv = (uint32_t)__builtin_amdgcn_readfirstlane(
                (int)(lds_v + (uint32_t)(((ALT ? ugrp : (x - 1) & 1) * C::TILE_V + (int)dma_j0 * C::PSV) * 2)));
            k_addr += k_step;
            v_addr += v_step;
            return d;
        };
        auto dma_issue = [&](const DmaPair& d, int k) {
            const uint32_t j = dma_j0 + (uint32_t)(k >> 1);
            const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((int)(4u * j * ((k & 1) ? v_row_b : k_row_b)));
            if (k & 1) {
                dma_load16_s(d.rv, dma_vv, so, d.mv + (uint32_t)((k >> 1) * C::PSV * 2));
            } else {
                dma_load16_s(d.rk, dma_vk, so, d.mk + (uint32_t)((k >> 1) * C::PSK * 2));
            }
        };

        // M(i): O += V(i-1)^T P(i-1) (i >= 1) then S(i) = K(i) Q^T (i < n), as one
        // stream of MFMAs whose LDS operands are read kOpDepth MFMAs ahead through
        // a small register ring; sched_barrier stops the compiler from hoisting
        // every read (which would need ~100 more VGPRs).
        auto mfma_stream = [&](auto do_pv_c, auto do_s_c, int i) {
            // The MFMA phase runs at raised wave priority: each SIMD also holds
            // the other group's wave in its softmax phase, whose VALU stream
            // otherwise delays the issue of the next MFMA (-1.2 % on causal GQA
            // B4 Hq32 Hkv8 S4096 D128 with RoPE and on B2 Hq32 Hkv8 S8192 D128 in
            // same-box A/B runs; the INT8 head_dim 128 kernel, whose softmax
            // side is its critical path, measured slower with it)
            __builtin_amdgcn_s_setprio(1);
            constexpr bool DO_PV = decltype(do_pv_c)::value;
            constexpr bool DO_S = decltype(do_s_c)::value;
            constexpr int NPV = DO_PV ? 4 * C::NDT : 0; // (u, dt)
            constexpr int NSK = DO_S ? 2 * C::NS : 0;   // (s, kt)
            constexpr int T = NPV + NSK;
            constexpr int DEPTH = T < kOpDepth ? T : kOpDepth;
            const int j16 = lane & 15;
            const _Float16* vrow = sVs + (ALT ? ugrp : (i - 1) & 1) * C::TILE_V + (4 * g + (j16 >> 2)) * C::LDV +
                                   16 * ((lane >> 4) & 1) + 4 * (j16 & 3);
            const _Float16* krow = sKs + (ALT ? ugrp : i & 1) * C::TILE_K + l32 * C::LDK + 8 * g;
            // DMA layout: K row l32 (+32 kt) is row b = l32 % 4 of group l32 / 4
            // (+8 kt), its chunk 2 st + g at position 2 (st ^ 2b) + g, i.e. at
            // 16 (st % 2) + 32 ((st / 2) ^ b) halves: one base per st / 2.  V
            // row 16u + 8h + 4g + j16 / 4 is row b = j16 / 4 of group 4u + 2h + g,
            // its columns 32 dt + 16 x + 4 (j16 % 4) at chunk quad dt ^ b: one
            // base per dt.
            const _Float16* kb[C::DMA ? 4 : 1];
            const _Float16* vb[C::DMA ? C::NDT : 1];
            if constexpr (C::DMA) {
                const int bk = l32 & 3, bv = (j16 >> 2) & 3;
                const _Float16* k0 = sKs + (ALT ? ugrp : i & 1) * C::TILE_K + (l32 >> 2) * C::PSK + 128 * bk + 8 * g;
                const _Float16* v0 = sVs + (ALT ? ugrp : (i - 1) & 1) * C::TILE_V + g * C::PSV + 128 * bv +
                                     16 * ((lane >> 4) & 1) + 4 * (j16 & 3);
#pragma unroll
                for (int s2 = 0; s2 < 4; s2++) {
                    kb[s2] = k0 + 32 * (s2 ^ bk);
                }
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
                    vb[dt] = v0 + 32 * (dt ^ bv);
                }
            }
            auto op = [&](int j) -> h8 {
                if (j < NPV) {
                    const int u = j / C::NDT, dt = j % C::NDT;
                    if constexpr (C::DMA) {
                        const _Float16* base = vb[dt] + (4 * u) * C::PSV;
                        h4 lo = lds_read_tr16(base);
                        h4 hi = lds_read_tr16(base + 2 * C::PSV);
                        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    }
                    const _Float16* base = vrow + (16 * u) * C::LDV + 32 * dt;
                    h4 lo = lds_read_tr16(base);
                    h4 hi = lds_read_tr16(base + 8 * C::LDV);
                    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                }
                const int js = j - NPV, st = js >> 1, kt = js & 1;
                if constexpr (C::DMA) {
                    return *reinterpret_cast<const h8*>(kb[st >> 1] + kt * 8 * C::PSK + 16 * (st & 1));
                }
                return *reinterpret_cast<const h8*>(krow + kt * 32 * C::LDK + 16 * st);
            };
            f16x acc0 = {}, acc1 = {};
            h8 ring[DEPTH > 0 ? DEPTH : 1];
#pragma unroll
            for (int j = 0; j < DEPTH; j++) {
                ring[j] = op(j);
            }
#pragma unroll
            for (int j = 0; j < T; j++) {
                const h8 a = ring[j % DEPTH];
                if (j + DEPTH < T) {
                    ring[j % DEPTH] = op(j + DEPTH);
                }
                if (j < NPV) {
                    const int u = j / C::NDT, dt = j % C::NDT;
                    oacc[dt] = mfma_32x32x16_f16(a, pb[u], oacc[dt]);
                } else {
                    const int js = j - NPV, st = js >> 1;
                    if (js & 1) {
                        acc1 = mfma_32x32x16_f16(a, qreg[st], (PRE && st == 0) ? minit : acc1);
                    } else {
                        acc0 = mfma_32x32x16_f16(a, qreg[st], (PRE && st == 0) ? minit : acc0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            if constexpr (DO_S) {
                sacc[0] = acc0;
                sacc[1] = acc1;
            }
        };
        auto phase_m = [&](int i) {
            if (!wave_active) {
                return;
            }
            const bool do_pv = i >= 1 && cls_prev != 0;
            const int cls_now = i < ng ? tile_class(tcls, tile_at(i)) : 0;
            using T_ = std::true_type;
            using F_ = std::false_type;
            if (do_pv && cls_now != 0) {
                mfma_stream(T_{}, T_{}, i);
            } else if (do_pv) {
                mfma_stream(T_{}, F_{}, i);
            } else if (cls_now != 0) {
                mfma_stream(F_{}, T_{}, i);
            }
            cls_prev = cls_now;
        };

        // V(i): softmax of S(i) -> pb, rescale O
        auto phase_v = [&](int i) {
            if (!wave_active || cls_prev == 0) {
                return;
            }
            if (cls_prev == 2) {
                const int kt0 = tile_at(i) * kBN;
                const int a = row_lo - kt0 - 4 * g;
                const int bnd = row_hi - kt0 - 4 * g;
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int off = kt * 32 + 8 * (e >> 2) + (e & 3);
                        sacc[kt][e] = (off < a || off > bnd) ? -INFINITY : sacc[kt][e];
                    }
                }
            }
            float mx = max_tree<32>([&](int e) { return sacc[e >> 4][e & 15]; });
            mx = pair_max(mx);
            // PRE: sacc = S c - m_use already; otherwise S
            const float m_new = PRE ? fmaxf(m_run, mx + m_use) : fmaxf(m_run, mx * p.c);
            const bool grow = m_new > m_run + kRescaleThreshold;
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
                const float m_use_new = (m_run == -INFINITY) ? 0.0f : m_run;
                if constexpr (PRE) {
                    // re-base this tile's exponents and the next tiles' start
                    const float shift = m_use - m_use_new;
#pragma unroll
                    for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            sacc[kt][e] += shift;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        minit[e] = -m_use_new;
                    }
                }
                m_use = m_use_new;
            }
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float x = PRE ? sacc[kt][e] : fmaf(sacc[kt][e], p.c, -m_use);
                    pb[kt * 2 + (e >> 3)][e & 7] = (_Float16)fast_exp2(x);
                }
            }
            l_run = sum_h8x4(pb, l_run);
        };

        // ---- prologue: pair 0 in LDS; each group's registers hold its next pair
        // (DMA: group B's K(0) in flight while Q stages)
        const bool dma_wave = __builtin_amdgcn_readfirstlane(grp) == 1;
        if constexpr (C::DMA) {
            if ((ALT || dma_wave) && n > 0) {
                const DmaPair d0 = dma_pair(0);
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    dma_issue(d0, k);
                }
            }
        } else if (n > 0) {
            load_pair(0);
        }
        stage_q();
        if constexpr (C::DMA) {
            if (ALT || dma_wave) {
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // K(0) landed (not tracked by the compiler)
            }
        } else if (n > 0) {
            store_pair(0);
            load_pair(1);
        }
        __syncthreads();
        read_q();
        // Both groups pass 2n + 2 barriers; group B starts one phase late.
        if constexpr (ALT) {
            // n2 steps of group A; group B's last may be missing
            const int n2 = (n + 1) / 2;
            if (n > 0) {
                if (dma_wave) {
                    __syncthreads();
                }
                for (int i = 0; i < n2; i++) {
                    phase_m(i);
                    __syncthreads();
                    if constexpr (C::DMA) {
                        const DmaPair d = dma_pair(i + 1);
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            dma_issue(d, k);
                        }
                    } else {
                        store_pair(i + 1);
                        load_pair(i + 2);
                    }
                    phase_v(i);
                    if constexpr (C::DMA) {
                        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // K(i + 1), V(i) landed
                    }
                    __syncthreads();
                }
                phase_m(n2);
                __syncthreads();
                if (!dma_wave) {
                    __syncthreads();
                }
            }
        } else if (n > 0) {
            if (grp == 0) {
                if constexpr (C::DMA) {
                    (void)dma_pair(0); // the address stepping starts at pair 0
                }
                for (int i = 0; i < n; i++) {
                    phase_m(i);
                    __syncthreads();
                    if constexpr (!C::DMA) {
                        store_pair(i + 1);
                        load_pair(i + 2);
                    } else {
                        // V(i) into V(i - 2)'s slot, last read in phase 2i - 1;
                        // first read in phase 2i + 2
                        const DmaPair d = dma_pair(i + 1);
#pragma unroll
                        for (int k = 1; k < 8; k += 2) {
                            dma_issue(d, k);
                        }
                    }
                    phase_v(i);
                    if constexpr (C::DMA) {
                        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // V(i) landed
                    }
                    __syncthreads();
                }
                phase_m(n);
                __syncthreads();
                __syncthreads();
            } else {
                // DMA: group B issues K(i + 2) at the start of its V(i) and
                // waits for it at the end of its M(i + 1); K(1) in phase 0
                if constexpr (C::DMA) {
                    if (1 < n) {
                        const DmaPair d1 = dma_pair(1);
#pragma unroll
                        for (int k = 0; k < 8; k += 2) {
                            dma_issue(d1, k);
                        }
                    }
                } else {
                    store_pair(1);
                    load_pair(2);
                }
                __syncthreads();
                for (int i = 0; i < n; i++) {
                    phase_m(i);
                    if constexpr (C::DMA) {
                        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0)); // K(i + 1) landed
                    }
                    __syncthreads();
                    if constexpr (C::DMA) {
                        if (i + 2 < n) {
                            const DmaPair d = dma_pair(i + 2);
#pragma unroll
                            for (int k = 0; k < 8; k += 2) {
                                dma_issue(d, k);
                            }
                        }
                    } else {
                        store_pair(i + 2);
                        load_pair(i + 3);
                    }
                    phase_v(i);
                    __syncthreads();
                }
                phase_m(n);
                __syncthreads();
            }
        }

        if constexpr (SPLIT) {
            const float l = pair_sum(l_run);
            if (wave_active && q < p.Sq) {
                const int64_t row = split * p.n_rows + ((int64_t)b * p.Hkv * p.ratio + h) * p.Sq + q;
                store_partial(oacc, m_run, l, g == 0, p.part_o, p.part_ml, row, D, 0, g,
                              [](int) { return 1.0f; });
            }
        } else if constexpr (ALT) {
            // group B's O into group A's: fp32 rows in the K/V area (free after
            // the last barrier), (m, l) in the unused half of sQ
            constexpr int LDM = D + 4;
            static_assert(ROW_WAVES * 32 * LDM * 4 <= (2 * C::TILE_K + 2 * C::TILE_V) * 2, "O fits the K/V area");
            float* const so = reinterpret_cast<float*>(smem) + (rw * 32 + l32) * LDM + 4 * g;
            float2* const sml = reinterpret_cast<float2*>(sQ + ROW_WAVES * 32 * C::LDQ) + rw * 32 + l32;
            const float l = pair_sum(l_run);
            if (grp == 1 && wave_active) {
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
#pragma unroll
                    for (int qq = 0; qq < 4; qq++) {
                        *reinterpret_cast<f4*>(so + 32 * dt + 8 * qq) = f4{oacc[dt][4 * qq], oacc[dt][4 * qq + 1],
                                                                           oacc[dt][4 * qq + 2], oacc[dt][4 * qq + 3]};
                    }
                }
                if (g == 0) {
                    *sml = float2{m_run, l};
                }
            }
            __syncthreads();
            if (grp == 0 && wave_active) {
                const float2 other = *sml;
                const float m = fmaxf(l > 0.0f ? m_run : -INFINITY, other.y > 0.0f ? other.x : -INFINITY);
                const float wa = l > 0.0f ? fast_exp2(m_run - m) : 0.0f;
                const float wb = other.y > 0.0f ? fast_exp2(other.x - m) : 0.0f;
                const float ls = l * wa + other.y * wb;
                const float inv = ls > 0.0f ? 1.0f / ls : 0.0f;
#pragma unroll
                for (int dt = 0; dt < C::NDT; dt++) {
#pragma unroll
                    for (int qq = 0; qq < 4; qq++) {
                        const f4 x = *reinterpret_cast<const f4*>(so + 32 * dt + 8 * qq);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            oacc[dt][4 * qq + e] = oacc[dt][4 * qq + e] * wa + x[e] * wb;
                        }
                    }
                }
                store_o_tile<D, C::LDQ>(oacc, [&](int) { return f4{inv, inv, inv, inv}; }, sQ + rw * 32 * C::LDQ,
                                        obase, q0, p.Sq, p.o_ss, lane);
            }
        } else if (wave_active) {
            // O = O^T / l, through this wave's sQ slot (free since read_q)
            const float l = pair_sum(l_run);
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            store_o_tile<D, C::LDQ>(oacc, [&](int) { return f4{inv, inv, inv, inv}; }, sQ + wave * 32 * C::LDQ,
                                    obase, q0, p.Sq, p.o_ss, lane);
        }
        if constexpr (C::PERSIST) {
            __syncthreads(); // the next row tile's Q staging writes every wave's slot
        }
    };
    if constexpr (C::PERSIST) {
        for (int item = 0;; item++) {
            const int wg = persistent_item(blockIdx.x, gridDim.x, item, p.n_items);
            if (wg < 0) {
                break;
            }
            run_tile(wg);
        }
    } else {
        run_tile(blockIdx.x);
    }
}

template <int D, bool PRE>
__global__ __launch_bounds__(kPPThreads, 1) void fa_fwd_f16_pp(PrefillParams p) {
    pp_body<D, PRE, PPMode::kWhole>(p);
}

template <int D, bool PRE>
__global__ __launch_bounds__(kPPThreads, 1) void fa_fwd_f16_pp_split(PrefillParams p) {
    pp_body<D, PRE, PPMode::kSplit>(p);
}

template <int D, bool PRE>
__global__ __launch_bounds__(kPPThreads, 1) void fa_fwd_f16_pp_alt(PrefillParams p) {
    pp_body<D, PRE, PPMode::kAlternate>(p);
}

template <int D, bool PRE>
int launch_pp_as(const PrefillParams& p, int64_t n_wg, hipStream_t stream, std::string& err) {
    // persistent: as many workgroups as the device holds at once, each
    // walking its share of the n_wg row tiles
    auto* const kernel = p.splits > 1   ? &fa_fwd_f16_pp_split<D, PRE>
                         : p.alternate ? &fa_fwd_f16_pp_alt<D, PRE>
                                       : &fa_fwd_f16_pp<D, PRE>;
    int64_t grid = n_wg;
    if (PPCfg<D>::PERSIST) {
        const int64_t resident = resident_workgroups(reinterpret_cast<const void*>(kernel), kPPThreads, err);
        if (resident <= 0) {
            return -1;
        }
        grid = std::min(n_wg, resident);
    }
    KernelTimerGuard timer(stream);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(kPPThreads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = hipGetErrorString(e);
        return -1;
    }
    return 0;
}

// Q pre-scaled into log2 units needs |q| c representable in fp16: c <= 1
// keeps |q c| <= |q|.  Not at D = 32, where the 16 registers of the start
// block would leave room for 3 waves per SIMD, not the 4 that let two
// workgroups share a compute unit.
template <int D>
int launch_pp(const PrefillParams& p, int64_t n_wg, hipStream_t stream, std::string& err) {
    if (D >= 64 && p.c <= 1.0f) {
        return launch_pp_as<D, D >= 64>(p, n_wg, stream, err);
    }
    return launch_pp_as<D, false>(p, n_wg, stream, err);
}

} // namespace

constexpr int64_t kMaxSeqStride = 1 << 24;

int xcd_head_group_chunk(int n_head_groups, int64_t kv_bytes) {
    constexpr int kXcds = 8;
    constexpr int64_t kL2Budget = 3 << 20; // of the 4 MB L2 per XCD
    if (n_head_groups % kXcds != 0 || kv_bytes <= 0) {
        return 0;
    }
    const int per_xcd = n_head_groups / kXcds;
    int c = (int)std::max<int64_t>(1, std::min<int64_t>(per_xcd, kL2Budget / kv_bytes));
    while (per_xcd % c != 0) {
        c--;
    }
    return c;
}

float softmax_log2_scale(float scale) {
    return std::max(std::fabs(scale) * kLog2e, 1e-30f);
}

// Query heads per prefill workgroup (G | Hq/Hkv, G <= 4).
static int prefill_group(const AttnArgs& a) {
    const int ratio = a.Hq / a.Hkv;
    return ratio % 4 == 0 ? 4 : (ratio % 2 == 0 ? 2 : 1);
}

int prefill_splits(const AttnArgs& a, int wg_rows, double tile_us, double alternate_us, double split_tile_us,
                   int launches, size_t max_partials) {
    // Too few workgroups for the CUs and many key tiles for each: split the
    // keys, by the least modelled time.  A workgroup takes about 5 us beside
    // its key tiles; the partials are written and read at about 2.5 MB/us, and
    // the combine launch adds about 5 us.  Measured, us a call, unsplit against
    // split: B1 Hq32 Hkv8 Sq256 Sk16640 D128 355 / 80 (8 splits, 79 of them
    // the 33.5 MB launch); Sq64 Sk4096 92 / 27; B2 Sq256 Sk8192 183 / 85; B1
    // Hq16 Hkv4 Sq128 Sk2000 D64 37 / 19.  Whole prompts this small stay
    // unsplit (1 x 8 heads, S 512, D64: 13.9 / 18.3; S 1024 causal 22.8 /
    // 23.2).  Above D = 128 the larger rows make it 7 us (D = 256, 128 kv heads
    // with one row, Sk 512: 17.5 / 19.5).  With more workgroups than CUs the
    // persistent grid balances them.
    const double merge_us = a.D > 128 ? 7.0 : 5.0;
    const int G = prefill_group(a);
    const int rows = wg_rows / G;
    const int64_t row_tiles = (a.Sq + rows - 1) / rows;
    const int64_t n_wg = row_tiles * a.B * (a.Hq / G);
    if (n_wg > 256) {
        return 1;
    }
    const MaskSpec mask{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    int64_t tiles = 0; // of the longest row tile: the last one, or one from the middle under a window
    for (int64_t rt : {row_tiles - 1, row_tiles / 2, int64_t{0}}) {
        int lo, hi;
        visible_key_range(mask, (int)(rt * rows), (int)std::min<int64_t>((rt + 1) * rows, a.Sq) - 1, lo, hi);
        tiles = std::max<int64_t>(tiles, hi >= lo ? hi / kBN + 1 - lo / kBN : 0);
    }
    int best_s = 1;
    double best = 0.0;
    for (int64_t s = 1; s <= std::min<int64_t>(tiles / 2, kMaxSplits); s++) {
        const size_t partials = splitk_partial_bytes(a, (int)s);
        if (region_bytes(partials) > max_partials) {
            break;
        }
        const double rounds = (double)((n_wg * s + 255) / 256);
        const double t = s == 1 ? 5.0 + (alternate_us > 0.0 && n_wg <= 128 ? (double)((tiles + 1) / 2) * alternate_us
                                                                           : (double)tiles * tile_us)
                                : rounds * (5.0 * launches + (double)((tiles + s - 1) / s) * split_tile_us) +
                                      merge_us * launches + 2.0 * (double)partials / 2.5e6;
        if (s == 1 || t < best) {
            best = t;
            best_s = (int)s;
        }
    }
    return best_s;
}

// Splits of an FP16 prefill call.  Up to D = 256; a 64-key tile takes about
// 1.4 us at D = 128 with 256 rows, or at D = 256 with 128.
static int f16_prefill_splits(const AttnArgs& a, size_t max_partials) {
    if (a.D > 256) {
        return 1;
    }
    const double tile_us = 0.4 + (a.D > 128 ? a.D / 256.0 : a.D / 128.0);
    return prefill_splits(a, a.D > 128 ? kKPairRows : 32 * kPPWaves, tile_us, a.D > 128 ? 0.0 : 1.4 * tile_us, tile_us,
                          1, max_partials);
}

// Steps of the longest sequence of row tiles that a workgroup of a persistent
// prefill launch walks, `fixed` steps added per row tile: `rows` rows of G heads
// per workgroup, `tiles_per_step` key tiles per step, head groups dealt to the
// XCDs `chunk` at a time.  Follows persistent_item and wg_tile for XCD 0 of 8
// with 32 workgroups (the others hold the same), of which every fourth and
// the last are looked at.
static double longest_walk(const AttnArgs& a, int rows, int tiles_per_step, double fixed, int chunk) {
    const MaskSpec mask{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    const int row_tiles = (a.Sq + rows - 1) / rows;
    const int head_groups = a.B * (a.Hq / prefill_group(a));
    const int items = row_tiles * head_groups;
    auto steps = [&](int rt) {
        int lo, hi;
        visible_key_range(mask, rt * rows, std::min((rt + 1) * rows, a.Sq) - 1, lo, hi);
        return hi >= lo ? (hi / kBN - lo / kBN + tiles_per_step) / tiles_per_step : 0;
    };
    double longest = 0.0;
    for (int w = 0; w < 32; w = w == 28 ? 31 : w + 4) {
        double walk = 0.0;
        for (int k = 0;; k++) {
            const int slot = 32 * k + ((k & 1) ? 31 - w : w);
            if (8 * slot >= items) {
                break;
            }
            const int rt = chunk > 0 ? slot % (chunk * row_tiles) / chunk : 8 * slot / head_groups;
            walk += fixed + steps(row_tiles - 1 - rt);
        }
        longest = std::max(longest, walk);
    }
    return longest;
}

bool prefill_alternate(const AttnArgs& a, double tile_us, double step_us, int chunk, int max_half_wg,
                       double half_margin) {
    // Twice as many row tiles of half as many steps, where the longest row
    // tile of a launch sets its time: up to two row tiles per CU.  A row tile
    // takes about 5 us beside its steps.
    const int rows = 32 * kPPWaves / prefill_group(a);
    const int head_groups = a.B * (a.Hq / prefill_group(a));
    const int64_t n_wg = (int64_t)((a.Sq + rows - 1) / rows) * head_groups;
    // Rows that fill at most half a row tile: as many workgroups as without, whose
    // second group had no rows and left each step shorter than the model's.
    const bool half = a.Sq <= rows / 2;
    if (a.Sk <= 2 * kBN || n_wg > (half ? max_half_wg : 512)) {
        return false;
    }
    return step_us * longest_walk(a, rows / 2, 2, 5.0 / step_us, chunk) <
           (half ? half_margin : 0.97) * tile_us * longest_walk(a, rows, 1, 5.0 / tile_us, chunk);
}

// Whether the two groups of a workgroup take the key tiles in turn (D <= 128).
// A step of 128 rows and two tiles takes about 1.4 times a step of 256 rows and
// one.  Measured, us a call, whole against alternating (Hq 32 Hkv 8, causal): B1
// S1024 D128 29.0 / 20.6, D64 22.5 / 15.8; B1 S2048 D128 55 / 45; B2 S1024 D128
// 31.8 / 30.5; and where the rule keeps whole row tiles: B1 S2048 D128 not
// causal 71 / 79, B2 S1500 49 / 58, B2 S2048 78 / 92.  Of rows that fill
// half a tile it does not pay at D = 32, where two workgroups share a CU, with more
// than 256 (512 kv heads of 33 to 128 rows, Sk 400 13.6 / 16.6), nor at D = 128 with
// more than 128, which stream their own K and V (256 kv heads of 64 rows, Sk 2048
// 52 / 57, Sk 512 18.7 / 20.1).
static bool f16_prefill_alternate(const AttnArgs& a, int chunk) {
    const double tile_us = 0.4 + a.D / 128.0;
    const int max_half_wg = a.D == 32 ? 256 : a.D == 128 ? 128 : 512;
    return a.D <= 128 && prefill_alternate(a, tile_us, 1.4 * tile_us, chunk, max_half_wg, 0.95);
}

static int f16_hg_chunk(const AttnArgs& a) {
    return xcd_head_group_chunk(a.B * (a.Hq / prefill_group(a)),
                                2 * (int64_t)a.Sk * a.D * (int64_t)sizeof(_Float16));
}

static CallPlan f16_prefill_plan(const AttnArgs& a, size_t max_partials) {
    CallPlan plan;
    plan.splits = f16_prefill_splits(a, max_partials);
    if (plan.splits > 1) {
        plan.form = CallForm::kSplit;
        plan.scratch = splitk_partial_bytes(a, plan.splits);
    } else if (f16_prefill_alternate(a, f16_hg_chunk(a))) {
        plan.form = CallForm::kAlternate;
    }
    return plan;
}

int fwd_f16_prefill(const AttnArgs& a, bool rope_q, hipStream_t stream, std::string& err, ScratchRegion* region) {
    CallPlan plan = f16_prefill_plan(a, region != nullptr ? region->bytes - region->used : SIZE_MAX);
    SplitRows out{};
    StreamScratch ws(ScratchUse::SplitKPartials, region);
    int rc = splitk_begin(a, plan.splits, ws, stream, out, err);
    if (rc == kScratchFull) {
        plan = f16_prefill_plan(a, 0); // keys not split
        rc = splitk_begin(a, plan.splits, ws, stream, out, err);
    }
    if (rc != 0) {
        return -1;
    }
    PrefillParams p{};
    p.q = static_cast<const _Float16*>(a.q);
    p.k = static_cast<const _Float16*>(a.k);
    p.v = static_cast<const _Float16*>(a.v);
    p.o = static_cast<_Float16*>(a.o);
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
    p.o_sb = a.os[0];
    p.o_sh = a.os[1];
    p.o_ss = a.os[2];
    p.Sq = a.Sq;
    p.Hkv = a.Hkv;
    p.ratio = a.Hq / a.Hkv;
    const bool kpair = a.D > 128 && a.D <= 256;
    const bool dpair = a.D > 256;
    // every kernel holds G query heads of one kv head (G | Hq/Hkv, G <= 4)
    // and 128 (query, head) rows per workgroup: 8 waves of 32 rows (D <= 128)
    // or 4 pairs of waves of 32 rows (D > 128)
    p.G = prefill_group(a);
    p.rows_per_wg = (kpair ? kKPairRows : dpair ? kDPairRows : 32 * kPPWaves) / p.G;
    p.groups_per_kv = p.ratio / p.G;
    p.n_head_groups = a.B * a.Hkv * p.groups_per_kv;
    p.hg_chunk = f16_hg_chunk(a);
    p.splits = plan.splits;
    p.alternate = plan.form == CallForm::kAlternate;
    if (p.alternate) {
        p.rows_per_wg /= 2;
    }
    p.n_row_tiles = (a.Sq + p.rows_per_wg - 1) / p.rows_per_wg;
    p.c = softmax_log2_scale(a.scale);
    p.q_sign = a.scale < 0.0f ? -1.0f : 1.0f;
    p.qmul = p.q_sign * p.c;
    p.mask = MaskSpec{a.Sk, a.Sk - a.Sq, a.causal ? 1 : 0, a.window > 0 ? a.window : 0};
    p.rope_q = rope_q ? 1 : 0;

    const int64_t n_wg = (int64_t)p.n_row_tiles * p.n_head_groups * p.splits;
    p.n_items = (int32_t)std::min<int64_t>(n_wg, INT32_MAX);
    if (n_wg <= 0) {
        err = "empty launch grid";
        return -1;
    }
    if (n_wg > INT32_MAX) {
        err = "launch grid too large";
        return -1;
    }
    p.part_o = out.part_o;
    p.part_ml = out.part_ml;
    p.n_rows = out.n_rows;
    rc = -1;
    switch (a.D) {
    case 32: rc = launch_pp<32>(p, n_wg, stream, err); break;
    case 64: rc = launch_pp<64>(p, n_wg, stream, err); break;
    case 96: rc = launch_pp<96>(p, n_wg, stream, err); break;
    case 128: rc = launch_pp<128>(p, n_wg, stream, err); break;
    default:
        if (kpair) {
            rc = launch_kpair(p, (int)a.D, n_wg, stream, err);
        } else if (dpair) {
            rc = launch_dpair(p, (int)a.D, n_wg, stream, err);
        } else {
            err = "unsupported head_dim (multiples of 32 from 32 to 512)";
        }
        break;
    }
    return rc != 0 ? rc : splitk_finish(a, out, stream, err);
}

bool splitk_supported(const AttnArgs& a);
bool splitk_built(const AttnArgs& a);

// Auto: the decode kernel for few query rows per kv head, the prefill tiles
// otherwise.  us a call, prefill / decode, each from an HBM-sized set of caches
// unless marked [r], where one cache is read again and again:
//   * up to Sk = 128 both are the launch (8.9 / 8.9); from there one decode
//     workgroup per kv head, no merge, is quicker as long as they run at once
//     (D = 128, 8 kv heads: 10.7 / 9.1 at 256, 13.4 / 9.7 at 400; D = 192, 256
//     kv heads: 22.6 / 18.4 at 511), but not from 1024 of them on (D = 128, Sk
//     256: 36 / 40)
//   * above D = 192 the decode kernel has one wave per SIMD.  It streams HBM
//     better (D = 256, 64 kv heads of Sk 8192: 102 / 91), and rows of eight
//     query heads together are read once and not per head (128 kv heads of
//     2048: 87 / 57).  A cache up to 64 MB is quicker through the prefill
//     kernel (8 kv heads of 4096: 17.3 / 18.9), and up to the 256 MiB that the
//     last-level cache holds it is when the cache is read again, since only
//     its loads are kept there (128 kv heads of 2048: 47.7 / 51.9 [r], 54.8 /
//     52.6 else)
bool prefer_splitk(const AttnArgs& a) {
    if (!splitk_built(a)) {
        return false;
    }
    const int64_t n_bkv = (int64_t)a.B * a.Hkv;
    if (a.D > 192) {
        const int64_t kv_bytes = n_bkv * a.Sk * a.D * (int64_t)(2 * sizeof(_Float16));
        return a.Sk >= 512 && (a.Hq > 4 * a.Hkv || kv_bytes > (int64_t)256 << 20);
    }
    return a.Sk >= 512 || (a.Sk > 128 && n_bkv <= 256);
}

int f16_call_plan(const AttnArgs& a, size_t max_partials, CallPlan& plan, std::string& err) {
    if (!prefer_splitk(a)) {
        plan = f16_prefill_plan(a, max_partials);
        return 0;
    }
    plan = CallPlan{CallForm::kDecode, 0, 0};
    SplitKPlan splits;
    if (splitk_plan(a, max_partials, splits, err) != 0) {
        return -1;
    }
    plan.splits = splits.splits;
    plan.scratch = splitk_partial_bytes(a, splits.splits);
    return 0;
}

int64_t fwd_f16_scratch_bytes(const AttnArgs& a, F16Path path, std::string& err) {
    const bool splitk = path == F16Path::SplitK || (path == F16Path::Auto && prefer_splitk(a));
    size_t bytes = 0;
    auto left = [&]() { return kNoAllocBytes - std::min(bytes, kNoAllocBytes); };
    if (a.has_rope && a.Sk > 0) {
        bytes += region_bytes((size_t)a.B * a.Hkv * a.Sk * a.D * sizeof(_Float16));
    }
    // fewer splits where the partials would not fit beside the K copy
    if (!splitk) {
        bytes += region_bytes(splitk_partial_bytes(a, f16_prefill_splits(a, left())));
    } else if (splitk_built(a)) {
        SplitKPlan plan;
        if (splitk_plan(a, left(), plan, err) != 0) {
            return -1;
        }
        bytes += region_bytes(splitk_partial_bytes(a, plan.splits));
    }
    return (int64_t)bytes;
}

int fwd_f16(const AttnArgs& in, F16Path path, hipStream_t stream, std::string& err, ScratchRegion* region) {
    AttnArgs a = in;
    // K/V rows are addressed with 32-bit byte offsets inside a 64-key tile
    if (a.ks[2] < 0 || a.vs[2] < 0 || a.ks[2] > kMaxSeqStride || a.vs[2] > kMaxSeqStride) {
        err = "key/value seq strides must be in [0, 2^24] elements";
        return -1;
    }
    const bool splitk = path == F16Path::SplitK || (path == F16Path::Auto && prefer_splitk(a));
    if (path == F16Path::SplitK && !splitk_supported(a)) {
        err = "split-K path needs head_dim in {32, 64, 128} and (num_heads / num_kv_heads) * seq_len <= 32";
        return -1;
    }
    StreamScratch krot(ScratchUse::RotatedK, region);
    if (a.has_rope && a.Sk > 0) {
        const size_t bytes = (size_t)a.B * a.Hkv * a.Sk * a.D * sizeof(_Float16);
        if (krot.alloc(bytes, stream, err) != 0 || rope_rotate_k(a, krot.ptr, stream, err) != 0) {
            return -1;
        }
        a.k = krot.ptr;
        a.ks[0] = (int64_t)a.Hkv * a.Sk * a.D;
        a.ks[1] = (int64_t)a.Sk * a.D;
        a.ks[2] = a.D;
    }
    return splitk ? fwd_f16_splitk(a, a.has_rope != 0, stream, err, region)
                  : fwd_f16_prefill(a, a.has_rope != 0, stream, err, region);
}

} // namespace rdna_amd
