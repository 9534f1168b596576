// Shared by the kernels that split the keys (device code): the split of a row
// tile, its partials, and the merges of a workgroup's waves and of the splits.
//
// A split leaves, per query row, O unnormalised in fp32 and (m, l): its
// reference maximum in log2 units and its row sum relative to it.  The merged
// row is sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s with M the largest m_s.
// A split without a visible key has l_s = 0 and an m_s that is -inf or another
// split's.  A score that is NaN or +inf makes l_s and O_s NaN; as in the kernels
// that see all keys of a row, so does it the row.
#pragma once

#include "fa_common.hpp"

namespace rdna_amd {

constexpr int kMaxSplits = 256; // weights of one row in the merge's LDS

// 2^(m - mref) for m <= mref; 1 for equal infinities (the NaN of their
// difference is dropped by the minimum).
__device__ __forceinline__ float part_weight(float m, float mref) {
    return fast_exp2(fminf(m - mref, 0.0f));
}

// The output rows of a launch and the partials of their splits.  Row
// (b * Hq + h) * Sq + q of split s is partial s * n_rows + row.
struct SplitRows {
    _Float16* o;
    int64_t o_sb, o_sh, o_ss;
    float* part_o;  // [splits][n_rows][D] unnormalised O (splits > 1)
    float* part_ml; // [splits][n_rows][2] (m in log2 units, l)
    int64_t n_rows; // B * Hq * Sq
    int32_t Sq, Hq, ratio, splits;

    __device__ __forceinline__ _Float16* row(int b, int h, int q) const {
        return o + b * o_sb + h * o_sh + (int64_t)q * o_ss;
    }
};

// Splits row tile index rt of a split grid into row tile and split, and the
// tile's n key tiles from t_begin on into the split's share of them.
__device__ __forceinline__ void split_row_tile(int n_row_tiles, int& rt, int& split) {
    split = rt / n_row_tiles;
    rt -= split * n_row_tiles;
}
__device__ __forceinline__ void split_key_tiles(int splits, int split, int& t_begin, int& n) {
    const int per = (n + splits - 1) / splits;
    const int first = min(split * per, n);
    t_begin += first;
    n = min(per, n - first);
}

// Partial of one query row per lane pair: O^T accumulators (lane: columns d0 ..
// d0 + 3, d0 = 32 dt + 8 qq + 4 g, of columns c0 .. c0 + 32 NDT - 1),
// unnormalised, relative to m with row sum l, times factors(d0).  A lane's 16
// bytes of a row meet the rest of their cache line in the L2 within the next
// three stores.
template <int NDT, class Factors>
__device__ __forceinline__ void store_partial(const f16x (&oacc)[NDT], float m, float l, bool write_ml, float* part_o,
                                              float* part_ml, int64_t row, int D, int c0, int g, Factors&& factors) {
    float* const o = part_o + row * D + c0;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
        for (int qq = 0; qq < 4; qq++) {
            const int d0 = 32 * dt + 8 * qq + 4 * g;
            *reinterpret_cast<f4*>(o + d0) =
                factors(d0) * f4{oacc[dt][4 * qq], oacc[dt][4 * qq + 1], oacc[dt][4 * qq + 2], oacc[dt][4 * qq + 3]};
        }
    }
    if (write_ml) {
        *reinterpret_cast<float2*>(part_ml + row * 2) = float2{m, l};
    }
}

// LDS of finish_rows: half of the waves' O (rows of D + 4 floats, conflict-free
// 16-byte accesses) and every wave's (m, l).
constexpr int finish_lds_bytes(int D, int waves) {
    return (waves / 2 * 32 * (D + 4) + waves * 32 * 2) * 4;
}

// Merges the O^T accumulators (32 columns, unnormalised, relative to m_run,
// with row sums l_run per half-wave) of a workgroup's WAVES waves through
// `lds` and writes split `split` of the rows of kv head `kvh` (column c is
// query row c % Sq of head kvh * ratio + c / Sq): the partial, or, of one split,
// the output.  The values go through scaled(f4, d) last (d the first of
// the four columns).  Every wave's own use of `lds` is over on entry.
template <int D, int WAVES, class Scaled>
__device__ __forceinline__ void finish_rows(f16x (&oacc)[D / 32], float m_run, float l_run, char* lds,
                                            const SplitRows& r, int b, int kvh, int split, Scaled&& scaled) {
    static_assert(WAVES % 2 == 0, "halves of the waves");
    constexpr int NDT = D / 32;
    constexpr int LDM = D + 4;
    constexpr int MERGE = WAVES / 2; // waves whose O is in LDS at once
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int l32 = tid & 31;
    const int g = (tid >> 5) & 1;
    const int M = r.ratio * r.Sq;
    const bool col_valid = l32 < M;
    float* const sm_o = reinterpret_cast<float*>(lds); // [MERGE][32][LDM]
    float* const sm_ml = sm_o + MERGE * 32 * LDM;      // [WAVES][32][2]
    __syncthreads();
    const float l_tot = pair_sum(l_run);
    if (g == 0) {
        sm_ml[(wave * 32 + l32) * 2 + 0] = m_run;
        sm_ml[(wave * 32 + l32) * 2 + 1] = l_tot;
    }
    __syncthreads();
    float mref = -INFINITY, lsum = 0.0f; // of column l32 over the waves
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        mref = fmaxf(mref, sm_ml[(w * 32 + l32) * 2 + 0]);
    }
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        lsum += sm_ml[(w * 32 + l32) * 2 + 1] * part_weight(sm_ml[(w * 32 + l32) * 2 + 0], mref);
    }
    const bool whole = r.splits == 1;
    float scale_w = part_weight(m_run, mref);
    if (whole) {
        scale_w *= lsum > 0.0f ? 1.0f / lsum : 0.0f;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
        oacc[dt] *= scale_w;
    }
    // the upper half of the waves through LDS into the lower half, then those
    // through LDS into whole rows
    float* const my_o = &sm_o[((wave % MERGE) * 32 + l32) * LDM + 4 * g];
    auto put_o = [&]() {
        if (col_valid) {
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++) {
                    *reinterpret_cast<f4*>(my_o + 32 * dt + 8 * e4) =
                        f4{oacc[dt][4 * e4], oacc[dt][4 * e4 + 1], oacc[dt][4 * e4 + 2], oacc[dt][4 * e4 + 3]};
                }
            }
        }
    };
    if (wave >= MERGE) {
        put_o();
    }
    __syncthreads();
    if (wave < MERGE && col_valid) {
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const f4 x = *reinterpret_cast<const f4*>(my_o + 32 * dt + 8 * e4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    oacc[dt][4 * e4 + e] += x[e];
                }
            }
        }
    }
    if (wave < MERGE) {
        put_o(); // its own slot, read above by the same lanes
    }
    // the group's rows are consecutive
    const int64_t part = split * r.n_rows + ((int64_t)b * r.Hq + kvh * r.ratio) * r.Sq;
    if (!whole && tid < M) { // M <= 32: the threads that hold mref, lsum of column tid
        r.part_ml[(part + tid) * 2 + 0] = mref;
        r.part_ml[(part + tid) * 2 + 1] = lsum;
    }
    __syncthreads();
    for (int e = tid; e < M * (D / 4); e += 64 * WAVES) {
        const int col = e / (D / 4);
        const int d = 4 * (e - col * (D / 4));
        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < MERGE; w++) {
            acc += *reinterpret_cast<const f4*>(&sm_o[(w * 32 + col) * LDM + d]);
        }
        acc = scaled(acc, d);
        if (whole) {
            const int ho = col / r.Sq;
            *reinterpret_cast<h4*>(r.row(b, kvh * r.ratio + ho, col - ho * r.Sq) + d) = __builtin_convertvector(acc, h4);
        } else {
            *reinterpret_cast<f4*>(&r.part_o[(part + col) * D + d]) = acc;
        }
    }
}

// Partials of one row: split s has its O at part_o[s * so] and its (m, l) at
// part_ml[s * sml].
struct SplitParts {
    const float* part_o;
    const float* part_ml;
    int64_t so, sml;
    int splits, D;
};

// LDS of merge_splits: a weight per split and one f4 per thread.
constexpr int merge_lds_floats(int splits, int threads) {
    return splits + 4 * threads;
}

// Merges one row with the T threads of a workgroup (a multiple of 64, D <= 4
// T) and hands every 4 output columns to store(d, f4).  What bounds it is
// latency: first the weights, the lanes side by side over the splits (every
// wave for itself), then O, spread over groups of splits with four loads in
// flight per thread.  A loop over the splits per thread, three times over,
// took 9.9 us for 32 rows of 16 splits, D = 128.
template <int T, class Store>
__device__ __forceinline__ void merge_splits(const SplitParts& p, float* lds, Store&& store) {
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    float* const wgt = lds;                                  // [kMaxSplits]
    f4* const red = reinterpret_cast<f4*>(lds + kMaxSplits); // [T]
    constexpr int PER = kMaxSplits / 64;
    float m[PER], l[PER];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int s = lane + 64 * i;
        m[i] = -INFINITY;
        l[i] = 0.0f;
        if (s < p.splits) {
            const float2 v = *reinterpret_cast<const float2*>(p.part_ml + s * p.sml);
            m[i] = v.x;
            l[i] = v.y;
        }
        mx = fmaxf(mx, m[i]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        m[i] = part_weight(m[i], mx);
        sum += l[i] * m[i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off);
    }
    // NaN: 0, as a row sum that is not positive gives in the prefill kernels; O
    // is NaN where the row is
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        if (tid < 64 && lane + 64 * i < p.splits) {
            wgt[lane + 64 * i] = l[i] != 0.0f ? m[i] * inv : -1.0f;
        }
    }
    __syncthreads();
    const int E = p.D / 4;
    const int SG = T / E; // groups of splits side by side
    const int sg = tid / E;
    const int e = tid - sg * E;
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    // a split without a visible key (weight -1) adds nothing
    auto add = [&](f4 x, float w) { acc += w < 0.0f ? f4{0.0f, 0.0f, 0.0f, 0.0f} : x * w; };
    if (sg < SG) {
        const float* o = p.part_o + 4 * e;
        int s = sg;
        for (; s + 3 * SG < p.splits; s += 4 * SG) {
            f4 x[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                x[i] = *reinterpret_cast<const f4*>(o + (s + i * SG) * p.so);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                add(x[i], wgt[s + i * SG]);
            }
        }
        for (; s < p.splits; s += SG) {
            add(*reinterpret_cast<const f4*>(o + s * p.so), wgt[s]);
        }
    }
    if (SG > 1) {
        red[tid] = acc;
        __syncthreads();
        if (sg == 0) {
            for (int i = 1; i < SG && i < p.splits; i++) {
                acc += red[i * E + e];
            }
        }
    }
    if (sg == 0) {
        store(4 * e, acc);
    }
}

} // namespace rdna_amd
