// Merge of key splits, shared by the split-K kernels (device code).
//
// A split leaves, per query row, O unnormalised in fp32 and (m, l): its
// reference maximum in log2 units and its row sum relative to it.  The merged
// row is sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s with M the largest m_s
// of the splits that saw a key (l_s > 0).
#pragma once

#include "fa_common.hpp"

namespace rdna_amd {

constexpr int kMaxSplits = 256; // weights of one row in the merge's LDS

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
        mx = l[i] > 0.0f ? fmaxf(mx, m[i]) : mx;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, off));
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        m[i] = l[i] > 0.0f ? fast_exp2(m[i] - mx) : 0.0f;
        sum += l[i] * m[i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off);
    }
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        if (tid < 64 && lane + 64 * i < p.splits) {
            wgt[lane + 64 * i] = m[i] * inv;
        }
    }
    __syncthreads();
    const int E = p.D / 4;
    const int SG = T / E; // groups of splits side by side
    const int sg = tid / E;
    const int e = tid - sg * E;
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    // a split without a visible key (weight 0) adds nothing
    auto add = [&](f4 x, float w) { acc += w > 0.0f ? x * w : f4{0.0f, 0.0f, 0.0f, 0.0f}; };
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
