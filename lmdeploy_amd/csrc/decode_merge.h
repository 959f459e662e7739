// What the decode attention kernels share about key splits: how many a sequence uses and how their results are joined.
// The splits of a (sequence, key head) meet inside the launch (tm_common.h): a merge launch of its own took 4.4 ... 6.8 us a layer, the ticket, one trip to memory
// and the join 0.4 ... 1.4.  One Llama-3-8B-shaped sequence, 8 layers W4: 11.1 -> 10.2 ms for 16 tokens; 8 fp16 sequences, 12 layers 43.3 -> 42.0; Fokonex
// width 4096, 32 sequences 118 -> 113.5.
#pragma once
#include "tm_common.h"
#include "tm_kernels.h"
#include <algorithm>

namespace tmk {

// Least tiles of a split for a launch of `wgs` workgroups without splits: a workgroup's four waves take a tile each, so fewer than four to a split only pay
// while compute units are idle, below 256 workgroups.  (8 sequences of ~150 fp16 entries, 8 heads: the same within 0.5 % for one, two and four tiles, 2 %
// slower with eight.)
inline int decode_split_tiles(int wgs)
{
    return std::min(4, std::max(1, wgs / 64));
}

int launch_decode_reduce(const DecodeAttnParams& p, hipStream_t st);  // attention_decode.hip: nothing where the splits meet inside the launch

// Joins the results of nsplit key splits, (m, l) pairs at pm[s * 2] and C channels at *at(s, c), into (m, l, o) (scale: of the exponents to base 2).  All
// loads of N splits are in flight at once: one trip to memory, which is what the merge costs.
template<int N, int C, class At>
__device__ __forceinline__ void merge_splits(const float* pm, At&& at, int nsplit, float scale, float& m, float& l, float (&o)[C])
{
    for (int s0 = 0; s0 < nsplit; s0 += N) {
        float mv[N], lv[N], ov[N][C];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int s = min(s0 + i, nsplit - 1);
            mv[i]       = agent_load(pm + s * 2);
            lv[i]       = agent_load(pm + s * 2 + 1);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                ov[i][c] = agent_load(at(s, c));
            }
        }
        float mn = m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            mn = fmaxf(mn, mv[i]);
        }
        const float a0 = m == -INFINITY ? 0.f : fast_exp2((m - mn) * scale);
        l *= a0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            o[c] *= a0;
        }
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float a = s0 + i >= nsplit || mv[i] == -INFINITY ? 0.f : fast_exp2((mv[i] - mn) * scale);
            l = fmaf(a, lv[i], l);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                o[c] = fmaf(a, ov[i][c], o[c]);
            }
        }
        m = mn;
    }
}

// channel d of query head hq of sequence b from the results of its splits
__device__ __forceinline__ void decode_merge(const DecodeAttnParams& p, int b, int hq, int d, int nsplit)
{
    constexpr int D    = 128;
    const size_t  slot = ((size_t)b * p.q_heads + hq) * p.splits;
    float         m = -INFINITY, l = 0.f, o[1] = {0.f};
    merge_splits<8>(p.partial_ml + slot * 2, [&](int s, int) { return p.partial_o + (slot + s) * D + d; }, nsplit, p.scale_log2, m, l, o);
    p.out[(size_t)b * p.q_heads * D + (size_t)hq * D + d] = (half_t)(o[0] / l);
}

}  // namespace tmk
