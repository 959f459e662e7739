// Paged causal attention for arbitrary head sizes (key size `dim`, value size `vdim`, grouped query heads), bf16 or fp32 cache,
// with the score modifiers of recent decoder designs as PARAMETERS (GeneralAttnParams), each off at its neutral value:
//   * query temperature by position: score *= 1 + coef * ln(floor((p + 1) / every) + 1)          (coef = 0: off)
//   * soft cap:                      score  = cap * tanh(score / cap)                               (cap <= 0: off)
//   * attention sink:                the softmax denominator also holds exp(sink[head]): a learned logit with no key and no value,
//                                    neither scaled nor capped                                      (sink = nullptr: off)
//   * distance penalty:              score -= r1[head] * ln(1 + r2[head] * (p - key position))      (dist_r1 = nullptr: off)
//   * chunked visibility:            a row sees the keys of its own chunk of positions only:
//                                    key >= floor(p / chunk) * chunk, chunks counted from position 0   (chunk = 0: off)
//   * output gate:                   head h of row t is multiplied by sigmoid(out_gate[t][h])        (out_gate = nullptr: off)
//   * sliding window:                a row at position p sees key j <= p only if p - j < window or j < keep_first: the window plus
//                                    the first tokens of the sequence, at their true positions             (window = 0: off)
//   * distance table:                score += dist_table[head][min(p - key position, len - 1)]: a learned bias per distance (a bucketed
//                                    table is expanded per distance by the caller)                   (dist_table = nullptr: off)
//   * key / value head counts of their own: the query heads form kv_heads groups; group g reads key head g % k_heads and value head
//                                    g % v_heads (two score maps over one set of values; one wide key with a value head per group)
// Scores, soft-max weights and the output accumulation are fp32 whatever the cache holds; out_f32 keeps the output rows in fp32 too.
//
// One launch serves every row of a forward, prefill portions and decoded tokens alike: row t belongs to sequence row_seq[t] at
// position row_pos[t] and sees the cache entries 0 .. row_pos[t] of that sequence (its own key was stored before the launch).
//   * row kernel : one wave per (row, query head, key split); lanes own keys for the scores and value channels for the output.
//                  What the others do not serve: odd sizes, keys of more than 256 channels, other block lengths; in fp32 many rows of few keys and few heads a key head.
//   * tile kernel: bf16 prefill on the matrix cores -- 64 query rows of one sequence x one query head per workgroup, four waves of 16
//                  rows; S^T = K Q^T and O^T += V^T P^T as v_mfma_f32_16x16x32_bf16 with every operand a 16-byte load straight from the
//                  cache (keys [token][channel], values stored transposed [channel][token]); online soft-max in fp32; no LDS, no barrier.
//   * staged kernel: the tile kernel's products over cache blocks that a workgroup brings into LDS once (head sizes of 64 ... 256).
//   * decode kernel: the same products with the query HEADS of one key head as the 16 rows (one row per sequence): a workgroup per
//                  (sequence, key head, key split), its four waves take every fourth cache block and merge at the end.
//   * heads kernel : that in fp32, for decoded rows and for prompts; a wave takes sixteen keys of every block.
// Cache block layout per layer: keys [kv_heads][64][dim], then values [kv_heads][vdim][64].
#include "tm_kernels.h"
#include "decode_merge.h"
#include "gemm_stream.h"  // stream_dma16
#include <algorithm>
#include <stdlib.h>

#define TM_TRY_RC(expr)      \
    do {                     \
        int _rc = (expr);    \
        if (_rc) {           \
            return _rc;      \
        }                    \
    } while (0)

namespace tmk {

__device__ __forceinline__ float ga_wave_max(float v)
{
    return group_max<64>(v);
}
__device__ __forceinline__ float ga_wave_sum(float v)
{
    return group_sum<64>(v);
}

__device__ __forceinline__ float ga_query_temp(const GeneralAttnParams& p, int pos)
{
    if (p.qtemp_coef == 0.f) {
        return 1.f;
    }
    const float steps = (float)floor((double)(pos + 1) / (double)p.qtemp_every);
    return 1.f + p.qtemp_coef * logf(steps + 1.f);
}

__device__ __forceinline__ float ga_modify(const GeneralAttnParams& p, float dot, float qscale)
{
    float s = dot * qscale;
    if (p.softcap > 0.f) {
        s = p.softcap * tanhf(s / p.softcap);
    }
    return s;
}

template<class T>
__device__ __forceinline__ float ga_dot(const T* __restrict__ k, const float* __restrict__ q, int D)
{
    float acc = 0.f;
    if constexpr (sizeof(T) == 2) {
        if ((D & 7) == 0) {
#pragma unroll 8
            for (int d = 0; d < D; d += 8) {
                const bf16x8 v = *(const bf16x8*)(k + d);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    acc = fmaf((float)v[i], q[d + i], acc);
                }
            }
            return acc;
        }
    }
    else {
        if ((D & 3) == 0) {
#pragma unroll 8
            for (int d = 0; d < D; d += 4) {
                const floatx4 v = *(const floatx4*)(k + d);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc = fmaf(v[i], q[d + i], acc);
                }
            }
            return acc;
        }
    }
    for (int d = 0; d < D; ++d) {
        acc = fmaf((float)k[d], q[d], acc);
    }
    return acc;
}

constexpr int kGaMaxDim = 1024;  // key size limit of the row kernel (q in LDS); value size: 64 * VC, VC value channels per lane

// first key of the contiguous range a row sees (its chunk's first position, or the window's)
__device__ __forceinline__ int ga_first_key(const GeneralAttnParams& p, int pos)
{
    const int f = p.chunk > 0 ? pos / p.chunk * p.chunk : 0;
    return p.window > 0 ? max(f, pos - p.window + 1) : f;
}
// keys below that range stay visible while they are among the first ga_keep() positions.  The blocks a row visits are then the
// `nk` blocks that hold such keys and lie before the range's first block `bf`, followed by bf .. (last block): ga_block_at maps an index of
// that list to the block; key splits divide the list.
__device__ __forceinline__ int ga_keep(const GeneralAttnParams& p)
{
    return p.window > 0 ? p.keep_first : 0;
}
__device__ __forceinline__ int ga_keep_blocks(const GeneralAttnParams& p, int first, int bf, int block_len)
{
    return min(bf, (min(ga_keep(p), first) + block_len - 1) / block_len);
}
__device__ __forceinline__ int ga_block_at(int bi, int nk, int bf)
{
    return bi < nk ? bi : bf + (bi - nk);
}

// blocks of a key split of a row that visits nvis blocks, and the splits it needs then (at least one): the others leave at once, and a row of one split
// is finished by it
__device__ __forceinline__ int ga_split_len(const GeneralAttnParams& p, int nvis)
{
    return max((nvis + p.splits - 1) / p.splits, p.split_blocks);
}
__device__ __forceinline__ int ga_split_count(const GeneralAttnParams& p, int nvis)
{
    const int per = ga_split_len(p, nvis);
    return max((nvis + per - 1) / per, 1);
}

// where head h of an output row starts: heads side by side unless the caller spaces them (a batched product reads them at a stride)
__device__ __forceinline__ size_t ga_out_head(const GeneralAttnParams& p, int h)
{
    return (size_t)h * (p.out_head_stride > 0 ? p.out_head_stride : p.vdim);
}

__device__ __forceinline__ float ga_out_gate(const GeneralAttnParams& p, int t, int h)
{
    return p.out_gate ? 1.f / (1.f + expf(-p.out_gate[(size_t)t * p.ld_gate + h])) : 1.f;
}

// key / value head of a group of query heads
__device__ __forceinline__ int ga_key_head(const GeneralAttnParams& p, int g)
{
    return p.k_heads > 0 ? g % p.k_heads : g;
}
__device__ __forceinline__ int ga_value_head(const GeneralAttnParams& p, int g)
{
    return p.v_heads > 0 ? g % p.v_heads : g;
}

// channel v of head h of output row t
template<class T>
__device__ __forceinline__ void ga_store(const GeneralAttnParams& p, int t, int h, int v, float val)
{
    const size_t at = (size_t)t * p.ldo + ga_out_head(p, h) + v;
    if (p.out_f32) {
        ((float*)p.out)[at] = val;
    }
    else {
        ((T*)p.out)[at] = (T)val;
    }
}

// four channels from v on (the hardware stores 8 and 16 bytes at any element's address)
typedef float ga_floatx4_any __attribute__((ext_vector_type(4), aligned(4)));
template<class T>
__device__ __forceinline__ void ga_store4(const GeneralAttnParams& p, int t, int h, int v, floatx4 val)
{
    typedef T    T4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    const size_t at = (size_t)t * p.ldo + ga_out_head(p, h) + v;
    if (p.out_f32) {
        *(ga_floatx4_any*)((float*)p.out + at) = val;
    }
    else {
        *(T4*)((T*)p.out + at) = T4{(T)val[0], (T)val[1], (T)val[2], (T)val[3]};
    }
}

// C channels of head h of row t from the results of its key splits (+ the sink): channel(c), those below vdim
template<class T, int C, class Channel>
__device__ __forceinline__ void ga_merge(const GeneralAttnParams& p, int t, int h, int nsplit, Channel&& channel)
{
    const size_t slot = ((size_t)t * p.q_heads + h) * p.splits;
    float        m = p.sink ? p.sink[h] : -1e30f, l = p.sink ? 1.f : 0.f, o[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        o[c] = 0.f;
    }
    merge_splits<C <= 4 ? 8 : 2>(p.partial_ml + slot * 2, [&](int s, int c) { return p.partial_o + (slot + s) * p.vdim + min(channel(c), p.vdim - 1); },
                                 nsplit, 1.4426950408889634f, m, l, o);
    const float inv = ga_out_gate(p, t, h) / l;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if (channel(c) < p.vdim) {
            ga_store<T>(p, t, h, channel(c), o[c] * inv);
        }
    }
}
template<class T, int VC>
__device__ __forceinline__ void ga_merge_row(const GeneralAttnParams& p, int t, int h, int nsplit)  // all channels, by one wave
{
    ga_merge<T, VC>(p, t, h, nsplit, [](int c) { return (int)(threadIdx.x & 63) + 64 * c; });
}

// grid (rows, ceil(q_heads / 4), splits), 256 threads: wave w -> head blockIdx.y * 4 + w.  A chain of dependent loads bounds it at a few rows: eight pieces
// of a key and four keys of a value channel are in flight at a time (3 rows of 16 heads over ~190 latent entries in fp32: 55 us with one of each, 31 so)
template<class T, int VC>
__global__ __launch_bounds__(256) void attn_rows_kernel(GeneralAttnParams p)
{
    typedef T T4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    __shared__ float qs[4][kGaMaxDim];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x, h = blockIdx.y * 4 + wave, sp = blockIdx.z;
    if (h >= p.q_heads) {
        return;
    }
    const int D = p.dim, V = p.vdim;
    const int s = p.row_seq[t], pos = p.row_pos[t];
    const int g = h / (p.q_heads / p.kv_heads);
    const uint64_t* table = p.block_ptrs + (size_t)(p.seq_slot ? p.seq_slot[s] : s) * p.block_stride;
    const T* q = (const T*)p.q + (size_t)t * p.ldq + (size_t)h * D;
    for (int d = lane; d < D; d += 64) {
        qs[wave][d] = (float)q[d];
    }
    const float qscale = p.scale * ga_query_temp(p, pos);
    const int   nkeys = pos + 1, nblk = (nkeys + p.block_len - 1) / p.block_len;
    const int   first = ga_first_key(p, pos), bf = first / p.block_len;  // the first key of the visible range and its block
    const int   keep = ga_keep(p), nk = ga_keep_blocks(p, first, bf, p.block_len), nvis = nk + nblk - bf;
    const int   per = ga_split_len(p, nvis), nsplit = ga_split_count(p, nvis);
    const int   i0 = sp * per, i1 = min(nvis, i0 + per);
    if (sp >= nsplit) {
        return;
    }
    const float r1 = p.dist_r1 ? p.dist_r1[h] : 0.f, r2 = p.dist_r1 ? p.dist_r2[h] : 0.f;
    float m = -1e30f, l = 0.f, o[VC];
#pragma unroll
    for (int c = 0; c < VC; ++c) {
        o[c] = 0.f;
    }
    // LDS writes of this wave are read by this wave only: a wave barrier is enough
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int bi = i0; bi < i1; ++bi) {
        const int   b    = ga_block_at(bi, nk, bf);
        const char* base = global_ptr(table[b]) + p.layer_offset;
        const T*    kb   = (const T*)base + (size_t)ga_key_head(p, g) * p.block_len * D;
        const T*    vb   = (const T*)(base + p.v_offset) + (size_t)ga_value_head(p, g) * p.block_len * V;  // [V][block_len]
        const int   n    = min(p.block_len, nkeys - b * p.block_len);
        const int   jlo  = first - b * p.block_len;  // keys below it lie in an earlier chunk / before the window ...
        const int   klo  = keep - b * p.block_len;   // ... and are seen only as kept first tokens: j < klo
        for (int j0 = klo > 0 ? 0 : max(0, jlo) / 64 * 64; j0 < n; j0 += 64) {
            const int  j     = j0 + lane;
            const bool valid = j < n && (j >= jlo || j < klo);
            float      sc    = -1e30f;
            if (valid) {
                sc = ga_modify(p, ga_dot<T>(kb + (size_t)j * D, qs[wave], D), qscale);
                if (p.dist_r1) {
                    sc -= r1 * log1pf(r2 * (float)(pos - (b * p.block_len + j)));
                }
                if (p.dist_table) {
                    sc += p.dist_table[(size_t)h * p.dist_table_len + min(pos - (b * p.block_len + j), p.dist_table_len - 1)];
                }
            }
            const float m_new = fmaxf(m, ga_wave_max(sc));
            const float alpha = __expf(m - m_new);
            const float pj    = valid ? __expf(sc - m_new) : 0.f;
            l                 = l * alpha + ga_wave_sum(pj);
            m                 = m_new;
#pragma unroll
            for (int c = 0; c < VC; ++c) {
                o[c] *= alpha;
            }
            const int cnt = min(64, n - j0);
            auto      wt  = [&](int jj) { return bit_cast<float>(__builtin_amdgcn_readlane(bit_cast<int>(pj), jj)); };
            auto      one = [&](int jj) {
                const float w  = wt(jj);
                const T*    vr = vb + (j0 + jj);
#pragma unroll
                for (int c = 0; c < VC; ++c) {
                    const int v = lane + 64 * c;
                    if (v < V) {
                        o[c] = fmaf(w, (float)vr[(size_t)v * p.block_len], o[c]);
                    }
                }
            };
            int jj = klo > 0 ? 0 : max(0, jlo - j0);
            for (; jj < cnt && (jj & 3); ++jj) {
                one(jj);
            }
#pragma unroll 2
            for (; jj + 4 <= cnt; jj += 4) {  // four keys of a channel a load
                const float w0 = wt(jj), w1 = wt(jj + 1), w2 = wt(jj + 2), w3 = wt(jj + 3);
                const T*    vr = vb + (j0 + jj);
#pragma unroll
                for (int c = 0; c < VC; ++c) {
                    const int v = lane + 64 * c;
                    if (v < V) {
                        const T4 x = *(const T4*)(vr + (size_t)v * p.block_len);
                        o[c]       = fmaf(w3, (float)x[3], fmaf(w2, (float)x[2], fmaf(w1, (float)x[1], fmaf(w0, (float)x[0], o[c]))));
                    }
                }
            }
            for (; jj < cnt; ++jj) {
                one(jj);
            }
        }
    }
    if (nsplit == 1) {
        float inv;
        if (p.sink) {
            const float sk = p.sink[h], mf = fmaxf(m, sk), a = __expf(m - mf);
            inv            = a / (l * a + __expf(sk - mf));
        }
        else {
            inv = 1.f / l;
        }
        inv *= ga_out_gate(p, t, h);
#pragma unroll
        for (int c = 0; c < VC; ++c) {
            const int v = lane + 64 * c;
            if (v < V) {
                ga_store<T>(p, t, h, v, o[c] * inv);
            }
        }
        return;
    }
    float* po = p.partial_o + (((size_t)t * p.q_heads + h) * p.splits + sp) * V;
    float* pm = p.partial_ml + (((size_t)t * p.q_heads + h) * p.splits + sp) * 2;
#pragma unroll
    for (int c = 0; c < VC; ++c) {
        const int v = lane + 64 * c;
        if (v < V) {
            agent_store(po + v, o[c]);
        }
    }
    if (lane == 0) {
        agent_store(pm, m);
        agent_store(pm + 1, l);
    }
    if (p.tickets && ticket_last_wave(p.tickets + (size_t)t * p.q_heads + h, nsplit)) {
        ga_merge_row<T, VC>(p, t, h, nsplit);
    }
}

// merge of the key splits as a launch of its own, for callers without tickets: grid (rows, q_heads), 64 threads
template<class T, int VC>
__global__ __launch_bounds__(64) void attn_rows_merge_kernel(GeneralAttnParams p)
{
    const int pos = p.row_pos[blockIdx.x], first = ga_first_key(p, pos), bf = first / p.block_len;
    const int nsplit = ga_split_count(p, ga_keep_blocks(p, first, bf, p.block_len) + (pos + p.block_len) / p.block_len - bf);
    if (nsplit > 1) {
        ga_merge_row<T, VC>(p, blockIdx.x, blockIdx.y, nsplit);
    }
}

template<class T>
static void launch_rows_merge(const GeneralAttnParams& p, hipStream_t st)
{
    if (p.vdim <= 256) {
        attn_rows_merge_kernel<T, 4><<<dim3(p.rows, p.q_heads), 64, 0, st>>>(p);
    }
    else {
        attn_rows_merge_kernel<T, 16><<<dim3(p.rows, p.q_heads), 64, 0, st>>>(p);
    }
}

template<class T>
static void launch_rows(const GeneralAttnParams& p, dim3 grid, hipStream_t st)
{
    if (p.vdim <= 256) {
        attn_rows_kernel<T, 4><<<grid, 256, 0, st>>>(p);
    }
    else {
        attn_rows_kernel<T, 16><<<grid, 256, 0, st>>>(p);
    }
}

size_t general_attention_workspace_bytes(int rows, int q_heads, int vdim, int splits)
{
    return (size_t)rows * q_heads * splits * (vdim + 2) * sizeof(float);
}

static unsigned* ga_tickets(const GeneralAttnParams& p)  // one per (row, head), or the splits' results are merged by a launch of their own
{
    return p.ticket_count >= p.rows * p.q_heads ? p.tickets : nullptr;
}

int launch_general_attention_rows(const GeneralAttnParams& p_in, hipStream_t st)
{
    GeneralAttnParams p = p_in;
    p.tickets           = ga_tickets(p_in);
    TM_REQUIRE(p.rows >= 0 && p.q_heads >= 1 && p.kv_heads >= 1 && p.q_heads % p.kv_heads == 0, "attention: head counts");
    TM_REQUIRE(p.dim >= 1 && p.dim <= kGaMaxDim && p.vdim >= 1 && p.vdim <= kGaMaxDim, "attention: 1 <= dim, vdim <= 1024");
    TM_REQUIRE(p.chunk >= 0 && (!p.dist_r1 || p.dist_r2) && (!p.out_gate || p.ld_gate >= p.q_heads), "attention: chunk / distance penalty / gate");
    TM_REQUIRE(p.window >= 0 && p.keep_first >= 0, "attention: window / kept first tokens");
    TM_REQUIRE(p.k_heads >= 0 && p.v_heads >= 0 && (!p.dist_table || p.dist_table_len >= 1), "attention: key / value head counts, distance table");
    TM_REQUIRE(p.block_len >= 1 && p.splits >= 1 && (p.splits == 1 || (p.partial_o && p.partial_ml)), "attention: splits / workspace");
    TM_REQUIRE(p.elem_bytes == 2 || p.elem_bytes == 4, "attention: bf16 or fp32");
    TM_REQUIRE(p.qtemp_coef == 0.f || p.qtemp_every > 0.f, "attention: query temperature period");
    if (p.rows == 0) {
        return 0;
    }
    const dim3 grid(p.rows, (p.q_heads + 3) / 4, p.splits);
    if (p.elem_bytes == 2) {
        launch_rows<__bf16>(p, grid, st);
    }
    else {
        launch_rows<float>(p, grid, st);
    }
    TM_HIP_CHECK(hipGetLastError());
    if (p.splits > 1 && !p.tickets) {
        if (p.elem_bytes == 2) {
            launch_rows_merge<__bf16>(p, st);
        }
        else {
            launch_rows_merge<float>(p, st);
        }
        TM_HIP_CHECK(hipGetLastError());
    }
    return 0;
}


// ---- matrix-core kernels (bf16) -------------------------------------------------------------------------------------------------------
// Per 64-key cache block a wave computes the TRANSPOSED scores S^T = K Q^T as four 16-key tiles (A = key rows, B = query rows; one
// 16-byte load per lane and 32 channels), so that a lane ends up with 16 scores of ONE query row (row = lane % 16): the soft-max
// statistics are per-lane scalars (two shuffles join the four lane groups) and the exponentiated accumulators ARE the B operand of
// O^T += V^T P^T.  Which 16 keys form a tile is free: tile kt, A-row i is key (kt / 2) * 32 + (i / 4) * 8 + (kt % 2) * 4 + i % 4, which
// leaves lane group lg with the EIGHT CONSECUTIVE keys ks * 32 + lg * 8 .. + 8 of k-step ks in its two tiles -- the A operand of the
// second product is then one 16-byte load from the transposed values.  No score or probability ever goes through memory.
constexpr int   kTileRows = 64;
constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;

__device__ __forceinline__ float ga_tanh_fast(float x)
{
    // 1 - 2 / (exp(2x) + 1): absolute error ~1e-7, exact limits at +-inf
    return 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f);
}

// one 64-key block for RT tiles of 16 query rows (the lane's row of tile rt is rt * 16 + lane % 16): updates (m, l, o) of those rows.
// Every key / value fragment is loaded ONCE and serves all RT row tiles; the value fragments are requested before the soft-max
// arithmetic so that their latency hides under it.  qf: the rows' query fragments; limit: last visible key of the lane's rows
// (block-relative; < 0: none); kb / vb: the key head's keys [64][D] and transposed values [V][64] of this block.
// lower: first key of the visible range of the lane's rows (block-relative, may be negative); keys below it are seen while < keep_rel
// (the kept first tokens, block-relative; <= 0: none); r1 / r2: the distance penalty of the lane's rows' head
// (r1 * log2(1 + r2 * (limit - key)) leaves the score, which lives in the log2 domain; bias = false: none); tab: the distance table's row
// of the lane's rows' head (nullptr: none)
template<int DS, int VT, int RT, bool MASK>
__device__ __forceinline__ void ga_block_step(const bf16x8 (&qf)[RT][DS], const __bf16* __restrict__ kb, const __bf16* __restrict__ vb, int D,
                                              int V, const int (&limit)[RT], const int (&lower)[RT], int keep_rel, const float (&qscale)[RT], float cap,
                                              float inv_cap, bool bias, float r1, float r2, float (&m)[RT], float (&l)[RT],
                                              floatx4 (&o)[RT][VT], const float* __restrict__ tab = nullptr, int tab_len = 0)
{
    const int    lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    floatx4      sc[RT][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sc[rt][kt] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const __bf16* kr = kb + (size_t)((kt >> 1) * 32 + (lr >> 2) * 8 + (kt & 1) * 4 + (lr & 3)) * D;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const int    d  = ds * 32 + lg * 8;
            const bf16x8 kf = d < D ? *(const bf16x8*)(kr + d) : zero8;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                sc[rt][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[rt][ds], sc[rt][kt], 0, 0, 0);
            }
        }
    }
    bf16x8 vf[VT][2];
#pragma unroll
    for (int t = 0; t < VT; ++t) {
        const int v = t * 16 + lr;
        const __bf16* vr = vb + (size_t)v * 64 + lg * 8;
        vf[t][0]         = v < V ? *(const bf16x8*)(vr) : zero8;
        vf[t][1]         = v < V ? *(const bf16x8*)(vr + 32) : zero8;
    }
    // lane holds S[row lr of tile rt][key (kt / 2) * 32 + lg * 8 + (kt % 2) * 4 + r].  From here on scores live in the log2 domain
    // (multiplied by log2 e) so that every exponential is one v_exp_f32: the capped score is
    //   cap2 * tanh(x / cap) = cap2 - 2 cap2 / (2^(x * 2 log2e / cap) + 1),  cap2 = cap * log2e
    // -- five VALU operations, two of them transcendental; the kernel is bound by exactly this arithmetic.
    bf16x8 pf[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float cap2 = cap * kLog2e, k1 = cap > 0.f ? qscale[rt] * inv_cap * (2.f * kLog2e) : qscale[rt] * kLog2e;
        float       bmax = -1e30f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = sc[rt][kt][r] * k1;
                if (cap > 0.f) {
                    v = fmaf(__builtin_amdgcn_rcpf(fast_exp2(v) + 1.f), -2.f * cap2, cap2);
                }
                const int key = (kt >> 1) * 32 + lg * 8 + (kt & 1) * 4 + r;
                if (bias) {  // (a key ahead of the row gives the logarithm of a number that may be negative: the mask below discards it)
                    v = fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, (float)(limit[rt] - key), 1.f)), v);
                }
                if (tab) {  // the lane's head's row of the distance table (a key ahead of the row reads entry 0 and is masked below)
                    v = fmaf(tab[min(max(limit[rt] - key, 0), tab_len - 1)], kLog2e, v);
                }
                if (MASK) {
                    v = (key <= limit[rt] && (key >= lower[rt] || key < keep_rel)) ? v : -1e30f;
                }
                sc[rt][kt][r] = v;
                bmax          = fmaxf(bmax, v);
            }
        }
        bmax = fmaxf(bmax, __shfl_xor(bmax, 16));
        bmax = fmaxf(bmax, __shfl_xor(bmax, 32));
        const float m_new = fmaxf(m[rt], bmax);
        const float alpha = fast_exp2(m[rt] - m_new);
        const float m_ref = fmaxf(m_new, -1e29f);  // a row that has seen no key yet (its chunk starts behind this block): every weight is 0
        float       bsum  = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = fast_exp2(sc[rt][kt][r] - m_ref);  // a masked score is -1e30: 2^(-1e30 - m) = 0
                bsum += e;
                pf[rt][kt >> 1][(kt & 1) * 4 + r] = (__bf16)e;
            }
        }
        bsum += __shfl_xor(bsum, 16);
        bsum += __shfl_xor(bsum, 32);
        l[rt] = l[rt] * alpha + bsum;
        m[rt] = m_new;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            o[rt][t] *= alpha;
        }
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                o[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[t][ks], pf[rt][ks], o[rt][t], 0, 0, 0);
            }
        }
    }
}

// Prefill: workgroup = 64 * RT query rows of one sequence x one query head, four independent waves of RT tiles of 16 rows.
template<int DS /* 32-channel steps of the key size */, int VT /* 16-channel tiles of the value size */, int RT>
__global__ __launch_bounds__(256) void attn_tiles_kernel(GeneralAttnParams p, int tiles_per_seq)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int s = blockIdx.x / tiles_per_seq, ti = blockIdx.x % tiles_per_seq, h = blockIdx.y;
    const int row_base = p.cu_q[s] - p.cu_q[0];
    const int q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int row0  = ti * (kTileRows * RT) + wave * (16 * RT);  // the wave's first row inside the sequence's portion
    if (row0 >= q_len) {
        return;
    }
    const int D = p.dim, V = p.vdim;
    const int g = h / (p.q_heads / p.kv_heads);
    const int pos0 = p.k_len[s] - q_len;  // position of the sequence's first row in this launch
    const int lr = lane & 15, lg = lane >> 4;
    const uint64_t* table = p.block_ptrs + (size_t)(p.seq_slot ? p.seq_slot[s] : s) * p.block_stride;
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const float cap = p.softcap, inv_cap = cap > 0.f ? 1.f / cap : 0.f;
    bf16x8  qf[RT][DS];  // B operand of S^T: row = lane % 16, channels ds * 32 + (lane / 16) * 8 .. + 8
    float   qscale[RT], m[RT], l[RT];
    int     pos[RT], first[RT];
    const bool  bias = p.dist_r1 != nullptr;
    const float r1 = bias ? p.dist_r1[h] : 0.f, r2 = bias ? p.dist_r2[h] : 0.f;
    const float* tab = p.dist_table ? p.dist_table + (size_t)h * p.dist_table_len : nullptr;
    bool    q_ok[RT];
    floatx4 o[RT][VT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int qi = row0 + rt * 16 + lr;
        q_ok[rt]     = qi < q_len;
        pos[rt]      = pos0 + qi;
        first[rt]    = ga_first_key(p, pos[rt]);
        const __bf16* q = (const __bf16*)p.q + (size_t)(row_base + (q_ok[rt] ? qi : 0)) * p.ldq + (size_t)h * D;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const int    d  = ds * 32 + lg * 8;
            const bf16x8 ql = *(const bf16x8*)(q + min(d, D - 8));
            qf[rt][ds]      = (q_ok[rt] && d < D) ? ql : zero8;
        }
        qscale[rt] = p.scale * ga_query_temp(p, pos[rt]);
        m[rt]      = -1e30f;
        l[rt]      = 0.f;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            o[rt][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const int last_pos = pos0 + min(q_len, row0 + 16 * RT) - 1;  // the wave's last row sees keys 0 .. last_pos
    const int nblk     = last_pos / 64 + 1;
    const int first_lo = ga_first_key(p, pos0 + row0), first_hi = ga_first_key(p, last_pos);  // of the wave's first and last row
    const int keep = ga_keep(p), bf = first_lo / 64, nk = ga_keep_blocks(p, first_lo, bf, 64);
    for (int bi = 0; bi < nk + nblk - bf; ++bi) {
        const int   b    = ga_block_at(bi, nk, bf);
        const char* base = global_ptr(table[b]) + p.layer_offset;
        int         limit[RT], lower[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            limit[rt] = q_ok[rt] ? pos[rt] - b * 64 : -1;
            lower[rt] = first[rt] - b * 64;
        }
        const __bf16 *kb = (const __bf16*)base + (size_t)ga_key_head(p, g) * 64 * D;
        const __bf16 *vb = (const __bf16*)(base + p.v_offset) + (size_t)ga_value_head(p, g) * 64 * V;
        // every row of the wave sees the whole block (rows beyond the portion are discarded anyway)
        if (b * 64 + 63 <= pos0 + row0 && b * 64 >= first_hi) {
            ga_block_step<DS, VT, RT, false>(qf, kb, vb, D, V, limit, lower, 0, qscale, cap, inv_cap, bias, r1, r2, m, l, o, tab, p.dist_table_len);
        }
        else {
            ga_block_step<DS, VT, RT, true>(qf, kb, vb, D, V, limit, lower, keep - b * 64, qscale, cap, inv_cap, bias, r1, r2, m, l, o, tab,
                                                   p.dist_table_len);
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (!q_ok[rt]) {
            continue;
        }
        float inv;
        if (p.sink) {  // m is in the log2 domain
            const float sk = p.sink[h] * kLog2e, mf = fmaxf(m[rt], sk), a = fast_exp2(m[rt] - mf);
            inv            = a / (l[rt] * a + fast_exp2(sk - mf));
        }
        else {
            inv = 1.f / l[rt];
        }
        inv *= ga_out_gate(p, row_base + row0 + rt * 16 + lr, h);
        // lane holds O[row lr][channels t * 16 + lg * 4 .. + 3] (V is a multiple of 8)
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            const int v = t * 16 + lg * 4;
            if (v < V) {
                ga_store4<__bf16>(p, row_base + row0 + rt * 16 + lr, h, v, o[rt][t] * inv);
            }
        }
    }
}

// The end of a kernel whose four waves hold, for the 16 heads from h0 on (nh of them exist) of row t, sums over different keys: lane (lr, lg) the channels
// 16 v + 4 lg .. + 3 of head h0 + lr, maximum and sum in the e^x domain.  Common maximum, rescaled sums, then the row's output or a split's results; the
// last split to arrive merges them
template<class T, int VT>
__device__ __forceinline__ void ga_close_heads(const GeneralAttnParams& p, int t, int sp, int nsplit, int h0, int nh, float m, float l, floatx4 (&o)[VT],
                                               float (&ml_s)[4][16][2], float (&o_s)[3][16][VT * 16 + 4], unsigned* last_s)
{
    const int  lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4, V = p.vdim;
    const bool h_ok = lr < nh;
    const int  h    = h0 + (h_ok ? lr : 0);
    const size_t slots  = (size_t)p.q_heads * p.splits;  // of row t
    const auto   row_o  = agent_base(p.partial_o + t * slots * V, slots * V * 4);
    const auto   row_ml = agent_base(p.partial_ml + t * slots * 2, slots * 8);
    if (lg == 0) {
        ml_s[wave][lr][0] = m;
        ml_s[wave][lr][1] = l;
    }
    __syncthreads();
    const float mf = fmaxf(fmaxf(ml_s[0][lr][0], ml_s[1][lr][0]), fmaxf(ml_s[2][lr][0], ml_s[3][lr][0]));
    const float a  = __expf(m - mf);
    if (wave > 0) {
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            *(floatx4*)&o_s[wave - 1][lr][v * 16 + lg * 4] = o[v] * a;
        }
    }
    __syncthreads();
    if (wave > 0) {
        if (nsplit == 1 || !p.tickets) {
            return;
        }
    }
    else {
        float lt = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            lt += ml_s[w][lr][1] * __expf(ml_s[w][lr][0] - mf);
        }
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            const int c = v * 16 + lg * 4;
            o[v]        = o[v] * a + ((*(const floatx4*)&o_s[0][lr][c] + *(const floatx4*)&o_s[1][lr][c]) + *(const floatx4*)&o_s[2][lr][c]);
        }
        if (nsplit == 1) {
            float inv;
            if (p.sink) {
                const float sk = p.sink[h], m2 = fmaxf(mf, sk), a2 = __expf(mf - m2);
                inv            = a2 / (lt * a2 + __expf(sk - m2));
            }
            else {
                inv = 1.f / lt;
            }
            inv *= ga_out_gate(p, t, h);
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const int c = v * 16 + lg * 4;
                if (h_ok && c < V) {
                    ga_store4<T>(p, t, h, c, o[v] * inv);
                }
            }
            return;
        }
        float* pm = p.partial_ml + (((size_t)t * p.q_heads + h) * p.splits + sp) * 2;
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            const int c = v * 16 + lg * 4;
            if (h_ok && c < V) {
                agent_store4(row_o, ((h * p.splits + sp) * V + c) * 4, o[v]);
            }
        }
        if (h_ok && lg == 0) {
            agent_store(pm, mf);
            agent_store(pm + 1, lt);
        }
    }
    if (p.tickets && ticket_last_workgroup(p.tickets + (size_t)t * p.q_heads + h0, nsplit, last_s)) {
        // The join of the splits (ga_merge), four channels a piece: everything that several splits have for all of a thread's pieces is asked for together.  Piece
        // by piece, and a channel at a time, 16 heads of 192 took three trips to memory: three fp32 rows over ~180 entries, 21.0 us then, 14.1 now
        constexpr int kPieces = (VT * 64 + 255) / 256, kSplits = kPieces <= 2 ? 8 : 4;
        const int     pieces = V / 4, n = nh * pieces;
        if ((int)threadIdx.x >= n) {
            return;
        }
        int     head[kPieces], c0[kPieces];
        float   mm[kPieces], ll[kPieces];
        floatx4 oo[kPieces];
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int at = min((int)threadIdx.x + i * 256, n - 1);
            head[i] = h0 + at / pieces, c0[i] = at % pieces * 4;
            mm[i] = p.sink ? p.sink[head[i]] : -1e30f, ll[i] = p.sink ? 1.f : 0.f;
            oo[i] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        for (int s0 = 0; s0 < nsplit; s0 += kSplits) {
            floatx2 ml[kPieces][kSplits];
            floatx4 ov[kPieces][kSplits];
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                if (i * 256 < n) {
#pragma unroll
                    for (int k = 0; k < kSplits; ++k) {
                        const int slot = head[i] * p.splits + min(s0 + k, nsplit - 1);
                        ml[i][k]       = agent_load2(row_ml, slot * 8);
                        ov[i][k]       = agent_load4(row_o, (slot * V + c0[i]) * 4);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                if (i * 256 < n) {
                    float mn = mm[i];
#pragma unroll
                    for (int k = 0; k < kSplits; ++k) {
                        mn = fmaxf(mn, ml[i][k][0]);
                    }
                    const float a0 = fast_exp2((mm[i] - mn) * kLog2e);
                    ll[i] *= a0;
                    oo[i] *= a0;
#pragma unroll
                    for (int k = 0; k < kSplits; ++k) {
                        const float ak = s0 + k < nsplit ? fast_exp2((ml[i][k][0] - mn) * kLog2e) : 0.f;
                        ll[i]          = fmaf(ak, ml[i][k][1], ll[i]);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            oo[i][c] = fmaf(ak, ov[i][k][c], oo[i][c]);
                        }
                    }
                    mm[i] = mn;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            if ((int)threadIdx.x + i * 256 < n) {
                ga_store4<T>(p, t, head[i], c0[i], oo[i] * (ga_out_gate(p, t, head[i]) / ll[i]));
            }
        }
    }
}

// Decode: grid (sequences, kv_heads * head chunks, splits).  The 16 rows are query heads g * group + chunk * 16 + (lane % 16) of row t;
// wave w takes the blocks b0 + w, b0 + w + 4, ... of the split; waves 1..3 hand their (m, l, O) to wave 0 through LDS.
template<int DS, int VT>
__global__ __launch_bounds__(256, VT <= 8 && DS * 16 + VT * 8 <= 128 ? 2 : 1) void attn_decode_kernel(GeneralAttnParams p, int chunks)
{
    __shared__ float    ml_s[4][16][2];
    __shared__ unsigned last_s;
    __shared__ float o_s[3][16][VT * 16 + 4];  // + 4: the sixteen rows start in different banks
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
    const int t = blockIdx.x, g = blockIdx.y / chunks, chunk = blockIdx.y % chunks, sp = blockIdx.z;
    const int D = p.dim, V = p.vdim, group = p.q_heads / p.kv_heads, h0 = g * group + chunk * 16, nh = min(16, group - chunk * 16);
    const int h = h0 + min(lr, nh - 1);  // (rows without a head repeat the last one's; they are not stored)
    const int s = p.row_seq[t], pos = p.row_pos[t];
    const uint64_t* table = p.block_ptrs + (size_t)(p.seq_slot ? p.seq_slot[s] : s) * p.block_stride;
    const int first = ga_first_key(p, pos), bf = first / 64;
    const int keep = ga_keep(p), nk = ga_keep_blocks(p, first, bf, 64);
    const int nvis = nk + pos / 64 + 1 - bf, per = ga_split_len(p, nvis), nsplit = ga_split_count(p, nvis);
    const int i1 = min(nvis, sp * per + per);
    if (sp >= nsplit) {
        return;
    }
    // A wave has one or two blocks, so latency is everything: all keys of a block are asked for at once, then all values, with unconditional addresses.  Left to
    // itself the compiler waits for each key fragment of 256 channels before it asks for the next, 32 trips to memory in a row; hence the barriers to its
    // scheduling and, for sizes that keys and values together do not fit in the registers, values that follow the first half of the products.  us, before / with it:
    // 4 rows of 16 / 1 heads of 256 / 192 over ~2040 entries 34.6 / 26.2, 32 rows of 32 / 8 heads of 128 over ~150 10.1 / 9.2
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const bool   tail  = D < DS * 32;  // channels that do not exist: zero on both sides
    const __bf16* const q = (const __bf16*)p.q + (size_t)t * p.ldq + (size_t)h * D;
    bf16x8       qf[DS], kf[4][DS], vf[VT][2];
    floatx4      o[VT];
    const __bf16 *kb = nullptr, *vb = nullptr;
    auto         load_keys = [&](int bi) {
        const char* base = global_ptr(table[ga_block_at(bi, nk, bf)]) + p.layer_offset;
        kb               = (const __bf16*)base + (size_t)ga_key_head(p, g) * 64 * D;
        vb               = (const __bf16*)(base + p.v_offset) + (size_t)ga_value_head(p, g) * 64 * V;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const uint32_t row = ((kt >> 1) * 32 + (lr >> 2) * 8 + (kt & 1) * 4 + (lr & 3)) * D;
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                kf[kt][ds] = *(const bf16x8*)(kb + row + (uint32_t)min(ds * 32 + lg * 8, D - 8));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_values = [&](int t0, int t1) {
#pragma unroll
        for (int v = t0; v < t1; ++v) {
            const uint32_t row = min(v * 16 + lr, V - 1) * 64 + lg * 8;  // (channels behind the last are not stored)
            vf[v][0]           = *(const bf16x8*)(vb + row);
            vf[v][1]           = *(const bf16x8*)(vb + row + 32);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
        qf[ds] = *(const bf16x8*)(q + min(ds * 32 + lg * 8, D - 8));
    }
#pragma unroll
    for (int v = 0; v < VT; ++v) {
        o[v] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    float m = -1e30f, l = 0.f;
    int   bi = sp * per + wave;
    if (bi < i1) {
        load_keys(bi);
        const float qscale = p.scale * ga_query_temp(p, pos), cap = p.softcap, cap2 = cap * kLog2e;
        const float k1     = cap > 0.f ? qscale / cap * (2.f * kLog2e) : qscale * kLog2e;  // (scores in the log2 domain, as in ga_block_step)
        const bool  bias   = p.dist_r1 != nullptr;
        const float r1 = bias ? p.dist_r1[h] : 0.f, r2 = bias ? p.dist_r2[h] : 0.f;  // of the lane's head
        const float* tab = p.dist_table + (size_t)h * p.dist_table_len;
        if (tail) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
                qf[ds] = ds * 32 + lg * 8 < D ? qf[ds] : zero8;
            }
        }
        for (;;) {
            const int b = ga_block_at(bi, nk, bf), limit = pos - b * 64, lower = first - b * 64, klo = keep - b * 64;
            floatx4   sc[4];
            constexpr int kEarly = DS * 16 + VT * 8 <= 128 ? VT : VT / 2;  // value tiles beside all keys
            if constexpr (DS * 16 + VT * 8 <= 128) {
                load_values(0, VT);
            }
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                if (tail) {
#pragma unroll
                    for (int ds = 0; ds < DS; ++ds) {
                        kf[kt][ds] = ds * 32 + lg * 8 < D ? kf[kt][ds] : zero8;
                    }
                }
                sc[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < DS; ++ds) {
                    sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt][ds], qf[ds], sc[kt], 0, 0, 0);
                }
                if constexpr (DS * 16 + VT * 8 > 128) {
                    if (kt == 1) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_values(0, kEarly);
                    }
                    if (kt == 3) {
                        __builtin_amdgcn_sched_barrier(0);
                        load_values(kEarly, VT);
                    }
                }
            }
            // lane: head lr, keys (kt / 2) * 32 + lg * 8 + (kt % 2) * 4 + r
            float add[4][4] = {};
            if (p.dist_table) {  // the lane's head's row of the distance table (a key ahead of the row reads entry 0 and is masked below)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key      = (i >> 3) * 32 + lg * 8 + (i & 7);
                    add[i >> 2][i & 3] = tab[min(max(limit - key, 0), p.dist_table_len - 1)];
                }
            }
            float bmax = -1e30f;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = sc[kt][r] * k1;
                    if (cap > 0.f) {
                        v = fmaf(__builtin_amdgcn_rcpf(fast_exp2(v) + 1.f), -2.f * cap2, cap2);
                    }
                    const int key = (kt >> 1) * 32 + lg * 8 + (kt & 1) * 4 + r;
                    if (bias) {  // (a key ahead of the row gives the logarithm of a number that may be negative: the mask below discards it)
                        v = fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, (float)(limit - key), 1.f)), v);
                    }
                    if (p.dist_table) {
                        v = fmaf(add[kt][r], kLog2e, v);
                    }
                    sc[kt][r] = key <= limit && (key >= lower || key < klo) ? v : -1e30f;
                    bmax      = fmaxf(bmax, sc[kt][r]);
                }
            }
            bmax              = fmaxf(bmax, __shfl_xor(bmax, 16));
            bmax              = fmaxf(bmax, __shfl_xor(bmax, 32));
            const float m_new = fmaxf(m, bmax), alpha = fast_exp2(m - m_new);
            const float m_ref = fmaxf(m_new, -1e29f);  // no key seen yet: every weight is 0
            float       bsum  = 0.f;
            bf16x8      pf[2];
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = fast_exp2(sc[kt][r] - m_ref);  // a masked score is -1e30: 2^(-1e30 - m) = 0
                    bsum += e;
                    pf[kt >> 1][(kt & 1) * 4 + r] = (__bf16)e;
                }
            }
            bsum += __shfl_xor(bsum, 16);
            bsum += __shfl_xor(bsum, 32);
            l = l * alpha + bsum;
            m = m_new;
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                o[v] *= alpha;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    o[v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[v][ks], pf[ks], o[v], 0, 0, 0);
                }
            }
            bi += 4;
            if (bi >= i1) {
                break;
            }
            load_keys(bi);
        }
    }
    // (back from the log2 domain: the merges use e^x)
    ga_close_heads<__bf16, VT>(p, t, sp, nsplit, h0, nh, m * kLn2, l, o, ml_s, o_s, &last_s);
}

bool general_attention_tiles_ok(const GeneralAttnParams& p)
{
    return p.elem_bytes == 2 && p.block_len == 64 && p.dim % 8 == 0 && p.vdim % 8 == 0 && p.dim <= 256 && p.vdim <= 256 && p.ldq % 8 == 0
           && p.cu_q && p.k_len && p.nseq >= 1 && p.max_q_len >= 1 && p.splits == 1 && p.q_heads % p.kv_heads == 0;
}

// ---- prefill over staged blocks -------------------------------------------------------------------------------------------------------
// Workgroup = W waves of RT tiles of 16 query rows of one sequence x one query head.  A cache block's keys and values are brought into LDS once per
// workgroup by DMA (no registers), double buffered, one barrier per block; the fragments come from there.  What bounds the kernel is the soft-max
// arithmetic (per score three transcendentals with a cap, one without, at quarter rate) beside about as many cycles of MFMA, so what matters is that two waves
// share a SIMD and run out of phase: under 256 registers a wave, 64 KB of LDS for 128 / 128 heads (two workgroups of four waves), one workgroup of eight
// waves for key size 256, one row tile a wave there (two spill: 640 us where one takes 271).
// A score's form is a template parameter: a plain score's scale and a cap's outer product go into the exponent (three and seven vector instructions a score beside the
// transcendentals, five and nine before).  A lane's four channels of an output row leave in one store: one by one they were 64 stores of two bytes a lane, as long as
// the products of four blocks.
// MI355X, us, before both / now: 4 x 2048 rows, 32 / 8 heads of 128 / 128 264 / 204 = 0.67 PFLOP/s (with a cap 298 / 246; 8000 rows 717 / 606 = 0.87), 16 / 1 heads of 256 / 192 236 / 194;
// 2 x 3000 rows, 16 / 8 heads of 64 / 128 with a cap 155 / 129; 40 x 100 rows, 16 / 1 heads of 256 / 192 58 / 38.
// Serves the sizes of staged_shape(); attn_tiles_kernel serves the rest (sizes that do not fill the pieces of a DMA or the 16-channel tiles).
typedef unsigned ga_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float ga_max_groups(float v)  // over the four lane groups (lanes l ^ 16, l ^ 32)
{
    unsigned       b = bit_cast<unsigned>(v);
    const ga_u32x2 r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    b                = bit_cast<unsigned>(fmaxf(bit_cast<float>((unsigned)r[0]), bit_cast<float>((unsigned)r[1])));
    const ga_u32x2 q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return fmaxf(bit_cast<float>((unsigned)q[0]), bit_cast<float>((unsigned)q[1]));
}

// 16-byte piece of a key row (2 D bytes) that holds channels 8 c .. 8 c + 7: fragment reads are served in groups of 16 lanes (eight rows each of two
// neighbouring pieces), whose pieces fall on 16 different slots of 256 bytes
template<int DS>
__device__ __forceinline__ int ga_key_swizzle(int row)
{
    return DS == 2 ? (row & 2) | ((row & 8) >> 1) : (row & 8) | ((row & 3) << 1);
}

// What a launch does with its scores, where the compiler knows it: nothing (the scale goes into the exponent), a soft cap, or any of the modifiers
enum { kScorePlain = 0, kScoreCap = 1, kScoreAny = 2 };

template<int DS, int VT, int RT, bool MASK, int MOD>
__device__ __forceinline__ void ga_staged_step(const bf16x8 (&qf)[RT][DS], const char* __restrict__ kt_lds, const char* __restrict__ vt_lds, const int (&limit)[RT],
                                               const int (&lower)[RT], int keep_rel, const float (&qscale)[RT], float cap, float inv_cap, bool bias, float r1,
                                               float r2, float (&m)[RT], float (&l)[RT], floatx4 (&o)[RT][VT], const float* __restrict__ tab, int tab_len)
{
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    floatx4   sc[RT][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sc[rt][kt] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const int   row = (kt >> 1) * 32 + (lr >> 2) * 8 + (kt & 1) * 4 + (lr & 3);
        const char* kr  = kt_lds + row * (DS * 64);
        const int   sw  = ga_key_swizzle<DS>(row);
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const bf16x8 kf = *(const bf16x8*)(kr + (((ds * 4 + lg) ^ sw) << 4));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                sc[rt][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[rt][ds], sc[rt][kt], 0, 0, 0);
            }
        }
    }
    bf16x8      pf[RT][2];
    const float cap2 = cap * kLog2e;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        // the exponent of a weight is base * (what each() leaves) + shift - maximum
        const bool  capped = MOD == kScoreCap || (MOD == kScoreAny && cap > 0.f);
        const float k1     = capped ? qscale[rt] * inv_cap * (2.f * kLog2e) : qscale[rt] * kLog2e;
        const float base = MOD == kScorePlain ? k1 : MOD == kScoreCap ? -2.f * cap2 : 1.f, shift = MOD == kScoreCap ? cap2 : 0.f;
        // (one loop per modifier, the branch outside: a branch per score would leave every score in a block of its own)
        auto each = [&](auto f) {
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sc[rt][kt][r] = f(sc[rt][kt][r], (kt >> 1) * 32 + lg * 8 + (kt & 1) * 4 + r);
                }
            }
        };
        if constexpr (MOD == kScoreCap) {  // cap tanh(x) = cap - 2 cap w with w = 1 / (e^2x + 1): the largest score has the smallest w
            each([&](float v, int) { return __builtin_amdgcn_rcpf(fast_exp2(v * k1) + 1.f); });
        }
        if constexpr (MOD == kScoreAny) {
            if (cap > 0.f) {
                each([&](float v, int) { return fmaf(__builtin_amdgcn_rcpf(fast_exp2(v * k1) + 1.f), -2.f * cap2, cap2); });
            }
            else {
                each([&](float v, int) { return v * k1; });
            }
            if (bias) {  // (a key ahead of the row gives the logarithm of a number that may be negative: the mask below discards it)
                each([&](float v, int key) { return fmaf(-r1, __builtin_amdgcn_logf(fmaf(r2, (float)(limit[rt] - key), 1.f)), v); });
            }
            if (tab) {  // (a key ahead of the row reads entry 0 and is masked below)
                each([&](float v, int key) { return fmaf(tab[min(max(limit[rt] - key, 0), tab_len - 1)], kLog2e, v); });
            }
        }
        constexpr float kUnseen = MOD == kScorePlain ? -INFINITY : MOD == kScoreCap ? INFINITY : -1e30f;  // (scaled scores below the maximum that stands in for none)
        if (MASK) {
            each([&](float v, int key) { return (key <= limit[rt] && (key >= lower[rt] || key < keep_rel)) ? v : kUnseen; });
        }
        float best = kUnseen;
        each([&](float v, int) {
            best = MOD == kScoreCap ? fminf(best, v) : fmaxf(best, v);
            return v;
        });
        // (a plain score's scale is not negative: plain_scores())
        const float m_new = fmaxf(m[rt], ga_max_groups(fmaf(best, base, shift)));
        const float m_ref = fmaxf(m_new, -1e29f);  // a row that has seen no key yet (its chunk starts behind this block): every weight is 0
        const float bend  = shift - m_ref;
        float       sum   = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (an unseen key's exponent is below -1e29, or -inf)
                const float e = fast_exp2(MOD == kScoreAny ? sc[rt][kt][r] - m_ref : fmaf(sc[rt][kt][r], base, bend));
                sum += e;
                pf[rt][kt >> 1][(kt & 1) * 4 + r] = (__bf16)e;
            }
        }
        if (__any(m_new != m[rt])) {  // (after the first blocks a row's maximum rarely moves)
            const float alpha = fast_exp2(m[rt] - m_new);
            l[rt] *= alpha;
#pragma unroll
            for (int t = 0; t < VT; ++t) {
                o[rt][t] *= alpha;
            }
        }
        l[rt] += sum;  // the lane's own sixteen keys: the lane groups meet at the end
        m[rt] = m_new;
    }
    const char* vr = vt_lds + lr * 128;
#pragma unroll
    for (int t = 0; t < VT; ++t) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const bf16x8 vf = *(const bf16x8*)(vr + t * 2048 + (((ks * 4 + lg) ^ (lr & 7)) << 4));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                o[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[rt][ks], o[rt][t], 0, 0, 0);
            }
        }
    }
}

template<int DS, int VT, int RT, int W, int MOD>
__global__ __launch_bounds__(W * 64, 2) void attn_staged_kernel(GeneralAttnParams p, int tiles_per_seq)
{
    constexpr int kKeyBytes = 64 * DS * 64, kBytes = kKeyBytes + VT * 16 * 128, kPieces = DS * 4 + VT * 2;  // of one block; DMA pieces of 1 KB
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroup i runs on XCD i % 8: consecutive heads (they share a key head) on one XCD; the longest rows of a sequence first
    int       i = blockIdx.x, h;
    const int H = p.q_heads;
    if (H % 8 == 0) {
        h = (i % 8) * (H / 8) + (i / 8) % (H / 8);
    }
    else {
        h = i % H;
    }
    i /= H;
    const int s = i % p.nseq, ti = tiles_per_seq - 1 - i / p.nseq;
    const int row_base = p.cu_q[s] - p.cu_q[0];
    const int q_len    = p.cu_q[s + 1] - p.cu_q[s];
    const int wg0      = ti * (W * RT * 16);  // the workgroup's first row inside the sequence's portion
    if (wg0 >= q_len) {
        return;
    }
    const int  row0   = wg0 + wave * (RT * 16);
    const bool active = row0 < q_len;  // (an inactive wave still stages and meets the barriers)
    const int  D = p.dim, V = p.vdim;
    const int  g = h / (H / p.kv_heads);
    const int  pos0 = p.k_len[s] - q_len;
    const int  lr = lane & 15, lg = lane >> 4;
    // (a scalar load, one block ahead: a vector load would be waited for together with the DMA in flight)
    typedef const __attribute__((address_space(4))) uint64_t ga_table;
    ga_table*   table = (ga_table*)(p.block_ptrs + (size_t)__builtin_amdgcn_readfirstlane(p.seq_slot ? p.seq_slot[s] : s) * p.block_stride);
    const float cap = p.softcap, inv_cap = cap > 0.f ? 1.f / cap : 0.f;
    const bool  bias = p.dist_r1 != nullptr;
    const float     r1 = bias ? p.dist_r1[h] : 0.f, r2 = bias ? p.dist_r2[h] : 0.f;
    const float*    tab = p.dist_table ? p.dist_table + (size_t)h * p.dist_table_len : nullptr;
    bf16x8     qf[RT][DS];
    float      qscale[RT], m[RT], l[RT] = {};
    int        pos[RT], first[RT];
    bool       q_ok[RT];
    floatx4    o[RT][VT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int qi = row0 + rt * 16 + lr;
        q_ok[rt]     = qi < q_len;
        pos[rt]      = pos0 + qi;
        first[rt]    = ga_first_key(p, pos[rt]);
        const __bf16* q = (const __bf16*)p.q + (size_t)(row_base + min(qi, q_len - 1)) * p.ldq + (size_t)h * D;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            qf[rt][ds] = *(const bf16x8*)(q + ds * 32 + lg * 8);
        }
        qscale[rt] = p.scale * ga_query_temp(p, pos[rt]);
        m[rt]      = -1e30f;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            o[rt][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // this wave's rows see keys up to last_w; those of the workgroup up to last
    const int last_w = pos0 + min(q_len, row0 + RT * 16) - 1, last = pos0 + min(q_len, wg0 + W * RT * 16) - 1;
    const int lo_w = ga_first_key(p, pos0 + min(row0, q_len - 1)), hi_w = ga_first_key(p, last_w);
    const int lo = ga_first_key(p, pos0 + wg0), keep = ga_keep(p);
    const int bf = __builtin_amdgcn_readfirstlane(lo / 64), nk = __builtin_amdgcn_readfirstlane(ga_keep_blocks(p, lo, bf, 64));
    const int n  = __builtin_amdgcn_readfirstlane(nk + last / 64 + 1 - bf);
    // DMA: lane L of a piece fetches the 16 bytes that belong into slot L.  Piece k of the keys: 1024 / 2 D rows, of the values: 8 channels
    constexpr int  kRowsPer = 1024 / (DS * 64);
    const unsigned lds0     = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
    const int      vsrc     = (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 3) & 7)) << 4);
    const int64_t  khead = p.layer_offset + (int64_t)ga_key_head(p, g) * kKeyBytes, vhead = p.layer_offset + p.v_offset + (int64_t)ga_value_head(p, g) * V * 128;
    uint64_t next = table[ga_block_at(0, nk, bf)];
    auto stage = [&](int bi, int buf) {
        const char* base = (const char*)next;
        next             = table[ga_block_at(min(bi + 1, n - 1), nk, bf)];
        const auto     rk   = __builtin_amdgcn_make_buffer_rsrc((void*)(base + khead), 0, kKeyBytes, 0x00020000);
        const auto     rv   = __builtin_amdgcn_make_buffer_rsrc((void*)(base + vhead), 0, VT * 2048, 0x00020000);
        const unsigned dst  = lds0 + buf * kBytes;
#pragma unroll
        for (int r = 0; r < (kPieces + W - 1) / W; ++r) {
            const int pc = r * W + wave;
            if (pc < DS * 4) {
                const int row = pc * kRowsPer + lane / (DS * 4), c = lane % (DS * 4);
                stream_dma16(rk, row * (DS * 64) + ((c ^ ga_key_swizzle<DS>(row)) << 4), 0, dst + pc * 1024);
            }
            else if (pc < kPieces) {
                stream_dma16(rv, vsrc, (pc - DS * 4) * 1024, dst + pc * 1024);
            }
        }
    };
    stage(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int bi = 0; bi < n; ++bi) {
        const int buf = bi & 1, b = ga_block_at(bi, nk, bf);
        if (bi + 1 < n) {
            stage(bi + 1, buf ^ 1);  // every wave is past the barrier behind its reads of that buffer
        }
        const char *kt = smem + buf * kBytes, *vt = kt + kKeyBytes;
        if (active && b * 64 <= last_w && (b * 64 + 63 >= lo_w || b * 64 < keep)) {
            int limit[RT], lower[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                limit[rt] = q_ok[rt] ? pos[rt] - b * 64 : -1;
                lower[rt] = first[rt] - b * 64;
            }
            const bool whole = b * 64 + 63 <= pos0 + row0 && b * 64 >= hi_w;  // every row of the wave sees the whole block
#define TM_STAGED(MASK_) \
    ga_staged_step<DS, VT, RT, MASK_, MOD>(qf, kt, vt, limit, lower, MASK_ ? keep - b * 64 : 0, qscale, cap, inv_cap, bias, r1, r2, m, l, o, tab, p.dist_table_len)
            if (whole) {
                TM_STAGED(false);
            }
            else {
                TM_STAGED(true);
            }
#undef TM_STAGED
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of the next block have landed ...
        __syncthreads();                                  // ... everybody's have, and everybody is done reading this one
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        float sum = l[rt];
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (!q_ok[rt]) {
            continue;
        }
        float inv;
        if (p.sink) {  // m is in the log2 domain
            const float sk = p.sink[h] * kLog2e, mf = fmaxf(m[rt], sk), a = fast_exp2(m[rt] - mf);
            inv            = a / (sum * a + fast_exp2(sk - mf));
        }
        else {
            inv = 1.f / sum;
        }
        const int t0 = row_base + row0 + rt * 16 + lr;
        inv *= ga_out_gate(p, t0, h);
#pragma unroll
        for (int t = 0; t < VT; ++t) {  // lane holds O[row lr][channels t * 16 + lg * 4 .. + 3]
            ga_store4<__bf16>(p, t0, h, t * 16 + lg * 4, o[rt][t] * inv);
        }
    }
}

template<int DS, int VT, int RT, int W, int MOD>
static int launch_staged_mod(const GeneralAttnParams& p, hipStream_t st)
{
    constexpr int lds = 2 * (64 * DS * 64 + VT * 16 * 128);
    const auto    k   = attn_staged_kernel<DS, VT, RT, W, MOD>;
    TM_TRY_RC(ensure_dynamic_lds((const void*)k, lds));
    const int tiles = (p.max_q_len + W * RT * 16 - 1) / (W * RT * 16);
    k<<<(unsigned)(p.nseq * tiles) * (unsigned)p.q_heads, W * 64, lds, st>>>(p, tiles);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<int DS, int VT, int RT, int W>
static int launch_staged(const GeneralAttnParams& p, hipStream_t st)
{
    const bool more = p.dist_r1 || p.dist_table || !(p.scale > 0.f) || !(p.qtemp_coef >= 0.f);  // (a plain score's largest has the largest weight)
    return more             ? launch_staged_mod<DS, VT, RT, W, kScoreAny>(p, st) :
           p.softcap > 0.f  ? launch_staged_mod<DS, VT, RT, W, kScoreCap>(p, st) :
                              launch_staged_mod<DS, VT, RT, W, kScorePlain>(p, st);
}

// key / value sizes of the staged kernel (0: none)
static int staged_shape(const GeneralAttnParams& p)
{
    static const int kShapes[][2] = {{64, 64}, {64, 128}, {128, 128}, {256, 128}, {256, 192}, {256, 256}};
    for (int i = 0; i < 6; ++i) {
        if (p.dim == kShapes[i][0] && p.vdim == kShapes[i][1]) {
            return i + 1;
        }
    }
    return 0;
}

// row tiles per wave of the prefill kernel (64 * RT query rows per workgroup): as many as the register file holds without scratch --
// every key / value fragment a wave loads then serves 16 * RT query rows.  (Key sizes up to 256 with value sizes up to 192 -- the latent
// space of latent attention -- still hold two: 256 VGPRs + 184 AGPRs.)
constexpr int tile_rt(int ds, int vt)
{
    return (ds <= 4 && vt <= 8) ? 4 : ((ds <= 4 || vt <= 8 || (ds <= 8 && vt <= 12)) ? 2 : 1);
}

// value sizes are served by the next even tile count (the kernels test channel < vdim), key sizes by 1, 2, 3, 4, 6 or 8 steps
template<int DS>
static void launch_tiles_ds(const GeneralAttnParams& p, int arg, dim3 grid, hipStream_t st, bool decode)
{
    const int vt = (p.vdim + 15) / 16;
    switch (vt <= 1 ? 1 : (vt + 1) / 2 * 2) {
#define TM_TILE_CASE(VT_)                                                           \
    case VT_:                                                                       \
        if (decode) {                                                               \
            attn_decode_kernel<DS, VT_><<<grid, 256, 0, st>>>(p, arg);              \
        }                                                                           \
        else {                                                                      \
            attn_tiles_kernel<DS, VT_, tile_rt(DS, VT_)><<<grid, 256, 0, st>>>(p, arg); \
        }                                                                           \
        break;
        TM_TILE_CASE(1) TM_TILE_CASE(2) TM_TILE_CASE(4) TM_TILE_CASE(6) TM_TILE_CASE(8) TM_TILE_CASE(10) TM_TILE_CASE(12) TM_TILE_CASE(14)
        TM_TILE_CASE(16)
#undef TM_TILE_CASE
    }
}

static int launch_mfma(const GeneralAttnParams& p, int arg, dim3 grid, hipStream_t st, bool decode)
{
    const int ds = (p.dim + 31) / 32;
    switch (ds <= 4 ? ds : (ds <= 6 ? 6 : 8)) {
        case 1: launch_tiles_ds<1>(p, arg, grid, st, decode); break;
        case 2: launch_tiles_ds<2>(p, arg, grid, st, decode); break;
        case 3: launch_tiles_ds<3>(p, arg, grid, st, decode); break;
        case 4: launch_tiles_ds<4>(p, arg, grid, st, decode); break;
        case 6: launch_tiles_ds<6>(p, arg, grid, st, decode); break;
        default: launch_tiles_ds<8>(p, arg, grid, st, decode); break;
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

bool general_attention_decode_ok(const GeneralAttnParams& p)
{
    return p.elem_bytes == 2 && p.block_len == 64 && p.dim % 8 == 0 && p.vdim % 8 == 0 && p.dim <= 256 && p.vdim <= 256 && p.ldq % 8 == 0
           && p.q_heads % p.kv_heads == 0 && p.splits >= 1 && (p.splits == 1 || (p.partial_o && p.partial_ml));
}

int launch_general_attention_decode(const GeneralAttnParams& p, hipStream_t st)
{
    TM_REQUIRE(general_attention_decode_ok(p), "attention decode kernel: bf16, 64-token blocks, dim and vdim multiples of 8 up to 256");
    if (p.rows == 0) {
        return 0;
    }
    // A workgroup takes four blocks at the time of one, so splits below four blocks only pay while the launch leaves compute units idle: 256 workgroups
    // without splits (64 * 4) are enough.  32 rows of 32 / 8 heads of 128, ~150 tokens, 8 splits: 13.2 us with splits of one block, 9.4 with at least four
    // (eight: the same), 21.9 when the splits without a block ran to the end as well; a merge launch took 4.6 more
    const int         chunks = (p.q_heads / p.kv_heads + 15) / 16, base = p.rows * p.kv_heads * chunks;
    GeneralAttnParams a      = p;
    a.tickets                = ga_tickets(p);
    a.split_blocks           = std::min(4, std::max(1, base / 64));
    TM_TRY_RC(launch_mfma(a, chunks, dim3(p.rows, p.kv_heads * chunks, p.splits), st, true));
    if (p.splits > 1 && !a.tickets) {
        launch_rows_merge<__bf16>(a, st);
        TM_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

// ---- fp32: the heads of a key head as a tile ------------------------------------------------------------------------------------------
// attn_decode_kernel's arrangement for an fp32 cache, v_mfma_f32_16x16x4: workgroup per (row, 16 heads of a key head, key split), each wave 16 of a block's 64
// keys.  S^T = K Q^T with the channels of a step dealt so that a lane's four are one load, and P^T then stands in the registers that O^T += V^T P^T reads.
// What bounds it is a CU's load path -- the row kernel brings every key once per query head through it -- and at few rows the chain of dependent loads.
// us, row kernel / this one: 16 / 1 heads of 256 / 192, 3 rows over ~180 tokens in a model 22.0 / 14.1; before this kernel's loads were in flight together, alone: 3 rows 21.0 / 15.1, 2 rows over 2000 61.3 / 27.4, 420 rows
// of three prompts 148 / 31, a prompt of 2000 7165 / 597; 32 / 8 heads of 128 / 128 14.9 / 9.9, 44.2 / 19.3, 147 / 66, 7690 / 1915; 16 / 16 heads of 128 / 128, where
// the tile holds one row of sixteen, 16.5 / 10.1, 56.8 / 22.1, 145 / 124, 10300 / 3850.  Where it loses: general_attention_heads_f32_pays.
template<int DS, int VT>
__global__ __launch_bounds__(256) void attn_heads_f32_kernel(GeneralAttnParams p, int chunks)
{
    __shared__ float    ml_s[4][16][2];
    __shared__ unsigned last_s;
    __shared__ float    o_s[3][16][VT * 16 + 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
    const int t = blockIdx.x, g = blockIdx.y / chunks, chunk = blockIdx.y % chunks, sp = blockIdx.z;
    const int D = p.dim, V = p.vdim, group = p.q_heads / p.kv_heads, h0 = g * group + chunk * 16, nh = min(16, group - chunk * 16);
    const int h = h0 + min(lr, nh - 1), pos = p.row_pos[t], s = p.row_seq[t];
    const uint64_t* table = p.block_ptrs + (size_t)(p.seq_slot ? p.seq_slot[s] : s) * p.block_stride;
    const int first = ga_first_key(p, pos), bf = first / 64;
    const int keep = ga_keep(p), nk = ga_keep_blocks(p, first, bf, 64);
    const int nvis = nk + pos / 64 + 1 - bf, per = ga_split_len(p, nvis), nsplit = ga_split_count(p, nvis);
    const int i0 = sp * per, i1 = min(nvis, i0 + per);
    if (sp >= nsplit) {
        return;
    }
    // Keys and values of a block are asked for all at once, before the queries are waited for; the barrier keeps the compiler from asking for them two at a time (420 rows of three prompts, 16 / 1 heads of 256 / 192: 36.6 -> 31.6 us)
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    const bool    tail = D < DS * 16;
    floatx4       q[DS], o[VT], k[DS], v4[VT];
#pragma unroll
    for (int i = 0; i < DS; ++i) {
        q[i] = *(const ga_floatx4_any*)((const float*)p.q + (size_t)t * p.ldq + (size_t)h * D + min(i * 16 + lg * 4, D - 4));
    }
#pragma unroll
    for (int v = 0; v < VT; ++v) {
        o[v] = zero;
    }
    float     m = -1e30f, l = 0.f;
    const int j0 = wave * 16;
    auto      unseen = [&](int bi) {  // none of the wave's keys of the block is seen
        const int b = ga_block_at(bi, nk, bf), limit = pos - b * 64, lower = first - b * 64, klo = keep - b * 64;
        return j0 > limit || (j0 + 15 < lower && j0 >= klo);
    };
    auto load = [&](int bi) {
        const char*  base = global_ptr(table[ga_block_at(bi, nk, bf)]) + p.layer_offset;
        const float* kb   = (const float*)base + (size_t)ga_key_head(p, g) * 64 * D;
        const float* vb   = (const float*)(base + p.v_offset) + (size_t)ga_value_head(p, g) * 64 * V;
#pragma unroll
        for (int i = 0; i < DS; ++i) {
            k[i] = *(const ga_floatx4_any*)(kb + (uint32_t)((j0 + lr) * D + min(i * 16 + lg * 4, D - 4)));
        }
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            v4[v] = *(const ga_floatx4_any*)(vb + (uint32_t)(min(v * 16 + lr, V - 1) * 64 + j0 + lg * 4));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int bi = i0;
    while (bi < i1 && unseen(bi)) {
        ++bi;
    }
    if (bi < i1) {
        load(bi);
        const float  qscale = p.scale * ga_query_temp(p, pos);
        const bool   bias   = p.dist_r1 != nullptr;
        const float  r1 = bias ? p.dist_r1[h] : 0.f, r2 = bias ? p.dist_r2[h] : 0.f;
        const float* tab = p.dist_table + (size_t)h * p.dist_table_len;
        if (tail) {
#pragma unroll
            for (int i = 0; i < DS; ++i) {
                q[i] = i * 16 + lg * 4 < D ? q[i] : zero;
            }
        }
        for (;;) {
            const int b = ga_block_at(bi, nk, bf), limit = pos - b * 64, lower = first - b * 64, klo = keep - b * 64;
            // two chains: a product that waits for the one before it takes longer than the matrix core needs
            floatx4 sc = zero, sc2 = zero;
#pragma unroll
            for (int i = 0; i < DS; i += 2) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    sc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][c], q[i][c], sc, 0, 0, 0);
                    if (i + 1 < DS) {
                        sc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i + 1][c], q[i + 1][c], sc2, 0, 0, 0);
                    }
                }
            }
            sc += sc2;
            float add[4] = {};
            if (p.dist_table) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    add[r] = tab[min(max(limit - (j0 + lg * 4 + r), 0), p.dist_table_len - 1)];
                }
            }
            bool  seen[4];
            float mx = -1e30f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = j0 + lg * 4 + r;
                seen[r]     = j <= limit && (j >= lower || j < klo);
                float x     = ga_modify(p, sc[r], qscale);
                if (bias) {
                    x -= r1 * log1pf(r2 * (float)(limit - j));
                }
                x += add[r];
                sc[r] = seen[r] ? x : -1e30f;
                mx    = fmaxf(mx, sc[r]);
            }
            const float m_new = fmaxf(m, ga_max_groups(mx)), alpha = __expf(m - m_new);
            m = m_new;
            l *= alpha;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[r] = seen[r] ? __expf(sc[r] - m_new) : 0.f;
                l += sc[r];
            }
            // entries that the row does not see -- behind its own, and before its window or chunk -- may hold anything: a weight of zero does not take them out
            const bool whole = j0 + 15 <= limit && (j0 >= lower || j0 + 15 < klo);
            if (!whole) {
#pragma unroll
                for (int v = 0; v < VT; ++v) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v4[v][r] = seen[r] ? v4[v][r] : 0.f;
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                o[v] *= alpha;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int v = 0; v < VT; ++v) {
                    o[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(v4[v][r], sc[r], o[v], 0, 0, 0);
                }
            }
            do {
                ++bi;
            } while (bi < i1 && unseen(bi));
            if (bi >= i1) {
                break;
            }
            load(bi);
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    ga_close_heads<float, VT>(p, t, sp, nsplit, h0, nh, m, l, o, ml_s, o_s, &last_s);
}

bool general_attention_heads_f32_ok(const GeneralAttnParams& p)
{
    return p.elem_bytes == 4 && p.block_len == 64 && p.dim % 4 == 0 && p.vdim % 4 == 0 && p.dim >= 4 && p.dim <= 256 && p.vdim >= 4 && p.vdim <= 256 && p.kv_heads >= 1
           && p.q_heads % p.kv_heads == 0 && p.splits >= 1 && (p.splits == 1 || (p.partial_o && p.partial_ml));
}

// The heads kernel or the row kernel.  Up to about two workgroups a CU latency counts, which the heads kernel has less of.  Beyond, a workgroup of it costs what a tile of sixteen
// heads costs however many of them exist, and the merge of its four waves: with a few heads a key head and few keys a row the row kernel's waves, each of them one head, do less.
// ns a tile or head where the chip is full, fitted to 1950 sizes (16 ... 256 channels, 1 ... 8 heads a key head, 1 ... 2000 rows, 17 ... 1000 keys).  us, row kernel / heads kernel:
// 32 / 32 heads of 12, 420 prompt rows 35 / 100; 32 / 32 of 128, 60 prompts of 33 267 / 736, a prompt of 1000 2631 / 2015; 32 / 8 of 64, 60 prompts of 33 125 / 96;
// 8 / 8 of 256, 128 decoded rows over 20 keys 19 / 47, three rows over 180 25 / 14.  What a row sees besides its own portion is not known here: a prompt counts as its own
// keys, a decoded row as half a block (4 heads of 256 a key head, 128 rows over 20 keys lose by it, 31 / 47; over 60 keys they gain)
bool general_attention_heads_f32_pays(const GeneralAttnParams& p, bool prefill)
{
    const int     group = p.q_heads / p.kv_heads, chunks = (group + 15) / 16, ds = (p.dim + 15) / 16, vt = (p.vdim + 15) / 16;
    const int     steps = ds <= 4 && vt <= 8 ? 4 + (vt <= 4 ? 4 : 8) : ds <= 8 && vt <= 8 ? 16 : 16 + (vt <= 8 ? 8 : vt <= 12 ? 12 : 16);  // channel steps of the instantiation
    const int64_t tiles = (int64_t)p.rows * p.kv_heads * chunks;
    if (tiles <= (steps > 16 ? 256 : 512)) {
        return true;
    }
    prefill     = prefill && p.max_q_len > 1;
    double keys = prefill ? p.max_q_len / 2.0 : 32.0;
    keys        = std::min(keys, p.chunk > 0 ? p.chunk / 2.0 : keys);
    keys        = std::min(keys, p.window > 0 ? (double)p.window + p.keep_first : keys);
    const double blocks = prefill ? keys / 64 + 0.5 : 1.0;
    const double tile   = steps > 16 ? steps * (0.6 + 0.62 * blocks) : steps * (0.3 + 0.6 * blocks);
    const double head   = 0.84 + 0.0035 * (p.dim + p.vdim) + (0.56 + 0.041 * (p.dim + p.vdim)) * keys / 64;
    return tile < head * group / chunks;
}

int launch_general_attention_heads_f32(const GeneralAttnParams& p, hipStream_t st)
{
    TM_REQUIRE(general_attention_heads_f32_ok(p), "attention over heads: fp32, 64-token blocks, dim and vdim multiples of 4 up to 256");
    TM_REQUIRE(p.rows >= 0 && p.chunk >= 0 && (!p.dist_r1 || p.dist_r2) && (!p.out_gate || p.ld_gate >= p.q_heads), "attention: chunk / distance penalty / gate");
    TM_REQUIRE(p.window >= 0 && p.keep_first >= 0, "attention: window / kept first tokens");
    TM_REQUIRE(p.k_heads >= 0 && p.v_heads >= 0 && (!p.dist_table || p.dist_table_len >= 1), "attention: key / value head counts, distance table");
    TM_REQUIRE(p.qtemp_coef == 0.f || p.qtemp_every > 0.f, "attention: query temperature period");
    if (p.rows == 0) {
        return 0;
    }
    const int         chunks = (p.q_heads / p.kv_heads + 15) / 16;
    GeneralAttnParams a      = p;
    a.tickets                = ga_tickets(p);
    a.split_blocks           = std::min(4, std::max(1, p.rows * p.kv_heads * chunks / 64));  // (as in the decode kernel)
    const dim3 grid(p.rows, p.kv_heads * chunks, p.splits);
    const int  ds = (p.dim + 15) / 16, vt = (p.vdim + 15) / 16;
#define TM_HEADS(DS_, VT_)                                            \
    if (ds <= DS_ && vt <= VT_) {                                     \
        attn_heads_f32_kernel<DS_, VT_><<<grid, 256, 0, st>>>(a, chunks); \
    }                                                                 \
    else
    TM_HEADS(4, 4) TM_HEADS(4, 8) TM_HEADS(8, 8) TM_HEADS(16, 8) TM_HEADS(16, 12)
    {
        attn_heads_f32_kernel<16, 16><<<grid, 256, 0, st>>>(a, chunks);
    }
#undef TM_HEADS
    TM_HIP_CHECK(hipGetLastError());
    if (p.splits > 1 && !a.tickets) {
        launch_rows_merge<float>(a, st);
        TM_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

int launch_general_attention_tiles(const GeneralAttnParams& p, hipStream_t st)
{
    TM_REQUIRE(general_attention_tiles_ok(p), "attention tile kernel: bf16, 64-token blocks, dim and vdim multiples of 8 up to 256, sequence description");
    if (p.rows == 0) {
        return 0;
    }
    switch (staged_shape(p)) {
        case 1: return launch_staged<2, 4, 2, 4>(p, st);
        case 2: return launch_staged<2, 8, 2, 4>(p, st);
        case 3: return launch_staged<4, 8, 2, 4>(p, st);
        case 4: return launch_staged<8, 8, 1, 8>(p, st);
        case 5: return launch_staged<8, 12, 1, 8>(p, st);
        case 6: return launch_staged<8, 16, 1, 8>(p, st);
        default: break;
    }
    const int ds = (p.dim + 31) / 32, vt = (p.vdim + 15) / 16;
    const int rows = kTileRows * tile_rt(ds <= 4 ? ds : (ds <= 6 ? 6 : 8), vt <= 1 ? 1 : (vt + 1) / 2 * 2);  // the instantiation launch_mfma picks
    const int tiles_per_seq = (p.max_q_len + rows - 1) / rows;
    return launch_mfma(p, tiles_per_seq, dim3(p.nseq * tiles_per_seq, p.q_heads), st, false);
}

int launch_general_attention(const GeneralAttnParams& p, bool prefill, hipStream_t st)
{
    static const bool tiles_on = !getenv("TM_ATTN_TILES") || atoi(getenv("TM_ATTN_TILES")) != 0;  // A/B switch: 0 = row kernel everywhere
    if (prefill && tiles_on && general_attention_tiles_ok(p)) {
        return launch_general_attention_tiles(p, st);
    }
    if (!prefill && tiles_on && general_attention_decode_ok(p)) {
        return launch_general_attention_decode(p, st);
    }
    if (tiles_on && general_attention_heads_f32_ok(p) && general_attention_heads_f32_pays(p, prefill)) {
        return launch_general_attention_heads_f32(p, st);
    }
    return launch_general_attention_rows(p, st);
}

}  // namespace tmk
