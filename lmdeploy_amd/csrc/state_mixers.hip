// Mixers with a recurrent state instead of a key / value cache: per head a matrix S [dim][vdim] in fp32 that every token updates.
//
//   linear attention ("lightning"):  S <- decay[head] S + k v^T                         o = S^T q      q, k, v = silu(projection)
//   generalized delta rule:          S <- diag(w) S - (a u)(u^T S) + k v^T              o = S^T r      u = k / sqrt(|k|^2 + 1e-6),
//                                    w, a per key channel (both terms read the old S)
//   gated delta rule:                S <- diag(g) S;  S <- S + k (beta (v - S^T k))^T   o = S^T q      is the same recurrence with
//                                    w = g, u = g k, a u = beta k and the key beta k (launch_gdelta_prep forms these vectors)
//   forget-gate linear attention:    S <- diag(f) S + (1 - f) v^T                      o = S^T q      q = silu(projection), f per key channel,
//                                    f = low + (1 - low) sigmoid(logit + bias)
//   retention:                       S <- decay[head] S + k v^T                         o = S^T q      q, k rotated by position, k scaled
//   bonus recurrence:                o = (S + diag(u) k v^T)^T q;  S <- diag(w) S + k v^T            w = exp(-exp(logit)) per key channel; the
//                                    current token enters o through the bonus u only
//   short convolution:               y_t = sum_j w[:, j] u_(t - taps + 1 + j) per channel; its state is the last taps - 1 inputs
//
// State pool: one state per (slot, layer run) -- slot = the engine's batch slot of the sequence, plus one parking slot for the decode
// rows of slots that hold no running sequence.  A sequence whose first row of a launch has position 0 starts from zero whatever the
// slot holds (slots are reused without clearing).  Everything here is fp32 in both number formats of the engine.
//
// The columns of S evolve independently (S[:, j] only meets v[j]), so the work is split over (sequence, head, 16 value columns): one wave
// owns a [dim][16] slab -- lane = (column pair c = lane % 8, row group rg = lane / 8), rows rg * dq + ii, dq = ceil(dim / 8), columns
// 2 c and 2 c + 1: DQ x 2 registers -- and walks the sequence's rows of this launch in order; the reductions over the key channels are a
// register sum + three lane shuffles.  (Two columns per lane: every per-token vector element read from LDS feeds two multiply-adds;
// with one the kernel is bound by LDS reads.)  Four waves (64 value columns) share a workgroup and the LDS stage of the per-token
// vectors (q, k, and w, a u, u for the delta rule), loaded TB tokens at a time: the next stage's global loads are issued before the
// current stage's tokens are walked and land in the other LDS buffer afterwards, so their latency hides under the recurrence.  A slab is
// stored as the wave holds it, [ii][column of the pair][lane]: loading and storing it are fully coalesced.
// The delta rule walks short portions, and portions of many heads x sequences, one token after the other (two dependent reductions per token; state_mix_chunks); the
// others, and every portion of the other mixers, run in chunks on the matrix cores (below).
// One kernel serves prompt portions (many rows per sequence) and decoded tokens (one row, TB = 1): the state traffic of a decode step,
// 2 * dim * vdim * 4 bytes per head, is what bounds it.
#include "tm_kernels.h"
#include "gemm_stream.h"  // stream_dma16
#include <algorithm>

namespace tmk {

constexpr int kStateCW = 8;   // lanes per row group; 64 / kStateCW row groups
constexpr int kStateNC = 2;   // value columns per lane: a wave owns kStateCW * kStateNC columns

__device__ __forceinline__ float sm_silu(float z)
{
    return z / (1.f + expf(-z));
}

// the delta rule's removal vector a u and decay from their logits
__device__ __forceinline__ float delta_rate(float u, float logit)
{
    return u / (1.f + expf(-logit));
}
__device__ __forceinline__ float delta_decay(float logit)
{
    return expf(-0.60653065971263342f / (1.f + expf(-logit)));
}

// staged vectors per token: q, k; the delta rule's decays, a u and u; the forget gates; the bonus recurrence's decays and u k
__host__ __device__ constexpr int state_vectors(int kind)
{
    return kind == kStateDelta ? 5 : kind == kStateBonus ? 4 : kind == kStateForget ? 3 : 2;
}

// channel d of a query / key head turned to position pos (first rot_dims channels; channel i pairs with i + rot_dims / 2), fp32
struct Rotation {
    float sn = 0.f, cs = 1.f;
    int   partner = 0;
    __device__ __forceinline__ Rotation(const StateMixParams& p, int pos, int d)
    {
        const int half = p.rot_dims >> 1;
        if (d < p.rot_dims) {
            sincosf((float)pos * p.inv_freq[d < half ? d : d - half], &sn, &cs);
            partner = d < half ? half : -half;
            sn      = d < half ? -sn : sn;
        }
    }
    __device__ __forceinline__ float operator()(const float* x) const  // x: the channel itself
    {
        return x[0] * cs + x[partner] * sn;
    }
};

size_t state_mix_floats(int heads, int dim, int vdim)
{
    const int wcols = kStateCW * kStateNC;
    return (size_t)heads * ((vdim + wcols - 1) / wcols) * ((dim + 7) / 8) * 64 * kStateNC;
}

// grid (nseq, heads, ceil(vdim / 64)), 256 threads, dynamic LDS = 2 * tb * (NV * dim + 64) floats; NV = 2 ... 5
// staged vectors per token, tb = min(TB, max_q_len) tokens per stage, TB: as many as keep the buffers under 64 KB.
// EXACT: dim == 8 * DQ -- every LDS stride is a compile-time constant and the per-token vectors are read 16 bytes at a time
template<int DQ, int KIND, int TB, bool EXACT>
__global__ __launch_bounds__(256) void state_mix_kernel(StateMixParams p)
{
    extern __shared__ __attribute__((aligned(16))) float lds_all[];
    constexpr bool DELTA = KIND == kStateDelta, LINEAR = KIND == kStateLinear, FORGET = KIND == kStateForget, RETAIN = KIND == kStateRetention,
                   BONUS = KIND == kStateBonus;
    constexpr int NV = state_vectors(KIND), CW = kStateCW, NC = kStateNC, RG = 64 / CW, WV = CW * NC, WC = 4 * WV;
    constexpr int PER  = (TB * DQ * RG + 255) / 256;  // staged elements per vector and thread (dim <= DQ * RG)
    constexpr int VPER = (TB * WC + 255) / 256;
    const int s = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int D = EXACT ? DQ * RG : p.dim, V = p.vdim, dq = EXACT ? DQ : (D + RG - 1) / RG, ncb = (V + WV - 1) / WV;
    const int Dp = dq * RG;  // staged vectors are padded to the row groups' share (zeros behind dim)
    const int cb = blockIdx.z * 4 + wave, c = lane % CW, rg = lane / CW, j0 = cb * WV + c * NC;
    const bool wave_on = cb < ncb;
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int pos0 = p.k_len[s] - q_len;
    int       slot = p.seq_slot ? p.seq_slot[s] : p.slot0 + s;
    if (p.active && !p.active[s]) {
        slot = p.park_slot;
    }
    float* slab = p.state + (size_t)slot * p.slot_stride + p.layer_offset + ((size_t)h * ncb + (wave_on ? cb : 0)) * dq * 64 * NC;
    float  S[DQ][NC];
#pragma unroll
    for (int ii = 0; ii < DQ; ++ii) {
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            S[ii][n] = (wave_on && pos0 > 0 && ii < dq) ? slab[(ii * NC + n) * 64 + lane] : 0.f;
        }
    }
    const float  decay = LINEAR || RETAIN ? p.decay_h[h] : 0.f;
    const int    tb    = min(TB, p.max_q_len);
    const size_t stage = (size_t)tb * (NV * Dp + WC);  // floats of one LDS buffer: [tb][NV][Dp] vectors, then [tb][WC] values
    float        rv[NV][PER], rval[VPER];
    // global loads of the stage that starts at token t0 (into registers) / their way into LDS buffer `buf`
    auto fetch = [&](int t0) {
        const int nt = min(tb, q_len - t0);
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int  i  = threadIdx.x + r * 256;
            const bool ok = i < nt * Dp && i % Dp < D;
            const int  t = ok ? i / Dp : 0, d = ok ? i % Dp : 0;
            const size_t row = (size_t)(row0 + t0 + t);
            const float* pr  = p.proj + row * p.ld + h * D + d;
            rv[0][r] = ok ? pr[p.c_q] : 0.f;
            if constexpr (RETAIN) {
                const Rotation ro(p, pos0 + t0 + t, d);
                rv[0][r] = ok ? ro(pr + p.c_q) : 0.f;
                rv[1][r] = ok ? ro(pr + p.c_k) * p.k_mult : 0.f;
            }
            else             if constexpr (FORGET) {  // gate logit and lower bound; padding gets a gate of one: nothing is written there
                rv[1][r] = ok ? pr[p.c_f] + p.f_bias[h * D + d] : 0.f;
                rv[2][r] = ok ? p.f_low[h * D + d] : 1.f;
            }
            else {
                rv[1][r] = ok ? pr[p.c_k] : 0.f;
            }
            if constexpr (BONUS) {
                rv[2][r] = ok ? p.decay_w[row * p.ld_w + h * D + d] : 0.f;
                rv[3][r] = ok ? p.bonus[h * D + d] : 0.f;
            }
            if constexpr (DELTA) {
                rv[2][r] = ok ? p.decay_w[row * p.ld_w + h * D + d] : 0.f;
                rv[3][r] = ok ? pr[p.c_a] : 0.f;
                rv[4][r] = ok ? p.unit[row * p.ld_u + h * D + d] : 0.f;
            }
        }
#pragma unroll
        for (int r = 0; r < VPER; ++r) {
            const int i = threadIdx.x + r * 256;
            const int t = i / WC, jj = blockIdx.z * WC + i % WC;
            rval[r]     = (i < nt * WC && jj < V) ? p.proj[(size_t)(row0 + t0 + t) * p.ld + p.c_v + h * V + jj] : 0.f;
        }
    };
    auto park = [&](int t0, int buf) {
        const int nt  = min(tb, q_len - t0);
        float*    lds = lds_all + buf * stage;
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int i = threadIdx.x + r * 256;
            if (i < nt * Dp) {
                const int t = i / Dp, d = i % Dp;
                if constexpr (FORGET) {
                    const float z = rv[1][r], low = rv[2][r], ez = expf(-fabsf(z)), hi = 1.f / (1.f + ez), lo = ez * hi;  // sigmoid(|z|), sigmoid(-|z|)
                    lds[(t * NV + 0) * Dp + d] = sm_silu(rv[0][r]);
                    lds[(t * NV + 1) * Dp + d] = (1.f - low) * (z > 0.f ? lo : hi);              // 1 - f without cancellation
                    lds[(t * NV + 2) * Dp + d] = fmaf(1.f - low, z > 0.f ? hi : lo, low);        // f
                }
                else if constexpr (BONUS) {
                    lds[(t * NV + 0) * Dp + d] = rv[0][r];
                    lds[(t * NV + 1) * Dp + d] = rv[1][r];
                    lds[(t * NV + 2) * Dp + d] = expf(-expf(rv[2][r]));
                    lds[(t * NV + 3) * Dp + d] = rv[3][r] * rv[1][r];
                }
                else {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        lds[(t * NV + v) * Dp + d] = DELTA || RETAIN ? rv[v][r] : sm_silu(rv[v][r]);
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < VPER; ++r) {
            const int i = threadIdx.x + r * 256;
            if (i < nt * WC) {
                lds[(size_t)tb * NV * Dp + i] = LINEAR ? sm_silu(rval[r]) : rval[r];
            }
        }
    };
    auto reduce_rg = [&](float a) {
        a += __shfl_xor(a, 8);
        a += __shfl_xor(a, 16);
        return a + __shfl_xor(a, 32);
    };
    auto store_out = [&](int t, const float (&o)[NC]) {
        float* out = p.out + (size_t)(row0 + t) * p.ldo + h * V + j0;
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            if (j0 + n < V) {
                out[n] = o[n];
            }
        }
    };
    fetch(0);
    park(0, 0);
    __syncthreads();
    int buf = 0;
    for (int t0 = 0; t0 < q_len; t0 += tb, buf ^= 1) {
        const int  nt   = min(tb, q_len - t0);
        const bool more = t0 + tb < q_len;
        if (more) {
            fetch(t0 + tb);
        }
        const float* lds = lds_all + buf * stage;
        const float* sv  = lds + (size_t)tb * NV * Dp + wave * WV + c * NC;  // the lane's columns of token t at sv[t * WC + n]
        for (int t = 0; wave_on && t < nt; ++t) {
            const float* q  = lds + (size_t)(t * NV + 0) * Dp + rg * dq;
            const float* k  = lds + (size_t)(t * NV + 1) * Dp + rg * dq;
            const float* w  = lds + (size_t)(t * NV + (LINEAR || RETAIN ? 0 : 2)) * Dp + rg * dq;
            const float* au = lds + (size_t)(t * NV + (DELTA || BONUS ? 3 : 0)) * Dp + rg * dq;  // a u, or bonus times key
            const float* u  = lds + (size_t)(t * NV + (DELTA ? 4 : 0)) * Dp + rg * dq;
            float        v[NC], us[NC], acc[NC];
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                v[n]  = sv[t * WC + n];
                us[n] = acc[n] = 0.f;
            }
            if constexpr (DELTA) {
#pragma unroll
                for (int ii = 0; ii < DQ; ++ii) {
                    if (EXACT || ii < dq) {  // (rows behind dim meet staged zeros and stay zero)
                        const float uv = u[ii];
#pragma unroll
                        for (int n = 0; n < NC; ++n) {
                            us[n] = fmaf(uv, S[ii][n], us[n]);
                        }
                    }
                }
#pragma unroll
                for (int n = 0; n < NC; ++n) {
                    us[n] = reduce_rg(us[n]);
                }
            }
#pragma unroll
            for (int ii = 0; ii < DQ; ++ii) {
                if (EXACT || ii < dq) {
                    const float wv = LINEAR || RETAIN ? decay : w[ii], av = au[ii], kv = k[ii], qv = q[ii];
#pragma unroll
                    for (int n = 0; n < NC; ++n) {
                        if constexpr (BONUS) {
                            acc[n]   = fmaf(fmaf(av, v[n], S[ii][n]), qv, acc[n]);
                            S[ii][n] = fmaf(wv, S[ii][n], kv * v[n]);
                            continue;
                        }
                        S[ii][n] = fmaf(wv, S[ii][n], DELTA ? fmaf(-av, us[n], kv * v[n]) : kv * v[n]);
                        acc[n]   = fmaf(S[ii][n], qv, acc[n]);
                    }
                }
            }
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                acc[n] = reduce_rg(acc[n]);
            }
            if (rg == (t & (RG - 1))) {
                store_out(t0 + t, acc);
            }
        }
        if (more) {
            park(t0 + tb, buf ^ 1);  // (the other buffer's readers passed the barrier that closed the previous stage)
        }
        __syncthreads();
    }
    if (wave_on) {
#pragma unroll
        for (int ii = 0; ii < DQ; ++ii) {
            if (ii < dq) {
#pragma unroll
                for (int n = 0; n < NC; ++n) {
                    slab[(ii * NC + n) * 64 + lane] = S[ii][n];
                }
            }
        }
    }
}

template<int KIND>
static void launch_state_dq(const StateMixParams& p, dim3 grid, hipStream_t st)
{
    const int  dp  = (p.dim + 7) / 8 * 8;
    constexpr bool DELTA = KIND == kStateDelta;
    auto       lds = [&](int tb) { return 2 * (size_t)tb * (state_vectors(KIND) * dp + 4 * kStateCW * kStateNC) * sizeof(float); };
    const bool one = p.max_q_len == 1;  // decoded tokens: one token per stage
#define TM_STATE_LAUNCH_TB(DQ_, TB_)                                                     \
    if (p.dim == 8 * DQ_) {                                                              \
        state_mix_kernel<DQ_, KIND, TB_, true><<<grid, 256, lds(TB_), st>>>(p);         \
    }                                                                                    \
    else {                                                                               \
        state_mix_kernel<DQ_, KIND, TB_, false><<<grid, 256, lds(TB_), st>>>(p);        \
    }
#define TM_STATE_LAUNCH(DQ_, TB_)                                             \
    if constexpr (!DELTA) { /* one token: portions take chunks */              \
        TM_STATE_LAUNCH_TB(DQ_, 1)                                            \
    }                                                                         \
    else if (one) {                                                           \
        TM_STATE_LAUNCH_TB(DQ_, 1)                                            \
    }                                                                         \
    else {                                                                    \
        TM_STATE_LAUNCH_TB(DQ_, TB_)                                          \
    }
    const int dq = dp / 8;
    if (dq <= 4) {
        TM_STATE_LAUNCH(4, 16)
    }
    else if (dq <= 8) {
        TM_STATE_LAUNCH(8, 16)
    }
    else if (dq <= 16) {
        TM_STATE_LAUNCH(16, 8)
    }
    else {
        TM_STATE_LAUNCH(32, 4)
    }
#undef TM_STATE_LAUNCH
#undef TM_STATE_LAUNCH_TB
}

// ---- linear attention with decays over prompt portions: chunks of 16 tokens on the fp32 matrix cores -------------------------------------
// Serves the forget-gate mixer (k = 1 - f), lightning attention (f = the head's decay; silu on q, k and v as they are loaded), retention (f = the head's
// decay, q and k rotated as they are loaded) and the bonus recurrence.
// 8 prompts of ~1000 tokens, 16 heads of 128 / 128, lightning: 84 + 143 us a layer; on the vector units (16 tokens at a time in LDS) 790.
// Per chunk, head and key channel d, with t, j counting tokens of the chunk and P(a..b) = prod of f_s[d] for a <= s <= b:
//   o_t = sum_d q_t P(0..t) S0[d] + sum_{j <= t} A[t][j] v_j,    A[t][j] = sum_d q_t k_j P(j+1..t)
//   S   = P(0..15) S0 + sum_j k_j P(j+1..15) v_j^T
// The bonus recurrence reads the state ahead of its token: P(0..t-1) and P(j+1..t-1) in o_t and A[t][j < t], and A[t][t] = sum_d q_t u k_t.
// Every factor is a running product of numbers in [0, 1]: nothing is divided by a decay, so gates near zero cost no precision.
//   decay_blocks_kernel: everything that does not depend on the state -- scaled queries, scaled keys, A, the chunk's whole decay -- for all
//                         chunks of the launch at once, one workgroup per (chunk, head), written in the order the second kernel's MFMA operands are read
//   decay_chunks_kernel: a wave owns 16 value columns of a head's state in MFMA accumulators and walks the sequence's chunks; the
//                         accumulator layout (row = lane / 16 * 4 + i) serves as the B operand of the query product as it is, the
//                         contraction index runs over (row tile, i) with lane group g on row 16 r + 4 g + i
// v_mfma_f32_16x16x4_f32: full 32-bit products and sums.  Block of a (chunk, head), DR = ceil(dim / 16) row tiles, floats:
//   scaled queries [DR][64 lanes][4], scaled keys [DR][64][4], A [64][4], chunk decay [DR * 16]
constexpr int kChunkT = 16;

__host__ __device__ inline int decay_tiles(int dim)  // row tiles of an instantiation
{
    const int n = (dim + 15) / 16;
    return n <= 2 ? 2 : n <= 4 ? 4 : n <= 8 ? 8 : 16;
}
__host__ __device__ constexpr int decay_block_floats_of(int dr, bool delta)  // whole pieces of 1 KB, as the DMA brings them
{
    return ((delta ? 4 : 2) * dr * 256 + (delta ? 3 : 1) * 256 + dr * 16 + 255) / 256 * 256;
}
__host__ __device__ inline size_t decay_block_floats(int dim, bool delta)
{
    return decay_block_floats_of(decay_tiles(dim), delta);
}
// chunk c of sequence s, whose first row is row0 of the launch: sequences take (rows before) / 16 + s onwards, which never overlaps
__device__ __forceinline__ size_t decay_chunk_index(int s, int row0, int c)
{
    return (size_t)(row0 / kChunkT + s + c);
}

size_t decay_workspace_floats(int rows, int nseq, int heads, int dim, bool delta)
{
    return ((size_t)rows / kChunkT + nseq + 1) * heads * decay_block_floats(dim, delta);
}

// grid (nseq * chunks, heads), 256 threads
template<int DR, int KIND>
__global__ __launch_bounds__(256) void decay_blocks_kernel(StateMixParams p, int chunks)
{
    constexpr int DP = DR * 16, LD = DP + 4, NM = (DP + 63) / 64;
    __shared__ __attribute__((aligned(16))) float sq[kChunkT * LD], sk[kChunkT * LD], sf[kChunkT * LD];
    constexpr bool FORGET = KIND == kStateForget, RETAIN = KIND == kStateRetention, BONUS = KIND == kStateBonus;
    const int s = blockIdx.x / chunks, c = blockIdx.x % chunks, h = blockIdx.y, D = p.dim, tid = threadIdx.x;
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int t0 = c * kChunkT, nt = min(kChunkT, q_len - t0);
    if (nt <= 0) {
        return;
    }
    float* out = p.blocks + (decay_chunk_index(s, row0, c) * p.heads + h) * decay_block_floats_of(DR, false);
    for (int i = tid; i < kChunkT * DP; i += 256) {
        const int  t = i / DP, d = i % DP;
        float      q = 0.f, k = 0.f, f = 1.f;  // tokens behind the portion and channels behind dim: nothing read, nothing written, nothing forgotten
        if (t < nt && d < D) {
            const size_t row = (size_t)(row0 + t0 + t);
            const float* pr  = p.proj + row * p.ld + h * D + d;
            if constexpr (FORGET) {
                const float z = pr[p.c_f] + p.f_bias[h * D + d], low = p.f_low[h * D + d];
                const float ez = expf(-fabsf(z)), hi = 1.f / (1.f + ez), lo = ez * hi;  // sigmoid(|z|), sigmoid(-|z|)
                q = sm_silu(pr[p.c_q]);
                k = (1.f - low) * (z > 0.f ? lo : hi);
                f = fmaf(1.f - low, z > 0.f ? hi : lo, low);
            }
            else if constexpr (RETAIN) {
                const Rotation ro(p, p.k_len[s] - q_len + t0 + t, d);
                q = ro(pr + p.c_q);
                k = ro(pr + p.c_k) * p.k_mult;
                f = p.decay_h[h];
            }
            else if constexpr (KIND == kStateLinear) {
                q = sm_silu(pr[p.c_q]);
                k = sm_silu(pr[p.c_k]);
                f = p.decay_h[h];
            }
            else {
                q = pr[p.c_q];
                k = pr[p.c_k];
                f = expf(-expf(p.decay_w[row * p.ld_w + h * D + d]));
            }
        }
        sq[t * LD + d] = q;
        sk[t * LD + d] = k;
        sf[t * LD + d] = f;
    }
    __syncthreads();
    {   // A[t][j]: 16 lanes share a key j, each with its channels; the key decays as t moves on
        const int j = tid >> 4, sl = tid & 15;
        floatx4   w[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int d = m * 64 + sl * 4;
            w[m]        = d < DP ? *(const floatx4*)(sk + j * LD + d) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
        float* A = out + DR * 64 * 4 * 2;
#pragma unroll
        for (int t = 0; t < kChunkT; ++t) {
            float dot = 0.f;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const int d = m * 64 + sl * 4;
                if (d < DP) {
                    const floatx4 q = *(const floatx4*)(sq + t * LD + d), f = *(const floatx4*)(sf + t * LD + d);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (BONUS) {  // the key meets its own token through the bonus, and decays behind each later one
                            dot = fmaf(q[i], t == j && d + i < D ? w[m][i] * p.bonus[h * D + d + i] : w[m][i], dot);
                            w[m][i] *= t > j ? f[i] : 1.f;
                        }
                        else {
                            w[m][i] *= t > j ? f[i] : 1.f;
                            dot = fmaf(q[i], w[m][i], dot);
                        }
                    }
                }
            }
            dot = group_sum<16>(dot);
            if (sl == t) {
                A[((j >> 2) * 16 + t) * 4 + (j & 3)] = t >= j ? dot : 0.f;  // operand order: lane = (j / 4) * 16 + t, element j % 4
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < 2 * DP; i += 256) {  // running products down the tokens (queries) and up (keys)
        const int d = i % DP;
        float     run = 1.f;
        if (i < DP) {
#pragma unroll
            for (int t = 0; t < kChunkT; ++t) {
                if constexpr (BONUS) {
                    sq[t * LD + d] *= run;
                    run *= sf[t * LD + d];
                }
                else {
                    run *= sf[t * LD + d];
                    sq[t * LD + d] *= run;
                }
            }
            out[DR * 64 * 4 * 2 + 256 + d] = run;
        }
        else {
#pragma unroll
            for (int t = kChunkT - 1; t >= 0; --t) {
                sk[t * LD + d] *= run;
                run *= sf[t * LD + d];
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < DR * 64; i += 256) {
        const int r = i >> 6, l = i & 63;
        *(floatx4*)(out + (size_t)i * 4) = *(const floatx4*)(sq + (l & 15) * LD + r * 16 + (l >> 4) * 4);
        floatx4 k;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            k[e] = sk[((l >> 4) * 4 + e) * LD + r * 16 + (l & 15)];
        }
        *(floatx4*)(out + (size_t)(DR * 64 + i) * 4) = k;
    }
}

// The delta rule, S_t = diag(w_t) S - b_t e_t + k_t v_t^T with b = a u and e_t = S^T u_t (S as the token finds it).  With
//   U0[t] = u_t P(0..t-1),   Auk[t][j < t] = sum_d u_t k_j P(j+1..t-1),   Aub likewise,   Aqk[t][j <= t] = sum_d q_t k_j P(j+1..t),   Aqb likewise
// the e of a chunk solve (I + Aub) E = U0 S0 + Auk V, and
//   o = Q0 S0 + Aqk V - Aqb E,   S = P(0..15) S0 + K1^T V - B1^T E      (Q0, K1 and B1 with their running products as above).
// Aub is strictly lower triangular: (I + Aub)^-1 is applied to the columns of U0 and Auk by forward substitution here, a column a thread, so that the walk
// over the chunks has E by products alone.  The substitution is the recurrence itself on those columns, token after token, and grows as that does: with |u| <= 1 and rates and
// decays in [0, 1] a factor diag(w) - b u^T may lengthen a vector where the rates differ from channel to channel, by 2 / sqrt 3 at most, and does not where they are alike.
// Block: as above, then U [DR][64][4], B1 [DR][64][4], Aqb [64][4], W = (I + Aub)^-1 Auk [64][4].  Dynamic LDS: delta_blocks_lds(DR)
constexpr int delta_blocks_lds(int dr)
{
    return (5 * kChunkT * (dr * 16 + 4) + 2 * kChunkT * kChunkT) * 4;
}
// RAW: key, removal-rate logits and decay logits come as the projections left them and are turned here as delta_prep_kernel turns them (8 x ~970 tokens, 16 heads of
// 128: 94 us of that launch and 236 of this one, 261 together)
template<int DR, bool RAW>
__global__ __launch_bounds__(256) void delta_blocks_kernel(StateMixParams p, int chunks)
{
    constexpr int DP = DR * 16, LD = DP + 4, NM = (DP + 63) / 64;
    extern __shared__ __attribute__((aligned(16))) float delta_lds[];
    float *sq = delta_lds, *sk = sq + kChunkT * LD, *sf = sk + kChunkT * LD, *sb = sf + kChunkT * LD, *su = sb + kChunkT * LD;
    float *ab = su + kChunkT * LD, *wk = ab + kChunkT * kChunkT;  // Aub, Auk [t][j]
    const int s = blockIdx.x / chunks, c = blockIdx.x % chunks, h = blockIdx.y, D = p.dim, tid = threadIdx.x;
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int t0 = c * kChunkT, nt = min(kChunkT, q_len - t0);
    if (nt <= 0) {
        return;
    }
    float* out = p.blocks + (decay_chunk_index(s, row0, c) * p.heads + h) * decay_block_floats_of(DR, true);
    float *oA = out + DR * 512, *oF = oA + 256, *oU = oF + DP, *oB = oU + DR * 256, *oAb = oB + DR * 256, *oW = oAb + 256;
    for (int i = tid; i < kChunkT * DP; i += 256) {
        const int  t = i / DP, d = i % DP;
        const bool ok = t < nt && d < D;  // tokens behind the portion and channels behind dim read, write and forget nothing
        const size_t row = (size_t)(row0 + t0 + (ok ? t : 0));
        const float* pr  = p.proj + row * p.ld + h * D + (ok ? d : 0);
        sq[t * LD + d] = ok ? pr[p.c_q] : 0.f;
        sk[t * LD + d] = ok ? pr[p.c_k] : 0.f;
        sb[t * LD + d] = ok ? pr[p.c_a] : 0.f;
        sf[t * LD + d] = ok ? p.decay_w[row * p.ld_w + h * D + d] : 1.f;
        if constexpr (!RAW) {
            su[t * LD + d] = ok ? p.unit[row * p.ld_u + h * D + d] : 0.f;
        }
    }
    __syncthreads();
    if constexpr (RAW) {
        const int t = tid >> 4, sl = tid & 15;  // 16 lanes a token
        float     ss = 0.f;
        for (int d = sl; d < DP; d += 16) {
            ss = fmaf(sk[t * LD + d], sk[t * LD + d], ss);
        }
        const float inv = 1.0f / sqrtf(group_sum<16>(ss) + 1e-6f);
        for (int d = sl; d < DP; d += 16) {
            const float u  = sk[t * LD + d] * inv;
            su[t * LD + d] = u;
            sb[t * LD + d] = delta_rate(u, sb[t * LD + d]);
            sf[t * LD + d] = t < nt && d < D ? delta_decay(sf[t * LD + d]) : 1.f;
        }
        __syncthreads();
    }
    {   // the four A: 16 lanes share a key j, each with its channels; the key and b decay as t moves on
        const int j = tid >> 4, sl = tid & 15;
        floatx4   k[NM], b[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int d = m * 64 + sl * 4;
            k[m]        = d < DP ? *(const floatx4*)(sk + j * LD + d) : floatx4{0.f, 0.f, 0.f, 0.f};
            b[m]        = d < DP ? *(const floatx4*)(sb + j * LD + d) : floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll 4
        for (int t = 0; t < kChunkT; ++t) {
            float uk = 0.f, ub = 0.f, qk = 0.f, qb = 0.f;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const int d = m * 64 + sl * 4;
                if (d < DP) {
                    const floatx4 q = *(const floatx4*)(sq + t * LD + d), f = *(const floatx4*)(sf + t * LD + d), u = *(const floatx4*)(su + t * LD + d);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uk = fmaf(u[i], k[m][i], uk);
                        ub = fmaf(u[i], b[m][i], ub);
                        const float w = t > j ? f[i] : 1.f;
                        k[m][i] *= w;
                        b[m][i] *= w;
                        qk = fmaf(q[i], k[m][i], qk);
                        qb = fmaf(q[i], b[m][i], qb);
                    }
                }
            }
            uk = group_sum<16>(uk), ub = group_sum<16>(ub), qk = group_sum<16>(qk), qb = group_sum<16>(qb);
            if (sl == t) {
                const int at = ((j >> 2) * 16 + t) * 4 + (j & 3);  // operand order: lane = (j / 4) * 16 + t, element j % 4
                oA[at]              = t >= j ? qk : 0.f;
                oAb[at]             = t >= j ? qb : 0.f;
                wk[t * kChunkT + j] = t > j ? uk : 0.f;
                ab[t * kChunkT + j] = t > j ? ub : 0.f;
            }
        }
    }
    __syncthreads();
    auto substitute = [&](float (&x)[kChunkT]) {  // (I + Aub) x = right side, in place
#pragma unroll
        for (int t = 1; t < kChunkT; ++t) {
            float r = x[t];
#pragma unroll
            for (int j = 0; j < t; ++j) {
                r = fmaf(-ab[t * kChunkT + j], x[j], r);
            }
            x[t] = r;
        }
    };
    for (int i = tid; i < 2 * DP; i += 256) {  // running products down the tokens (queries, u) and up (keys, b); the solution's columns
        const int d = i % DP;
        float     run = 1.f, x[kChunkT];
        if (i < DP) {
#pragma unroll
            for (int t = 0; t < kChunkT; ++t) {
                x[t] = su[t * LD + d] * run;
                run *= sf[t * LD + d];
                sq[t * LD + d] *= run;
            }
            oF[d] = run;
            substitute(x);
#pragma unroll
            for (int t = 0; t < kChunkT; ++t) {
                su[t * LD + d] = x[t];
            }
        }
        else {
#pragma unroll
            for (int t = kChunkT - 1; t >= 0; --t) {
                sk[t * LD + d] *= run;
                sb[t * LD + d] *= run;
                run *= sf[t * LD + d];
            }
            if (d < kChunkT) {
#pragma unroll
                for (int t = 0; t < kChunkT; ++t) {
                    x[t] = wk[t * kChunkT + d];
                }
                substitute(x);
#pragma unroll
                for (int t = 0; t < kChunkT; ++t) {
                    wk[t * kChunkT + d] = x[t];
                }
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < DR * 64; i += 256) {
        const int r = i >> 6, l = i & 63, row = (l & 15) * LD + r * 16 + (l >> 4) * 4;
        *(floatx4*)(out + (size_t)i * 4) = *(const floatx4*)(sq + row);
        *(floatx4*)(oU + (size_t)i * 4)  = *(const floatx4*)(su + row);
        floatx4 k, b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            k[e] = sk[((l >> 4) * 4 + e) * LD + r * 16 + (l & 15)];
            b[e] = sb[((l >> 4) * 4 + e) * LD + r * 16 + (l & 15)];
        }
        *(floatx4*)(out + (size_t)(DR * 64 + i) * 4) = k;
        *(floatx4*)(oB + (size_t)i * 4)              = b;
    }
    if (tid < 64) {
        *(floatx4*)(oW + tid * 4) = *(const floatx4*)(wk + (tid & 15) * kChunkT + (tid >> 4) * 4);
    }
}

// grid (nseq, heads, ceil(vdim / 64)), 384 threads: waves 0 - 3 -> 16 value columns each, waves 4 and 5 bring blocks and values into LDS by DMA, a ring of stages
// deep.  SILU: on the values; DELTA: blocks of delta_blocks_kernel.  The walk is as long as the longest prompt, with one wave a SIMD for the products: what
// bounds it is that wave's issue slots, so the products' waves do nothing else (with their own share of the DMA, about sixty instructions a chunk for addresses,
// lightning took 180 us and the delta rule 287).  8 prompts of ~1000 tokens, 16 heads of 128 / 128: lightning 190 us -> 143, the delta rule 226 (with its
// blocks and what prepares them 487; a token at a time on the vector units 1184)
constexpr int kValueStage = kChunkT * 64;  // floats of the workgroup's 64 value columns
constexpr int decay_chunk_stages(int dr, bool delta)
{
    return dr > 8 && delta ? 2 : 3;
}
constexpr int decay_chunks_lds(int dr, bool delta)
{
    return decay_chunk_stages(dr, delta) * (decay_block_floats_of(dr, delta) + kValueStage) * 4;
}
// 64 consecutive words of LDS from 64 addresses
__device__ __forceinline__ void chunk_dma4(__amdgpu_buffer_rsrc_t rs, int voff, unsigned lds)
{
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "buffer_load_dword %1, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(voff), "s"(lds), "s"(rs)
                 : "memory");
}
template<int DR, bool SILU, bool DELTA>
__global__ __launch_bounds__(384) void decay_chunks_kernel(StateMixParams p)
{
    constexpr int NC = kStateNC, WV = kStateCW * kStateNC, BF = decay_block_floats_of(DR, DELTA), DP = DR * 16, NB = decay_chunk_stages(DR, DELTA);
    extern __shared__ __attribute__((aligned(16))) char chunk_lds[];
    const int s = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int D = p.dim, V = p.vdim, dq = (D + 7) / 8, ncb = (V + WV - 1) / WV, cb = blockIdx.z * 4 + wave;
    const bool wave_on = wave < 4 && cb < ncb;
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int pos0 = p.k_len[s] - q_len, g = lane >> 4, col = cb * 16 + (lane & 15);
    int       slot = p.seq_slot ? p.seq_slot[s] : p.slot0 + s;
    if (p.active && !p.active[s]) {
        slot = p.park_slot;
    }
    float* slab = p.state + (size_t)slot * p.slot_stride + p.layer_offset + ((size_t)h * ncb + (wave_on ? cb : 0)) * dq * 64 * NC;
    // element (d, column) of the slab as state_mix_kernel keeps it
    auto at = [&](int d) { return ((d % dq) * NC + (lane & 15) % NC) * 64 + d / dq * kStateCW + (lane & 15) / NC; };
    floatx4 S[DR];
#pragma unroll
    for (int r = 0; r < DR; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = r * 16 + g * 4 + i;
            S[r][i]     = wave_on && pos0 > 0 && d < D ? slab[at(d)] : 0.f;
        }
    }
    const int    chunks = (q_len + kChunkT - 1) / kChunkT;
    const float* blk    = p.blocks + (decay_chunk_index(s, row0, 0) * p.heads + h) * BF;
    const size_t next   = (size_t)p.heads * BF;
    const float* val    = p.proj + (size_t)row0 * p.ld + p.c_v + h * V;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)chunk_lds);
    const int      vcol = min((int)blockIdx.z * 64 + lane, V - 1) * 4;
    constexpr int  kStage = (BF + kValueStage) * 4, kPieces = BF / 256, kOps = kPieces / 2 + kChunkT / 2;  // bytes; pieces of 1 KB; the fewest operations of a wave
    auto dma = [&](int c) {  // waves 4, 5: every other piece, every other token
        const unsigned dst = lds0 + __builtin_amdgcn_readfirstlane(c % NB * kStage);
        const auto     rs  = __builtin_amdgcn_make_buffer_rsrc((void*)(blk + (size_t)c * next), 0, BF * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < kPieces; i += 2) {
            const int at = __builtin_amdgcn_readfirstlane((i + wave - 4) * 1024);
            if (at < BF * 4) {
                stream_dma16(rs, lane * 16, at, dst + at);
            }
        }
        const int  last = min(kChunkT, q_len - c * kChunkT) - 1;  // (keys behind the portion are zero: any finite value will do)
        const auto rv   = __builtin_amdgcn_make_buffer_rsrc((void*)(val + (size_t)c * kChunkT * p.ld), 0, (last * p.ld + V) * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < kChunkT; i += 2) {
            const int t = __builtin_amdgcn_readfirstlane(i + wave - 4);
            chunk_dma4(rv, min(t, last) * p.ld * 4 + vcol, dst + BF * 4 + t * 256);
        }
    };
    float* out  = p.out + (size_t)(row0 + g * 4) * p.ldo + h * V + col;
    auto   step = [&](const float* b, floatx4 vv, int t0) {
        auto    lane4 = [&](int at) { return *(const floatx4*)(b + at + lane * 4); };
        const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
        floatx4       add[DR], y[4], z[4], ya[2], yb[2];  // short chains of sums: independent products for the matrix core and less rounding
        auto outer = [&](int at, const floatx4& x) {  // add += (scaled keys at `at`)^T x: neighbouring products meet different sums
            floatx4 k[DR];
#pragma unroll
            for (int r = 0; r < DR; ++r) {
                k[r] = lane4(at + r * 256);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int r = 0; r < DR; ++r) {
                    add[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[r][e], x[e], add[r], 0, 0, 0);
                }
            }
        };
        auto inner = [&](floatx4 (&o)[2], int at, const floatx4& x) {  // o += (triangle at `at`) x
            const floatx4 a = lane4(at);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], x[e], o[e & 1], 0, 0, 0);
            }
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            y[i] = z[i] = ya[i & 1] = yb[i & 1] = zero;
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {
            add[r] = zero;
        }
        constexpr int oA = DR * 512, oF = oA + 256, oU = oF + DP, oB = oU + DR * 256, oAb = oB + DR * 256, oW = oAb + 256;
        if constexpr (DELTA) {
            const floatx4 w = lane4(oW);
#pragma unroll
            for (int r = 0; r < DR; ++r) {
                const floatx4 u = lane4(oU + r * 256);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    z[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[i], S[r][i], z[i], 0, 0, 0);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                z[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], vv[e], z[e], 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {  // (vector work between the products, which take 32 cycles each)
            const floatx4 q = lane4(r * 256);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                y[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i], S[r][i], y[i], 0, 0, 0);
            }
            if constexpr (SILU) {
#pragma unroll
                for (int e = r * 4 / DR; e < (r + 1) * 4 / DR; ++e) {
                    vv[e] = sm_silu(vv[e]);
                }
            }
        }
        inner(ya, oA, vv);
        outer(DR * 256, vv);
        if constexpr (DELTA) {
            const floatx4 e = -((z[0] + z[1]) + (z[2] + z[3]));
            inner(yb, oAb, e);
            outer(oB, e);
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {  // (one rounding of the state a chunk)
            const floatx4 f = *(const floatx4*)(b + oF + r * 16 + g * 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                S[r][i] = fmaf(S[r][i], f[i], add[r][i]);
            }
        }
        const floatx4 sum = ((y[0] + y[1]) + (y[2] + y[3])) + ((ya[0] + ya[1]) + (yb[0] + yb[1]));
        float* o = out + (size_t)t0 * p.ldo;
        if (col < V) {
            if (t0 + kChunkT <= q_len) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[i * p.ldo] = sum[i];
                }
            }
            else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (t0 + g * 4 + i < q_len) {
                        o[i * p.ldo] = sum[i];
                    }
                }
            }
        }
    };
    if (wave >= 4) {
        for (int c = 0; c < NB - 1 && c < chunks; ++c) {
            dma(c);
        }
        for (int c = 0; c < chunks; ++c) {
            if (NB > 2 && c + NB - 2 < chunks) {  // the stages behind this one may still be on their way
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * kOps) : "memory");
            }
            else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            __syncthreads();  // stage c has landed, and nobody reads the stage before it any more
            if (c + NB - 1 < chunks) {
                dma(c + NB - 1);
            }
        }
        return;
    }
    for (int c = 0; c < chunks; ++c) {
        __syncthreads();
        if (wave_on) {
            const float* b = (const float*)chunk_lds + c % NB * (kStage / 4);
            floatx4      v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = b[BF + (g * 4 + e) * 64 + wave * 16 + (lane & 15)];
            }
            step(b, v, c * kChunkT);
        }
    }
    if (!wave_on) {
        return;
    }
#pragma unroll
    for (int r = 0; r < DR; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = r * 16 + g * 4 + i;
            if (d < dq * 8) {  // (the slab's padding rows are stored as the zeros they are)
                slab[at(d)] = S[r][i];
            }
        }
    }
}

// The walk of short portions (at most 128 channels; not the delta rule): as above, without LDS.  Each wave fetches its own operands, the next chunk's under this chunk's products:
// nothing has to come through two barriers first, and more workgroups fit on a CU.  us with the blocks, this / the one above, forget gate, 16 heads of 128: one portion of 20
// tokens 18.7 / 20.5, of 33 21.0 / 21.9, of 64 23.1 / 23.2, of 1000 156 / 108; 32 portions of 20 53 / 62; 32 heads of 32, 32 portions of 64 30 / 35, of 256 85 / 90.
// grid (nseq, heads, ceil(vdim / 64)), 256 threads: wave -> 16 value columns; SILU: on the values
template<int DR, bool SILU>
__global__ __launch_bounds__(256) void decay_chunks_short_kernel(StateMixParams p)
{
    constexpr int NC = kStateNC, WV = kStateCW * kStateNC;
    const int s = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, cb = blockIdx.z * 4 + (threadIdx.x >> 6);
    const int D = p.dim, V = p.vdim, dq = (D + 7) / 8, ncb = (V + WV - 1) / WV;
    if (cb >= ncb) {
        return;
    }
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int pos0 = p.k_len[s] - q_len, g = lane >> 4, col = cb * 16 + (lane & 15);
    int       slot = p.seq_slot ? p.seq_slot[s] : p.slot0 + s;
    if (p.active && !p.active[s]) {
        slot = p.park_slot;
    }
    float* slab = p.state + (size_t)slot * p.slot_stride + p.layer_offset + ((size_t)h * ncb + cb) * dq * 64 * NC;
    // element (d, column) of the slab as state_mix_kernel keeps it
    auto at = [&](int d) { return ((d % dq) * NC + (lane & 15) % NC) * 64 + d / dq * kStateCW + (lane & 15) / NC; };
    floatx4 S[DR];
#pragma unroll
    for (int r = 0; r < DR; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = r * 16 + g * 4 + i;
            S[r][i]     = pos0 > 0 && d < D ? slab[at(d)] : 0.f;
        }
    }
    constexpr size_t bf = decay_block_floats_of(DR, false);
    const float* blk = p.blocks + (decay_chunk_index(s, row0, 0) * p.heads + h) * bf;
    struct Operands {
        floatx4 q[DR], k[DR], f[DR], a, v;
    };
    auto fetch = [&](Operands& o, int t0, const float* b) {
#pragma unroll
        for (int r = 0; r < DR; ++r) {
            o.q[r] = *(const floatx4*)(b + (size_t)(r * 64 + lane) * 4);
            o.k[r] = *(const floatx4*)(b + (size_t)((DR + r) * 64 + lane) * 4);
            o.f[r] = *(const floatx4*)(b + DR * 64 * 4 * 2 + 256 + r * 16 + g * 4);
        }
        o.a = *(const floatx4*)(b + DR * 64 * 4 * 2 + lane * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = min(t0 + g * 4 + e, q_len - 1);  // (keys behind the portion are zero: any finite value will do)
            o.v[e]      = p.proj[(size_t)(row0 + t) * p.ld + p.c_v + h * V + min(col, V - 1)];
        }
    };
    auto step = [&](Operands& o, int t0) {
        if constexpr (SILU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o.v[e] = sm_silu(o.v[e]);
            }
        }
        floatx4 y[4], ya = {0.f, 0.f, 0.f, 0.f};  // short chains of sums: independent products for the matrix core and less rounding
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            y[i] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                y[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[r][i], S[r][i], y[i], 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            ya = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[e], o.v[e], ya, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < DR; ++r) {
            S[r] *= o.f[r];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int r = 0; r < DR; ++r) {
                S[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[r][e], o.v[e], S[r], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + g * 4 + i;
            if (t < q_len && col < V) {
                p.out[(size_t)(row0 + t) * p.ldo + h * V + col] = ((y[0][i] + y[1][i]) + (y[2][i] + y[3][i])) + ya[i];
            }
        }
    };
    const size_t next = (size_t)p.heads * bf;
    Operands a, b;
    if (q_len > 0) {
        fetch(a, 0, blk);
    }
    for (int t0 = 0; t0 < q_len; t0 += 2 * kChunkT, blk += 2 * next) {
        const bool more = t0 + kChunkT < q_len;
        if (more) {
            fetch(b, t0 + kChunkT, blk + next);
        }
        step(a, t0);
        if (t0 + 2 * kChunkT < q_len) {
            fetch(a, t0 + 2 * kChunkT, blk + 2 * next);
        }
        if (more) {
            step(b, t0 + kChunkT);
        }
    }
#pragma unroll
    for (int r = 0; r < DR; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = r * 16 + g * 4 + i;
            if (d < dq * 8) {  // (the slab's padding rows are stored as the zeros they are)
                slab[at(d)] = S[r][i];
            }
        }
    }
}

// Up to three chunks, and heads of few channels that fill the chip several times over, whose blocks are small against what the other walk's stages take of a CU
bool state_mix_short(const StateMixParams& p)
{
    return decay_tiles(p.dim) <= 8 && (p.max_q_len <= 3 * kChunkT || (decay_tiles(p.dim) == 2 && (int64_t)p.nseq * p.heads * ((p.vdim + 63) / 64) >= 1024));
}

template<int DR, int KIND>
static int launch_decay_chunks_dr(const StateMixParams& p, hipStream_t st)
{
    constexpr bool DELTA = KIND == kStateDelta;
    constexpr int  lds    = decay_chunks_lds(DR, DELTA);
    const int      chunks = (p.max_q_len + kChunkT - 1) / kChunkT;
    const dim3     gb(p.nseq * chunks, p.heads), gc(p.nseq, p.heads, (p.vdim + 63) / 64);
    if constexpr (DELTA) {
        const auto blocks = p.raw ? delta_blocks_kernel<DR, true> : delta_blocks_kernel<DR, false>;
        if (const int rc = ensure_dynamic_lds((const void*)blocks, delta_blocks_lds(DR))) {
            return rc;
        }
        blocks<<<gb, 256, delta_blocks_lds(DR), st>>>(p, chunks);
    }
    else {
        decay_blocks_kernel<DR, KIND><<<gb, 256, 0, st>>>(p, chunks);
        if constexpr (DR <= 8) {
            if (state_mix_short(p)) {
                decay_chunks_short_kernel<DR, KIND == kStateLinear><<<gc, 256, 0, st>>>(p);
                TM_HIP_CHECK(hipGetLastError());
                return 0;
            }
        }
    }
    const auto k = decay_chunks_kernel<DR, KIND == kStateLinear, DELTA>;
    if (const int rc = ensure_dynamic_lds((const void*)k, lds)) {
        return rc;
    }
    k<<<gc, 384, lds, st>>>(p);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<int KIND>
static int launch_decay_chunks(const StateMixParams& p, hipStream_t st)
{
    TM_REQUIRE(p.blocks && p.blocks_floats >= decay_workspace_floats(p.rows, p.nseq, p.heads, p.dim, KIND == kStateDelta), "state mixer: chunk workspace");
    switch (decay_tiles(p.dim)) {
        case 2: return launch_decay_chunks_dr<2, KIND>(p, st);
        case 4: return launch_decay_chunks_dr<4, KIND>(p, st);
        case 8: return launch_decay_chunks_dr<8, KIND>(p, st);
        default: return launch_decay_chunks_dr<16, KIND>(p, st);
    }
}

// Portions of the delta rule in chunks, or walked token by token.  A few heads x sequences leave the walk a chain of tokens, which chunks shorten; where there are enough of
// them to fill the chip the walk is bound by its work, and chunks do about as much of it and more for the last, part-filled one.  A model of both in microseconds, fitted
// to 800 sizes (32 ... 256 channels, 2 ... 2048 heads x sequences, 33 ... 1000 tokens): what it takes is at most 6 % slower than the walk and 1.4 % slower than the better one on average.  us, walk with the launch
// that prepares its operands / chunks: 128 channels, 16 heads, one prompt of 33 tokens 35 / 31, 8 of 1000 974 / 411, 32 of 33 85 / 111, 32 of 64 146 / 137; 256 channels, 32 heads, 32 of
// 33 530 / 881, of 64 1005 / 1136, of 256 3890 / 3855.  Up to 32 tokens it was never chunks (one prompt of 32 29 / 31).  Without logits (raw: 0) the operands are prepared either way.
bool state_mix_chunks(const StateMixParams& p)
{
    if (p.max_q_len <= 2 * kChunkT) {
        return false;
    }
    const double rows = p.rows > 0 ? p.rows : (double)p.nseq * p.max_q_len, state = (double)p.dim * p.vdim;
    const double walk = 5 + std::max((0.31 + 0.005 * p.dim) * p.max_q_len, (0.00055 + 2.1e-7 * state) * p.heads * rows)
                        - (p.raw ? 0.0 : 2 + 5e-6 * p.heads * rows * p.dim);
    const int    chunks = (p.max_q_len + kChunkT - 1) / kChunkT, dp = decay_tiles(p.dim) * 16;
    const double whole = std::min((double)p.nseq * chunks * kChunkT, rows + (kChunkT - 1.0) * p.nseq), tile = (double)dp * std::max(p.vdim, dp / 2);
    const double blocks = 9.9 + 0.081 * dp + std::max((0.035 + 0.0013 * dp) * chunks * kChunkT, (0.00038 + 1.6e-7 * tile) * p.heads * whole) + 3.3e-6 * p.heads * p.nseq * tile;
    return 1.12 * blocks < walk;
}

int launch_state_mix(const StateMixParams& p, int kind, hipStream_t st)
{
    TM_REQUIRE(p.nseq >= 0 && p.heads >= 1 && p.dim >= 1 && p.dim <= 256 && p.vdim >= 1 && p.max_q_len >= 1, "state mixer: sizes (dim <= 256)");
    TM_REQUIRE(p.cu_q && p.k_len && p.state && p.proj && p.out && p.ld >= 1 && p.ldo >= p.heads * p.vdim, "state mixer: operands");
    TM_REQUIRE(kind == kStateDelta ? (p.decay_w && p.ld_w >= p.heads * p.dim && (p.raw || (p.unit && p.ld_u >= p.heads * p.dim))) :
               kind == kStateForget ? (p.f_bias && p.f_low) :
               kind == kStateBonus ? (p.decay_w && p.bonus && p.ld_w >= p.heads * p.dim) : ((kind == kStateLinear || kind == kStateRetention) && p.decay_h),
               "state mixer: decay operands");
    if (p.nseq == 0) {
        return 0;
    }
    TM_REQUIRE(kind != kStateRetention || (p.rot_dims >= 0 && p.rot_dims % 2 == 0 && p.rot_dims <= p.dim && (p.rot_dims == 0 || p.inv_freq)),
               "state mixer: rotation");
    if (p.max_q_len > 1 && kind == kStateLinear) {
        return launch_decay_chunks<kStateLinear>(p, st);
    }
    if (p.max_q_len > 1 && kind == kStateForget) {
        return launch_decay_chunks<kStateForget>(p, st);
    }
    if (p.max_q_len > 1 && kind == kStateRetention) {
        return launch_decay_chunks<kStateRetention>(p, st);
    }
    if (p.max_q_len > 1 && kind == kStateBonus) {
        return launch_decay_chunks<kStateBonus>(p, st);
    }
    TM_REQUIRE(!p.raw || (kind == kStateDelta && state_mix_chunks(p)), "state mixer: logits only for chunks of the delta rule");
    if (kind == kStateDelta && state_mix_chunks(p)) {
        return launch_decay_chunks<kStateDelta>(p, st);
    }
    const int  wcols = 4 * kStateCW * kStateNC;  // value columns of a workgroup
    const dim3 grid(p.nseq, p.heads, (p.vdim + wcols - 1) / wcols);
    if (kind == kStateDelta) {
        launch_state_dq<kStateDelta>(p, grid, st);
    }
    else if (kind == kStateForget) {
        launch_state_dq<kStateForget>(p, grid, st);
    }
    else if (kind == kStateRetention) {
        launch_state_dq<kStateRetention>(p, grid, st);
    }
    else if (kind == kStateBonus) {
        launch_state_dq<kStateBonus>(p, grid, st);
    }
    else {
        launch_state_dq<kStateLinear>(p, grid, st);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// delta rule, per (row, head): the fused projection's key, removal-rate logits and the decay logits become what the recurrence reads --
//   unit[row][h d]  = u = k / sqrt(sum k^2 + 1e-6)
//   proj[.. c_a ..] = sigmoid(logit) * u            (in place)
//   decay[row][h d] = exp(-e^(-1/2) sigmoid(logit)) (in place)
__global__ __launch_bounds__(256) void delta_prep_kernel(float* __restrict__ proj, int ld, int c_k, int c_a, float* __restrict__ decay, int ld_w,
                                                         float* __restrict__ unit, int ld_u, int H, int D)
{
    const int t = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= H) {
        return;
    }
    float*       pr = proj + (size_t)t * ld;
    const float* k  = pr + c_k + h * D;
    float        ss = 0.f;
    for (int i = lane; i < D; i += 64) {
        ss = fmaf(k[i], k[i], ss);
    }
    const float inv = 1.0f / sqrtf(group_sum<64>(ss) + 1e-6f);
    for (int i = lane; i < D; i += 64) {
        const float u  = k[i] * inv;
        float&      a  = pr[c_a + h * D + i];
        float&      w  = decay[(size_t)t * ld_w + h * D + i];
        a              = delta_rate(u, a);
        w              = delta_decay(w);
        unit[(size_t)t * ld_u + h * D + i] = u;
    }
}

int launch_delta_prep(float* proj, int ld, int c_k, int c_a, float* decay, int ld_w, float* unit, int ld_u, int rows, int heads, int dim,
                      hipStream_t st)
{
    TM_REQUIRE(proj && decay && unit && heads >= 1 && dim >= 1, "delta prep: operands");
    if (rows == 0) {
        return 0;
    }
    delta_prep_kernel<<<dim3(rows, (heads + 3) / 4), 256, 0, st>>>(proj, ld, c_k, c_a, decay, ld_w, unit, ld_u, heads, dim);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// gated delta rule: one wave per (row, head) turns the convolved queries / keys and the decay logits into the vectors of the recurrence
__global__ __launch_bounds__(256) void gdelta_prep_kernel(float* __restrict__ src, int ld, int c_q, int c_k, int c_qo, int c_ko,
                                                          const float* __restrict__ beta_logit, int ld_b, float* __restrict__ decay, int ld_w,
                                                          const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                                                          float* __restrict__ unit, int ld_u, int H, int G, int D)
{
    const int t = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= H) {
        return;
    }
    const int    c  = h / (H / G);
    float*       pr = src + (size_t)t * ld;
    const float *q = pr + c_q + c * D, *k = pr + c_k + c * D;
    float        sq = 0.f, sk = 0.f;
    for (int i = lane; i < D; i += 64) {
        sq = fmaf(q[i], q[i], sq);
        sk = fmaf(k[i], k[i], sk);
    }
    const float qinv = 1.0f / (sqrtf(group_sum<64>(sq) + 1e-6f) * sqrtf((float)D));
    const float kinv = 1.0f / sqrtf(group_sum<64>(sk) + 1e-6f);
    const float beta = 1.f / (1.f + expf(-beta_logit[(size_t)t * ld_b + h]));
    const float A    = expf(a_log[h]);
    for (int i = lane; i < D; i += 64) {
        const float ku = k[i] * kinv;
        float&      w  = decay[(size_t)t * ld_w + h * D + i];
        const float z  = w + (dt_bias ? dt_bias[h * D + i] : 0.f);
        const float g  = expf(-A * (z > 20.f ? z : log1pf(expf(z))));
        w                                  = g;
        pr[c_qo + h * D + i]               = q[i] * qinv;
        pr[c_ko + h * D + i]               = beta * ku;
        unit[(size_t)t * ld_u + h * D + i] = g * ku;
    }
}

int launch_gdelta_prep(float* src, int ld, int c_q, int c_k, int c_qo, int c_ko, const float* beta_logit, int ld_b, float* decay, int ld_w,
                       const float* a_log, const float* dt_bias, float* unit, int ld_u, int rows, int heads, int kv_heads, int dim, hipStream_t st)
{
    TM_REQUIRE(src && beta_logit && decay && a_log && unit && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0 && dim >= 1, "gdelta prep: operands");
    TM_REQUIRE(c_qo >= c_q + kv_heads * dim && c_qo >= c_k + kv_heads * dim && c_ko >= c_qo + heads * dim && ld >= c_ko + heads * dim,
               "gdelta prep: the per-head vectors lie behind the convolved ones");
    if (rows == 0) {
        return 0;
    }
    gdelta_prep_kernel<<<dim3(rows, (heads + 3) / 4), 256, 0, st>>>(src, ld, c_q, c_k, c_qo, c_ko, beta_logit, ld_b, decay, ld_w, a_log, dt_bias, unit,
                                                                    ld_u, heads, kv_heads, dim);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// short causal convolution: thread = (sequence, channel, segment of kConvSeg rows); it keeps the last taps - 1 inputs in registers, so every
// input is read once.  A segment's first rows read the rows before it from x (x is not written: the output goes elsewhere) or, before the
// launch's first row, from the sequence's state; the thread of segment 0 then stores the state's new content -- nobody else touches it.
// MT: register window, taps <= MT; weights are right-aligned in it (unused taps weigh zero)
constexpr int kConvSeg = 64;

template<int MT>
__global__ __launch_bounds__(256) void short_conv_kernel(float* __restrict__ y, int ldy, const float* __restrict__ x, int ldx, int x_col,
                                                         const float* __restrict__ w, int C, int taps, int act, StateMixParams p)
{
    const int s = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x, seg = blockIdx.z;
    const int row0 = p.cu_q[s] - p.cu_q[0], q_len = p.cu_q[s + 1] - p.cu_q[s];
    const int t0 = seg * kConvSeg, t1 = min(q_len, t0 + kConvSeg);
    if (c >= C || (t0 >= q_len && seg > 0)) {
        return;
    }
    const int pos0 = p.k_len[s] - q_len, nh = taps - 1;
    int       slot = p.seq_slot ? p.seq_slot[s] : p.slot0 + s;
    if (p.active && !p.active[s]) {
        slot = p.park_slot;
    }
    float* st = p.state + (size_t)slot * p.slot_stride + p.layer_offset;  // [taps - 1][C]
    // input at row t of the launch's rows of this sequence (t < 0: history)
    auto input = [&](int t) -> float {
        if (t >= 0) {
            return x[(size_t)(row0 + t) * ldx + x_col + c];
        }
        return (pos0 > 0 && t + nh >= 0) ? st[(size_t)(t + nh) * C + c] : 0.f;
    };
    float wt[MT], win[MT - 1];
#pragma unroll
    for (int k = 0; k < MT; ++k) {
        const int j = k - (MT - taps);  // tap index
        wt[k]       = j >= 0 ? w[(size_t)c * taps + j] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < MT - 1; ++k) {
        const int j = k - (MT - 1 - nh);  // history index 0 .. nh - 1, oldest first
        win[k]      = j >= 0 ? input(t0 - nh + j) : 0.f;
    }
    for (int t = t0; t < t1; ++t) {
        const float u   = x[(size_t)(row0 + t) * ldx + x_col + c];
        float       acc = 0.f;
#pragma unroll
        for (int k = 0; k < MT - 1; ++k) {
            acc = fmaf(wt[k], win[k], acc);
        }
        acc = fmaf(wt[MT - 1], u, acc);
#pragma unroll
        for (int k = 0; k + 1 < MT - 1; ++k) {
            win[k] = win[k + 1];
        }
        if (MT > 1) {
            win[MT - 2] = u;
        }
        y[(size_t)(row0 + t) * ldy + c] = act == 1 ? sm_silu(acc) : acc;
    }
    if (seg == 0) {  // new state: the inputs q_len - nh .. q_len - 1; ascending j reads st behind what it has written
        for (int j = 0; j < nh; ++j) {
            st[(size_t)j * C + c] = input(q_len - nh + j);
        }
    }
}

int launch_short_conv(float* y, int ldy, const float* x, int ldx, int x_col, const float* w, int channels, int taps, int act,
                      const StateMixParams& p, hipStream_t st)
{
    TM_REQUIRE(y && x && w && channels >= 1 && ldy >= channels && ldx >= x_col + channels && taps >= 1 && taps <= 16, "short conv: operands (1 <= taps <= 16)");
    TM_REQUIRE(p.cu_q && p.k_len && (taps == 1 || p.state) && p.max_q_len >= 1, "short conv: sequences / state");
    if (p.nseq == 0) {
        return 0;
    }
    const dim3 grid(p.nseq, (channels + 255) / 256, (p.max_q_len + kConvSeg - 1) / kConvSeg);
    if (taps <= 4) {
        short_conv_kernel<4><<<grid, 256, 0, st>>>(y, ldy, x, ldx, x_col, w, channels, taps, act, p);
    }
    else if (taps <= 8) {
        short_conv_kernel<8><<<grid, 256, 0, st>>>(y, ldy, x, ldx, x_col, w, channels, taps, act, p);
    }
    else {
        short_conv_kernel<16><<<grid, 256, 0, st>>>(y, ldy, x, ldx, x_col, w, channels, taps, act, p);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// y[row][g * n + i] = x[row][g * n + i] / sqrt(mean_i(x[row][g, :]^2) + eps) * w[g * n + i] * sigmoid(gate[row][g * n + i]):
// the output norm of the state mixers over groups of n channels (all heads together, or head by head) and their sigmoid gate (gate == nullptr: none).
// One workgroup per row: a single group is reduced by the whole workgroup, several groups are dealt to its four waves (and to grid y
// workgroups where the rows are too few to fill the device).
template<class T>
__global__ __launch_bounds__(256) void gated_group_norm_kernel(T* __restrict__ y, int ldy, const float* __restrict__ x, int ldx,
                                                               const float* __restrict__ w, const float* __restrict__ gate, int ldg, int groups,
                                                               int n, float eps, int silu, float mult)
{
    __shared__ float red[4];
    const int    t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* xr = x + (size_t)t * ldx;
    auto close = [&](float o, size_t c) {  // weight, gate, factor
        o *= w ? w[c] : 1.f;
        if (gate) {
            const float g = gate[(size_t)t * ldg + c];
            o             = (silu ? o * g : o) / (1.f + expf(-g));
        }
        return o * mult;
    };
    if (groups == 1) {
        float ss = 0.f;
        for (int i = threadIdx.x; i < n; i += 256) {
            ss = fmaf(xr[i], xr[i], ss);
        }
        ss = group_sum<64>(ss);
        if (lane == 0) {
            red[wave] = ss;
        }
        __syncthreads();
        const float inv = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)n + eps);
        for (int i = threadIdx.x; i < n; i += 256) {
            y[(size_t)t * ldy + i] = (T)close(xr[i] * inv, i);
        }
        return;
    }
    for (int g = blockIdx.y * 4 + wave; g < groups; g += gridDim.y * 4) {
        const float* xg = xr + (size_t)g * n;
        float        ss = 0.f;
        for (int i = lane; i < n; i += 64) {
            ss = fmaf(xg[i], xg[i], ss);
        }
        const float inv = 1.0f / sqrtf(group_sum<64>(ss) / (float)n + eps);
        for (int i = lane; i < n; i += 64) {
            const size_t c = (size_t)g * n + i;
            y[(size_t)t * ldy + c] = (T)close(xg[i] * inv, c);
        }
    }
}

// the same for groups that fit a workgroup's (one group: up to 8192 channels) or a wave's registers (several: up to 256), in pieces of four channels on
// 16-byte aligned operands: the row, its weights and its gates are requested together ahead of the reduction.  8 rows of 2048 in one group with a gate:
// the loop above 9.1 us a launch, this kernel 5.2.
template<class T, int NQ /* pieces of four channels a thread */, bool WIDE /* one group */>
__global__ __launch_bounds__(256) void gated_group_norm_reg_kernel(T* __restrict__ y, int ldy, const float* __restrict__ x, int ldx,
                                                                   const float* __restrict__ w, const float* __restrict__ gate, int ldg, int groups,
                                                                   int n, float eps, int silu, float mult)
{
    typedef T        T4 __attribute__((ext_vector_type(4)));
    __shared__ float red[4];
    constexpr int    NT = WIDE ? 256 : 64;
    const int        t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int        id = WIDE ? threadIdx.x : lane;
    for (int g = WIDE ? 0 : blockIdx.y * 4 + wave; g < groups; g += gridDim.y * 4) {
        const size_t c0 = (size_t)g * n;
        floatx4      v[NQ], wv[NQ], gv[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int i = min((id + q * NT) * 4, n - 4);
            v[q]        = *(const floatx4*)(x + (size_t)t * ldx + c0 + i);
            wv[q]       = floatx4{1.f, 1.f, 1.f, 1.f};
            gv[q]       = floatx4{0.f, 0.f, 0.f, 0.f};
            if (w) {
                wv[q] = *(const floatx4*)(w + c0 + i);
            }
            if (gate) {
                gv[q] = *(const floatx4*)(gate + (size_t)t * ldg + c0 + i);
            }
        }
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const bool in = (id + q * NT) * 4 < n;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ss = in ? fmaf(v[q][e], v[q][e], ss) : ss;
            }
        }
        ss = group_sum<64>(ss);
        if constexpr (WIDE) {
            if (lane == 0) {
                red[wave] = ss;
            }
            __syncthreads();
            ss = (red[0] + red[1]) + (red[2] + red[3]);
        }
        const float inv = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int i = (id + q * NT) * 4;
            if (i < n) {
                T4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float o = v[q][e] * inv * wv[q][e];
                    if (gate) {
                        o = (silu ? o * gv[q][e] : o) / (1.f + expf(-gv[q][e]));
                    }
                    out[e] = (T)(o * mult);
                }
                *(T4*)(y + (size_t)t * ldy + c0 + i) = out;
            }
        }
        if constexpr (WIDE) {
            return;
        }
    }
}

template<class T>
static void launch_gated_group_norm_t(T* y, int ldy, const float* x, int ldx, const float* w, const float* gate, int ldg, dim3 grid, int groups, int n,
                                      float eps, int silu, float mult, hipStream_t st)
{
    auto aligned = [](const void* p, size_t bytes) { return (uintptr_t)p % bytes == 0; };
    if (n % 4 || ldx % 4 || ldy % 4 || (gate && ldg % 4) || !aligned(x, 16) || !aligned(w, 16) || !aligned(gate, 16) || !aligned(y, 4 * sizeof(T))
        || n > (groups == 1 ? 8192 : 256)) {
        gated_group_norm_kernel<T><<<grid, 256, 0, st>>>(y, ldy, x, ldx, w, gate, ldg, groups, n, eps, silu, mult);
    }
    else if (groups > 1) {
        gated_group_norm_reg_kernel<T, 1, false><<<grid, 256, 0, st>>>(y, ldy, x, ldx, w, gate, ldg, groups, n, eps, silu, mult);
    }
    else if (n <= 2048) {
        gated_group_norm_reg_kernel<T, 2, true><<<grid, 256, 0, st>>>(y, ldy, x, ldx, w, gate, ldg, groups, n, eps, silu, mult);
    }
    else if (n <= 4096) {
        gated_group_norm_reg_kernel<T, 4, true><<<grid, 256, 0, st>>>(y, ldy, x, ldx, w, gate, ldg, groups, n, eps, silu, mult);
    }
    else {
        gated_group_norm_reg_kernel<T, 8, true><<<grid, 256, 0, st>>>(y, ldy, x, ldx, w, gate, ldg, groups, n, eps, silu, mult);
    }
}

int launch_gated_group_norm(void* y, int ldy, int out_elem_bytes, const float* x, int ldx, const float* w, const float* gate, int ldg, int rows,
                            int groups, int n, float eps, hipStream_t st, bool silu, float mult)
{
    TM_REQUIRE(y && x && groups >= 1 && n >= 1 && ldy >= groups * n && ldx >= groups * n && (!gate || ldg >= groups * n), "gated norm: operands");
    if (rows == 0) {
        return 0;
    }
    const dim3 grid(rows, groups > 4 && rows <= 256 ? (groups + 3) / 4 : 1);
    if (out_elem_bytes == 2) {
        launch_gated_group_norm_t((__bf16*)y, ldy, x, ldx, w, gate, ldg, grid, groups, n, eps, silu, mult, st);
    }
    else {
        launch_gated_group_norm_t((float*)y, ldy, x, ldx, w, gate, ldg, grid, groups, n, eps, silu, mult, st);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace tmk
