// Causal flash-attention for prefill on MFMA (gfx950), over the linear fp16 scratch produced by
// flatten_kv (K [kv_heads][k_stride][D], V transposed [kv_heads][D][k_stride]).
//
// Replaces: dispatchAttention -> attention_kernel<...AttentionCtaMap...> (src/turbomind/kernels/attention/
//           attention.cu:12-28, attention_template.h:13-85, kernel/attention_sm80_128.cu:21-37).
// Like the reference, prefill attention sees the round-tripped (quantised -> dequantised) KV.
//
// Layout trick (wave64, v_mfma_f32_16x16x32_f16): the scores are computed TRANSPOSED, S^T = K Q^T, so the
// accumulator of a lane (col = query row, rows = 4 consecutive keys) is, after exp2 and a cast to fp16,
// directly the B operand of the second contraction O^T = V^T P^T -- no LDS round trip, no cross-lane shuffle for P.
// The k-slot <-> key mapping of that second MFMA is (g, e) -> key 4g+e (e<4) / 16+4g+(e-4) (e>=4), which is
// why V is kept transposed: a lane fetches its 8 keys of one head-dim row with one 16-byte read.
// Softmax state is per lane.  Key order inside a 32-key step is permuted so that a lane's 8 probabilities
// belong to 8 CONSECUTIVE keys: score tile A row 4g+r <-> key 8g+r, tile B row 4g+r <-> key 8g+4+r.
//
// A workgroup is four waves of RT row tiles of 16 rows for HW query heads of a kv head (large launches: 128 rows of one head); a stage = 64 keys (K 16 KB + V^T 16 KB) comes in ONCE per
// workgroup by LDS-DMA (buffer_load ... lds: no staging registers), double buffered, one barrier per stage; the XOR swizzles that make the 16-byte
// fragment reads bank-conflict free sit on the DMA's source addresses (the DMA writes lane L to slot L of its 1 KB piece).  What bounds it is the
// softmax's VALU issue (v_exp_f32 at quarter rate) beside about as many matrix-pipe cycles: two waves share a SIMD, out of phase, under 256 registers
// each; a lane keeps its own partial row sum (the lane groups meet once, at the end) and the accumulators are rescaled only when a row's maximum moved.
// MI355X, Llama-3-8B heads (32 / 8), rocprofv3: 8192 rows of two sequences of ~8000 621 us a launch (~0.85 PFLOP/s), 8 x ~1024 rows 137 us.  (Sixteen rows
// of four query heads in one wave spilled: 1236 and 237 us.)
#include "gemm_stream.h"  // stream_dma16
#include "tm_common.h"
#include "tm_kernels.h"

namespace tmk {

// Swizzle term of K-tile row r (16-byte slot = chunk ^ ksw(r)).  A ds_read_b128 is served in four groups of 16 lanes --
// {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31}, ... (MI355X_MICROARCH.md, LDS) -- i.e. two neighbouring g with eight score-tile
// rows each; row i16 of a score tile is key 8 (i16 >> 2) + (i16 & 3), so the eight rows of either half differ in
// (bit 3, bits 1..0) of the key row: those three bits, shifted to slot bits 3..1, leave slot bit 0 to g -- 16 distinct slots
// per group.  (XOR with the plain row number, the first version, was a 2-way conflict on every K fragment read.)
__device__ __forceinline__ int ksw(int r)
{
    return (r & 8) | ((r & 3) << 1);
}

// max over the lane pairs l ^ 16 and l ^ 32 with gfx950's row / half swaps: two VALU ops each instead of a ds_bpermute round
// trip through the LDS crossbar in the middle of the softmax's dependency chain.  permlane16_swap(a, a) returns
// ([row0, row0, row2, row2], [row1, row1, row3, row3]), permlane32_swap(a, a) ([lo, lo], [hi, hi]).
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float max_xor16(float v)
{
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const u32x2_t  r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ __forceinline__ float max_xor32(float v)
{
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const u32x2_t  r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ __forceinline__ float sum_xor16_xor32(float v)
{
    unsigned       b = __builtin_bit_cast(unsigned, v);
    const u32x2_t  r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    b                = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]));
    const u32x2_t  q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return __builtin_bit_cast(float, (unsigned)q[0]) + __builtin_bit_cast(float, (unsigned)q[1]);
}

// Running maxima start at a large negative FINITE value: every difference / product in the online softmax then stays finite
// or is a clean -inf (masked score -> exp2(-inf) = 0), and the "-inf so far" selects around each exp disappear.
constexpr float kMinScore = -1.0e30f;

// NK: 32-key halves of the stage that hold visible keys
template<bool MASK, int RT, int NK>
__device__ __forceinline__ void prefill_step(const half8_t (&qf)[RT][4], const char* __restrict__ kt, const char* __restrict__ vt,
                                             const int (&limit)[RT], float sc, float (&m)[RT], float (&l)[RT],
                                             floatx4 (&O)[RT][8])
{
    const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
    floatx4   s[RT][2 * NK];
#pragma unroll
    for (int t = 0; t < 2 * NK; ++t) {  // score tile t, row i16: key 32 (t / 2) + 8 (i16 / 4) + 4 (t % 2) + i16 % 4 of the stage
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            s[rt][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const int   row = (t >> 1) * 32 + (i16 >> 2) * 8 + (t & 1) * 4 + (i16 & 3);
        const char* kr  = kt + row * 256;
        const int   sw  = ksw(row);
#pragma unroll
        for (int dd = 0; dd < 4; ++dd) {
            const half8_t kf = *(const half8_t*)(kr + (((4 * dd + g) ^ sw) << 4));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                s[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[rt][dd], s[rt][t], 0, 0, 0);
            }
        }
    }
    half8_t pf[RT][NK];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        // lane holds S[key 32 (t / 2) + 8 g + 4 (t % 2) + r][q = i16]
        float tmax = kMinScore;
#pragma unroll
        for (int t = 0; t < 2 * NK; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (MASK) {
                    s[rt][t][r] = (t >> 1) * 32 + 8 * g + (t & 1) * 4 + r <= limit[rt] ? s[rt][t][r] : -INFINITY;
                }
                tmax = fmaxf(tmax, s[rt][t][r]);
            }
        }
        tmax             = max_xor32(max_xor16(tmax));
        const float mnew = fmaxf(m[rt], tmax);  // finite (kMinScore at least)
        const float ms   = mnew * sc;
        float       psum = 0.f;
#pragma unroll
        for (int t = 0; t < 2 * NK; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float pv = fast_exp2(__builtin_fmaf(s[rt][t][r], sc, -ms));  // masked score: exp2(-inf) = 0
                psum += pv;
                pf[rt][t >> 1][(t & 1) * 4 + r] = (half_t)pv;
            }
        }
        if (__any(mnew != m[rt])) {
            const float alpha = fast_exp2((m[rt] - mnew) * sc);
            l[rt] *= alpha;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                O[rt][dt] *= alpha;
            }
        }
        l[rt] += psum;
        m[rt] = mnew;
    }
    // O^T += V^T P^T: one 16-byte V^T fragment (8 consecutive keys of one head-dim row) feeds both row tiles
    const char* vr = vt + i16 * 128;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
            const half8_t vf = *(const half8_t*)(vr + dt * 2048 + (((4 * ks + g) ^ (i16 & 7)) << 4));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                O[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pf[rt][ks], O[rt][dt], 0, 0, 0);
            }
        }
    }
}

// HW waves side by side take HW query heads of one kv head, 4 / HW row blocks of 16 RT rows each
template<int RT, int HW>
__global__ __launch_bounds__(256, 2) void prefill_attention_kernel(PrefillAttnParams p)
{
    constexpr int kRows = 16 * RT, kRowsGroup = 4 / HW * kRows;
    constexpr int D = 128, KS = 64, KTILE = KS * D * 2, STG = 2 * KTILE;  // keys per stage; bytes of a K tile (and of a V^T tile)
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, g = lane >> 4;
    // workgroups are dealt to the eight XCDs in turn, heads first: the query heads of a kv head on one XCD where the head count allows it; the longest row
    // blocks of every sequence first (longest-processing-time order: the short ones fill the tail)
    const int HG = gridDim.x, b = blockIdx.y, bx = gridDim.z - 1 - blockIdx.z;
    const int hg = HG % 8 == 0 ? (blockIdx.x % 8) * (HG / 8) + blockIdx.x / 8 : blockIdx.x;
    const int hq = hg * HW + wave % HW;
    const int q_beg = p.cu_q_len[b];
    const int qlen  = p.cu_q_len[b + 1] - q_beg;
    const int klen  = p.k_len[b];
    const int hist  = klen - qlen;
    if (bx * kRowsGroup >= qlen) {
        return;  // workgroup-uniform
    }
    const int  q0     = bx * kRowsGroup + wave / HW * kRows;
    const bool active = q0 < qlen;  // wave-uniform; an inactive wave still stages tiles and meets the barriers
    const int  kvh    = hg * HW / (p.q_heads / p.kv_heads);

    // Q^T fragments (B operand): lane (j = query row, g) holds Q[row j][32*dd + 8g .. +8)
    half8_t qf[RT][4];
    floatx4 O[RT][8];
    float   m[RT], l[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const half_t* qptr = p.q + (size_t)(q_beg + min(q0 + rt * 16 + i16, qlen - 1)) * p.q_stride + (size_t)hq * D;
#pragma unroll
        for (int dd = 0; dd < 4; ++dd) {
            qf[rt][dd] = *(const half8_t*)(qptr + dd * 32 + g * 8);
        }
        m[rt] = kMinScore;
        l[rt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            O[rt][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // the sequence's region of the scratch is 64-key aligned, its V^T tail is zero-filled (flatten_kv_kernel): a 64-key stage
    // never leaves the region; K rows past klen may hold stale data, their scores are masked below
    const half_t* kbase    = p.k + ((size_t)kvh * p.k_stride + p.cu_k_off[b]) * D;
    const half_t* vbase    = p.vt + (size_t)kvh * D * p.k_stride + p.cu_k_off[b];
    const int     klen_pad = (klen + KS - 1) / KS * KS;
    const auto    rs_k     = __builtin_amdgcn_make_buffer_rsrc((void*)kbase, 0, klen_pad * D * 2, 0x00020000);
    const auto    rs_v     = __builtin_amdgcn_make_buffer_rsrc((void*)vbase, 0, (int)(((size_t)(D - 1) * p.k_stride + klen_pad) * 2), 0x00020000);
    // DMA pieces of 1 KB: K piece pc = key rows 4pc .. 4pc+3 (256 B each, 16 chunks), V^T piece pc = head-dim rows 8pc .. 8pc+7
    // (128 B each, 8 chunks); wave w moves pieces 4r + w, r = 0..3.  Lane L lands in slot L: it fetches the chunk that belongs there.
    // piece 4r + w: K rows 16r + 4w + (L >> 4), V^T rows 32r + 8w + (L >> 3) -- the swizzle terms (row & 15, d & 7) do not depend on
    // r (ksw looks at bits 3 and 1..0 only), so one per-lane offset each serves all four pieces and r moves into the scalar offset
    const int krow0 = 4 * wave + (lane >> 4);
    const int kdo   = krow0 * 256 + (((lane & 15) ^ ksw(krow0)) << 4);
    const int vrow0 = 8 * wave + (lane >> 3);
    const int vdo   = vrow0 * p.k_stride * 2 + (((lane & 7) ^ (vrow0 & 7)) << 4);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
    auto stage_in = [&](int ks, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const unsigned dk = lds0 + buf * STG + (4 * r + wave) * 1024;
            stream_dma16(rs_k, kdo, ks * D * 2 + r * 16 * 256, dk);
            stream_dma16(rs_v, vdo, ks * 2 + r * 32 * p.k_stride * 2, dk + KTILE);
        }
    };
    const int kend_w  = active ? min(klen, hist + q0 + kRows) : 0;      // keys visible to the last row of this wave
    const int kend_wg = min(klen, hist + (bx + 1) * kRowsGroup);            // ... of this workgroup

    stage_in(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int buf = 0;
    for (int ks0 = 0; ks0 < kend_wg; ks0 += KS, buf ^= 1) {
        if (ks0 + KS < kend_wg) {
            stage_in(ks0 + KS, buf ^ 1);  // every wave is past the barrier behind its reads of that buffer
        }
        const char *kt = smem + buf * STG, *vt = kt + KTILE;
        if (ks0 < kend_w) {  // wave-uniform: causal end of this wave (or an inactive wave)
            int limit[RT];  // last visible key of the lane's rows in this stage (rows past the portion: none)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int r = q0 + rt * 16 + i16;
                limit[rt]   = r < qlen ? hist + r - ks0 : -1;
            }
            // the whole stage lies at or below the diagonal for every row of the wave: no masking needed (all but the last stages)
            if (ks0 + KS - 1 <= hist + q0 && q0 + kRows <= qlen) {
                prefill_step<false, RT, 2>(qf, kt, vt, limit, p.scale_log2, m, l, O);
            }
            else if (ks0 + KS / 2 < kend_w) {
                prefill_step<true, RT, 2>(qf, kt, vt, limit, p.scale_log2, m, l, O);
            }
            else {
                prefill_step<true, RT, 1>(qf, kt, vt, limit, p.scale_log2, m, l, O);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of the next stage have landed ...
        __syncthreads();                                  // ... everybody's have, and everybody is done reading this one
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const float lh = sum_xor16_xor32(l[rt]);
        const int   r  = q0 + rt * 16 + i16;
        if (r < qlen) {
            half_t*     optr = p.out + (size_t)(q_beg + r) * p.q_heads * D + (size_t)hq * D;
            const float inv  = 1.0f / lh;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                half4_t o = {(half_t)(O[rt][dt][0] * inv), (half_t)(O[rt][dt][1] * inv), (half_t)(O[rt][dt][2] * inv),
                             (half_t)(O[rt][dt][3] * inv)};
                *(half4_t*)(optr + dt * 16 + g * 4) = o;
            }
        }
    }
}

template<int RT, int HW>
static int launch_prefill(const PrefillAttnParams& p, hipStream_t st)
{
    constexpr int lds = 2 * 2 * 64 * 128 * 2;  // two stages of (K tile + V^T tile)
    const auto    k   = prefill_attention_kernel<RT, HW>;
    if (const int rc = ensure_dynamic_lds((const void*)k, lds)) {
        return rc;
    }
    const int tiles = (p.max_q_len + 64 / HW * RT - 1) / (64 / HW * RT);
    k<<<dim3(p.q_heads / HW, p.batch, tiles), 256, lds, st>>>(p);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_prefill_attention(const PrefillAttnParams& p, hipStream_t st)
{
    TM_REQUIRE(p.q_heads % p.kv_heads == 0, "q_heads % kv_heads");
    TM_REQUIRE(p.k_stride % 64 == 0, "k_stride must be a multiple of 64");
    if (p.batch == 0 || p.max_q_len == 0) {
        return 0;
    }
    // us, heads / kv heads, rows x sequences + context.  Two row tiles a wave read each key and value half as often, but need 512 workgroups of 128 rows, two a
    // CU, to be faster than one (32/8: 1024 x 8 104 | 128, 500 x 4 22.6 | 22.6; 64/8: 512 x 2 + 3000 138 | 160; 8/8: 500 x 4 17.5 | 11.7, 16 x 2 + 4000 106 | 75; 5/1:
    // 4000 x 1 96 | 70) and rows that fill them (28/4: 129 x 16 23.8 | 21.6).  Short prompts of many heads: 16 or 32 rows of four or two heads side by side
    // leave no wave idle and share keys and values (32/8: 10 x 64 one head 12.0, two 7.6, four 5.5; 20 x 100 24.5, 18.0, 19.6; fewer than two workgroups
    // a CU: 17 x 1 3.6, 3.9, 4.4)
    const int     group = p.q_heads / p.kv_heads;
    const int64_t r64 = (p.max_q_len + 63) / 64, r128 = (p.max_q_len + 127) / 128, per_row_block = (int64_t)p.batch * p.q_heads;
    if (r128 * per_row_block >= 512 && r128 * 200 <= r64 * 115) {
        return launch_prefill<2, 1>(p, st);
    }
    if (per_row_block > 512) {
        if (p.max_q_len <= 16 && group % 4 == 0) {
            return launch_prefill<1, 4>(p, st);
        }
        if (p.max_q_len <= 32 && group % 2 == 0) {
            return launch_prefill<1, 2>(p, st);
        }
    }
    return launch_prefill<1, 1>(p, st);
}

}  // namespace tmk
