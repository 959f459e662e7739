// Mixture-of-experts routing for gfx950: router (gate) + top-k + routing tables + weighted combine.
//
// Replaces: MoeFfnLayerImpl::Gate, invokeMoeGate_V2 (softmax / top-k / norm_topk / routed_scale and the f2n / en2f /
// offsets tables) and invokeMoeCombine (src/turbomind/models/llama/moe_ffn_layer.cc:43-53,133-325;
// kernels/gemm/moe_utils_v2.cu:355-690).  The expert FFNs run as grouped GEMMs (gemm_w4a16.hip, `groups` descriptors)
// over the token rows listed per expert.
//   gate:   logits[t][e] = sum_h x[t][h] * Wg[h][e] in fp32; top-k on the logits (ties: lower expert id);
//           norm_topk: w_j = exp(l_j - max) / sum over the SELECTED experts, else softmax over all experts;
//           w_j *= routed_scale.
//   route:  for every expert the tokens that selected it, in ascending token order:
//           offsets[e] .. offsets[e+1] index the flat pair list; f2n[f] = token; en2f[j][t] = f.
//   combine: out[t] = fp16( sum_j w[t][j] * float(y[en2f[j][t]]) ).
#include "fp8_quant.h"
#include "tm_common.h"
#include "tm_kernels.h"

#define TM_TRY_RC(expr)       \
    do {                     \
        const int _rc = (expr); \
        if (_rc) {           \
            return _rc;      \
        }                    \
    } while (0)

namespace tmk {

constexpr int kMaxExperts = 64;
constexpr int kMaxTopK    = 8;
constexpr int kRouteTokens = 64, kRouteExperts = 256, kRoutePairs = 2048;  // what one workgroup's masks hold (moe_route_masks_kernel)

// the largest v of a wave, the lower index on a tie (i = INT_MAX: no candidate, else i % 64 is the lane); every lane ends up with the choice
__device__ __forceinline__ void wave_argmax(float& v, int& i)
{
    const bool in = i != 0x7fffffff;
    if (__ballot(in && !(v == v)) == 0) {
        // the maximum over DPP, then who has it: the twelve shuffles through LDS, one behind the other, cost 0.2 - 0.3 us a choice more
        const float              mx  = group_max<64>(in ? v : -INFINITY);
        const bool               has = in && v == mx;
        const unsigned long long any = __ballot(has);
        if (any) {
            int low = 0;
            while (!__ballot(has && i < (low + 1) * 64)) {  // (some lane has it: the loop ends)
                ++low;
            }
            const int lane = __builtin_ctzll(__ballot(has && i < (low + 1) * 64));
            v = mx, i = low * 64 + lane;
        }
        return;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {  // (with numbers that are none: as they compare)
        const float ov = __shfl_xor(v, d);
        const int   oi = __shfl_xor(i, d);
        if (oi != 0x7fffffff && (i == 0x7fffffff || ov > v || (ov == v && oi < i))) {
            v = ov, i = oi;
        }
    }
}

// One 256-thread workgroup per token; Wg fp16 [H][E] (input-major like every other weight).  V experts share a pass over the token (V = 8: E a multiple of
// eight, 16-byte loads of Wg), so the row is read E / V times and every load is independent of the last, sixteen rounds of them in flight (V = 1: a short pass an expert,
// which loads beyond the row's end would only lengthen: eight; 60 experts of H = 2048, one token, a whole expert block 87 us, with sixteen 107); one wave picks the
// experts.  Bound by that chain: H = 4096, 8 experts: 24.6 us with a pass per expert and one thread picking, 8.0 us with eight
// rounds in flight, 6.4 with the tail beside it:
// workgroups behind the tokens' quantise the rows, and of up to 64 tokens the last one's writes the routing tables.  16 tokens, fp8 experts: 8.0 + 4.7 (tables) + 4.8 us
// (codes) -> 6.4.  More tokens keep the tables' own launch, which takes a workgroup an expert.
template<int V>
__global__ __launch_bounds__(256) void moe_gate_kernel(int* __restrict__ topk_ids,      // [T][k]
                                                       float* __restrict__ topk_w,      // [T][k]
                                                       float* __restrict__ logits_out,  // [T][E] or nullptr
                                                       const half_t* __restrict__ x,
                                                       int ldx,
                                                       const half_t* __restrict__ wg,
                                                       int H,
                                                       int E,
                                                       int k,
                                                       int norm_topk,
                                                       float routed_scale,
                                                       int T,
                                                       MoeGateTail tail)
{
    if ((int)blockIdx.x >= T) {
        quant_fp8_groups(blockIdx.x - T, tail.xq, tail.sx, x, ldx, T, H, tail.ldsx);
        return;
    }
    typedef half_t HV __attribute__((ext_vector_type(V)));
    __shared__ float              part[4][kMaxExperts];
    __shared__ unsigned long long mask[64];
    __shared__ int                first[64];
    const int        t    = blockIdx.x;
    const int        lane = threadIdx.x & 63;
    const int        wave = threadIdx.x >> 6;
    const half_t*    xr   = x + (size_t)t * ldx;
    for (int e = 0; e < E; e += V) {
        float acc[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
            acc[i] = 0.f;
        }
        if constexpr (V == 1) {
#pragma unroll 8
            for (int h = threadIdx.x; h < H; h += 256) {
                acc[0] = __builtin_fmaf((float)xr[h], (float)wg[(size_t)h * E + e], acc[0]);
            }
        }
        for (int h0 = threadIdx.x; V > 1 && h0 < H; h0 += 256 * 16) {
            half_t xv[16];
            HV     wv[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {  // (the row's last channel again beyond its end)
                const int h = min(h0 + r * 256, H - 1);
                xv[r]       = xr[h];
                wv[r]       = *(const HV*)(wg + (size_t)h * E + e);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const bool in = h0 + r * 256 < H;
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    acc[i] = in ? __builtin_fmaf((float)xv[r], (float)wv[r][i], acc[i]) : acc[i];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < V; ++i) {
            acc[i] = group_sum<64>(acc[i]);
            if (lane == 0) {
                part[wave][e + i] = acc[i];
            }
        }
    }
    __syncthreads();
    if (wave > 0) {
        return;
    }
    const bool  in    = lane < E;  // lane = expert
    const float logit = in ? (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]) : -INFINITY;
    if (in && logits_out) {
        logits_out[(size_t)t * E + lane] = logit;
    }
    const float mx    = group_max<64>(logit);
    bool        taken = !in;
    int         id    = 0;       // lane j < k: choice j
    float       val   = 0.f, denom = 0.f;
    for (int j = 0; j < k; ++j) {
        float v = logit;
        int   i = taken ? 0x7fffffff : lane;
        wave_argmax(v, i);
        i     = __builtin_amdgcn_readfirstlane(i);
        v     = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
        taken = taken || lane == i;
        id    = lane == j ? i : id;
        val   = lane == j ? v : val;
        denom += __builtin_expf(v - mx);
    }
    if (!norm_topk) {
        denom = group_sum<64>(in ? __builtin_expf(logit - mx) : 0.f);
    }
    if (lane < k) {
        topk_w[(size_t)t * k + lane] = __builtin_expf(val - mx) * (1.0f / denom) * routed_scale;
        __hip_atomic_store(topk_ids + (size_t)t * k + lane, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!tail.ticket || !ticket_last_wave(tail.ticket, T)) {
        return;
    }
    // The tables by one wave, as moe_route_masks_kernel builds them: at most 64 tokens and 64 experts, an expert on each lane
    constexpr int kPairs = kRouteTokens * kMaxTopK / 64;
    int           ids[kPairs];
#pragma unroll
    for (int r = 0; r < kPairs; ++r) {
        if (r * 64 < T * k) {
            ids[r] = __hip_atomic_load(topk_ids + min(r * 64 + lane, T * k - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    mask[lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll
    for (int r = 0; r < kPairs; ++r) {
        if (r * 64 + lane < T * k) {
            atomicOr(&mask[ids[r]], 1ull << ((r * 64 + lane) / k));
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    const int n = __popcll(mask[lane]);
    int       f = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(f, d);
        f += lane >= d ? y : 0;
    }
    first[lane] = f - n;
    if (lane < E) {
        tail.offsets[lane] = f - n;
    }
    if (lane == 0) {
        tail.offsets[E] = T * k;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
#pragma unroll
    for (int r = 0; r < kPairs; ++r) {
        const int p = r * 64 + lane;
        if (p < T * k) {
            const int to = p / k, at = first[ids[r]] + __popcll(mask[ids[r]] & ((1ull << to) - 1));
            tail.f2n[at]                               = to;
            tail.en2f[(size_t)(p - to * k) * T + to] = at;
        }
    }
}

template<class X>
struct MoeGather {  // rows of x, H channels, to xs in the experts' order; shared: and all of them behind
    X*       xs     = nullptr;
    int      lds    = 0;
    const X* x      = nullptr;
    int      ldx    = 0;
    int      H      = 0;
    int      shared = 0;
};

// Routing tables of up to kRouteTokens tokens and kRouteExperts experts in one workgroup: an expert's tokens are a 64-bit mask in LDS, a pair's place the
// expert's first row (a wave's scan over the experts) plus the tokens ahead of it in the mask -- no pass over the experts.  PICK: the experts are first
// chosen here, one wave per token, as moe_topk_softmax_kernel does (expert e on lane e % 64).  A chain of latencies: 8 tokens, 8 experts, 2 a token take
// 4.8 us, the two kernels for any size 5.7 + 9.5.
// V > 0: every workgroup makes the tables for itself, the first one writes them, and each copies four of the rows that moe_gather_kernel would (V channels a load, the
// first of them asked for ahead of the routing).  8 tokens of 2048, three rows a token: 5.0 us, the two launches
// 4.8 + 2.6.
template<bool PICK, class X = __bf16, int V = 0>
__global__ __launch_bounds__(1024) void moe_route_masks_kernel(int* __restrict__ offsets, int* __restrict__ f2n, int* __restrict__ en2f, int* topk_ids,
                                                               float* __restrict__ w, const float* __restrict__ logits, int ld, int T, int E, int k,
                                                               float scale, MoeGather<X> g)
{
    constexpr int NE = kRouteExperts / 64;
    typedef X XV __attribute__((ext_vector_type(V ? V : 1)));
    __shared__ unsigned long long mask[kRouteExperts];
    __shared__ int                first[kRouteExperts];
    __shared__ unsigned short     chosen[V ? kRoutePairs : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kk = k + g.shared, job = blockIdx.x * 4 + (tid >> 8), jt = min(job / kk, T - 1), jj = job % kk, c0 = (tid & 255) * V;
    const X* const src = V ? g.x + (size_t)jt * g.ldx : nullptr;
    XV             head{};
    if constexpr (V > 0) {
        if (c0 < g.H) {
            head = *(const XV*)(src + c0);
        }
    }
    const bool writes = blockIdx.x == 0;
    if (tid < kRouteExperts) {
        mask[tid] = 0;
    }
    __syncthreads();
    if constexpr (PICK) {
        for (int t = wave; t < T; t += 16) {
            float z[NE], mx = -INFINITY, den = 0.f;
            bool  taken[NE];
#pragma unroll
            for (int q = 0; q < NE; ++q) {
                const int e = q * 64 + lane;
                taken[q]    = e >= E;
                z[q]        = e < E ? logits[(size_t)t * ld + e] : -INFINITY;
                mx          = fmaxf(mx, z[q]);
            }
            mx = group_max<64>(mx);
#pragma unroll
            for (int q = 0; q < NE; ++q) {
                den += taken[q] ? 0.f : expf(z[q] - mx);
            }
            den = group_sum<64>(den);
            for (int j = 0; j < k; ++j) {
                float v = 0.f;
                int   i = 0x7fffffff;
#pragma unroll
                for (int q = 0; q < NE; ++q) {
                    if (!taken[q] && (i == 0x7fffffff || z[q] > v)) {
                        v = z[q], i = q * 64 + lane;
                    }
                }
                wave_argmax(v, i);
                i = __builtin_amdgcn_readfirstlane(i);
#pragma unroll
                for (int q = 0; q < NE; ++q) {
                    taken[q] = taken[q] || q * 64 + lane == i;
                }
                if (lane == 0) {
                    if (writes) {
                        topk_ids[(size_t)t * k + j] = i;
                        w[(size_t)t * k + j]        = scale * (expf(v - mx) / den);
                    }
                    if constexpr (V > 0) {
                        chosen[t * k + j] = (unsigned short)i;
                    }
                    atomicOr(&mask[i], 1ull << t);
                }
            }
        }
    }
    else {
        for (int p = tid; p < T * k; p += 1024) {
            atomicOr(&mask[topk_ids[p]], 1ull << (p / k));
        }
    }
    __syncthreads();
    if (wave == 0) {
        int n[NE], sum = 0;
#pragma unroll
        for (int q = 0; q < NE; ++q) {
            n[q] = __popcll(mask[lane * NE + q]);
            sum += n[q];
        }
        int x = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(x, d);
            x += lane >= d ? y : 0;
        }
        x -= sum;
#pragma unroll
        for (int q = 0; q < NE; ++q) {
            first[lane * NE + q] = x;
            x += n[q];
        }
    }
    __syncthreads();
    if (writes) {
        if (tid <= E) {
            offsets[tid] = tid < E ? first[tid] : T * k;
        }
        if (V > 0 && tid == 0 && g.shared) {
            offsets[E + 1] = T * kk;
        }
        for (int p = tid; p < T * k; p += 1024) {
            const int t = p / k, e = V ? chosen[p] : topk_ids[p], f = first[e] + __popcll(mask[e] & ((1ull << t) - 1));
            f2n[f]                          = t;
            en2f[(size_t)(p - t * k) * T + t] = f;
        }
    }
    if constexpr (V > 0) {
        if (job < T * kk) {
            int f = T * k + jt;  // the copy behind the routed rows
            if (jj < k) {
                const int e = chosen[jt * k + jj];
                f           = first[e] + __popcll(mask[e] & ((1ull << jt) - 1));
            }
            X* const dst = g.xs + (size_t)f * g.lds;
            if (c0 < g.H) {
                *(XV*)(dst + c0) = head;
            }
            for (int i = c0 + 256 * V; i < g.H; i += 256 * V) {
                *(XV*)(dst + i) = *(const XV*)(src + i);
            }
        }
    }
}

// Routing tables of any number of tokens: offsets [E+1], f2n [T*k], en2f [k][T].  A workgroup an expert: each reads all choices (they stay in L2), counts those of
// lower experts, which is where its rows begin, and its own ahead of every thread's run of tokens; a second look at them writes its rows in token order.  Two
// short passes over T k numbers instead of one workgroup's walk over the experts with barriers for each: 8 experts, 2 choices: 8000 tokens 70 -> 14 us, 4000
// 36.7 -> 7.3.
__global__ __launch_bounds__(1024) void moe_route_kernel(int* __restrict__ offsets, int* __restrict__ f2n, int* __restrict__ en2f,
                                                         const int* __restrict__ topk_ids, int T, int E, int k)
{
    __shared__ int s_mine[16], s_lower[16];
    const int      tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, e = blockIdx.x;
    const int      run = (T + 1023) / 1024 * k;  // choices of a thread: whole tokens
    const int      p0 = min(tid * run, T * k), p1 = min(p0 + run, T * k);
    int            mine = 0, lower = 0;
#pragma unroll 8
    for (int p = p0; p < p1; ++p) {
        const int id = topk_ids[p];
        mine += id == e;
        lower += (unsigned)id < (unsigned)e;
    }
    int x = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        x += lane >= d ? y : 0;
        lower += __shfl_xor(lower, d);
    }
    if (lane == 63) {
        s_mine[wave]  = x;
        s_lower[wave] = lower;
    }
    __syncthreads();
    int f = x - mine;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        f += s_lower[w] + (w < wave ? s_mine[w] : 0);
    }
    if (tid == 0) {
        offsets[e] = f;
    }
    if (tid == 1023 && e == E - 1) {
        offsets[E] = f + mine;
    }
    if (mine == 0) {
        return;
    }
    for (int p = p0; p < p1; ++p) {
        if (topk_ids[p] == e) {
            const int t                       = p / k;
            f2n[f]                            = t;
            en2f[(size_t)(p - t * k) * T + t] = f;
            ++f;
        }
    }
}

// out[t][h] = fp16( sum_j w[t][j] * y[en2f[j][t]][h] ); 8 columns per thread
__global__ __launch_bounds__(256) void moe_combine_kernel(half_t* __restrict__ out, int ldo, const half_t* __restrict__ y, int ldy,
                                                          const float* __restrict__ topk_w, const int* __restrict__ en2f, int T,
                                                          int H, int k)
{
    const int t = blockIdx.y;
    const int h = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (h >= H) {
        return;
    }
    float acc[8] = {};
    for (int j = 0; j < k; ++j) {
        const int     f = en2f[(size_t)j * T + t];
        const float   w = topk_w[(size_t)t * k + j];
        const half8_t v = *(const half8_t*)(y + (size_t)f * ldy + h);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            acc[e] = __builtin_fmaf(w, (float)v[e], acc[e]);
        }
    }
    half8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        o[e] = (half_t)acc[e];
    }
    *(half8_t*)(out + (size_t)t * ldo + h) = o;
}

int launch_moe_gate(int* topk_ids, float* topk_w, float* logits_out, const half_t* x, int ldx, const half_t* wg, int T, int H,
                    int E, int k, bool norm_topk, float routed_scale, hipStream_t st, const MoeGateTail& tail)
{
    TM_REQUIRE(E >= 1 && E <= kMaxExperts && k >= 1 && k <= kMaxTopK && k <= E, "moe: 1 <= top_k <= experts <= 64, top_k <= 8");
    TM_REQUIRE(!tail.ticket || T <= kRouteTokens, "moe gate: the tables of at most 64 tokens");
    TM_REQUIRE(!tail.xq || (H % 128 == 0 && ldx % 8 == 0 && tail.ldsx >= T), "moe gate: fp8 rows of 128-channel groups, 16-byte aligned, ldsx >= T");
    if (T == 0) {
        return 0;
    }
    const int  grid = T + (tail.xq ? (T * (H / 128) + 15) / 16 : 0);
    const auto gate = E % 8 == 0 && (uintptr_t)wg % 16 == 0 ? moe_gate_kernel<8> : moe_gate_kernel<1>;
    gate<<<grid, 256, 0, st>>>(topk_ids, topk_w, logits_out, x, ldx, wg, H, E, k, norm_topk ? 1 : 0, routed_scale, T, tail);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_moe_route(int* offsets, int* f2n, int* en2f, const int* topk_ids, int T, int E, int k, hipStream_t st)
{
    if (T <= kRouteTokens && E <= kRouteExperts) {
        moe_route_masks_kernel<false><<<1, 1024, 0, st>>>(offsets, f2n, en2f, (int*)topk_ids, nullptr, nullptr, 0, T, E, k, 0.f, {});
    }
    else {
        moe_route_kernel<<<E, 1024, 0, st>>>(offsets, f2n, en2f, topk_ids, T, E, k);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

int launch_moe_combine(half_t* out, int ldo, const half_t* y, int ldy, const float* topk_w, const int* en2f, int T, int H, int k,
                       hipStream_t st)
{
    TM_REQUIRE(H % 8 == 0, "moe combine: H % 8 == 0");
    if (T == 0) {
        return 0;
    }
    moe_combine_kernel<<<dim3((H / 8 + 255) / 256, T), 256, 0, st>>>(out, ldo, y, ldy, topk_w, en2f, T, H, k);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---- one MoE FFN block (host object shared by the C-ABI operator and the engine) -------------------------------------
size_t moe_workspace_bytes(const MoeBlock& m, int tokens)
{
    const size_t pairs = (size_t)tokens * m.top_k;
    size_t       b     = 0;
    b += pairs * 4;                  // topk_ids
    b += pairs * 4;                  // topk_w
    b += (size_t)(m.experts + 1) * 4;  // offsets
    b += pairs * 4;                  // f2n
    b += pairs * 4;                  // en2f
    b  = (b + 255) / 256 * 256;
    b += pairs * m.inter * 2;        // act  [pairs][I]
    b  = (b + 255) / 256 * 256;
    b += pairs * m.hidden * 2;       // y2   [pairs][H]
    b  = (b + 255) / 256 * 256;
    // fp8 x fp8 experts: codes + scales of x (per token) and of the gated-SiLU output (per (token, expert) row)
    b += fp8_act_workspace_bytes(tokens, m.hidden) + fp8_act_workspace_bytes((int)pairs, m.inter);
    return b + 256;
}

int moe_prepare(MoeBlock& m, hipStream_t st)
{
    TM_REQUIRE((int)m.w13.size() == m.experts && (int)m.w2.size() == m.experts && m.gate, "moe: gate and every expert must be set");
    TM_TRY_RC(moe_build_groups(&m.groups13, m.w13.data(), m.experts, st));
    TM_TRY_RC(moe_build_groups(&m.groups2, m.w2.data(), m.experts, st));
    if (fp8_mfma_supported(m.w13[0]) && fp8_mfma_supported(m.w2[0])) {  // device tables of the experts' P8 unit pointers
        std::vector<const void*> h13(m.experts), h2(m.experts);
        for (int e = 0; e < m.experts; ++e) {
            TM_REQUIRE(m.w13[e].packed8 && m.w2[e].packed8, "moe: fp8 expert without its P8 image");
            h13[e] = m.w13[e].packed8;
            h2[e]  = m.w2[e].packed8;
        }
        if (!m.groups13_p8) {
            TM_HIP_CHECK(hipMalloc(&m.groups13_p8, sizeof(void*) * m.experts));
            TM_HIP_CHECK(hipMalloc(&m.groups2_p8, sizeof(void*) * m.experts));
        }
        TM_HIP_CHECK(hipMemcpyAsync(m.groups13_p8, h13.data(), sizeof(void*) * m.experts, hipMemcpyHostToDevice, st));
        TM_HIP_CHECK(hipMemcpyAsync(m.groups2_p8, h2.data(), sizeof(void*) * m.experts, hipMemcpyHostToDevice, st));
        TM_HIP_CHECK(hipStreamSynchronize(st));
    }
    return 0;
}

// (rows: the sum is left to the caller, out is not written; ticket: a counter of the caller's stream, zero between launches, for one launch instead of two)
// out[t] = sum_j w_j * W2_e( silu(W1_e x_t) * (W3_e x_t) ) over the top_k experts e of token t
int moe_forward(const MoeBlock& m, half_t* out, int ldo, const half_t* x, int ldx, int tokens, void* workspace, int* topk_ids_out,
                float* topk_w_out, hipStream_t st, MoeRows* rows, unsigned* ticket)
{
    TM_REQUIRE(m.groups13 && m.groups2, "moe: not prepared");
    if (rows) {
        *rows = MoeRows{};
    }
    if (tokens == 0) {
        return 0;
    }
    const size_t pairs = (size_t)tokens * m.top_k;
    char*        w     = (char*)workspace;
    int*         ids   = (int*)w;
    float*       tw    = (float*)(w + pairs * 4);
    int*         offs  = (int*)(w + pairs * 8);
    int*         f2n   = offs + (m.experts + 1);
    int*         en2f  = f2n + pairs;
    size_t       o     = ((char*)(en2f + pairs) - w + 255) / 256 * 256;
    half_t*      act   = (half_t*)(w + o);
    o                  = (o + pairs * m.inter * 2 + 255) / 256 * 256;
    half_t*      y2    = (half_t*)(w + o);
    MoeGateTail tail;
    if (ticket && tokens <= kRouteTokens) {
        tail.ticket = ticket, tail.offsets = offs, tail.f2n = f2n, tail.en2f = en2f;
    }
    o                 = (o + pairs * m.hidden * 2 + 255) / 256 * 256;
    uint8_t*  xq      = (uint8_t*)(w + o);
    const int ldsx1   = (tokens + 3) / 4 * 4;
    float*    sx1     = (float*)(xq + (size_t)tokens * m.hidden);
    if (m.groups13_p8) {
        TM_REQUIRE(ldx == m.hidden || tokens == 1, "moe fp8: x must be row-contiguous");
        tail.xq = xq, tail.sx = sx1, tail.ldsx = ldsx1;
    }
    TM_TRY_RC(launch_moe_gate(ids, tw, nullptr, x, ldx, m.gate, tokens, m.hidden, m.experts, m.top_k, m.norm_topk, m.routed_scale, st, tail));
    if (!tail.ticket) {
        TM_TRY_RC(launch_moe_route(offs, f2n, en2f, ids, tokens, m.experts, m.top_k, st));
    }
    // expert FFNs: gathered rows of x -> act (gated SiLU fused) -> y2, both grouped over the experts
    const int hint = (int)((pairs + m.experts - 1) / m.experts);  // expected rows per expert
    if (m.groups13_p8) {
        // e4m3 experts on the fp8 matrix cores (the reference's fp8 path: QuantizeSymm + fp8 GEMM, LlamaLinear.cu:67-127):
        // x was quantised once per token beside the router, the gated-SiLU output once per (token, expert) row
        o                  = (o + fp8_act_workspace_bytes(tokens, m.hidden) + 255) / 256 * 256;
        uint8_t*     aq    = (uint8_t*)(w + o);
        const int    ldsx2 = ((int)pairs + 3) / 4 * 4;
        float*       sx2   = (float*)(aq + pairs * m.inter);
        TM_TRY_RC(launch_linear_fp8_grouped(m.w13[0], m.groups13_p8, m.experts, xq, sx1, ldsx1, tokens, act, m.inter, tokens, (int)pairs, hint, true,
                                            offs, f2n, st));
        TM_TRY_RC(launch_quant_fp8_rows(aq, sx2, act, m.inter, (int)pairs, m.inter, ldsx2, st));
        TM_TRY_RC(launch_linear_fp8_grouped(m.w2[0], m.groups2_p8, m.experts, aq, sx2, ldsx2, (int)pairs, y2, m.hidden, tokens, (int)pairs, hint, false,
                                            offs, nullptr, st));
    }
    else {
        TM_TRY_RC(launch_linear_grouped(m.w13[0], m.groups13, m.experts, x, ldx, tokens, act, m.inter, tokens, hint, true, offs, f2n, st));
        TM_TRY_RC(launch_linear_grouped(m.w2[0], m.groups2, m.experts, act, m.inter, (int)pairs, y2, m.hidden, tokens, hint, false, offs,
                                        nullptr, st));
    }
    if (rows) {
        *rows = MoeRows{y2, tw, en2f, m.top_k, nullptr};
    }
    else {
        TM_TRY_RC(launch_moe_combine(out, ldo, y2, m.hidden, tw, en2f, tokens, m.hidden, m.top_k, st));
    }
    if (topk_ids_out) {
        TM_HIP_CHECK(hipMemcpyAsync(topk_ids_out, ids, pairs * 4, hipMemcpyDeviceToDevice, st));
    }
    if (topk_w_out) {
        TM_HIP_CHECK(hipMemcpyAsync(topk_w_out, tw, pairs * 4, hipMemcpyDeviceToDevice, st));
    }
    return 0;
}

void moe_free(MoeBlock& m)
{
    for (auto& l : m.w13) {
        linear_weight_free(l);
    }
    for (auto& l : m.w2) {
        linear_weight_free(l);
    }
    for (void* q : {(void*)m.gate, m.groups13, m.groups2, m.groups13_p8, m.groups2_p8}) {
        if (q) {
            (void)hipFree(q);
        }
    }
    m.gate = nullptr;
    m.groups13 = m.groups2 = nullptr;
    m.groups13_p8 = m.groups2_p8 = nullptr;
}

// ---- mixture of experts on the fp32 residual stream (layer-list family) -------------------------------------------------------------
// Router scores sigmoid(logit) from fp32 logits; the `k` largest win (ties: the lower index); the weights are the scores as they are.
__global__ void moe_topk_sigmoid_kernel(int* __restrict__ ids, float* __restrict__ w, const float* __restrict__ logits, int ld, int T, int E, int k)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) {
        return;
    }
    const float* z = logits + (size_t)t * ld;
    for (int j = 0; j < k; ++j) {
        int   best = -1;
        float bz   = 0.f;
        for (int e = 0; e < E; ++e) {
            bool taken = false;
            for (int q = 0; q < j; ++q) {
                taken = taken || ids[(size_t)t * k + q] == e;
            }
            if (!taken && (best < 0 || z[e] > bz)) {  // the sigmoid is monotonic: order by the logit
                best = e;
                bz   = z[e];
            }
        }
        ids[(size_t)t * k + j] = best;
        w[(size_t)t * k + j]   = 1.f / (1.f + expf(-bz));
    }
}

int launch_moe_topk_sigmoid(int* ids, float* w, const float* logits, int ld, int T, int E, int k, hipStream_t st)
{
    TM_REQUIRE(ids && w && logits && E >= 1 && k >= 1 && k <= E && ld >= E, "moe top-k: operands");
    if (T == 0) {
        return 0;
    }
    moe_topk_sigmoid_kernel<<<(T + 63) / 64, 64, 0, st>>>(ids, w, logits, ld, T, E, k);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// Router scores soft-max(logits) over all experts from fp32 logits; the `k` largest win (ties: the lower index); weight = scale * score.
__global__ void moe_topk_softmax_kernel(int* __restrict__ ids, float* __restrict__ w, const float* __restrict__ logits, int ld, int T, int E, int k,
                                        float scale)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) {
        return;
    }
    const float* z  = logits + (size_t)t * ld;
    float        mx = z[0];
    for (int e = 1; e < E; ++e) {
        mx = fmaxf(mx, z[e]);
    }
    float den = 0.f;
    for (int e = 0; e < E; ++e) {
        den += expf(z[e] - mx);
    }
    for (int j = 0; j < k; ++j) {
        int   best = -1;
        float bz   = 0.f;
        for (int e = 0; e < E; ++e) {
            bool taken = false;
            for (int q = 0; q < j; ++q) {
                taken = taken || ids[(size_t)t * k + q] == e;
            }
            if (!taken && (best < 0 || z[e] > bz)) {  // the soft-max is monotonic: order by the logit
                best = e;
                bz   = z[e];
            }
        }
        ids[(size_t)t * k + j] = best;
        w[(size_t)t * k + j]   = scale * (expf(bz - mx) / den);
    }
}

int launch_moe_softmax_route(int* ids, float* w, int* offsets, int* f2n, int* en2f, const float* logits, int ld, int T, int E, int k, float scale,
                             hipStream_t st)
{
    TM_REQUIRE(ids && w && logits && E >= 1 && k >= 1 && k <= E && ld >= E, "moe top-k: operands");
    if (T == 0) {
        return launch_moe_route(offsets, f2n, en2f, ids, T, E, k, st);
    }
    if (T <= kRouteTokens && E <= kRouteExperts) {
        moe_route_masks_kernel<true><<<1, 1024, 0, st>>>(offsets, f2n, en2f, ids, w, logits, ld, T, E, k, scale, {});
        TM_HIP_CHECK(hipGetLastError());
        return 0;
    }
    moe_topk_softmax_kernel<<<(T + 63) / 64, 64, 0, st>>>(ids, w, logits, ld, T, E, k, scale);
    TM_HIP_CHECK(hipGetLastError());
    return launch_moe_route(offsets, f2n, en2f, ids, T, E, k, st);
}

// Grouped router, one wave per token (four tokens per workgroup): the choice scores of a token lie in LDS, the lanes share the searches.
constexpr int kGroupedMaxExperts = 1024, kGroupedMaxGroups = 256;

__global__ __launch_bounds__(256) void moe_topk_grouped_kernel(int* __restrict__ ids, float* __restrict__ w, const float* __restrict__ logits, int ld,
                                                               const float* __restrict__ corr, int T, int E, int groups, int keep, int k, int renorm)
{
    extern __shared__ float lds_topk[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t = blockIdx.x * 4 + wave;
    float*    choice = lds_topk + (size_t)wave * (2 * E + groups);  // [E], choice score; then the group's place in the order below
    float*    score  = choice + E;                                   // [E]
    float*    gsum   = score + E;                                    // [groups]
    const bool on = t < T;
    if (on) {
        for (int e = lane; e < E; e += 64) {
            const float s = 1.f / (1.f + expf(-logits[(size_t)t * ld + e]));
            score[e]  = s;
            choice[e] = s + (corr ? corr[e] : 0.f);
        }
    }
    __syncthreads();
    const int per = E / groups;
    if (on && keep < groups) {
        for (int g = lane; g < groups; g += 64) {
            float a = -INFINITY, b = -INFINITY;  // the group's two best
            for (int e = g * per; e < (g + 1) * per; ++e) {
                const float c = choice[e];
                if (c > a) {
                    b = a, a = c;
                }
                else if (c > b) {
                    b = c;
                }
            }
            gsum[g] = per > 1 ? a + b : a;
        }
    }
    __syncthreads();
    if (on && keep < groups) {
        // group g stays if fewer than `keep` groups come before it; the others' experts leave the competition
        for (int g = lane; g < groups; g += 64) {
            int before = 0;
            for (int o = 0; o < groups; ++o) {
                before += gsum[o] > gsum[g] || (gsum[o] == gsum[g] && o < g);
            }
            if (before >= keep) {
                for (int e = g * per; e < (g + 1) * per; ++e) {
                    choice[e] = -INFINITY;
                }
            }
        }
    }
    __syncthreads();
    float sum = 0.f;
    for (int j = 0; j < k; ++j) {
        float v = -INFINITY;
        int   i = 0x7fffffff;
        if (on) {
            for (int e = lane; e < E; e += 64) {
                if (choice[e] > v) {
                    v = choice[e], i = e;
                }
            }
        }
        wave_argmax(v, i);
        i = min(i, E - 1);  // (the kept groups hold at least k experts: there is always a candidate)
        if (on) {
            const float s = score[i];
            sum += s;
            if (lane == 0) {
                ids[(size_t)t * k + j] = i;
                w[(size_t)t * k + j]   = s;
                choice[i]              = -INFINITY;
            }
        }
        __syncthreads();
    }
    if (on && renorm) {
        const float inv = 1.f / (sum + 1e-20f);
        for (int j = lane; j < k; j += 64) {
            w[(size_t)t * k + j] *= inv;  // (written by lane 0 of this wave, ahead of the barrier above)
        }
    }
}

int launch_moe_topk_grouped(int* ids, float* w, const float* logits, int ld, const float* correction, int T, int E, int groups, int keep, int k,
                            bool renorm, hipStream_t st)
{
    TM_REQUIRE(ids && w && logits && E >= 1 && E <= kGroupedMaxExperts && ld >= E, "moe grouped top-k: operands");
    TM_REQUIRE(groups >= 1 && groups <= kGroupedMaxGroups && E % groups == 0 && keep >= 1 && keep <= groups && k >= 1 && k <= E / groups * keep,
               "moe grouped top-k: the kept groups hold at least k experts");
    if (T == 0) {
        return 0;
    }
    const size_t lds = (size_t)4 * (2 * E + groups) * sizeof(float);
    moe_topk_grouped_kernel<<<(T + 3) / 4, 256, lds, st>>>(ids, w, logits, ld, correction, T, E, groups, keep, k, renorm);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// rows sorted by expert: xs[en2f[j][t]] = (scale ? w[t][j] : 1) * x[t] -- the weight on the expert's INPUT; V neighbouring channels a thread
template<class T, int V>
__global__ __launch_bounds__(256) void moe_gather_kernel(T* __restrict__ xs, int lds, const T* __restrict__ x, int ldx, const float* __restrict__ w,
                                                         const int* __restrict__ en2f, int Tn, int H, int k, int scale, int* __restrict__ shared_offsets,
                                                         int E)
{
    typedef T TV __attribute__((ext_vector_type(V)));
    const int kk = k + (shared_offsets ? 1 : 0);
    const int t = blockIdx.x / kk, j = blockIdx.x % kk;
    if (j == k) {  // the copy behind the routed rows
        if (t == 0 && threadIdx.x == 0) {
            shared_offsets[E + 1] = Tn * kk;
        }
        for (int i = threadIdx.x * V; i < H; i += 256 * V) {
            *(TV*)(xs + ((size_t)Tn * k + t) * lds + i) = *(const TV*)(x + (size_t)t * ldx + i);
        }
        return;
    }
    const int f = en2f[(size_t)j * Tn + t];
    const float a = scale ? w[(size_t)t * k + j] : 1.f;
    for (int i = threadIdx.x * V; i < H; i += 256 * V) {
        TV v = *(const TV*)(x + (size_t)t * ldx + i);
        if (scale) {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                v[e] = (T)(a * (float)v[e]);
            }
        }
        *(TV*)(xs + (size_t)f * lds + i) = v;
    }
}

template<class T>
static void launch_moe_gather_t(T* xs, int lds, const T* x, int ldx, const float* w, const int* en2f, int Tn, int H, int k, bool scale, int* shared_offsets,
                                int E, hipStream_t st)
{
    constexpr int V = 16 / sizeof(T);
    const int     wgs = Tn * (k + (shared_offsets ? 1 : 0));
    if (H % V == 0 && lds % V == 0 && ldx % V == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)xs % 16 == 0) {
        moe_gather_kernel<T, V><<<wgs, 256, 0, st>>>(xs, lds, x, ldx, w, en2f, Tn, H, k, scale, shared_offsets, E);
    }
    else {
        moe_gather_kernel<T, 1><<<wgs, 256, 0, st>>>(xs, lds, x, ldx, w, en2f, Tn, H, k, scale, shared_offsets, E);
    }
}

int launch_moe_gather(void* xs, int lds, const void* x, int ldx, int elem_bytes, const float* w, const int* en2f, int T, int H, int k, bool scale,
                      hipStream_t st, int* shared_offsets, int E)
{
    TM_REQUIRE(xs && x && w && en2f && lds >= H && ldx >= H, "moe gather: operands");
    if (T == 0) {
        return 0;
    }
    if (elem_bytes == 2) {
        launch_moe_gather_t((__bf16*)xs, lds, (const __bf16*)x, ldx, w, en2f, T, H, k, scale, shared_offsets, E, st);
    }
    else {
        launch_moe_gather_t((float*)xs, lds, (const float*)x, ldx, w, en2f, T, H, k, scale, shared_offsets, E, st);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class T>
static void launch_route_gather_t(int* ids, float* w, int* offsets, int* f2n, int* en2f, const float* logits, int ld, const MoeGather<T>& g, int Tn, int E, int k,
                                  float scale, hipStream_t st)
{
    constexpr int V   = 16 / sizeof(T);
    const int     wgs = (Tn * (k + g.shared) + 3) / 4;
    if (g.H % V == 0 && g.lds % V == 0 && g.ldx % V == 0 && (uintptr_t)g.x % 16 == 0 && (uintptr_t)g.xs % 16 == 0) {
        moe_route_masks_kernel<true, T, V><<<wgs, 1024, 0, st>>>(offsets, f2n, en2f, ids, w, logits, ld, Tn, E, k, scale, g);
    }
    else {
        moe_route_masks_kernel<true, T, 1><<<wgs, 1024, 0, st>>>(offsets, f2n, en2f, ids, w, logits, ld, Tn, E, k, scale, g);
    }
}

int launch_moe_softmax_route_gather(int* ids, float* w, int* offsets, int* f2n, int* en2f, const float* logits, int ld, void* xs, int lds, const void* x, int ldx,
                                    int elem_bytes, int T, int H, int E, int k, float scale, bool shared, hipStream_t st)
{
    // (more tokens than a mask has bits, or more choices than its list: one workgroup's tables no longer cost less than a launch of their own)
    if (T == 0 || T > kRouteTokens || E > kRouteExperts || T * k > kRoutePairs) {
        TM_TRY_RC(launch_moe_softmax_route(ids, w, offsets, f2n, en2f, logits, ld, T, E, k, scale, st));
        return launch_moe_gather(xs, lds, x, ldx, elem_bytes, w, en2f, T, H, k, false, st, shared ? offsets : nullptr, E);
    }
    TM_REQUIRE(ids && w && logits && E >= 1 && k >= 1 && k <= E && ld >= E, "moe top-k: operands");
    TM_REQUIRE(xs && x && lds >= H && ldx >= H, "moe gather: operands");
    if (elem_bytes == 2) {
        launch_route_gather_t(ids, w, offsets, f2n, en2f, logits, ld, MoeGather<__bf16>{(__bf16*)xs, lds, (const __bf16*)x, ldx, H, shared ? 1 : 0}, T, E, k, scale, st);
    }
    else {
        launch_route_gather_t(ids, w, offsets, f2n, en2f, logits, ld, MoeGather<float>{(float*)xs, lds, (const float*)x, ldx, H, shared ? 1 : 0}, T, E, k, scale, st);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// resid[t] += gate(t) * sum_j (weighted ? w[t][j] : 1) * y[en2f[j][t]], gate(t)[i] = sigmoid(gate[t][i] + gate_bias[i]) (gate == nullptr: 1);
// VEC neighbouring channels per thread (VEC = 4: H is a multiple of four)
template<int VEC>
__global__ void moe_combine_f32_kernel(float* __restrict__ resid, const float* __restrict__ y, const float* __restrict__ w, const int* __restrict__ en2f,
                                       const float* __restrict__ gate, int ldg, const float* __restrict__ gate_bias, int Tn, int H, int k, int weighted,
                                       int overwrite, const float* __restrict__ add, const float* __restrict__ add_gate, int ld_ag)
{
    typedef float VF __attribute__((ext_vector_type(VEC)));
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    if (i >= (size_t)Tn * H) {
        return;
    }
    const int t = (int)(i / H), c = (int)(i % H);
    VF        s = 0.f;
    for (int j = 0; j < k; j += 2) {  // two rows in flight
        const int   j1 = min(j + 1, k - 1);
        const int   f0 = en2f[(size_t)j * Tn + t], f1 = en2f[(size_t)j1 * Tn + t];
        const float w0 = weighted ? w[(size_t)t * k + j] : 1.f, w1 = weighted ? w[(size_t)t * k + j1] : 1.f;
        const VF    v0 = *(const VF*)(y + (size_t)f0 * H + c), v1 = *(const VF*)(y + (size_t)f1 * H + c);
        s += w0 * v0;
        if (j + 1 < k) {
            s += w1 * v1;
        }
    }
    if (gate) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            s[e] = s[e] / (1.f + expf(-(gate[(size_t)t * ldg + c + e] + gate_bias[c + e])));
        }
    }
    if (add) {
        const VF a = *(const VF*)(add + i);
        s = (add_gate ? a / (1.f + expf(-add_gate[(size_t)t * ld_ag])) : a) + s;
    }
    VF* out = (VF*)(resid + i);
    *out    = overwrite ? s : *out + s;
}

int launch_moe_combine_f32(float* resid, const float* y, const float* w, const int* en2f, const float* gate, int ldg, const float* gate_bias, int T,
                           int H, int k, bool weighted, hipStream_t st, bool overwrite, const float* add, const float* add_gate, int ld_add_gate)
{
    TM_REQUIRE(resid && y && w && en2f && (!gate || (gate_bias && ldg >= H)) && (!add || overwrite) && (!add_gate || add), "moe combine: operands");
    const size_t total = (size_t)T * H;
    if (total == 0) {
        return 0;
    }
    if (H % 4 == 0) {
        moe_combine_f32_kernel<4><<<(total / 4 + 255) / 256, 256, 0, st>>>(resid, y, w, en2f, gate, ldg, gate_bias, T, H, k, weighted, overwrite, add, add_gate, ld_add_gate);
    }
    else {
        moe_combine_f32_kernel<1><<<(total + 255) / 256, 256, 0, st>>>(resid, y, w, en2f, gate, ldg, gate_bias, T, H, k, weighted, overwrite, add, add_gate, ld_add_gate);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace tmk
