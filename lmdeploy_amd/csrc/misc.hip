// Small HBM-bound helpers: embedding lookup, greedy argmax, row gather, unfused SiLU*up, and the
// group-wise u4 quantiser used to fabricate synthetic AWQ weights on the device.
//
// Replaces: embeddingLookup (src/turbomind/kernels/decoding_kernels.cu via language_model.cc:232),
//           top-k(=1) sampling (generation/sampling.cc:92-183), CollectHiddenStates
//           (unified_decoder.cc:355-372), Activation (kernels/activation.cu:27-130),
//           QuantizeGroupwise / IntegralQuantizer (kernels/quantization.cu:384-440,515-676).
#include "tm_common.h"
#include "tm_kernels.h"
#include <algorithm>
#include <map>
#include <mutex>

namespace tmk {

__global__ __launch_bounds__(256) void embedding_kernel(half_t* __restrict__ out,
                                                        const half_t* __restrict__ table,
                                                        const int* __restrict__ ids,
                                                        int H,
                                                        int vocab)
{
    const int t  = blockIdx.x;
    int       id = ids[t];
    id           = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    for (int v = threadIdx.x; v < H / 8; v += 256) {
        *(half8_t*)(out + (size_t)t * H + v * 8) = *(const half8_t*)(table + (size_t)id * H + v * 8);
    }
}

int launch_embedding(half_t* out, const half_t* table, const int* ids, int T, int H, int vocab, hipStream_t st)
{
    TM_REQUIRE(H % 8 == 0, "H % 8");
    if (T == 0) {
        return 0;
    }
    embedding_kernel<<<T, 256, 0, st>>>(out, table, ids, H, vocab);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void gather_rows_kernel(half_t* __restrict__ out,
                                                          const half_t* __restrict__ in,
                                                          const int* __restrict__ rows,
                                                          int H)
{
    const int r = rows[blockIdx.x];
    for (int v = threadIdx.x; v < H / 8; v += 256) {
        *(half8_t*)(out + (size_t)blockIdx.x * H + v * 8) = *(const half8_t*)(in + (size_t)r * H + v * 8);
    }
}

int launch_gather_rows(half_t* out, const half_t* in, const int* rows, int n, int H, hipStream_t st)
{
    if (n == 0) {
        return 0;
    }
    gather_rows_kernel<<<n, 256, 0, st>>>(out, in, rows, H);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// greedy: argmax over fp32-cast logits, lowest index wins ties. One 1024-thread workgroup per row.
__global__ __launch_bounds__(1024) void argmax_kernel(int* __restrict__ out_ids,
                                                      half_t* __restrict__ out_val,
                                                      const half_t* __restrict__ logits,
                                                      int V,
                                                      int ld,
                                                      int id_offset)
{
    __shared__ float sv[16];
    __shared__ int   si[16];
    const int     row  = blockIdx.x;
    const half_t* lp   = logits + (size_t)row * ld;
    float         best = -INFINITY;
    int           bi   = 0x7fffffff;
    const int     nvec = V / 8;
    for (int v = threadIdx.x; v < nvec; v += 1024) {
        const half8_t x = *(const half8_t*)(lp + (size_t)v * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float f = (float)x[e];
            if (f > best) {  // ascending scan: strict > keeps the lowest index
                best = f;
                bi   = v * 8 + e;
            }
        }
    }
    for (int i = nvec * 8 + threadIdx.x; i < V; i += 1024) {
        const float f = (float)lp[i];
        if (f > best || (f == best && i < bi)) {
            best = f;
            bi   = i;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(best, off);
        const int   oi = __shfl_xor(bi, off);
        if (ov > best || (ov == best && oi < bi)) {
            best = ov;
            bi   = oi;
        }
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sv[wave] = best;
        si[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) {
            if (sv[w] > best || (sv[w] == best && si[w] < bi)) {
                best = sv[w];
                bi   = si[w];
            }
        }
        out_ids[row] = (bi == 0x7fffffff ? 0 : bi) + id_offset;
        if (out_val) {
            out_val[row] = (half_t)best;
        }
    }
}

int launch_argmax(int* out_ids, half_t* out_val, const half_t* logits, int B, int V, int ld, int id_offset, hipStream_t st)
{
    TM_REQUIRE(ld % 8 == 0, "logits rows must be 16-byte aligned");
    if (B == 0) {
        return 0;
    }
    argmax_kernel<<<B, 1024, 0, st>>>(out_ids, out_val, logits, V, ld, id_offset);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---- the end of a step: the greedy token of every row, and what a decode step does with it ----------------------------------------------
// Latency-bound: 256 KB a row at most, and what follows is a few words.  A row is shared by `parts` workgroups (kGreedyVec 16-byte vectors a thread, all
// in flight at once) that meet inside the launch; the last of a row writes its token, and for a decode step also the current id and the record, the last
// of all rows counts the step.  The layer-list families' fp32 logits become the fp16 rows on the way.  One workgroup a row, a copy and a record launch took
// 9.5 + 4.2 + 3.9 us of a step at one row of 128256 (64 rows: 10.5 + 4.5 + 4.1), this launch 5.3 (11.5); 32 fp32 rows of 32000 with the conversion 18.6, now 6.8.
constexpr int kGreedyVec = 4;
static int greedy_parts(int ld)
{
    return (ld / 8 + 256 * kGreedyVec - 1) / (256 * kGreedyVec);
}
size_t greedy_workspace_floats(int rows, int ld)
{
    return (size_t)rows * greedy_parts(ld) * 2;
}

__device__ __forceinline__ void greedy_better(float& v, int& i, float ov, int oi)
{
    const bool b = ov > v || (ov == v && oi < i);
    v            = b ? ov : v;
    i            = b ? oi : i;
}

// 8 logits of the fp16 rows: read there, or made of the fp32 row (pad columns can never win an arg-max)
template<class T, bool WIDE>
__device__ __forceinline__ half8_t greedy_load(const T* __restrict__ row, int c, int V)
{
    if constexpr (sizeof(T) == 2) {
        return *(const half8_t*)(row + c);
    }
    else {
        float f[8];
        if constexpr (WIDE) {
            const floatx4 a = *(const floatx4*)(row + min(c, V - 4)), b = *(const floatx4*)(row + min(c + 4, V - 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = a[e], f[4 + e] = b[e];
            }
        }
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                f[e] = row[min(c + e, V - 1)];
            }
        }
        half8_t h;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            h[e] = (half_t)(c + e < V ? fminf(fmaxf(f[e], -65504.f), 65504.f) : -65504.f);
        }
        return h;
    }
}

template<class T, bool WIDE>
__global__ __launch_bounds__(256) void greedy_kernel(int* __restrict__ out_ids, half_t* __restrict__ rows16, int ld, const T* __restrict__ logits, int ldl, int V,
                                                     float* __restrict__ ws, unsigned* __restrict__ tickets, StepCommit cm)
{
    __shared__ float sv[4];
    __shared__ int   si[4];
    const int row = blockIdx.y, parts = gridDim.x, tid = threadIdx.x, nvec = ld / 8;
    // (asked for ahead of the row: it changes only once every row's token is out)
    const int step = cm.step ? __hip_atomic_load(cm.step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    half8_t   x[kGreedyVec];
    int       at[kGreedyVec];
#pragma unroll
    for (int u = 0; u < kGreedyVec; ++u) {  // (the last vector again beyond the row's end: it is not lower in index, nor higher in value)
        at[u] = min(((int)blockIdx.x * kGreedyVec + u) * 256 + tid, nvec - 1);
        x[u]  = greedy_load<T, WIDE>(logits + (size_t)row * ldl, at[u] * 8, V);
    }
    float best = -INFINITY;
    int   bi   = 0x7fffffff;
#pragma unroll
    for (int u = 0; u < kGreedyVec; ++u) {
        if constexpr (sizeof(T) == 4) {
            *(half8_t*)(rows16 + (size_t)row * ld + (size_t)at[u] * 8) = x[u];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float f = (float)x[u][e];
            if (f > best) {  // ascending scan: strict > keeps the lowest index
                best = f;
                bi   = at[u] * 8 + e;
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(best, off);
        const int   oi = __shfl_xor(bi, off);
        greedy_better(best, bi, ov, oi);
    }
    if ((tid & 63) == 0) {
        sv[tid >> 6] = best;
        si[tid >> 6] = bi;
    }
    __syncthreads();
    if (tid >= 64) {
        return;
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        greedy_better(best, bi, sv[w], si[w]);
    }
    if (parts > 1) {
        float* const mine = ws + ((size_t)row * parts + blockIdx.x) * 2;
        if (tid == 0) {
            agent_store(mine, best);
            agent_store(mine + 1, __int_as_float(bi));
        }
        if (!ticket_last_wave(tickets + row, parts)) {
            return;
        }
        best = -INFINITY;
        bi   = 0x7fffffff;
        for (int p = tid; p < parts; p += 64) {
            const float* o = ws + ((size_t)row * parts + p) * 2;
            greedy_better(best, bi, agent_load(o), __float_as_int(agent_load(o + 1)));
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(best, off);
            const int   oi = __shfl_xor(bi, off);
            greedy_better(best, bi, ov, oi);
        }
    }
    if (tid != 0) {
        return;
    }
    const int id = bi == 0x7fffffff ? 0 : bi;
    out_ids[row] = id;
    if (cm.cur_ids) {
        cm.cur_ids[row] = id;
    }
    if (cm.step) {
        if (step < cm.max_new) {
            cm.generated[(size_t)row * cm.max_new + step] = id;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (ticket_last(tickets + gridDim.y, gridDim.y)) {
            __hip_atomic_store(cm.step, step + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

int launch_greedy(int* out_ids, half_t* rows16, int ld, const float* logits32, int V, int rows, float* ws, size_t ws_floats, unsigned* tickets, int ticket_count,
                  const StepCommit& cm, hipStream_t st)
{
    TM_REQUIRE(out_ids && rows16 && ws && tickets && ld >= V && V >= 1 && ld % 8 == 0, "greedy: operands (logits rows of 16-byte vectors)");
    TM_REQUIRE(!cm.step || (cm.cur_ids && cm.generated), "greedy: a step's record");
    TM_REQUIRE(greedy_workspace_floats(rows, ld) <= ws_floats && rows < ticket_count && rows <= 65535, "greedy: workspace");
    if (rows == 0) {
        return 0;
    }
    const dim3 grid(greedy_parts(ld), rows);
    if (!logits32) {
        greedy_kernel<half_t, true><<<grid, 256, 0, st>>>(out_ids, nullptr, ld, rows16, ld, V, ws, tickets, cm);
    }
    else if (V % 4 == 0 && (uintptr_t)logits32 % 16 == 0) {
        greedy_kernel<float, true><<<grid, 256, 0, st>>>(out_ids, rows16, ld, logits32, V, V, ws, tickets, cm);
    }
    else {
        greedy_kernel<float, false><<<grid, 256, 0, st>>>(out_ids, rows16, ld, logits32, V, V, ws, tickets, cm);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// the same commit for tokens that another kernel chose: ids become the current ids and are appended to generated[b][step]; step++ (a single thread does the
// counter after everybody read it)
__global__ void commit_kernel(const int* __restrict__ ids, int n, StepCommit cm)
{
    const int step = cm.step ? *cm.step : 0;
    for (int b = threadIdx.x; b < n; b += blockDim.x) {
        const int id  = ids[b];
        cm.cur_ids[b] = id;
        if (cm.step && step < cm.max_new) {
            cm.generated[(size_t)b * cm.max_new + step] = id;
        }
    }
    __syncthreads();
    if (cm.step && threadIdx.x == 0) {
        *cm.step = step + 1;
    }
}

int launch_commit(const int* ids, int n, const StepCommit& cm, hipStream_t st)
{
    TM_REQUIRE(ids && cm.cur_ids && (!cm.step || cm.generated), "commit: operands");
    commit_kernel<<<1, std::min(1024, std::max(64, (n + 63) / 64 * 64)), 0, st>>>(ids, n, cm);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// unfused activation on a [M][2*inter] buffer laid out [gate | up]
// Pseudo-random fp16 values in (-amp, amp) -- stand-in activations for the start-up GEMM tuner.  Not zeros: the matrix pipe
// of MI355X is power-limited, and a GEMM over all-zero activations runs at the full 2.4 GHz instead of the ~1.6 GHz it sustains
// on real data (measured: the fused w1w3 prefill tile 1152 us on zeros, 1697 us on N(0,1) rows) -- timings on zeros rank
// compute-bound candidates wrongly.
__global__ __launch_bounds__(256) void fill_uniform_f16_kernel(half_t* __restrict__ out, size_t n, float amp, uint32_t seed)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    uint32_t h = (uint32_t)i * 0x9E3779B1u + (uint32_t)(i >> 32) + seed;  // one round of a 32-bit integer hash
    h ^= h >> 16;
    h *= 0x7feb352du;
    h ^= h >> 15;
    h *= 0x846ca68bu;
    h ^= h >> 16;
    out[i] = (half_t)(((float)(h >> 8) * (1.0f / 8388608.0f) - 1.0f) * amp);
}

int launch_fill_uniform_f16(half_t* out, size_t n, float amp, uint32_t seed, hipStream_t st)
{
    if (n == 0) {
        return 0;
    }
    fill_uniform_f16_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(out, n, amp, seed);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void silu_mul_kernel(half_t* __restrict__ out,
                                                       const half_t* __restrict__ gate_up,
                                                       int M,
                                                       int inter)
{
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)M * inter / 8) {
        return;
    }
    const int     m = idx / (inter / 8);
    const int     c = (idx - (size_t)m * (inter / 8)) * 8;
    const half8_t g = *(const half8_t*)(gate_up + (size_t)m * 2 * inter + c);
    const half8_t u = *(const half8_t*)(gate_up + (size_t)m * 2 * inter + inter + c);
    half8_t       o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float gf = (float)g[e];
        o[e]           = (half_t)(silu_f32(gf) * (float)u[e]);
    }
    *(half8_t*)(out + (size_t)m * inter + c) = o;
}

int launch_silu_mul(half_t* out, const half_t* gate_up, int M, int inter, hipStream_t st)
{
    TM_REQUIRE(inter % 8 == 0, "inter % 8");
    const size_t total = (size_t)M * inter / 8;
    if (total == 0) {
        return 0;
    }
    silu_mul_kernel<<<(total + 255) / 256, 256, 0, st>>>(out, gate_up, M, inter);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// IntegralQuantizer<half,4>: groups of `group` along K for every output column n.
//   scale_ = max(max-min, 1e-5)/15 ; zero_ = clamp(-rint(min/scale_), 0, 15)
//   q = clamp(rint(x/scale_) + zero_, 0, 15) ; d = h(q - zero_) * h(scale_)
// Output in the boundary layout: qweight int32 [K][N/8] (nibble j of word c = column 8c+j).
__global__ __launch_bounds__(256) void quantize_groupwise_u4_kernel(int32_t* __restrict__ qweight,
                                                                    half_t* __restrict__ scales,
                                                                    half_t* __restrict__ zeros,
                                                                    half_t* __restrict__ dequant,
                                                                    const half_t* __restrict__ w,
                                                                    int K,
                                                                    int N,
                                                                    int group)
{
    // one thread per (group, 8 consecutive columns)
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int    nc  = N / 8;
    if (idx >= (size_t)(K / group) * nc) {
        return;
    }
    const int gi = idx / nc;
    const int c  = idx - (size_t)gi * nc;
    float     mn[8], mx[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        mn[e] = INFINITY;
        mx[e] = -INFINITY;
    }
    for (int k = gi * group; k < (gi + 1) * group; ++k) {
        const half8_t x = *(const half8_t*)(w + (size_t)k * N + c * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mn[e] = fminf(mn[e], (float)x[e]);
            mx[e] = fmaxf(mx[e], (float)x[e]);
        }
    }
    float sc[8];
    int   zp[8];
    half8_t s_out, z_out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        sc[e]    = fmaxf(mx[e] - mn[e], 1e-5f) / 15.0f;
        int z    = (int)(-__builtin_rintf(mn[e] / sc[e]));
        zp[e]    = z < 0 ? 0 : (z > 15 ? 15 : z);
        s_out[e] = (half_t)sc[e];
        z_out[e] = (half_t)(float)zp[e];
    }
    *(half8_t*)(scales + (size_t)gi * N + c * 8) = s_out;
    *(half8_t*)(zeros + (size_t)gi * N + c * 8)  = z_out;
    for (int k = gi * group; k < (gi + 1) * group; ++k) {
        const half8_t x = *(const half8_t*)(w + (size_t)k * N + c * 8);
        uint32_t      word = 0;
        half8_t       d;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            int q = (int)__builtin_rintf((float)x[e] / sc[e]) + zp[e];
            q     = q < 0 ? 0 : (q > 15 ? 15 : q);
            word |= (uint32_t)q << (4 * e);
            d[e] = (half_t)(float)(q - zp[e]) * s_out[e];
        }
        qweight[(size_t)k * nc + c] = (int32_t)word;
        if (dequant) {
            *(half8_t*)(dequant + (size_t)k * N + c * 8) = d;
        }
    }
}

int launch_quantize_groupwise_u4(int32_t* qweight, half_t* scales, half_t* zeros, half_t* dequant, const half_t* w,
                                 int K, int N, int group, hipStream_t st)
{
    TM_REQUIRE(N % 8 == 0 && K % group == 0, "N % 8 == 0, K % group == 0");
    const size_t total = (size_t)(K / group) * (N / 8);
    if (total == 0) {
        return 0;
    }
    quantize_groupwise_u4_kernel<<<(total + 255) / 256, 256, 0, st>>>(qweight, scales, zeros, dequant, w, K, N, group);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

int ensure_dynamic_lds(const void* kernel, int bytes)
{
    static std::mutex                               mu;
    static std::map<std::pair<const void*, int>, int> done;  // (kernel, device) -> bytes granted
    int dev = 0;
    TM_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    auto                        it = done.find({kernel, dev});
    if (it != done.end() && it->second >= bytes) {
        return 0;
    }
    TM_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    done[{kernel, dev}] = bytes;
    return 0;
}


// The embedding rows as the fp32 stream, grid (row, chunk of V * 256 columns).  A decode step's first launch: row t is sequence t's one token, so its context
// length grows here (begin.active: where a sequence runs) and its place is written, which were launches of their own: 14.1 -> 4.7 us (32 rows of 4096).
// Four columns a thread, no division: 8192 rows of 4096 bf16 channels 94 -> 37 us.
template<class T, int V>
__global__ __launch_bounds__(256) void embedding_f32_kernel(float* __restrict__ out, const T* __restrict__ table, const int* __restrict__ ids, int H, int vocab,
                                                            float scale, float* __restrict__ out2, StepBegin begin, int* __restrict__ row_seq, int* __restrict__ row_pos)
{
    typedef T     TV __attribute__((ext_vector_type(V)));
    typedef float FV __attribute__((ext_vector_type(V)));
    const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * V;
    int       id = ids[t];
    id           = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    if (begin.k_len && blockIdx.y == 0 && threadIdx.x == 0) {
        const int len = begin.k_len[t] + (!begin.active || begin.active[t] ? 1 : 0);
        begin.k_len[t] = len;
        row_seq[t]     = t;
        row_pos[t]     = len - 1;
    }
    if (c < H) {
        const TV v = *(const TV*)(table + (size_t)id * H + c);
        FV       o;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            o[e] = (float)v[e] * scale;
        }
        *(FV*)(out + (size_t)t * H + c) = o;
        if (out2) {
            *(FV*)(out2 + (size_t)t * H + c) = o;
        }
    }
}

int launch_embedding_f32(float* out, const void* table, int table_elem_bytes, const int* ids, int T, int H, int vocab, hipStream_t st, float scale,
                         float* out2, const StepBegin& begin, int* row_seq, int* row_pos)
{
    TM_REQUIRE(out && table && ids && (table_elem_bytes == 2 || table_elem_bytes == 4), "embedding_f32: operands");
    TM_REQUIRE(!begin.k_len || (row_seq && row_pos), "embedding_f32: a step's rows");
    if (T == 0 || H == 0) {
        return 0;
    }
    const bool four = H % 4 == 0 && ((uintptr_t)out | (uintptr_t)out2 | (uintptr_t)table) % 16 == 0;
    const dim3 grid(T, four ? (H + 1023) / 1024 : (H + 255) / 256);
#define TM_EMBED(T_, V_) embedding_f32_kernel<T_, V_><<<grid, 256, 0, st>>>(out, (const T_*)table, ids, H, vocab, scale, out2, begin, row_seq, row_pos)
    if (table_elem_bytes == 2) {
        four ? TM_EMBED(__bf16, 4) : TM_EMBED(__bf16, 1);
    }
    else {
        four ? TM_EMBED(float, 4) : TM_EMBED(float, 1);
    }
#undef TM_EMBED
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

__global__ void f32_to_f16_rows_kernel(half_t* __restrict__ out, int ld, const float* __restrict__ in, int n, int V)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (size_t)n * ld) {
        const int r = (int)(i / ld), c = (int)(i % ld);
        const float v = c < V ? in[(size_t)r * V + c] : -65504.f;  // pad columns can never win an arg-max
        out[i] = (half_t)fminf(fmaxf(v, -65504.f), 65504.f);
    }
}

int launch_f32_to_f16_rows(half_t* out, int ld, const float* in, int n, int V, hipStream_t st)
{
    TM_REQUIRE(out && in && ld >= V, "f32_to_f16_rows: operands");
    const size_t cnt = (size_t)n * ld;
    if (cnt > 0) {
        f32_to_f16_rows_kernel<<<(cnt + 255) / 256, 256, 0, st>>>(out, ld, in, n, V);
        TM_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

// ---- fp32 stream helpers of the layer-list family ------------------------------------------------------------------------------------
// out[m] = [a[m] | b[m]] in the activation type: two fp32 streams side by side as the operand of one product
template<class T>
__global__ void concat2_kernel(T* __restrict__ out, int ldo, const float* __restrict__ a, const float* __restrict__ b, int H, size_t total)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) {
        const size_t m = i / (2 * H);
        const int    c = (int)(i % (2 * H));
        out[m * ldo + c] = (T)(c < H ? a[m * H + c] : b[m * H + c - H]);
    }
}

int launch_concat2(void* out, int ldo, int out_elem_bytes, const float* a, const float* b, int M, int H, hipStream_t st)
{
    TM_REQUIRE(out && a && b && ldo >= 2 * H && (out_elem_bytes == 2 || out_elem_bytes == 4), "concat2: operands");
    const size_t total = (size_t)M * 2 * H;
    if (total == 0) {
        return 0;
    }
    if (out_elem_bytes == 2) {
        concat2_kernel<__bf16><<<(total + 255) / 256, 256, 0, st>>>((__bf16*)out, ldo, a, b, H, total);
    }
    else {
        concat2_kernel<float><<<(total + 255) / 256, 256, 0, st>>>((float*)out, ldo, a, b, H, total);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---- mixer outputs on their way to the output projection ------------------------------------------------------------------------------
// differential attention: one wave per (row, head) joins the head's two maps, o = a1 - lambda a2, and scales o to unit RMS (times mult)
template<class T>
__global__ __launch_bounds__(256) void diff_head_norm_kernel(T* __restrict__ y, int ldy, const float* __restrict__ a, int lda,
                                                             const float* __restrict__ lambda, float mult, int heads, int n, float eps)
{
    const int t = blockIdx.x, h = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= heads) {
        return;
    }
    const float  lam = lambda[0];
    const float *a1 = a + (size_t)t * lda + (size_t)h * n, *a2 = a1 + (size_t)heads * n;
    float        ss = 0.f;
    for (int i = lane; i < n; i += 64) {
        const float o = fmaf(-lam, a2[i], a1[i]);
        ss            = fmaf(o, o, ss);
    }
    const float inv = mult / sqrtf(group_sum<64>(ss) / (float)n + eps);
    for (int i = lane; i < n; i += 64) {
        y[(size_t)t * ldy + (size_t)h * n + i] = (T)(fmaf(-lam, a2[i], a1[i]) * inv);
    }
}

int launch_diff_head_norm(void* y, int ldy, int out_elem_bytes, const float* a, int lda, const float* lambda, float mult, int rows, int heads, int n,
                          float eps, hipStream_t st)
{
    TM_REQUIRE(y && a && lambda && heads >= 1 && n >= 1 && ldy >= heads * n && lda >= 2 * heads * n && (out_elem_bytes == 2 || out_elem_bytes == 4),
               "diff_head_norm: operands");
    if (rows == 0) {
        return 0;
    }
    const dim3 grid(rows, (heads + 3) / 4);
    if (out_elem_bytes == 2) {
        diff_head_norm_kernel<__bf16><<<grid, 256, 0, st>>>((__bf16*)y, ldy, a, lda, lambda, mult, heads, n, eps);
    }
    else {
        diff_head_norm_kernel<float><<<grid, 256, 0, st>>>((float*)y, ldy, a, lda, lambda, mult, heads, n, eps);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class T>
__global__ void sigmoid_gate_mul_kernel(T* __restrict__ y, int ldy, const float* __restrict__ x, int ldx, const float* __restrict__ gate, int ldg,
                                        int rows, int n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (size_t)rows * n) {
        const int t = (int)(i / n), c = (int)(i % n);
        y[(size_t)t * ldy + c] = (T)(x[(size_t)t * ldx + c] / (1.f + expf(-gate[(size_t)t * ldg + c])));
    }
}

int launch_sigmoid_gate_mul(void* y, int ldy, int out_elem_bytes, const float* x, int ldx, const float* gate, int ldg, int rows, int n, hipStream_t st)
{
    TM_REQUIRE(y && x && gate && n >= 1 && ldy >= n && ldx >= n && ldg >= n && (out_elem_bytes == 2 || out_elem_bytes == 4), "sigmoid_gate_mul: operands");
    const size_t total = (size_t)rows * n;
    if (total == 0) {
        return 0;
    }
    if (out_elem_bytes == 2) {
        sigmoid_gate_mul_kernel<__bf16><<<(total + 255) / 256, 256, 0, st>>>((__bf16*)y, ldy, x, ldx, gate, ldg, rows, n);
    }
    else {
        sigmoid_gate_mul_kernel<float><<<(total + 255) / 256, 256, 0, st>>>((float*)y, ldy, x, ldx, gate, ldg, rows, n);
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

__global__ void softcap_f32_kernel(float* __restrict__ x, size_t n, float cap)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x[i] = cap * tanhf(x[i] / cap);
    }
}

int launch_softcap_f32(float* x, size_t n, float cap, hipStream_t st)
{
    TM_REQUIRE(x && cap > 0.f, "softcap_f32: operands");
    if (n > 0) {
        softcap_f32_kernel<<<(n + 255) / 256, 256, 0, st>>>(x, n, cap);
        TM_HIP_CHECK(hipGetLastError());
    }
    return 0;
}

}  // namespace tmk
