// Dense linears with unquantised weights: y = x . W^T for W stored [N][K] (the checkpoint's own orientation), in two number formats.
//
//   bf16 : weights and activations bfloat16, fp32 accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).
//   fp32 : activations fp32, weights as they come (bf16, every one an fp32 number), multiplied and added in 32 bits: a row's numbers are split
//          into three of bf16 on the way to the matrix cores (StreamOp).
//
// The kernels are gemm_stream.h's: the weight stream for up to 64 rows (a decode step), tiles staged in LDS for more (prompts).
// Weights are kept as zero-padded images of Np x Kp elements in fragment order (Np % 128 == 0, Kp % 32 == 0; dense_frag_index): no bounds
// test in any inner loop.  Activation rows have a leading dimension >= Kp; what lies in their pad columns only has to be finite, it
// meets zero weights.
//
// The epilogue is chosen per call (DenseEpilogue): plain store, relu(x)^2 (the squared-ReLU feed-forward), accumulate into the fp32
// residual stream with a multiplier (resid += alpha * acc: the output projection of a residual block closes the block in the GEMM),
// (optionally with a copy of the new stream in the activation type), act(acc) times a row of a table chosen by the row's token id,
// or alpha * acc as fp32 (scaled logits), acc + bias[n] as fp32, or the sigmoid-gated residual sum
// resid += sigmoid(gate[m][n] + gate_bias[n]) * acc (a block whose sublayers are gated element by element).
//
// A launch may be BATCHED (DenseCall::count > 1, grid z): item g multiplies with image g of the weight (images at a fixed stride), reads
// x at column g * x_col_stride and writes y at column g * y_col_stride -- per-head projections of one activation row -- or, with
// row_offsets, owns the rows [row_offsets[g], row_offsets[g + 1]) of x and y: the experts of a mixture over rows sorted by expert.
// A launch may also have SEGMENTS (DenseCall::n_seg): ranges of output columns that read x at columns of their own -- the projections of
// several inputs derived from one token (each its own mix of the token and its predecessor) as one product of any widths.
#include "tm_kernels.h"
#include "gemm_stream.h"
#include <algorithm>
#include <numeric>

namespace tmk {

// gate / up pairs of a gated feed-forward (the branch on the activation is outside the loop: N independent chains)
template<int N>
__device__ __forceinline__ void dense_gated(const DenseCall& c, const float (&g)[N], const float (&u)[N], float (&r)[N])
{
    if (c.act == kActClamped) {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const float gc = fminf(g[e], c.act_limit), uc = fminf(fmaxf(u[e], -c.act_limit), c.act_limit);
            r[e]           = gc / (1.f + expf(-c.act_alpha * gc)) * (uc + 1.f);
        }
    }
    else if (c.act == kActGeluTanh) {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            r[e] = act_apply(kActGeluTanh, g[e]) * u[e];
        }
    }
    else if (c.act == kActSilu) {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            r[e] = act_apply(kActSilu, g[e]) * u[e];
        }
    }
    else {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            r[e] = act_apply(c.act, g[e]) * u[e];
        }
    }
}

// where an item of a batched launch starts (bytes), and its row count (<= 0: nothing to do)
struct DenseItem {
    int64_t x_off, w_off;
    int     row_base, col_base, M;
};

// N consecutive elements of a row, as one store where the row allows it (`vec`: rows and columns aligned to the vector)
template<class O, int N>
__device__ __forceinline__ void store_run(O* y, size_t i, const float (&v)[N], bool vec, int left)
{
    typedef O run_t __attribute__((ext_vector_type(N)));
    if (vec && left >= N) {
        run_t o;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            o[e] = (O)v[e];
        }
        *(run_t*)(y + i) = o;
        return;
    }
#pragma unroll
    for (int e = 0; e < N; ++e) {
        if (e < left) {
            y[i + e] = (O)v[e];
        }
    }
}

// Epilogues on four consecutive columns n .. n + 3 of row m.  EPI >= 0: known at compile time (a kernel with many outputs per thread must not
// carry every epilogue per output: the unroller gives up and the accumulators land in scratch memory); -1: the call's own
template<class T, int EPI>
struct DenseEpi {
    DenseCall c;
    int       vec;  // rows of y (and of the operands read beside it) start at multiples of 16 bytes

    static constexpr bool kPairs = EPI == kDenseGatedAct && sizeof(T) == 2;
    static constexpr bool kTileRuns = true;
    // What an output needs besides its product: the stream's element or its bias.  Where a lane of a 256 x 256 tile has its outputs, their operands are
    // asked for together (read), before the first of them is stored (join): a load that follows a store which may have written there waits in line, and a tile's 64
    // outputs a lane paid 64 trips to memory one after the other.  us, one by one / sixteen together: 8010 rows of bf16 into the stream, (2048, 2048) 104 / 85,
    // (8448, 2048) 275 / 253; 8000 rows of (2048, 2050) 97 / 92.  Not in the smaller tiles, whose other workgroup on the CU covers the trips: 128 x 128 and 256 x 128
    // took 1 - 7 % longer with it ((2048, 2048) 2500 rows 39.7 / 41.4), a ragged edge 16 % ((1000, 3000) 2500 rows 32.2 / 37.4)
    static constexpr int kReads = EPI == kDenseResidAdd || EPI == kDenseBiasF32 ? 16 : 0;  // so many at a time
    struct Operand {
        floatx4 v;
    };
    template<bool WHOLE>
    __device__ __forceinline__ Operand read(const StreamArgs& a, const DenseItem& it, int m, int n) const
    {
        typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));
        const float*  at = EPI == kDenseBiasF32 ? c.bias + n : (const float*)a.y + (size_t)(m + it.row_base) * a.ldy + it.col_base + n;
        if constexpr (WHOLE) {
            return {*(const float4_any*)at};
        }
        Operand o = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (n + e < a.N) {
                o.v[e] = at[e];
            }
        }
        return o;
    }
    // the operands of N outputs: output j is row at(j).x of the item, columns at(j).y .. + 3
    template<int N, class At>
    __device__ __forceinline__ void operands(const StreamArgs& a, const DenseItem& it, At&& at, Operand (&op)[N]) const
    {
        bool whole = true;  // (the loads need no alignment but their elements')
#pragma unroll
        for (int j = 0; j < N; ++j) {
            whole = whole && at(j).y + 4 <= a.N;
        }
        if (whole) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                op[j] = read<true>(a, it, at(j).x, at(j).y);
            }
        }
        else {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                op[j] = read<false>(a, it, at(j).x, at(j).y);
            }
        }
    }
    __device__ __forceinline__ void join(const StreamArgs& a, const DenseItem& it, int m, int n, floatx4 acc, const Operand& op) const
    {
        const int left = a.N - n;
        if (left <= 0) {
            return;
        }
        m += it.row_base;
        const size_t i = (size_t)m * a.ldy + it.col_base + n;
        float        r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            r[e] = EPI == kDenseBiasF32 ? acc[e] + op.v[e] : op.v[e] + c.alpha * acc[e];
        }
        store_run<float, 4>((float*)a.y, i, r, vec, left);
        if (EPI == kDenseResidAdd && c.y2) {
            store_run<T, 4>((T*)c.y2, (size_t)m * c.ldy2 + n, r, vec, left);
        }
    }
    __device__ __forceinline__ const int* row_offsets() const
    {
        return c.row_offsets;
    }
    __device__ __forceinline__ int items() const
    {
        return c.count;
    }
    __device__ __forceinline__ DenseItem item(int g, int M, int n0) const
    {
        DenseItem it{(int64_t)g * c.x_col_stride, (int64_t)g * (int64_t)c.w_stride, 0, g * c.y_col_stride, M};
#pragma unroll
        for (int s = 1; s < kDenseMaxSeg; ++s) {  // (the segment of this workgroup's columns: the plan takes no tile that holds a border)
            it.x_off += s < c.n_seg && n0 >= c.seg_n0[s] ? c.x_col_stride : 0;
        }
        if (c.row_offsets) {
            it.row_base = c.row_offsets[g];
            it.x_off += (int64_t)it.row_base * c.ldx;
            it.M = c.row_offsets[g + 1] - it.row_base;
        }
        it.x_off *= sizeof(T), it.w_off *= 2;
        return it;
    }
    // asks early for what an output is added to (its first element brings the line); whoever calls it keeps the result until rows()
    __device__ __forceinline__ unsigned touch(const StreamArgs& a, const DenseItem& it, int m, int n) const
    {
        const int epi = EPI >= 0 ? EPI : c.epi;
        return epi == kDenseResidAdd || epi == kDenseResidGate ? ((const unsigned*)a.y)[(size_t)(m + it.row_base) * a.ldy + it.col_base + n] : 0u;
    }
    // acc[j]: columns n + 16 j .. + 3
    template<int NT>
    __device__ __forceinline__ void rows(const StreamArgs& a, const DenseItem& it, int m, int n, const floatx4 (&acc)[NT]) const
    {
        const int epi = EPI >= 0 ? EPI : c.epi;
        m += it.row_base;
        if (epi == kDenseGatedAct) {
            if constexpr (sizeof(T) == 4) {  // the four columns are gate, gate, up, up of two outputs
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int   o    = (n + 16 * j) >> 1;
                    const float g[2] = {acc[j][0], acc[j][1]}, u[2] = {acc[j][2], acc[j][3]};
                    float       r[2];
                    dense_gated(c, g, u, r);
                    store_run<T, 2>((T*)a.y, (size_t)m * a.ldy + it.col_base + o, r, vec, c.n_out - o);
                }
            }
            else if constexpr (NT % 2 == 0) {  // tiles 2 j, 2 j + 1 of the image are the gate / up halves of output tile j
#pragma unroll
                for (int j = 0; j < NT; j += 2) {
                    const int n16 = n & ~15, o = (n16 >> 1) + (n & 15) + 8 * j;
                    const float g[4] = {acc[j][0], acc[j][1], acc[j][2], acc[j][3]}, u[4] = {acc[j + 1][0], acc[j + 1][1], acc[j + 1][2], acc[j + 1][3]};
                    float       r[4];
                    dense_gated(c, g, u, r);
                    store_run<T, 4>((T*)a.y, (size_t)m * a.ldy + it.col_base + o, r, vec, c.n_out - o);
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            one(a, it, m, n + 16 * j, acc[j], epi);
        }
    }
    __device__ __forceinline__ void one(const StreamArgs& a, const DenseItem& it, int m, int n, floatx4 acc, int epi) const
    {
        const int left = a.N - n;
        if (left <= 0) {
            return;
        }
        if (epi == kDenseStoreRelu2) {
            float r[4];
            if (n >= c.split_n) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float z = fmaxf(acc[e], 0.f);
                    r[e]          = z * z;
                }
                store_run<T, 4>((T*)c.y2, (size_t)m * c.ldy2 + n - c.split_n, r, vec, left);
                return;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r[e] = acc[e];
            }
            if (EPI >= 0 || !c.kv.block_ptrs || n + 4 <= c.kv.k_col) {
                if (n < c.first_n) {
                    store_run<T, 4>((T*)a.y, (size_t)m * a.ldy + n, r, vec, c.first_n - n);
                }
                return;
            }
            const int s = c.kv.row_seq[m], pos = c.kv.row_pos[m], ti = pos % c.kv.block_len;
            char* const base = global_ptr(c.kv.block_ptrs[(size_t)(c.kv.seq_slot ? c.kv.seq_slot[s] : s) * c.kv.block_stride + pos / c.kv.block_len]) + c.kv.layer_offset;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = n + e;
                if (col >= c.first_n) {
                    break;
                }
                if (col < c.kv.k_col) {
                    ((T*)a.y)[(size_t)m * a.ldy + col] = (T)r[e];
                }
                else if (col < c.kv.v_col) {
                    const int g = (col - c.kv.k_col) / c.kv.dim, d = (col - c.kv.k_col) % c.kv.dim;
                    ((T*)base)[((size_t)g * c.kv.block_len + ti) * c.kv.dim + d] = (T)r[e];
                }
                else {
                    const int g = (col - c.kv.v_col) / c.kv.vdim, d = (col - c.kv.v_col) % c.kv.vdim;
                    ((T*)(base + c.kv.v_offset))[((size_t)g * c.kv.vdim + d) * c.kv.block_len + ti] = (T)r[e];
                }
            }
            return;
        }
        const size_t i = (size_t)m * a.ldy + it.col_base + n;
        float        r[4];
        if (epi == kDenseStore || epi == kDenseRelu2 || epi == kDenseXielu || epi == kDenseActTable) {
            if (epi == kDenseXielu) {
                const float p = c.act_par[0], q = c.act_par[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float z = acc[e];
                    r[e]          = z > 0.f ? fmaf(p * z, z, 0.5f * z) : fmaf(q, expm1f(z) - z, 0.5f * z);
                }
            }
            else if (epi == kDenseActTable) {
                const int     id  = min(max(c.ids[m], 0), c.table_rows - 1);
                const __bf16* row = (const __bf16*)c.table + (size_t)id * c.ld_table + c.table_col + n;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    r[e] = e < left ? act_apply(c.act, acc[e]) * (float)row[e] : 0.f;
                }
            }
            else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float z = epi == kDenseRelu2 ? fmaxf(acc[e], 0.f) : acc[e];
                    r[e]          = epi == kDenseRelu2 ? z * z : z;
                }
            }
            store_run<T, 4>((T*)a.y, i, r, vec, left);
            return;
        }
        float* y = (float*)a.y;
        if (epi == kDenseScaleF32 || epi == kDenseBiasF32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r[e] = epi == kDenseScaleF32 ? c.alpha * acc[e] : acc[e] + (e < left ? c.bias[n + e] : 0.f);
            }
            store_run<float, 4>(y, i, r, vec, left);
            return;
        }
        // the residual stream is read and written
        floatx4 old = {0.f, 0.f, 0.f, 0.f}, g = old;
        if (vec && left >= 4) {
            old = *(const floatx4*)(y + i);
        }
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                old[e] = e < left ? y[i + e] : 0.f;
            }
        }
        if (epi == kDenseResidAdd) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r[e] = old[e] + c.alpha * acc[e];
            }
            store_run<float, 4>(y, i, r, vec, left);
            if (c.y2) {
                store_run<T, 4>((T*)c.y2, (size_t)m * c.ldy2 + n, r, vec, left);
            }
            return;
        }
        // kDenseResidGate
        const float* gp = c.gate + (size_t)m * c.ldg + n;
        if (vec && left >= 4) {
            g = *(const floatx4*)gp;
        }
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g[e] = e < left ? gp[e] : 0.f;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float z = g[e] + (e < left ? c.gate_bias[n + e] : 0.f);
            r[e]          = old[e] + acc[e] / (1.f + expf(-z));
        }
        store_run<float, 4>(y, i, r, vec, left);
    }
};

// ---- weight images ----------------------------------------------------------------------------------------------------------------
// src: bf16 [rows][cols] (checkpoint bytes) -> dst at dense_frag_index of (row0 + r, col0 + c); half (1, 2): rows of a paired image, in the order of fp32 outputs or not
__global__ void dense_place_kernel(__bf16* __restrict__ dst, int steps, int row0, int col0, const __bf16* __restrict__ src, int rows, int cols,
                                   int transpose, int half, int f32)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (size_t)rows * cols) {
        const int r = (int)(i / cols), c = (int)(i % cols);
        int       n = row0 + (transpose ? c : r);  // transposed: the block's columns become output rows
        const int k = col0 + (transpose ? r : c);
        if (half) {
            n = dense_pair_row(n, half - 1, f32);
        }
        dst[dense_frag_index(n, k, steps)] = src[i];
    }
}

int dense_weight_alloc(DenseWeight& d, int K, int N, int dtype, hipStream_t st, int count)
{
    TM_REQUIRE(K >= 1 && N >= 1 && count >= 1 && (dtype == kDenseBf16 || dtype == kDenseF32), "dense weight: K, N, count >= 1, dtype bf16 | f32");
    d.K     = K;
    d.N     = N;
    d.Kp    = (K + 31) / 32 * 32;
    d.Np    = (N + 127) / 128 * 128;
    d.dtype = dtype;
    d.count = count;
    d.bytes = (size_t)d.Kp * d.Np * count * 2;
    TM_HIP_CHECK(hipMalloc(&d.w, d.bytes));
    TM_HIP_CHECK(hipMemsetAsync(d.w, 0, d.bytes, st));
    return 0;
}

int dense_weight_place(DenseWeight& d, int row0, int col0, const void* src_bf16, int rows, int cols, hipStream_t st, int item, bool transpose,
                       int half)
{
    TM_REQUIRE(d.w && row0 >= 0 && col0 >= 0 && item >= 0 && item < d.count && half >= 0 && half <= 2, "dense weight: part outside the image");
    TM_REQUIRE((half ? dense_pair_rows(row0 + (transpose ? cols : rows)) : row0 + (transpose ? cols : rows)) <= d.N
                   && col0 + (transpose ? rows : cols) <= d.K,
               "dense weight: part outside the image");
    const size_t n = (size_t)rows * cols, at = (size_t)item * d.Np * d.Kp;
    if (n == 0) {
        return 0;
    }
    dense_place_kernel<<<(n + 255) / 256, 256, 0, st>>>((__bf16*)d.w + at, d.Kp / 32, row0, col0, (const __bf16*)src_bf16, rows, cols, transpose, half, d.dtype == kDenseF32);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

void dense_weight_free(DenseWeight& d)
{
    if (d.w) {
        (void)hipFree(d.w);
    }
    d.w = nullptr;
}

// The lines between the kernels are a model of one CU's time in microseconds, fitted to measurements of this file's kernels (graph replays, weights from HBM).
//   tile kernels: (tiles of the fullest CU) x (steps x time of a step with the CU full + prologue and results), at least one tile alone.  16-bit, 8192
//     rows, (K, N) = (4096, 21504): 256 x 256 1155 us (1.25 PFLOP/s), 256 x 128 1281, 128 x 128 1520, 64 x 64 2714; (2048, 256) with 8000 rows: 46,
//     33, 23, 20 us; (2048, 2048) with 2600 rows: 50, 36, 35, 48 us; fp16 (5120, 5120) with 400 rows: -, 74, 44, 57, (4096, 4096) with 200: -, 69, 38, 20
//   few rows of one item (few_rows_cost): what the workgroups of the fullest CU stream, at 32 - 33 GB/s of weights a CU with a line of x (from L2) at a fraction
//     of the price of a line of weights; 6.1 TB/s for all of them; a workgroup's chain of steps; for slices the way through memory.  Of 184 sizes
//     (K 768 ... 25600, N 768 ... 32000, 1 ... 64 rows, 64 and 96 columns a workgroup, 1 ... 16 slices and the narrow kernel) what it takes is on
//     average 0.8 % and at most 10 % slower than the best.  us, bf16: (4096, 21504) 32 rows, 64 columns 38.9 (two workgroups on some CUs), 96 columns 30.1; (25600,
//     4096) 32 rows, one slice 95, four 36, eight 39; (4096, 6144) 32 rows, 96 columns four slices 14.8, 64 columns four 15.8, one 18.6; (2048, 2048) 8
//     rows, narrow 5.1, four slices 6.3, one 7.9; (14336, 4096) 16 rows, narrow 27.3, four slices 21.6; 128 columns where nearly every CU gets one workgroup of them, of 64 two, and
//     x is long: bf16 (4096, 27648) 32 rows 39.0 / 37.3, 64 rows 44.3 / 41.3, (4096, 32000) 64 rows 47.5 / 44.6; not (2048, 28160) 32 rows 22.0 / 22.4, (4096, 27648) 8 rows 36.7 / 36.6
//   items with rows of their own: blocks of as many rows as an item has at most (the tokens of a routed mixture, not its rows in total).  Febivik width 2048, whole
//     batches: 8 tokens 35.4 -> 35.0 ms, 16 tokens 32.5 -> 30.5 (48 rows, blocks of 64 before), 22 tokens 38.9 -> 37.5 (66 rows, tiles before), 32 the same
//   items, pairs: as many slices of k as give every CU a workgroup, none of fewer than 16 steps; nine items of (2048, 2816): one 21, three 31; pairs, four rows,
//     (2048, 11264): one 17, two 23
// us; cw: column tiles a workgroup (0: narrow kernel), ss: steps of one of sp slices
static double few_rows_cost(int steps, int cols, int rows, int cw, int sp, int ss)
{
    const int    mt = rows <= 16 ? 1 : rows <= 32 ? 2 : 4, wgs = cw ? (cols / 16 + cw - 1) / cw * sp : cols / 16;
    const double per_cu = wgs <= 1024 ? (wgs + 255) / 256 : wgs / 256.0;
    const double all    = cols * 64e-6 * steps / 6.1;
    if (cw == 0) {
        return 2.4 + std::max(all, per_cu * steps * 64 * (16 + 0.82 * rows) / 33e3);
    }
    return 2.6 + std::max({all, per_cu * ss * 64 * (cw * 16 + 0.26 * rows) / 32e3, ss * (0.018 + 0.037 * mt)}) + (sp > 1 ? 2.4 + 0.66 * sp * rows * cols * 4e-6 : 0.0);
}

// The same for fp32 rows, whose lines are twice as many: blocks of 64 rows side by side up to 256, and (cw < 0) 64 x 64 tiles.  Of 486 sizes (K 64 ... 14336, N 256 ... 32000, 1 ...
// 256 rows) what it took without the two terms at the line to tiles (stream_plan) was on average 1.6 % slower than the best, at most 45 % ((256, 24500) 129 rows).  us: (2048, 2048) 3 rows, narrow 5.3, four slices 7.0; (8448, 2048) 3
// rows, narrow 14.9, six slices 12.5; (2048, 8448) 32 rows, 96 columns two slices 16.1, 64 columns one 18.3, narrow 28.9; (2048, 1024) 90 rows, eight slices 15.9, tiles 17.2; (2048,
// 32000) 48 rows, slices 62, tiles 35 (up to 64 rows tiles are taken where the model sees 15 % in them)
static double few_rows_cost_f32(int steps, int cols, int rows, int cw, int sp, int ss)
{
    const int    mt = rows <= 16 ? 1 : rows <= 32 ? 2 : 4, rb = (rows + 63) / 64, wgs = (cw < 0 ? (cols + 63) / 64 : cw ? (cols / 16 + cw - 1) / cw * sp : cols / 16) * rb;
    const double per_cu = cw < 0 || wgs <= 1024 ? (wgs + 255) / 256 : wgs / 256.0, all = cols * 64e-6 * steps / 5.9, lines = per_cu * ss * 64e-3;
    if (cw < 0) {
        return std::max(per_cu * (0.143 * steps + 1.49), 0.168 * steps + 2.41);
    }
    if (cw == 0) {
        return 2.95 + 0.124 * ((steps + 31) / 32) * mt + std::max(all, lines * (16 + 1.36 * std::min(rows, 64)) / 31.1);
    }
    return 2.19 + 0.07 * mt + std::max({all, lines * (cw * 16 + 1.48 * std::min(rows, 64)) / 35.5, ss * 0.18}) + (sp > 1 ? 3.62 + 0.378 * sp * rows * cols * 4e-6 : 0.0);
}

StreamPlan stream_plan(int steps, int cols, int rows, int items, bool own_rows, int elem, bool pairs, size_t ws_bytes, int tickets, int border,
                       bool k_major, int item_rows, bool cut_ok, bool few_only)
{
    struct Tile {
        int    rows, cols;
        double full16, alone16, full32, alone32, fixed;
    };
    static const Tile kTiles[] = {{256, 256, 0.83, 0.83, 1e9, 1e9, 8.0}, {256, 128, 0.46, 0.55, 1e9, 1e9, 5.0}, {128, 128, 0.283, 0.30, 0.61, 0.73, 3.0},
                                  {64, 64, 0.125, 0.15, 0.20, 0.30, 1.0}};
    StreamPlan        best{};
    double            cost = 1e30;
    // row tiles: items with rows of their own fill half of their last one on average, and each that has rows needs one
    auto row_tiles = [&](int bm) -> int64_t {
        return own_rows ? std::max(rows / bm + (items + 1) / 2 + (bm == 256), std::min(rows, items)) : (int64_t)((rows + bm - 1) / bm) * items;
    };
    auto rounds = [&](int k, int n_cols) {  // of tiles of shape k over n_cols columns, 256 tiles a round
        const Tile& t = kTiles[k];
        return (row_tiles(t.rows) * ((n_cols + t.cols - 1) / t.cols) + 255) / 256;
    };
    auto tile_cost = [&](int k, int n_cols) {
        const Tile&  t     = kTiles[k];
        const double full  = elem == 4 ? t.full32 : t.full16, alone = elem == 4 ? t.alone32 : t.alone16;
        const double fixed = k == 0 && pairs ? 22.0 : t.fixed;  // (an activation per output, and no other workgroup on the CU meanwhile)
        return border % t.cols ? 1e30 : std::max(rounds(k, n_cols) * (full * steps + fixed), alone * steps + fixed);  // (a workgroup reads x at one place)
    };
    for (int k = 0; k < 4; ++k) {
        if (const double c = tile_cost(k, cols); c < cost) {
            cost = c, best.tile = k;
        }
    }
    // A last round that few tiles are left for: whole rounds of 256 x 256 tiles, and the columns behind them in smaller tiles of a launch of their own, if the
    // model above sees 1 % in it after 4 us for the launch.  us, one launch / two: fp16 (14336, 4096) 4100 rows 591 / 449, (2048, 8448) 2040 rows 96 / 75, 8010 rows 283 /
    // 262, (5120, 27648) gated 1030 rows 399 / 335, (4096, 6144) 5888 rows 303 / 262, least of 17 sizes (5120, 27648) 8010 rows 1873 / 1879; bf16 (4096, 27648) 8192
    // rows 1469 / 1458
    // Items with rows of their own, nine of (2048, 2816) and (2816, 2048), one launch / two: 23800 rows 314 / 302 and 344 / 306, 12400 rows the first 174 / 166, 16500 rows
    // the second 232 / 237 (the line is drawn wider for them: their last tiles are not known here)
    if (cut_ok && (items == 1 || own_rows) && elem == 2 && border % 256 == 0) {
        const int64_t rt = row_tiles(256);
        for (int64_t full = rounds(0, cols) - 1; full >= 1 && full >= rounds(0, cols) - 2; --full) {
            const int cut = (int)(full * 256 / rt) * 256;
            if (cut <= 0 || cut >= cols) {
                continue;
            }
            for (int k = 1; k < 4; ++k) {
                const double c = tile_cost(0, cut) + tile_cost(k, cols - cut) + 4.0;
                if (c < (own_rows ? 0.97 : 0.99) * cost) {
                    cost = c, best.tile = 0, best.cut = cut, best.tile2 = k;
                }
            }
        }
    }
    const int block = own_rows && item_rows > 0 ? std::min(rows, item_rows) : rows;  // rows that a workgroup may meet
    if (own_rows ? block > 64 : rows > 256 || (elem == 4 && rows > 64 && items > 1)) {  // (an item's rows are one block of the skinny kernel)
        return best;
    }
    const int mt = block <= 16 ? 1 : block <= 32 ? 2 : 4, rb = (block + 16 * mt - 1) / (16 * mt);
    best.mt = mt, best.row_blocks = rb, best.cw = pairs ? 8 : 4, best.splits = 1, best.split_steps = (steps + 7) / 8 * 8;
    if (items == 1 && !pairs && rows <= (elem == 4 && !own_rows ? 256 : 64)) {
        auto few = [&](int cw, int sp, int ss) { return elem == 4 ? few_rows_cost_f32(steps, cols, rows, cw, sp, ss) : few_rows_cost(steps, cols, rows, cw, sp, ss); };
        // (the waves of a narrow workgroup read pieces of 4 KB that lie far apart in a k-major image: fp16 (2048, 16384) 8 rows, narrow 14.6, 64 columns 11.9,
        // (2048, 4096) 48 rows 10.2 and 9.4)
        double least = k_major && cols > (rows > 32 ? 2048 : 8192) ? 1e30 : few(0, 1, steps);
        best.skinny = best.narrow = true;
        for (int cw : {4, 6, 8}) {
            const int groups = (cols / 16 + cw - 1) / cw;
            if (border % (16 * cw) || (cw == 8 && (elem == 4 || k_major || rows <= 16 || steps < 128 || groups < 192 || groups > 256))) {
                continue;
            }
            for (int sp = 1; sp <= 16 && (sp == 1 || steps / sp >= (elem == 4 ? 8 : 16)); ++sp) {
                const int ss = ((steps + sp - 1) / sp + 7) / 8 * 8;
                if ((steps + ss - 1) / ss != sp || (sp > 1 && ((size_t)sp * rows * cols * 4 > ws_bytes || groups * rb > tickets))) {
                    continue;
                }
                const double c = few(cw, sp, ss) * (cw == 8 ? 0.95 : 1.0);
                if (c < least) {
                    least = c, best.narrow = false, best.cw = cw, best.splits = sp, best.split_steps = ss;
                }
            }
        }
        if (elem == 4 && !few_only && border % 64 == 0) {
            // what a workgroup of the weight stream stages and splits of the rows are whole tiles of 16, and four of them take its stages twice as often, which weighs where the
            // model's other terms are short (1320 sizes without slices, both timed: this line is 0.9 % over the better one in the mean, 23 % at most; without these two terms
            // 2.5 % and 93 %.  us, stream / tile: (256, 32000) 256 rows 44 / 23, (1536, 8448) 33 rows 26 / 16, (256, 2048) 33 rows 7.6 / 5.8)
            const bool   one  = best.splits == 1;
            const double held = one && !best.narrow ? few_rows_cost_f32(steps, cols, rows <= 64 ? 16 * mt : rows, best.cw, 1, best.split_steps) + (mt < 4 ? 0.0 : rows <= 64 ? 0.7 : 2.5) : least;
            if (few(-1, 1, steps) < (rows <= 64 ? 0.85 : one ? 1.1 : 1.0) * held) {
                best.skinny = false, best.tile = 3;
            }
        }
        return best;
    }
    const int    wg_cols = pairs ? 128 : 64, groups = (cols + wg_cols - 1) / wg_cols * items * rb;
    const double step = 64.0 * (wg_cols + (elem == 4 ? 1.4 : 0.7) * std::min(block, 16 * mt)) / 25e3;
    int          sp   = groups >= (pairs ? 80 : 200) ? 1 : (256 + groups - 1) / groups;  // about one workgroup a CU
    sp          = std::max(1, std::min({sp, steps / 16, 16}));
    for (int more = sp; sp > 1 && more < 2 * sp && more <= 16; ++more) {  // slices of equal length
        if (steps % (8 * more) == 0) {
            sp = more;
            break;
        }
    }
    best.narrow = groups <= 64 && !pairs && rows <= 16 && steps <= 64;  // short sums: the way through memory costs more than it gives
    if (best.narrow) {
        sp = 1;
    }
    if (sp > 1 && ((size_t)items * sp * rows * cols * 4 > ws_bytes || groups > tickets)) {
        sp = 1, best.narrow = true;
    }
    // One slice: 96 columns a workgroup where the fullest CU then streams fewer, if of items with rows of their own nearly all have some (less than one is expected to have none,
    // rows dealt at random).  Where fewer have rows the CUs that get a second workgroup of 64 columns wait less for it than six waves of one CU for their loads.  us a routed layer in
    // a step, 64 | 96 columns: nine items, top 2, (4096, 2048) 8 rows 102.6 | 96.0, 16 rows 114.2 | 106.5; seventeen, top 2, (4096, 2048) 4 rows 123.6 | 129.2, (1408, 2048) 4 rows
    // 66.2 | 69.6; nine, (2048, 2816) 4 rows 73.3 | 75.6; seventeen, top 4, (2048, 1536) 6 rows 82.8 | 85.3, (2048, 1024) 12 rows 73.4 | 69.5
    const bool all = !own_rows || items * std::pow(1.0 - 1.0 / items, rows) < 0.85;
    const int  g64 = (cols + 63) / 64 * items * rb, g96 = (cols + 95) / 96 * items * rb;
    if (sp == 1 && items > 1 && elem == 2 && !pairs && !best.narrow && border % 96 == 0 && all && g64 <= 1024 && (g96 + 255) / 256 * 6 < (g64 + 255) / 256 * 4) {
        best.cw = 6;
    }
    const int    ss = ((steps + sp - 1) / sp + 7) / 8 * 8;
    const double c  = std::max(1.0, groups * sp / 256.0) * ss * step + 3.0;
    if (rows <= 64 || c < cost) {
        best.skinny = true, best.splits = (steps + ss - 1) / ss, best.split_steps = ss;
    }
    return best;
}

int launch_dense_linear(const DenseWeight& d, const void* x, int ldx, void* y, int ldy, int M, int epi, float alpha, hipStream_t st)
{
    DenseCall c;
    c.epi   = epi;
    c.alpha = alpha;
    return launch_dense_call(d, x, ldx, y, ldy, M, c, st);
}

// one instantiation per epilogue
#define TM_EPI_SWITCH(LAUNCH)                                \
    switch (epi) {                                           \
        case kDenseStore: LAUNCH(kDenseStore); break;        \
        case kDenseRelu2: LAUNCH(kDenseRelu2); break;        \
        case kDenseResidAdd: LAUNCH(kDenseResidAdd); break;  \
        case kDenseScaleF32: LAUNCH(kDenseScaleF32); break;  \
        case kDenseBiasF32: LAUNCH(kDenseBiasF32); break;    \
        case kDenseResidGate: LAUNCH(kDenseResidGate); break; \
        case kDenseGatedAct: LAUNCH(kDenseGatedAct); break;  \
        case kDenseXielu: LAUNCH(kDenseXielu); break;        \
        case kDenseActTable: LAUNCH(kDenseActTable); break;  \
        case kDenseStoreRelu2: LAUNCH(kDenseStoreRelu2); break; \
    }

template<class T, int MT, int NT, int CW, int KP>
static int launch_dense_skinny(const StreamArgs& a, const DenseCall& call, int vec, dim3 grid, hipStream_t st)
{
    stream_skinny_kernel<T, DenseEpi<T, -1>, MT, NT, CW, KP><<<grid, CW * KP * 64, 0, st>>>(a, DenseEpi<T, -1>{call, vec});
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class T, int MT, int NT>
static int launch_dense_narrow(const StreamArgs& a, const DenseCall& call, int vec, int items, hipStream_t st)
{
    const dim3 grid((a.tiles + NT - 1) / NT, items * a.row_blocks);
    if (MT * NT <= 2 && stream_narrow_waves(a) == 16) {
        stream_narrow_kernel<T, DenseEpi<T, -1>, MT, NT, MT * NT <= 2 ? 16 : 8><<<grid, 1024, 0, st>>>(a, DenseEpi<T, -1>{call, vec});
    }
    else {
        stream_narrow_kernel<T, DenseEpi<T, -1>, MT, NT, 8><<<grid, 512, 0, st>>>(a, DenseEpi<T, -1>{call, vec});
    }
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

static dim3 stream_tile_grid(const StreamArgs& a, int bm, int bn, const DenseCall& call)
{
    const unsigned tns = ((a.col1 ? a.col1 : a.tiles * 16) - a.col0 + bn - 1) / bn;
    return call.row_offsets ? dim3((a.M / bm + call.count) * tns) : dim3((a.M + bm - 1) / bm * tns, call.count);
}

template<class T, int EPI, int BM, int BN, int WM, int WN>
static int launch_dense_tile(const StreamArgs& a, const DenseCall& call, int vec, hipStream_t st)
{
    constexpr int lds = stream_tile_bufs(BM, BN) * (BM + BN) * 64;
    const auto    k   = stream_tile_kernel<T, DenseEpi<T, EPI>, BM, BN, WM, WN>;
    if (const int rc = ensure_dynamic_lds((const void*)k, lds)) {
        return rc;
    }
    k<<<stream_tile_grid(a, BM, BN, call), 256, lds, st>>>(a, DenseEpi<T, EPI>{call, vec});
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<int EPI, int BM, int BN, int KP>
static int launch_dense_tile_split(const StreamArgs& a, const DenseCall& call, int vec, hipStream_t st)
{
    constexpr int lds = KP * stream_split_bufs(BM, KP) * (BM * 2 + BN) * 64;
    const auto    k   = stream_tile_split_kernel<DenseEpi<float, EPI>, BM, BN, KP>;
    if (const int rc = ensure_dynamic_lds((const void*)k, lds)) {
        return rc;
    }
    k<<<stream_tile_grid(a, BM, BN, call), 256 * KP, lds, st>>>(a, DenseEpi<float, EPI>{call, vec});
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class T, int EPI>
static int launch_dense_tile256(const StreamArgs& a, const DenseCall& call, int vec, hipStream_t st)
{
    constexpr int lds = stream_tile_bufs(256, 256) * 512 * 64;
    const auto    k   = stream_tile256_kernel<T, DenseEpi<T, EPI>>;
    if (const int rc = ensure_dynamic_lds((const void*)k, lds)) {
        return rc;
    }
    k<<<stream_tile_grid(a, 256, 256, call), 256, lds, st>>>(a, DenseEpi<T, EPI>{call, vec});
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

template<class T>
static int launch_dense_tiles(const StreamArgs& a, const DenseCall& call, int tile, int vec, hipStream_t st)
{
    const int  epi   = call.epi;
    const dim3 grid  = stream_tile_grid(a, 64, 64, call);
    const bool alone = a.steps >= 32 && grid.x * grid.y <= 256;  // (fp32: four groups of waves a tile, see stream_tile_split_kernel; at 24 steps it is a tie)
#define TM_TILE(EPI_)                                                                        \
    if constexpr (sizeof(T) == 4) {                                                          \
        return tile == 2 ? launch_dense_tile_split<EPI_, 128, 128, 1>(a, call, vec, st) :    \
               alone     ? launch_dense_tile_split<EPI_, 64, 64, 4>(a, call, vec, st) :      \
                           launch_dense_tile_split<EPI_, 64, 64, 1>(a, call, vec, st);       \
    }                                                                                        \
    else {                                                                                   \
        if constexpr (EPI_ != kDenseActTable) {                                              \
            if (tile == 0) {                                                                 \
                return launch_dense_tile256<T, EPI_>(a, call, vec, st);                      \
            }                                                                                \
        }                                                                                    \
        return tile <= 1 ? launch_dense_tile<T, EPI_, 256, 128, 2, 2>(a, call, vec, st) :    \
               tile == 2 ? launch_dense_tile<T, EPI_, 128, 128, 2, 2>(a, call, vec, st) :    \
                           launch_dense_tile<T, EPI_, 64, 64, 2, 2>(a, call, vec, st);       \
    }
    TM_EPI_SWITCH(TM_TILE)
#undef TM_TILE
    return 0;
}

template<class T>
static int launch_dense_typed(const DenseWeight& d, const void* x, int ldx, void* y, int ldy, int M, const DenseCall& call, hipStream_t st)
{
    const int  epi = call.epi, G = call.count;
    StreamArgs a{};
    a.x = (const char*)x, a.ldx = (int64_t)ldx * sizeof(T);
    a.w = (const char*)d.w, a.steps = d.Kp / 32, a.tiles = d.Np / 16;
    a.w_tile = (int64_t)a.steps * 1024, a.w_quad = 4096;
    a.y = y, a.ldy = ldy, a.M = M, a.N = d.N;
    const bool f32_out = epi == kDenseResidAdd || epi == kDenseScaleF32 || epi == kDenseBiasF32 || epi == kDenseResidGate;
    const int  align   = f32_out || sizeof(T) == 4 ? 4 : 8;  // elements of 16 bytes
    const int  vec     = ldy % align == 0 && (uintptr_t)y % 16 == 0 && call.y_col_stride % align == 0
                    && (!call.y2 || (call.ldy2 % 8 == 0 && (uintptr_t)call.y2 % 16 == 0))
                    && (epi != kDenseResidGate || (call.ldg % 4 == 0 && (uintptr_t)call.gate % 16 == 0));
    int border = 0;  // the segments begin at multiples of this many columns
    for (int s = 1; s < call.n_seg; ++s) {
        border = std::gcd(border, call.seg_n0[s]);
    }
    const StreamPlan p = stream_plan(a.steps, d.Np, M, G, call.row_offsets != nullptr, sizeof(T), epi == kDenseGatedAct && sizeof(T) == 2,
                                     d.scratch ? d.scratch->bytes : 0, d.scratch ? d.scratch->count : 0, border, false, call.item_rows, true, call.kv.block_ptrs != nullptr);
    TM_REQUIRE(p.skinny || !call.kv.block_ptrs, "dense linear: cache columns belong to products of few rows");
    if (p.skinny) {
        a.split_steps = p.split_steps;
        a.row_blocks  = p.row_blocks;
        a.slabs       = p.splits > 1 ? d.scratch->slabs : nullptr;
        a.tickets     = p.splits > 1 ? d.scratch->tickets : nullptr;
        const dim3 grid((unsigned)((a.tiles + p.cw - 1) / p.cw), G * p.row_blocks, p.splits);
        const bool pairs = epi == kDenseGatedAct && sizeof(T) == 2;
#define TM_SKINNY(MT_, NT_, CW_, KP_)                                                    \
    if (p.mt == MT_ && p.cw == CW_ * NT_ && pairs == (NT_ == 2)) {                       \
        if (p.narrow) {                                                                  \
            return launch_dense_narrow<T, MT_, NT_>(a, call, vec, G, st);                \
        }                                                                                \
        return launch_dense_skinny<T, MT_, NT_, CW_, KP_>(a, call, vec, grid, st);       \
    }
        TM_STREAM_SHAPES(TM_SKINNY)
        if constexpr (sizeof(T) == 2) {
            TM_STREAM_SHAPES_WIDE(TM_SKINNY) TM_STREAM_SHAPES_PAIRS(TM_SKINNY)
        }
#undef TM_SKINNY
    }
    if (p.cut > 0) {
        StreamArgs rest = a;
        rest.col0       = p.cut;
        a.col1          = p.cut;
        if (const int rc = launch_dense_tiles<T>(a, call, p.tile, vec, st)) {
            return rc;
        }
        return launch_dense_tiles<T>(rest, call, p.tile2, vec, st);
    }
    return launch_dense_tiles<T>(a, call, p.tile, vec, st);
}

int launch_dense_call(const DenseWeight& d, const void* x, int ldx, void* y, int ldy, int M, DenseCall call, hipStream_t st)
{
    const int epi = call.epi;
    TM_REQUIRE(d.w && x && y && M >= 0 && call.count >= 1 && call.count <= d.count, "dense linear: operands");
    const int n_y = epi == kDenseGatedAct ? call.n_out : epi == kDenseStoreRelu2 ? call.first_n : d.N;
    TM_REQUIRE(ldx >= d.Kp + (call.count - 1) * call.x_col_stride && ldy >= n_y + (call.count - 1) * call.y_col_stride, "dense linear: row lengths");
    TM_REQUIRE(epi >= kDenseStore && epi <= kDenseStoreRelu2 && (epi != kDenseXielu || call.act_par), "dense linear: epilogue");
    TM_REQUIRE(epi != kDenseGatedAct || (call.n_out >= 1 && dense_pair_rows(call.n_out) <= d.N), "dense linear: paired image");
    TM_REQUIRE(epi != kDenseBiasF32 || call.bias, "dense linear: bias");
    TM_REQUIRE(!call.y2 || epi == kDenseStoreRelu2 || (epi == kDenseResidAdd && call.ldy2 >= d.N && call.count == 1), "dense linear: second output");
    TM_REQUIRE(epi != kDenseStoreRelu2 || (call.y2 && call.count == 1 && call.first_n >= 1 && call.first_n <= call.split_n && call.split_n % 4 == 0 && call.split_n < d.N
                                           && call.ldy2 >= d.N - call.split_n),
               "dense linear: two outputs");
    TM_REQUIRE(!call.kv.block_ptrs || (epi == kDenseStoreRelu2 && M <= kDenseSinkRows && call.kv.row_seq && call.kv.row_pos && call.kv.dim >= 1 && call.kv.vdim >= 1
                                       && call.kv.block_stride >= 1 && call.kv.k_col <= call.kv.v_col && call.kv.v_col <= call.first_n),
               "dense linear: cache columns");
    TM_REQUIRE(epi != kDenseActTable || (call.table && call.ids && call.count == 1 && call.table_rows >= 1 && call.table_col >= 0
                                         && call.table_col + d.N <= call.ld_table),
               "dense linear: table");
    TM_REQUIRE(epi != kDenseResidGate || (call.gate && call.gate_bias && call.ldg >= d.N), "dense linear: gate");
    TM_REQUIRE(call.n_seg >= 0 && call.n_seg <= kDenseMaxSeg && (call.n_seg == 0 || (call.count == 1 && call.seg_n0[0] == 0 && ldx >= d.Kp + (call.n_seg - 1) * call.x_col_stride)),
               "dense linear: segments");
    for (int s = 1; s < call.n_seg; ++s) {
        TM_REQUIRE(call.seg_n0[s] % 128 == 0 && call.seg_n0[s] > call.seg_n0[s - 1] && call.seg_n0[s] < d.N, "dense linear: segment borders");
    }
    TM_REQUIRE(call.act != kActClamped || epi == kDenseGatedAct, "dense linear: the clamped activation takes a gate / up pair");
    if (M == 0) {
        return 0;
    }
    call.w_stride = (size_t)d.Np * d.Kp;
    call.ldx      = ldx;
    if (d.dtype == kDenseF32) {
        TM_REQUIRE(ldx % 4 == 0, "dense linear (fp32): rows must be 16-byte aligned");
        TM_REQUIRE(call.x_col_stride % 4 == 0, "dense linear (fp32): items must be 16-byte aligned");
        return launch_dense_typed<float>(d, x, ldx, y, ldy, M, call, st);
    }
    TM_REQUIRE(ldx % 8 == 0 && call.x_col_stride % 8 == 0, "dense linear (bf16): rows and items must be 16-byte aligned");
    return launch_dense_typed<__bf16>(d, x, ldx, y, ldy, M, call, st);
}

}  // namespace tmk
