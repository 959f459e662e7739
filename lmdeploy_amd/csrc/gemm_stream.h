// Building blocks of the unquantised products y = x . W^T (gemm_dense.hip: bf16 and fp32 checkpoint weights; gemm_f16.hip: the fp16
// linears of the Llama family), one set for the three number formats.
//
// Weight image: 16 output columns x 32 k of a 16-bit format are one contiguous KB in MFMA fragment order, lane l holds column l % 16 and its eight k at
// (l / 16) * 8 (v_mfma_f32_16x16x32).  A "step" below is such a range of 32 k: 64 bytes of a weight column, and 64 of a row of x in 16 bits, 128 in fp32.
// fp32 products have bf16 weights (as every checkpoint of these models) and fp32 rows: a row's number is the sum of three bf16 numbers, exactly (StreamOp).
//
// The weight is the MFMA's A operand: a lane's four results are four CONSECUTIVE output columns of one row of x, so results leave in
// 8- or 16-byte stores, and a gate / up pair of a feed-forward is in one lane.
#pragma once
#include "tm_common.h"
#include <type_traits>

namespace tmk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template<class T>
struct StreamOp;
template<>
struct StreamOp<__bf16> {
    static __device__ __forceinline__ floatx4 mma(u32x4 a, u32x4 b, floatx4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bit_cast<bf16x8>(a), bit_cast<bf16x8>(b), c, 0, 0, 0);
    }
};
template<>
struct StreamOp<half_t> {
    static __device__ __forceinline__ floatx4 mma(u32x4 a, u32x4 b, floatx4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(bit_cast<half8_t>(a), bit_cast<half8_t>(b), c, 0, 0, 0);
    }
};
// fp32 rows: 24 bits of significand are three times the eight of bf16, so x = high + middle + low exactly (each part the rest's leading bits, cut off; a part that
// underflows is below 2^-126), and a product of two bf16 numbers is exact in fp32: three bf16 matrix instructions multiply as exactly as fp32 ones do, in 48
// cycles instead of 256.  They cut the sum off where v_mfma_f32_16x16x4 rounds it, so sums of one sign would drift: every kSplitSteps steps begin at zero and are
// added to the others in fp32, and few rows sum the low and middle parts apart from the high ones.  What remains of an infinity after its leading part is what remains of the
// largest number, and a NaN whose leading half is that of an infinity (its payload in the lower one) is a NaN in the middle part: the median of three numbers is the least of
// them where one is a NaN, and a signalling NaN where that comes last.
struct SplitRow {
    u32x4 part[3];  // low, middle, high
};
__device__ __forceinline__ float stream_most()
{
    float most = 3.402823466e38f;
    asm("" : "+s"(most));  // (the compiler may not know the value: it puts constants last.  Once a kernel: once a split, it moved the splits of the 128 x 128 tile behind their barrier, 7 %)
    return most;
}
__device__ __forceinline__ SplitRow stream_split(u32x4 a, u32x4 b, float most)
{
    SplitRow o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float r[2] = {bit_cast<float>(i < 2 ? a[2 * i] : b[2 * i - 4]), bit_cast<float>(i < 2 ? a[2 * i + 1] : b[2 * i - 3])};
#pragma unroll
        for (int p = 2; p >= 0; --p) {
            o.part[p][i] = __builtin_amdgcn_perm(bit_cast<uint32_t>(r[1]), bit_cast<uint32_t>(r[0]), 0x07060302);  // both leading halves
#pragma unroll
            for (int e = 0; p > 0 && e < 2; ++e) {
                if (p == 2) {
                    r[e] = __builtin_amdgcn_fmed3f(most, -most, r[e]);
                }
                r[e] -= bit_cast<float>(bit_cast<uint32_t>(r[e]) & 0xffff0000u);
            }
        }
    }
    return o;
}
template<>
struct StreamOp<float> {
    static __device__ __forceinline__ floatx4 mma(u32x4 a, u32x4 b, floatx4 c)
    {
        return StreamOp<__bf16>::mma(a, b, c);
    }
};
template<class T>
constexpr int kStreamParts = sizeof(T) == 4 ? 3 : 1;  // matrix instructions a fragment of x takes
template<class T>
constexpr int kStreamXStep = 32 * sizeof(T);          // bytes of a row of x in a step
constexpr int kSplitSteps = 8;                        // most steps of fp32 rows that the matrix cores add up by themselves

struct StreamArgs {
    const char* x;       // rows of ldx bytes, 16-byte aligned
    int64_t     ldx;
    const char* w;       // image of the first item
    int64_t     w_tile;  // bytes from one 16-column tile to the next ...
    int64_t     w_quad;  // ... and from four steps to the next four (the four are contiguous)
    int         tiles;   // 16-column tiles the image holds
    int         steps;   // steps of k
    int         split_steps;  // skinny kernel: steps of one slice of k (grid z), a multiple of 8
    int         col0, col1;   // tile kernels: the columns of the launch, multiples of its tile (col1 0: to the image's end)
    int         row_blocks;   // skinny kernel: blocks of 16 MT rows (grid y = item * row_blocks + block)
    void*       y;
    int         ldy, M, N;
    float*      slabs;        // skinny kernel, several slices: their partial sums, [item][slice][M][16 tiles]
    unsigned*   tickets;      // ... and an arrival counter per (column group, row block, item), zero between launches (nullptr: the slabs are the result)
};
// The step that stands first in a tile of an image whose tiles are one behind the other (Epi::kTileRuns).  A launch reads a thousand tiles at about the same step.
// Where tiles are a multiple of 64 KB long those places fall on a part of the memory channels, so tiles of 128 KB and more are turned: they begin with another step,
// 4 KB further in some order for every 16 tiles, and end with the steps ahead of it.  bf16, weights from HBM, plain / turned / tiles 4 KB apart (which reach over one
// page more): (4096, 27648) 8 rows 41.1 / 38.1 / 37.0 us, 32 rows 44.6 / 41.3 / 41.5, 200 rows 78 / 80 / 81; (4096, 4096) 32 rows 14.7 / 14.1 / 13.8, 640 rows 43.9 / 43.5
// / 45.9; (8192, 2048) 32 rows 23.1 / 21.7 / 21.9, 4096 rows 135 / 132 / 144.  Tiles of 64 KB gain nothing: (2048, 12288) 8 rows 11.5 / 12.7 / 11.6, 65 rows 17.9 /
// 18.1 / 20.8; (2048, 8448) 65 rows 16.1 / 17.7 / 17.9 (and with the number of the sixteen alone, or three, five or seven times it, (2048, 32000) 32 rows 25 / 28).
__host__ __device__ inline int stream_turn(int tile, int steps)
{
    return steps % 64 == 0 && steps >= 128 ? (((tile >> 4) ^ (tile >> 8)) * 11 & 15) * 4 : 0;
}
// where step s is in a tile (turn: the step that stands first)
template<class Epi>
__device__ __forceinline__ int64_t stream_step_at(const StreamArgs& a, int s, int turn)
{
    if constexpr (Epi::kTileRuns) {
        const int at = s + turn;
        return (at < a.steps ? at : at - a.steps) * 1024;
    }
    return (s >> 2) * a.w_quad + (s & 3) * 1024;
}
// from the first block of a column tile to the end of the image's last block
__device__ __forceinline__ int64_t stream_weight_bytes(const StreamArgs& a, int tile)
{
    return (int64_t)(a.tiles - 1 - tile) * a.w_tile + (int64_t)((a.steps - 1) >> 2) * a.w_quad + ((a.steps - 1) & 3) * 1024 + 1024;
}

// ---- few rows: the weight stream ---------------------------------------------------------------------------------------------------
// What bounds it: a CU keeps about 440 cache lines in flight whatever their source, so a line of x that comes from L2 costs nearly what a
// line of weights costs.  One workgroup therefore covers CW x NT column tiles with ONE copy of its rows of x in LDS (double buffered, eight
// steps at a time), and few columns are spread over the CUs by cutting k instead of the column group: KP waves share a column
// tile inside the workgroup and meet in LDS, grid z slices of k meet in the last workgroup of a column group to arrive, which adds the
// slices in slice order (the sum never depends on the order of arrival; no workgroup waits for another).
// Weights run one chunk of eight steps ahead of the MFMAs in a second register buffer; all loads of a stage are unconditional (clamped).  Loads return in
// order, so a stage's x is asked for ahead of its weights: the wait for x then leaves the weights in flight (the other way round every stage drained the
// queue: 8 rows fp16 of (2048, 16384) 14.6 us, now 11.9 = 5.6 TB/s; bf16 of (2048, 8448) 12.0, 9.9).
// 32 rows bf16, weights from HBM: (K, N) = (25600, 4096) 38 us = 5.5 TB/s, (4096, 21504) 30 us = 5.9 TB/s with 96 columns a workgroup, one for nearly every CU
// (39 us with 64, of which some CUs get two; with every wave reading x for itself, no slices: 76 and 50).  The loop fetches without a branch: with one around the
// loads, and 64 columns, the two took 52 and 42.  Its last two stages stand behind it and fetch nothing beyond the slice: 8 rows bf16 of (8448, 2048) then took
// 15.1 -> 11.8.
template<class T, class Epi, int MT, int NT, int CW, int KP>
__global__ __launch_bounds__(CW* KP * 64) void stream_skinny_kernel(StreamArgs a, Epi epi)
{
    constexpr int kParts = kStreamParts<T>, kXS = kStreamXStep<T>;
    constexpr int kThreads = CW * KP * 64, kChunk = kParts > 1 && MT == 4 ? 4 : 8;
    constexpr int kXVecs  = KP * MT * kChunk * 64;                          // fragments' pieces of eight k of one x stage
    constexpr int kXPer   = (kXVecs + kThreads - 1) / kThreads;             // ... per thread (kXVecs is a multiple of kThreads or of 64)
    constexpr int kRaw    = kXS / 64;                                       // 16-byte loads of a piece
    constexpr int kRed    = KP > 1 ? (KP - 1) * CW * MT * NT * 64 * 16 : 0;  // the other k-phases' sums
    constexpr int kStage  = kParts * kXVecs * 16, kXBytes = 2 * kStage;
    __shared__ __attribute__((aligned(16))) char smem[kXBytes > kRed ? kXBytes : kRed];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wave % CW, ph = wave / CW;
    const int tile0 = (blockIdx.x * CW + cw) * NT;
    const int  mb   = blockIdx.y % a.row_blocks * (MT * 16);
    const auto item = epi.item(blockIdx.y / a.row_blocks, a.M, blockIdx.x * CW * NT * 16);
    const int  M    = min(item.M - mb, MT * 16);
    if (M <= 0) {
        return;
    }
    const char* x = a.x + item.x_off + mb * a.ldx;
    const char* w = a.w + item.w_off + lane * 16;
    const int   s0 = blockIdx.z * a.split_steps, s1 = min(a.steps, s0 + a.split_steps);
    const char* wp[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        wp[j] = w + (int64_t)min(tile0 + j, a.tiles - 1) * a.w_tile;
    }
    const float most = stream_most();
    const int turn = stream_turn(tile0, a.steps);
    u32x4     wa[kChunk][NT], wb[kChunk][NT], xr[kXPer][kRaw];
    auto  fetch = [&](u32x4(&buf)[kChunk][NT], int base) {
#pragma unroll
        for (int kk = 0; kk < kChunk; ++kk) {
            const int s = min(base + kk, a.steps - 1);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                buf[kk][j] = __builtin_nontemporal_load((const u32x4*)(wp[j] + stream_step_at<Epi>(a, s, turn)));
            }
        }
    };
    // x stage: [phase][row tile][pair of steps] blocks of 16 rows x 128 bytes, 16-byte piece c of row r at r * 128 + ((c ^ (r & 7)) * 16): a
    // fragment read meets every bank once, a row's 128 bytes (256 in fp32) are whole lines of memory.  fp32 rows are split once, by who stores them: a stage for each part
    auto fetch_x = [&](int base) {
#pragma unroll
        for (int i = 0; i < kXPer; ++i) {
            const int v = tid + i * kThreads;
            const int c = v & 7, r = (v >> 3) & 15, blk = v >> 7;
            const int pair = blk % (kChunk / 2), rt = blk / (kChunk / 2) % MT, p = blk / (kChunk / 2) / MT;
            const int row = min(rt * 16 + r, M - 1);
            const int64_t col = min((int64_t)(base + p * kChunk + pair * 2) * kXS + c * 16 * kRaw, (int64_t)a.steps * kXS - 16 * kRaw);
#pragma unroll
            for (int h = 0; h < kRaw; ++h) {
                xr[i][h] = *(const u32x4*)(x + row * a.ldx + col + 16 * h);
            }
        }
    };
    auto stash_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kXPer; ++i) {
            const int v = tid + i * kThreads;
            if (kXVecs % kThreads == 0 || v < kXVecs) {
                const int   c = v & 7, r = (v >> 3) & 15, blk = v >> 7;
                char* const at = smem + buf * kStage + blk * 2048 + r * 128 + ((c ^ (r & 7)) << 4);
                if constexpr (kParts > 1) {
                    const SplitRow f = stream_split(xr[i][0], xr[i][1], most);
#pragma unroll
                    for (int p = 0; p < kParts; ++p) {
                        *(u32x4*)(at + p * kXVecs * 16) = f.part[p];
                    }
                }
                else {
                    *(u32x4*)at = xr[i][0];
                }
            }
        }
    };
    floatx4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            acc[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const int   fr = lane & 15, fc = lane >> 4;
    const char* xf = smem + ph * (MT * (kChunk / 2) * 2048) + fr * 128;
    floatx4     sum[2][MT][NT];  // (fp32: of the chunk, the low and middle parts' and the high parts')
    auto        one = [&](const u32x4(&buf)[kChunk][NT], int xbuf, int kk) {
#pragma unroll
        for (int p = 0; p < kParts; ++p) {
            floatx4(&to)[MT][NT] = kParts > 1 ? sum[p / 2] : acc;
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const u32x4 b = *(const u32x4*)(xf + xbuf * kStage + p * kXVecs * 16 + (t * (kChunk / 2) + (kk >> 1)) * 2048 + ((((kk & 1) * 4 + fc) ^ (fr & 7)) << 4));
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    to[t][j] = StreamOp<T>::mma(buf[kk][j], b, to[t][j]);
                }
            }
        }
    };
    auto compute = [&](const u32x4(&buf)[kChunk][NT], int xbuf, int base) {
        static_assert(kParts == 1 || kChunk <= kSplitSteps, "sums of fp32 rows");
        if constexpr (kParts > 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    sum[0][t][j] = sum[1][t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
        if (base + kChunk <= s1) {
#pragma unroll
            for (int kk = 0; kk < kChunk; ++kk) {
                one(buf, xbuf, kk);
            }
        }
        else {
#pragma unroll
            for (int kk = 0; kk < kChunk; ++kk) {
                if (base + kk < s1) {
                    one(buf, xbuf, kk);
                }
            }
        }
        if constexpr (kParts > 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    acc[t][j] += sum[0][t][j] + sum[1][t][j];
                }
            }
        }
    };
    constexpr int kStride = KP * kChunk;
    const int     first   = ph * kChunk;  // of this k-phase in a stage
    auto load = [&](u32x4(&buf)[kChunk][NT], int at) {
        fetch_x(at);
        asm volatile("" ::: "memory");
        fetch(buf, at + first);
        asm volatile("" ::: "memory");
    };
    load(wa, s0);
    stash_x(0);
    __syncthreads();
    int base = s0;
    for (; base + 2 * kStride < s1; base += 2 * kStride) {  // three stages lie ahead
        load(wb, base + kStride);
        compute(wa, 0, base + first);
        stash_x(1);  // its readers finished before the last barrier
        __syncthreads();
        load(wa, base + 2 * kStride);
        compute(wb, 1, base + kStride + first);
        stash_x(0);
        __syncthreads();
    }
    if (base + kStride < s1) {  // the last two stages, or the last: nothing is fetched that is not used
        load(wb, base + kStride);
        compute(wa, 0, base + first);
        stash_x(1);
        __syncthreads();
        compute(wb, 1, base + kStride + first);
    }
    else {
        compute(wa, 0, base + first);
    }
    __syncthreads();
    if constexpr (KP > 1) {  // (the last barrier freed the x buffers)
        floatx4* red = (floatx4*)smem;
        if (ph > 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    red[(((ph - 1) * CW + cw) * MT * NT + t * NT + j) * 64 + lane] = acc[t][j];
                }
            }
        }
        __syncthreads();
        if (ph == 0) {
#pragma unroll
            for (int p = 1; p < KP; ++p) {  // fixed order
#pragma unroll
                for (int t = 0; t < MT; ++t) {
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        acc[t][j] += red[(((p - 1) * CW + cw) * MT * NT + t * NT + j) * 64 + lane];
                    }
                }
            }
        }
    }
    if (gridDim.z > 1) {
        // slabs [item][slice][row][column] of all the columns the image holds.  Without counters they are the result; else they are written through to
        // memory (sc1) and drained before the counter moves, and the last workgroup reads them past its L1 (sc1)
        const int     ld   = a.tiles * 16, n = tile0 * 16 + fc * 4;
        const int64_t rows = (int64_t)a.M * ld * 4;  // bytes of one slice
        const auto    rs   = __builtin_amdgcn_make_buffer_rsrc((void*)((char*)a.slabs + blockIdx.y / a.row_blocks * gridDim.z * rows), 0, (int)(gridDim.z * rows), 0x00020000);
        if (ph == 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if (t * 16 + fr < M) {
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        const int at = ((mb + t * 16 + fr) * ld + n + 16 * j) * 4;
                        if (n + 16 * j < ld) {
                            __builtin_amdgcn_raw_buffer_store_b128(bit_cast<u32x4>(acc[t][j]), rs, at, (int)(blockIdx.z * rows), /*sc1*/ 16);
                        }
                    }
                }
            }
        }
        if (!a.tickets) {
            return;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned* last = (unsigned*)smem;  // (every reader of the x buffers and of `red` has passed a barrier)
        unsigned* mine = a.tickets + blockIdx.y * gridDim.x + blockIdx.x;
        if (tid == 0) {
            *last = __hip_atomic_fetch_add(mine, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (*last != gridDim.z - 1) {
            return;
        }
        if (tid == 0) {
            __hip_atomic_store(mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (ph > 0) {
            return;
        }
        // in the order of the slices, several of them and what the outputs are added to asked for at once: the seven slices of (8192, 2048) were four trips to memory in a
        // row, and the outputs a fifth (fp16, 8 rows 10.3 -> 9.8 us in a model)
        constexpr int kZ = MT * NT >= 4 ? 2 : 8 / (MT * NT);
        unsigned      warm[MT][NT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                acc[t][j]  = floatx4{0.f, 0.f, 0.f, 0.f};
                warm[t][j] = epi.touch(a, item, mb + min(t * 16 + fr, M - 1), min(n + 16 * j, a.N - 1));
            }
        }
        for (int z0 = 0; z0 < (int)gridDim.z; z0 += kZ) {
            u32x4 part[MT][NT][kZ];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int at = ((mb + min(t * 16 + fr, M - 1)) * ld + min(n + 16 * j, ld - 4)) * 4;
#pragma unroll
                    for (int z = 0; z < kZ; ++z) {
                        part[t][j][z] = __builtin_amdgcn_raw_buffer_load_b128(rs, at, (int)(min(z0 + z, (int)gridDim.z - 1) * rows), /*sc1*/ 16);
                    }
                }
            }
#pragma unroll
            for (int z = 0; z < kZ; ++z) {
                if (z0 + z < (int)gridDim.z) {
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
#pragma unroll
                        for (int j = 0; j < NT; ++j) {
                            acc[t][j] += bit_cast<floatx4>(part[t][j][z]);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                asm volatile("" ::"v"(warm[t][j]));
            }
        }
    }
    if (KP > 1 && ph > 0) {
        return;
    }
    // results: row m = t * 16 + lane % 16, columns tile * 16 + (lane / 16) * 4 + 0 .. 3
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + fr;
        if (m < M) {
            epi.template rows<NT>(a, item, mb + m, tile0 * 16 + fc * 4, acc[t]);
        }
    }
}

// The same without slices across workgroups, for callers that bring no scratch and where slices cost more than they give (stream_plan): a workgroup owns NT
// column tiles, its W waves take chunks of steps in turn, each reading its own rows of x, and meet in LDS in wave order.
template<class T, class Epi, int MT, int NT, int W>
__global__ __launch_bounds__(W * 64) void stream_narrow_kernel(StreamArgs a, Epi epi)
{
    constexpr int  kParts = kStreamParts<T>, kXS = kStreamXStep<T>, kRaw = kXS / 64;
    constexpr bool kAhead = MT == 1 || (MT == 2 && kParts == 1);
    constexpr int  kChunk = (MT * NT > 1 || kParts > 1) && kAhead ? 4 : 8 / NT;
    __shared__ __attribute__((aligned(16))) floatx4 red[W][MT * NT][64];
    const int  lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int  mb   = blockIdx.y % a.row_blocks * (MT * 16), tile0 = blockIdx.x * NT;
    const auto item = epi.item(blockIdx.y / a.row_blocks, a.M, tile0 * 16);
    const int  M    = min(item.M - mb, MT * 16);
    if (M <= 0) {
        return;
    }
    const int   fr = lane & 15, fc = lane >> 4;
    const char* xp[MT];
    const char* wp[NT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        xp[t] = a.x + item.x_off + (int64_t)(mb + min(t * 16 + fr, M - 1)) * a.ldx + fc * 16 * kRaw;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        wp[j] = a.w + item.w_off + (int64_t)min(tile0 + j, a.tiles - 1) * a.w_tile + lane * 16;
    }
    floatx4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            acc[t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // Up to 16 rows, and up to 32 of a 16-bit format, x of a chunk leaves with its weights, ahead of them: loads return in order, and a load of x where it is used would
    // wait for the next chunk's weights (fp16, 8 rows: (2048, 4096) 5.9 -> 5.4 us, (2048, 2048) 5.1 -> 4.8; bf16, 17
    // rows, (4096, 4096) 11.9 -> 10.8).  More rows take more registers for it than they leave for weights: x there | where it is used, 64 rows: bf16 (2048, 2048)
    // 11.8 | 11.4 us
    const float most = stream_most();
    const int turn = stream_turn(tile0, a.steps);
    struct Raw {
        u32x4 h[kRaw];
    };
    auto load_x = [&](int t, int s) {
        Raw r;
#pragma unroll
        for (int h = 0; h < kRaw; ++h) {
            r.h[h] = *(const u32x4*)(xp[t] + (int64_t)s * kXS + 16 * h);
        }
        return r;
    };
    u32x4     wa[kChunk][NT], wb[kChunk][NT];
    Raw       xa[kChunk][MT], xb[kChunk][MT];
    auto  fetch = [&](u32x4(&buf)[kChunk][NT], Raw(&xbuf)[kChunk][MT], int base) {
        if constexpr (kAhead) {
#pragma unroll
            for (int kk = 0; kk < kChunk; ++kk) {
                const int s = min(base + kk, a.steps - 1);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    xbuf[kk][t] = load_x(t, s);
                }
            }
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int kk = 0; kk < kChunk; kk += 4) {
            const int64_t at   = stream_step_at<Epi>(a, min(base + kk, a.steps - 1) & ~3, turn);  // (four steps are contiguous)
            const int     last = a.steps - 1 - (min(base + kk, a.steps - 1) & ~3);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    buf[kk + e][j] = __builtin_nontemporal_load((const u32x4*)(wp[j] + at + min(e, last) * 1024));
                }
            }
        }
        if constexpr (kAhead) {
            asm volatile("" ::: "memory");
        }
    };
    floatx4 sum[2][MT][NT];  // (fp32: of the chunk, the low and middle parts' and the high parts')
    auto    compute = [&](const u32x4(&buf)[kChunk][NT], const Raw(&xbuf)[kChunk][MT], int base) {
        static_assert(kParts == 1 || kChunk <= kSplitSteps, "sums of fp32 rows");
        if constexpr (kParts > 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    sum[0][t][j] = sum[1][t][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
#pragma unroll
        for (int kk = 0; kk < kChunk; ++kk) {
            if (base + kk < a.steps) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    Raw b;
                    if constexpr (kAhead) {
                        b = xbuf[kk][t];
                    }
                    else {
                        b = load_x(t, base + kk);
                    }
                    SplitRow f;
                    if constexpr (kParts > 1) {
                        f = stream_split(b.h[0], b.h[1], most);
                    }
                    else {
                        f.part[0] = b.h[0];
                    }
#pragma unroll
                    for (int p = 0; p < kParts; ++p) {
                        floatx4(&to)[MT][NT] = kParts > 1 ? sum[p / 2] : acc;
#pragma unroll
                        for (int j = 0; j < NT; ++j) {
                            to[t][j] = StreamOp<T>::mma(buf[kk][j], f.part[p], to[t][j]);
                        }
                    }
                }
            }
        }
        if constexpr (kParts > 1) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    acc[t][j] += sum[0][t][j] + sum[1][t][j];
                }
            }
        }
    };
    constexpr int kStride = W * kChunk;
    int           base    = wave * kChunk;
    if (base < a.steps) {
        fetch(wa, xa, base);
        for (; base + 2 * kStride < a.steps; base += 2 * kStride) {
            fetch(wb, xb, base + kStride);
            compute(wa, xa, base);
            fetch(wa, xa, base + 2 * kStride);
            compute(wb, xb, base + kStride);
        }
        if (base + kStride < a.steps) {  // the last two chunks, or the last: nothing is fetched that is not used
            fetch(wb, xb, base + kStride);
            compute(wa, xa, base);
            compute(wb, xb, base + kStride);
        }
        else {
            compute(wa, xa, base);
        }
    }
    unsigned warm = 0;  // (what the outputs are added to is on its way while the waves meet; two tiles of columns have no register for it)
    if (NT == 1 && wave < MT) {
        warm = epi.touch(a, item, mb + min(wave * 16 + fr, M - 1), min(tile0 * 16 + fc * 4, a.N - 1));
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            red[wave][t * NT + j][lane] = acc[t][j];
        }
    }
    __syncthreads();
    if (wave < MT) {  // wave t: row tile t
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            floatx4 s = red[0][wave * NT + j][lane];
            for (int v = 1; v < W; ++v) {
                s += red[v][wave * NT + j][lane];
            }
            acc[0][j] = s;
        }
        if constexpr (NT == 1) {
            asm volatile("" ::"v"(warm));
        }
        const int m = wave * 16 + fr;
        if (m < M) {
            epi.template rows<NT>(a, item, mb + m, tile0 * 16 + fc * 4, acc[0]);
        }
    }
}

// ---- many rows: tiles staged in LDS by DMA -------------------------------------------------------------------------------------------
// Workgroup tile BM x BN, 4 waves of (BM / WM) x (BN / WN) outputs, one step of k (64 bytes a row) per stage, B = three to six stages in LDS.  The fragments of
// step s + 1 are read into a second register set under the MFMAs of step s, so the stage of step s is free when step s begins: the DMA of stage s + B
// is issued there and has B - 1 steps to land.  One barrier a step.  Weight blocks are lane-linear in memory and in LDS; a row of x is four
// 16-byte pieces, piece c of row r at c ^ ((r >> 1) & 3) (the swizzle is on the DMA's source address): fragment reads meet every bank once.
__device__ __forceinline__ void stream_dma16(__amdgpu_buffer_rsrc_t rs, int voff, int soff, unsigned lds)
{
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(voff), "s"(lds), "s"(rs), "s"(soff)
                 : "memory");
}

// Which tile a workgroup owns.  XCD-aware order: workgroup i runs on XCD i % 8; each XCD gets a contiguous eighth of the tiles, walked in bands of
// BAND row tiles, so that what its CUs hold at a time shares operands in its L2.  Items with rows of their own (row_offsets): the row tiles of all
// items are one list, which the XCDs share evenly.  The launch has workgroups for rows / BM + items row tiles, as many as there can be; those past the list's end leave (they
// were the last XCD's share before: nine experts of (2048, 2816), 12400 rows in 256 x 128 tiles 180 us, now 174; 1500 rows, a forward of eight layers 2.53 ms, now 2.36)
struct StreamTile {
    int tm, tn, item;  // item < 0: past the end of the list
};
template<int BM, int BN, int BAND>
__device__ __forceinline__ StreamTile stream_tile_of(const StreamArgs& a, const int* row_offsets, int items)
{
    const int lane = threadIdx.x & 63, tns = ((a.col1 ? a.col1 : a.tiles * 16) - a.col0 + BN - 1) / BN;
    auto      count = [&](int g) { return g < items ? (row_offsets[g + 1] - row_offsets[g] + BM - 1) / BM : 0; };  // row tiles of an item
    auto      prefix = [&](int n) {  // inclusive sums over the lanes
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const int up = __shfl_up(n, d);
            n += lane >= d ? up : 0;
        }
        return n;
    };
    int tms = (a.M + BM - 1) / BM, n = 0, sum = 0;
    if (row_offsets) {
        tms = 0;
        for (int base = 0; base < items; base += 64) {
            n   = count(base + lane);
            sum = prefix(n);
            tms += __builtin_amdgcn_readlane(sum, 63);
        }
    }
    const int total = tms * tns, i = blockIdx.x, q = total >> 3, rem = total & 7, xcd = i & 7;
    if (i >= total) {
        return StreamTile{0, 0, -1};
    }
    const int lin  = xcd * q + min(xcd, rem) + (i >> 3);
    const int band = lin / (BAND * tns), in = lin - band * BAND * tns, h = min(BAND, tms - band * BAND);
    StreamTile t{band * BAND + in % h, in / h, (int)blockIdx.y};
    if (row_offsets) {
        for (int base = 0; base < items; base += 64) {
            if (items > 64) {
                n   = count(base + lane);
                sum = prefix(n);
            }
            const uint64_t past = __ballot(t.tm < sum);
            if (past) {
                const int f = __builtin_ctzll(past);
                t.item      = base + f;
                t.tm -= __builtin_amdgcn_readlane(sum - n, f);
                break;
            }
            t.tm -= __builtin_amdgcn_readlane(sum, 63);
        }
        t.item = __builtin_amdgcn_readfirstlane(t.item);
        t.tm   = __builtin_amdgcn_readfirstlane(t.tm);
    }
    return t;
}

// Stages of a tile in LDS.  The small tiles are what a few hundred rows of a narrow product get, about one workgroup a CU: only the bytes in flight hide the
// way to memory.  fp16, weights from HBM, 200 rows of (4096, 4096) in 64 x 64 tiles: three stages 38 us, four 28, six 19.9, eight 18.6 (300 rows, two tiles on
// some CUs: 41, 37, 37, 38); 400 rows of (5120, 5120) in 128 x 128 tiles: three 57, four 44
constexpr int stream_tile_bufs(int bm, int bn)
{
    return bm == 64 && bn == 64 ? 6 : bm == 128 && bn == 128 || bm == 256 && bn == 256 ? 4 : 3;
}

constexpr int stream_split_bufs(int bm, int kp)  // ... of a group of waves of a tile whose rows are fp32
{
    return bm == 64 && kp == 1 ? 4 : 3;
}

template<class T, class Epi, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256, BM* BN > 256 * 128 ? 1 : 2) void stream_tile_kernel(StreamArgs a, Epi epi)
{
    static_assert(WM * WN == 4, "four waves");
    constexpr int MI = BM / WM / 16, NI = BN / WN / 16;
    constexpr int kXB = BM * 64, kWB = BN * 64, kStage = kXB + kWB, kBufs = stream_tile_bufs(BM, BN);
    constexpr int kXP = BM / 16 / 4, kWP = BN / 16 / 4;  // DMA pieces of one KB per wave and stage
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const StreamTile t = stream_tile_of<BM, BN, 8>(a, epi.row_offsets(), epi.items());
    if (t.item < 0) {
        return;
    }
    const int  m0 = t.tm * BM, n0 = a.col0 + t.tn * BN;
    const auto item = epi.item(t.item, a.M, n0);
    const int  Mloc = min(item.M - m0, BM);
    if (Mloc <= 0) {  // an item with fewer rows than the launch's largest
        return;
    }
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + item.x_off + m0 * a.ldx), 0, (int)((Mloc - 1) * a.ldx + (int64_t)a.steps * 64), 0x00020000);
    const int64_t w_left = stream_weight_bytes(a, n0 >> 4);
    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + item.w_off + (int64_t)(n0 >> 4) * a.w_tile), 0, (int)min(w_left, (int64_t)0xffffffff), 0x00020000);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
    int            xoff[kXP];
#pragma unroll
    for (int r = 0; r < kXP; ++r) {
        const int row = 16 * (kXP * wave + r) + (lane >> 2);
        xoff[r]       = (int)(min(row, Mloc - 1) * a.ldx) + ((lane & 3) ^ ((row >> 1) & 3)) * 16;
    }
    int woff[kWP];
#pragma unroll
    for (int r = 0; r < kWP; ++r) {
        woff[r] = (int)(min(kWP * wave + r, a.tiles - 1 - (n0 >> 4)) * a.w_tile) + lane * 16;
    }
    const int turn = stream_turn(n0 >> 4, a.steps);
    auto      dma  = [&](int s, int buf) {
        const int      ws  = (int)stream_step_at<Epi>(a, s, turn);
        const unsigned dst = lds0 + buf * kStage;
#pragma unroll
        for (int r = 0; r < kXP; ++r) {
            stream_dma16(rs_x, xoff[r], s * 64, dst + (kXP * wave + r) * 1024);
        }
#pragma unroll
        for (int r = 0; r < kWP; ++r) {
            stream_dma16(rs_w, woff[r], ws, dst + kXB + (kWP * wave + r) * 1024);
        }
    };
    floatx4 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const int wm = wave / WN, wn = wave % WN;
    const int fr = lane & 15, fc = lane >> 4;
    const int xf = (wm * (BM / WM) + fr) * 64 + ((fc ^ ((fr >> 1) & 3)) << 4);
    const int wf = kXB + wn * NI * 1024 + lane * 16;
    const int steps = a.steps;
    u32x4     fx[2][MI], fw[2][NI];
    auto      read = [&](int q, int buf) {
        const char* st = smem + buf * kStage;
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            fw[q][j] = *(const u32x4*)(st + wf + j * 1024);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            fx[q][i] = *(const u32x4*)(st + xf + i * 1024);
        }
    };
    constexpr int kPieces = kXP + kWP;
    // no branch inside a step (the reads and MFMAs of one block are interleaved): past the end the DMA fetches the last stage again, into
    // buffers that are not read any more
#pragma unroll
    for (int b = 0; b < kBufs; ++b) {
        dma(min(b, steps - 1), b);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kBufs - 1) * kPieces) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    int  buf  = 0;  // stage of step s
    auto step = [&](auto Q, int s) {
        constexpr int q   = decltype(Q)::value;
        const int     nxt = buf == kBufs - 1 ? 0 : buf + 1;
        // this wave's fragments of step s are in registers and its pieces of stage s + 1 have landed; then everybody's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kBufs - 2) * kPieces) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        dma(min(s + kBufs, steps - 1), buf);
        read(q ^ 1, nxt);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                acc[i][j] = StreamOp<T>::mma(fw[q][j], fx[q][i], acc[i][j]);
            }
        }
#pragma unroll
        for (int g = 0; g < MI + NI; ++g) {  // the next step's fragment reads go between the MFMAs
            __builtin_amdgcn_sched_group_barrier(0x008, MI * NI / (MI + NI), 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        buf = nxt;
    };
    for (int s = 0; s < steps; s += 2) {
        step(std::integral_constant<int, 0>{}, s);
        if (s + 1 < steps) {
            step(std::integral_constant<int, 1>{}, s + 1);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the DMA writes this workgroup's LDS)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + wm * (BM / WM) + i * 16 + fr;
        if (m < item.M) {
            epi.template rows<NI>(a, item, m, n0 + wn * NI * 16 + fc * 4, acc[i]);
        }
    }
}

// ---- many rows in fp32: tiles whose rows are split on the way to the matrix cores ---------------------------------------------------------
// As above with rows of 128 bytes a step in LDS, piece c of row r at c ^ ((r >> 1) & 7); the waves share out the rows and each has all columns of the tile, since a
// fragment of x takes 52 vector instructions to split and 48 cycles of matrix work for every 16 columns.  us, fp32 weights and matrix instructions before / now:
// (2048, 8448) 450 rows 153 / 69, 6000 rows 1506 / 524 (128 x 128 tiles, 1.2 PFLOP/s of bf16 products); (2048, 2048) 450 rows 38 / 24: one tile a CU, whose 12 KB a step
// come at 36 GB/s, what a CU's lines in flight give over the way to memory.  Relative error against 64 bits (2-norm), before / now: normal rows, K 2048 8.1e-7 / 1.7e-7;
// sums of one sign 6.3e-7 / 6.3e-8 (in one run of all steps 9.8e-7: see kSplitSteps)
// KP groups of four waves share out k, each with stages of its own, and meet in LDS in their order: where every tile has a CU to itself, four groups have more on their way
// (one / four, us: (2048, 2048) 200 rows 21.9 / 17.8, 450 rows 23.3 / 21.8; (8448, 2048) 300 rows 81 / 59; (768, 2048) 200 rows 10.4 / 10.6).
template<class Epi, int BM, int BN, int KP>
__global__ __launch_bounds__(256 * KP, KP == 1 ? 2 : 4) void stream_tile_split_kernel(StreamArgs a, Epi epi)
{
    constexpr int MI = BM / 64, NI = BN / 16;
    constexpr int kXB = BM * 128, kWB = BN * 64, kStage = kXB + kWB, kBufs = stream_split_bufs(BM, KP);
    constexpr int kXP = BM / 32, kWP = BN / 64;  // DMA pieces of one KB per wave and stage
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, ph = __builtin_amdgcn_readfirstlane(tid >> 8);
    const StreamTile t = stream_tile_of<BM, BN, 8>(a, epi.row_offsets(), epi.items());
    if (t.item < 0) {
        return;
    }
    const int  m0 = t.tm * BM, n0 = a.col0 + t.tn * BN;
    const auto item = epi.item(t.item, a.M, n0);
    const int  Mloc = min(item.M - m0, BM);
    if (Mloc <= 0) {  // an item with fewer rows than the launch's largest
        return;
    }
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + item.x_off + m0 * a.ldx), 0, (int)((Mloc - 1) * a.ldx + (int64_t)a.steps * 128), 0x00020000);
    const int64_t w_left = stream_weight_bytes(a, n0 >> 4);
    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + item.w_off + (int64_t)(n0 >> 4) * a.w_tile), 0, (int)min(w_left, (int64_t)0xffffffff), 0x00020000);
    char* const    stages = smem + ph * (kBufs * kStage);
    const unsigned lds0   = __builtin_amdgcn_readfirstlane((unsigned)(size_t)stages);
    int            xoff[kXP], woff[kWP];
#pragma unroll
    for (int r = 0; r < kXP; ++r) {
        const int row = 8 * (kXP * wave + r) + (lane >> 3);
        xoff[r]       = (int)(min(row, Mloc - 1) * a.ldx) + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int r = 0; r < kWP; ++r) {
        woff[r] = (int)(min(kWP * wave + r, a.tiles - 1 - (n0 >> 4)) * a.w_tile) + lane * 16;
    }
    const int turn = stream_turn(n0 >> 4, a.steps);
    auto      dma  = [&](int s, int buf) {
        const int      ws  = (int)stream_step_at<Epi>(a, s, turn);
        const unsigned dst = lds0 + buf * kStage;
#pragma unroll
        for (int r = 0; r < kXP; ++r) {
            stream_dma16(rs_x, xoff[r], s * 128, dst + (kXP * wave + r) * 1024);
        }
#pragma unroll
        for (int r = 0; r < kWP; ++r) {
            stream_dma16(rs_w, woff[r], ws, dst + kXB + (kWP * wave + r) * 1024);
        }
    };
    const float most = stream_most();
    floatx4 acc[MI][NI], sum[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const int fr = lane & 15, fc = lane >> 4;
    const int xrow = (wave * (BM / 4) + fr) * 128, sw = (fr >> 1) & 7;
    const int wf = kXB + lane * 16;
    // a group's steps begin at s0; all groups walk as many as the first has, for the barriers, the last ones some without products
    const int run = ((a.steps + KP - 1) / KP + kSplitSteps - 1) / kSplitSteps * kSplitSteps, s0 = min(ph * run, a.steps - 1);
    const int steps = min(a.steps - ph * run, run), walk = min(run, a.steps);
    u32x4     fx[2][MI][2], fw[2][NI];
    auto      read = [&](int q, int buf) {
        const char* st = stages + buf * kStage;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                fx[q][i][h] = *(const u32x4*)(st + xrow + i * 2048 + (((2 * fc + h) ^ sw) << 4));
            }
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            fw[q][j] = *(const u32x4*)(st + wf + j * 1024);
        }
    };
    constexpr int kPieces = kXP + kWP;
#pragma unroll
    for (int b = 0; b < kBufs; ++b) {
        dma(s0 + max(min(b, steps - 1), 0), b);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kBufs - 1) * kPieces) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    int  buf  = 0;  // stage of step s
    auto step = [&](auto Nth, int s) {  // step N of a run of kSplitSteps
        constexpr int n = decltype(Nth)::value, q = n & 1;
        const int     nxt = buf == kBufs - 1 ? 0 : buf + 1;
        // this wave's fragments of step s are in registers and its pieces of stage s + 1 have landed; then everybody's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kBufs - 2) * kPieces) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        dma(s0 + max(min(s + kBufs, steps - 1), 0), buf);
        read(q ^ 1, nxt);
        buf = nxt;
        if (KP > 1 && s >= steps) {
            return;
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const SplitRow f = stream_split(fx[q][i][0], fx[q][i][1], most);
#pragma unroll
            for (int p = 0; p < 3; ++p) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    sum[i][j] = StreamOp<float>::mma(fw[q][j], f.part[p], n == 0 && p == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : sum[i][j]);
                }
            }
        }
    };
    for (int s = 0; s < walk; s += kSplitSteps) {
        static_assert(kSplitSteps == 8, "the steps below");
        step(std::integral_constant<int, 0>{}, s);
#define TM_STEP(N)                                           \
    if (s + N < walk) {                                       \
        step(std::integral_constant<int, N>{}, s + N);       \
    }
        TM_STEP(1) TM_STEP(2) TM_STEP(3) TM_STEP(4) TM_STEP(5) TM_STEP(6) TM_STEP(7)
#undef TM_STEP
        if (KP == 1 || s < steps) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    acc[i][j] += sum[i][j];
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the DMA writes this workgroup's LDS)
    if constexpr (KP > 1) {
        static_assert(kBufs * kStage * KP >= (KP - 1) * BM * BN * 4, "the groups' sums lie where their stages were");
        __syncthreads();
        floatx4* const red = (floatx4*)smem;
        if (ph > 0) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    red[(((ph - 1) * 4 + wave) * MI * NI + i * NI + j) * 64 + lane] = acc[i][j];
                }
            }
        }
        __syncthreads();
        if (ph > 0) {
            return;
        }
#pragma unroll
        for (int p = 0; p < KP - 1; ++p) {  // fixed order
#pragma unroll
            for (int i = 0; i < MI; ++i) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    acc[i][j] += red[((p * 4 + wave) * MI * NI + i * NI + j) * 64 + lane];
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + wave * (BM / 4) + i * 16 + fr;
        if (m < item.M) {
            epi.template rows<NI>(a, item, m, n0 + fc * 4, acc[i]);
        }
    }
}

// ---- many rows of a 16-bit format: 256 x 256 tiles -----------------------------------------------------------------------------------
// 4 waves of 128 x 128 outputs (v_mfma_f32_16x16x32, 256 accumulator registers, one wave per SIMD): a step moves 32 KB into a CU and 64 KB out of its LDS per
// 1024 cycles of matrix work, where the 256 x 128 tiles above move 48 and 96.  Power holds the clock, and what a multiply-add costs depends on the
// instruction: from registers alone, on normal operands, 16x16x32 reaches 1.98 PFLOP/s on this card and 32x32x16 1.72 (2.40 and 2.43 on zeros); neighbours in
// the order of issue share an operand, which is another 1 %.  bf16, 8192 rows, MI355X: (K, N) = (4096, 21504) 1162 us, (25600, 4096) 1280 us =
// 1.34 PFLOP/s, (8448, 2048) 212; with 32x32x16 1225, 1374 and 230, 256 x 128 tiles 1281 and 1670 (first two).
// The MFMAs are asm so that the accumulators are accumulation registers and nothing else (left to the register allocator, it spills fragments); they
// and the fragment reads stay in the order written.
template<class T>
__device__ __forceinline__ void stream_mma_acc(floatx4& c, const u32x4& a, const u32x4& b)
{
    if constexpr (std::is_same<T, __bf16>::value) {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
    else {
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    }
}

template<class T, class Epi>
__global__ __launch_bounds__(256, 1) void stream_tile256_kernel(StreamArgs a, Epi epi)
{
    constexpr int BM = 256, BN = 256, kXB = BM * 64, kStage = kXB + BN * 64, kBufs = stream_tile_bufs(BM, BN);
    constexpr int kXP = 4, kWP = 4, kPieces = 8;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const StreamTile t = stream_tile_of<BM, BN, 4>(a, epi.row_offsets(), epi.items());
    if (t.item < 0) {
        return;
    }
    const int  m0 = t.tm * BM, n0 = a.col0 + t.tn * BN;
    const auto item = epi.item(t.item, a.M, n0);
    const int  Mloc = min(item.M - m0, BM);
    if (Mloc <= 0) {
        return;
    }
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + item.x_off + m0 * a.ldx), 0, (int)((Mloc - 1) * a.ldx + (int64_t)a.steps * 64), 0x00020000);
    const int64_t w_left = stream_weight_bytes(a, n0 >> 4);
    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)(a.w + item.w_off + (int64_t)(n0 >> 4) * a.w_tile), 0, (int)min(w_left, (int64_t)0xffffffff), 0x00020000);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
    int            xoff[kXP], woff[kWP];
#pragma unroll
    for (int r = 0; r < kXP; ++r) {
        const int row = 16 * (kXP * wave + r) + (lane >> 2);
        xoff[r]       = (int)(min(row, Mloc - 1) * a.ldx) + ((lane & 3) ^ ((row >> 1) & 3)) * 16;
        woff[r]       = (int)(min(kWP * wave + r, a.tiles - 1 - (n0 >> 4)) * a.w_tile) + lane * 16;
    }
    const int turn      = stream_turn(n0 >> 4, a.steps);
    auto      dma_piece = [&](int s, int buf, int n) {
        const unsigned dst = lds0 + buf * kStage + (4 * wave + (n & 3)) * 1024;
        if (n < 4) {
            stream_dma16(rs_x, xoff[n], s * 64, dst);
        }
        else {
            stream_dma16(rs_w, woff[n - 4], (int)stream_step_at<Epi>(a, s, turn), dst + kXB);
        }
    };
    floatx4 acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const int wm = wave >> 1, wn = wave & 1;
    const int fr = lane & 15, fc = lane >> 4;
    // x: row r at r * 64, piece c at c ^ ((r >> 1) & 3)
    const int xf = (wm * 128 + fr) * 64 + ((fc ^ ((fr >> 1) & 3)) << 4);
    const int wf = kXB + wn * 8192 + lane * 16;
    // The fragments of step s + 1 are read under the MFMAs of step s, so the step's own stage is free behind its barrier: the DMA of stage s + kBufs goes there
    u32x4     fx[2][8], fw[2][8];
    const int steps = a.steps;
    auto      read  = [&](auto Q, const char* st, int n) {
        constexpr int q = decltype(Q)::value;
        if (n < 8) {
            fw[q][n] = *(const u32x4*)(st + wf + n * 1024);
        }
        else {
            fx[q][n - 8] = *(const u32x4*)(st + xf + (n - 8) * 1024);
        }
    };
#pragma unroll
    for (int b = 0; b < kBufs; ++b) {
#pragma unroll
        for (int n = 0; n < kPieces; ++n) {
            dma_piece(min(b, steps - 1), b, n);
        }
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kBufs - 1) * kPieces) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int n = 0; n < 16; ++n) {
        read(std::integral_constant<int, 0>{}, smem, n);
    }
    int  buf  = 0;  // stage of step s
    auto step = [&](auto Q, int s) {
        constexpr int q   = decltype(Q)::value;
        const int     nxt = buf == kBufs - 1 ? 0 : buf + 1;
        // this wave's fragments of step s are in registers and its pieces of stage s + 1 have landed; then everybody's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kBufs - 2) * kPieces) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const char* st = smem + nxt * kStage;
        const int   sd = min(s + kBufs, steps - 1);
#pragma unroll
        for (int n = 0; n < 64; ++n) {
            if (n % 3 == 0 && n < 48) {
                read(std::integral_constant<int, q ^ 1>{}, st, n / 3);
            }
            if (n % 8 == 4) {
                dma_piece(sd, buf, n >> 3);
            }
            const int i = n >> 3, j = i & 1 ? 7 - (n & 7) : n & 7;
            stream_mma_acc<T>(acc[i][j], fw[q][j], fx[q][i]);
        }
        buf = nxt;
    };
    int s = 0;
    for (; s + 1 < steps; s += 2) {
        step(std::integral_constant<int, 0>{}, s);
        step(std::integral_constant<int, 1>{}, s + 1);
    }
    if (s < steps) {
        step(std::integral_constant<int, 0>{}, s);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the DMA writes this workgroup's LDS)
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // (the last results are passes behind their issue)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            asm volatile("s_nop 7" : "+a"(acc[i][c]));
        }
    }
    // A lane's results are four columns each of 16 rows apart; through the wave's own 16 KB of LDS they leave as whole runs of a row (512 bytes of fp32): 32
    // rows at a time, piece p (four columns) of row r at p ^ r
    __builtin_amdgcn_s_barrier();  // every wave is through with the stages
    asm volatile("" ::: "memory");
    floatx4* const sw = (floatx4*)(smem + wave * 16384);
    const int      l31 = lane & 31, half = lane >> 5;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int n = 0; n < 16; ++n) {  // row 16 (n / 8) + fr, columns 16 (n % 8) + 4 fc + 0 .. 3
            const int r = (n >> 3) * 16 + fr;
            sw[r * 32 + ((4 * (n & 7) + fc) ^ r)] = acc[2 * i + (n >> 3)][n & 7];
        }
        __builtin_amdgcn_wave_barrier();
        const int mb = m0 + wm * 128 + i * 32, nb = n0 + wn * 128;
        if constexpr (Epi::kPairs) {  // gate and up are 16 columns (four pieces) apart: a lane has both
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                const int     r = n * 4 + (lane >> 4), p = ((lane & 15) >> 2) * 8 + (lane & 3);
                const floatx4 v[2] = {sw[r * 32 + (p ^ r)], sw[r * 32 + ((p + 4) ^ r)]};
                if (mb + r < item.M) {
                    epi.template rows<2>(a, item, mb + r, nb + p * 4, v);
                }
            }
        }
        else if constexpr (Epi::kReads > 0) {  // what kReads outputs need is on its way together (DenseEpi)
            constexpr int kOps = Epi::kReads;
#pragma unroll 1
            for (int n0 = 0; n0 < 16; n0 += kOps) {
                typename Epi::Operand op[kOps];
                epi.template operands<kOps>(a, item, [&](int n) { return int2{min(mb + (n0 + n) * 2 + half, item.M - 1), nb + l31 * 4}; }, op);
#pragma unroll
                for (int n = 0; n < kOps; ++n) {
                    const int     r = (n0 + n) * 2 + half;
                    const floatx4 v = sw[r * 32 + (l31 ^ r)];
                    if (mb + r < item.M) {
                        epi.join(a, item, mb + r, nb + l31 * 4, v, op[n]);
                    }
                }
            }
        }
        else {
#pragma unroll
            for (int n = 0; n < 16; ++n) {
                const int     r = n * 2 + half;
                const floatx4 v[1] = {sw[r * 32 + (l31 ^ r)]};
                if (mb + r < item.M) {
                    epi.template rows<1>(a, item, mb + r, nb + l31 * 4, v);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ---- weight images of bf16 and fp32 linears ----------------------------------------------------------------------------------------
// Images are stored in FRAGMENT ORDER: the 16 rows x 64 bytes block (n / 16, k / step) is one contiguous KB laid out as the 64 lanes of
// its MFMA fragment (16 bytes each: lane = piece * 16 + n % 16), blocks of one 16-row tile consecutive along k -- a wave's fragment
// load is one contiguous KB and a workgroup streams whole contiguous runs of HBM instead of 64-byte pieces of 16 rows
// (from stream_turn's step on)
__host__ __device__ inline size_t dense_frag_index(int n, int k, int steps)
{
    constexpr int E = 8, S = 4 * E;  // elements of a 16-byte piece, of a step
    const int     at = k / S + stream_turn(n >> 4, steps);
    return (((size_t)(n >> 4) * steps + (at < steps ? at : at - steps)) * 64 + (k % S) / E * 16 + (n & 15)) * E + k % E;
}

// ---- which kernel, which shape -------------------------------------------------------------------------------------------------------
// (row tiles, column tiles a wave, column waves, k-phases) of the skinny kernels that exist: 64 columns a workgroup of four waves, 96 of six where those
// fill the CUs more evenly; bf16 beyond 16 rows also 128 of eight, which read x less often; and 128 columns where a wave needs a pair of column tiles.  k-phases gave nothing at 184 sizes.
#define TM_STREAM_SHAPES(X) X(1, 1, 4, 1) X(2, 1, 4, 1) X(4, 1, 4, 1) X(1, 1, 6, 1) X(2, 1, 6, 1) X(4, 1, 6, 1)
#define TM_STREAM_SHAPES_WIDE(X) X(2, 1, 8, 1) X(4, 1, 8, 1)
#define TM_STREAM_SHAPES_PAIRS(X) X(1, 2, 4, 2) X(2, 2, 4, 2) X(4, 2, 4, 1)

// waves of the narrow kernel (row tiles x column tiles <= 2): eight where sixteen would have nothing to do, or would keep a second workgroup off the CU
inline int stream_narrow_waves(const StreamArgs& a)
{
    return a.steps <= 64 || a.tiles > 256 ? 8 : 16;
}

struct StreamPlan {
    bool skinny, narrow;  // narrow: no slices across workgroups
    int  mt, cw, splits, split_steps, row_blocks;  // skinny kernel (cw: column tiles a workgroup)
    int  tile;                                 // 0: 256 x 256 (16-bit formats), 1: 256 x 128, 2: 128 x 128, 3: 64 x 64
    int  cut, tile2;                           // > 0: columns [0, cut) in `tile`, the others in a launch of tile2
};
// steps of k, image columns, rows, items (own_rows: each with rows of its own, `rows` in total), bytes of an element; pairs: a wave needs two
// column tiles; ws_bytes / tickets: what slices of k may use (0: no slices); border: x is read elsewhere from multiples of this many columns on (a
// multiple of 128; 0: nowhere); k_major: the image holds four steps of every column tile before the next four; item_rows: own_rows, the most an item has (0: rows);
// cut_ok: the columns may go to two launches; few_only: up to 64 rows no tiles (their epilogues store no cache columns)
StreamPlan stream_plan(int steps, int cols, int rows, int items, bool own_rows, int elem, bool pairs, size_t ws_bytes, int tickets, int border = 0,
                       bool k_major = false, int item_rows = 0, bool cut_ok = false, bool few_only = false);
constexpr size_t kStreamWsBytes = (size_t)16 << 20;  // scratch and arrival counters that serve every plan
constexpr int    kStreamTickets = 4096;

}  // namespace tmk
