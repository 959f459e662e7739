// Products of a few rows that make the norm of their rows themselves: every workgroup brings the residual rows into LDS, norms them there, and then streams its columns'
// weights past them.
//
// What bounds such a step is its launches: a norm of a few rows is a chain of latencies, 1.8 us of a graph's chain of launches on its own and 3.3 among a model's other
// kernels.  Made by every workgroup of the product behind it, it reads no byte more than the normed rows would and runs under the first weights' way from memory:
// fp16, 8 rows of (2048, 16384) 13.6 us, rows that need no norm 13.2, norm and product apart 15.2.  The residual is therefore added where the sublayer's output is made
// (F16EpiAdd): as a second operand here, eight rows of it in every CU, which takes 33 KB a microsecond from wherever it comes, cost the whole gain.  So did a
// norm whose pieces were dealt to the threads without regard to rows (four sums over lanes a wave and two barriers: 15.8 us); a wave with a whole row needs one.
// The weights are asked for behind the rows (loads return in order) and ahead of the sums.  Behind the last barrier no wave waits for another until the k-phases meet:
// all of k is in LDS.
#pragma once
#include "gemm_stream.h"
#include <algorithm>

namespace tmk {

constexpr int kRowsPad = 16;  // bytes behind a row in LDS: 16 rows' pieces of the same k then lie in different banks

// The rows of rmsnorm_kernel (norm_row.h), a multiple of 512 channels: as many waves a row as there are for it (`team`), RPW rows a wave, P pieces of 512 channels of each.
// A wave that has a whole row needs no other wave's sum, and one barrier does.
template<int RPW, int P>
struct NormRows {
    const half_t* resid;
    const half_t* weight;
    float         eps;
    int           team;  // waves a row, a power of two
    struct Regs {
        half8_t r[RPW][P], w[P];
    };
    __device__ __forceinline__ int piece(int nv, int wave, int lane, int q) const
    {
        return min(((wave & (team - 1)) * P + q) * 64, nv - 64) + lane;
    }
    __device__ __forceinline__ bool mine(int nv, int wave, int q) const
    {
        return ((wave & (team - 1)) * P + q) * 64 < nv;
    }
    __device__ __forceinline__ void load(Regs& g, int M, int n, int wave, int lane, int waves) const
    {
        const int nv = n * 4;
#pragma unroll
        for (int j = 0; j < RPW; ++j) {
            const int m = min(wave / team + j * (waves / team), M - 1);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                g.r[j][q] = *(const half8_t*)(resid + ((size_t)m * nv + piece(nv, wave, lane, q)) * 8);
            }
        }
#pragma unroll
        for (int q = 0; q < P; ++q) {
            g.w[q] = *(const half8_t*)(weight + (size_t)piece(nv, wave, lane, q) * 8);
        }
    }
    // put(m, piece of eight channels, values): where they go; every wave comes here, and a barrier stands behind it
    template<class Put>
    __device__ __forceinline__ void finish(Regs& g, int M, int n, float* sums, int wave, int lane, int waves, Put put) const
    {
        const int nv = n * 4;
        float     ss[RPW];
#pragma unroll
        for (int j = 0; j < RPW; ++j) {
            ss[j] = 0.f;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                if (mine(nv, wave, q)) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float f = (float)g.r[j][q][e];
                        ss[j]         = __builtin_fmaf(f, f, ss[j]);
                    }
                }
            }
            ss[j] = group_sum<64>(ss[j]);
        }
        if (team > 1) {  // (RPW is one then)
            if (lane == 0) {
                sums[wave] = ss[0];
            }
            __syncthreads();
            ss[0] = 0.f;
            for (int i = 0; i < team; ++i) {
                ss[0] += sums[(wave & ~(team - 1)) + i];
            }
        }
#pragma unroll
        for (int j = 0; j < RPW; ++j) {
            const int   m   = wave / team + j * (waves / team);
            const float inv = 1.0f / __builtin_sqrtf(ss[j] / (float)(nv * 8) + eps);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                if (m < M && mine(nv, wave, q)) {  // (the same for the whole wave)
                    half8_t y;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        y[e] = (half_t)__builtin_fmaf((float)g.r[j][q][e], inv, -0.f);  // (a product: one instruction with both conversions)
                    }
                    put(m, piece(nv, wave, lane, q), y * g.w[q]);
                }
            }
        }
        __syncthreads();
    }
};

// Up to 16 rows; CW column tiles x KP k-phases of waves, R steps of weights in flight a wave.  Grid: column groups
template<class T, class Epi, class Rows, int CW, int KP, int R>
__global__ __launch_bounds__(CW* KP * 64) void stream_rows_kernel(StreamArgs a, Epi epi, Rows rows)
{
    constexpr int kWaves = CW * KP, kChunk = 8;
    static_assert(R % kChunk == 0, "whole chunks");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int  lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int  cw = wave % CW, ph = wave / CW, tile = blockIdx.x * CW + cw;
    const auto item = epi.item(0, a.M, blockIdx.x * CW * 16);
    const int  M = a.M, n = a.steps, pitch = n * 64 + kRowsPad;

    typename Rows::Regs g;
    rows.load(g, M, n, wave, lane, kWaves);
    asm volatile("" ::: "memory");
    // a wave takes every KP-th chunk of eight steps: its step i of `count` is ...
    const int   chunks = (n + kChunk - 1) / kChunk, mine = (chunks - ph + KP - 1) / KP;
    const int   count  = mine <= 0 ? 0 : mine * kChunk - ((chunks - 1) % KP == ph ? chunks * kChunk - n : 0);
    auto        step   = [&](int i) { return ((i / kChunk) * KP + ph) * kChunk + i % kChunk; };
    const char* wp     = a.w + (int64_t)min(tile, a.tiles - 1) * a.w_tile + lane * 16;
    const int   turn   = stream_turn(min(tile, a.tiles - 1), a.steps);
    u32x4       ring[R];
    auto        load = [&](int i) { return __builtin_nontemporal_load((const u32x4*)(wp + stream_step_at<Epi>(a, min(step(min(i, max(count - 1, 0))), n - 1), turn))); };
#pragma unroll
    for (int k = 0; k < R; ++k) {
        ring[k] = load(k);
    }
    asm volatile("" ::: "memory");
    rows.finish(g, M, n, (float*)(smem + M * pitch), wave, lane, kWaves, [&](int m, int piece, half8_t y) { *(half8_t*)(smem + m * pitch + piece * 16) = y; });

    const int   fr = lane & 15, fc = lane >> 4;
    const char* xf  = smem + min(fr, M - 1) * pitch + fc * 16;
    floatx4     acc = {0.f, 0.f, 0.f, 0.f};
    int         i   = 0;
    for (; i + 2 * R <= count; i += R) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            acc     = StreamOp<T>::mma(ring[k], *(const u32x4*)(xf + step(i + k) * 64), acc);
            ring[k] = load(i + R + k);
        }
    }
    // fewer than 2 R are left; nothing is fetched that is not used, but for the end of a last part
    if (i + R < count) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            acc     = StreamOp<T>::mma(ring[k], *(const u32x4*)(xf + step(i + k) * 64), acc);
            ring[k] = load(i + R + k);
        }
        i += R;
    }
    if (i + R <= count) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            acc = StreamOp<T>::mma(ring[k], *(const u32x4*)(xf + step(i + k) * 64), acc);
        }
    }
    else {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (i + k < count) {
                acc = StreamOp<T>::mma(ring[k], *(const u32x4*)(xf + step(i + k) * 64), acc);
            }
        }
    }
    if constexpr (KP > 1) {
        __syncthreads();
        floatx4* red = (floatx4*)smem;
        if (ph > 0) {
            red[((ph - 1) * CW + cw) * 64 + lane] = acc;
        }
        __syncthreads();
        if (ph > 0) {
            return;
        }
#pragma unroll
        for (int p = 1; p < KP; ++p) {  // fixed order
            acc += red[((p - 1) * CW + cw) * 64 + lane];
        }
    }
    if (fr >= M) {
        return;
    }
    const floatx4 r[1] = {acc};
    epi.template rows<1>(a, item, fr, tile * 16 + fc * 4, r);
}

// dynamic LDS of a launch: the rows and their partial sums, or the k-phases' sums
inline int stream_rows_lds(int M, int steps, int cw, int kp)
{
    return std::max(M * (steps * 64 + kRowsPad) + cw * kp * 4, (kp - 1) * cw * 1024);
}

}  // namespace tmk
