// W4A16 products of up to 16 rows: all rows of a workgroup's slice of k in LDS, the weights streamed past them, scales and zero points applied to sums.
//
// Replaces: LlamaLinear::Forward -> gemm::Gemm::Run for small decode batches (src/turbomind/models/llama/LlamaLinear.cu:140-216), dequant
//           kernels/gemm/transform.h:34-74, gated-SiLU epilogue kernels/gemm/epilogue.h:159-176.
//
// What bounds it: the weight stream, 33 KB a microsecond into a CU, as long as nothing else holds a wave up.  gemm_dec32_kernel (32 rows a workgroup, a barrier for
// every four k-blocks, 13 operations to make eight weights) does with few rows.  Here
//   * the rows come once, ahead of the weights, and behind one barrier (two with more than eight rows) every wave runs through its own k-blocks, two units in flight;
//     more of them in flight, or 16 waves where 8 do, are slower ((4096, 28672) one row, 4 x 4 waves with one, two units 14.8, four 16; a ring of eight 19.7);
//   * v_mfma_f32_16x16x32: a P32 dword is 8 k of one of 32 columns, v_permlane16_swap of the dwords of two neighbouring 16-k steps makes the operands of the
//     unit's two column halves; lane group g = lane / 16 then holds k = 16 (g & 1) + 8 (g >> 1) + 0 .. 7 of 32, and the rows are read in that order;
//   * a weight is never made.  y = sum over groups of 128 k of  s (sum q x) - z s (sum x):  the matrix core contracts the codes as fp16 with the exponent bits that an
//     `and or` gives them, 1024 + q and 64 + q (five operations for eight); sums start at what those bits will add, negated, and a group's sums meet scale and zero
//     point in fp32, two multiply-adds for 32 weights.  Error against 64 bits, (4096, 4096) 8 rows: 2.08e-4 of the results'
//     root mean square, 2.07e-4 of it their own rounding to fp16 (weights rounded to fp16: 2.79e-4); rows that are all positive 2.30e-4 (4.75e-4).
// us, one launch and a tiny one ahead of it, (4096, 28672) gated / (4096, 6144) / (4096, 4096) / (14336, 4096), the last two with the norm behind them, gemm_dec32_kernel | here: one row
// 17.9 | 14.8, 9.1 | 7.3, 10.6 | 9.4, 14.7 | 12.6; 8 rows 17.5 | 15.6, 9.2 | 7.8, 11.1 | 9.9, 15.2 | 14.3; 16 rows 18.5 | 17.8, 9.4 | 8.8, 11.3 | 10.2, 15.9 | 16.1 (not taken).
#include "gemm_decode_common.h"
#include "gemm_rows.h"
#include "tm_kernels.h"
#include <algorithm>

namespace tmk {

// 16 columns x 32 k of a unit on v_mfma_f32_16x16x32_f16: codes as fp16 with their exponent bits still on, 1024 + q (pairs 0, 2 of a dword) and 64 + q (pairs 1, 3);
// what these add to a sum of products is taken off per 128 k with the scale and the zero point, in fp32
__device__ __forceinline__ half8_t w4_rows_codes(uint32_t w, uint32_t m1024, uint32_t m64)
{
    const uint32_t hi = w >> 8;
    const half2_t  p0 = bit_cast<half2_t>((w & 0x000f000fu) | m1024), p1 = bit_cast<half2_t>((w & 0x00f000f0u) | m64);
    const half2_t  p2 = bit_cast<half2_t>((hi & 0x000f000fu) | m1024), p3 = bit_cast<half2_t>((hi & 0x00f000f0u) | m64);
    return half8_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

constexpr int kW4RowsPad = 16;

// CW column groups (32 columns) x KP k-phases of waves, R units in flight a wave.  Grid (column groups / CW, slices of k).  MANY: more than eight rows.  NP > 0: the rows
// are made here, the norm of p.resid's (gemm_rows.h: as many waves a row as there are, NP pieces each; one slice of k): one row, gate / up of Llama-3-8B between a model's
// other kernels 13.5 us, its norm and gemm_dec32_kernel 4.6 + 15.0
template<int CW, int KP, int R, int XB, bool MANY, int NP>
__global__ __launch_bounds__(CW* KP * 64) void gemm_w4_rows_kernel(Dec32Params p, int team)
{
    constexpr int T = CW * KP * 64;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    asm volatile("" ::"s"(p.x), "s"(p.wp), "s"(p.y), "s"(p.partial), "s"(p.ldx), "s"(p.ldy), "s"(p.M), "s"(p.N), "s"(p.KB), "s"(p.ncg), "s"(p.kb_per_split),
                 "s"(p.epilogue));  // (one batch of scalar loads)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wave % CW, ph = wave / CW, fr = lane & 15, fc = lane >> 4;
    const int M = p.M, cg = blockIdx.x * CW + cw, cgc = min(cg, p.ncg - 1);
    const int kb0 = blockIdx.y * p.kb_per_split, nkb = min(p.kb_per_split, p.KB - kb0);
    const int pitch = nkb * 256 + kW4RowsPad;
    float2* const sums = (float2*)(smem + M * pitch);  // [k-block][row]: -(what the codes' exponent bits add), the sum of x
    // rows: 16-byte piece c of k-block kb, row m; 16 neighbouring lanes have a row's k-block
    const int per = nkb * 16, pieces = M * per;
    u32x4     xr[XB];
    auto      x_of = [&](int i) { const int m = i / per; return (const u32x4*)(p.x + (size_t)m * p.ldx + (size_t)kb0 * 128 + (i - m * per) * 8); };
    const NormRows<1, NP ? NP : 1>           norm{p.resid, p.norm_w, p.ss_eps, team};
    typename NormRows<1, NP ? NP : 1>::Regs g;
    if constexpr (NP > 0) {
        norm.load(g, M, nkb * 4, wave, lane, CW * KP);
    }
    else {
#pragma unroll
        for (int r = 0; r < XB; ++r) {
            xr[r] = *x_of(min(tid + r * T, pieces - 1));
        }
    }
    asm volatile("" ::: "memory");
    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)p.wp, 0, (int)((size_t)p.KB * p.ncg * kP32Unit), 0x00020000);
    const int  n    = (nkb - ph + KP - 1) / KP;  // k-blocks of this wave: ph, ph + KP, ...
    u32x4      w[R][2], sz[R][2];
    auto       load = [&](int s, int i) {
        const int uo = ((kb0 + min(ph + i * KP, nkb - 1)) * p.ncg + cgc) * kP32Unit;
        w[s][0]  = __builtin_amdgcn_raw_buffer_load_b128(rs_w, lane * 16, uo, /*nt*/ 2);
        w[s][1]  = __builtin_amdgcn_raw_buffer_load_b128(rs_w, lane * 16 + 1024, uo, /*nt*/ 2);
        sz[s][0] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, 2048 + fc * 16, uo, 0);
        sz[s][1] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, 2112 + fc * 16, uo, 0);
    };
#pragma unroll
    for (int s = 0; s < R; ++s) {
        load(s, min(s, max(n - 1, 0)));
    }
    asm volatile("" ::: "memory");
    // (in: the same for 16 neighbouring lanes)
    auto park = [&](int m, int at, half8_t h, bool in) {
        float c, t;
        if constexpr (!MANY) {
            const float a = ((float)h[0] + (float)h[1]) + ((float)h[4] + (float)h[5]), b = ((float)h[2] + (float)h[3]) + ((float)h[6] + (float)h[7]);
            c = group_sum<16>(-1024.f * a - 64.f * b), t = group_sum<16>(a + b);
        }
        if (in) {
            *(half8_t*)(smem + m * pitch + at * 16) = h;
            if (!MANY && fr == 0) {
                sums[(at >> 4) * M + m] = float2{c, t};
            }
        }
    };
    if constexpr (NP > 0) {
        norm.finish(g, M, nkb * 4, (float*)(sums + M * nkb), wave, lane, CW * KP, [&](int m, int at, half8_t h) { park(m, at, h, true); });
    }
    else {
#pragma unroll
        for (int r = 0; r < XB; ++r) {
            const int i = tid + r * T, m = i / per;
            park(m, i - m * per, bit_cast<half8_t>(xr[r]), i < pieces);
        }
        for (int i = tid + XB * T; i - tid < pieces; i += T) {
            const int m = i / per;
            park(m, i - m * per, bit_cast<half8_t>(*x_of(min(i, pieces - 1))), i < pieces);
        }
        __syncthreads();
    }

    uint32_t m1024 = 0x64006400u, m64 = 0x54005400u;
    asm volatile("" : "+v"(m1024), "+v"(m64));  // magic numbers in VGPRs: one v_and_or_b32 per pair
    const int     row = min(fr, M - 1);
    const char*   xf  = smem + row * pitch + (fc & 1) * 32 + (fc >> 1) * 16;  // (lane group g holds k = 16 (g & 1) + 8 (g >> 1) + 0 .. 7 of 32)
    if constexpr (MANY) {  // the sums: an A operand whose first row is what a code's exponent bits are, negated, and whose second row is ones
        const half2_t c0 = fr == 0 ? half2_t{(half_t)-1024.f, (half_t)-1024.f} : fr == 1 ? half2_t{(half_t)1.f, (half_t)1.f} : half2_t{(half_t)0.f, (half_t)0.f};
        const half2_t c1 = fr == 0 ? half2_t{(half_t)-64.f, (half_t)-64.f} : c0;
        const half8_t ones = {c0[0], c0[1], c1[0], c1[1], c0[0], c0[1], c1[0], c1[1]};
        for (int kb = wave; kb < nkb; kb += CW * KP) {
            floatx4 cs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                cs = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, *(const half8_t*)(xf + kb * 256 + t * 64), cs, 0, 0, 0);
            }
            if (lane < M) {
                sums[kb * M + lane] = float2{cs[0], cs[1]};
            }
        }
        __syncthreads();
    }
    const float2* sf = sums + row;
    floatx4       out[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    float         odd    = 0.f;  // NaN once a sum of x is not finite
    auto          compute = [&](int s, int i) {
        const int    kb = ph + i * KP;
        const float2 cs  = sf[kb * M];
        half8_t      x  = *(const half8_t*)(xf + kb * 256);
        __builtin_amdgcn_sched_barrier(0);  // (asked for ahead of the wait for the weights)
        floatx4 acc[2] = {{cs.x, cs.x, cs.x, cs.x}, {cs.x, cs.x, cs.x, cs.x}};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            x = t == 0 ? x : *(const half8_t*)(xf + kb * 256 + t * 64);
            const auto    d = __builtin_amdgcn_permlane16_swap(w[s][t >> 1][2 * t & 3], w[s][t >> 1][(2 * t & 3) + 1], false, false);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_rows_codes(d[u], m1024, m64), x, acc[u], 0, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const half2_t pr = bit_cast<half2_t>(sz[s][u][e]);  // s, -z s
                out[u][e]        = __builtin_fmaf((float)pr[0], acc[u][e], __builtin_fmaf((float)pr[1], cs.y, out[u][e]));
            }
        }
        odd = __builtin_fmaf(cs.x, 0.f, odd);
    };
    int i = 0;
    for (; i + 2 * R <= n; i += R) {
#pragma unroll
        for (int s = 0; s < R; ++s) {
            compute(s, i + s);
            load(s, i + R + s);
        }
    }
    if (i + R < n) {  // fewer than 2 R are left: the refills of a last part may repeat its last unit
#pragma unroll
        for (int s = 0; s < R; ++s) {
            compute(s, i + s);
            load(s, min(i + R + s, n - 1));
        }
        i += R;
    }
    half4_t stream[2] = {};  // what the results are added to, asked for ahead of the last products: behind them it was two trips to memory in a row
    // (one sequence, 8 layers of Llama-3-8B's shapes: 8.62 -> 8.54 ms for 37 tokens and 16 more)
    if constexpr (NP == 0) {
        if (p.epilogue == 4 && ph == 0) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                stream[u] = *(const half4_t*)(p.y + (size_t)min(fr, M - 1) * p.ldy + cgc * 32 + u * 16 + fc * 4);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < R; ++s) {
        if (i + s < n) {
            compute(s, i + s);
        }
    }
    // A row that holds an infinity: with the codes' exponent bits on every sum of it is infinity less infinity.  Its results are then made from weights.
    if (__ballot(odd != odd) != 0) {
        floatx4 alt[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        for (int j = 0; j < n; ++j) {
            const int   kb   = ph + j * KP;
            const char* unit = (const char*)p.wp + ((size_t)(kb0 + kb) * p.ncg + cgc) * kP32Unit;
            half2_t     s2[2], z2[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const half2_t pr = *(const half2_t*)(unit + 2048 + (u * 16 + fr) * 4);
                s2[u] = half2_t{pr[0], pr[0]}, z2[u] = half2_t{pr[1], pr[1]};
            }
#pragma unroll 1
            for (int t = 0; t < 4; ++t) {
                const half8_t   x = *(const half8_t*)(xf + kb * 256 + t * 64);
                const uint32_t* q = (const uint32_t*)(unit + (t >> 1) * 1024 + lane * 16) + (2 * t & 3);
                const auto      d = __builtin_amdgcn_permlane16_swap(q[0], q[1], false, false);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    alt[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dequant8_p32(d[u], s2[u], z2[u], m1024, m64), x, alt[u], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                out[u][e] = odd != odd ? alt[u][e] : out[u][e];
            }
        }
    }
    if constexpr (KP > 1) {
        __syncthreads();
        floatx4* red = (floatx4*)smem;
        if (ph > 0) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                red[(((ph - 1) * CW + cw) * 2 + u) * 64 + lane] = out[u];
            }
        }
        __syncthreads();
        if (ph > 0) {
            return;
        }
#pragma unroll
        for (int k = 1; k < KP; ++k) {  // fixed order
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                out[u] += red[(((k - 1) * CW + cw) * 2 + u) * 64 + lane];
            }
        }
    }
    if (fr >= M || cg >= p.ncg) {
        return;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int     c = cg * 32 + u * 16 + fc * 4;
        const floatx4 a = out[u];
        if (p.epilogue == 2) {
            store_wt((floatx4*)(p.partial + ((size_t)blockIdx.y * M + fr) * p.N + c), a);
        }
        else if (p.epilogue == 1) {
            const float s0 = silu_f32(a[0]);
            const float s1 = silu_f32(a[2]);
            *(half2_t*)(p.y + (size_t)fr * p.ldy + (c >> 1)) = half2_t{(half_t)(s0 * a[1]), (half_t)(s1 * a[3])};
        }
        else {
            half4_t* y = (half4_t*)(p.y + (size_t)fr * p.ldy + c);
            half4_t  h = {(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3]};
            if (p.epilogue == 4) {  // the residual stream: the product's fp16 rounding, then an addition in fp16
                h = stream[u] + h;
            }
            *y = h;
        }
    }
}

static int w4_rows_lds(int M, int nkb, int cw, int kp)
{
    return std::max(M * (nkb * 256 + kW4RowsPad) + M * nkb * 8 + cw * kp * 4, (kp - 1) * cw * 2048);
}

// ---- which shape, how many slices of k -------------------------------------------------------------------------------------------------
// Waves of a workgroup: column groups of 32 x k-phases.  Of the six shapes that were timed (1 x 4, 4 x 2 too) these four are within 0.9 % of the best of all.
struct W4RowsShape {
    int cw, kp;
};
static const W4RowsShape kW4RowsShapes[] = {{1, 8}, {2, 4}, {2, 8}, {4, 4}};

// A model of the fullest CU's time in microseconds, fitted to which of these shapes and 1, 2, 4 or 8 slices was fastest, with the launch that consumes the slabs, at 140
// sizes (K 2048 ... 14336, N 768 ... 28672, 1, 4, 8, 16 rows; weights from HBM): what it takes is on average 0.8 % slower than the best and 1.16 x as fast as
// gemm_dec32_kernel's choice, slower than that at one size ((4096, 5120) 16 rows, 1.6 %).  Best | this | dec32, us: (2048, 4096) 4 rows 8.7 | 8.7 | 9.9, (4096, 10240) gated one row
// 9.8 | 9.8 | 13.4, (8192, 2048) one row 9.3 | 10.1 | 11.4, (4096, 6144) 8 rows 11.7 | 11.7 | 13.0, (8192, 8192) 16 rows 16.3 | 16.3 | 17.9.
static double w4_rows_cost(int ncg, int nkb, int M, const W4RowsShape& s, int slices)
{
    const int    wgs = (ncg + s.cw - 1) / s.cw * slices, per_cu = (wgs + 255) / 256, waves = s.cw * s.kp;
    const double load  = per_cu * nkb * (s.cw * 2.18 + M * 0.16) / 135;
    const double chain = (nkb + s.kp - 1) / s.kp * 0.134 * (1 + 0.14 * std::max(0.0, per_cu * waves / 4.0 - 1));
    const double rows  = M * nkb * 16 / (waves * 64.0) * 0.2 * per_cu;
    return std::max(load, chain) + 0.11 * std::min(load, chain) + rows + 1.08 * per_cu * waves / 16 + (slices > 1 ? 0.49 + 0.565 * slices * M * ncg * 32 * 4e-6 : 0.0);
}

static int w4_rows_slice(int KB, int slices)
{
    return (KB + slices - 1) / slices;
}

// the cheapest shape that `slices` slices leave room for; -1: none
static int w4_rows_shape(int ncg, int KB, int M, int slices, double* cost)
{
    const int nkb  = w4_rows_slice(KB, slices);
    int       best = -1;
    for (int i = 0; i < 4; ++i) {
        const W4RowsShape& s = kW4RowsShapes[i];
        if (w4_rows_lds(M, nkb, s.cw, s.kp) > 160 * 1024) {
            continue;
        }
        const double c = w4_rows_cost(ncg, nkb, M, s, slices);
        if (best < 0 || c < *cost) {
            best = i, *cost = c;
        }
    }
    return best;
}

bool w4_rows_supported(const LinearWeight& w, int M, int slices)
{
    const int KB = w.K / 128;
    double    cost;
    return M >= 1 && M <= 16 && slices >= 1 && slices <= 16 && (slices == 1 || (KB + w4_rows_slice(KB, slices) - 1) / w4_rows_slice(KB, slices) == slices)
           && (size_t)KB * (w.N / 32) * kP32Unit < ((size_t)1 << 31) && w4_rows_shape(w.N / 32, KB, M, slices, &cost) >= 0;
}

// Products below what was timed stay with gemm_dec32_kernel (whose rows have the bits that they have in forwards of more rows), and so do more than eight rows of a long
// k: (14336, 4096) 16 rows 16.1 here, 15.9 there.  A slice has eight k-blocks at least; a gate / up product's slabs are nobody's to sum but a launch's of its own: in
// a model's step 1 us of the model above's, also against one slice that makes its norm (176 sizes, K 4096 ... 8192, N 3584 ... 14336: on average 0.05 us a layer from the best).  us a
// layer, gemm_dec32_kernel | one slice | four: (8192, 3584) 9 rows 48.8 | 53.6 | 48.0, 8 rows 48.8 | 51.4 | 47.5, (7168, 4096) 9 rows 45.3 | 48.1 | 44.0, (8192, 7168) 4 rows 51.4 | 48.0 | 48.9.
// Wide products whose rows do not fit in LDS whole would have slices only for that, and slabs of all columns: where gemm_dec32_kernel needs none, it keeps them, unless more than a
// quarter of its last round of 128-column workgroups stays empty.  us, there | here in two slices: (5120, 20480) 16 rows 16.9 | 22.5, (6144, 28672) 14 rows 22.5 | 26.7, (8192, 57344)
// 12 rows 54.6 | 59.6, (16384, 20480) 8 rows 42.7 | 47.6, 4 rows 45.1 | 40.8; (8192, 40960), 1.25 rounds, 12 rows 50.8 | 44.9
bool w4_rows_plan(const LinearWeight& w, int M, int* slices)
{
    const int KB = w.K / 128, ncg = w.N / 32;
    if (M > 16 || (M > 8 && w.K > 8192) || w.K < 2048 || w.N < 512) {
        return false;
    }
    double best = 0;
    *slices     = 0;
    for (const int s : {1, 2, 4, 8}) {
        double cost;
        if ((s > 1 && KB / s < 8) || !w4_rows_supported(w, M, s) || w4_rows_shape(ncg, KB, M, s, &cost) < 0) {
            continue;
        }
        cost += s > 1 && w.role == 3 ? 1.0 : 0.0;
        if (*slices == 0 || cost < best) {
            *slices = s, best = cost;
        }
    }
    if (*slices > 1 && M > 4 && w.N >= 16384) {
        int shape, splits;
        dec32_pick_plain(w, M, &shape, &splits, false);
        const int wgs = (w.N + 127) / 128, rounds = (wgs + 255) / 256;
        if (splits == 1 && (rounds == 1 || wgs > 192 * rounds)) {
            return false;
        }
    }
    return *slices > 0;
}

template<int CW, int KP, bool MANY, int NP>
static int launch_w4_rows_shape(const Dec32Params& p, int slices, int team, hipStream_t st)
{
    const auto kernel = gemm_w4_rows_kernel<CW, KP, 2, CW * KP == 16 ? 2 : 4, MANY, NP>;
    const int  lds    = w4_rows_lds(p.M, p.kb_per_split, CW, KP);
    if (const int rc = ensure_dynamic_lds((const void*)kernel, lds)) {
        return rc;
    }
    kernel<<<dim3((p.ncg + CW - 1) / CW, slices), CW * KP * 64, lds, st>>>(p, team);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

static Dec32Params w4_rows_params(const LinearWeight& w, half_t* y, int ldy, int M, int slices)
{
    Dec32Params p{};
    p.wp = w.packed32, p.y = y, p.ldy = ldy;
    p.M = M, p.N = w.N, p.K = w.K, p.KB = w.K / 128, p.ncg = w.N / 32;
    p.kb_per_split = w4_rows_slice(p.KB, slices);
    return p;
}

// as launch_linear_dec32: several slices leave fp32 slabs [slice][M][N] in the workspace; add (one slice): y += x . W, rounded to fp16 first
int launch_w4_rows(const LinearWeight& w, const half_t* x, int ldx, half_t* y, int ldy, int M, bool gated, int slices, float* workspace, int* slabs, hipStream_t st, bool add)
{
    TM_REQUIRE(w.packed32 && w.N % 32 == 0 && w.K % 128 == 0 && ldx % 8 == 0 && w4_rows_supported(w, M, slices) && (slices == 1 || workspace), "W4 product of few rows");
    TM_REQUIRE(!add || (slices == 1 && !gated), "W4 product of few rows: a residual addition");
    Dec32Params p = w4_rows_params(w, y, ldy, M, slices);
    p.x = x, p.ldx = ldx, p.partial = workspace;
    p.epilogue = slices > 1 ? 2 : gated ? 1 : add ? 4 : 0;
    if (slabs) {
        *slabs = slices;
    }
    double cost;
#define TM_W4_ROWS(CW, KP) return M > 8 ? launch_w4_rows_shape<CW, KP, true, 0>(p, slices, 0, st) : launch_w4_rows_shape<CW, KP, false, 0>(p, slices, 0, st)
    switch (w4_rows_shape(p.ncg, p.KB, M, slices, &cost)) {
        case 0: TM_W4_ROWS(1, 8);
        case 1: TM_W4_ROWS(2, 4);
        case 2: TM_W4_ROWS(2, 8);
        default: TM_W4_ROWS(4, 4);
    }
#undef TM_W4_ROWS
}

// `first` in one slice of k, adding to the residual stream, and the norm made by `next`, instead of the plan's slices and a norm launch that sums them: it spares a launch, costs what
// one slice is slower by, and every workgroup of the next product norms all rows once more.  Fitted to 180 pairs in the steps of 19 models (hidden 2048 ... 8192, 1 ... 8
// rows): on average 0.04 us a layer from the better side, 0.9 at most.  us a layer, launch | pair: (4096, 4096) and (4096, 28672) one row 50.1 | 49.1, 8 rows 53.3 | 55.5; (5120, 5120)
// and (5120, 55296) one row 80.5 | 78.8, 4 rows 80.5 | 83.4, 8 rows 85.6 | 92.1; (2048, 2048) and (2048, 16384) 8 rows 37.3 | 36.1; (8192, 2048) and (2048, 4096) one row 35.6 | 34.6, 4 rows 36.8 | 37.9
bool w4_norm_pays(const LinearWeight& first, const LinearWeight& next, int M)
{
    int    slices;
    double one, best;
    return w4_rows_plan(first, M, &slices) && w4_rows_supported(first, M, 1) && w4_rows_shape(first.N / 32, first.K / 128, M, 1, &one) >= 0
           && w4_rows_shape(first.N / 32, first.K / 128, M, slices, &best) >= 0 && one - best + 0.6 * M * (next.K / 8192.0) * (next.N / 28672.0) <= 1.25;
}

bool w4_norm_rows_supported(const LinearWeight& w, int M)
{
    return M <= 8 && w.K % 512 == 0 && w.K <= 8192 && w4_rows_supported(w, M, 1);
}

template<int CW, int KP>
static int launch_w4_norm_rows_shape(const Dec32Params& p, hipStream_t st)
{
    int teams = 1;
    while (teams < p.M) {
        teams *= 2;
    }
    const int team = CW * KP / teams, pieces = (p.K / 512 + team - 1) / team;
    return pieces <= 1 ? launch_w4_rows_shape<CW, KP, false, 1>(p, 1, team, st) :
           pieces <= 2 ? launch_w4_rows_shape<CW, KP, false, 2>(p, 1, team, st) :
           pieces <= 4 ? launch_w4_rows_shape<CW, KP, false, 4>(p, 1, team, st) :
           pieces <= 8 ? launch_w4_rows_shape<CW, KP, false, 8>(p, 1, team, st) :
                         launch_w4_rows_shape<CW, KP, false, 16>(p, 1, team, st);
}

// y = rmsnorm(resid) . W
int launch_w4_norm_rows(const LinearWeight& w, const half_t* resid, const half_t* norm_w, float eps, half_t* y, int ldy, int M, bool gated, hipStream_t st)
{
    TM_REQUIRE(w.packed32 && w4_norm_rows_supported(w, M) && resid && norm_w && y, "W4 product with its norm");
    Dec32Params p = w4_rows_params(w, y, ldy, M, 1);
    p.resid = const_cast<half_t*>(resid), p.norm_w = norm_w, p.ss_eps = eps;
    p.epilogue = gated ? 1 : 0;
    double cost;
    switch (w4_rows_shape(p.ncg, p.KB, M, 1, &cost)) {
        case 0: return launch_w4_norm_rows_shape<1, 8>(p, st);
        case 1: return launch_w4_norm_rows_shape<2, 4>(p, st);
        case 2: return launch_w4_norm_rows_shape<2, 8>(p, st);
        default: return launch_w4_norm_rows_shape<4, 4>(p, st);
    }
}

}  // namespace tmk
