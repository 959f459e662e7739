// FP8 x FP8 linear on the CDNA4 fp8 matrix cores (v_mfma_f32_32x32x16_fp8_fp8): e4m3 weights with 128 x 128 block scales,
// activations quantised on the fly per row and 128-channel group.  Plain and grouped (mixture-of-experts) form.
//
// Replaces: the fp8 path of LlamaLinear::Forward (src/turbomind/models/llama/LlamaLinear.cu:67-127: QuantizeSymm of the
//           input, then the fp8 GEMM with activation scales U and weight scales V), QuantizeSymm itself
//           (kernels/quantization.cu:28-125), the weight format lmdeploy/turbomind/weight_format.py:349-393, and for
//           experts the grouped launch with idxs / offsets (LlamaLinear.cu:95-127, moe_ffn_layer.cc:133-300).
// Arithmetic (oracle: tm_oracle.fp8_quant_rows / fp8_act_linear_acc):
//   activation: absmax over 128 channels (clamped to 1e-8), scale = absmax / 448, q = e4m3_rne_sat(x * (448 / absmax));
//   y[m, n] = sum_g  sx[g, m] * sw[g, n / 128] * sum_{k in g} xq[m, k] * wq[k, n]        (fp32)
//   the inner sum runs on the matrix core (products of two e4m3 values are exact in fp32), one k-group = 8 MFMAs.
//
// MI355X design -- the structure of gemm_decode.hip with the fp8 data path:
//   * the weights go from HBM straight into the MFMA: no dequantisation VALU at all.  Layout "P8": unit (kb, cg) =
//     32 columns x 128 k = 4096 B in A-operand order (lane l: column 32cg + (l & 31), 16-B vector v holds the 16-k steps
//     2v and 2v+1, 8 bytes = k 16j + 8(l >> 5) .. +8) followed by the two fp32 block scales of its even / odd columns
//     (they differ only for the fused w1w3 linear, whose (gate_j, up_j)-interleaved columns come from separately
//     quantised w1 / w3) -- 4224-byte units, one descriptor, k-block-major like P32;
//   * x codes go global -> LDS by LDS-DMA in stages of S k-blocks (128 B per row and k-block: half the fp16 volume), 16-byte
//     units XOR-swizzled by (row >> 1) & 7 on the source address; B fragments are ds_read_b64;
//   * per k-group the partial tile is scaled into the running fp32 accumulators with one fma per element: the lane's
//     row scale sx (a lane owns ONE row of the D tile) times the even / odd column scale;
//   * CG column groups x WK k-phases per workgroup, partial tiles of the k-phases summed through LDS, whole-row stores
//     (fp16, gated SiLU, fp32 split-K slabs) -- as in gemm_decode.hip;
//   * grouped: device-side row segments (`seg`), x rows gathered through `row_idx`, per-expert weight pointers; tiles of 32, 64 or 128
//     rows, only row blocks that hold rows, those of a column tile side by side; many rows an expert: tiles of 256 x 256 on the scaled 16x16x128 instruction
//     (gemm_fp8_tile256_kernel).
#include "fp8_quant.h"
#include "tm_common.h"
#include "tm_kernels.h"
#include <algorithm>
#include <cmath>
#include <stdlib.h>
#include <type_traits>

namespace tmk {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kP8Unit = 4096 + 128;

// ---- activation quantiser ----------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void quant_fp8_rows_kernel(uint8_t* __restrict__ xq, float* __restrict__ sx, const half_t* __restrict__ x,
                                                             int ldx, int M, int K, int ldsx)
{
    quant_fp8_groups(blockIdx.x, xq, sx, x, ldx, M, K, ldsx);
}

int launch_quant_fp8_rows(uint8_t* xq, float* sx, const half_t* x, int ldx, int M, int K, int ldsx, hipStream_t st)
{
    TM_REQUIRE(K % 128 == 0 && ldx % 8 == 0 && ldsx >= M, "fp8 row quantiser: K % 128 == 0, 16-byte aligned rows, ldsx >= M");
    if (M == 0) {
        return 0;
    }
    const int n = M * (K / 128);
    quant_fp8_rows_kernel<<<(n + 15) / 16, 256, 0, st>>>(xq, sx, x, ldx, M, K, ldsx);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---- load-time repack ---------------------------------------------------------------------------------------------
__global__ void repack_p8_kernel(uint32_t* __restrict__ out, const uint8_t* __restrict__ w, const float* __restrict__ block_scales, int K,
                                 int N, int gated)
{
    const size_t idx   = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // one dword
    const int    ncg   = N / 32;
    const size_t total = (size_t)(K / 128) * ncg * (kP8Unit / 4);
    if (idx >= total) {
        return;
    }
    const size_t unit = idx / (kP8Unit / 4);
    const int    d    = (int)(idx % (kP8Unit / 4));
    const int    cg   = (int)(unit % ncg);
    const int    kb   = (int)(unit / ncg);
    if (d >= 1024) {  // [even column scale, odd column scale, padding]
        const int nb = (N + 127) / 128;
        float     s  = 0.f;
        if (d - 1024 < 2) {
            const int n = cg * 32 + (d - 1024);
            const int b = gated ? (n & 1) * (nb / 2) + (n >> 1) / 128 : n / 128;
            s           = block_scales[(size_t)kb * nb + b];
        }
        out[idx] = bit_cast<uint32_t>(s);
        return;
    }
    // dword d: vector v = d >> 8, lane = (d >> 2) & 63, dword-in-vector dd = d & 3 -> j = 2v + (dd >> 1), bytes 4(dd & 1) .. +4
    const int v    = d >> 8;
    const int lane = (d >> 2) & 63;
    const int dd   = d & 3;
    const int j    = 2 * v + (dd >> 1);
    const int n    = cg * 32 + (lane & 31);
    const int k0   = kb * 128 + 16 * j + 8 * (lane >> 5) + 4 * (dd & 1);
    uint32_t  o    = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o |= (uint32_t)w[(size_t)(k0 + e) * N + n] << (8 * e);
    }
    out[idx] = o;
}

size_t p8_bytes(int K, int N)
{
    return (size_t)(K / 128) * (N / 32) * kP8Unit;
}

int launch_repack_p8(void* out, const uint8_t* weight, const float* block_scales, int K, int N, bool gated, hipStream_t st)
{
    const size_t total = p8_bytes(K, N) / 4;
    repack_p8_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>((uint32_t*)out, weight, block_scales, K, N, gated ? 1 : 0);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

// ---- GEMM -----------------------------------------------------------------------------------------------------------
struct Fp8Params {
    const uint8_t* xq;   // [rows][K] e4m3 codes
    const float*   sx;   // [K/128][ldsx] activation scales
    int            ldsx;
    const void*    wp;   // P8 units (plain) ...
    const void* const* groups;  // ... or device [experts] unit pointers (grouped)
    const int*     seg;         // grouped: device [experts + 1] flat-row offsets
    const int*     row_idx;     // grouped: x / sx row of flat row f (nullptr: f)
    int            experts, ct8, one_block;  // grouped: at most 64 experts; column tiles over eight; no expert has more rows than a block
    half_t*        y;
    int            ldy;
    float*         partial;
    int            M, N, K, KB, ncg;  // M: rows (plain) / flat rows in total (grouped, slab stride)
    int            x_rows;            // rows of xq / sx (descriptor bounds)
    int            kb_per_split;
    int            epilogue;  // 0 fp16, 1 gated SiLU fp16, 2 fp32 slab of split blockIdx.y
};

template<int N, class F, int I = 0>
__device__ __forceinline__ void static_for8(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for8<N, F, I + 1>(static_cast<F&&>(f));
    }
}

// Grouped: the tile of this workgroup, e < 0: none.  One-dimensional grid over (expert, column tile, row block) with only the row blocks that hold rows, the
// row blocks of a column tile on consecutive turns of one XCD (workgroups are dealt to the eight in turn): its second-level cache serves a weight unit to
// all of them.  (Empty blocks in between would leave the shader engines they fall on idle: up to 1.9 times slower.)
struct Fp8Tile {
    int e, ct, m0, row0, Mloc;
};
template<int ROWS, int CG>
__device__ __forceinline__ Fp8Tile fp8_tile_of(const Fp8Params& p)
{
    const int turn = blockIdx.x >> 3;
    int       e, n_e = 1, in_e;
    if (p.one_block) {  // decode: no expert has more rows than a block
        e    = turn / p.ct8;
        in_e = turn - e * p.ct8;
    }
    else {
        const int ln = threadIdx.x & 63, nb = ln < p.experts ? (p.seg[ln + 1] - p.seg[ln] + ROWS - 1) / ROWS : 0;
        int       upto = nb;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(upto, d);
            upto += ln >= d ? o : 0;
        }
        e = __popcll(__ballot(upto * p.ct8 <= turn));  // experts whose workgroups come before this turn
        if (e >= p.experts) {
            return {-1, 0, 0, 0, 0};
        }
        n_e  = __builtin_amdgcn_readlane(nb, e);
        in_e = turn - (__builtin_amdgcn_readlane(upto, e) - n_e) * p.ct8;
    }
    const int ct = in_e / n_e * 8 + (blockIdx.x & 7), m0 = in_e % n_e * ROWS, row0 = p.seg[e], Mloc = min(ROWS, p.seg[e + 1] - row0 - m0);
    return {ct * CG >= p.ncg || Mloc <= 0 ? -1 : e, ct, m0, row0, Mloc};
}

template<int MH, int CG, int WK, int S, bool GRP>
__global__ __launch_bounds__(CG* WK * 64) void gemm_fp8_kernel(Fp8Params p)
{
    constexpr int WAVES = CG * WK;
    constexpr int T     = WAVES * 64;
    constexpr int ROWS  = 32 * MH;
    constexpr int KBB   = ROWS * 128;  // LDS bytes of one k-block of codes
    constexpr int STG   = S * KBB;
    constexpr int BPS   = S / WK;
    constexpr int PF    = 2 * BPS;     // ring = two stages
    constexpr int NPC   = S * ROWS / 8;  // 1-KiB DMA pieces (8 rows x 128 B) per stage
    constexpr int DR    = (NPC + WAVES - 1) / WAVES;
    static_assert(S % WK == 0, "tile parameters");
    (void)T;

    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cgl  = wave % CG;
    const int wk   = wave / CG;
    const int l31  = lane & 31;
    const int half = lane >> 5;

    // rows and columns of this workgroup
    int         m0 = blockIdx.z * ROWS, row0 = 0, Mloc = min(ROWS, p.M - m0), ct = blockIdx.x;
    const void* wbase = p.wp;
    if constexpr (GRP) {
        const Fp8Tile tl = fp8_tile_of<ROWS, CG>(p);
        if (tl.e < 0) {
            return;  // whole workgroup, before any barrier
        }
        ct = tl.ct, m0 = tl.m0, row0 = tl.row0, Mloc = tl.Mloc;
        wbase = p.groups[tl.e];
    }
    const int cg  = ct * CG + cgl;
    const int cgc = min(cg, p.ncg - 1);
    const int kb0 = blockIdx.y * p.kb_per_split;
    const int nkb = min(p.kb_per_split, p.KB - kb0);
    const int nst = (nkb + S - 1) / S;

    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)wbase, 0, (int)((size_t)p.KB * p.ncg * kP8Unit), 0x00020000);
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)p.xq, 0, (int)((size_t)p.x_rows * p.K), 0x00020000);
    const auto rs_s = __builtin_amdgcn_make_buffer_rsrc((void*)p.sx, 0, (int)((size_t)p.KB * p.ldsx * 4), 0x00020000);

    // x / sx row of local row m (clamped duplicates past Mloc only feed rows that are never stored)
    auto xrow = [&](int m) {
        const int f = row0 + m0 + min(m, Mloc - 1);
        return (GRP && p.row_idx) ? p.row_idx[f] : f;
    };

    floatx16 acc[MH];
#pragma unroll
    for (int h = 0; h < MH; ++h) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[h][r] = 0.f;
        }
    }
    int sxoff[MH];  // byte offset of this lane's row in one k-group row of sx
#pragma unroll
    for (int h = 0; h < MH; ++h) {
        sxoff[h] = xrow(32 * h + l31) * 4;
    }
    // B fragment of 16-k step j: row (l & 31) [+ 32h], 16-byte unit j XOR-swizzled by (row >> 1) & 7, 8-byte half (l >> 5)
    int coff[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        coff[j] = l31 * 128 + ((j ^ ((l31 >> 1) & 7)) << 4) + half * 8;
    }
    // DMA pieces of a stage: piece pc = r * WAVES + wave = k-block pc / (ROWS / 8), rows 8 (pc % (ROWS / 8)) + (lane >> 3);
    // lane L lands at slot L & 7 of its row and therefore fetches unit (L & 7) ^ ((row >> 1) & 7)
    int            doff[DR];
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
#pragma unroll
    for (int r = 0; r < DR; ++r) {
        const int pc  = min(r * WAVES + wave, NPC - 1);
        const int kbi = pc / (ROWS / 8);
        const int row = (pc % (ROWS / 8)) * 8 + (lane >> 3);
        const int u   = (lane & 7) ^ ((row >> 1) & 7);
        doff[r]       = xrow(row) * p.K + kbi * 128 + u * 16;
    }
    const int my_dr = NPC % WAVES == 0 ? DR : (wave < NPC - (DR - 1) * WAVES ? DR : DR - 1);  // wave-uniform
#define F8_DMA_X(t, buf)                                                                                          \
    _Pragma("unroll") for (int r = 0; r < DR; ++r)                                                                \
    {                                                                                                             \
        if (r < my_dr) {                                                                                          \
            unsigned       keep_;                                                                                 \
            const unsigned dst_ = lds0 + (buf)*STG + (r * WAVES + wave) * 1024;                                   \
            const int      so_  = (kb0 + (t)*S) * 128;                                                            \
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"                                       \
                         "buffer_load_dwordx4 %1, %2, %4 offen lds\n\ts_mov_b32 m0, %0"                               \
                         : "=&s"(keep_)                                                                           \
                         : "v"(doff[r]), "s"(rs_x), "s"(dst_), "s"(so_)                                           \
                         : "memory");                                                                             \
        }                                                                                                         \
    }

    u32x4 ring[PF][4];
    u32x2 swr[PF];      // (even, odd) column scale of the unit
    float sxr[PF][MH];  // this lane's row scale(s) for the k-group
    const int vw = lane * 16;
#define F8_LOAD_W(slot, b)                                                                                        \
    {                                                                                                             \
        const int kbx_ = kb0 + min((b), nkb - 1);                                                                 \
        const int uo_  = (kbx_ * p.ncg + cgc) * kP8Unit;                                                          \
        _Pragma("unroll") for (int v = 0; v < 4; ++v)                                                             \
        {                                                                                                         \
            ring[slot][v] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, vw + v * 1024, uo_, /*nt*/ 2);            \
        }                                                                                                         \
        swr[slot] = __builtin_amdgcn_raw_buffer_load_b64(rs_w, 4096, uo_, 0);                                     \
        _Pragma("unroll") for (int h = 0; h < MH; ++h)                                                            \
        {                                                                                                         \
            sxr[slot][h] = bit_cast<float>(__builtin_amdgcn_raw_buffer_load_b32(rs_s, sxoff[h], kbx_ * p.ldsx * 4, 0)); \
        }                                                                                                         \
    }
    constexpr int LPB = 4 + 1 + MH;  // loads per ring slot

    if (nst > 0) {
        F8_DMA_X(0, 0);
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            F8_LOAD_W(q, (q / BPS) * S + wk + (q % BPS) * WK);
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LPB * PF) : "memory");  // everything older than the ring: x(0)
        __syncthreads();

        auto stage = [&](auto U, const int t) __attribute__((always_inline)) {
            constexpr int u   = decltype(U)::value;
            const int     buf = u & 1;
            // make hipcc wait for this stage's ring slots HERE, then start the (invisible to its waitcnt pass) DMA of x(t+1)
#pragma unroll
            for (int i = 0; i < BPS; ++i) {
                asm volatile("" ::"v"(ring[u * BPS + i][0]), "v"(ring[u * BPS + i][3]), "v"(swr[u * BPS + i]), "v"(sxr[u * BPS + i][MH - 1]));
            }
            if (t + 1 < nst) {  // uniform; see gemm_dec32_kernel: a DMA behind the last stage could land on the reduction image
                F8_DMA_X(t + 1, buf ^ 1);
            }
#pragma unroll
            for (int i = 0; i < BPS; ++i) {
                const int  slot = u * BPS + i;
                const int  kbi  = wk + i * WK;
                const bool live = t * S + kbi < nkb;
                const char* xb  = smem + buf * STG + kbi * KBB;
                floatx16    tt[MH];
                static_for8<8>([&](auto J) {
                    constexpr int j  = decltype(J)::value;
                    const u32x4   wv = ring[slot][j >> 1];
                    const long    a  = bit_cast<long>(u32x2{wv[(j & 1) * 2], wv[(j & 1) * 2 + 1]});
#pragma unroll
                    for (int h = 0; h < MH; ++h) {
                        const long b = *(const long*)(xb + h * 4096 + coff[j]);
                        if constexpr (j == 0) {
                            tt[h] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a, b, floatx16{}, 0, 0, 0);
                        }
                        else {
                            tt[h] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a, b, tt[h], 0, 0, 0);
                        }
                    }
                });
                if (live) {  // wave-uniform; a k-block past the slice contributes nothing (its operands are clamped re-reads)
                    const float s_even = bit_cast<float>(swr[slot][0]);
                    const float s_odd  = bit_cast<float>(swr[slot][1]);
#pragma unroll
                    for (int h = 0; h < MH; ++h) {
                        const float se = sxr[slot][h] * s_even, so = sxr[slot][h] * s_odd;
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            acc[h][r] = __builtin_fmaf(tt[h][r], (r & 1) ? so : se, acc[h][r]);
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < BPS; ++i) {
                F8_LOAD_W(u * BPS + i, (t + 2) * S + wk + i * WK);
            }
            asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LPB * BPS) : "memory");  // my DMA pieces of x(t+1) have landed
            __syncthreads();
        };
        int t0 = 0;
        for (; t0 + 2 <= nst; t0 += 2) {
            static_for8<2>([&](auto U) { stage(U, t0 + decltype(U)::value); });
        }
        if (t0 < nst) {
            stage(std::integral_constant<int, 0>{}, t0);
        }
    }
#undef F8_DMA_X
#undef F8_LOAD_W

    // ---- k-phase reduction + whole-row stores (as gemm_decode.hip) ------------------------------------------------------
    {
        constexpr int C4 = CG * 8;
        floatx4*      red = (floatx4*)smem;
#pragma unroll
        for (int h = 0; h < MH; ++h) {
            const int m = 32 * h + l31;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int c4 = cgl * 8 + 2 * g4 + half;
                red[(wk * ROWS + m) * C4 + (c4 ^ (m & 7))] =
                    floatx4{acc[h][4 * g4], acc[h][4 * g4 + 1], acc[h][4 * g4 + 2], acc[h][4 * g4 + 3]};
            }
        }
        __syncthreads();
        constexpr int NE    = ROWS * C4;
        const int     ncol0 = ct * CG * 32;
#pragma unroll
        for (int e0 = 0; e0 < NE; e0 += T) {
            const int e = e0 + tid;
            if (NE % T != 0 && e >= NE) {
                break;
            }
            const int m  = e / C4;
            const int c4 = e % C4;
            floatx4   a  = red[m * C4 + (c4 ^ (m & 7))];
#pragma unroll
            for (int k = 1; k < WK; ++k) {
                a += red[(k * ROWS + m) * C4 + (c4 ^ (m & 7))];
            }
            const int n = ncol0 + c4 * 4;
            if (m >= Mloc || n >= p.N) {
                continue;
            }
            const size_t mg = (size_t)row0 + m0 + m;  // (flat) output row
            if (p.epilogue == 2) {
                *(floatx4*)(p.partial + ((size_t)blockIdx.y * p.M + mg) * p.N + n) = a;
            }
            else if (p.epilogue == 1) {
                const float s0 = silu_f32(a[0]);
                const float s1 = silu_f32(a[2]);
                half2_t     o  = {(half_t)(s0 * a[1]), (half_t)(s1 * a[3])};
                *(half2_t*)(p.y + mg * p.ldy + (n >> 1)) = o;
            }
            else {
                half4_t o = {(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3]};
                *(half4_t*)(p.y + mg * p.ldy + n) = o;
            }
        }
    }
}

// ---- many rows: 256 x 256 tiles ---------------------------------------------------------------------------------------------------------------------
// The kernel above gives a weight unit to 128 rows at most and runs at the 16-bit instructions' rate; here a k-block of 256 rows x 256 columns meets in LDS
// (66 KB, two stages: the next one is on its way by LDS-DMA during this one's products), and one v_mfma_f32_16x16x128_f8f6f4 is a whole scale block of
// 16 x 16 outputs at twice that rate.  Eight waves of 64 rows x 128 columns: the fp32 accumulators are vector operands of the scaling, which the
// accumulation registers cannot be, so 128 a lane is the most there are.  Products and scaling take turns one by one (behind each other in groups of four
// and sixteen the two hardly overlapped: matrix cores 36 % busy, now 46 %); the rest is the barrier a k-block and LDS (192 KB read, 66 KB written a k-block).
// Expert block 4096 x 14336, 8 experts, top 2, 4000 tokens: 3104 -> 1765 us, 8000: 6170 -> 2985 (1.89 PFLOP/s with routing and quantisation).
// Lane l of an A operand holds column l & 15 and 32 of the 128 channels, those of a P8 unit's vectors 2 (l >> 5), 2 (l >> 5) + 1 and half (l >> 4) & 1; B
// takes the same channels of row l & 15, so the order the instruction gives them in does not matter.
typedef int intx8 __attribute__((ext_vector_type(8)));

// LDS-DMA of 16 or 4 bytes a lane to consecutive places from dst on
__device__ __forceinline__ void fp8_dma16(const __amdgpu_buffer_rsrc_t rs, int off, int soff, unsigned dst)
{
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(off), "s"(dst), "s"(rs), "s"(soff)
                 : "memory");
}
__device__ __forceinline__ void fp8_dma4(const __amdgpu_buffer_rsrc_t rs, int off, int soff, unsigned dst)
{
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                 "buffer_load_dword %1, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(off), "s"(dst), "s"(rs), "s"(soff)
                 : "memory");
}

constexpr int kFp8TileX     = 256 * 128;                       // codes of 256 rows
constexpr int kFp8TileW     = 8 * kP8Unit + 128;               // eight units
constexpr int kFp8TileStage = kFp8TileX + kFp8TileW + 256 * 4;  // and the rows' scales
constexpr int kFp8TileOut   = 64 * 288;                        // a wave's results on their way out, 64 rows
constexpr int kFp8TileLds   = 8 * kFp8TileOut > 2 * kFp8TileStage ? 8 * kFp8TileOut : 2 * kFp8TileStage;

__global__ __launch_bounds__(512) void gemm_fp8_tile256_kernel(Fp8Params p)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int     tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Fp8Tile tl = fp8_tile_of<256, 8>(p);
    if (tl.e < 0) {
        return;  // whole workgroup, before any barrier
    }
    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)p.groups[tl.e], 0, (int)((size_t)p.KB * p.ncg * kP8Unit), 0x00020000);
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)p.xq, 0, (int)((size_t)p.x_rows * p.K), 0x00020000);
    const auto rs_s = __builtin_amdgcn_make_buffer_rsrc((void*)p.sx, 0, (int)((size_t)p.KB * p.ldsx * 4), 0x00020000);
    auto       xrow = [&](int m) {  // (clamped duplicates past Mloc only feed rows that are never stored)
        const int f = tl.row0 + tl.m0 + min(m, tl.Mloc - 1);
        return p.row_idx ? p.row_idx[f] : f;
    };
    // DMA of a k-block: wave w takes 32 rows of x (pieces of 8 rows x 128 bytes; 16-byte unit u of row r at u ^ ((r >> 1) & 7)), weight unit w (its last piece, 256
    // bytes, runs into the next unit's head: the same bytes that land there anyway, or the room behind the eighth) and the scales of 64 rows (two waves the same)
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);
    int            xoff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = (4 * wave + r) * 8 + (lane >> 3);
        xoff[r]       = xrow(row) * p.K + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
    const int soff = xrow((wave & 3) * 64 + lane) * 4, w0 = (tl.ct * 8 + wave) * kP8Unit, wstep = p.ncg * kP8Unit;
    auto      fetch = [&](int kb, int buf, int n) {  // piece n = 0 .. 9 of this wave
        const unsigned dst = lds0 + buf * kFp8TileStage;
        if (n < 4) {
            fp8_dma16(rs_x, xoff[n], kb * 128, dst + (4 * wave + n) * 1024);
        }
        else if (n < 8) {
            fp8_dma16(rs_w, lane * 16 + (n - 4) * 1024, w0 + kb * wstep, dst + kFp8TileX + wave * kP8Unit + (n - 4) * 1024);
        }
        else if (n == 8) {
            fp8_dma4(rs_w, lane * 4 + 4096, w0 + kb * wstep, dst + kFp8TileX + wave * kP8Unit + 4096);
        }
        else {
            fp8_dma4(rs_s, soff, kb * p.ldsx * 4, dst + kFp8TileX + kFp8TileW + (wave & 3) * 256);
        }
    };
    const int c = lane & 15, q = lane >> 4, wr = wave >> 1, wc = wave & 1;
    int       xf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        xf[j] = (wr * 64 + c) * 128 + (((4 * (q >> 1) + j) ^ (c >> 1)) << 4) + (q & 1) * 8;
    }
    const int wf = kFp8TileX + wc * 4 * kP8Unit + (q >> 1) * 2048 + (c + 32 * (q & 1)) * 16;
    const int sf = kFp8TileX + kFp8TileW + (wr * 64 + c) * 4;

    floatx4 acc[4][2][4];  // unit, column half, row tile
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                acc[u][h][t] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
#pragma unroll
    for (int n = 0; n < 10; ++n) {
        fetch(0, 0, n);
    }
    for (int kb = 0; kb < p.KB; ++kb) {
        // this wave's pieces of the k-block have landed and its reads of the other stage are over; then everybody's
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int   nxt = min(kb + 1, p.KB - 1), nbuf = (kb + 1) & 1;  // (behind the last block: again, into the stage that nobody reads)
        const char* st  = smem + (kb & 1) * kFp8TileStage;
        intx8       a[2], b[4];
        auto        read_a = [&](int i) {  // column tile i = 0 .. 7
            const u32x4 a0 = *(const u32x4*)(st + wf + (i >> 1) * kP8Unit + (i & 1) * 256);
            const u32x4 a1 = *(const u32x4*)(st + wf + (i >> 1) * kP8Unit + (i & 1) * 256 + 1024);
            a[i & 1]       = intx8{(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
        };
        read_a(0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int off = (int)(st - smem) + xf[j] + t * 2048;
                asm("" : "+v"(off));  // (two tiles' rows in one instruction, as the compiler would have them, meet in the same banks)
                const u32x2 v   = *(const u32x2*)(smem + off);
                b[t][2 * j]     = (int)v[0];
                b[t][2 * j + 1] = (int)v[1];
            }
        }
        float sx[4], sw[4][2];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            sx[t]       = *(const float*)(st + sf + t * 64);
            const u32x2 v = *(const u32x2*)(st + kFp8TileX + (wc * 4 + t) * kP8Unit + 4096);
            sw[t][0] = bit_cast<float>(v[0]), sw[t][1] = bit_cast<float>(v[1]);
        }
        floatx4 tt[2][4];
        auto    scale = [&](int i, int t) {  // the results of column tile i, row tile t join the sums
            const float se = sx[t] * sw[i >> 1][0], so = sx[t] * sw[i >> 1][1];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[i >> 1][i & 1][t][r] = __builtin_fmaf(tt[i & 1][t][r], (r & 1) ? so : se, acc[i >> 1][i & 1][t][r]);
            }
        };
        // A product of column tile i, the scaling of one of tile i - 1 under it, in turn: 32 cycles of the matrix core, 24 of the vector unit; the next tile's
        // operand and, first, the pieces of the next k-block with them
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i < 7) {
                read_a(i + 1);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {  // (formats 0: e4m3; both scales 0: the form without scales)
                tt[i & 1][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i & 1], b[t], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                if (i > 0) {
                    scale(i - 1, t);
                }
                if (4 * i + t < 10) {
                    fetch(nxt, nbuf, 4 * i + t);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            scale(7, t);
        }
    }
    // A lane's results are four columns each of its rows; through the wave's own LDS they leave as whole runs of a row
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave is through with the stages
    asm volatile("" ::: "memory");
    char* const out   = smem + wave * kFp8TileOut;
    const bool  gated = p.epilogue == 1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const floatx4 a   = acc[u][h][t];
                char* const   row = out + (t * 16 + c) * 288;
                if (gated) {
                    const float s0 = silu_f32(a[0]);
                    const float s1 = silu_f32(a[2]);
                    *(half2_t*)(row + u * 32 + h * 16 + q * 4) = half2_t{(half_t)(s0 * a[1]), (half_t)(s1 * a[3])};
                }
                else {
                    *(half4_t*)(row + u * 64 + h * 32 + q * 8) = half4_t{(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3]};
                }
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
    const int n0 = (tl.ct * 256 + wc * 128) >> (gated ? 1 : 0), N = p.N >> (gated ? 1 : 0), run = gated ? 8 : 16;  // 16-byte runs of a row
    const int rr = gated ? lane >> 3 : lane >> 4, rc = lane & (run - 1), n = n0 + rc * 8;
#pragma unroll 4
    for (int r = rr; r < 64; r += 64 / run) {
        const int m = wr * 64 + r;
        if (m < tl.Mloc && n < N) {
            *(half8_t*)(p.y + (size_t)(tl.row0 + tl.m0 + m) * p.ldy + n) = *(const half8_t*)(out + r * 288 + rc * 16);
        }
    }
}

template<int MH, int CG, int WK, bool GRP>
static int launch_fp8_one(const Fp8Params& p, dim3 grid, hipStream_t st)
{
    constexpr int S     = 4;
    constexpr int stage = 2 * S * 32 * MH * 128;
    constexpr int red   = WK * 32 * MH * CG * 128;
    constexpr int lds   = stage > red ? stage : red;
    if (const int rc = ensure_dynamic_lds((const void*)gemm_fp8_kernel<MH, CG, WK, S, GRP>, lds)) {
        return rc;
    }
    gemm_fp8_kernel<MH, CG, WK, S, GRP><<<grid, CG * WK * 64, lds, st>>>(p);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

bool fp8_mfma_supported(const LinearWeight& w)
{
    const char* ev = getenv("TM_FP8_MFMA");  // 0: keep e4m3 weights on the weight-only (dequantise to f16) path
    const int   on = ev ? atoi(ev) : 1;
    return on && w.type == 2 && w.packed8 != nullptr && w.N % 32 == 0 && w.K % 128 == 0;
}

size_t fp8_act_workspace_bytes(int rows, int K)
{
    // codes [rows][K] + scales [K/128][rows rounded up to 4]
    return (size_t)rows * K + (size_t)(K / 128) * ((rows + 3) / 4 * 4) * sizeof(float) + 256;
}

static int fp8_splits(int col_wgs, int KB, int want)
{
    if (want > 0) {
        return want;
    }
    int splits = 1;
    for (int s = 2; s <= 16; ++s) {
        int per = (KB + s - 1) / s;
        per     = (per + 3) / 4 * 4;
        if ((KB + per - 1) / per == s && col_wgs * s <= 256 && per >= 4) {
            splits = s;
        }
    }
    return splits;
}

// y = fp8 x fp8 linear of PRE-QUANTISED activations (xq, sx from launch_quant_fp8_rows).  splits = 0: heuristic.
int launch_linear_fp8(const LinearWeight& w, const uint8_t* xq, const float* sx, int ldsx, half_t* y, int ldy, int M, bool gated_silu,
                      int splits, float* workspace, int* slabs_out, hipStream_t st)
{
    // (the TM_FP8_MFMA switch is evaluated where the path is CHOSEN -- fp8_mfma_supported at load / dispatch time --, not per launch)
    TM_REQUIRE(w.type == 2 && w.packed8 != nullptr && w.N % 32 == 0 && w.K % 128 == 0, "fp8 MFMA linear: e4m3 weights in P8 layout, N % 32 == 0");
    if (slabs_out) {
        *slabs_out = 1;
    }
    if (M == 0) {
        return 0;
    }
    Fp8Params p{};
    p.xq = xq, p.sx = sx, p.ldsx = ldsx, p.wp = w.packed8, p.y = y, p.ldy = ldy, p.partial = workspace;
    p.M = M, p.N = w.N, p.K = w.K, p.KB = w.K / 128, p.ncg = w.N / 32, p.x_rows = M;
    const int rows_per = M <= 32 ? 32 : 64;
    const int zb       = (M + rows_per - 1) / rows_per;
    const int col_wgs  = (p.ncg + 3) / 4 * zb;
    int       sp       = workspace ? fp8_splits(col_wgs, p.KB, splits) : 1;
    int       per      = (p.KB + sp - 1) / sp;
    per                = std::min((per + 3) / 4 * 4, p.KB);
    sp                 = (p.KB + per - 1) / per;
    p.kb_per_split     = per;
    p.epilogue         = sp > 1 ? 2 : (gated_silu ? 1 : 0);
    dim3 grid((p.ncg + 3) / 4, sp, zb);
    const int rc = M <= 32 ? launch_fp8_one<1, 4, 4, false>(p, grid, st) : launch_fp8_one<2, 4, 2, false>(p, grid, st);
    if (rc) {
        return rc;
    }
    if (slabs_out) {
        *slabs_out = sp;
    }
    return 0;
}

// grouped: flat rows seg[e] .. seg[e+1] of expert e, x / sx row of flat row f = row_idx ? row_idx[f] : f; m_hint = expected rows
// per expert (tile height), m_cap = upper bound
int launch_linear_fp8_grouped(const LinearWeight& proto, const void* d_groups, int E, const uint8_t* xq, const float* sx, int ldsx,
                              int x_rows, half_t* y, int ldy, int m_cap, int total_rows, int m_hint, bool gated_silu, const int* seg,
                              const int* row_idx, hipStream_t st)
{
    TM_REQUIRE(E <= 64 && proto.type == 2 && proto.N % 32 == 0 && proto.K % 128 == 0, "grouped fp8 MFMA linear: e4m3 experts, N % 32 == 0");
    if (m_cap == 0 || E == 0) {
        return 0;
    }
    Fp8Params p{};
    p.xq = xq, p.sx = sx, p.ldsx = ldsx, p.groups = (const void* const*)d_groups, p.seg = seg, p.row_idx = row_idx;
    p.y = y, p.ldy = ldy, p.M = m_cap, p.N = proto.N, p.K = proto.K, p.KB = proto.K / 128, p.ncg = proto.N / 32, p.x_rows = x_rows;
    p.kb_per_split = p.KB;
    p.epilogue     = gated_silu ? 1 : 0;
    const int want = std::min(m_cap, std::max(1, 2 * m_hint));
    int       tv[4];
    const bool measured = gen_table_get(kGenGrouped + 2, 0, proto.K, proto.N, dec32_m_bucket(m_cap), tv);  // tm_engine_tune_gemm
    // Rows of a tile, by the expected rows of an expert: a weight unit costs a workgroup the same for 128 rows as for 32, but rows that are not there cost as
    // much as those that are.  Mixtral-sized experts (4096 x 14336, 8, top 2), us a layer with 32 / 64 / 128 rows: 16 expected 259 / 302 / 427, 48: 398 / 326
    // / 428, 64: 469 / 478 / 430, 100: 612 / 522 / 447, 128: 735 / 641 / 697, 256: 1304 / 1088 / 1013, 1024: 4915 / 3857 / 3264 (0.88 PFLOP/s; 64 rows with
    // the row blocks of a column tile far apart: 4868).  128 / 256 rows (the kernel of 256 x 256 tiles): 80 expected 489 / 544, 100: 452 / 499, 110: 561 / 489, 160: 773 / 506,
    // 1000: 3104 / 1765; 32 experts of 4096 x 1536: 80: 283 / 293, 150: 509 / 351.  What the larger tile saves is a second round of the smaller ones: while those (of
    // the rows that an expert has with the spread of a random choice) are about a round, the chip is emptier with a quarter as many.  One product, 128 rows and
    // the difference of 256: (1024, 1024) 4 experts, 500 rows 128 tiles 48 us + 6; (14336, 4096) 8 experts, 110 rows 256 tiles + 62 of 439, 160 rows 512 tiles
    // - 23 of 770; (4096, 4096) 4 experts, 160 rows 256 tiles + 14 of 132, 250 rows 384 tiles - 15 of 194; (6144, 2048) 2 experts, 1000 rows 288 tiles + 24 of 132
    // (2000: - 66 of 299); (3584, 1024) 8 experts, 300 rows 192 tiles + 17 of 139, 500 rows 320 tiles - 9 of 208
    const bool wide = ldy % 8 == 0 && (uintptr_t)y % 16 == 0;  // (rows leave in 16-byte runs)
    const int  t128 = E * (int)std::ceil((m_hint + std::sqrt((double)m_hint)) / 128.0) * ((p.ncg + 3) / 4);
    int        rows = measured ? tv[0] : want <= 32 ? 32 : m_hint < 56 ? 64 : m_hint < 105 || t128 <= 288 ? 128 : 256;
    rows            = rows == 256 && !wide ? 128 : rows;
    p.experts      = E;
    p.ct8          = ((p.ncg + 3) / 4 + 7) / 8;
    p.one_block    = m_cap <= rows;
    if (rows == 256) {
        p.ct8 = ((p.ncg + 7) / 8 + 7) / 8;
        if (const int rc = ensure_dynamic_lds((const void*)gemm_fp8_tile256_kernel, kFp8TileLds)) {
            return rc;
        }
        gemm_fp8_tile256_kernel<<<p.ct8 * 8 * (p.one_block ? E : std::min(E * ((m_cap + rows - 1) / rows), total_rows / rows + E)), 512, kFp8TileLds, st>>>(p);
        TM_HIP_CHECK(hipGetLastError());
        return 0;
    }
    const dim3 grid(p.ct8 * 8 * (p.one_block ? E : std::min(E * ((m_cap + rows - 1) / rows), total_rows / rows + E)));
    return rows == 32 ? launch_fp8_one<1, 4, 4, true>(p, grid, st) :
           rows == 64 ? launch_fp8_one<2, 4, 2, true>(p, grid, st) : launch_fp8_one<4, 4, 2, true>(p, grid, st);
}

}  // namespace tmk
