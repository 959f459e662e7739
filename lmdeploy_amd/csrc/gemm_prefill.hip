// W4A16 prefill GEMM for gfx950: 256 x 256 output tiles, each u4 weight dequantised ONCE per workgroup tile, in registers.
//
// Replaces: the large-M end of gemm::Gemm::Run (src/turbomind/kernels/gemm/gemm.cu:257-344, tile family
//           kernels/gemm/kernel/sm80_16816_4.cu:18-61), dequant kernels/gemm/transform.h:34-74, gated-SiLU epilogue
//           kernels/gemm/epilogue.h:159-176.  Same operand as every other W4A16 kernel here: w = h(fma(h(q), s, h(-z*s))).
//
// What bounds it: power.  A matrix kernel on real data holds the clock near 1.6 GHz, so what counts is the energy of a multiply-add and of
// everything beside it:
//   * v_mfma_f32_16x16x32 instead of 32x32x16: from registers alone, u4 grid x normal rows, 2.05 against 1.73 PFLOP/s (2.40 and 2.43 on zeros).  It wants
//     16 columns x 32 k where a P32 dword is 8 k of one of 32 columns: v_permlane16_swap of the dwords of two neighbouring 16-k steps makes the
//     operands of the unit's two column halves; lane group g = lane / 16 then holds k = 16 (g & 1) + 8 (g >> 1) + 0 .. 7 of the 32, and the rows are read in that order;
//   * 4 waves side by side, 256 rows x 64 columns each: no weight is dequantised twice in a workgroup (13 packed operations for 16 MFMAs), 256
//     accumulator registers, one wave per SIMD;
//   * rows AND raw weight units come by LDS-DMA (a unit goes to the wave that owns its columns): one counted queue, nothing staged in registers.
// A step is 32 k: 64 MFMAs a wave, 16 row fragments read a whole step ahead, the next step's four weight fragments dequantised three or four operations per four
// MFMAs; four row stages of 16 KB, two slots of weight units; one barrier a step.
// 8192 rows, MI355X, one launch after another: (K, N) = (4096, 28672) gated 1508 us = 1.28 PFLOP/s (between a model's other kernels 1530 - 1670), (14336, 4096) 700 = 1.37, (4096, 6144) 319, (4096, 4096) 218; tiles of 128 x 512 on
// 32x32x16 1638, 779, 366 and 247 on the same box; 256 x 256 tiles that dequantised through LDS for 32x32x16 were no faster than those.
// fp16 results leave in 16-byte pieces (eight and four bytes a lane: (2048, 16384) gated, 4096 rows 272 us against 258).
// grid = (ceil(N / 256), splits, ceil(M / 256)); epilogue straight from the accumulators (fp16, gated SiLU, fp32 slabs).
#include "gemm_decode_common.h"

namespace tmk {

template<int BYTES>  // a lane
__device__ __forceinline__ void pre256_dma(__amdgpu_buffer_rsrc_t rs, int voff, int soff, unsigned lds)
{
    unsigned keep;
    if constexpr (BYTES == 16) {
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "buffer_load_dwordx4 %1, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep)
                     : "v"(voff), "s"(lds), "s"(rs), "s"(soff)
                     : "memory");
    }
    else {
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "buffer_load_dword %1, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep)
                     : "v"(voff), "s"(lds), "s"(rs), "s"(soff)
                     : "memory");
    }
}

// asm: the accumulators are accumulation registers and nothing else.  The operands are VALU results of the step before (the hardware wants two
// operations between, the step's wait and barrier stand there) or LDS reads, which the compiler waits for
__device__ __forceinline__ void pre256_mma(floatx4& c, const u32x4& a, const u32x4& b)
{
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// one 32-bit part (two weights) of dequant8_p32
template<int P>
__device__ __forceinline__ uint32_t pre256_dequant2(uint32_t w, half2_t s2, half2_t z2, uint32_t m1024, uint32_t m64)
{
    const uint32_t v = P >= 2 ? w >> 8 : w;
    const half2_t  q = P & 1 ? bit_cast<half2_t>((v & 0x00f000f0u) | m64) - half2_t{(half_t)64.0f, (half_t)64.0f} :
                               bit_cast<half2_t>((v & 0x000f000fu) | m1024) - half2_t{(half_t)1024.0f, (half_t)1024.0f};
    return bit_cast<uint32_t>(h2_fma(q, s2, z2));
}

// r[j] of lane group g (16 lanes) <-> r[g] of lane group j
__device__ __forceinline__ void pre256_transpose(uint32_t (&r)[4])
{
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const auto s = __builtin_amdgcn_permlane32_swap(r[j], r[j + 2], false, false);
        r[j] = s[0], r[j + 2] = s[1];
    }
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
        const auto s = __builtin_amdgcn_permlane16_swap(r[j], r[j + 1], false, false);
        r[j] = s[0], r[j + 1] = s[1];
    }
}

constexpr int kPre256X      = 256 * 64;            // bytes of one row stage: 256 rows x 32 k
constexpr int kPre256W      = 2 * 2048 + 256;      // ... of a wave's two units of a k-block: codes, then the scales of both
constexpr int kPre256Lds    = 4 * kPre256X + 2 * 4 * kPre256W;
constexpr int kPre256XPiece = 4, kPre256WPiece = 5;  // DMA operations of a wave: per row stage, per k-block of weights

__global__ __launch_bounds__(256, 1) void gemm_pre256_kernel(Dec32Params p)
{
    constexpr int BM = 256;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int tid  = threadIdx.x;
    const int wgid = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (p.dbg && tid == 0) {
        p.dbg[wgid * 8 + 0] = __builtin_amdgcn_s_memrealtime();
    }
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fc = lane >> 4;

    // XCD-aware order: workgroup i runs on XCD i % 8; each XCD gets a contiguous eighth of the tiles, walked in bands of four row tiles, so that what its
    // CUs hold at a time shares operands in its L2
    int tn = blockIdx.x, tm = blockIdx.z;
    if (gridDim.y == 1) {
        const int tns = gridDim.x, tms = gridDim.z, total = tns * tms;
        const int i = tm * tns + tn, xcd = i & 7, lin = xcd * (total >> 3) + min(xcd, total & 7) + (i >> 3);
        const int band = lin / (4 * tns), in = lin - band * 4 * tns, h = min(4, tms - band * 4);
        tm = band * 4 + in % h, tn = in / h;
    }
    const int kb0  = blockIdx.y * p.kb_per_split;
    const int nkb  = min(p.kb_per_split, p.KB - kb0);
    const int m0   = tm * BM;
    const int Mloc = min(BM, p.M - m0);

    const auto rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)p.wp, 0, (int)((size_t)p.KB * p.ncg * kP32Unit), 0x00020000);
    const auto rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)(p.x + (size_t)m0 * p.ldx), 0,
                                                        (int)(((size_t)(Mloc - 1) * p.ldx + p.K) * 2), 0x00020000);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);

    // rows: piece (1 KB) 4 wave + r of a stage is rows 16 (4 wave + r) .. + 15; 16-byte piece c of row r at c ^ ((r >> 1) & 3), the swizzle is on the source
    int xoff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * (4 * wave + r) + (lane >> 2);
        xoff[r]       = min(row, Mloc - 1) * p.ldx * 2 + ((lane & 3) ^ ((row >> 1) & 3)) * 16;
    }
    auto dma_x = [&](int kb, int q, int r) {
        pre256_dma<16>(rs_x, xoff[r], (kb0 + kb) * 256 + q * 64, lds0 + q * kPre256X + (4 * wave + r) * 1024);
    };
    // weights: this wave's units of a k-block (past the last column group: the last again, its results are not stored)
    const int cg0 = min(tn * 8 + 2 * wave, p.ncg - 1), cg1 = min(tn * 8 + 2 * wave + 1, p.ncg - 1);
    const int scale_off = 2048 + (lane & 31) * 4 + (lane >> 5) * (cg1 - cg0) * kP32Unit;
    auto      dma_w     = [&](int kb, int n) {
        const unsigned dst = lds0 + 4 * kPre256X + ((kb & 1) * 4 + wave) * kPre256W;
        const int      at  = (kb0 + min(kb, nkb - 1)) * p.ncg;
        if (n < 4) {
            pre256_dma<16>(rs_w, lane * 16, (at + (n < 2 ? cg0 : cg1)) * kP32Unit + (n & 1) * 1024, dst + n * 1024);
        }
        else {
            pre256_dma<4>(rs_w, scale_off, (at + cg0) * kP32Unit, dst + 4096);
        }
    };

    floatx4 acc[16][4];  // [row tile][column tile]
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
    const char* const xf = smem + fr * 64 + (((2 * (fc & 1) + (fc >> 1)) ^ ((fr >> 1) & 3)) << 4);
    const char* const wf = smem + 4 * kPre256X + wave * kPre256W;
    uint32_t          m1024 = 0x64006400u, m64 = 0x54005400u;
    asm volatile("" : "+v"(m1024), "+v"(m64));

    u32x4    fx[2][16], fw[2][4];  // fragments of a step and of the next
    u32x4    raw[2];               // per unit: the codes of two steps
    uint32_t sc[4], d[4];          // per column tile: (s, -z s); the codes of the step that is being dequantised
    auto     read_raw = [&](int kb, int h) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            raw[u] = *(const u32x4*)(wf + (kb & 1) * 4 * kPre256W + (2 * u + h) * 1024 + lane * 16);
        }
    };
    auto read_scale = [&](uint32_t(&s)[4], int kb) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = *(const uint32_t*)(wf + (kb & 1) * 4 * kPre256W + 4096 + (j * 16 + fr) * 4);
        }
    };
    auto swap = [&](int q) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const auto r = __builtin_amdgcn_permlane16_swap(raw[u][2 * q & 3], raw[u][(2 * q & 3) + 1], false, false);
            d[2 * u] = r[0], d[2 * u + 1] = r[1];
        }
    };
    auto part = [&](auto B, auto N, const uint32_t(&s)[4]) {  // part N & 3 of weight fragment N >> 2
        constexpr int b = decltype(B)::value, j = decltype(N)::value >> 2, e = decltype(N)::value & 3;
        const half2_t pr = bit_cast<half2_t>(s[j]);
        fw[b][j][e]      = pre256_dequant2<e>(d[j], half2_t{pr[0], pr[0]}, half2_t{pr[1], pr[1]}, m1024, m64);
    };
    if (nkb > 0) {
#pragma unroll
        for (int n = 0; n < 2 * kPre256WPiece; ++n) {
            dma_w(n / kPre256WPiece, n % kPre256WPiece);
        }
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            dma_x(0, n >> 2, n & 3);
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * kPre256XPiece) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (p.dbg && tid == 0) {
            p.dbg[wgid * 8 + 1] = __builtin_amdgcn_s_memrealtime();
            p.dbg[wgid * 8 + 5] = __builtin_amdgcn_s_memtime();  // shader-clock counter: (d6 - d5) / loop time = the clock
        }
        read_raw(0, 0);
        read_scale(sc, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            fx[0][i] = *(const u32x4*)(xf + i * 1024);
        }
        swap(0);
        static_for<16>([&](auto N) { part(std::integral_constant<int, 0>{}, N, sc); });
        for (int kb = 0; kb < nkb; ++kb) {
            uint32_t sn[4];
            static_for<4>([&](auto Q) {
                constexpr int q = decltype(Q)::value, b = q & 1;
                const int     kx = min(kb + 1, nkb - 1);
                // this wave's fragments of the step are in registers and its pieces of the next row stage have landed (and, at q = 2, the next k-block's
                // units: they left five steps ago); then everybody's.  Behind those pieces: the row pieces of two steps, the units that left at q = 1
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * kPre256XPiece + (q >= 2 ? kPre256WPiece : 0)) : "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const char* const st = xf + (q + 1 & 3) * kPre256X;
                if constexpr (q == 3) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        sc[j] = sn[j];
                    }
                }
                swap(q + 1 & 3);
                // codes of the step after next (q = 0, 2), scales of the next k-block
                if constexpr (q == 0) {
                    read_raw(kb, 1);
                }
                if constexpr (q == 2) {
                    read_raw(kb + 1, 0);
                    read_scale(sn, kb + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                static_for<16>([&](auto I) {
                    constexpr int i = decltype(I)::value;
                    auto          mma = [&](int k) {
                        const int j = i & 1 ? 3 - k : k;  // neighbours share an operand
                        pre256_mma(acc[i][j], fw[b][j], fx[b][i]);
                    };
                    mma(0);
                    fx[b ^ 1][i] = *(const u32x4*)(st + i * 1024);
                    mma(1);
                    part(std::integral_constant<int, b ^ 1>{}, I, sc);
                    mma(2);
                    if constexpr (i % 4 == 2) {  // the step's own row stage is free: the rows of four steps on
                        dma_x(kx, q, i >> 2);
                    }
                    if constexpr (q == 1 && i % 2 == 1 && i < 10) {  // the k-block's units are in registers since the step before
                        dma_w(kb + 2, i >> 1);
                    }
                    mma(3);
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the DMA writes this workgroup's LDS)
    }
    if (p.dbg && tid == 0) {
        p.dbg[wgid * 8 + 2] = __builtin_amdgcn_s_memrealtime();
        p.dbg[wgid * 8 + 6] = __builtin_amdgcn_s_memtime();
        p.dbg[wgid * 8 + 7] = p.dbg[wgid * 8 + 2];
    }
    // ---- epilogue: straight from the accumulators.  Lane holds, per row tile i and column tile j: row m = 16 i + fr, columns 64 wave + 16 j + 4 fc + 0 .. 3.
    // fp16 results change places between the lane groups, so that lane group fc has all 16 columns (8 gated) of column tile fc and stores them in 16-byte pieces
    const bool wide = p.epilogue != 2 && (p.ldy & 7) == 0 && ((uintptr_t)p.y & 15) == 0;
    const int  n0   = tn * 256 + wave * 64;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            asm volatile("s_nop 7" : "+a"(acc[i][j]));  // (the last results are passes behind their issue)
        }
        const int    m  = 16 * i + fr;
        const size_t mg = (size_t)m0 + m;
        if (p.epilogue == 2) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = n0 + 16 * j + 4 * fc;
                if (m < Mloc && n < p.N) {
                    floatx4* dst = (floatx4*)(p.partial + ((size_t)blockIdx.y * p.M + mg) * p.N + n);
                    if (p.wt & 1) {
                        store_wt(dst, acc[i][j], p.wt >> 4);
                    }
                    else {
                        *dst = acc[i][j];
                    }
                }
            }
        }
        else if (p.epilogue == 1) {
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const floatx4 a = acc[i][j];
                o[j]            = bit_cast<uint32_t>(half2_t{(half_t)(silu_f32(a[0]) * a[1]), (half_t)(silu_f32(a[2]) * a[3])});
            }
            if (wide) {
                pre256_transpose(o);
                if (m < Mloc && n0 + 16 * fc < p.N) {
                    *(u32x4*)(p.y + mg * p.ldy + (n0 >> 1) + 8 * fc) = u32x4{o[0], o[1], o[2], o[3]};
                }
            }
            else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + 16 * j + 4 * fc;
                    if (m < Mloc && n < p.N) {
                        *(uint32_t*)(p.y + mg * p.ldy + (n >> 1)) = o[j];
                    }
                }
            }
        }
        else {
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const floatx4 a = acc[i][j];
                lo[j]           = bit_cast<uint32_t>(half2_t{(half_t)a[0], (half_t)a[1]});
                hi[j]           = bit_cast<uint32_t>(half2_t{(half_t)a[2], (half_t)a[3]});
            }
            if (wide) {
                pre256_transpose(lo);
                pre256_transpose(hi);
                if (m < Mloc && n0 + 16 * fc < p.N) {
                    u32x4* dst = (u32x4*)(p.y + mg * p.ldy + n0 + 16 * fc);
                    dst[0]     = u32x4{lo[0], hi[0], lo[1], hi[1]};
                    dst[1]     = u32x4{lo[2], hi[2], lo[3], hi[3]};
                }
            }
            else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + 16 * j + 4 * fc;
                    if (m < Mloc && n < p.N) {
                        *(u32x2*)(p.y + mg * p.ldy + n) = u32x2{lo[j], hi[j]};
                    }
                }
            }
        }
    }
    if (p.dbg && tid == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        p.dbg[wgid * 8 + 3] = __builtin_amdgcn_s_memrealtime();
    }
}

// shape kShapePre256: grid = (ceil(ncg / 8), splits, ceil(M / 256))
int launch_pre256(const Dec32Params& p, dim3 grid, hipStream_t st)
{
    if (const int rc = ensure_dynamic_lds((const void*)gemm_pre256_kernel, kPre256Lds)) {
        return rc;
    }
    gemm_pre256_kernel<<<grid, 256, kPre256Lds, st>>>(p);
    TM_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace tmk
