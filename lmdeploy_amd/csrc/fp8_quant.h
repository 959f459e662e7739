// e4m3 codes of fp16 rows, one scale per row and 128 channels (launch_quant_fp8_rows, and the workgroups behind the router's in moe.hip).
// Replaces: QuantizeSymm (src/turbomind/kernels/quantization.cu:28-125).
#pragma once
#include "tm_common.h"

namespace tmk {

// 256 threads, 16 (row, group)s: 16 lanes = one of them, 8 halves per lane, absmax by DPP, 8 codes (one 8-byte store) per lane
__device__ __forceinline__ void quant_fp8_groups(int block, uint8_t* __restrict__ xq, float* __restrict__ sx, const half_t* __restrict__ x, int ldx, int M, int K,
                                                 int ldsx)
{
    const int groups = K / 128;
    const int gid    = block * 16 + (threadIdx.x >> 4);  // (row, group) index
    const int l16    = threadIdx.x & 15;
    const bool ok    = gid < M * groups;
    const int gc     = ok ? gid : M * groups - 1;
    const int m      = gc / groups;
    const int g      = gc - m * groups;
    const half8_t v  = *(const half8_t*)(x + (size_t)m * ldx + g * 128 + l16 * 8);
    float amax       = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        amax = fmaxf(amax, fabsf((float)v[e]));
    }
    amax = group_max<16>(amax);
    amax = fmaxf(amax, 1e-8f);
    const float inv = 448.0f / amax;
    float       f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        f[e] = fminf(fmaxf((float)v[e] * inv, -448.0f), 448.0f);  // saturating RNE (the conversion below rounds to nearest even)
    }
    int w0 = 0, w1 = 0;
    w0     = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], w0, false);
    w0     = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
    w1     = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], w1, false);
    w1     = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
    if (ok) {
        *(u32x2*)(xq + (size_t)m * K + g * 128 + l16 * 8) = u32x2{(uint32_t)w0, (uint32_t)w1};
        if (l16 == 0) {
            sx[(size_t)g * ldsx + m] = amax / 448.0f;
        }
    }
}

}  // namespace tmk
