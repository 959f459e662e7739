// Common device/host helpers for the MI355X-native TurboMind hot path (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string>

namespace tmk {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float    floatx4 __attribute__((ext_vector_type(4)));
typedef float    floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

// ---- error plumbing (C-ABI never throws) -----------------------------------------------
void        set_last_error(const std::string& msg);
const char* get_last_error();
// Raise a kernel's dynamic-LDS limit on the CURRENT device, once per (kernel, device): hipFuncAttributeMaxDynamicSharedMemorySize
// is a per-device function attribute.  Thread-safe (engines of several devices / threads launch concurrently).
int         ensure_dynamic_lds(const void* kernel, int bytes);

#define TM_HIP_CHECK(expr)                                                                         \
    do {                                                                                           \
        hipError_t _e = (expr);                                                                    \
        if (_e != hipSuccess) {                                                                    \
            ::tmk::set_last_error(std::string(#expr) + ": " + hipGetErrorString(_e) + " @" + __FILE__ + ":" \
                                 + std::to_string(__LINE__));                                      \
            return 5; /* TM_FAIL */                                                                \
        }                                                                                          \
    } while (0)

#define TM_REQUIRE(cond, msg)                                                                      \
    do {                                                                                           \
        if (!(cond)) {                                                                             \
            ::tmk::set_last_error(std::string("invalid argument: ") + (msg) + " (" #cond ")");      \
            return 1; /* TM_INVALID */                                                             \
        }                                                                                          \
    } while (0)

// ---- tiny device helpers ---------------------------------------------------------------
template<class To, class From>
__device__ __forceinline__ To bit_cast(const From& f)
{
    return __builtin_bit_cast(To, f);
}

// z / (1 + e^-z) in fp32, the one silu of every product's epilogue: a call's numbers do not depend on which tile makes them
__device__ __forceinline__ float silu_f32(float z)
{
    return z / (1.0f + __builtin_expf(-z));
}

__device__ __forceinline__ half2_t h2_fma(half2_t a, half2_t b, half2_t c)
{
    return __builtin_elementwise_fma(a, b, c);  // v_pk_fma_f16, single rounding
}

// DPP lane exchange inside a row of 16 lanes (no LDS).  ctrl: quad_perm / row_* codes.
template<int CTRL>
__device__ __forceinline__ float dpp_f32(float v)
{
    return bit_cast<float>(__builtin_amdgcn_update_dpp(0, bit_cast<int>(v), CTRL, 0xF, 0xF, false));
}
template<int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}

constexpr int DPP_XOR1  = 0xB1;   // quad_perm [1,0,3,2]
constexpr int DPP_XOR2  = 0x4E;   // quad_perm [2,3,0,1]
constexpr int DPP_HMIRR = 0x141;  // row_half_mirror (lane i <-> 7-i in each 8)
constexpr int DPP_ROR8  = 0x128;  // row_ror:8      (lane i <- i^8 in each 16)

// butterfly all-reduce (sum / max) over groups of N consecutive lanes, N in {8,16,64}
template<int N>
__device__ __forceinline__ float group_sum(float v)
{
    v += dpp_f32<DPP_XOR1>(v);
    v += dpp_f32<DPP_XOR2>(v);
    v += dpp_f32<DPP_HMIRR>(v);
    if constexpr (N >= 16) {
        v += dpp_f32<DPP_ROR8>(v);
    }
    if constexpr (N >= 64) {
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
    }
    return v;
}
template<int N>
__device__ __forceinline__ float group_max(float v)
{
    v = fmaxf(v, dpp_f32<DPP_XOR1>(v));
    v = fmaxf(v, dpp_f32<DPP_XOR2>(v));
    v = fmaxf(v, dpp_f32<DPP_HMIRR>(v));
    if constexpr (N >= 16) {
        v = fmaxf(v, dpp_f32<DPP_ROR8>(v));
    }
    if constexpr (N >= 64) {
        v = fmaxf(v, __shfl_xor(v, 16));
        v = fmaxf(v, __shfl_xor(v, 32));
    }
    return v;
}

// reduce across the lanes that differ in bits >= log2(LOW) (i.e. keep the low LOW lanes distinct)
template<int LOW>
__device__ __forceinline__ float upper_sum(float v)
{
    if constexpr (LOW <= 8) {
        v += dpp_f32<DPP_ROR8>(v);
    }
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    return v;
}
template<int LOW>
__device__ __forceinline__ float upper_max(float v)
{
    if constexpr (LOW <= 8) {
        v = fmaxf(v, dpp_f32<DPP_ROR8>(v));
    }
    v = fmaxf(v, __shfl_xor(v, 16));
    v = fmaxf(v, __shfl_xor(v, 32));
    return v;
}

__device__ __forceinline__ float fast_exp2(float x)
{
    return __builtin_amdgcn_exp2f(x);  // v_exp_f32 (no denormal range handling needed here)
}

// A pointer that a table holds as a number.  Cast to a plain pointer its loads are flat ones, which count as LDS traffic too and return in no order that a
// wait could use: whatever is in flight has to arrive before the first of them is used (fp32 attention, 16 / 1 heads of 256 / 192, a prompt
// of 2000: 667 -> 597 us, row kernel 7810 -> 7165; 2 decoded rows over 2000 29.4 -> 27.4)
__device__ __forceinline__ char* global_ptr(uint64_t address)
{
    return (char*)(__attribute__((address_space(1))) char*)address;
}

// ---- results of several workgroups met in one launch ----
// Partial results are written through to the device's memory (agent_store), drained, and counted in a ticket that is zero between launches; who arrives last
// reads them past its caches (agent_load) and finishes.  No workgroup waits for another.
__device__ __forceinline__ void agent_store(float* p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float agent_load(const float* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The same for several neighbours, at `at` bytes behind a base that all lanes share (agent_base: its first `bytes` bytes): buffer instructions with the agent's scope (sc1),
// which need no more than the four-byte alignment of a float
__device__ __forceinline__ auto agent_base(const float* base, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}
template<class Base>
__device__ __forceinline__ void agent_store4(Base base, int at, floatx4 v)
{
    __builtin_amdgcn_raw_buffer_store_b128(bit_cast<u32x4>(v), base, at, 0, /*sc1*/ 16);
}
template<class Base>
__device__ __forceinline__ floatx4 agent_load4(Base base, int at)
{
    return bit_cast<floatx4>(__builtin_amdgcn_raw_buffer_load_b128(base, at, 0, /*sc1*/ 16));
}
template<class Base>
__device__ __forceinline__ floatx2 agent_load2(Base base, int at)
{
    return bit_cast<floatx2>(__builtin_amdgcn_raw_buffer_load_b64(base, at, 0, /*sc1*/ 16));
}
// of n arrivals: is this the last one (which also clears the ticket)?  One lane calls it after the stores are drained
__device__ __forceinline__ bool ticket_last(unsigned* ticket, int n)
{
    const bool last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (unsigned)n;
    if (last) {
        __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return last;
}
// the same for a wave (the lanes that are active; lane 0 is one of them) and for a whole workgroup (flag: one word of LDS)
__device__ __forceinline__ bool ticket_last_wave(unsigned* ticket, int n)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int last = 0;
    if ((threadIdx.x & 63) == 0) {
        last = ticket_last(ticket, n);
    }
    return __builtin_amdgcn_readfirstlane(last) != 0;
}
__device__ __forceinline__ bool ticket_last_workgroup(unsigned* ticket, int n, unsigned* flag)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        *flag = ticket_last(ticket, n);
    }
    __syncthreads();
    return *flag != 0;
}

}  // namespace tmk
