// mfma_device.h — device-side helpers shared by the matrix-core kernels: operand types, the
// XCD-aware tile order, row exponents, and buffer -> LDS loads with their waits.
#pragma once
#include "formats.h"
#include "nbits_device.h"

namespace msnb {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));

constexpr int kBsStride = 40;   // fp16 per LDS weight row (32 + 8 pad)

// tile index of workgroup `bid` among tiles_m*tiles_n tiles (m-major), so that
// XCD x = bid % 8 owns the contiguous tile range [x*per, (x+1)*per).
__device__ __forceinline__ int xcd_tile(int bid, int tiles)
{
    const int per = (tiles + kXcds - 1) / kXcds;
    return (bid % kXcds) * per + bid / kXcds;
}

// Base offset of a row beyond the matrix: above every buffer the kernels that use
// it read (the host checks each is smaller), so loads from it return zero.
constexpr int kPipeFar = 0x40000000;

__device__ __forceinline__ float max_abs8(const float4& lo, const float4& hi)
{
    return fmaxf(fmaxf(fmaxf(fabsf(lo.x), fabsf(lo.y)), fmaxf(fabsf(lo.z), fabsf(lo.w))),
                 fmaxf(fmaxf(fabsf(hi.x), fabsf(hi.y)), fmaxf(fabsf(hi.z), fabsf(hi.w))));
}

// Exponent e of a row whose largest magnitude is mx: mx * 2^-e lies in [2^14, 2^15)
// (mx in [2^(E-1), 2^E) with E = frexp exponent, e = E - 15). Rows that are all zero,
// or hold an inf (fmaxf skips NaN), take e = 0: their sums are zero or non-finite
// whatever the scaling.
__device__ __forceinline__ int row_exponent(float mx)
{
    return (mx > 0.0f && mx <= 3.402823466e38f) ? __builtin_amdgcn_frexp_expf(mx) - 15 : 0;
}

// Largest value of x over the workgroup of 256 threads, in every thread.
__device__ __forceinline__ float block256_max(float x, float* red4)
{
    x = row16_max_all(x);
    x = fmaxf(x, xor16_value(x));
    x = fmaxf(x, xor32_value(x));
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) red4[wave] = x;
    __syncthreads();
    return fmaxf(fmaxf(red4[0], red4[1]), fmaxf(red4[2], red4[3]));
}

typedef __attribute__((address_space(3))) uint8_t lds_byte_t;
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(lds_byte_t*)p; }

// buffer -> LDS loads: lane i's bytes land at LDS m0 + 16*i (x4) or m0 + 4*i (ushort).
// The s_nop keeps the wait states that the compiler does not insert before inline asm: one
// between a write of m0 and the load, five between a vector instruction's write of a scalar
// operand (a resource reloaded from a spill by v_readlane) and the load. A kernel whose scalar
// operands are all written by scalar instructions takes one (NOP 0): five cost mfma_w4_pipe 1%
// (M=512, K=3584 MLP: 332 -> 337 us). test_lds_load_wait_states.py reads both off the built code.
template <int NOP = 4>
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, int voff, int soff, uint32_t m0v)
{
    asm volatile("s_nop %4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff), "{m0}"(m0v), "n"(NOP)
                 : "memory");
}
template <int NOP = 4>
__device__ __forceinline__ void lds_load4(__amdgpu_buffer_rsrc_t r, int voff, int soff, uint32_t m0v)
{
    asm volatile("s_nop %4\n\tbuffer_load_dword %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff), "{m0}"(m0v), "n"(NOP)
                 : "memory");
}
template <int NOP = 4>
__device__ __forceinline__ void lds_load2(__amdgpu_buffer_rsrc_t r, int voff, int soff, uint32_t m0v)
{
    asm volatile("s_nop %4\n\tbuffer_load_ushort %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff), "{m0}"(m0v), "n"(NOP)
                 : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace msnb
