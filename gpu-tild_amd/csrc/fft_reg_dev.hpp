// fft_reg_dev.hpp -- helpers of the register-resident FFT passes.
#pragma once
#include "device.hpp"

namespace tild {

// Products that the LDS-staged pass writes to LDS before its next stage adds them:
// kept out of FMA contraction with those additions, as they are there.
__device__ __forceinline__ float2 scaled(float s, float2 a) {
#pragma clang fp contract(off)
    return make_float2(s * a.x, s * a.y);
}
__device__ __forceinline__ float2 grad_line(float k, float2 a) {
#pragma clang fp contract(off)
    return make_float2(k * a.y, k * a.x);
}

// A twiddle from LDS, as one value read where it is used: which product of a sum the
// compiler fuses follows the order and form of its operands' reads, and this is the
// LDS-staged passes' (which read theirs from global memory).
__device__ __forceinline__ float2 lds_twiddle(const float2* p) {
    f2v v = *(const f2v*)p;
    asm volatile("" : "+v"(v));
    return make_float2(v.x, v.y);
}

}  // namespace tild
