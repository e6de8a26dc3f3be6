// fft_reg_dev.hpp -- plans, butterflies and helpers of the register-resident FFT passes.
//
// A plan is two groups of Stockham stages, (A0 A1) and (B0 B1).  In a transform of length
// N = R1 R2, R1 = A0 A1 and R2 = B0 B1:
//   first group   thread i < R2 takes x[i + R2 r], r < R1, and leaves y[i R1 + q], q < R1;
//   second group  thread i < R1 takes y[i + R1 s], s < R2, and leaves X[i + R1 q], q < R2.
// A group of two stages (a, b) runs both in registers: the stages of the LDS-staged
// transform on the same values with the same twiddles, without the exchange between them.
#pragma once
#include "device.hpp"
#include "fft_dev.hpp"
#include "launch.hpp"

namespace tild {

template <int A0_, int A1_, int B0_, int B1_> struct RegPlan {
    static constexpr int A0 = A0_, A1 = A1_, B0 = B0_, B1 = B1_;
    static constexpr int R1 = A0 * A1, R2 = B0 * B1, N = R1 * R2;
    static constexpr int RM = R1 > R2 ? R1 : R2;
    static constexpr int NTW = N - R1;             // twiddles of the second group
    static constexpr bool REV = A1 == 1 && B1 == 1;   // the last axis' inverse runs reversed
    static constexpr bool KEPT = reg_plan_kept(N);
};

// Twiddles of the second group of an N-point plan: N - R1 (uniform).
__device__ __forceinline__ int reg_ntw(int key, int N) {
    switch (key) {
#define TILD_CASE(A0, A1, B0, B1) case reg_plan_key(A0, A1, B0, B1): return N - (A0) * (A1);
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: return 0;
    }
}

// Complex product with its fused operations spelled out: those of the LDS-staged stages,
// whatever surrounds the product here.
__device__ __forceinline__ float2 cmul_fused(float2 a, float2 b) {
#pragma clang fp contract(off)
    const float yy = a.y * b.y, yx = a.y * b.x;
    return make_float2(__builtin_fmaf(a.x, b.x, -yy), __builtin_fmaf(a.x, b.y, yx));
}
// ... those of the kept plans in the forward plane pass and the fused last-axis pass,
// which are compiled into several kernels: a replica's bits may not depend on which of
// them its set runs
__device__ __forceinline__ float2 cmul_kept(float2 a, float2 b) {
#pragma clang fp contract(off)
    const float yy = a.y * b.y, xy = a.x * b.y;
    return make_float2(__builtin_fmaf(a.x, b.x, -yy), __builtin_fmaf(a.y, b.x, xy));
}
template <bool FUSED> __device__ __forceinline__ float2 cmul_as(float2 a, float2 b) {
    if constexpr (FUSED) return cmul_fused(a, b);
    else return cmul_kept(a, b);
}

// The n values are computed here: a sum that the compiler moves to its use in a later block
// (past a barrier) rounds its product there, which is fused into the sum here.
template <int n> __device__ __forceinline__ void settle(float2* v) {
#pragma unroll
    for (int r = 0; r < n; ++r) asm volatile("" : "+v"(v[r].x), "+v"(v[r].y));
}

// Stages (A, B) on v[r], r < A B, in place (output q natural): stage A over r = r2 + B r1
// for each r2, twiddles w_{AB}^{r2 k} at tw[k (B - 1) + r2 - 1], stage B.
template <int A, int B>
__device__ __forceinline__ void first_group(float2* v, const float2* tw) {
    if constexpr (B == 1) {
        Dft<A>::run(v);
    } else {
        float2 z[B][A];
#pragma unroll
        for (int r2 = 0; r2 < B; ++r2) {
            float2 a[A];
#pragma unroll
            for (int r1 = 0; r1 < A; ++r1) a[r1] = v[r2 + B * r1];
            Dft<A>::run(a);
#pragma unroll
            for (int k = 0; k < A; ++k) z[r2][k] = a[k];
        }
#pragma unroll
        for (int k = 0; k < A; ++k) {
            float2 u[B];
            u[0] = z[0][k];
#pragma unroll
            for (int r2 = 1; r2 < B; ++r2) u[r2] = k == 0 ? z[r2][0] : cmul_fused(z[r2][k], gld(tw + (k * (B - 1) + r2 - 1)));
            Dft<B>::run(u);
#pragma unroll
            for (int q = 0; q < B; ++q) v[k + A * q] = u[q];
        }
    }
}
// The first group of plan P; tw2 = the second group's twiddles, which follow the first
// group's in the table.
template <class P>
__device__ __forceinline__ void plan_first(float2* v, const float2* tw2) {
    first_group<P::A0, P::A1>(v, tw2 - P::A0 * (P::A1 - 1));
}

// Index in the second group's table of the m-th twiddle (1 <= m < R2) of thread i: the
// first stage's w^{r i}, r = m < B0, then the second stage's w^{t (i + R1 q)},
// m = B0 + q (B1 - 1) + t - 1.
template <class P>
__device__ __forceinline__ int tw2_index(int i, int m) {
    if (m < P::B0) return i * (P::B0 - 1) + m - 1;
    const int u = m - P::B0, q = u / (P::B1 > 1 ? P::B1 - 1 : 1), t = u - q * (P::B1 - 1);
    return P::R1 * (P::B0 - 1) + (i + P::R1 * q) * (P::B1 - 1) + t;
}

// The second group of plan P on w[s], s < R2, in place (output q natural); tw(m) = the m-th
// twiddle of this thread.  FUSED: products as the LDS-staged stages fuse them, else cmul_kept.
template <class P, bool FUSED, class TW>
__device__ __forceinline__ void plan_second(float2* w, TW tw) {
    constexpr int C = P::B0, D = P::B1;
    if constexpr (D == 1) {
#pragma unroll
        for (int r = 1; r < C; ++r) w[r] = cmul_as<FUSED>(w[r], tw(r));
        Dft<C>::run(w);
    } else {
        float2 y[C][D];
#pragma unroll
        for (int t = 0; t < D; ++t) {
            float2 u[C];
#pragma unroll
            for (int r = 0; r < C; ++r) u[r] = r == 0 ? w[t] : cmul_fused(w[t + D * r], tw(r));
            Dft<C>::run(u);
#pragma unroll
            for (int q = 0; q < C; ++q) y[q][t] = u[q];
        }
#pragma unroll
        for (int q = 0; q < C; ++q) {
            float2 u[D];
#pragma unroll
            for (int t = 0; t < D; ++t) u[t] = t == 0 ? y[q][0] : cmul_fused(y[q][t], tw(C + q * (D - 1) + t - 1));
            Dft<D>::run(u);
#pragma unroll
            for (int q2 = 0; q2 < D; ++q2) w[q + C * q2] = u[q2];
        }
    }
}
// ... with its twiddles in LDS
template <class P, bool FUSED>
__device__ __forceinline__ void plan_second_lds(float2* w, const float2* TW, int i) {
    plan_second<P, FUSED>(w, [&](int m) { return TW[tw2_index<P>(i, m)]; });
}

// Frequency of n = i + S r, i < S (fi = (float)i), on an axis of N points, 0 at N/2.  Which
// side of N/2 the S values of one r lie on is known when the loop over r is unrolled, but
// for the r that holds N/2: spelled out, since i's bound is not visible to the compiler and
// the selects, conversions and address terms of every element were most of a short phase.
template <int S, int N>
__device__ __forceinline__ float freq_of(int i, float fi, int r) {
    const int lo = S * r, hi = lo + S - 1;
    if (2 * hi < N) return fi + (float)lo;
    if (2 * lo > N) return fi + (float)(lo - N);
    const int n2 = 2 * (i + lo);
    const float f = 2 * lo == N || n2 > N ? fi + (float)(lo - N) : fi + (float)lo;
    return N % 2 == 0 && n2 == N ? 0.f : f;
}
// The same n as an entry of a half spectrum: column kk = n, or N - n with the conjugate
// (upper; N/2 as either), self: its own conjugate, k: the frequency kk, 0 at N/2.
struct HalfEntry {
    bool upper, self;
    int kk;
    float k;
};
template <int S, int N>
__device__ __forceinline__ HalfEntry half_entry(int i, float fi, int r) {
    const int lo = S * r, hi = lo + S - 1;
    const bool mid = 2 * lo <= N && N <= 2 * hi;   // N/2 is among the S values
    const bool nyq = N % 2 == 0 && mid && 2 * (i + lo) == N;
    HalfEntry e;
    e.upper = 2 * hi <= N ? false : (2 * lo >= N ? true : 2 * (i + lo) > N);
    e.kk = e.upper ? (N - lo) - i : i + lo;
    e.k = e.upper ? (float)(N - lo) - fi : fi + (float)lo;
    if (nyq) e.k = 0.f;
    e.self = (r == 0 && i == 0) || nyq;
    return e;
}

// Products that the LDS-staged passes write to LDS before a later stage adds them: kept
// out of FMA contraction with those additions, as they are there.
__device__ __forceinline__ float2 scaled(float s, float2 a) {
#pragma clang fp contract(off)
    return make_float2(s * a.x, s * a.y);
}
__device__ __forceinline__ float2 grad_line(float k, float2 a) {
#pragma clang fp contract(off)
    return make_float2(k * a.y, k * a.x);
}
__device__ __forceinline__ float2 x_gradient(float kx, float2 a) {   // -i k_x a
#pragma clang fp contract(off)
    return make_float2(kx * a.y, -kx * a.x);
}
// on ? a : b, with both computed: a select, where the compiler branches around the products
// of every element and waits for its loads one by one
__device__ __forceinline__ float2 pick(bool on, float2 a, float2 b) {
    settle<1>(&a);
    return make_float2(on ? a.x : b.x, on ? a.y : b.y);
}
__device__ __forceinline__ float half_of(float a) {
#pragma clang fp contract(off)
    return 0.5f * a;
}

}  // namespace tild
