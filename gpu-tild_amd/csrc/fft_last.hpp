// fft_last.hpp -- the fused last-axis pass with register-resident columns, k_last_reg
// (CDNA4 / gfx950), shared by the files that compile one class of its variants each.
//
// k_last_reg: the same operation as k_last_fused (kernels.hip) -- last-axis forward FFT of every
// field, the k-space coupling w_I = sum_J C_IJ rho_J (+ the charge row), and the
// inverse transforms of w and -i k_la w -- for last axes with a plan of TILD_REG_PLANS,
// N = R1 R2.  Each thread keeps its values in registers through a group of stages, so a
// block makes three LDS exchanges and three barriers, where the LDS-staged form stages
// every value through LDS and ends each of its nine or more phases with a barrier:
//
//   A   thread (b, i < R2, f): rows i + R2 r of column b of field f, read from HBM
//       straight into registers; first group; exchange.
//   B1  thread (b, i < R1, f): second group -> rho_f(k) at k = i + R1 q, back to the rows
//       it read, where the other threads find it.
//   B2  w_f(k) = sum_J C_fJ rho_J and the first group of the field's two inverse lines
//       conj(w), conj(-i k w); exchange.  Plans of two stages run the inverse reversed,
//       R2 x R1: thread (b, i < R1, f) couples the k = i + R1 q it holds.  Other plans run it
//       as they are: thread (b, i < R2, f) couples k = i + R2 q.
//   C   the second group of the lines, one task per (b, line, index); rows stored.
//
// One field per thread in the middle stages: a thread that took every field (and one of
// the two inverse lines, so that two threads repeated the forward stage) issued 1.5 times
// the instructions and held up to 256 registers; the stage was the longest of the block
// (2.7 of 7.7 us on a 192-point film's 13 blocks, where it ran one wave per SIMD).
// The transforms and sums are those of the LDS-staged pass (whose inverse runs the same
// plan, RepDev::axr), bit for bit but for the kept plans (reg_plan_kept), whose twiddle
// products fuse the other of their two sums' terms here (cmul_kept).
#pragma once
#include "device.hpp"
#include "fft_dev.hpp"
#include "fft_reg_dev.hpp"
#include "launch.hpp"

namespace tild {

namespace {

// One block: NB = last_reg_cols adjacent columns q0 .. q0 + NB - 1 of the last-axis lines
// (fewer in the last block), TT types and CH charge fields (NF = TT + CH).
// LDS: the forward exchange (N x ldx), the inverse exchange (N x ldy), the second group's
// twiddles of the inverse, then the ramp weights (last_reg_lds_bytes).
template <class P, int NT, int TT, int CH>
__device__ __forceinline__ void last_reg_block(const RepDev& r, int blk, float2* lds, int koff) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N, NF = TT + CH, NB = last_reg_cols(R1, R2, NF);
    constexpr bool REV = P::REV;
    constexpr int ldx = NF * NB + 1, ldy = 2 * NF * NB + 1;
    constexpr int NT2 = REV ? N - R2 : N - R1;      // twiddles of the inverse's second group
    constexpr int RC = REV ? R2 : R1;               // spectrum values a thread couples
    constexpr bool XCH = NF > 1 || !REV;            // the spectrum changes threads
    static_assert(NB >= 1 && NB * P::RM * NF <= NT && NT2 <= NT, "k_last_reg: one task of each stage per thread");
    const int la = r.dim - 1, D = r.dim;
    const int Q = la == 2 ? r.Ny * r.Nxh : r.Nxh;   // plane size = line stride
    const int q0 = blk * NB;
    const int nb = min(NB, Q - q0);
    float2* X1 = lds;                               // N x ldx: forward exchange
    float2* Y1 = lds + N * ldx;                     // N x ldy: inverse exchange
    float2* TW2 = Y1 + N * ldy;
    float* rw = (float*)(TW2 + NT2);                // ramp weights of this step
    // lanes: column, then field, then i (the fields' LDS rows are NB values apart, which
    // spreads a wave's accesses over the banks)
    const int b = (int)threadIdx.x % NB, f = ((int)threadIdx.x / NB) % NF, i = (int)threadIdx.x / (NB * NF);
    const bool liveA = b < nb && i < R2, liveB = b < nb && i < R1;
    const bool liveC = REV ? liveB : liveA;         // couples k = i + R1 q (REV) or i + R2 q
    constexpr int KS = REV ? R1 : R2;
    // grid buffers below 4 GiB (required on the host): 32-bit element offsets
    const uint32_t Qu = (uint32_t)Q, Mhu = (uint32_t)r.Mh;
    const float2* const tw = la == 2 ? r.reg_tw[2] : r.reg_tw[1];

    // everything the block reads is requested before the first wait: this thread's rows
    // of the spectrum, its twiddles of both groups and its coupling rows
    float2 t2 = make_float2(0.f, 0.f);
    if ((int)threadIdx.x < NT2) t2 = gld(r.reg_twr + threadIdx.x);
    float2 v[R1];
    if (liveA) {
#pragma unroll
        for (int rr = 0; rr < R1; ++rr)
            v[rr] = gld(at32((const float2*)r.H, (uint32_t)f * Mhu + (uint32_t)(i + R2 * rr) * Qu + (uint32_t)(q0 + b)));
    }
    // coupling rows of w_f: pidx(lo, hi) = lo TT - lo (lo - 1) / 2 + (hi - lo) for the
    // types, the charge row for the charge field.  Element (n, row) of column b:
    // cb0 + (n nrows + row) NB from the uniform table base.
    const int nrows = r.ctab_rows;
    const uint32_t cb0 = (uint32_t)blk * (uint32_t)(N * nrows * NB) + (uint32_t)b;
    auto ctab = [&](int n, int row) { return G(at32(r.Ctab, cb0 + (uint32_t)((n * nrows + row) * NB)))[0]; };
    const bool isq = CH && f == TT;
    auto pidx = [&](int J) {
        const int lo = min(f, J), hi = max(f, J);
        return lo * TT - lo * (lo - 1) / 2 + (hi - lo);
    };
    float2 t1[R2];
    float c[RC][TT];
    if (liveB) {
#pragma unroll
        for (int m = 1; m < R2; ++m) t1[m] = gld(tw + tw2_index<P>(i, m));
    }
    if (liveC) {
#pragma unroll
        for (int J = 0; J < TT; ++J) {
            const int row = isq ? r.ctab_charge : pidx(J);
#pragma unroll
            for (int q = 0; q < RC; ++q) c[q][J] = ctab(i + KS * q, row);
        }
    }
    if ((int)threadIdx.x < r.nramp) rw[threadIdx.x] = ramp_weight(r, threadIdx.x, r.step + koff);

    // ---- A: first group on rows i + R2 r (out[i R1 + q])
    if (liveA) {
        plan_first<P>(v, tw);
#pragma unroll
        for (int q = 0; q < R1; ++q) X1[(i * R1 + q) * ldx + f * NB + b] = v[q];
    }
    if ((int)threadIdx.x < NT2) TW2[threadIdx.x] = t2;
    __syncthreads();

    // ---- B1: second group -> rho_f(k), k = i + R1 q
    float2 w[RC > R2 ? RC : R2];
    if (liveB) {
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = X1[(i + R1 * rr) * ldx + f * NB + b];
        plan_second<P, !P::KEPT>(w, [&](int m) { return t1[m]; });
        if constexpr (XCH) {
#pragma unroll
            for (int q = 0; q < R2; ++q) X1[(i + R1 * q) * ldx + f * NB + b] = w[q];
        }
    }
    if constexpr (XCH) __syncthreads();

    // ---- B2: coupling and the first group of the two inverse lines
    if (liveC) {
        for (int j = 0; j < r.nramp; ++j) {   // ramped styles add their weighted rows (uniform trip count)
            const float wj = rw[j];
            const int rp = r.ramp_pair[j];
#pragma unroll
            for (int J = 0; J < TT; ++J) {
                const bool on = !isq && rp == pidx(J);
#pragma unroll
                for (int q = 0; q < RC; ++q) {
                    const float cr = wj * ctab(i + KS * q, r.ramp_row0 + j);
                    c[q][J] += on ? cr : 0.f;
                }
            }
        }
        if constexpr (!REV) {   // this thread's values of its own field
#pragma unroll
            for (int q = 0; q < RC; ++q) w[q] = X1[(i + KS * q) * ldx + f * NB + b];
        }
        // w_f = sum_J C_fJ rho_J; charges w_c = G_c rho_c
#pragma unroll
        for (int q = 0; q < RC; ++q) {
            float2 acc = make_float2(0.f, 0.f);
#pragma unroll
            for (int J = 0; J < TT; ++J) {
                const float2 rh = NF > 1 ? X1[(i + KS * q) * ldx + J * NB + b] : w[q];
                acc.x += c[q][J] * rh.x; acc.y += c[q][J] * rh.y;
            }
            w[q] = isq ? scaled(c[q][0], w[q]) : acc;
        }
        // the inverse is conj(FFT(conj)): conj(w) = (w.x, -w.y), then conj(-i k_la w) =
        // (k w.y, k w.x), k_la = 0 on the Nyquist plane
        auto inverse_first = [&](float2* z, int line) {
            if constexpr (REV) {   // plan R2 x R1: radix R2, out[i R2 + q]
                Dft<R2>::run(z);
#pragma unroll
                for (int q = 0; q < R2; ++q) Y1[(i * R2 + q) * ldy + line * NB + b] = z[q];
            } else {
                plan_first<P>(z, tw);
#pragma unroll
                for (int q = 0; q < R1; ++q) Y1[(i * R1 + q) * ldy + line * NB + b] = z[q];
            }
        };
        const float fi = (float)i;
        float2 z[RC];
#pragma unroll
        for (int q = 0; q < RC; ++q) z[q] = make_float2(w[q].x, -w[q].y);
        inverse_first(z, f);
#pragma unroll
        for (int q = 0; q < RC; ++q) {
            const float kl = r.kfac[la] * freq_of<KS, N>(i, fi, q);
            z[q] = grad_line(kl, w[q]);
        }
        inverse_first(z, NF + f);
    }
    __syncthreads();

    // ---- C: second group of the inverse (REV: radix R1, twiddles w_N^{j r}, including the
    // unit ones of j = 0 as the staged pass multiplies them) -> rows j + RC q.  One task
    // per (column, line, j), spread over all threads.
    constexpr int RJ = REV ? R2 : R1, RV = REV ? R1 : R2;
    for (int task = threadIdx.x; task < NB * RJ * 2 * NF; task += NT) {
        const int bc = task % NB, rest = task / NB, line = rest % (2 * NF), j = rest / (2 * NF);   // line = o NF + f
        if (bc >= nb) continue;
        const int o = line >= NF ? 1 : 0, fl = line - o * NF;
        float2 z[RV];
#pragma unroll
        for (int rr = 0; rr < RV; ++rr) z[rr] = Y1[(j + RJ * rr) * ldy + line * NB + bc];
        if constexpr (REV) {
#pragma unroll
            for (int rr = 1; rr < R1; ++rr) z[rr] = cmul_as<!P::KEPT>(z[rr], TW2[j * (R1 - 1) + rr - 1]);
            Dft<R1>::run(z);
        } else {
            plan_second_lds<P, true>(z, TW2, j);
        }
        const uint32_t o0 = (uint32_t)(fl * D + (o == 0 ? 0 : la)) * Mhu + (uint32_t)j * Qu + (uint32_t)(q0 + bc);
        const uint32_t step = (uint32_t)RJ * Qu;
#pragma unroll
        for (int q = 0; q < RV; ++q) gst(at32(r.Gk, o0 + (uint32_t)q * step), conjf2(z[q]));
    }
}

template <class P, int NT, int TT, int CH, int CLS>
__device__ __forceinline__ void last_reg_variant_block(const RepDev& r, int blk, float2* lds, int koff) {
    if constexpr (last_reg_variant(P::A0, P::R1, P::R2, P::REV, TT) && last_reg_held(last_reg_class(P::N, TT), CLS))
        last_reg_block<P, NT, TT, CH>(r, blk, lds, koff);
}

template <class P, int NT, int CLS>
__device__ __forceinline__ void last_reg_types(const RepDev& r, int blk, float2* lds, int koff) {
    const bool ch = r.nf > r.ntypes;
    switch (r.ntypes * 2 + (ch ? 1 : 0)) {
        case 2: last_reg_variant_block<P, NT, 1, 0, CLS>(r, blk, lds, koff); break;
        case 3: last_reg_variant_block<P, NT, 1, 1, CLS>(r, blk, lds, koff); break;
        case 4: last_reg_variant_block<P, NT, 2, 0, CLS>(r, blk, lds, koff); break;
        case 5: last_reg_variant_block<P, NT, 2, 1, CLS>(r, blk, lds, koff); break;
        case 6: last_reg_variant_block<P, NT, 3, 0, CLS>(r, blk, lds, koff); break;
        case 7: last_reg_variant_block<P, NT, 3, 1, CLS>(r, blk, lds, koff); break;
        case 8: last_reg_variant_block<P, NT, 4, 0, CLS>(r, blk, lds, koff); break;
        case 9: last_reg_variant_block<P, NT, 4, 1, CLS>(r, blk, lds, koff); break;
        default: break;   // excluded by last_reg_plan on the host
    }
}

}  // namespace

// One instantiation per class of variants (last_reg_class), each compiled in a file of
// its own: a class's registers do not lower the occupancy of another's, and the classes
// compile side by side.  In a set of several classes those of class 0 join the launch of
// another (films of 64 and 128 points in one launch 7.5 us a step, in two 12.7; six 64^3 and
// six 64 x 64 x 128 melts 35.9 and 43.2): the kernel of class 2 holds them too, at no cost to
// it, and kernel 3 holds classes 0 and 1 for such sets, since class 1 alone lost by it
// (coacervate on 64^3 8.8 -> 9.7 us).
template <int NT, int CLS>
__global__ void __launch_bounds__(NT) k_last_reg(const RepDev* __restrict__ reps, const WorkItem* __restrict__ wmap,
                                                 int koff) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    warm_desc<0, 1, 6, 7>(r);
    switch (r.dim == 3 ? r.reg_key[2] : r.reg_key[1]) {   // uniform per block
#define TILD_CASE(A0, A1, B0, B1) \
    case reg_plan_key(A0, A1, B0, B1): last_reg_types<RegPlan<A0, A1, B0, B1>, NT, CLS>(r, wi.blk, lds, koff); break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by last_reg_plan on the host
    }
}

// launch and attributes of one class (defined per file)
#define TILD_LAST_REG_CLASS(CLS)                                                                                    \
    hipError_t launch_last_reg_##CLS(const LaunchCtx& c, int koff) {                                                \
        TILD_LAUNCH(c, (k_last_reg<kLastRegThreads, CLS>), dim3(c.n), dim3(kLastRegThreads), c.lds, c.reps, c.wmap, \
                    koff);                                                                                          \
        return hipGetLastError();                                                                                   \
    }                                                                                                               \
    hipError_t configure_last_reg_##CLS() {                                                                         \
        return hipFuncSetAttribute((const void*)k_last_reg<kLastRegThreads, CLS>,                                   \
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPlaneLds);                     \
    }

}  // namespace tild
