// fft_last.hpp -- the fused last-axis pass with register-resident columns, k_last_reg
// (CDNA4 / gfx950), shared by the files that compile one class of its variants each.
//
// k_last_reg: the same operation as k_last_fused (kernels.hip) -- last-axis forward FFT of every
// field, the k-space coupling w_I = sum_J C_IJ rho_J (+ the charge row), and the
// inverse transforms of w and -i k_la w -- for last axes with a two-stage plan
// N = R1 R2 (TILD_REG_PLANS; R1 >= R2).  Each
// thread keeps its Stockham columns in registers between the stages, so a block makes
// three LDS exchanges and three barriers, where the LDS-staged form stages every value
// through LDS and ends each of its nine phases with a barrier:
//
//   A   thread (b, i < R2, f): rows i + R2 r of column b of field f, read from HBM
//       straight into registers; DFT_R1; exchange.
//   B1  thread (b, i < R1, f): twiddles w_N^{i r}, DFT_R2 -> rho_f(k) at k = i + R1 q,
//       back to the rows it read, where the threads of the other fields find it.
//   B2  thread (b, i, f): w_f(k) = sum_J C_fJ rho_J at those k, and the first stage of its
//       two inverse lines conj(w), conj(-i k w) by the Stockham plan R2 x R1, whose first
//       stage (radix R2, no twiddles) reads exactly the values k = i + R1 q; exchange.
//   C   task (b, j < R2, line): twiddles w_N^{j r}, DFT_R1 -> rows j + R2 q; store.
//
// One field per thread in the middle stages: a thread that took every field (and one of
// the two inverse lines, so that two threads repeated the forward stage) issued 1.5 times
// the instructions and held up to 256 registers; the stage was the longest of the block
// (2.7 of 7.7 us on a 192-point film's 13 blocks, where it ran one wave per SIMD).
// The transforms and sums are those of the LDS-staged pass (whose inverse also runs the
// reversed plan RepDev::axr); the two agree to rounding, since the compiler contracts
// multiplies into the following additions differently where one keeps in registers
// what the other stages through LDS.
#pragma once
#include "device.hpp"
#include "fft_dev.hpp"
#include "fft_reg_dev.hpp"
#include "launch.hpp"

namespace tild {

namespace {

// One block: NB = last_reg_cols(R1, NF) adjacent columns q0 .. q0 + NB - 1 of the
// last-axis lines (fewer in the last block), TT types and CH charge fields (NF = TT + CH).
// LDS: the forward exchange (N x ldx), the inverse exchange (N x ldy), the inverse
// stage's twiddles, then the ramp weights (last_reg_lds_bytes).
template <int R1, int R2, int NT, int TT, int CH>
__device__ __forceinline__ void last_reg_block(const RepDev& r, int blk, float2* lds, int koff) {
    constexpr int N = R1 * R2, NF = TT + CH, NB = last_reg_cols(R1, NF);
    constexpr int ldx = NF * NB + 1, ldy = 2 * NF * NB + 1;
    constexpr int NT2 = R2 * (R1 - 1);
    static_assert(R2 <= R1 && NB * R1 * NF <= NT && NT2 <= NT, "k_last_reg: one middle-stage task per thread");
    const int la = r.dim - 1, D = r.dim;
    const int Q = la == 2 ? r.Ny * r.Nxh : r.Nxh;   // plane size = line stride
    const int q0 = blk * NB;
    const int nb = min(NB, Q - q0);
    float2* X1 = lds;                               // N x ldx: forward exchange
    float2* Y1 = lds + N * ldx;                     // N x ldy: inverse exchange
    float2* TW2 = Y1 + N * ldy;                     // w_N^{j r}, j < R2, 1 <= r < R1 (inverse stage 2)
    float* rw = (float*)(TW2 + NT2);                // ramp weights of this step
    // lanes: column, then field, then i (the fields' LDS rows are NB values apart, which
    // spreads a wave's accesses over the banks)
    const int b = (int)threadIdx.x % NB, f = ((int)threadIdx.x / NB) % NF, i = (int)threadIdx.x / (NB * NF);
    const bool live = b < nb && i < R1;
    // grid buffers below 4 GiB (required on the host): 32-bit element offsets
    const uint32_t Qu = (uint32_t)Q, Mhu = (uint32_t)r.Mh;

    // everything the block reads is requested before the first wait: this thread's rows
    // of the spectrum, its twiddles of both stages and its coupling rows
    float2 t2 = make_float2(0.f, 0.f);
    if ((int)threadIdx.x < NT2) t2 = gld(r.reg_twr + threadIdx.x);
    float2 v[R1];
    const bool liveA = b < nb && i < R2;
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
    float c[R2][TT];
    if (live) {
        const float2* tw1 = la == 2 ? r.reg_tw[2] : r.reg_tw[1];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) t1[rr] = gld(tw1 + (i * (R2 - 1) + rr - 1));
#pragma unroll
        for (int J = 0; J < TT; ++J) {
            const int row = isq ? r.ctab_charge : pidx(J);
#pragma unroll
            for (int q = 0; q < R2; ++q) c[q][J] = ctab(i + R1 * q, row);
        }
    }
    if ((int)threadIdx.x < r.nramp) rw[threadIdx.x] = ramp_weight(r, threadIdx.x, r.step + koff);

    // ---- A: DFT_R1 of rows i + R2 r (Stockham stage 1: out[i R1 + q])
    if (liveA) {
        Dft<R1>::run(v);
#pragma unroll
        for (int q = 0; q < R1; ++q) X1[(i * R1 + q) * ldx + f * NB + b] = v[q];
    }
    if ((int)threadIdx.x < NT2) TW2[threadIdx.x] = t2;
    __syncthreads();

    // ---- B1: stage 2 (radix R2, twiddles w_N^{i r}) -> rho_f(k), k = i + R1 q
    float2 w[R2];
    if (live) {
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = X1[(i + R1 * rr) * ldx + f * NB + b];
        // With four types or charges the twiddles count as read here: which of a sum's two products
        // the compiler fuses follows the order their operands are read in, and this order
        // keeps the rounding that such decks have had.
        if constexpr (TT == 4 || CH) {
#pragma unroll
            for (int rr = 1; rr < R2; ++rr) asm volatile("" : "+v"(t1[rr].x), "+v"(t1[rr].y));
        }
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) w[rr] = cmul(w[rr], t1[rr]);
        Dft<R2>::run(w);
        if constexpr (NF > 1) {
#pragma unroll
            for (int q = 0; q < R2; ++q) X1[(i + R1 * q) * ldx + f * NB + b] = w[q];
        }
    }
    if constexpr (NF > 1) __syncthreads();

    // ---- B2: coupling and the first stage of the two inverse lines
    if (live) {
        for (int j = 0; j < r.nramp; ++j) {   // ramped styles add their weighted rows (uniform trip count)
            const float wj = rw[j];
            const int rp = r.ramp_pair[j];
#pragma unroll
            for (int J = 0; J < TT; ++J) {
                const bool on = !isq && rp == pidx(J);
#pragma unroll
                for (int q = 0; q < R2; ++q) {
                    const float cr = wj * ctab(i + R1 * q, r.ramp_row0 + j);
                    c[q][J] += on ? cr : 0.f;
                }
            }
        }
        // w_f = sum_J C_fJ rho_J; charges w_c = G_c rho_c
#pragma unroll
        for (int q = 0; q < R2; ++q) {
            float2 acc = make_float2(0.f, 0.f);
#pragma unroll
            for (int J = 0; J < TT; ++J) {
                const float2 rh = NF > 1 ? X1[(i + R1 * q) * ldx + J * NB + b] : w[q];
                acc.x += c[q][J] * rh.x; acc.y += c[q][J] * rh.y;
            }
            w[q] = isq ? scaled(c[q][0], w[q]) : acc;
        }
        // the inverse is conj(FFT(conj)): conj(w) = (w.x, -w.y), then conj(-i k_la w) =
        // (k w.y, k w.x), k_la = 0 on the Nyquist plane; first stage of the R2 x R1 plan:
        // radix R2, out[i R2 + q]
        float2 z[R2];
#pragma unroll
        for (int q = 0; q < R2; ++q) z[q] = make_float2(w[q].x, -w[q].y);
        Dft<R2>::run(z);
#pragma unroll
        for (int q = 0; q < R2; ++q) Y1[(i * R2 + q) * ldy + f * NB + b] = z[q];
#pragma unroll
        for (int q = 0; q < R2; ++q) {
            const int n = i + R1 * q;
            const float kl = 2 * n == N ? 0.f : r.kfac[la] * (float)(2 * n < N ? n : n - N);
            z[q] = grad_line(kl, w[q]);
        }
        Dft<R2>::run(z);
#pragma unroll
        for (int q = 0; q < R2; ++q) Y1[(i * R2 + q) * ldy + (NF + f) * NB + b] = z[q];
    }
    __syncthreads();

    // ---- C: stage 2 of the R2 x R1 plan (radix R1, twiddles w_N^{j r}, including the
    // unit ones of j = 0 as the staged pass multiplies them) -> rows j + R2 q.  One task
    // per (column, line, j), spread over all threads.
    for (int task = threadIdx.x; task < NB * R2 * 2 * NF; task += NT) {
        const int bc = task % NB, rest = task / NB, line = rest % (2 * NF), j = rest / (2 * NF);   // line = o NF + f
        if (bc >= nb) continue;
        const int o = line >= NF ? 1 : 0, fl = line - o * NF;
        float2 z[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) z[rr] = Y1[(j + R2 * rr) * ldy + line * NB + bc];
#pragma unroll
        for (int rr = 1; rr < R1; ++rr) z[rr] = cmul(z[rr], TW2[j * (R1 - 1) + rr - 1]);
        Dft<R1>::run(z);
        const uint32_t o0 = (uint32_t)(fl * D + (o == 0 ? 0 : la)) * Mhu + (uint32_t)j * Qu + (uint32_t)(q0 + bc);
        const uint32_t step = (uint32_t)R2 * Qu;
#pragma unroll
        for (int q = 0; q < R1; ++q) gst(at32(r.Gk, o0 + (uint32_t)q * step), conjf2(z[q]));
    }
}

template <int R1, int R2, int NT, int TT, int CH, int CLS>
__device__ __forceinline__ void last_reg_variant_block(const RepDev& r, int blk, float2* lds, int koff) {
    if constexpr (last_reg_variant(R1, R2, TT, CH) && last_reg_class(R1, R2, TT) == CLS)
        last_reg_block<R1, R2, NT, TT, CH>(r, blk, lds, koff);
}

template <int R1, int R2, int NT, int CLS>
__device__ __forceinline__ void last_reg_types(const RepDev& r, int blk, float2* lds, int koff) {
    const bool ch = r.nf > r.ntypes;
    switch (r.ntypes * 2 + (ch ? 1 : 0)) {
        case 2: last_reg_variant_block<R1, R2, NT, 1, 0, CLS>(r, blk, lds, koff); break;
        case 3: last_reg_variant_block<R1, R2, NT, 1, 1, CLS>(r, blk, lds, koff); break;
        case 4: last_reg_variant_block<R1, R2, NT, 2, 0, CLS>(r, blk, lds, koff); break;
        case 5: last_reg_variant_block<R1, R2, NT, 2, 1, CLS>(r, blk, lds, koff); break;
        case 6: last_reg_variant_block<R1, R2, NT, 3, 0, CLS>(r, blk, lds, koff); break;
        case 7: last_reg_variant_block<R1, R2, NT, 3, 1, CLS>(r, blk, lds, koff); break;
        case 8: last_reg_variant_block<R1, R2, NT, 4, 0, CLS>(r, blk, lds, koff); break;
        case 9: last_reg_variant_block<R1, R2, NT, 4, 1, CLS>(r, blk, lds, koff); break;
        default: break;   // excluded by last_reg_plan on the host
    }
}

}  // namespace

// One instantiation per class of variants (last_reg_class), each compiled in a file of
// its own: a class's registers do not lower the occupancy of another's, and the classes
// compile side by side.
template <int NT, int CLS>
__global__ void __launch_bounds__(NT) k_last_reg(const RepDev* __restrict__ reps, const WorkItem* __restrict__ wmap,
                                                 int koff) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    warm_desc<0, 1, 6, 7>(r);
    switch (r.dim == 3 ? r.reg_key[2] : r.reg_key[1]) {   // uniform per block
#define TILD_CASE(A, B) case A * 32 + B: last_reg_types<A, B, NT, CLS>(r, wi.blk, lds, koff); break;
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
