// fft_last.hpp -- the fused last-axis pass with register-resident columns, k_last_reg
// (CDNA4 / gfx950), shared by the files that compile one class of its variants each.
//
// k_last_reg: the same operation as k_last_fused (kernels.hip) -- last-axis forward FFT of every
// field, the k-space coupling w_I = sum_J C_IJ rho_J (+ the charge row), and the
// inverse transforms of w and -i k_la w -- for last axes with a two-stage plan
// N = R1 R2 (TILD_REG_PLANS; R1 >= R2).  Each
// thread keeps its Stockham columns in registers between the stages, so a block makes
// two LDS exchanges and two barriers, where the LDS-staged form stages every value
// through LDS and ends each of its nine phases with a barrier:
//
//   A  task (b, i < R2, field): rows i + R2 r (r < R1) of column b, read from HBM
//      straight into registers; DFT_R1; exchange.
//   B  thread (b, i < R1, h < 2): twiddles w_N^{i r}, DFT_R2 -> rho_f(k) at
//      k = i + R1 q; the coupling in registers; inverse direction h (conj(w) or
//      conj(-i k w)) is transformed by the Stockham plan R2 x R1, whose first stage
//      (radix R2, no twiddles) reads exactly the values k = i + R1 q this thread holds;
//      exchange.
//   C  task (b, j < R2, line): twiddles w_N^{j r}, DFT_R1 -> rows j + R2 q; store.
//
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

// One block: NB = NT / (2 R1) adjacent columns q0 .. q0 + NB - 1 of the last-axis lines
// (fewer in the last block), TT types and CH charge fields (NF = TT + CH fields).  Two
// threads share each (column, i) of the middle stage: both run the forward stage and
// the coupling, and each transforms one of the two inverse directions.
// LDS: the forward exchange (N x ldx), the inverse exchange (N x ldy), both stages'
// twiddles, then the ramp weights (last_reg_lds_bytes).
template <int R1, int R2, int NT, int TT, int CH>
__device__ __forceinline__ void last_reg_block(const RepDev& r, int blk, float2* lds, int koff) {
    constexpr int N = R1 * R2, NF = TT + CH, NR = TT * (TT + 1) / 2, NB = NT / (2 * R1);
    constexpr int ldx = NF * NB + 1, ldy = 2 * NF * NB + 1;
    constexpr int NT1 = R1 * (R2 - 1), NT2 = R2 * (R1 - 1);
    const int la = r.dim - 1, D = r.dim;
    const int Q = la == 2 ? r.Ny * r.Nxh : r.Nxh;   // plane size = line stride
    const int q0 = blk * NB;
    const int nb = min(NB, Q - q0);
    float2* X1 = lds;                               // N x ldx: forward exchange
    float2* Y1 = lds + N * ldx;                     // N x ldy: inverse exchange
    float2* TW1 = Y1 + N * ldy;                     // w_N^{i r}, i < R1, 1 <= r < R2 (forward stage 2)
    float2* TW2 = TW1 + NT1;                        // w_N^{j r}, j < R2, 1 <= r < R1 (inverse stage 2)
    float* rw = (float*)(TW2 + NT2);                // ramp weights of this step
    // phase B: thread (b, i, h), h = the inverse direction it transforms
    const int b = (int)threadIdx.x % NB, i = ((int)threadIdx.x / NB) % R1, h = (int)threadIdx.x / (NB * R1);
    // grid buffers below 4 GiB (required on the host): 32-bit element offsets
    const uint32_t Qu = (uint32_t)Q, Mhu = (uint32_t)r.Mh;
    const bool liveB = h < 2 && b < nb;

    // set-up, visible after the first barrier: twiddles and ramp weights into LDS
    {
        const float2* tw1 = la == 2 ? r.reg_tw[2] : r.reg_tw[1];
        const float2* tw2 = r.reg_twr;
        for (int t = threadIdx.x; t < NT1; t += NT) TW1[t] = gld(tw1 + t);
        for (int t = threadIdx.x; t < NT2; t += NT) TW2[t] = gld(tw2 + t);
        if ((int)threadIdx.x < r.nramp) rw[threadIdx.x] = ramp_weight(r, threadIdx.x, r.step + koff);
    }
    // coupling rows of this thread's phase-B nodes, requested before anything else
    const int nrows = r.ctab_rows;
    // element (n, row) of this thread's column: cb0 + (n nrows + row) NB, from the
    // uniform table base (every offset 32-bit)
    const uint32_t cb0 = (uint32_t)blk * (uint32_t)(N * nrows * NB) + (uint32_t)b;
    auto ctab = [&](int n, int row) { return G(at32(r.Ctab, cb0 + (uint32_t)((n * nrows + row) * NB)))[0]; };
    // up to three types every row of the thread's nodes is requested at block start
    // and held through the forward stages; with four (ten rows per node) each node's
    // rows are requested where the coupling uses them, which keeps the pass within 256
    // registers
    constexpr bool kEarly = NR <= 6;
    constexpr int QE = kEarly ? R2 : 1;
    float c[QE][NR], cq[QE];
    auto load_rows = [&](int q, int slot) {
#pragma unroll
        for (int k = 0; k < NR; ++k) c[slot][k] = ctab(i + R1 * q, k);
        cq[slot] = CH ? ctab(i + R1 * q, r.ctab_charge) : 0.f;
    };
    if (kEarly && liveB) {
#pragma unroll
        for (int q = 0; q < R2; ++q) load_rows(q, q < QE ? q : 0);
    }

    // ---- A: task (b, i < R2, f): rows i + R2 r of field f, DFT_R1 (Stockham stage 1:
    // out[i R1 + q])
    // lanes: column, then field, then i (the fields' LDS rows are NB values apart,
    // which spreads a wave's writes over the banks)
    for (int task = threadIdx.x; task < NB * R2 * NF; task += NT) {
        const int ba = task % NB, f = (task / NB) % NF, ia = task / (NB * NF);
        if (ba >= nb) continue;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr)
            v[rr] = gld(at32((const float2*)r.H, (uint32_t)f * Mhu + (uint32_t)(ia + R2 * rr) * Qu + (uint32_t)(q0 + ba)));
        Dft<R1>::run(v);
#pragma unroll
        for (int q = 0; q < R1; ++q) X1[(ia * R1 + q) * ldx + f * NB + ba] = v[q];
    }
    __syncthreads();

    // ---- B: stage 2 (radix R2, twiddles w_N^{i r}) -> rho_f(k), k = i + R1 q
    if (liveB) {
        float2 w[NF][R2];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int rr = 0; rr < R2; ++rr) w[f][rr] = X1[(i + R1 * rr) * ldx + f * NB + b];
        float2 t[R2];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) t[rr] = TW1[i * (R2 - 1) + rr - 1];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
#pragma unroll
            for (int rr = 1; rr < R2; ++rr) w[f][rr] = cmul(w[f][rr], t[rr]);
            Dft<R2>::run(w[f]);
        }
        // coupling: w_I = sum_J C_IJ rho_J over the symmetric rows pidx(lo, hi) =
        // lo TT - lo (lo - 1) / 2 + (hi - lo); ramped styles add their weighted rows;
        // charges w_c = G_c rho_c
#pragma unroll
        for (int q = 0; q < R2; ++q) {
            const int n = i + R1 * q;
            const int cs = kEarly ? q : 0;     // slot of this node's rows
            if (!kEarly) load_rows(q, 0);
            for (int j = 0; j < r.nramp; ++j) {   // uniform trip count
                const float v = rw[j] * ctab(n, r.ramp_row0 + j);
#pragma unroll
                for (int k = 0; k < NR; ++k) c[cs][k] += r.ramp_pair[j] == k ? v : 0.f;
            }
            float2 rh[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) rh[f] = w[f][q];
#pragma unroll
            for (int I = 0; I < TT; ++I) {
                float2 acc = make_float2(0.f, 0.f);
#pragma unroll
                for (int J = 0; J < TT; ++J) {
                    const int lo = I < J ? I : J, hi = I < J ? J : I;
                    const float cc = c[cs][lo * TT - lo * (lo - 1) / 2 + (hi - lo)];
                    acc.x += cc * rh[J].x; acc.y += cc * rh[J].y;
                }
                w[I][q] = acc;
            }
            if (CH) w[TT][q] = scaled(cq[cs], rh[TT]);
        }
        // this thread's inverse lines (the inverse is conj(FFT(conj))): h = 0
        // conj(w) = (w.x, -w.y), h = 1 conj(-i k_la w) = (k w.y, k w.x), k_la = 0 on the
        // Nyquist plane; first stage of the R2 x R1 plan: radix R2, out[i R2 + q]
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            float2 z[R2];
#pragma unroll
            for (int q = 0; q < R2; ++q) {
                const int n = i + R1 * q;
                const float2 a = w[f][q];
                const float kl = 2 * n == N ? 0.f : r.kfac[la] * (float)(2 * n < N ? n : n - N);
                z[q] = h == 0 ? make_float2(a.x, -a.y) : grad_line(kl, a);
            }
            Dft<R2>::run(z);
#pragma unroll
            for (int q = 0; q < R2; ++q) Y1[(i * R2 + q) * ldy + (h * NF + f) * NB + b] = z[q];
        }
    }
    __syncthreads();

    // ---- C: stage 2 of the R2 x R1 plan (radix R1, twiddles w_N^{j r}, including the
    // unit ones of j = 0 as the staged pass multiplies them) -> rows j + R2 q.  One task
    // per (column, j, line), spread over all threads.
    // lanes: column, then line, then j (lines NB values apart in LDS: a wave's reads of
    // one row fall in distinct banks)
    for (int task = threadIdx.x; task < NB * R2 * 2 * NF; task += NT) {
        const int bc = task % NB, rest = task / NB, line = rest % (2 * NF), j = rest / (2 * NF);   // line = o NF + f
        if (bc >= nb) continue;
        const int o = line >= NF ? 1 : 0, f = line - o * NF;
        float2 z[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) z[rr] = Y1[(j + R2 * rr) * ldy + line * NB + bc];
#pragma unroll
        for (int rr = 1; rr < R1; ++rr) z[rr] = cmul(z[rr], TW2[j * (R1 - 1) + rr - 1]);
        Dft<R1>::run(z);
        const uint32_t o0 = (uint32_t)(f * D + (o == 0 ? 0 : la)) * Mhu + (uint32_t)j * Qu + (uint32_t)(q0 + bc);
        const uint32_t step = (uint32_t)R2 * Qu;
#pragma unroll
        for (int q = 0; q < R1; ++q) gst(at32(r.Gk, o0 + (uint32_t)q * step), conjf2(z[q]));
    }
}

template <int R1, int R2, int NT, int TT, int CH, int CLS>
__device__ __forceinline__ void last_reg_variant_block(const RepDev& r, int blk, float2* lds, int koff) {
    if constexpr (last_reg_variant(R1, R2, TT, CH) && last_reg_class(R1, TT) == CLS)
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
