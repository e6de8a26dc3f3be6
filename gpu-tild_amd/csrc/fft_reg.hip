// fft_reg.hip -- FFT passes of the step with register-resident columns (CDNA4 / gfx950):
// the forward plane pass (k_plane_reg), the y inverse of the gradient spectra
// (k_grad_reg), the inverse plane pass (k_plane_inv) and the inverse x transform into the
// gather records (k_c2r_reg); the fused last-axis pass is in fft_last.hpp, the x transform
// of the deposit in spread_tiled.hip.  Each takes axes with a plan of TILD_REG_PLANS, two
// groups of one or two Stockham stages; a thread keeps its columns in registers through a
// group, so a pass makes one to three LDS exchanges where the LDS-staged forms
// (kernels.hip) stage every value through LDS with a barrier after each phase.
#include "device.hpp"
#include "fft_dev.hpp"
#include "fft_reg_dev.hpp"
#include "launch.hpp"

namespace tild {

RegDims reg_dims(const AxisPlan& pl) {
    if (pl.nst < 2 || pl.nst > 4) return RegDims{0, 0, 0, 0};
    int key = pl.rad[0];
    for (int s = 1; s < pl.nst; ++s) key = key * 32 + pl.rad[s];
    switch (key) {
#define TILD_CASE(A0, A1, B0, B1) \
    case reg_plan_key(A0, A1, B0, B1): return RegDims{key, (A0) * (A1), (B0) * (B1), A1 > 1 ? 2 : 1};
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: return RegDims{0, 0, 0, 0};
    }
}

// ------------------------------------------------------------------ y inverse (3D)
// The y-axis inverse of the gradient spectra (the operation of k_mid_grad, kernels.hip)
// for y plans of groups R1 x R2, columns in registers between the groups: per (field,
// z) plane and NB = NT / max(R1, R2) adjacent x columns,
//   A  thread (b, i), i < R2: rows i + R2 r of U (slot 0) and V (slot 2), the three
//      lines conj(U), conj(-i k_y U), conj(V), first group; exchange;
//   B  thread (b, i), i < R1: second group -> rows i + R1 q of the three outputs (slots
//      0, 1, 2).
// One barrier; bound by its loads and stores (18.4 us LDS-staged, 9.4 here on 96^3).  A block reads its columns of slots 0 and 2 before it writes any slot,
// and no other block touches them.
namespace {
template <class P, int NT>
__device__ __forceinline__ void grad_reg_block(const RepDev& r, int blk, float2* lds) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N, NB = NT / P::RM, ld = 3 * NB + 1;
    const int Nxh = r.Nxh;
    const int nchunk = (Nxh + NB - 1) / NB;
    const int o = blk / nchunk, c = blk - o * nchunk;   // o = f Nz + z
    const int f = o / r.Nz, z = o - f * r.Nz;
    const int b0 = c * NB, nb = min(NB, Nxh - b0);
    float2* X1 = lds;                 // N x ld
    float2* TW1 = X1 + N * ld;        // the second group's twiddles
    const int b = (int)threadIdx.x % NB, i = (int)threadIdx.x / NB;
    const float2* const tw = r.reg_tw[1];
    for (int t = threadIdx.x; t < P::NTW; t += NT) TW1[t] = gld(tw + t);
    // element (n, column b) of slot s: 32-bit offsets from the uniform base
    const uint32_t Mhu = (uint32_t)r.Mh, Nxu = (uint32_t)Nxh;
    const uint32_t plane = (uint32_t)z * (uint32_t)N * Nxu + (uint32_t)(b0 + b);
    const uint32_t sU = (uint32_t)(f * 3 + 0) * Mhu + plane, sY = (uint32_t)(f * 3 + 1) * Mhu + plane,
                   sV = (uint32_t)(f * 3 + 2) * Mhu + plane;
    if (i < R2 && b < nb) {
        float2 u[R1], v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const uint32_t n = (uint32_t)(i + R2 * rr) * Nxu;
            u[rr] = gld(at32((const float2*)r.Gk, sU + n));
            v[rr] = gld(at32((const float2*)r.Gk, sV + n));
        }
        float2 L[3][R1];
        const float fi = (float)i;
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const float ky = r.kfac[1] * freq_of<R2, N>(i, fi, rr);
            // lines of the conj(FFT(conj)) inverse: conj(u), conj(-i ky u), conj(v)
            L[0][rr] = make_float2(u[rr].x, -u[rr].y);
            L[1][rr] = grad_line(ky, u[rr]);
            L[2][rr] = make_float2(v[rr].x, -v[rr].y);
        }
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            plan_first<P>(L[l], tw);
#pragma unroll
            for (int q = 0; q < R1; ++q) X1[(i * R1 + q) * ld + l * NB + b] = L[l][q];
        }
    }
    __syncthreads();
    if (i < R1 && b < nb) {
        float2 t[R2];
#pragma unroll
        for (int m = 1; m < R2; ++m) t[m] = TW1[tw2_index<P>(i, m)];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            float2 w[R2];
#pragma unroll
            for (int rr = 0; rr < R2; ++rr) w[rr] = X1[(i + R1 * rr) * ld + l * NB + b];
            plan_second<P, true>(w, [&](int m) { return t[m]; });
            const uint32_t s0 = l == 0 ? sU : (l == 1 ? sY : sV);
#pragma unroll
            for (int q = 0; q < R2; ++q)
                gst(at32(r.Gk, s0 + (uint32_t)(i + R1 * q) * Nxu), conjf2(w[q]));
        }
    }
}

}  // namespace

// ALL: some replica of the set has a grouped y plan; without them 121 registers and four waves
// per SIMD, with them 210 and two (y of 80 points, 160 x 80 x 80: 9.6 us, and 11.5 in the
// kernel of all plans; 128^3: 21 and 24).
template <int NT, bool ALL>
__global__ void __launch_bounds__(NT) k_grad_reg(const RepDev* __restrict__ reps, const WorkItem* __restrict__ wmap) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    warm_desc<0, 1, 6, 7>(r);
    switch (r.reg_key[1]) {   // uniform per block
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr ((A0) * (A1) <= 16 && (ALL || !reg_plan_grouped(A1, B1)))     \
            grad_reg_block<RegPlan<A0, A1, B0, B1>, NT>(r, wi.blk, lds);           \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by grad_reg_plan on the host
    }
}

// ------------------------------------------------------------------ plane forward (3D)
// x R2C and y FFT of one (field, z) density plane (the operation of k_plane_r2c,
// kernels.hip) for even square planes Nx = Ny with a kept two-stage plan R1 x R2:
//   A  task (pair j, i < R2): rows 2j and 2j+1 at x = i + R2 r as one complex line, DFT_R1;
//   B  task (j, i < R1): twiddles, DFT_R2 -> Z_j(k), k = i + R1 q; exchange;
//   C  task (column k < Nxh, i < R2): the half spectra of rows y = i + R2 r unpacked on
//      the fly from Z_{y/2}(k) and Z_{y/2}(N - k), DFT_R1;
//   D  task (k, i < R1): twiddles, DFT_R2 -> H(y = i + R1 q, k), stored.
// Three barriers, where the staged pass has seven; loads and stores go straight to and
// from registers.
namespace {
template <int R1, int R2, int NT>
__device__ __forceinline__ void plane_reg_block(const RepDev& r, int blk, float2* lds) {
    constexpr int N = R1 * R2, NP = N / 2, NXH = N / 2 + 1, ldp = NP | 1, ldc = NXH | 1;
    constexpr int NT1 = R1 * (R2 - 1), LDA = (N * ldp > N * ldc) ? N * ldp : N * ldc;
    const int z = blk % r.Nz, f = blk / r.Nz;
    float2* Xa = lds;                  // x stage-1 output, later the y stage-1 output (N x ldc)
    float2* Xb = Xa + LDA;             // Z: x transforms of the row pairs (N x ldp)
    float2* TWx = Xb + N * ldp;        // w_N^{i r} of the x plan and of the y plan
    float2* TWy = TWx + NT1;
    {
        const float2* tx = r.reg_tw[0];
        const float2* ty = r.reg_tw[1];
        for (int t = threadIdx.x; t < NT1; t += NT) { TWx[t] = gld(tx + t); TWy[t] = gld(ty + t); }
    }
    const uint32_t pbase = (uint32_t)f * (uint32_t)r.M + (uint32_t)z * (uint32_t)(N * N);
    // A: pairs of rows as complex lines, stage 1 of the x plan
    for (int task = threadIdx.x; task < NP * R2; task += NT) {
        const int i = task % R2, j = task / R2;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const uint32_t o = pbase + (uint32_t)(2 * j * N + i + R2 * rr);
            v[rr] = make_float2(G(at32((const float*)r.rho, o))[0], G(at32((const float*)r.rho, o + N))[0]);
        }
        Dft<R1>::run(v);
#pragma unroll
        for (int q = 0; q < R1; ++q) Xa[(i * R1 + q) * ldp + j] = v[q];
    }
    __syncthreads();
    // B: stage 2 of the x plan -> Z_j(k)
    for (int task = threadIdx.x; task < NP * R1; task += NT) {
        const int i = task % R1, j = task / R1;
        float2 v[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) v[rr] = Xa[(i + R1 * rr) * ldp + j];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) v[rr] = cmul_kept(v[rr], TWx[i * (R2 - 1) + rr - 1]);
        Dft<R2>::run(v);
#pragma unroll
        for (int q = 0; q < R2; ++q) Xb[(i + R1 * q) * ldp + j] = v[q];
    }
    __syncthreads();
    // C: unpack rows y = i + R2 r of column k (even y: the real row's spectrum
    // (Z_k + conj Z_{N-k}) / 2, odd y: the imaginary row's (Z_k - conj Z_{N-k}) / 2i),
    // stage 1 of the y plan
    for (int task = threadIdx.x; task < NXH * R2; task += NT) {
        const int k = task % NXH, i = task / NXH;
        const int km = k == 0 ? 0 : N - k;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const int y = i + R2 * rr, j = y >> 1;
            const float2 Zk = Xb[k * ldp + j], Zm = Xb[km * ldp + j];
            v[rr] = (y & 1) == 0 ? make_float2(half_of(Zk.x + Zm.x), half_of(Zk.y - Zm.y))
                                 : make_float2(half_of(Zk.y + Zm.y), half_of(Zm.x - Zk.x));
        }
        Dft<R1>::run(v);
#pragma unroll
        for (int q = 0; q < R1; ++q) Xa[(i * R1 + q) * ldc + k] = v[q];
    }
    __syncthreads();
    // D: stage 2 of the y plan -> H(y, k)
    const uint32_t hbase = ((uint32_t)f * (uint32_t)r.Nz + (uint32_t)z) * (uint32_t)(N * NXH);
    for (int task = threadIdx.x; task < NXH * R1; task += NT) {
        const int k = task % NXH, i = task / NXH;
        float2 v[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) v[rr] = Xa[(i + R1 * rr) * ldc + k];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) v[rr] = cmul_kept(v[rr], TWy[i * (R2 - 1) + rr - 1]);
        Dft<R2>::run(v);
#pragma unroll
        for (int q = 0; q < R2; ++q) gst(at32(r.H, hbase + (uint32_t)((i + R1 * q) * NXH + k)), v[q]);
    }
}
}  // namespace

// The same for any even plane of compiled plans (sides of equal or unequal plans): the x
// phases compiled per x plan, the y phases per y plan, bit for bit the LDS-staged pass.
namespace {
template <class P, int NT>
__device__ __forceinline__ void plane_rect_x(const RepDev& r, uint32_t pbase, float2* Xa, float2* Xb, const float2* TW) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N;
    const int np = r.Ny / 2, ldp = np | 1;
    const float2* const tw = r.reg_tw[0];
    // A: pairs of rows as complex lines, first group of the x plan
    for (int task = threadIdx.x; task < np * R2; task += NT) {
        const int i = task % R2, j = task / R2;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const uint32_t o = pbase + (uint32_t)(2 * j * N + i + R2 * rr);
            v[rr] = make_float2(G(at32((const float*)r.rho, o))[0], G(at32((const float*)r.rho, o + N))[0]);
        }
        plan_first<P>(v, tw);
#pragma unroll
        for (int q = 0; q < R1; ++q) Xa[(i * R1 + q) * ldp + j] = v[q];
    }
    __syncthreads();
    // B: second group -> Z_j(k)
    const FastDiv dnp(np);
    for (int task = threadIdx.x; task < np * R1; task += NT) {
        int j;
        const int i = dnp.div(task, j);
        float2 v[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) v[rr] = Xa[(i + R1 * rr) * ldp + j];
        plan_second_lds<P, true>(v, TW, i);
#pragma unroll
        for (int q = 0; q < R2; ++q) Xb[(i + R1 * q) * ldp + j] = v[q];
    }
    __syncthreads();
}

template <class P, int NT>
__device__ __forceinline__ void plane_rect_y(const RepDev& r, uint32_t hbase, float2* Xa, const float2* Xb, const float2* TW) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N;
    const int Nx = r.Nx, nxh = r.Nxh, ldp = (N / 2) | 1, ldc = nxh | 1;
    const float2* const tw = r.reg_tw[1];
    const FastDiv dnx(nxh);
    // C: unpack rows y = i + R2 r of column k, first group of the y plan
    for (int task = threadIdx.x; task < nxh * R2; task += NT) {
        int k;
        const int i = dnx.div(task, k);
        const int km = k == 0 ? 0 : Nx - k;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const int y = i + R2 * rr, j = y >> 1;
            const float2 Zk = Xb[k * ldp + j], Zm = Xb[km * ldp + j];
            v[rr] = (y & 1) == 0 ? make_float2(half_of(Zk.x + Zm.x), half_of(Zk.y - Zm.y))
                                 : make_float2(half_of(Zk.y + Zm.y), half_of(Zm.x - Zk.x));
        }
        plan_first<P>(v, tw);
#pragma unroll
        for (int q = 0; q < R1; ++q) Xa[(i * R1 + q) * ldc + k] = v[q];
    }
    __syncthreads();
    // D: second group -> H(y, k)
    for (int task = threadIdx.x; task < nxh * R1; task += NT) {
        int k;
        const int i = dnx.div(task, k);
        float2 v[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) v[rr] = Xa[(i + R1 * rr) * ldc + k];
        plan_second_lds<P, true>(v, TW, i);
#pragma unroll
        for (int q = 0; q < R2; ++q) gst(at32(r.H, hbase + (uint32_t)((i + R1 * q) * nxh + k)), v[q]);
    }
}

template <int NT>
__device__ __forceinline__ void plane_rect_block(const RepDev& r, int blk, float2* lds) {
    const int Nx = r.Nx, Ny = r.Ny, nxh = r.Nxh, ldp = (Ny / 2) | 1, ldc = nxh | 1;
    const int z = blk % r.Nz, f = blk / r.Nz;
    float2* Xa = lds;                                   // x first-group output, later the y one
    float2* Xb = Xa + max(Nx * ldp, Ny * ldc);          // Z: x transforms of the row pairs
    float2* TWx = Xb + Nx * ldp;
    float2* TWy = TWx + Nx;
    // second groups' twiddles: fewer than N of each (N - R1), visible after the first barrier
    {
        const int nx = reg_ntw(r.reg_key[0], Nx), ny = reg_ntw(r.reg_key[1], Ny);
        for (int t = threadIdx.x; t < nx; t += NT) TWx[t] = gld(r.reg_tw[0] + t);
        for (int t = threadIdx.x; t < ny; t += NT) TWy[t] = gld(r.reg_tw[1] + t);
    }
    const uint32_t pbase = (uint32_t)f * (uint32_t)r.M + (uint32_t)z * (uint32_t)(Nx * Ny);
    const uint32_t hbase = ((uint32_t)f * (uint32_t)r.Nz + (uint32_t)z) * (uint32_t)(Ny * nxh);
    switch (r.reg_key[0]) {   // uniform per block
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr ((A0) * (A1) <= 16 && (B0) * (B1) <= 16) plane_rect_x<RegPlan<A0, A1, B0, B1>, NT>(r, pbase, Xa, Xb, TWx); \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by plane_rect_plan on the host
    }
    switch (r.reg_key[1]) {
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr ((A0) * (A1) <= 16 && (B0) * (B1) <= 16) plane_rect_y<RegPlan<A0, A1, B0, B1>, NT>(r, hbase, Xa, Xb, TWy); \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;
    }
}

// Forward y FFT of the half spectra of a (field, z) plane's columns in place (the operation
// of k_mid, kernels.hip), where the deposit transforms x (odd sides): kYfwdThreads threads
// take NB columns, so that a block takes several such pieces; live: the piece exists.
template <class P>
__device__ __forceinline__ void yfwd_piece(const RepDev& r, int piece, bool live, float2* lds) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N, NB = kYfwdThreads / P::RM, ld = NB + 1;
    const int Nxh = r.Nxh, nchunk = (Nxh + NB - 1) / NB;
    const int o = piece / nchunk, c = piece - o * nchunk;   // o = f Nz + z
    const int b0 = c * NB, nb = live ? min(NB, Nxh - b0) : 0;
    float2* X1 = lds;                 // N x ld
    float2* TW1 = X1 + N * ld;
    const int tid = (int)threadIdx.x % kYfwdThreads, b = tid % NB, i = tid / NB;
    const float2* const tw = r.reg_tw[1];
    const uint32_t Nxu = (uint32_t)Nxh, s0 = (uint32_t)o * (uint32_t)N * Nxu + (uint32_t)(b0 + b);
    float2 v[R1];
    if (i < R2 && b < nb) {
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) v[rr] = gld(at32((const float2*)r.H, s0 + (uint32_t)(i + R2 * rr) * Nxu));
    }
    for (int t = tid; t < P::NTW; t += kYfwdThreads) TW1[t] = gld(tw + t);
    if (i < R2 && b < nb) {
        plan_first<P>(v, tw);
#pragma unroll
        for (int q = 0; q < R1; ++q) X1[(i * R1 + q) * ld + b] = v[q];
    }
    __syncthreads();
    if (i < R1 && b < nb) {
        float2 w[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = X1[(i + R1 * rr) * ld + b];
        plan_second_lds<P, true>(w, TW1, i);
#pragma unroll
        for (int q = 0; q < R2; ++q) gst(at32(r.H, s0 + (uint32_t)(i + R1 * q) * Nxu), w[q]);
    }
}
}  // namespace

// ANY: some replica of the set takes one of the two other forms; without them the kernel
// holds the kept squares only, and its registers (74 against 89, three blocks to a CU
// against two).  One launch for the forms: the sweep of 24 replicas spends 11.7 us a step
// here, and 19.3 with a launch for each.
template <int NT, bool ANY>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) k_plane_reg(const RepDev* __restrict__ reps,
                                                                                        const WorkItem* __restrict__ wmap) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    if (ANY) warm_desc<0, 1, 6, 7, 8>(r);
    else warm_desc<0, 1, 6, 7>(r);
    if constexpr (ANY) {   // uniform per block, like the switches
        if (r.plane_rect) {
            plane_rect_block<NT>(r, wi.blk, lds);
            return;
        }
        if (r.yfwd_reg) {
            const int sub = (int)threadIdx.x / kYfwdThreads, piece = wi.blk * (NT / kYfwdThreads) + sub;
            switch (r.reg_key[1]) {
#define TILD_CASE(A0, A1, B0, B1)                                                                    \
    case reg_plan_key(A0, A1, B0, B1):                                                               \
        if constexpr ((A0) * (A1) <= 16 && (B0) * (B1) <= 16) {                                      \
            using P = RegPlan<A0, A1, B0, B1>;                                                       \
            constexpr int NB = kYfwdThreads / P::RM, elems = P::N * (NB + 2);                        \
            yfwd_piece<P>(r, piece, piece < r.nf * r.Nz * ((r.Nxh + NB - 1) / NB), lds + sub * elems); \
        }                                                                                            \
        break;
                TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
                default: break;   // excluded by yfwd_reg_plan on the host
            }
            return;
        }
    }
    switch (r.reg_key[0]) {
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr (reg_plan_kept(A0 * A1 * B0 * B1) && A0 * B0 % 2 == 0 && A0 * B0 <= 128) plane_reg_block<A0, B0, NT>(r, wi.blk, lds); \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by plane_reg_plan on the host
    }
}

// ------------------------------------------------------------------ plane inverse (3D)
// The y inverse of the gradient spectra and the x C2R into gather records of one
// (field, z) plane in one block (the operations of k_grad_reg and k_x_c2r, kernels.hip,
// without the half spectra of the y inverses going through HBM), for square planes
// Nx = Ny = N with a kept two-stage plan R1 x R2 (an odd N pairs its last row's z derivative
// with an all-zero line):
//   A  task (column k < N/2 + 1, i < R2): rows i + R2 r of U and V (slots 0 and 2),
//      the lines conj(U), conj(-i k_y U), conj(V), DFT_R1;
//   B  task (k, i < R1): twiddles, DFT_R2 -> the y inverses Y_l(y, k), y = i + R1 q,
//      written back over the rows the task read;
//   C  task (x line c, i < R2): the complex lines of the x inverse -- per row y the
//      x derivative (-i k_x applied) plus i times the y derivative, per row pair the
//      z derivatives of rows 2p and 2p + 1 -- extended to the full spectrum by
//      Hermitian symmetry at k = i + R2 r, DFT_R1; held across a barrier, then written
//      over the y inverses;
//   D  task (c, i < R1): twiddles, DFT_R2 -> the real lines at x = i + R1 q, held
//      across a barrier, then laid out as the plane's records in LDS and copied out.
// Six barriers; the y and x transforms and the conjugation and Hermitian rules are
// those of the two staged passes, which the records match to rounding (the x lines
// pair components differently).  Records carry no density mask (see k_x_c2r).
namespace {
template <int R1, int R2, int NT>
__device__ __forceinline__ void plane_inv_block(const RepDev& r, int blk, float2* lds) {
    constexpr int N = R1 * R2, NXH = N / 2 + 1, NT1 = R1 * (R2 - 1);
    constexpr int LA = (3 * NXH) | 1;          // row stride of the y inverses: [y][line][k]
    constexpr int NCL = N + (N + 1) / 2;       // x lines: N rows + the row pairs
    constexpr int LC = NCL | 1;                // row stride of the x exchange
    constexpr int CT = (NCL * R2 + NT - 1) / NT;   // stage C tasks per thread
    constexpr int DT = (NCL * R1 + NT - 1) / NT;   // stage D tasks per thread
    static_assert(LC <= LA && 3 * N * N <= 2 * N * LA, "plane_inv_block: exchange and records within the y buffer");
    const int z = blk % r.Nz, f = blk / r.Nz;
    float2* X = lds;                   // N x LA: y stages, then the x exchange (N x LC)
    float2* TW = X + N * LA;           // w_N^{i r}, i < R1, 1 <= r < R2 (same plan on x and y)
    {
        const float2* tw = r.reg_tw[1];
        for (int t = threadIdx.x; t < NT1; t += NT) TW[t] = gld(tw + t);
    }
    const uint32_t Mhu = (uint32_t)r.Mh;
    const uint32_t plane = (uint32_t)z * (uint32_t)(N * NXH);
    const uint32_t sU = (uint32_t)(f * 3 + 0) * Mhu + plane, sV = (uint32_t)(f * 3 + 2) * Mhu + plane;
    const float kfy = r.kfac[1], kfx = r.kfac[0];
    // A: y stage 1 of the three lines of column k
    for (int task = threadIdx.x; task < NXH * R2; task += NT) {
        const int k = task % NXH, i = task / NXH;
        float2 u[R1], v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const uint32_t o = (uint32_t)((i + R2 * rr) * NXH + k);
            u[rr] = gld(at32((const float2*)r.Gk, sU + o));
            v[rr] = gld(at32((const float2*)r.Gk, sV + o));
        }
        float2 L[3][R1];
        const float fi = (float)i;
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const float ky = kfy * freq_of<R2, N>(i, fi, rr);
            // lines of the conj(FFT(conj)) inverse: conj(u), conj(-i ky u), conj(v)
            L[0][rr] = make_float2(u[rr].x, -u[rr].y);
            L[1][rr] = grad_line(ky, u[rr]);
            L[2][rr] = make_float2(v[rr].x, -v[rr].y);
        }
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            Dft<R1>::run(L[l]);
#pragma unroll
            for (int q = 0; q < R1; ++q) X[(i * R1 + q) * LA + l * NXH + k] = L[l][q];
        }
    }
    __syncthreads();
    // B: y stage 2; Y_l(y, k) = conj of the result, over the rows the task read
    for (int task = threadIdx.x; task < NXH * R1; task += NT) {
        const int k = task % NXH, i = task / NXH;
        float2 t[R2];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) t[rr] = TW[i * (R2 - 1) + rr - 1];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            float2 w[R2];
#pragma unroll
            for (int rr = 0; rr < R2; ++rr) w[rr] = X[(i + R1 * rr) * LA + l * NXH + k];
#pragma unroll
            for (int rr = 1; rr < R2; ++rr) w[rr] = cmul(w[rr], t[rr]);
            Dft<R2>::run(w);
#pragma unroll
            for (int q = 0; q < R2; ++q) X[(i + R1 * q) * LA + l * NXH + k] = conjf2(w[q]);
        }
    }
    __syncthreads();
    // C: x stage 1.  Line c < N is row y = c: A = -i k_x Y_0, B = Y_1; line N + p pairs
    // A = Y_2(2p), B = Y_2(2p + 1).  Z = A + i B with Z_{N-k} = conj A_k + i conj B_k;
    // the self-conjugate columns (0, N/2) drop their imaginary parts; conj(Z) is
    // transformed (the inverse as conj(FFT(conj))).
    float2 hold[CT][R1];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int task = (int)threadIdx.x + ct * NT;
        if (task >= NCL * R2) break;
        const int c = task % NCL, i = task / NCL;
        const bool rowline = c < N;
        const int ya = rowline ? c : 2 * (c - N), yb = rowline ? c : ya + 1;
        const int la = rowline ? 0 : 2, lb = rowline ? 1 : 2;
        const float fi = (float)i;
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const HalfEntry e = half_entry<R2, N>(i, fi, rr);   // of the full-spectrum index
            float2 A = X[ya * LA + la * NXH + e.kk];
            float2 B = yb < N ? X[yb * LA + lb * NXH + e.kk] : make_float2(0.f, 0.f);
            if (rowline) {   // the x derivative: -i k_x (0 on the Nyquist column)
                const float kx = kfx * e.k;
                A = make_float2(kx * A.y, -kx * A.x);
            }
            if (e.self) { A.y = 0.f; B.y = 0.f; }
            hold[ct][rr] = e.upper ? make_float2(A.x + B.y, A.y - B.x) : make_float2(A.x - B.y, -(A.y + B.x));
        }
        Dft<R1>::run(hold[ct]);
    }
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int task = (int)threadIdx.x + ct * NT;
        if (task >= NCL * R2) break;
        const int c = task % NCL, i = task / NCL;
#pragma unroll
        for (int q = 0; q < R1; ++q) X[(i * R1 + q) * LC + c] = hold[ct][q];
    }
    __syncthreads();
    // D: x stage 2 -> the real lines A = res.x, B = -res.y at x = i + R1 q, held across
    // a barrier and laid out as the plane's records [y][x](g_x, g_y, g_z) over the
    // exchange; the plane's records are one contiguous run of HBM, copied out in 16-byte
    // pieces
    float2 out[DT][R2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int task = (int)threadIdx.x + dt * NT;
        if (task >= NCL * R1) break;
        const int i = task % R1, c = task / R1;   // adjacent lanes: adjacent x
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) out[dt][rr] = X[(i + R1 * rr) * LC + c];
#pragma unroll
        for (int rr = 1; rr < R2; ++rr) out[dt][rr] = cmul(out[dt][rr], TW[i * (R2 - 1) + rr - 1]);
        Dft<R2>::run(out[dt]);
    }
    __syncthreads();
    float* rec = (float*)X;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int task = (int)threadIdx.x + dt * NT;
        if (task >= NCL * R1) break;
        const int i = task % R1, c = task / R1;   // adjacent lanes: adjacent x
#pragma unroll
        for (int q = 0; q < R2; ++q) {
            const int x = i + R1 * q;
            if (c < N) {   // row y = c: (g_x, g_y)
                rec[(c * N + x) * 3 + 0] = out[dt][q].x;
                rec[(c * N + x) * 3 + 1] = -out[dt][q].y;
            } else {       // rows 2p and 2p + 1: g_z
                const int y0 = 2 * (c - N);
                rec[(y0 * N + x) * 3 + 2] = out[dt][q].x;
                if (y0 + 1 < N) rec[((y0 + 1) * N + x) * 3 + 2] = -out[dt][q].y;
            }
        }
    }
    __syncthreads();
    const uint32_t rec0 = (uint32_t)f * (uint32_t)r.M + (uint32_t)z * (uint32_t)(N * N);
    if constexpr (N % 2 == 0) {   // 12 rec0 bytes, 16-byte aligned
        float4* dst = (float4*)((char*)r.G3 + ((rec0 << 3) + (rec0 << 2)));
        const float4* src = (const float4*)rec;
        for (int t = threadIdx.x; t < 3 * N * N / 4; t += NT) gst(dst + t, src[t]);
    } else {
        float* dst = (float*)((char*)r.G3 + ((rec0 << 3) + (rec0 << 2)));
        for (int t = threadIdx.x; t < 3 * N * N; t += NT) G(dst)[t] = rec[t];
    }
}
}  // namespace

// The inverse plane pass of any other plane of compiled plans, bit for bit the y inverse
// and the x pass it stands for.  That x pass takes the real lines of a row (line f 3 + d of
// field f's component d) two to a complex line, so a block takes one such pair of lines of
// a z plane (more where that leaves threads idle, plane_pairs): their y inverses over the
// plane's columns, the paired x transform of its rows, and their components of the records.
// One pair of 96 x 96 points fits half a CU's LDS where a field's three lines do not.
// Bound by instruction issue on few waves (96 x 96: 2,700 a wave, two waves per SIMD):
// 96^3 22.8 us and 45 x 36 x 60 6.8 where the y inverse and the x pass took 26.8 and 9.2.
namespace {
template <class P, int NT>
__device__ __forceinline__ void plane_pair_y(const RepDev& r, int z, int l0, int nl, int la, float2* X, const float2* TW) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N;
    const int nxh = r.Nxh;   // rows: [line][k]
    const float2* const tw = r.reg_tw[1];
    const uint32_t Mhu = (uint32_t)r.Mh, plane = (uint32_t)z * (uint32_t)(N * nxh);
    const FastDiv dnx(nxh);
    // A: first group of column k of line l0 + s
    for (int task = threadIdx.x; task < nl * nxh * R2; task += NT) {
        int k;
        const int rest = dnx.div(task, k), i = rest % R2, s = rest / R2;
        const int l = l0 + s, f = l / 3, d = l - 3 * f;
        const uint32_t src = (uint32_t)(f * 3 + (d == 2 ? 2 : 0)) * Mhu + plane + (uint32_t)k;
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) v[rr] = gld(at32((const float2*)r.Gk, src + (uint32_t)((i + R2 * rr) * nxh)));
        const float fi = (float)i;
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            // lines of the conj(FFT(conj)) inverse: conj(u), conj(-i ky u), conj(v)
            v[rr] = pick(d == 1, grad_line(r.kfac[1] * freq_of<R2, N>(i, fi, rr), v[rr]), make_float2(v[rr].x, -v[rr].y));
        }
        plan_first<P>(v, tw);
#pragma unroll
        for (int q = 0; q < R1; ++q) X[(i * R1 + q) * la + s * nxh + k] = v[q];
    }
    __syncthreads();
    // B: second group over the rows the task read; conj of the result
    for (int task = threadIdx.x; task < nl * nxh * R1; task += NT) {
        int k;
        const int rest = dnx.div(task, k), i = rest % R1, s = rest / R1;
        float2* Xc = X + s * nxh + k;
        float2 w[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = Xc[(i + R1 * rr) * la];
        plan_second_lds<P, true>(w, TW, i);
#pragma unroll
        for (int q = 0; q < R2; ++q) Xc[(i + R1 * q) * la] = conjf2(w[q]);
    }
    __syncthreads();
}

template <class P, int NT>
__device__ __forceinline__ void plane_pair_x(const RepDev& r, int z, int l0, int nl, int la, float2* X, const float2* TW) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N, NXH = N / 2 + 1;
    constexpr int CT = plane_pair_hold(R1);      // tasks of a thread
    const int ny = r.Ny, np = (nl + 1) / 2, ncl = ny * np, lc = ncl | 1;   // complex lines (row y, pair j)
    const float2* const tw = r.reg_tw[0];
    const float kf = r.kfac[0];
    const FastDiv dncl(ncl), dnp(np);
    // C: first group of line c, held across a barrier: the exchange takes the rows' place
    float2 hold[CT][R1];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int task = (int)threadIdx.x + ct * NT;
        if (task >= ncl * R2) break;
        int c, j;
        const int i = dncl.div(task, c), y = dnp.div(c, j);
        const int la0 = l0 + 2 * j, d0 = la0 - 3 * (la0 / 3), d1 = d0 == 2 ? 0 : d0 + 1;
        const bool two = 2 * j + 1 < nl;
        const float2* ra = X + y * la + 2 * j * NXH;
        const float2* rb = ra + (two ? NXH : 0);
        const float fi = (float)i;
        float2 a[R1], b[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const int kk = half_entry<R2, N>(i, fi, rr).kk;
            a[rr] = ra[kk];
            b[rr] = rb[kk];
        }
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const HalfEntry e = half_entry<R2, N>(i, fi, rr);   // of the full-spectrum index
            const float kx = kf * e.k;
            float2 A = pick(d0 == 0, x_gradient(kx, a[rr]), a[rr]), B = pick(d1 == 0, x_gradient(kx, b[rr]), b[rr]);
            if (!two) B = make_float2(0.f, 0.f);
            if (e.self) { A.y = 0.f; B.y = 0.f; }
            hold[ct][rr] = e.upper ? make_float2(A.x + B.y, A.y - B.x) : make_float2(A.x - B.y, -(A.y + B.x));
        }
        plan_first<P>(hold[ct], tw);
        settle<R1>(hold[ct]);
    }
    __syncthreads();
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int task = (int)threadIdx.x + ct * NT;
        if (task >= ncl * R2) break;
        int c;
        const int i = dncl.div(task, c);
#pragma unroll
        for (int q = 0; q < R1; ++q) X[(i * R1 + q) * lc + c] = hold[ct][q];
    }
    __syncthreads();
    // D: second group -> the pairs' components of the records at x = i + R1 q (adjacent
    // lanes: adjacent x)
    const uint32_t M3 = 3u * (uint32_t)r.M, base = 3u * (uint32_t)(z * N * ny);
    for (int task = threadIdx.x; task < ncl * R1; task += NT) {
        const int i = task % R1, c = task / R1;
        int j;
        const int y = dnp.div(c, j);
        const int la0 = l0 + 2 * j, f0 = la0 / 3, d0 = la0 - 3 * f0;
        float2 w[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = X[(i + R1 * rr) * lc + c];
        plan_second_lds<P, true>(w, TW, i);
        settle<R2>(w);
        const uint32_t o = base + 3u * (uint32_t)(y * N + i) + (uint32_t)f0 * M3;
        const uint32_t p0 = o + (uint32_t)d0, p1 = d0 == 2 ? o + M3 : p0 + 1;
#pragma unroll
        for (int q = 0; q < R2; ++q) G(at32((float*)r.G3, p0 + 3u * R1 * q))[0] = w[q].x;
        if (2 * j + 1 < nl) {
#pragma unroll
            for (int q = 0; q < R2; ++q) G(at32((float*)r.G3, p1 + 3u * R1 * q))[0] = -w[q].y;
        }
    }
}

template <int NT>
__device__ __forceinline__ void plane_pair_block(const RepDev& r, int blk, float2* lds) {
    const int nlines = 3 * r.nf, per = 2 * r.plane_pair, nb = (nlines + per - 1) / per;
    const int z = blk / nb, l0 = per * (blk - z * nb), nl = min(per, nlines - l0), la = (per * r.Nxh) | 1;
    float2* TWy = lds + plane_pair_elems(r.Nx, r.Ny, r.plane_pair);   // second groups' twiddles
    float2* TWx = TWy + r.Ny;
    {
        const int ny = reg_ntw(r.reg_key[1], r.Ny), nx = reg_ntw(r.reg_key[0], r.Nx);
        for (int t = threadIdx.x; t < ny; t += NT) TWy[t] = gld(r.reg_tw[1] + t);
        for (int t = threadIdx.x; t < nx; t += NT) TWx[t] = gld(r.reg_tw[0] + t);
    }
    switch (r.reg_key[1]) {   // uniform per block
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr ((A0) * (A1) <= 16 && (B0) * (B1) <= 16) plane_pair_y<RegPlan<A0, A1, B0, B1>, NT>(r, z, l0, nl, la, lds, TWy); \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by plane_pairs on the host
    }
    switch (r.reg_key[0]) {
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr ((A0) * (A1) <= 16 && (B0) * (B1) <= 16) plane_pair_x<RegPlan<A0, A1, B0, B1>, NT>(r, z, l0, nl, la, lds, TWx); \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;
    }
}
}  // namespace

template <int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) k_plane_inv(const RepDev* __restrict__ reps, const WorkItem* __restrict__ wmap) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    warm_desc<0, 1, 3, 6, 7, 8>(r);
    if (r.plane_pair) {   // uniform per block, like the switch
        plane_pair_block<NT>(r, wi.blk, lds);
        return;
    }
    switch (r.reg_key[1]) {
#define TILD_CASE(A0, A1, B0, B1)          \
    case reg_plan_key(A0, A1, B0, B1):     \
        if constexpr (reg_plan_kept(A0 * A1 * B0 * B1) && (A0 * B0 / 2 + 1) * (A0 > B0 ? A0 : B0) <= NT) \
            plane_inv_block<A0, B0, NT>(r, wi.blk, lds);                                                 \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // excluded by plane_inv_plan on the host
    }
}

// ------------------------------------------------------------------ x C2R
// Inverse x transform of the half spectra into the gather records (the operation of
// k_x_c2r, kernels.hip) for compiled x plans, where no plane pass runs it (2D, and planes
// above half a CU's LDS; c2r_reg_plan); nr_c2r rows per block, nc complex lines per row:
//   A  task (line b, i < R2): Z = A + i B at k = i + R2 r of the full spectrum straight
//      from the half spectra (the upper half by Hermitian symmetry), first group; exchange;
//   B  task (b, i < R1): second group -> the real lines, over the values the task read;
//   C  the records (g_x, g_y, g_z), stored in order.
// Two barriers; the staged form has four and waits for its second stage's twiddles (film
// 64^2 5.6 -> 4.3 us, the latency of a launch of few blocks; 192^2 5.2 -> 4.8).  It reads
// each half-spectrum value twice, the second time from cache.
namespace {
template <class P, int NT>
__device__ __forceinline__ void c2r_reg_block(const RepDev& r, int blk, float2* lds) {
    constexpr int R1 = P::R1, R2 = P::R2, N = P::N, NXH = N / 2 + 1, NT1 = P::NTW;
    static_assert(NT1 <= NT, "c2r_reg_block: one twiddle per thread");
    const int D = r.dim, NL = r.nf * D, nc = (NL + 1) / 2;
    const int nrows = r.M / N;                 // rows of one field
    const int row0 = blk * r.nr_c2r;
    const int rows = min(r.nr_c2r, nrows - row0);
    const int nb = rows * nc, ldb = nb | 1;
    float2* X = lds;                           // N x ldb
    float2* TW = X + N * ((r.nr_c2r * nc) | 1);
    float2 tw = make_float2(0.f, 0.f);
    if ((int)threadIdx.x < NT1) tw = gld(r.reg_tw[0] + threadIdx.x);
    const float kf = r.kfac[0];
    const uint32_t line = (uint32_t)nrows * (uint32_t)NXH;   // one line's half spectra
    const FastDiv dnc(nc);
    const bool fuse = D == 2 && r.nf == 2;
    for (int task = threadIdx.x; task < nb * R2; task += NT) {
        const int i = task % R2, b = task / R2;
        int j;
        const int rr0 = dnc.div(b, j);
        const int la = 2 * j, lb = la + 1;
        const bool two = lb < NL;
        const bool xa = D == 3 ? la % 3 == 0 : true, xb = D == 3 && lb % 3 == 0;   // x derivatives (2D: every even line)
        const uint32_t o = (uint32_t)la * line + (uint32_t)(row0 + rr0) * (uint32_t)NXH;
        const float fi = (float)i;
        float2 A[R1], B[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const uint32_t kk = (uint32_t)half_entry<R2, N>(i, fi, rr).kk;
            A[rr] = gld(at32((const float2*)r.Gk, o + kk));
            B[rr] = gld(at32((const float2*)r.Gk, o + (two ? line : 0u) + kk));
        }
        float2 v[R1];
#pragma unroll
        for (int rr = 0; rr < R1; ++rr) {
            const HalfEntry e = half_entry<R2, N>(i, fi, rr);
            const float kx = kf * e.k;
            float2 a = A[rr], c = two ? B[rr] : make_float2(0.f, 0.f);
            a = pick(xa, x_gradient(kx, a), a);
            c = pick(xb, x_gradient(kx, c), c);
            if (e.self) { a.y = 0.f; c.y = 0.f; }
            // conj(Z) is transformed (the inverse as conj(FFT(conj))); products round before
            // they are added, as in the staged form, except where that form fuses them: the
            // lower half's real part with two fields in 2D
            const float re = fuse ? __builtin_fmaf(kx, A[rr].y, -c.y) : a.x - c.y;
            v[rr] = e.upper ? make_float2(a.x + c.y, a.y - c.x) : make_float2(re, -(a.y + c.x));
        }
        plan_first<P>(v, r.reg_tw[0]);
#pragma unroll
        for (int q = 0; q < R1; ++q) X[(i * R1 + q) * ldb + b] = v[q];
    }
    if ((int)threadIdx.x < NT1) TW[threadIdx.x] = tw;
    __syncthreads();
    const FastDiv dnb(nb);
    for (int task = threadIdx.x; task < nb * R1; task += NT) {
        int b;
        const int i = dnb.div(task, b);
        float2 w[R2];
#pragma unroll
        for (int rr = 0; rr < R2; ++rr) w[rr] = X[(i + R1 * rr) * ldb + b];
        plan_second_lds<P, true>(w, TW, i);
#pragma unroll
        for (int q = 0; q < R2; ++q) X[(i + R1 * q) * ldb + b] = w[q];
    }
    __syncthreads();
    const FastDiv dnf(r.nf);
    for (int task = threadIdx.x; task < rows * r.nf * N; task += NT) {
        const int x = task % N;
        int f;
        const int rr0 = dnf.div(task / N, f);
        float g[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d < D) {
                const int l = f * D + d;
                const float2 z = X[x * ldb + rr0 * nc + l / 2];
                g[d] = (l & 1) ? -z.y : z.x;   // conj of the forward result
            }
        }
        const uint32_t fn = (uint32_t)f * (uint32_t)r.M + (uint32_t)(row0 + rr0) * (uint32_t)N + (uint32_t)x;
        gst3((float*)((char*)r.G3 + ((fn << 3) + (fn << 2))), g[0], g[1], g[2]);   // 12 fn bytes, no mask (see k_x_c2r)
    }
}
}  // namespace

// ALL: as in k_grad_reg (114 registers and four waves per SIMD, 165 and three; 128^2 x 160
// 27.2 us against 32.5, 80 x 160 x 80 13.6 against 15.7).
template <int NT, bool ALL>
__global__ void __launch_bounds__(NT) k_c2r_reg(const RepDev* __restrict__ reps, const WorkItem* __restrict__ wmap) {
    extern __shared__ float2 lds[];
    const WorkItem wi = wmap[blockIdx.x];
    const RepDev& r = reps[wi.rep];
    warm_desc<0, 1, 3, 6, 7, 8>(r);
    switch (r.reg_key[0]) {   // uniform per block
#define TILD_CASE(A0, A1, B0, B1)                                                  \
    case reg_plan_key(A0, A1, B0, B1):                                             \
        if constexpr (ALL || !reg_plan_grouped(A1, B1))                            \
            c2r_reg_block<RegPlan<A0, A1, B0, B1>, NT>(r, wi.blk, lds);            \
        break;
        TILD_REG_PLANS(TILD_CASE)
#undef TILD_CASE
        default: break;   // reg_key holds compiled plans only
    }
}

// x plans for the register form.  In three dimensions not 160 points, whose LDS-staged form runs
// its two stages compiled (lds_fft2), nor 125, where a group of 5 leaves a fifth of the threads
// for the other's 25 values: staged and register form, us, 160 x 80 x 24 6.8 and 8.3, 160 x 80 x
// 80 14.7 and 15.5, 160^3 44.6 and 43.3; 125 x 100 x 100 22.3 and 23.7, with four types and
// charges 125 x 125 x 40 24.6 and 32.0.  The others gain, at any number of planes: 80 x 160 x 80
// 14.0 and 13.2, 100^3 17.2 and 14.1, 128 x 128 x 24 9.3 and 8.0, x 160 36.6 and 27.2, 180 x 180
// x 50 35.2 and 23.4; and films gain or are alike at every length.
bool c2r_reg_plan(const AxisPlan& pl, int dim) {
    const RegDims d = reg_dims(pl);
    return dim == 2 || !((d.R1 == 16 && d.R2 == 10) || d.R2 >= 5 * d.R1);
}

hipError_t launch_c2r_reg(const LaunchCtx& c) {
    if (!c.n) return hipSuccess;
    if (c.allforms) TILD_LAUNCH(c, (k_c2r_reg<kC2rRegThreads, true>), dim3(c.n), dim3(kC2rRegThreads), c.lds, c.reps, c.wmap);
    else TILD_LAUNCH(c, (k_c2r_reg<kC2rRegThreads, false>), dim3(c.n), dim3(kC2rRegThreads), c.lds, c.reps, c.wmap);
    return hipGetLastError();
}

bool plane_inv_plan(const AxisPlan& px, const AxisPlan& py) {
    if (!(px.N == py.N && reg_dims(py).key && reg_plan_kept(py.N))) return false;
    const int rmax = py.rad[0] > py.rad[1] ? py.rad[0] : py.rad[1];
    return (py.N / 2 + 1) * rmax <= kPlaneInvThreads && plane_inv_lds_bytes(py) <= kPlaneLds / 2;
}

// Pairs of lines to a block: as many as leave a task of the largest phase to every thread,
// spread evenly over the plane's blocks (a 21 x 21 x 225 slab with a pair to each of 675
// blocks of 462 / 3 tasks 9.7 us, with three 6.1; 27^3 alike with one and two).  Groups
// above 16 would spill the registers of two blocks to a CU.
int plane_pairs(const AxisPlan& px, const AxisPlan& py, int nf) {
    const RegDims x = reg_dims(px), y = reg_dims(py);
    if (!x.key || !y.key || x.R1 > 16 || y.R1 > 16 || x.R2 > 16 || y.R2 > 16) return 0;
    const int np = (3 * nf + 1) / 2, nxh = px.N / 2 + 1;
    const int tasks = std::max(2 * nxh * std::max(y.R1, y.R2), py.N * std::max(x.R1, x.R2));
    int g = std::max(1, std::min(np, kPlaneInvThreads / tasks));
    const int nb = (np + g - 1) / g;
    g = (np + nb - 1) / nb;
    return g * py.N * x.R2 <= plane_pair_hold(x.R1) * kPlaneInvThreads && plane_pair_lds_bytes(px.N, py.N, g) <= kPlaneLds / 2
               ? g : 0;
}

hipError_t launch_plane_inv(const LaunchCtx& c) {
    if (!c.n) return hipSuccess;
    TILD_LAUNCH(c, k_plane_inv<kPlaneInvThreads>, dim3(c.n), dim3(kPlaneInvThreads), c.lds, c.reps, c.wmap);
    return hipGetLastError();
}

static hipError_t allow_lds(const void* kernel, size_t bytes) {
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

hipError_t configure_plane_inv() {
    return allow_lds((const void*)k_plane_inv<kPlaneInvThreads>, kPlaneLds / 2);
}

// the kept square plans
bool plane_reg_plan(const AxisPlan& px, const AxisPlan& py) {
    return px.N == py.N && reg_dims(px).key && reg_plan_kept(px.N);
}

bool plane_rect_plan(const AxisPlan& px, const AxisPlan& py) {
    const RegDims x = reg_dims(px), y = reg_dims(py);
    return x.key && y.key && std::max(std::max(x.R1, x.R2), std::max(y.R1, y.R2)) <= 16 &&
           plane_rect_lds_bytes(px.N, py.N) <= kPlaneLds;
}

bool yfwd_reg_plan(const AxisPlan& pl) {
    const RegDims d = reg_dims(pl);
    return d.key && d.R1 <= 16 && d.R2 <= 16 && yfwd_reg_lds_bytes(pl) <= kPlaneLds;
}

hipError_t launch_plane_reg(const LaunchCtx& c) {
    if (!c.n) return hipSuccess;
    if (c.allforms) TILD_LAUNCH(c, (k_plane_reg<kPlaneRegThreads, true>), dim3(c.n), dim3(kPlaneRegThreads), c.lds, c.reps, c.wmap);
    else TILD_LAUNCH(c, (k_plane_reg<kPlaneRegThreads, false>), dim3(c.n), dim3(kPlaneRegThreads), c.lds, c.reps, c.wmap);
    return hipGetLastError();
}

hipError_t configure_plane_reg() {
    const hipError_t e = allow_lds((const void*)k_plane_reg<kPlaneRegThreads, false>, kPlaneLds);
    return e != hipSuccess ? e : allow_lds((const void*)k_plane_reg<kPlaneRegThreads, true>, kPlaneLds);
}

bool grad_reg_plan(const AxisPlan& pl) {
    const RegDims d = reg_dims(pl);
    return d.key && d.R1 <= 16;
}

hipError_t launch_grad_reg(const LaunchCtx& c) {
    if (!c.n) return hipSuccess;
    if (c.allforms) TILD_LAUNCH(c, (k_grad_reg<kGradRegThreads, true>), dim3(c.n), dim3(kGradRegThreads), c.lds, c.reps, c.wmap);
    else TILD_LAUNCH(c, (k_grad_reg<kGradRegThreads, false>), dim3(c.n), dim3(kGradRegThreads), c.lds, c.reps, c.wmap);
    return hipGetLastError();
}

bool last_reg_plan(const AxisPlan& pl, int ntypes, int nf) {
    const RegDims d = reg_dims(pl);
    if (!d.key || ntypes < 1 || ntypes > 4 || nf > ntypes + 1) return false;
    return last_reg_variant(pl.rad[0], d.R1, d.R2, pl.nst == 2, ntypes) && last_reg_cols(d.R1, d.R2, nf) >= 1;
}

hipError_t launch_last_reg(const LaunchCtx& c, int koff, int cls) {
    if (!c.n) return hipSuccess;
    switch (cls == 1 && c.allforms ? kLastRegShort : cls) {
        case 0: return launch_last_reg_0(c, koff);
        case 1: return launch_last_reg_1(c, koff);
        case 2: return launch_last_reg_2(c, koff);
        default: return launch_last_reg_3(c, koff);
    }
}

hipError_t configure_last_reg() {
    for (hipError_t e : {configure_last_reg_0(), configure_last_reg_1(), configure_last_reg_2(), configure_last_reg_3()})
        if (e != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace tild
