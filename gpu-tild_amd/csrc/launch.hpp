// launch.hpp -- block geometry of every pass (shared by kernels and host launchers)
// and the host-side launcher declarations.
#pragma once
#include "device.hpp"

#include <hip/hip_ext.h>

namespace tild {

// Largest batch of complex values one FFT block transforms at once (two LDS
// ping-pong buffers of this size).
constexpr int kFftBudget = kFftElems * kFftThreads;        // 2048
constexpr size_t kMaxLds = 65536;

// Strided pass along y (axis 1) or z (axis 2) of nfb half-spectrum fields.
struct MidGeom {
    int N, lstride, batch, nouter, ostride, nl, nchunk;
};
__host__ __device__ inline MidGeom mid_geom(const RepDev& r, int axis, int nfb) {
    MidGeom g;
    const int Nz = r.dim == 3 ? r.Nz : 1;
    if (axis == 1) {
        g.N = r.Ny; g.lstride = r.Nxh; g.batch = r.Nxh;
        g.nouter = nfb * Nz; g.ostride = r.Ny * r.Nxh;
    } else {
        g.N = r.Nz; g.lstride = r.Ny * r.Nxh; g.batch = r.Ny * r.Nxh;
        g.nouter = nfb; g.ostride = r.Nz * r.Ny * r.Nxh;
    }
    int nl = (r.mid_elems > 0 ? r.mid_elems : kFftBudget) / g.N;
    if (nl < 1) nl = 1;
    if (nl > g.batch) nl = g.batch;
    g.nchunk = (g.batch + nl - 1) / nl;
    g.nl = (g.batch + g.nchunk - 1) / g.nchunk;     // balanced chunks
    return g;
}
// 3D y-inverse of the gradient spectra: y lines of (field, z) planes, three line sets
// per column in one batch
__host__ __device__ inline MidGeom mid_grad_geom(const RepDev& r) {
    MidGeom g;
    g.N = r.Ny; g.lstride = r.Nxh; g.batch = r.Nxh;
    g.nouter = r.nf * r.Nz; g.ostride = r.Ny * r.Nxh;
    int nl = (r.mid_elems > 0 ? r.mid_elems : kFftBudget) / (3 * g.N);
    if (nl < 1) nl = 1;
    if (nl > g.batch) nl = g.batch;
    g.nchunk = (g.batch + nl - 1) / nl;
    g.nl = (g.batch + g.nchunk - 1) / g.nchunk;     // balanced chunks
    return g;
}
// one FFT buffer of N x nlines complex values, and the ping-pong pair a pass needs
inline size_t fft_buf_bytes(int N, int nlines) { return (size_t)N * (size_t)(nlines | 1) * sizeof(float2); }
inline size_t lds_bytes(int N, int nlines) { return 2 * fft_buf_bytes(N, nlines); }
// fused last-axis pass: coupled fields (nf*nl lines, unpadded: only read and written
// element by element) + two buffers of nf*DB*nl lines (DB inverse outputs per batch)
// + the ramp weights of the step
inline size_t last_lds_bytes(int N, int nf, int DB, int nl) {
    return (size_t)N * nf * nl * sizeof(float2) + 2 * fft_buf_bytes(N, nf * DB * nl) + kMaxRamp * sizeof(float);
}

// x transforms of a deposit launch: none (the forward plane passes make them), the LDS-staged one,
// or also those of the compiled plans
enum { kXNone = 0, kXStaged = 1, kXRegister = 2 };
struct LaunchCtx {
    const RepDev* reps;
    const WorkItem* wmap;
    int n;              // blocks
    size_t lds;         // dynamic LDS bytes
    hipStream_t stream;
    // step profile: events that take the kernel's own start and stop times
    hipEvent_t t0 = nullptr, t1 = nullptr;
    int threads = 0;    // block size where a pass has more than one (0: its default)
    int xfft = kXRegister;   // tiled deposit: the x transforms its replicas run
    // some replica of the set needs the instantiation that holds every form.  Deposit:
    // position records; particles: orders above 1; forward plane pass: rectangles and y
    // columns; y inverse, x C2R: plans with a group of two stages;
    // fused last-axis pass, class 1: class 0 with it
    bool allforms = true;
};

// Launch on c.stream; with c.t0 set, through hipExtLaunchKernel, whose events take
// the start and stop times of the kernel itself.
#define TILD_LAUNCH(c, kernel, grid, block, lds, ...)                                                   \
    do {                                                                                               \
        if ((c).t0) hipExtLaunchKernelGGL(kernel, grid, block, lds, (c).stream, (c).t0, (c).t1, 0, __VA_ARGS__); \
        else hipLaunchKernelGGL(kernel, grid, block, lds, (c).stream, __VA_ARGS__);                   \
    } while (0)

hipError_t launch_spread(const LaunchCtx& c, int koff);
hipError_t launch_x_r2c(const LaunchCtx& c, bool from_acc, int nrows_override, const float* in, float2* out);
hipError_t launch_mid(const LaunchCtx& c, int axis, int use_gk, int nfb, int inverse, float2* buf);
hipError_t launch_last_fused(const LaunchCtx& c, int store_spectrum, int koff);
hipError_t launch_x_c2r(const LaunchCtx& c, bool records, int nlines, const float2* in, float* out);
// claim: integrating steps of LDS-tiled replicas also claim the next step's records
hipError_t launch_particles(const LaunchCtx& c, bool integrate, int write_forces, int koff, bool claim);
hipError_t launch_advance(hipStream_t s, RepDev* reps, const int* which, int n, int nsteps,
                          hipEvent_t t0 = nullptr, hipEvent_t t1 = nullptr);
constexpr int kPlaneThreads = 512;                      // block of the plane forward pass
constexpr int kLastThreads = 256;                       // block of the fused last-axis pass
constexpr int kGradThreads = 256;                       // block of the y inverse pass
constexpr int kC2rThreads = 256;                        // block of the inverse x pass (records)
constexpr size_t kPlaneLds = 163840;                    // LDS one block may use (MI355X)
hipError_t launch_mid_grad(const LaunchCtx& c);
// Stockham plans the register-resident passes are compiled for, as two groups of stages
// (A0 A1) (B0 B1) (1: no second stage): a thread runs a group's stages on the R1 = A0 A1
// and then on the R2 = B0 B1 values it holds, so that a plan of three or four stages takes
// one exchange through LDS like one of two.  The radices and their order are the planner's.
#define TILD_REG_PLANS(X)                                                                            \
    X(8, 1, 3, 1) X(5, 1, 5, 1) X(10, 1, 3, 1) X(8, 1, 4, 1) X(8, 1, 5, 1) X(16, 1, 3, 1)            \
    X(10, 1, 5, 1) X(8, 1, 8, 1) X(10, 1, 8, 1) X(16, 1, 8, 1) X(16, 1, 10, 1) /* 24 ... 160 */      \
    X(7, 1, 3, 1) X(7, 1, 4, 1) X(7, 1, 5, 1) X(10, 1, 10, 1)                  /* 21 28 35 100 */     \
    X(3, 1, 3, 3) X(4, 1, 3, 3) X(5, 1, 3, 3) X(7, 1, 3, 3) X(5, 1, 4, 3)      /* 27 36 45 63 60 */   \
    X(8, 1, 3, 3) X(5, 1, 5, 3) X(10, 1, 3, 3) X(8, 1, 4, 3) X(8, 1, 5, 3)     /* 72 75 90 96 120 */  \
    X(5, 1, 5, 5) X(16, 1, 3, 3) X(10, 1, 5, 3) X(8, 1, 8, 3) X(8, 1, 5, 5)    /* 125 144 150 192 200 */ \
    X(10, 1, 8, 3) X(3, 3, 3, 2) X(4, 3, 3, 3) X(5, 4, 3, 3) X(8, 3, 3, 3)     /* 240 54 108 180 216 */ \
    X(5, 5, 3, 3)                                                              /* 225 */
// the radices in order, five bits each
__host__ __device__ constexpr int reg_plan_key(int a0, int a1, int b0, int b1) {
    int k = a0;
    if (a1 > 1) k = k * 32 + a1;
    k = k * 32 + b0;
    return b1 > 1 ? k * 32 + b1 : k;
}
// Plans of the first two lines: the fused z pass and the plane passes of square planes have run
// these in registers all along, and fuse the other product of a twiddle's two sums (cmul_kept;
// the inverse plane pass as the compiler does); every other register pass fuses them as the
// LDS-staged pass it stands for, so that no length's results depend on which of the two runs.
__host__ __device__ constexpr bool reg_plan_kept(int n) {
    return n == 24 || n == 25 || n == 30 || n == 32 || n == 40 || n == 48 || n == 50 || n == 64 || n == 80 || n == 128 ||
           n == 160;
}
// Plans with a group of two stages hold more values a thread (reg_plan_grouped): sets without
// them run kernels compiled without them, whose registers leave room for more waves.
__host__ __device__ constexpr bool reg_plan_grouped(int A1, int B1) { return A1 > 1 || B1 > 1; }
// x transform of the tiled deposit: in registers for compiled plans, but for films of 80 and 160
// points, whose LDS-staged form runs its two stages compiled (lds_fft2) in 71 registers against
// 128: staged and in registers, us, 160 x 64 6.5 and 7.1, 160 x 1024 7.6 and 8.1, 80 x 1024 6.2 and
// 7.0; odd-sided boxes 160 x 125 x 24 12.3 and 11.0, 80 x 45 x 60 with five fields 12.0 and 10.2.
__host__ __device__ constexpr bool deposit_xreg(int key, int dim) {
    return key != 0 && !(dim == 2 && (key == reg_plan_key(16, 1, 10, 1) || key == reg_plan_key(10, 1, 8, 1)));
}
// key, group sizes and first stage of the second group of an axis plan (key 0: not compiled)
struct RegDims {
    int key, R1, R2, group2;
};
RegDims reg_dims(const AxisPlan& pl);
// Fused last-axis pass with register-resident columns (fft_last.hpp): last axes with one
// of those plans, at most four types (two on axes above 100 points or of first radix 16)
// plus charges.  Blocks of kLastRegThreads threads hold nl_last = last_reg_cols columns.
constexpr int kLastRegThreads = 256;
// Plans of two stages run the inverse reversed (RepDev::axr), others as they are; a thread
// of the coupling stage holds a coefficient per type for each of its R2 (R1) values, at
// most 50.
__host__ __device__ constexpr bool last_reg_variant(int A0, int R1, int R2, bool rev, int TT) {
    return TT <= (R1 * R2 > 100 || A0 == 16 ? 2 : 4) && TT * (rev ? R2 : R1) <= 50;
}
// the kernel instantiation of a variant: axes up to 100 points with up to two types (class
// 0) or three and four (class 1), and longer axes (class 2)
__host__ __device__ constexpr int last_reg_class(int N, int TT) { return N > 100 ? 2 : (TT >= 3 ? 1 : 0); }
constexpr int kLastRegShort = 3;   // the kernel of classes 0 and 1
// whether the kernel of class k holds class c
__host__ __device__ constexpr bool last_reg_held(int c, int k) {
    return c == k || (c == 0 && k == 2) || (c <= 1 && k == kLastRegShort);
}
bool last_reg_plan(const AxisPlan& pl, int ntypes, int nf);
// columns of a block: one thread per (column, index of the larger group, field)
__host__ __device__ constexpr int last_reg_cols(int R1, int R2, int nf) {
    return kLastRegThreads / ((R1 > R2 ? R1 : R2) * nf);
}
inline int last_reg_lines(const AxisPlan& pl, int nf) { return last_reg_cols(reg_dims(pl).R1, reg_dims(pl).R2, nf); }
// the two exchange buffers, the inverse stage's twiddles and the ramp weights
inline size_t last_reg_lds_bytes(const AxisPlan& pl, int nf) {
    const size_t N = (size_t)pl.N, nl = (size_t)last_reg_lines(pl, nf);
    return (N * (3 * (size_t)nf * nl + 2) + N) * sizeof(float2) + kMaxRamp * sizeof(float);
}
hipError_t launch_last_reg(const LaunchCtx& c, int koff, int cls);
hipError_t launch_last_reg_0(const LaunchCtx& c, int koff);   // one per class, in files of their own
hipError_t launch_last_reg_1(const LaunchCtx& c, int koff);
hipError_t launch_last_reg_2(const LaunchCtx& c, int koff);
hipError_t launch_last_reg_3(const LaunchCtx& c, int koff);
hipError_t configure_last_reg_0();
hipError_t configure_last_reg_1();
hipError_t configure_last_reg_2();
hipError_t configure_last_reg_3();
// The y inverse of the gradient spectra with register-resident columns (3D, y plans as
// above with R1 <= 16): blocks of kGradRegThreads threads, grad_reg_lines(plan) columns
// each, grad_reg_chunks per (field, z) plane.
constexpr int kGradRegThreads = 128;
bool grad_reg_plan(const AxisPlan& pl);
inline int grad_reg_lines(const AxisPlan& pl) {
    const RegDims d = reg_dims(pl);
    return kGradRegThreads / (d.R1 > d.R2 ? d.R1 : d.R2);
}
inline int grad_reg_chunks(const AxisPlan& pl, int Nxh) { return (Nxh + grad_reg_lines(pl) - 1) / grad_reg_lines(pl); }
inline size_t grad_reg_lds_bytes(const AxisPlan& pl) {
    return ((size_t)pl.N * (3 * (size_t)grad_reg_lines(pl) + 1) + (size_t)pl.N) * sizeof(float2);
}
hipError_t launch_grad_reg(const LaunchCtx& c);
// The forward plane pass with register-resident columns: blocks of kPlaneRegThreads
// threads.  plane_reg: a (field, z) plane of the kept two-stage plans, square; plane_rect:
// any other of compiled plans; yfwd: columns of planes whose deposit transforms x.
constexpr int kPlaneRegThreads = 512;
bool plane_reg_plan(const AxisPlan& px, const AxisPlan& py);
inline size_t plane_reg_lds_bytes(const AxisPlan& pl) {
    const size_t N = (size_t)pl.N, ldp = (size_t)((pl.N / 2) | 1), ldc = (size_t)((pl.N / 2 + 1) | 1);
    return (N * (ldp > ldc ? ldp : ldc) + N * ldp + 2 * N) * sizeof(float2);
}
inline size_t plane_rect_lds_bytes(int Nx, int Ny) {
    const size_t a = (size_t)Nx * (size_t)((Ny / 2) | 1), b = (size_t)Ny * (size_t)((Nx / 2 + 1) | 1);
    return ((a > b ? a : b) + a + (size_t)Nx + (size_t)Ny) * sizeof(float2);
}
hipError_t launch_plane_reg(const LaunchCtx& c);
bool plane_rect_plan(const AxisPlan& px, const AxisPlan& py);
// yfwd: pieces of kYfwdThreads threads, their exchange and twiddles side by side
constexpr int kYfwdThreads = 128, kYfwdPieces = kPlaneRegThreads / kYfwdThreads;
inline int yfwd_reg_lines(const AxisPlan& pl) {
    const RegDims d = reg_dims(pl);
    return kYfwdThreads / (d.R1 > d.R2 ? d.R1 : d.R2);
}
inline int yfwd_reg_blocks(const AxisPlan& pl, int Nxh, int planes) {
    const int nl = yfwd_reg_lines(pl);
    return (planes * ((Nxh + nl - 1) / nl) + kYfwdPieces - 1) / kYfwdPieces;
}
inline size_t yfwd_reg_lds_bytes(const AxisPlan& pl) {
    return (size_t)kYfwdPieces * (size_t)pl.N * (size_t)(yfwd_reg_lines(pl) + 2) * sizeof(float2);
}
bool yfwd_reg_plan(const AxisPlan& pl);
hipError_t configure_plane_reg();
// Register-resident inverse plane pass (y inverse + x C2R into the gather records) of
// square planes with a kept two-stage plan: one block of kPlaneInvThreads threads per
// (field, z) plane, two blocks to a CU.
constexpr int kPlaneInvThreads = 512;
inline size_t plane_inv_lds_bytes(const AxisPlan& pl) {
    const size_t N = (size_t)pl.N, la = (size_t)((3 * (pl.N / 2 + 1)) | 1);
    return (N * la + (size_t)pl.rad[0] * (pl.rad[1] - 1)) * sizeof(float2);
}
bool plane_inv_plan(const AxisPlan& px, const AxisPlan& py);
// The same for any other plane of compiled plans with R1, R2 <= 16, in the same kernel: one
// block per z plane and plane_pairs pairs of the x pass' lines, two blocks to a CU.  A thread
// holds plane_pair_hold(R1) first groups, 24 values, at once.
__host__ __device__ constexpr int plane_pair_hold(int R1) { return R1 > 24 ? 1 : 24 / R1; }
__host__ __device__ constexpr int plane_pair_elems(int Nx, int Ny, int g) {   // the rows' half spectra, or the x exchange
    return Ny * ((2 * g * (Nx / 2 + 1)) | 1) > Nx * ((Ny * g) | 1) ? Ny * ((2 * g * (Nx / 2 + 1)) | 1) : Nx * ((Ny * g) | 1);
}
inline size_t plane_pair_lds_bytes(int Nx, int Ny, int g) {
    return (size_t)(plane_pair_elems(Nx, Ny, g) + Nx + Ny) * sizeof(float2);
}
int plane_pairs(const AxisPlan& px, const AxisPlan& py, int nf);   // 0: no such pass
hipError_t launch_plane_inv(const LaunchCtx& c);
hipError_t configure_plane_inv();
hipError_t configure_last_reg();
hipError_t launch_plane_r2c(const LaunchCtx& c);
// LDS of the forward plane pass: two buffers holding either the Ny/2 row pairs of
// length Nx or the Ny x Nxh half spectra
inline size_t plane_r2c_lds(const RepDev& h) {
    const size_t a = (size_t)h.Nx * (size_t)((h.Ny / 2) | 1), b = (size_t)h.Ny * (size_t)(h.Nxh | 1);
    return 2 * (a > b ? a : b) * sizeof(float2);
}
// x C2R into the gather records with register-resident columns (compiled x plans, no
// field phases): one exchange buffer and the second group's twiddles.
constexpr int kC2rRegThreads = 256;
inline size_t c2r_reg_lds_bytes(int N, int nlines) { return fft_buf_bytes(N, nlines) + (size_t)N * sizeof(float2); }
bool c2r_reg_plan(const AxisPlan& pl, int dim);
hipError_t launch_c2r_reg(const LaunchCtx& c);
// One-time kernel attributes (dynamic LDS above 64 KiB for the plane pass).
hipError_t configure_kernels();
hipError_t launch_kprops(const LaunchCtx& c, int nq_max);
hipError_t launch_sk_accumulate(hipStream_t s, const RepDev* reps, int rep, int type, int Mh, double* acc);
hipError_t launch_bond_props(const LaunchCtx& c);
hipError_t launch_reduce_rows(hipStream_t s, const double* in, int nrows, int n, double* out);
constexpr int kCountBlock = 256;                        // beads per block of the bucket claims
hipError_t launch_tile_count(const LaunchCtx& c, int koff);
hipError_t launch_tile_scan(const LaunchCtx& c);
hipError_t launch_tile_claim(const LaunchCtx& c, int koff);
hipError_t launch_tile_reset(const LaunchCtx& c, int koff);
hipError_t launch_tile_regions(hipStream_t s, const RepDev* reps, int rep);
// c.threads: 512 for sets whose tiles hold many beads, else 256
hipError_t launch_tile_deposit(const LaunchCtx& c, int koff);
hipError_t launch_bins(hipStream_t s, const RepDev* reps, int rep, int ns, int* out);
hipError_t launch_virial_source(hipStream_t s, const RepDev* reps, int rep, int M, const float* fr, float* vr);

// Buffers of the periodic spatial reorder (one set per replica that reorders).
struct ReorderBufs {
    uint32_t* keys[2] = {nullptr, nullptr};   // ns row keys (unsorted, sorted)
    int* vals[2] = {nullptr, nullptr};        // ns slot ids (identity, new order)
    void* tmp = nullptr;                      // radix-sort scratch
    size_t tmp_bytes = 0;
};
size_t reorder_tmp_bytes(int ns, int bits);

// Site-order copy of a permuted per-bead array of D floats: dst[pid[p]] = src[p] (to_site)
// or dst[p] = src[pid[p]].
hipError_t launch_site_order(hipStream_t s, const float* src, const int* pid, float* dst, int ns, int D, bool to_site);

// Neighbour-list build (device buffers, all indexed by site id except cell_slots).
struct NlistArgs {
    const unsigned char* member;   // ns group-membership flags
    int* cell_of;                  // ns cell of each member (-1 outside the group)
    int* counts;                   // ns list lengths
    int* neigh;                    // ns * cap sorted neighbour site ids
    int* cell_count;               // ncells
    int* cell_slots;               // ncells * cmax slots
    int* overflow;                 // 1: a cell exceeded cmax, 2: a list exceeded cap
    float Lc[3];
    int nc[3];
    float rc;
    int cmax, cap;
};
hipError_t launch_nlist(hipStream_t s, const RepDev* reps, int rep, int ns, const NlistArgs& a);
// Sort the replica's beads by grid row (stable), permute every per-bead array and
// swap the live and spare buffers in the device descriptor.
hipError_t launch_reorder(hipStream_t s, RepDev* reps, int rep, int ns, int bits, ReorderBufs& b);
// Tiled replicas: each tile's beads (from an exact binning, tkey and toff) sorted by
// site id, then the same permutation.
hipError_t launch_reorder_tiles(hipStream_t s, RepDev* reps, int rep, int ns, int ntiles, ReorderBufs& b);
// The same for a set of tiled replicas at once: `beads` maps 256-bead blocks, `tiles`
// one block per tile and `reps1` one block per replica (scratch in RepDev::rsrc etc.).
hipError_t launch_reorder_tiles_set(const LaunchCtx& beads, const LaunchCtx& tiles, const LaunchCtx& reps1);
// Bucket regions (k_tile_regions) of every replica of a set, one block each.
hipError_t launch_tile_regions_set(const LaunchCtx& reps1);

}  // namespace tild
