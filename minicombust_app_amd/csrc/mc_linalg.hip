// mc_linalg.hip -- Krylov solvers and the aggregation-AMG hierarchy.
//
// Replaces the AmgX solves of the reference GPU path (gpu/FlowSolver.inl:
// 716-782, 943-969) and PETSc's KSPBCGS / KSPFGMRES+PCGAMG of the CPU path
// (FlowSolver.hpp:513-527, FlowSolver.inl:1341-1375, 2203-2273).
//
// Storage.  Matrices are assembled in the PETSc CSR pattern.  When a pattern
// has exactly 7 distinct diagonals (the box mesh's 7-point coupling) or 27
// (a coarse level of the regular 2x2x2 aggregation of that mesh), the solver
// also keeps a diagonal-indexed copy, v[d*n + i] = A[i, i + off_d] (zero
// where the pattern has no entry): one thread per row, no column indices to
// stream, and all ND loads of a row independent and coalesced.  Any other
// pattern runs the CSR kernels: 8 lanes per row, the row sum reduced with 3
// cross-lane shuffles.  A ND-template drives every kernel through for_rows().
//
// Reductions: fixed-order two-level block sums finished by the last block
// (deterministic, no host round trip).  Solver scalars live in device memory;
// kernels of a converged system return at once, and the host polls a flag
// after a number of iterations predicted from the observed convergence rate.
//
//  * BiCGStab: van der Vorst's unpreconditioned method, x0 = 0 (momentum and
//    scalar equations; the reference's KSPBCGS+PCNONE), up to 4 RHS sharing
//    each matrix read.
//  * Pressure: PCG preconditioned by an unsmoothed-aggregation AMG V-cycle
//    (damped Jacobi nu/nu, scaled coarse correction, dense regularised inverse
//    on the coarsest level) on the singular Neumann system with the RHS
//    projected to mean zero.  Mixed form: FP32 PCG-AMG (SpMV, smoothers,
//    hierarchy) inside FP64 iterative refinement; the refinement residual,
//    the update and the coarsest solve stay FP64.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <set>

#include "mc_internal.hpp"

namespace mc {

// ------------------------------------------------------------ layout --
constexpr int RED_MAX_BLOCKS = 8192;   // partial sums: at most 12 per block (RED_PARTIALS)
static_assert(12 * RED_MAX_BLOCKS <= RED_PARTIALS, "reduction partials buffer");
constexpr int BLOCK = 256;

struct Grid {
    int blocks;
    int chunk;   // rows per block (multiple of BLOCK)
};

static Grid grid_for(int n)
{
    const int64_t g = div_up(n, BLOCK);
    int blocks = (int)std::min<int64_t>(g, RED_MAX_BLOCKS);
    if (blocks < 1) blocks = 1;
    const int64_t per = div_up(g, blocks);
    Grid gr;
    gr.chunk = (int)(per * BLOCK);
    gr.blocks = div_up(n, gr.chunk);
    if (gr.blocks < 1) gr.blocks = 1;
    return gr;
}

// Grid of a CSR level's smoothing passes, without reductions: eight lanes a row,
// so 32 rows a block ask for everything in one go.  With grid_for's 256 a thread
// visited eight rows one after the other, each waiting for its row pointers,
// then columns, then x: 8,984 rows (modifier 33's second level, FP32) k_jac
// 7.3 -> 4.1 us, k_jac_first2 8.5 -> 3.2, k_jac_prolong 8.5 -> 4.6.
static Grid grid_csr(int n)
{
    Grid g;
    const int rows = BLOCK / 8;
    g.chunk = rows * std::max(1, div_up(n, rows * (1 << 20)));
    g.blocks = std::max(1, div_up(n, g.chunk));
    return g;
}

// alpha, omega, rho and beta formed by their consumers (fold_sums)
static bool fold_on(const Ctx *c, const Grid &g) { return g.blocks <= FOLD_BLOCKS && !(c->plain & MC_PLAIN_FINISH); }

// Device scalars of one Krylov solve (NR <= 4 systems).
struct KState {
    double rho_old[4], alpha[4], omega[4], rho[4], beta[4];
    double tol[4], bnorm[4], rnorm[4], sn[4], mean;
    double atol;
    int done[4], half[4], iters[4], conv[4];
    int zero_start[4];   // BiCGStab: the initial guess is dropped for x0 = 0
    int all_done, nr, maxit, pad;
};

// ------------------------------------------------------- matrix view --
template <typename T>
struct Mat {
    int n;
    const int *rp, *col;
    const T *csr;
    const T *dia;          // diagonal storage, nullptr -> CSR kernels
    int nd;
    int off[DIA_MAX];
    int sym;               // symmetric: dia holds diagonals nd/2 .. nd-1 (offsets >= 0) only
};

// Entry (i, i + off[d]) of a diagonal-storage matrix.  Symmetric storage
// (SYM) keeps the main diagonal and the upper ones; a lower entry is the
// stored upper entry of the transposed position (row i + off[d], diagonal
// nd-1-d), zero where that row does not exist.  Reading it there touches the
// words a later row reads as its upper entry, so each value crosses HBM once.
// SYM is a compile-time choice (negative ND in the kernels' dispatch): a
// run-time branch here slows every diagonal-storage kernel.
template <bool SYM, typename T>
__device__ __forceinline__ double dia_at(const Mat<T> &A, int d, int i)
{
    if constexpr (!SYM) {
        return (double)A.dia[(size_t)d * A.n + i];
    } else {
        const int h = A.nd >> 1;
        if (d >= h) return (double)A.dia[(size_t)(d - h) * A.n + i];
        const int j = i + A.off[d];
        return j >= 0 ? (double)A.dia[(size_t)(A.nd - 1 - d - h) * A.n + j] : 0.0;
    }
}

// bytes of one pass over a matrix: the stored diagonals (symmetric storage:
// the main and upper ones), or CSR values + columns + row pointers
template <typename T>
static double mat_bytes(const Mat<T> &A, int64_t nnz, size_t vsize)
{
    if (A.nd) return (double)vsize * (A.sym ? A.nd / 2 + 1 : A.nd) * A.n;
    return (double)(vsize + 4) * nnz + 4.0 * (A.n + 1);
}


__device__ __forceinline__ int clampi(int j, int n) { return j < 0 ? 0 : (j >= n ? n - 1 : j); }

// The V-cycle's row expressions, contraction written out: the per-pass kernels
// and the one-workgroup tail of the cycle use them in different surroundings
// and form the same bits.
template <typename T>
__device__ __forceinline__ T vc_fma(T a, T b, T c)
{
    if constexpr (sizeof(T) == 8) return (T)fma((double)a, (double)b, (double)c);
    else return (T)fmaf((float)a, (float)b, (float)c);
}
// y + omega D^-1 (b - A y)
template <typename T>
__device__ __forceinline__ T vc_jac(T y, T omega, T di, T b, double ax)
{
#pragma clang fp contract(off)
    return vc_fma(omega * di, b - (T)ax, y);
}
// w D^-1 b
template <typename T>
__device__ __forceinline__ T vc_first(T w, T di, T b)
{
#pragma clang fp contract(off)
    return (w * di) * b;
}
// two sweeps from zero: x1 + w2 D^-1 (b - A x1), x1 = w1 D^-1 b
template <typename T>
__device__ __forceinline__ T vc_first2(T w1, T w2, T di, T b, double ax)
{
#pragma clang fp contract(off)
    return vc_fma(w1 * di, b, (w2 * di) * (b - (T)ax));
}
// x + cs xc
template <typename T>
__device__ __forceinline__ T vc_prolong(T x, T cs, T xc) { return vc_fma(cs, xc, x); }

// Visit the rows [r0, r1) handled by this thread and call f(row, A x) once
// per row.  ND > 0: one thread per row over ND diagonals (compile-time, fully
// unrolled); ND == 0: CSR, 8 lanes per row, lane 0 calls f.  X(k, j) yields
// operand k at column j, so fused producers (prolongation, p-update) feed the
// product without a separate pass.
template <int ND, int NR, typename T, typename XF, typename F>
__device__ __forceinline__ void for_rows(const Mat<T> &A, int r0, int r1, XF X, F f)
{
    constexpr bool SYM = ND < 0;
    constexpr int NA = SYM ? -ND : ND;
    if constexpr (NA > 0) {
        for (int i = r0 + (int)threadIdx.x; i < r1; i += BLOCK) {
            double acc[NR];
#pragma unroll
            for (int k = 0; k < NR; k++) acc[k] = 0.0;
            double a[NA];
            int j[NA];
#pragma unroll
            for (int d = 0; d < NA; d++) {
                a[d] = dia_at<SYM>(A, d, i);
                j[d] = clampi(i + A.off[d], A.n);
            }
#pragma unroll
            for (int d = 0; d < NA; d++) {
#pragma unroll
                for (int k = 0; k < NR; k++) acc[k] = fma(a[d], X(k, j[d]), acc[k]);
            }
            f(i, acc);
        }
    } else {
        const int lane8 = threadIdx.x & 7;
        for (int base = r0; base < r1; base += BLOCK / 8) {
            const int r = base + (threadIdx.x >> 3);
            double acc[NR];
#pragma unroll
            for (int k = 0; k < NR; k++) acc[k] = 0.0;
            if (r < r1) {
                const int beg = A.rp[r], end = A.rp[r + 1];
                for (int e = beg + lane8; e < end; e += 8) {
                    const int jj = A.col[e];
                    const double a = (double)A.csr[e];
#pragma unroll
                    for (int k = 0; k < NR; k++) acc[k] += a * X(k, jj);
                }
            }
#pragma unroll
            for (int k = 0; k < NR; k++) {
                acc[k] = lane8_sum(acc[k]);
            }
            if (lane8 == 0 && r < r1) f(r, acc);
        }
    }
}

// Launch a kernel template over the supported diagonal counts; KERNEL names
// the count ND_ (7, 27, or 0 for the CSR path).
// Kernels take the storage as a compile-time ND: the number of diagonals,
// negative for symmetric storage, 0 for CSR.
template <typename T>
inline int nd_code(const Mat<T> &A)
{
    return A.dia ? (A.sym ? -A.nd : A.nd) : 0;
}

#define MC_DISPATCH_ND(code, KERNEL, ...)                                                         \
    do {                                                                                          \
        const int code_ = (code);                                                                 \
        if (code_ == 7) { constexpr int ND_ = 7; hipLaunchKernelGGL(KERNEL, __VA_ARGS__); }        \
        else if (code_ == -7) { constexpr int ND_ = -7; hipLaunchKernelGGL(KERNEL, __VA_ARGS__); } \
        else if (code_ == 27) { constexpr int ND_ = 27; hipLaunchKernelGGL(KERNEL, __VA_ARGS__); } \
        else if (code_ == -27) { constexpr int ND_ = -27; hipLaunchKernelGGL(KERNEL, __VA_ARGS__); } \
        else { constexpr int ND_ = 0; hipLaunchKernelGGL(KERNEL, __VA_ARGS__); }                  \
    } while (0)

// ------------------------------------------ CSR -> diagonal storage --
// Offsets of a pattern; diagonal storage when there are exactly 7 or 27.
static bool dia_analyze(int n, const int *rp, const int *col, std::vector<int> &offs, std::vector<int> &map)
{
    std::set<int> s;
    for (int i = 0; i < n; i++)
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            s.insert(col[k] - i);
            if (s.size() > 27) return false;
        }
    if (s.size() != 7 && s.size() != 27) return false;
    offs.assign(s.begin(), s.end());
    map.resize(rp[n]);
    for (int i = 0; i < n; i++)
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            const int d = (int)(std::lower_bound(offs.begin(), offs.end(), col[k] - i) - offs.begin());
            map[k] = d * n + i;
        }
    return true;
}

// The pattern of a box: nx x ny x nz cells numbered x fastest, each row the
// cell and its neighbours in -z, -y, -x, +x, +y, +z that exist.
static bool box_analyze(int n, const int *rp, const int *col, int &nx, int &ny, int &nz)
{
    // a corner cell's row names the strides: 0, 1, nx, nx ny
    if (n < 8 || rp[1] - rp[0] != 4 || col[0] != 0 || col[1] != 1) return false;
    const int a = col[2], b = col[3];
    if (a < 2 || b % a || b / a < 2 || n % b || n / b < 2) return false;
    nx = a; ny = b / a; nz = n / b;
    for (int z = 0, i = 0; z < nz; z++)
        for (int y = 0; y < ny; y++)
            for (int x = 0; x < nx; x++, i++) {
                int k = rp[i];
                const int e = rp[i + 1];
                if (e - k != 1 + (z > 0) + (y > 0) + (x > 0) + (x + 1 < nx) + (y + 1 < ny) + (z + 1 < nz)) return false;
                if (z > 0 && col[k++] != i - b) return false;
                if (y > 0 && col[k++] != i - a) return false;
                if (x > 0 && col[k++] != i - 1) return false;
                if (col[k++] != i) return false;
                if (x + 1 < nx && col[k++] != i + 1) return false;
                if (y + 1 < ny && col[k++] != i + a) return false;
                if (z + 1 < nz && col[k++] != i + b) return false;
            }
    return true;
}

__global__ void k_csr_to_dia(int nnz, const int *map, const double *csr, double *dia, float *dia32)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnz) return;
    const double v = csr[k];
    dia[map[k]] = v;
    if (dia32) dia32[map[k]] = (float)v;
}

int dia_setup_fine(Ctx *c)
{
    MemScope ms(c, MC_MEM_MATRIX);
    std::vector<int> rp(c->N + 1), col(c->nnz), offs, map;
    MC_HIP(c, hipMemcpy(rp.data(), c->row_ptr, (size_t)(c->N + 1) * 4, hipMemcpyDeviceToHost));
    MC_HIP(c, hipMemcpy(col.data(), c->col, (size_t)c->nnz * 4, hipMemcpyDeviceToHost));
    c->fine_nd = 0;
    c->box_nx = c->box_ny = c->box_nz = 0;
    if (!dia_analyze(c->N, rp.data(), col.data(), offs, map)) return MC_OK;
    if (!box_analyze(c->N, rp.data(), col.data(), c->box_nx, c->box_ny, c->box_nz))
        c->box_nx = c->box_ny = c->box_nz = 0;
    c->fine_nd = (int)offs.size();
    for (int d = 0; d < c->fine_nd; d++) c->fine_off[d] = offs[d];
    MC_TRY(dalloc(c, &c->fine_map, c->nnz));
    MC_HIP(c, hipMemcpy(c->fine_map, map.data(), (size_t)c->nnz * 4, hipMemcpyHostToDevice));
    MC_TRY(dalloc(c, &c->A_dia, (size_t)c->fine_nd * c->N));
    MC_TRY(dalloc(c, &c->A_dia2, (size_t)c->fine_nd * c->N));
    // entries outside the pattern (missing neighbours) stay zero for good
    MC_HIP(c, hipMemset(c->A_dia, 0, (size_t)c->fine_nd * c->N * 8));
    MC_HIP(c, hipMemset(c->A_dia2, 0, (size_t)c->fine_nd * c->N * 8));
    return MC_OK;
}

const double *fine_dia_of(const Ctx *c, const double *csr)
{
    if (!c->fine_nd) return nullptr;
    if (csr == c->A_vals) return c->A_dia;
    if (csr == c->A_vals2) return c->A_dia2;
    return nullptr;
}

__global__ void k_dia_to_csr(int nnz, const int *map, const double *dia, double *csr)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nnz) csr[k] = dia[map[k]];
}

int dia_to_csr(Ctx *c, const double *dia, double *csr)
{
    hipLaunchKernelGGL(k_dia_to_csr, dim3(div_up(c->nnz, 256)), dim3(256), 0, c->stream, c->nnz, c->fine_map, dia, csr);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

static Mat<double> fine_mat(Ctx *c, const double *csr, const double *dia)
{
    Mat<double> A;
    A.n = c->N; A.rp = c->row_ptr; A.col = c->col; A.csr = csr;
    A.dia = (c->fine_nd && dia) ? dia : nullptr;
    A.nd = A.dia ? c->fine_nd : 0;
    A.sym = 0;
    for (int d = 0; d < DIA_MAX; d++) A.off[d] = d < c->fine_nd ? c->fine_off[d] : 0;
    return A;
}

// CSR values (set through the array access) into the diagonal storage.
int csr_to_dia(Ctx *c, const double *csr, double *dia)
{
    if (!c->fine_nd) return MC_OK;
    hipLaunchKernelGGL(k_csr_to_dia, dim3(div_up(c->nnz, 256)), dim3(256), 0, c->stream, c->nnz, c->fine_map, csr, dia,
                       (float *)nullptr);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

// ------------------------------------------------------------ SpMV --
template <int ND>
__global__ void __launch_bounds__(BLOCK) k_spmv(Mat<double> A, const double *x, double *y, int chunk)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * chunk, r1 = min(A.n, r0 + chunk);
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return x[j]; }, [&](int i, const double (&ax)[1]) { y[i] = ax[0]; });
}

int spmv(Ctx *c, const double *vals, const double *x, double *y)
{
    const Grid g = grid_for(c->N);
    // the momentum / scalar matrices through their diagonal storage, any other
    // (the pressure matrix) through CSR
    const Mat<double> A = fine_mat(c, vals, fine_dia_of(c, vals));
    MC_DISPATCH_ND(nd_code(A), (k_spmv<ND_>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, x, y, g.chunk);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

// ------------------------------------------------------- BiCGStab --
// One iteration is three streaming kernels, each followed by a one-block
// finishing kernel for its dot products:
//   pv: p = r + beta (p' - omega v'), formed on the fly (also where a row
//       reads it at a neighbour); v = A p; (r^, v)       -> alpha
//   st: s = r - alpha v, formed on the fly; t = A s;
//       (t, s), (t, t), (s, s)                           -> half-step test, omega
//   xr: x += alpha p + omega s; r = s - omega t;
//       (r, r), (r^, r)                                  -> convergence, rho, beta
// p and v alternate between two buffers, since rows read the previous
// iteration's values at their neighbours while others write the new ones.
struct BiVecs {
    double *x[4], *r[4], *s[4], *t[4];
    double *p[4], *v[4];            // this iteration's
    const double *po[4], *vo[4];    // the previous iteration's
    const double *rh[4];            // r^ (= b, never written)
    const double *b[4];
};

template <int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_init(int n, BiVecs w, double *partials, int chunk)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = b * chunk, i1 = min(n, i0 + chunk);
    double acc[NR];
#pragma unroll
    for (int k = 0; k < NR; k++) acc[k] = 0.0;
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const double bi = w.b[k][i];
            w.x[k][i] = 0.0; w.r[k][i] = bi;
            acc[k] += bi * bi;
        }
    }
    block_partials<NR>(acc, partials, b, gridDim.x);
}

// Warm start: r = b - A x0 with the starting values the caller left in x;
// partials of (b, b), (r, r) and (r^, r) with r^ = b.
template <int ND, int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_init_x0(Mat<double> A, BiVecs w, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double acc[3 * NR];
#pragma unroll
    for (int k = 0; k < 3 * NR; k++) acc[k] = 0.0;
    for_rows<ND, NR>(A, r0, r1, [&](int k, int j) { return w.x[k][j]; }, [&](int i, const double (&ax)[NR]) {
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const double bi = w.b[k][i], ri = bi - ax[k];
            w.r[k][i] = ri;
            acc[3 * k] += bi * bi;
            acc[3 * k + 1] += ri * ri;
            acc[3 * k + 2] += bi * ri;
        }
    });
    block_partials<3 * NR>(acc, partials, bb, gridDim.x);
}

// The same partials when the assembly already formed r = b - A x0.
template <int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_init_r0(int n, BiVecs w, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = bb * chunk, i1 = min(n, i0 + chunk);
    double acc[3 * NR];
#pragma unroll
    for (int k = 0; k < 3 * NR; k++) acc[k] = 0.0;
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const double bi = w.b[k][i], ri = w.r[k][i];
            acc[3 * k] += bi * bi;
            acc[3 * k + 1] += ri * ri;
            acc[3 * k + 2] += bi * ri;
        }
    }
    block_partials<3 * NR>(acc, partials, bb, gridDim.x);
}

// The criterion stays ||r|| <= rtol ||b|| (PETSc's default test, as with a
// zero start).  A guess whose residual is not below ||b|| is dropped: that
// right-hand side restarts from x0 = 0 (in the first k_bi_pv), so a warm start
// never converges later than the zero start would.
template <int NR>
struct EpiBiInitX0 {
    KState *ks;
    double rtol;
    int maxit;
    __device__ void operator()(const double (&v)[3 * NR]) const
    {
        int all = 1;
        for (int k = 0; k < NR; k++) {
            const double bn = sqrt(v[3 * k]), rn = sqrt(v[3 * k + 1]);
            const int zs = !(rn < bn);
            ks->zero_start[k] = zs;
            ks->bnorm[k] = bn; ks->tol[k] = rtol * bn; ks->rnorm[k] = zs ? bn : rn;
            ks->rho_old[k] = 1.0; ks->alpha[k] = 1.0; ks->omega[k] = 1.0;
            ks->rho[k] = zs ? v[3 * k] : v[3 * k + 2];   // (r^, r0)
            ks->beta[k] = 0.0;
            ks->iters[k] = 0; ks->half[k] = 0; ks->sn[k] = 0.0;
            const double r0n = zs ? bn : rn;
            ks->done[k] = (bn == 0.0 || r0n <= ks->tol[k]) ? 1 : 0;
            ks->conv[k] = ks->done[k];
            all &= ks->done[k];
        }
        ks->nr = NR; ks->maxit = maxit;
        ks->all_done = all;
    }
};

template <int NR>
struct EpiBiInit {
    KState *ks;
    double rtol;
    int maxit;
    __device__ void operator()(const double (&v)[NR]) const
    {
        int all = 1;
        for (int k = 0; k < NR; k++) {
            const double bn = sqrt(v[k]);
            ks->bnorm[k] = bn; ks->tol[k] = rtol * bn; ks->rnorm[k] = bn;
            ks->rho_old[k] = 1.0; ks->alpha[k] = 1.0; ks->omega[k] = 1.0;
            ks->rho[k] = v[k];  // (r^, r) with r^ = r = b
            ks->beta[k] = 0.0;
            ks->iters[k] = 0; ks->half[k] = 0; ks->sn[k] = 0.0;
            ks->done[k] = (bn == 0.0) ? 1 : 0;
            ks->conv[k] = (bn == 0.0) ? 1 : 0;
            all &= ks->done[k];
        }
        ks->nr = NR; ks->maxit = maxit;
        ks->all_done = all;
    }
};

// v = A p with p formed on the fly ; partials of (r^, v)
template <int ND, int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_pv(Mat<double> A, BiVecs w, const KState *ks, double *partials,
                                                 int chunk, int warm)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * chunk, r1 = min(A.n, r0 + chunk);
    bool skip[NR], first[NR], zs[NR];
    double beta[NR], om[NR], dsum[NR];
    bool any = false;
#pragma unroll
    for (int k = 0; k < NR; k++) {
        // first iteration after a warm start: a right-hand side whose guess
        // was dropped (b = 0 included: its solution is zero) restarts from
        // x = 0, r = b, converged or not; p is then read from b, since other
        // blocks are writing r
        zs[k] = warm && (ks->zero_start[k] || ks->bnorm[k] == 0.0);
        any |= zs[k];
    }
    if (any)
        for (int i = r0 + (int)threadIdx.x; i < r1; i += BLOCK)
#pragma unroll
            for (int k = 0; k < NR; k++)
                if (zs[k]) { w.x[k][i] = 0.0; w.r[k][i] = w.b[k][i]; }
    if (ks->all_done) return;
#pragma unroll
    for (int k = 0; k < NR; k++) {
        skip[k] = ks->done[k] != 0;
        first[k] = ks->iters[k] == 0;
        beta[k] = ks->beta[k];
        om[k] = ks->omega[k];
        dsum[k] = 0.0;
    }
    auto P = [&](int k, int j) -> double {
        if (zs[k]) return w.b[k][j];
        if (first[k]) return w.r[k][j];
        return fma(beta[k], fma(-om[k], w.vo[k][j], w.po[k][j]), w.r[k][j]);
    };
    for_rows<ND, NR>(A, r0, r1, [&](int k, int j) { return skip[k] ? 0.0 : P(k, j); },
                     [&](int r, const double (&ax)[NR]) {
#pragma unroll
                         for (int k = 0; k < NR; k++) {
                             if (skip[k]) continue;
                             w.p[k][r] = P(k, r);
                             w.v[k][r] = ax[k];
                             dsum[k] += w.rh[k][r] * ax[k];
                         }
                     });
    block_partials<NR>(dsum, partials, b, gridDim.x);
}

template <int NR>
struct EpiBiAlpha {
    KState *ks;
    __device__ void operator()(const double (&v)[NR]) const
    {
        if (ks->all_done) return;
        for (int k = 0; k < NR; k++)
            if (!ks->done[k]) ks->alpha[k] = ks->rho[k] / v[k];
    }
};

// t = A s with s = r - alpha v formed on the fly ; partials of (t,s), (t,t), (s,s)
template <int ND, int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_st(Mat<double> A, BiVecs w, KState *ks, const double *fold,
                                                 double *partials, int chunk)
{
    if (ks->all_done) return;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = b * chunk, r1 = min(A.n, r0 + chunk);
    bool skip[NR];
    double al[NR], dsum[3 * NR];
    if (fold) {   // EpiBiAlpha here; no block reads the alpha that block 0 stores for k_bi_xr
        double v[NR];
        fold_sums<NR>(fold, gridDim.x, v);
#pragma unroll
        for (int k = 0; k < NR; k++) {
            al[k] = ks->rho[k] / v[k];
            if (blockIdx.x == 0 && threadIdx.x == 0 && !ks->done[k]) ks->alpha[k] = al[k];
        }
    }
#pragma unroll
    for (int k = 0; k < NR; k++) {
        skip[k] = ks->done[k] != 0;
        if (!fold) al[k] = ks->alpha[k];
        dsum[3 * k] = dsum[3 * k + 1] = dsum[3 * k + 2] = 0.0;
    }
    auto S = [&](int k, int j) -> double { return fma(-al[k], w.v[k][j], w.r[k][j]); };
    for_rows<ND, NR>(A, r0, r1, [&](int k, int j) { return skip[k] ? 0.0 : S(k, j); },
                     [&](int r, const double (&ax)[NR]) {
#pragma unroll
                         for (int k = 0; k < NR; k++) {
                             if (skip[k]) continue;
                             const double sv = S(k, r);
                             w.s[k][r] = sv;
                             w.t[k][r] = ax[k];
                             dsum[3 * k] += ax[k] * sv;
                             dsum[3 * k + 1] += ax[k] * ax[k];
                             dsum[3 * k + 2] += sv * sv;
                         }
                     });
    block_partials<3 * NR>(dsum, partials, b, gridDim.x);
}

template <int NR>
struct EpiBiOmega {
    KState *ks;
    __device__ void operator()(const double (&v)[3 * NR]) const
    {
        if (ks->all_done) return;
        for (int k = 0; k < NR; k++) {
            if (ks->done[k]) continue;
            const double sn = sqrt(v[3 * k + 2]);
            ks->sn[k] = sn;
            ks->half[k] = (sn <= ks->tol[k]) ? 1 : 0;
            if (!ks->half[k]) ks->omega[k] = v[3 * k] / v[3 * k + 1];
        }
    }
};

// x += alpha p + omega s ; r = s - omega t ; partials of (r,r), (r^,r)
template <int NR>
__global__ void __launch_bounds__(BLOCK) k_bi_xr(int n, BiVecs w, KState *ks, const double *fold, double *partials,
                                                 int chunk)
{
    if (ks->all_done) return;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = b * chunk, i1 = min(n, i0 + chunk);
    bool skip[NR], half[NR];
    double al[NR], om[NR], acc[2 * NR];
    if (fold) {   // EpiBiOmega here; what block 0 stores is read by EpiBiXr only
        double v[3 * NR];
        fold_sums<3 * NR>(fold, gridDim.x, v);
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const double sn = sqrt(v[3 * k + 2]);
            half[k] = sn <= ks->tol[k];
            om[k] = v[3 * k] / v[3 * k + 1];
            if (blockIdx.x == 0 && threadIdx.x == 0 && !ks->done[k]) {
                ks->sn[k] = sn;
                ks->half[k] = half[k] ? 1 : 0;
                if (!half[k]) ks->omega[k] = om[k];
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NR; k++) {
        skip[k] = ks->done[k] != 0;
        al[k] = ks->alpha[k];
        if (!fold) {
            half[k] = ks->half[k] != 0;
            om[k] = ks->omega[k];
        }
        acc[2 * k] = acc[2 * k + 1] = 0.0;
    }
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
#pragma unroll
        for (int k = 0; k < NR; k++) {
            if (skip[k]) continue;
            if (half[k]) {
                w.x[k][i] = fma(al[k], w.p[k][i], w.x[k][i]);
            } else {
                const double sv = w.s[k][i];
                w.x[k][i] = fma(om[k], sv, fma(al[k], w.p[k][i], w.x[k][i]));
                const double r = fma(-om[k], w.t[k][i], sv);
                w.r[k][i] = r;
                acc[2 * k] += r * r;
                acc[2 * k + 1] += w.rh[k][i] * r;
            }
        }
    }
    block_partials<2 * NR>(acc, partials, b, gridDim.x);
}

template <int NR>
struct EpiBiXr {
    KState *ks;
    __device__ void operator()(const double (&v)[2 * NR]) const
    {
        if (ks->all_done) return;
        int all = 1;
        for (int k = 0; k < NR; k++) {
            if (!ks->done[k]) {
                ks->iters[k] += 1;
                if (ks->half[k]) {
                    ks->rnorm[k] = ks->sn[k];
                    ks->done[k] = 1; ks->conv[k] = 1;
                } else {
                    const double rn = sqrt(v[2 * k]);
                    ks->rnorm[k] = rn;
                    ks->rho_old[k] = ks->rho[k];
                    ks->rho[k] = v[2 * k + 1];
                    if (rn <= ks->tol[k]) { ks->done[k] = 1; ks->conv[k] = 1; }
                    else if (ks->rho[k] == 0.0 || ks->iters[k] >= ks->maxit || !(rn == rn)) ks->done[k] = 1;
                    else ks->beta[k] = (ks->rho[k] / ks->rho_old[k]) * (ks->alpha[k] / ks->omega[k]);
                }
            }
            all &= ks->done[k];
        }
        ks->all_done = all;
    }
};

static_assert(sizeof(KState) % 8 == 0 && sizeof(KState) / 8 <= 500, "published as doubles below the mirror's other slots");

int wait_pub(Ctx *c)
{
    const unsigned long long *flag = (const unsigned long long *)(c->hscal + PUB_FLAG);
    for (unsigned spin = 1;; spin++) {
        if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == c->pub_seq) return MC_OK;
        if ((spin & 0x3fff) == 0) {
            // the stream must still be at work on it: one that has drained or
            // failed without publishing ends the wait
            const hipError_t e = hipStreamQuery(c->stream);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();
                continue;
            }
            MC_HIP(c, e);
            if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == c->pub_seq) return MC_OK;
            c->err = "a published result did not arrive";
            return MC_ERR_HIP;
        }
    }
}

// A solver's state copied back and waited for (graph replays, which hold no
// publication).
static int poll_done(Ctx *c, KState *ks, KState *host)
{
    MC_HIP(c, hipMemcpyAsync(host, ks, sizeof(KState), hipMemcpyDeviceToHost, c->stream));
    MC_HIP(c, hipStreamSynchronize(c->stream));
    return MC_OK;
}

// Iterations to enqueue before the next host poll: the remaining count
// predicted from the last observed residual reduction rate (at least 1).
static int predict_batch(double rn_prev, double rn, int its, double tol, int cap)
{
    if (its <= 0 || !(rn > 0) || !(rn_prev > 0) || rn >= rn_prev) return 1;
    const double rate = std::pow(rn / rn_prev, 1.0 / its);
    const double need = std::log(tol / rn) / std::log(rate);
    int k = (int)std::floor(need);
    return std::max(1, std::min(k, cap));
}

template <int NR>
static int bicgstab_nr(Ctx *c, const double *vals, double *const *b, double *const *x, double rtol, int maxit,
                       mc_solve_status *st, bool warm, double *const *r0)
{
    static_assert(NR <= 4, "NR");
    const int n = c->N;
    // seven work vectors per RHS (r, s, t and two each of p, v) from the 24
    // FP64 work vectors and the 8 scratch vectors (sized for doubles)
    double *pool[32];
    int np = 0;
    for (int i = 0; i < 24; i++) pool[np++] = c->wk[i];
    for (int i = 0; i < 8; i++) pool[np++] = (double *)c->wk32[i];
    BiVecs w[2] = {};
    int q = 0;
    for (int k = 0; k < NR; k++) {
        double *r = pool[q++], *s = pool[q++], *t = pool[q++];
        double *pa = pool[q++], *pb = pool[q++], *va = pool[q++], *vb = pool[q++];
        for (int e = 0; e < 2; e++) {
            w[e].b[k] = b[k]; w[e].x[k] = x[k]; w[e].rh[k] = b[k];
            w[e].r[k] = r; w[e].s[k] = s; w[e].t[k] = t;
        }
        w[0].p[k] = pa; w[0].v[k] = va; w[0].po[k] = pb; w[0].vo[k] = vb;
        w[1].p[k] = pb; w[1].v[k] = vb; w[1].po[k] = pa; w[1].vo[k] = va;
    }
    const double *dia = fine_dia_of(c, vals);
    if (c->fine_nd && !dia) { c->err = "bicgstab: matrix without its diagonal storage"; return MC_ERR_STATE; }
    const Mat<double> A = fine_mat(c, vals, dia);
    KState *ks = (KState *)c->dscal;
    KState *hs = (KState *)c->hscal;
    const Grid g = grid_for(n);
    // short grids: alpha and omega are formed by their consumers (fold_sums);
    // a folding kernel reads one half of the partials buffer and writes the other
    const bool fold = fold_on(c, g);
    double *red2 = fold ? c->red + RED_PARTIALS / 2 : c->red;
    if (warm && r0) {
        // the assembly formed r = b - A x0 (same x0, same matrix): it is the r vector
        for (int k = 0; k < NR; k++) w[0].r[k] = w[1].r[k] = r0[k];
        hipLaunchKernelGGL(k_bi_init_r0<NR>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, w[0], c->red, g.chunk);
        launch_finish<3 * NR>(c->stream, c->red, g.blocks, EpiBiInitX0<NR>{ks, rtol, maxit});
    } else if (warm) {
        MC_DISPATCH_ND(nd_code(A), (k_bi_init_x0<ND_, NR>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, w[0], c->red,
                       g.chunk);
        launch_finish<3 * NR>(c->stream, c->red, g.blocks, EpiBiInitX0<NR>{ks, rtol, maxit});
    } else {
        hipLaunchKernelGGL(k_bi_init<NR>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, w[0], c->red, g.chunk);
        launch_finish<NR>(c->stream, c->red, g.blocks, EpiBiInit<NR>{ks, rtol, maxit});
    }
    MC_LAUNCH_CHECK(c);
    // A; r, p', v', r^ read and p, v written per RHS
    const double mbytes = mat_bytes(A, c->nnz, 8) + 48.0 * NR * n;
    // first batch: as many iterations as the last solve for these unknowns
    // took (surplus iterations return at once on the device), so a solve that
    // repeats its count needs one host poll
    int hslot = -1;
    for (int k = 0; k < Ctx::BI_HIST && hslot < 0; k++)
        if (c->bi_hist_key[k] == x[0]) hslot = k;
    int it = 0, batch = hslot >= 0 ? std::max(1, std::min(c->bi_hist_its[hslot], 8)) : 1;
    double rn_prev = -1.0;
    for (;;) {
        for (int j = 0; j < batch && it < maxit; j++, it++) {
            const BiVecs &W = w[it & 1];
            {
                KTimer kt(c, MC_KC_BICG, mbytes);
                MC_DISPATCH_ND(nd_code(A), (k_bi_pv<ND_, NR>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, W, ks, c->red,
                               g.chunk, warm && it == 0 ? 1 : 0);
            }
            if (!fold) launch_finish<NR>(c->stream, c->red, g.blocks, EpiBiAlpha<NR>{ks});
            MC_DISPATCH_ND(nd_code(A), (k_bi_st<ND_, NR>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, W, ks,
                           fold ? (const double *)c->red : nullptr, red2, g.chunk);
            if (!fold) launch_finish<3 * NR>(c->stream, red2, g.blocks, EpiBiOmega<NR>{ks});
            hipLaunchKernelGGL(k_bi_xr<NR>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, W, ks,
                               fold ? (const double *)red2 : nullptr, c->red, g.chunk);
            const bool last = j == batch - 1 || it == maxit - 1;
            launch_finish<2 * NR>(c->stream, c->red, g.blocks, EpiBiXr<NR>{ks},
                                  last ? make_pub(c, ks, 0, sizeof(KState)) : Pub());
        }
        MC_LAUNCH_CHECK(c);
        MC_TRY(wait_pub(c));
        c->st.host_polls++;
        if (hs->all_done || it >= maxit) break;
        double rn = 0.0;
        for (int k = 0; k < NR; k++)
            if (!hs->done[k]) rn = std::max(rn, hs->rnorm[k] / std::max(hs->tol[k], 1e-300));
        batch = predict_batch(rn_prev, rn, batch, 1.0, 8);
        rn_prev = rn;
    }
    {
        int its = 0;
        for (int k = 0; k < NR; k++) its = std::max(its, hs->iters[k]);
        if (hslot < 0) {   // a free slot, else the oldest entry's
            hslot = 0;
            while (hslot < Ctx::BI_HIST - 1 && c->bi_hist_key[hslot]) hslot++;
            if (c->bi_hist_key[hslot]) {
                for (int k = 0; k + 1 < Ctx::BI_HIST; k++) {
                    c->bi_hist_key[k] = c->bi_hist_key[k + 1];
                    c->bi_hist_its[k] = c->bi_hist_its[k + 1];
                }
                hslot = Ctx::BI_HIST - 1;
            }
            c->bi_hist_key[hslot] = x[0];
        }
        c->bi_hist_its[hslot] = its;
    }
    if (st) {
        st->iterations = 0; st->converged = 1; st->relres = 0.0; st->outer = 0; st->guess_used = 0; st->bnorm = 0.0;
        for (int k = 0; k < NR; k++) {
            st->iterations += hs->iters[k];
            st->converged &= hs->conv[k];
            const double rr = hs->bnorm[k] > 0 ? hs->rnorm[k] / hs->bnorm[k] : 0.0;
            st->relres = std::max(st->relres, rr);
            st->bnorm = std::max(st->bnorm, hs->bnorm[k]);
        }
    }
    return MC_OK;
}

int bicgstab_solve(Ctx *c, const double *vals, int nr, double *const *b, double *const *x, double rtol, int maxit,
                   mc_solve_status *st, bool warm, double *const *r0)
{
    switch (nr) {
    case 1: return bicgstab_nr<1>(c, vals, b, x, rtol, maxit, st, warm, r0);
    case 2: return bicgstab_nr<2>(c, vals, b, x, rtol, maxit, st, warm, r0);
    case 3: return bicgstab_nr<3>(c, vals, b, x, rtol, maxit, st, warm, r0);
    case 4: return bicgstab_nr<4>(c, vals, b, x, rtol, maxit, st, warm, r0);
    default: c->err = "bicgstab: 1..4 right-hand sides"; return MC_ERR_ARG;
    }
}

// ------------------------------------------------- generic reductions --
__global__ void __launch_bounds__(BLOCK) k_sum(int n, const double *v, double *partials, int chunk)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = b * chunk, i1 = min(n, i0 + chunk);
    double acc[1] = {0.0};
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) acc[0] += v[i];
    block_partials<1>(acc, partials, b, gridDim.x);
}

struct EpiScale {
    double *out;
    double scale;
    __device__ void operator()(const double (&v)[1]) const { *out = v[0] * scale; }
};

// *out = scale * sum(v[0..n)) on the stream
static void sum_scaled(Ctx *c, const double *v, int n, double *out, double scale)
{
    const Grid g = grid_for(n);
    hipLaunchKernelGGL(k_sum, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, v, c->red, g.chunk);
    launch_finish<1>(c->stream, c->red, g.blocks, EpiScale{out, scale});
}

__global__ void k_sub_scalar(int n, const double *in, const double *s, double *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[i] - *s;
}

int mean_project(Ctx *c, const double *b, double *out, int n)
{
    double *mean = c->dscal + 512;
    sum_scaled(c, b, n, mean, 1.0 / (double)n);
    hipLaunchKernelGGL(k_sub_scalar, dim3(div_up(n, BLOCK)), dim3(BLOCK), 0, c->stream, n, b, mean, out);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

// max(PP[0], max_{i>=1} |PP[i]|), the reference's Pressure_correction_max
// (FlowSolver.inl:2371-2378): block maxima, then one block combines them
__global__ void __launch_bounds__(BLOCK) k_maxabs(int n, const double *v, double *partials, int chunk)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = b * chunk, i1 = min(n, i0 + chunk);
    double m = 0.0;
    for (int i = max(i0, 1) + threadIdx.x; i < i1; i += BLOCK) m = fmax(m, fabs(v[i]));
    __shared__ double lds[BLOCK / 64];
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) partials[b] = fmax(fmax(lds[0], lds[1]), fmax(lds[2], lds[3]));
}

__global__ void __launch_bounds__(BLOCK) k_maxabs_finish(const double *v, const double *partials, int nblocks,
                                                         double *out, Pub pub)
{
    double mm = 0.0;
    for (int i = threadIdx.x; i < nblocks; i += BLOCK) mm = fmax(mm, partials[i]);
    __shared__ double lds[BLOCK / 64];
    for (int off = 32; off > 0; off >>= 1) mm = fmax(mm, __shfl_down(mm, off, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = mm;
    __syncthreads();
    if (threadIdx.x == 0) {
        mm = fmax(fmax(lds[0], lds[1]), fmax(lds[2], lds[3]));
        const double p0 = v[0];
        *out = (p0 != p0) ? p0 : ((mm > p0) ? mm : p0);
    }
    publish(pub);
}

int reduce_maxabs_pp(Ctx *c, const double *v, double *out_host)
{
    const Grid g = grid_for(c->N);
    double *d = c->dscal + 520;
    hipLaunchKernelGGL(k_maxabs, dim3(g.blocks), dim3(BLOCK), 0, c->stream, c->N, v, c->red, g.chunk);
    hipLaunchKernelGGL(k_maxabs_finish, dim3(1), dim3(BLOCK), 0, c->stream, v, c->red, g.blocks, d,
                       make_pub(c, d, 520, sizeof(double)));
    MC_LAUNCH_CHECK(c);
    MC_TRY(wait_pub(c));
    *out_host = c->hscal[520];
    return MC_OK;
}

// =================================================================== AMG ==
// Host-side aggregation: three passes of greedy pairwise matching (strongest
// unmatched neighbour, ties to the lowest column) per level -> aggregates of
// at most 8 cells.  Done once per context; later matrices on the same pattern
// only recompute the Galerkin values on the GPU.
struct HostCSR {
    int n = 0;
    std::vector<int> rp, col;
    std::vector<double> val;
};

static void pairwise_pass(const HostCSR &A, std::vector<int> &agg, int &nc)
{
    agg.assign(A.n, -1);
    nc = 0;
    for (int i = 0; i < A.n; i++) {
        if (agg[i] >= 0) continue;
        int best = -1;
        double bw = 0.0;
        for (int k = A.rp[i]; k < A.rp[i + 1]; k++) {
            const int j = A.col[k];
            if (j == i || agg[j] >= 0) continue;
            const double w = -A.val[k];
            if (w > bw * (1.0 + 1e-12)) { best = j; bw = w; }
        }
        agg[i] = nc;
        if (best >= 0) agg[best] = nc;
        nc++;
    }
}

// Galerkin product with piecewise-constant prolongation; also returns, for
// every coarse nonzero, the list of fine nonzeros summed into it.
static void galerkin(const HostCSR &A, const std::vector<int> &agg, int nc, HostCSR &Ac, std::vector<int> *gptr,
                     std::vector<int> *gmap)
{
    std::vector<int> mp(nc + 1, 0), mem(A.n);
    for (int i = 0; i < A.n; i++) mp[agg[i] + 1]++;
    for (int I = 0; I < nc; I++) mp[I + 1] += mp[I];
    {
        std::vector<int> pos(mp.begin(), mp.end() - 1);
        for (int i = 0; i < A.n; i++) mem[pos[agg[i]]++] = i;
    }
    Ac.n = nc;
    Ac.rp.assign(nc + 1, 0);
    Ac.col.clear();
    Ac.val.clear();
    std::vector<std::pair<int, int>> ent;  // (coarse col, fine nnz)
    std::vector<int> gp, gm;
    gp.push_back(0);
    for (int I = 0; I < nc; I++) {
        ent.clear();
        for (int t = mp[I]; t < mp[I + 1]; t++) {
            const int i = mem[t];
            for (int k = A.rp[i]; k < A.rp[i + 1]; k++) ent.emplace_back(agg[A.col[k]], k);
        }
        std::sort(ent.begin(), ent.end());
        for (size_t e = 0; e < ent.size();) {
            const int J = ent[e].first;
            double s = 0.0;
            size_t f = e;
            for (; f < ent.size() && ent[f].first == J; f++) {
                s += A.val[ent[f].second];
                gm.push_back(ent[f].second);
            }
            Ac.col.push_back(J);
            Ac.val.push_back(s);
            gp.push_back((int)gm.size());
            e = f;
        }
        Ac.rp[I + 1] = (int)Ac.col.size();
    }
    if (gptr) *gptr = std::move(gp);
    if (gmap) *gmap = std::move(gm);
}

__global__ void k_gather_sum(int nnzc, const int *gptr, const int *gmap, const double *vf, double *vc)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nnzc) return;
    double s = 0.0;
    for (int t = gptr[k]; t < gptr[k + 1]; t++) s += vf[gmap[t]];
    vc[k] = s;
}

__global__ void k_diag_inv(int n, const int *rp, const int *col, const double *v, double *dinv, float *dinv32,
                           float *v32, int nnz)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        double d = 0.0;
        for (int k = rp[i]; k < rp[i + 1]; k++) if (col[k] == i) d = v[k];
        const double di = (d != 0.0) ? 1.0 / d : 0.0;
        dinv[i] = di;
        dinv32[i] = (float)di;
    }
    for (int k = i; k < nnz; k += gridDim.x * blockDim.x) v32[k] = (float)v[k];
}

// A level with diagonal storage: one pass over its CSR rows fills the FP64 and
// FP32 diagonal copies and the inverse diagonal.
__global__ void k_level_dia(int n, const int *rp, const int *col, const int *map, const double *v, double *dia,
                            float *dia32, double *dinv, float *dinv32, int sym_skip, _Float16 *hoff, float *diag32)
{
    // sym_skip > 0: the FP64 copy is symmetric storage without the sym_skip
    // lower diagonals; the FP32 copy keeps all of them
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double d = 0.0;
    const size_t shift = (size_t)sym_skip * n;
    for (int k = rp[i]; k < rp[i + 1]; k++) {
        const double x = v[k];
        const int m = map[k];
        if (col[k] == i) d = x;
        dia32[m] = (float)x;
        if (!sym_skip || col[k] >= i) dia[(size_t)m - shift] = x;
    }
    const double di = (d != 0.0) ? 1.0 / d : 0.0;
    dinv[i] = di;
    dinv32[i] = (float)di;
    if (hoff) {   // 7 diagonals, the main one in the middle
        diag32[i] = (float)d;
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            if (col[k] == i) continue;
            const int dd = (map[k] - i) / n;
            hoff[(size_t)(dd < 3 ? dd : dd - 1) * n + i] = (_Float16)(v[k] / d);
        }
    }
}

// Dense regularised coarsest operator A + alpha 11^T (alpha = mean diag / n):
// for a mean-zero right-hand side its inverse returns the mean-zero solution
// of the singular Neumann system.  In-place Gauss-Jordan inversion (SPD, no
// pivoting) of n <= 128 rows in one workgroup of 1024 threads, the matrix
// held in registers and padded with zeros to 128 x 128.  Only the first n
// pivots are taken; the zero padding then stays zero and the leading n x n
// block holds the inverse.
// One CU, a chain of n steps: what counts is a step's length.  Thread t owns
// the 4 x 4 tile at rows 4 (t / 32), columns 4 (t % 32), so a step needs four
// values of the pivot row and four of the pivot column (64 bytes of LDS reads
// a thread; a 1 x 16 strip needs 136), and the half wave that holds the pivot row
// scales it before it is published, so one barrier a step suffices (row and
// column are double-buffered by the step's parity).  Four pivots an iteration:
// the pivot's place in a tile is then a constant and a step is 16 products and
// no selection of registers (by a running index the selections were most of a
// step, and the kernel the more slowed by others' waves on its CU).  128 rows
// with the device idle 235 -> 70 us, beside the learned guess at modifier 128
// 245 -> 170 us.
//
// The matrix: CSR, or a box level's symmetric diagonals (main, +x, +y, +z).
struct DenseSrc {
    int n;
    const int *rp, *col;
    const double *v;        // CSR values, or the box level's dia
    int bx, by;             // box: row length, rows per plane (0: CSR)
};
__device__ __forceinline__ double dense_src_at(const DenseSrc &s, int i, int j)
{
    if (!s.bx) {
        for (int k = s.rp[i]; k < s.rp[i + 1]; k++)
            if (s.col[k] == j) return s.v[k];
        return 0.0;
    }
    // the upper entry of the pair (lo, lo + stride); each direction's
    // diagonal holds zero where the neighbour does not exist
    const int lo = i < j ? i : j, d = i < j ? j - i : i - j;
    if (d == 0) return s.v[i];
    double r = 0.0;
    if (d == 1) r += s.v[(size_t)s.n + lo];
    if (d == s.bx) r += s.v[2 * (size_t)s.n + lo];
    if (d == s.bx * s.by) r += s.v[3 * (size_t)s.n + lo];
    return r;
}

__global__ void __launch_bounds__(1024) k_dense_inverse(DenseSrc src, double *inv)
{
    constexpr int TQ = DENSE_MAX / 32;   // tile edge
    static_assert(TQ == 4, "32 x 32 threads of 4 x 4");
    __shared__ __align__(16) double colk[2][DENSE_MAX];
    __shared__ __align__(16) double rowk[2][DENSE_MAX];
    __shared__ double red[1024 / 64];
    const int tid = threadIdx.x, n = src.n;
    const int i0 = TQ * (tid >> 5), j0 = TQ * (tid & 31);
    double s = (tid < n) ? dense_src_at(src, tid, tid) : 0.0;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < 1024 / 64; w++) tot += red[w];
    const double alpha = (tot / n) / n;
    double m[TQ][TQ];
#pragma unroll
    for (int a = 0; a < TQ; a++) {
        const int i = i0 + a;
#pragma unroll
        for (int b = 0; b < TQ; b++) {
            m[a][b] = (i < n && j0 + b < n) ? alpha : 0.0;
            if (src.bx && i < n && j0 + b < n) m[a][b] += dense_src_at(src, i, j0 + b);
        }
        if (!src.bx && i < n)   // a CSR row is read once for its four elements
            for (int k = src.rp[i]; k < src.rp[i + 1]; k++) {
                const int jb = src.col[k] - j0;
                const double v = src.v[k];
#pragma unroll
                for (int b = 0; b < TQ; b++)
                    if (b == jb) m[a][b] += v;
            }
    }
    const int rg = tid >> 5, cg = tid & 31;
    for (int k0 = 0; k0 < n; k0 += TQ)
#pragma unroll
        for (int q = 0; q < TQ; q++) {
            const int buf = q & 1;
            if (k0 + q >= n) break;
            const bool rows = rg == k0 / TQ, cols = cg == k0 / TQ;   // this tile holds row / column k0 + q
            if (rows) {
                // the pivot is the value of the half wave's lane k0 / 4
                const double rk = 1.0 / __shfl(m[q][q], (tid & 32) | (k0 / TQ), 64);
#pragma unroll
                for (int b = 0; b < TQ; b++) rowk[buf][j0 + b] = ((cols && b == q) ? 1.0 : m[q][b]) * rk;
            }
            if (cols)
#pragma unroll
                for (int a = 0; a < TQ; a++) { colk[buf][i0 + a] = m[a][q]; m[a][q] = 0.0; }
            __syncthreads();
            double pr[TQ], pc[TQ];
#pragma unroll
            for (int b = 0; b < TQ; b++) pr[b] = rowk[buf][j0 + b];
#pragma unroll
            for (int a = 0; a < TQ; a++) pc[a] = colk[buf][i0 + a];
#pragma unroll
            for (int a = 0; a < TQ; a++)
#pragma unroll
                for (int b = 0; b < TQ; b++) m[a][b] = m[a][b] - pc[a] * pr[b];
            if (rows)
#pragma unroll
                for (int b = 0; b < TQ; b++) m[q][b] = pr[b];
        }
    // stored transposed: k_dense_apply's threads (rows) then read consecutive words
#pragma unroll
    for (int a = 0; a < TQ; a++)
#pragma unroll
        for (int b = 0; b < TQ; b++)
            if (i0 + a < n && j0 + b < n) inv[(size_t)(j0 + b) * n + i0 + a] = m[a][b];
}

// Pairwise matching on a box of even sides pairs along x, y and z in turn: the
// aggregates are its 2 x 2 x 2 blocks, numbered in order.  Such a level's transfers
// need no index arrays (k_box_restrict, k_box_jac_prolong).
static void regular_level(AmgLevel &L, const HostCSR &A, const std::vector<int> &agg, int nc)
{
    if (L.nd != 7 || L.off[4] != 1 || L.off[5] <= 1 || L.off[6] <= L.off[5]) return;
    const int nx = L.off[5], nxny = L.off[6];
    for (int d = 0; d < 7; d++)
        if (L.off[d] != -L.off[6 - d]) return;
    if (nxny % nx || A.n % nxny) return;
    const int ny = nxny / nx, nz = A.n / nxny, cx = (nx + 1) >> 1, cy = (ny + 1) >> 1, cz = (nz + 1) >> 1;
    if (nc != cx * cy * cz) return;
    int i = 0;
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < ny; y++)
            for (int x = 0; x < nx; x++, i++) {
                if (agg[i] != (x >> 1) + cx * ((y >> 1) + cy * (z >> 1))) return;
                for (int k = A.rp[i]; k < A.rp[i + 1]; k++) {   // entries of coordinate neighbours only
                    const int o = A.col[k] - i;
                    if ((o == 1 && x + 1 == nx) || (o == -1 && x == 0) || (o == nx && y + 1 == ny) ||
                        (o == -nx && y == 0))
                        return;
                }
            }
    L.rx = nx; L.ry = ny; L.rz = nz;
}


static int amg_build(Ctx *c, const double *vals);

// Aggregation-AMG hierarchy from the pressure matrix (host aggregation and
// Galerkin pattern, then the first values on the device); the wall time up to
// the first values' completion goes to the statistics
int amg_setup(Ctx *c, const double *vals)
{
    const auto t0 = std::chrono::steady_clock::now();
    MC_TRY(amg_build(c, vals));
    MC_HIP(c, hipStreamSynchronize(c->stream));
    c->st.amg_setups += 1;
    c->st.amg_setup_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return MC_OK;
}

// --------------------------------------------------- box hierarchy --
// On a box pattern the hierarchy is built by halving: aggregates are 2 x 2 x 2
// cells (odd lengths leave a thinner last layer), every level is again a box
// of 7 diagonals, and nothing is formed on the host.  Pairwise matching gives
// the same aggregates where all lengths are powers of two; elsewhere its
// aggregates are irregular from the second level on and every coarse level
// falls back to CSR.  Measured on a 100 x 50 x 50 box, mixed form to 1e-11: 15
// -> 8 PCG iterations, a solve 7.6 -> 1.36 ms; on lognormal momentum diagonals
// (sigma 0.2 / 1 / 2 / 3, 66 x 33 x 33, 1e-10) 21 / 22 / 38 / 120 -> 8 / 12 /
// 30 / 97 iterations.
// A direction is halved when the first matrix's mean coupling along it is at
// least a quarter of the strongest direction's (the usual strength threshold:
// point smoothing does not reach errors along weaker ones), so a stretched
// box is coarsened along its strong directions first.
struct BoxDims {
    int nx, ny, nz, n;       // this level
    int cx, cy, cz, nc;      // the next one
    int sx, sy, sz;          // shift per direction: 1 halved, 0 kept
};

static BoxDims box_dims(const AmgLevel &L)
{
    BoxDims b;
    b.n = L.n;
    if (L.bx) {
        b.nx = L.bx; b.ny = L.by; b.nz = L.bz;
        b.sx = L.sx; b.sy = L.sy; b.sz = L.sz;
    } else {
        b.nx = L.rx; b.ny = L.ry; b.nz = L.rz;
        b.sx = b.sy = b.sz = 1;
    }
    b.cx = (b.nx + b.sx) >> b.sx; b.cy = (b.ny + b.sy) >> b.sy; b.cz = (b.nz + b.sz) >> b.sz;
    b.nc = b.cx * b.cy * b.cz;
    return b;
}

// sums of -A[i, i + stride] over the CSR matrix's upper entries, per direction
__global__ void __launch_bounds__(BLOCK) k_box_strength(int n, const int *rp, const int *col, const double *v, int nx,
                                                        int nxny, double *partials, int chunk)
{
    const int i0 = blockIdx.x * chunk, i1 = min(n, i0 + chunk);
    double acc[3] = {0.0, 0.0, 0.0};
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK)
        for (int k = rp[i]; k < rp[i + 1]; k++) {
            const int d = col[k] - i;
            if (d == 1) acc[0] -= v[k];
            else if (d == nx) acc[1] -= v[k];
            else if (d == nxny) acc[2] -= v[k];
        }
    block_partials<3>(acc, partials, blockIdx.x, gridDim.x);
}

struct EpiStore3 {
    double *out;
    __device__ void operator()(const double (&v)[3]) const { out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; }
};

// Galerkin product P^T A P of a box level with piecewise-constant P, symmetric
// storage (main, +x, +y, +z): a coarse cell's main entry is its members' main
// entries plus twice the couplings between them, its upper entry the sum of
// the couplings across that face.  One thread per coarse cell; the FP32 copy
// (all seven diagonals) takes the upper entry in both rows.
__global__ void __launch_bounds__(BLOCK) k_box_galerkin(BoxDims b, const double *dia, double *cdia, float *cdia32,
                                                        double *cdinv, float *cdinv32)
{
    const int I = blockIdx.x * BLOCK + threadIdx.x;
    if (I >= b.nc) return;
    const int X = I % b.cx, Y = (I / b.cx) % b.cy, Z = I / (b.cx * b.cy);
    const size_t n = b.n;
    double d = 0.0, off = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
    for (int k = 0; k <= b.sz; k++)
        for (int j = 0; j <= b.sy; j++)
            for (int i = 0; i <= b.sx; i++) {
                const int x = (X << b.sx) + i, y = (Y << b.sy) + j, z = (Z << b.sz) + k;
                if (x >= b.nx || y >= b.ny || z >= b.nz) continue;
                const size_t f = x + (size_t)b.nx * (y + (size_t)b.ny * z);
                d += dia[f];
                const double ax = dia[n + f], ay = dia[2 * n + f], az = dia[3 * n + f];
                if (i < b.sx) off += ax; else ux += ax;   // (a missing neighbour's entry is zero)
                if (j < b.sy) off += ay; else uy += ay;
                if (k < b.sz) off += az; else uz += az;
            }
    const double D = d + 2.0 * off;
    const size_t nc = b.nc;
    cdia[I] = D; cdia[nc + I] = ux; cdia[2 * nc + I] = uy; cdia[3 * nc + I] = uz;
    const double di = (D != 0.0) ? 1.0 / D : 0.0;
    cdinv[I] = di; cdinv32[I] = (float)di;
    // FP32: diagonals -z -y -x main +x +y +z
    cdia32[3 * nc + I] = (float)D;
    if (X + 1 < b.cx) { cdia32[4 * nc + I] = (float)ux; cdia32[2 * nc + I + 1] = (float)ux; }
    if (Y + 1 < b.cy) { cdia32[5 * nc + I] = (float)uy; cdia32[1 * nc + I + b.cx] = (float)uy; }
    if (Z + 1 < b.cz) { cdia32[6 * nc + I] = (float)uz; cdia32[0 * nc + I + (size_t)b.cx * b.cy] = (float)uz; }
}

static int level_vectors(Ctx *c, AmgLevel &L)
{
    MC_TRY(dalloc(c, &L.dinv, L.n));
    MC_TRY(dalloc(c, &L.dinv32, L.n));
    MC_TRY(dalloc(c, &L.x, L.n)); MC_TRY(dalloc(c, &L.b, L.n)); MC_TRY(dalloc(c, &L.t, L.n));
    MC_TRY(dalloc(c, &L.x32, L.n)); MC_TRY(dalloc(c, &L.b32, L.n)); MC_TRY(dalloc(c, &L.t32, L.n));
    return MC_OK;
}

// a hierarchy rebuilt (after a change of options) first releases the
// old one: every allocation charged to MC_MEM_AMG is made by its build
static int amg_release(Ctx *c)
{
    if (c->amg.empty()) return MC_OK;
    c->amg.clear();
    c->amg_dense = nullptr;
    c->amg_ready = false;
    return dfree_category(c, MC_MEM_AMG);
}

// rows up to which a level is the dense coarsest one
static int amg_coarse_bound(const Ctx *c) { return std::max(8, std::min(c->opt.amg_coarse_max, DENSE_MAX)); }

static bool box_wanted(const Ctx *c);

static int amg_finish_build(Ctx *c, const double *vals)
{
    const int nco = c->amg.back().n;
    c->amg_coarse_n = nco;
    MC_TRY(dalloc(c, &c->amg_dense, (size_t)nco * nco));
    c->amg_ready = true;
    c->amg_box_wanted = box_wanted(c);
    c->amg_updates = 0;
    // level 0's diagonal copies were just allocated and zeroed: whatever an
    // earlier pressure assembly wrote went to the hierarchy released above
    c->pa_dia_fresh = false;
    return amg_update_values(c, vals);
}

// Which solves take it: a relative tolerance of 1e-9 or below, no gradient
// limiter.  The preconditioner does not change what a solve converges to, only
// which of the vectors within its tolerance it stops at.  At 1e-8 that choice
// still shows: the cross-stream velocities after one timestep differ by up to
// 5e-9 (relative, modifiers 33 to 100) between the two hierarchies, so those
// runs keep the matched aggregates and with them their results.  At 1e-10 the
// two differ by 3e-11 and less, and the faster one is taken.  With the limiter
// on, cross-stream velocities that are zero up to rounding follow the last bit
// of every solve.
constexpr double BOX_RTOL = 1e-9;

// The options' choice.  A hierarchy built for the other one is replaced before
// the next solve (amg_current), so results depend on the options in force and
// not on the ones before them.
static bool box_wanted(const Ctx *c)
{
    return c->box_nx && c->fine_nd == 7 && c->N > amg_coarse_bound(c) && c->opt.p_rtol <= BOX_RTOL && !c->opt.limit_grad;
}

static bool amg_current(const Ctx *c) { return c->amg_ready && c->amg_box_wanted == box_wanted(c); }

// *built = false: not wanted (above), or no positive coupling to choose
// directions by (the pairwise build then decides)
static int amg_build_box(Ctx *c, const double *vals, bool *built)
{
    *built = false;
    const int coarse_max = amg_coarse_bound(c);
    if (!box_wanted(c)) return MC_OK;
    const int nx = c->box_nx, ny = c->box_ny, nz = c->box_nz;
    double st[3];
    {
        const Grid g = grid_for(c->N);
        double *d = c->dscal + 630;
        hipLaunchKernelGGL(k_box_strength, dim3(g.blocks), dim3(BLOCK), 0, c->stream, c->N, c->row_ptr, c->col, vals,
                           nx, nx * ny, c->red, g.chunk);
        launch_finish<3>(c->stream, c->red, g.blocks, EpiStore3{d});
        MC_LAUNCH_CHECK(c);
        MC_HIP(c, hipMemcpyAsync(c->hscal + 630, d, 3 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
        MC_HIP(c, hipStreamSynchronize(c->stream));
        const double faces[3] = {(double)(nx - 1) * ny * nz, (double)nx * (ny - 1) * nz, (double)nx * ny * (nz - 1)};
        for (int k = 0; k < 3; k++) st[k] = c->hscal[630 + k] / faces[k];
    }
    // the levels' lengths first: a hierarchy that stops shrinking is not built
    std::vector<AmgLevel> lv;
    AmgLevel L;
    L.bx = nx; L.by = ny; L.bz = nz; L.n = c->N;
    while (L.n > coarse_max) {
        const int len[3] = {L.bx, L.by, L.bz};
        double top = 0.0;
        for (int k = 0; k < 3; k++) if (len[k] > 1) top = std::max(top, st[k]);
        if (!(top > 0.0)) return MC_OK;
        int sh[3];
        for (int k = 0; k < 3; k++) sh[k] = len[k] > 1 && st[k] >= 0.25 * top;
        L.sx = sh[0]; L.sy = sh[1]; L.sz = sh[2];
        const BoxDims b = box_dims(L);
        if (b.nc > (int)(0.75 * L.n)) return MC_OK;
        L.nc = b.nc;
        lv.push_back(L);
        // a halved direction doubles the couplings across the others' faces
        for (int k = 0; k < 3; k++)
            for (int e = 0; e < 3; e++) if (e != k && sh[e]) st[k] *= 2.0;
        L = AmgLevel();
        L.bx = b.cx; L.by = b.cy; L.bz = b.cz; L.n = b.nc;
    }
    lv.push_back(L);
    MC_TRY(amg_release(c));
    c->graph_gen++;   // the PCG graphs hold the old levels' buffers
    for (size_t l = 0; l < lv.size(); l++) {
        AmgLevel &Q = lv[l];
        const int nxny = Q.bx * Q.by;
        const int off[7] = {-nxny, -Q.bx, -1, 0, 1, Q.bx, nxny};
        Q.nd = 7; Q.sym = 1;
        for (int d = 0; d < 7; d++) Q.off[d] = off[d];
        MC_TRY(level_vectors(c, Q));
        MC_TRY(dalloc(c, &Q.dia, (size_t)4 * Q.n));
        MC_TRY(dalloc(c, &Q.dia32, (size_t)7 * Q.n));
        MC_HIP(c, hipMemsetAsync(Q.dia, 0, (size_t)4 * Q.n * 8, c->stream));
        MC_HIP(c, hipMemsetAsync(Q.dia32, 0, (size_t)7 * Q.n * 4, c->stream));
        if (l == 0) {
            Q.row_ptr = c->row_ptr; Q.col = c->col; Q.nnz = c->nnz;
            Q.vals = c->PA_vals;       // the fine level reads the pressure matrix in place
            Q.dia_map = c->fine_map;   // the same pattern and diagonals
            if (c->opt.amg_half) {
                MC_TRY(dalloc(c, &Q.hoff, (size_t)6 * Q.n));
                MC_TRY(dalloc(c, &Q.diag32, (size_t)Q.n));
                MC_HIP(c, hipMemsetAsync(Q.hoff, 0, (size_t)6 * Q.n * sizeof(_Float16), c->stream));
            }
        }
    }
    c->amg = lv;
    *built = true;
    return amg_finish_build(c, vals);
}

static int amg_build(Ctx *c, const double *vals)
{
    MemScope ms(c, MC_MEM_AMG);
    {
        bool built = false;
        MC_TRY(amg_build_box(c, vals, &built));
        if (built) return MC_OK;
    }
    HostCSR A;
    A.n = c->N;
    A.rp.resize(c->N + 1);
    A.col.resize(c->nnz);
    A.val.resize(c->nnz);
    MC_HIP(c, hipMemcpyAsync(A.rp.data(), c->row_ptr, (size_t)(c->N + 1) * 4, hipMemcpyDeviceToHost, c->stream));
    MC_HIP(c, hipMemcpyAsync(A.col.data(), c->col, (size_t)c->nnz * 4, hipMemcpyDeviceToHost, c->stream));
    MC_HIP(c, hipMemcpyAsync(A.val.data(), vals, (size_t)c->nnz * 8, hipMemcpyDeviceToHost, c->stream));
    MC_HIP(c, hipStreamSynchronize(c->stream));
    MC_TRY(amg_release(c));
    const int coarse_max = amg_coarse_bound(c);
    c->graph_gen++;   // the PCG graphs hold the old levels' buffers
    HostCSR cur = std::move(A);
    bool first = true;
    for (;;) {
        AmgLevel L;
        L.n = cur.n;
        L.nnz = (int)cur.col.size();
        if (first) {
            L.row_ptr = c->row_ptr; L.col = c->col;
        } else {
            MC_TRY(dalloc(c, &L.row_ptr, L.n + 1));
            MC_TRY(dalloc(c, &L.col, L.nnz));
            MC_HIP(c, hipMemcpy(L.row_ptr, cur.rp.data(), (size_t)(L.n + 1) * 4, hipMemcpyHostToDevice));
            MC_HIP(c, hipMemcpy(L.col, cur.col.data(), (size_t)L.nnz * 4, hipMemcpyHostToDevice));
        }
        if (first) L.vals = c->PA_vals;   // the fine level reads the pressure matrix in place
        else MC_TRY(dalloc(c, &L.vals, L.nnz));
        MC_TRY(level_vectors(c, L));
        // diagonal storage for this level's pattern
        {
            std::vector<int> offs, map;
            L.nd = 0;
            if (cur.n > coarse_max && dia_analyze(cur.n, cur.rp.data(), cur.col.data(), offs, map)) {
                L.nd = (int)offs.size();
                for (int d = 0; d < L.nd; d++) L.off[d] = offs[d];
                // pressure levels are symmetric: the fine matrix entry for a face is one value
                // written to both rows, and Galerkin levels of it are taken as their upper part
                L.sym = (L.nd % 2 == 1);
                for (int d = 0; d < L.nd && L.sym; d++) L.sym = (L.off[d] == -L.off[L.nd - 1 - d]);
                const int ns = L.sym ? L.nd / 2 + 1 : L.nd;
                MC_TRY(dalloc(c, &L.dia_map, L.nnz));
                MC_HIP(c, hipMemcpy(L.dia_map, map.data(), (size_t)L.nnz * 4, hipMemcpyHostToDevice));
                MC_TRY(dalloc(c, &L.dia, (size_t)ns * L.n));
                MC_TRY(dalloc(c, &L.dia32, (size_t)L.nd * L.n));
                MC_HIP(c, hipMemset(L.dia, 0, (size_t)ns * L.n * 8));
                MC_HIP(c, hipMemset(L.dia32, 0, (size_t)L.nd * L.n * 4));
                if (first && L.nd == 7 && L.sym && c->opt.amg_half) {
                    MC_TRY(dalloc(c, &L.hoff, (size_t)6 * L.n));
                    MC_TRY(dalloc(c, &L.diag32, (size_t)L.n));
                    MC_HIP(c, hipMemset(L.hoff, 0, (size_t)6 * L.n * sizeof(_Float16)));
                }
            }
            if (!L.nd) MC_TRY(dalloc(c, &L.vals32, L.nnz));   // FP32 CSR only where no diagonal copy
        }
        if (cur.n <= coarse_max) {
            c->amg.push_back(L);
            break;
        }
        std::vector<int> agg(cur.n), a1;
        std::iota(agg.begin(), agg.end(), 0);
        HostCSR g = cur;
        int nc = cur.n;
        for (int pass = 0; pass < 3; pass++) {
            int ncn = 0;
            pairwise_pass(g, a1, ncn);
            for (int i = 0; i < cur.n; i++) agg[i] = a1[agg[i]];
            HostCSR gn;
            galerkin(g, a1, ncn, gn, nullptr, nullptr);
            g = std::move(gn);
            nc = ncn;
            if (nc <= coarse_max) break;
        }
        if (nc > (int)(0.75 * cur.n)) { c->err = "aggregation stalled"; return MC_ERR_STATE; }
        HostCSR Ac;
        std::vector<int> gp, gm;
        galerkin(cur, agg, nc, Ac, &gp, &gm);
        L.nc = nc;
        regular_level(L, cur, agg, nc);
        MC_TRY(dalloc(c, &L.agg, L.n));
        MC_HIP(c, hipMemcpy(L.agg, agg.data(), (size_t)L.n * 4, hipMemcpyHostToDevice));
        {
            std::vector<int> mp(nc + 1, 0), mem(L.n);
            for (int i = 0; i < L.n; i++) mp[agg[i] + 1]++;
            for (int I = 0; I < nc; I++) mp[I + 1] += mp[I];
            int maxm = 0;
            for (int I = 0; I < nc; I++) maxm = std::max(maxm, mp[I + 1] - mp[I]);
            if (maxm > 8) { c->err = "aggregate larger than 8"; return MC_ERR_STATE; }
            std::vector<int> pos(mp.begin(), mp.end() - 1);
            for (int i = 0; i < L.n; i++) mem[pos[agg[i]]++] = i;
            MC_TRY(dalloc(c, &L.agg_ptr, nc + 1));
            MC_TRY(dalloc(c, &L.agg_members, L.n));
            MC_HIP(c, hipMemcpy(L.agg_ptr, mp.data(), (size_t)(nc + 1) * 4, hipMemcpyHostToDevice));
            MC_HIP(c, hipMemcpy(L.agg_members, mem.data(), (size_t)L.n * 4, hipMemcpyHostToDevice));
        }
        MC_TRY(dalloc(c, &L.gptr, gp.size()));
        MC_TRY(dalloc(c, &L.gmap, gm.size()));
        MC_HIP(c, hipMemcpy(L.gptr, gp.data(), gp.size() * 4, hipMemcpyHostToDevice));
        MC_HIP(c, hipMemcpy(L.gmap, gm.data(), gm.size() * 4, hipMemcpyHostToDevice));
        c->amg.push_back(L);
        cur = std::move(Ac);
        first = false;
    }
    return amg_finish_build(c, vals);
}

// The main stream waits for the coarsest inverse formed on the side stream.
static int dense_join(Ctx *c)
{
    if (!c->dense_pending) return MC_OK;
    MC_HIP(c, hipStreamWaitEvent(c->stream, c->ev_dense, 0));
    c->dense_pending = false;
    return MC_OK;
}

static int box_coarsen(Ctx *c, size_t l)
{
    const BoxDims b = box_dims(c->amg[l]);
    AmgLevel &Lc = c->amg[l + 1];
    hipLaunchKernelGGL(k_box_galerkin, dim3(div_up(b.nc, BLOCK)), dim3(BLOCK), 0, c->stream, b, c->amg[l].dia, Lc.dia,
                       Lc.dia32, Lc.dinv, Lc.dinv32);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

int amg_update_values(Ctx *c, const double *vals)
{
    if (!amg_current(c)) return amg_setup(c, vals);
    MC_TRY(dense_join(c));   // the previous inverse still reads the coarsest values
    const double *vf = vals;
    // the pressure assembly wrote level 0's diagonal copies with the values
    const bool l0_done = c->pa_dia_fresh && vals == c->PA_vals;
    c->pa_dia_fresh = false;
    // between refreshes the coarse levels keep the values of an earlier
    // matrix: the V-cycle stays a fixed symmetric operator for the solve
    const bool coarse =
        c->amg.size() == 1 || c->opt.amg_refresh <= 1 || c->amg_updates % c->opt.amg_refresh == 0;
    c->amg_updates++;
    for (size_t l = 0; l < c->amg.size(); l++) {
        AmgLevel &L = c->amg[l];
        if (L.bx && (l > 0 || l0_done)) {   // a coarse box level: written by the Galerkin pass below
            if (l + 1 < c->amg.size()) {
                if (!coarse) return MC_OK;
                MC_TRY(box_coarsen(c, l));
            }
            continue;
        }
        if (L.vals != vf)
            MC_HIP(c, hipMemcpyAsync(L.vals, vf, (size_t)L.nnz * 8, hipMemcpyDeviceToDevice, c->stream));
        if (!(l == 0 && l0_done)) {
            if (L.nd)
                hipLaunchKernelGGL(k_level_dia, dim3(div_up(L.n, 256)), dim3(256), 0, c->stream, L.n, L.row_ptr,
                                   L.col, L.dia_map, L.vals, L.dia, L.dia32, L.dinv, L.dinv32, L.sym ? L.nd / 2 : 0,
                                   L.hoff, L.diag32);
            else
                hipLaunchKernelGGL(k_diag_inv, dim3(div_up(L.n, 256)), dim3(256), 0, c->stream, L.n, L.row_ptr,
                                   L.col, L.vals, L.dinv, L.dinv32, L.vals32, L.nnz);
            MC_LAUNCH_CHECK(c);
        }
        if (l + 1 < c->amg.size()) {
            if (!coarse) return MC_OK;
            if (L.bx) { MC_TRY(box_coarsen(c, l)); continue; }
            AmgLevel &Lc = c->amg[l + 1];
            hipLaunchKernelGGL(k_gather_sum, dim3(div_up(Lc.nnz, 256)), dim3(256), 0, c->stream, Lc.nnz, L.gptr, L.gmap,
                               L.vals, Lc.vals);
            MC_LAUNCH_CHECK(c);
            vf = Lc.vals;
        }
    }
    AmgLevel &Lc = c->amg.back();
    if (Lc.n > DENSE_MAX) { c->err = "coarsest AMG level larger than the dense limit"; return MC_ERR_STATE; }
    // one workgroup for ~0.2 ms: run it beside the work that precedes the
    // first coarsest-level solve (residual, first V-cycle's descent)
    MC_HIP(c, hipEventRecord(c->ev_coarse, c->stream));
    MC_HIP(c, hipStreamWaitEvent(c->side, c->ev_coarse, 0));
    const DenseSrc src{Lc.n, Lc.row_ptr, Lc.col, Lc.bx ? Lc.dia : Lc.vals, Lc.bx, Lc.by};
    hipLaunchKernelGGL(k_dense_inverse, dim3(1), dim3(1024), 0, c->side, src, c->amg_dense);
    MC_LAUNCH_CHECK(c);
    MC_HIP(c, hipEventRecord(c->ev_dense, c->side));
    c->dense_pending = true;
    return MC_OK;
}

template <typename T>
static Mat<T> level_mat(AmgLevel &L)
{
    Mat<T> A;
    A.n = L.n; A.rp = L.row_ptr; A.col = L.col;
    if constexpr (sizeof(T) == 8) { A.csr = (const T *)L.vals; A.dia = L.nd ? (const T *)L.dia : nullptr; }
    else { A.csr = (const T *)L.vals32; A.dia = L.nd ? (const T *)L.dia32 : nullptr; }
    A.sym = (sizeof(T) == 8) ? L.sym : 0;   // FP32 copies keep every diagonal (faster there, measured)
    A.nd = L.nd;
    for (int d = 0; d < DIA_MAX; d++) A.off[d] = d < L.nd ? L.off[d] : 0;
    return A;
}

// ------------------------------------------------------ V-cycle kernels --
// first two pre-smoothing sweeps from x = 0: x1 = w1 D^-1 b, x2 = x1 + w2 D^-1 (b - A x1)
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_jac_first2(Mat<T> A, const T *dinv, const T *b, T *xout, T w1, T w2,
                                                      int chunk, int two, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    if (!two) {
        for (int i = r0 + threadIdx.x; i < r1; i += BLOCK) xout[i] = vc_first(w1, dinv[i], b[i]);
        return;
    }
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return (double)vc_first(w1, dinv[j], b[j]); },
                    [&](int r, const double (&ax)[1]) {
                        xout[r] = vc_first2(w1, w2, dinv[r], b[r], ax[0]);
                    });
}

// Jacobi weights of the nu smoothing sweeps: all amg_omega, or, with
// amg_cheb_ratio > 0, the reciprocals of the Chebyshev nodes of degree nu on
// [2 / ratio, 2] -- a Chebyshev smoother written as nu Jacobi sweeps (the
// spectrum of D^-1 A lies in [0, 2] for the zero-row-sum M-matrices of every
// level).  Pre-smoothing uses them in this order, post-smoothing in reverse,
// so the V-cycle stays symmetric.
static void smoother_weights(const Ctx *c, int nu, double *w)
{
    const double ratio = c->opt.amg_cheb_ratio;
    if (!(ratio > 1.0)) {
        for (int k = 0; k < nu; k++) w[k] = c->opt.amg_omega;
        return;
    }
    const double lo = 2.0 / ratio, hi = 2.0;
    for (int k = 0; k < nu; k++) {
        const double node = 0.5 * (hi + lo) + 0.5 * (hi - lo) * std::cos(M_PI * (2.0 * k + 1.0) / (2.0 * nu));
        w[k] = 1.0 / node;
    }
}

// x_out = x + w D^-1 (b - A x).  With dotv != nullptr the last sweep also
// forms the block partials of (dotv, x_out): the PCG's (r, z), finished into
// rho / beta by EpiRz.
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_jac(Mat<T> A, const T *dinv, const T *b, const T *x, T *xout, T omega,
                                               int chunk, const T *dotv, double *partials, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double acc[1] = {0.0};
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return (double)x[j]; }, [&](int r, const double (&ax)[1]) {
        const T o = vc_jac(x[r], omega, dinv[r], b[r], ax[0]);
        xout[r] = o;
        if (dotv) acc[0] += (double)dotv[r] * (double)o;
    });
    if (dotv) block_partials<1>(acc, partials, bb, gridDim.x);
}

// y = x + cs * xc[agg] in place: the prolongation of the coarse correction,
// one pass before the post-smoothing sweeps (folded into the first sweep it
// was 15 us slower per fine-level V-cycle at m = 128: every row gathered
// its seven neighbours' aggregates and corrections)
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_prolong(int n, const int *agg, const T *xc, T cs, T *x, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) x[i] = vc_prolong(x[i], cs, xc[agg[i]]);
}

// rho = (r, z), beta = rho / rho_old of the PCG
struct EpiRz {
    KState *ks;
    __device__ void operator()(const double (&v)[1]) const
    {
        if (ks->all_done) return;
        ks->rho[0] = v[0];
        ks->beta[0] = (ks->iters[0] == 0) ? 0.0 : v[0] / ks->rho_old[0];
        ks->rho_old[0] = v[0];
    }
};

// bc[I] = sum_{i in aggregate I} (b_i - (A x)_i) on a CSR level: residual
// fused with restriction.  A wave per coarse row, eight lanes per member (at
// most eight members: the host's aggregation checks it), the lanes striding over
// the member's entries; each lane's sum then takes the members in order and the
// eight lanes' sums are added.  With eight lanes per coarse row and the members
// one after the other every member waited for its own chain of row pointers,
// columns and x: 1,124 coarse rows of 8,984 (modifier 33, FP32) 8.0 -> 3.9 us.
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_resid_restrict(Mat<T> A, int nc, const int *aptr, const int *amem,
                                                          const T *b, const T *x, T *bc, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int I = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    if (I >= nc) return;   // whole waves
    const int lane = threadIdx.x & 63, lane8 = lane & 7, m = lane >> 3;
    const int t0 = aptr[I], cnt = aptr[I + 1] - t0;
    double acc = 0.0, bi = 0.0;
    if (m < cnt) {
        const int i = amem[t0 + m];
        bi = (double)b[i];
        for (int e = A.rp[i] + lane8; e < A.rp[i + 1]; e += 8) acc += (double)A.csr[e] * (double)x[A.col[e]];
    }
    double s = 0.0;
    for (int t = 0; t < cnt; t++) {
        const double bt = __shfl(bi, 8 * t, 64), at = __shfl(acc, 8 * t + lane8, 64);
        if (lane8 == 0) s += bt;
        s -= at;
    }
    s = lane8_sum(s);
    if (lane == 0) bc[I] = (T)s;
}

// r = b - A x in row order (diagonal storage: coalesced), then the
// restriction sums each aggregate's members: two passes that replace the
// member-ordered fused kernel, whose row gathers follow the aggregates.
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_resid(Mat<T> A, const T *b, const T *x, T *r, int chunk, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return (double)x[j]; },
                    [&](int i, const double (&ax)[1]) { r[i] = (T)((double)b[i] - ax[0]); });
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) k_restrict(int nc, const int *aptr, const int *amem, const T *r, T *bc,
                                                    const KState *stop)
{
    if (stop && stop->all_done) return;
    const int I = blockIdx.x * BLOCK + threadIdx.x;
    if (I >= nc) return;
    const int t0 = aptr[I], cnt = aptr[I + 1] - t0;
    // at most eight members (the host's aggregation checks it), asked for together
    int mem[8];
    T v[8];
#pragma unroll
    for (int t = 0; t < 8; t++) mem[t] = amem[t0 + min(t, cnt - 1)];
#pragma unroll
    for (int t = 0; t < 8; t++) v[t] = r[mem[t]];
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < 8; t++)
        if (t < cnt) s += (double)v[t];
    bc[I] = (T)s;
}

// k_resid then k_restrict in one launch, for the coarse levels in diagonal
// storage (a launch there costs more than the pass): 8 lanes per coarse row,
// lane m forms member m's residual as k_resid does (rounded to T), and the
// first lane adds the members' residuals in member order as k_restrict does,
// so bc holds the same bits as the two passes give.  Aggregates have at most
// 8 members (the host's aggregation checks it).
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_resid_restrict_seq(Mat<T> A, int nc, const int *aptr, const int *amem,
                                                              const T *b, const T *x, T *bc, const KState *stop)
{
    if (stop && stop->all_done) return;
    constexpr bool SYM = ND < 0;
    constexpr int NA = SYM ? -ND : ND;
    const int I = blockIdx.x * (BLOCK / 8) + (threadIdx.x >> 3);
    const int lane8 = threadIdx.x & 7;
    int t0 = 0, cnt = 0;
    double r = 0.0;
    if (I < nc) {
        t0 = aptr[I];
        cnt = aptr[I + 1] - t0;
        if (lane8 < cnt) {
            const int i = amem[t0 + lane8];
            double a[NA > 0 ? NA : 1];
            int j[NA > 0 ? NA : 1];
#pragma unroll
            for (int d = 0; d < NA; d++) {
                a[d] = dia_at<SYM>(A, d, i);
                j[d] = clampi(i + A.off[d], A.n);
            }
            double acc = 0.0;
#pragma unroll
            for (int d = 0; d < NA; d++) acc = fma(a[d], (double)x[j[d]], acc);
            r = (double)(T)((double)b[i] - acc);
        }
    }
    double s = 0.0;
    const int base = threadIdx.x & ~7;
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const double v = __shfl(r, base + m, 64);
        if (m < cnt) s += v;
    }
    if (lane8 == 0 && I < nc) bc[I] = (T)s;
}

// The first post-smoothing sweep with the prolongation folded in: every x
// value it reads is the prolonged x_j + cs xc[agg_j], formed by k_prolong's
// expression, so the sweep's output equals k_prolong then k_jac bit for bit
// and the prolonged vector is never stored.  For the coarse levels, where a
// launch costs more than the gathered aggregate ids (on the finest level the
// separate pass is faster).
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_jac_prolong(Mat<T> A, const T *dinv, const T *b, const T *x, const int *agg,
                                                       const T *xc, T cs, T *xout, T omega, int chunk,
                                                       const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    auto xp = [&](int j) -> T { return vc_prolong(x[j], cs, xc[agg[j]]); };
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return (double)xp(j); }, [&](int r, const double (&ax)[1]) {
        xout[r] = vc_jac(xp(r), omega, dinv[r], b[r], ax[0]);
    });
}

// coarsest level: x = Ainv b in FP64.  One workgroup of 1024 threads: thread
// t sums row t % 128 over the 16 columns of part t / 128 (consecutive lanes
// read consecutive words of the transposed inverse), then the 8 part sums of
// a row are added in part order.
template <typename T>
__global__ void __launch_bounds__(1024) k_dense_apply(int n, const double *inv, const T *b, T *x, const KState *stop)
{
    if (stop && stop->all_done) return;
    constexpr int PARTS = 1024 / DENSE_MAX, PLEN = DENSE_MAX / PARTS;
    __shared__ double bs[DENSE_MAX];
    __shared__ double part[PARTS][DENSE_MAX];
    const int t = threadIdx.x;
    if (t < n) bs[t] = (double)b[t];
    __syncthreads();
    const int i = t % DENSE_MAX, p = t / DENSE_MAX;
    double s = 0.0;
    if (i < n) {
        const int j0 = p * PLEN;
#pragma unroll
        for (int jj = 0; jj < PLEN; jj++) {
            const int j = j0 + jj;
            if (j < n) s = fma(inv[(size_t)j * n + i], bs[j], s);
        }
    }
    part[p][i] = s;
    __syncthreads();
    if (t < n) {
        double y = 0.0;
#pragma unroll
        for (int q = 0; q < PARTS; q++) y += part[q][t];
        x[t] = (T)y;
    }
}

// partials of (r, z) when no smoothing sweep can carry them
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_rz(int n, const T *r, const T *z, const KState *ks, double *partials,
                                              int chunk)
{
    if (ks->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = bb * chunk, i1 = min(n, i0 + chunk);
    double acc[1] = {0.0};
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) acc[0] += (double)r[i] * (double)z[i];
    block_partials<1>(acc, partials, bb, gridDim.x);
}

template <typename T> static T *lv_x(AmgLevel &L);
template <typename T> static T *lv_b(AmgLevel &L);
template <typename T> static T *lv_t(AmgLevel &L);
template <typename T> static T *lv_dinv(AmgLevel &L);
template <> double *lv_x<double>(AmgLevel &L) { return L.x; }
template <> double *lv_b<double>(AmgLevel &L) { return L.b; }
template <> double *lv_t<double>(AmgLevel &L) { return L.t; }
template <> double *lv_dinv<double>(AmgLevel &L) { return L.dinv; }
template <> float *lv_x<float>(AmgLevel &L) { return L.x32; }
template <> float *lv_b<float>(AmgLevel &L) { return L.b32; }
template <> float *lv_t<float>(AmgLevel &L) { return L.t32; }
template <> float *lv_dinv<float>(AmgLevel &L) { return L.dinv32; }

// ------------------------------- V-cycle tail of a matched hierarchy --
// The small levels of a hierarchy from pairwise matching, and the dense
// coarsest level, in one workgroup of 1024 threads: the six launches of a
// level (7 to 10 us each with their gaps on a CSR level of any size) become
// passes separated by barriers.  A pass is bound by one round trip to L2 for
// the matrix: x and b of every level stay in LDS, CSR row pointers too, and all
// of a thread's entries are asked for together.  Rows in diagonal storage take
// a thread each; CSR rows eight lanes, lane l the entries l, l + 8, ..., as in
// the per-pass kernels.  Every row is formed by those kernels' expressions
// (k_jac_first2, k_jac, k_resid_restrict_seq / k_resid_restrict, k_jac_prolong,
// k_dense_apply) in the same order, so the result is the same.
// Sizes: LDS holds VT_SUM rows in all; a first level beyond VT_ROWS takes
// longer on one CU than its launches do on all of them.  Measured when it also
// took hierarchies of CSR levels only (now k_csr_tail's): modifier 33 mixed, 13
// launches of the two levels below 8,985 rows into one, ten timesteps 92 -> 82 ms.
constexpr int VT_LEVELS = 4, VT_ROWS = 2304, VT_SUM = 4096, TAIL_THREADS = 1024;

template <typename T>
struct VtLevel {
    Mat<T> A;                       // dia: 7 diagonals; else CSR
    const T *dinv;
    const int *agg, *aptr, *amem;   // aggregation to the next level
    int nc;
    int off, rpo;                   // the level's place in the LDS vectors / row pointers
};

template <typename T>
struct VtArgs {
    VtLevel<T> lv[VT_LEVELS];
    int nl;                             // smoothed levels
    const T *b;                         // right-hand side and solution of the first
    T *x;
    const double *inv;                  // dense inverse, transposed
    int nd;                             // dense level size
    int nu;
    T cs;
    double w[8];
};

// f(i, (A src)_i, D^-1_i) for every row i, by one thread each
template <bool SYM, typename T, typename F>
__device__ __forceinline__ void vt_rows(const VtLevel<T> &L, const T *src, const int *rp, F f)
{
    const int n = L.A.n, tid = threadIdx.x;
    if (L.A.dia) {
        constexpr int R = (VT_ROWS + TAIL_THREADS - 1) / TAIL_THREADS;
        double a[R][7];
        T di[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (TAIL_THREADS * r >= n) break;
            const int i = min(tid + TAIL_THREADS * r, n - 1);
#pragma unroll
            for (int d = 0; d < 7; d++) a[r][d] = dia_at<SYM>(L.A, d, i);
            di[r] = L.dinv[i];
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (TAIL_THREADS * r >= n) break;
            const int i = tid + TAIL_THREADS * r;
            if (i >= n) continue;
            double acc = 0.0;
#pragma unroll
            for (int d = 0; d < 7; d++) acc = fma(a[r][d], (double)src[clampi(i + L.A.off[d], n)], acc);
            f(i, acc, di[r]);
        }
    } else {
        constexpr int B = 3, E = 3;   // rows in flight, entries per lane fetched ahead
        const int lane8 = tid & 7, g = tid >> 3;
        for (int r0 = 0; r0 < n; r0 += 128 * B) {
            double v[B][E];
            int c[B][E], beg[B], end[B];
            T di[B];
#pragma unroll
            for (int q = 0; q < B; q++) {
                const int i = min(r0 + 128 * q + g, n - 1);
                beg[q] = rp[i];
                end[q] = rp[i + 1];
                di[q] = L.dinv[i];
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const int k = beg[q] + lane8 + 8 * e;
                    const bool in = k < end[q];
                    const int kk = in ? k : beg[q];
                    c[q][e] = L.A.col[kk];
                    v[q][e] = in ? (double)L.A.csr[kk] : 0.0;
                }
            }
#pragma unroll
            for (int q = 0; q < B; q++) {
                double acc = 0.0;
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (beg[q] + lane8 + 8 * e < end[q]) acc = fma(v[q][e], (double)src[c[q][e]], acc);
                for (int k = beg[q] + lane8 + 8 * E; k < end[q]; k += 8)
                    acc = fma((double)L.A.csr[k], (double)src[L.A.col[k]], acc);
                acc = lane8_sum(acc);
                const int i = r0 + 128 * q + g;
                if (lane8 == 0 && i < n) f(i, acc, di[q]);
            }
        }
    }
}

template <bool SYM, typename T>
__global__ void __launch_bounds__(TAIL_THREADS) k_vtail(VtArgs<T> a, const KState *stop)
{
    if (stop && stop->all_done) return;
    __shared__ T xs[VT_SUM], bl[VT_SUM], alt[VT_ROWS];
    __shared__ int rps[VT_SUM + VT_LEVELS];
    __shared__ double bs[DENSE_MAX];
    __shared__ T xd[DENSE_MAX];
    __shared__ double part[TAIL_THREADS / DENSE_MAX][DENSE_MAX];
    const int tid = threadIdx.x, nu = a.nu;
    for (int l = 0; l < a.nl; l++)
        if (!a.lv[l].A.dia)
            for (int i = tid; i <= a.lv[l].A.n; i += TAIL_THREADS) rps[a.lv[l].rpo + i] = a.lv[l].A.rp[i];
    for (int i = tid; i < a.lv[0].A.n; i += TAIL_THREADS) bl[i] = a.b[i];
    __syncthreads();
    for (int l = 0; l < a.nl; l++) {
        const VtLevel<T> &L = a.lv[l];
        const int n = L.A.n;
        T *x = xs + L.off;
        const T *b = bl + L.off;
        const int *rp = rps + L.rpo;
        const T w1 = (T)a.w[0], w2 = (T)a.w[nu >= 2 ? 1 : 0];
        for (int i = tid; i < n; i += TAIL_THREADS) x[i] = vc_first(w1, L.dinv[i], b[i]);
        __syncthreads();
        T *cur = x, *oth = alt;
        for (int k = 1; k < nu; k++) {
            const T omega = (T)a.w[k];
            if (k == 1)
                vt_rows<SYM>(L, cur, rp, [&](int i, double ax, T di) { oth[i] = vc_first2(w1, w2, di, b[i], ax); });
            else
                vt_rows<SYM>(L, cur, rp, [&](int i, double ax, T di) { oth[i] = vc_jac(cur[i], omega, di, b[i], ax); });
            __syncthreads();
            T *sw = cur; cur = oth; oth = sw;
        }
        if (cur != x) {   // x keeps the value; alt is free
            for (int i = tid; i < n; i += TAIL_THREADS) x[i] = cur[i];
            __syncthreads();
        }
        const bool dense = l + 1 == a.nl;
        T *bc = dense ? nullptr : bl + a.lv[l + 1].off;
        if (L.A.dia) {
            vt_rows<SYM>(L, x, rp, [&](int i, double ax, T) { alt[i] = (T)((double)b[i] - ax); });
            __syncthreads();
            for (int I = tid; I < L.nc; I += TAIL_THREADS) {
                double sum = 0.0;
                for (int t = L.aptr[I]; t < L.aptr[I + 1]; t++) sum += (double)alt[L.amem[t]];
                if (dense) bs[I] = (double)(T)sum; else bc[I] = (T)sum;
            }
        } else {
            const int lane8 = tid & 7;
            for (int I0 = 0; I0 < L.nc; I0 += 128) {
                const int I = I0 + (tid >> 3);
                double s = 0.0;
                if (I < L.nc)
                    for (int t = L.aptr[I]; t < L.aptr[I + 1]; t++) {
                        const int i = L.amem[t];
                        double acc = 0.0;
                        for (int e = rp[i] + lane8; e < rp[i + 1]; e += 8)
                            acc = fma((double)L.A.csr[e], (double)x[L.A.col[e]], acc);
                        if (lane8 == 0) s += (double)b[i];
                        s -= acc;
                    }
                s = lane8_sum(s);
                if (lane8 == 0 && I < L.nc) { if (dense) bs[I] = (double)(T)s; else bc[I] = (T)s; }
            }
        }
        __syncthreads();
    }
    {   // dense coarsest level, as k_dense_apply
        constexpr int PARTS = TAIL_THREADS / DENSE_MAX, PLEN = DENSE_MAX / PARTS;
        const int nd = a.nd;
        const int i = tid % DENSE_MAX, p = tid / DENSE_MAX;
        double sum = 0.0;
        if (i < nd) {
            const int j0 = p * PLEN;
#pragma unroll
            for (int jj = 0; jj < PLEN; jj++) {
                const int j = j0 + jj;
                if (j < nd) sum = fma(a.inv[(size_t)j * nd + i], bs[j], sum);
            }
        }
        part[p][i] = sum;
        __syncthreads();
        if (tid < nd) {
            double y = 0.0;
#pragma unroll
            for (int q = 0; q < PARTS; q++) y += part[q][tid];
            xd[tid] = (T)y;
        }
        __syncthreads();
    }
    for (int l = a.nl - 1; l >= 0; l--) {
        const VtLevel<T> &L = a.lv[l];
        const int n = L.A.n;
        const T *xc = l + 1 == a.nl ? xd : xs + a.lv[l + 1].off;
        T *x = xs + L.off;
        const T *b = bl + L.off;
        for (int i = tid; i < n; i += TAIL_THREADS) x[i] = vc_prolong(x[i], a.cs, xc[L.agg[i]]);
        __syncthreads();
        T *cur = x, *oth = alt;
        for (int k = 0; k < nu; k++) {
            const T omega = (T)a.w[nu - 1 - k];
            vt_rows<SYM>(L, cur, rps + L.rpo,
                         [&](int i, double ax, T di) { oth[i] = vc_jac(cur[i], omega, di, b[i], ax); });
            __syncthreads();
            T *sw = cur; cur = oth; oth = sw;
        }
        T *dst = l == 0 ? a.x : x;
        if (cur != dst) {
            for (int i = tid; i < n; i += TAIL_THREADS) dst[i] = cur[i];
            __syncthreads();
        }
    }
}

// The same cycle where every level left is in CSR storage and small enough for
// a thread to keep its entries in registers: eight lanes a row, nine rows a
// thread, the first sixteen entries of a row (the pairwise levels below a box of
// odd sides have 7 on average and up to 19; the rest is fetched again on each
// pass).  In k_vtail each of a level's seven passes waits three times for its
// entries; here they are loaded once on the way down and once on the way up (the
// last level once), and a pass reads x from LDS only.  It is then bound by LDS and
// vector instructions of one CU, so the rows' own work is spread: lane l of the
// eight finishes the thread's row l (every lane has every sum).  x is held as
// doubles, rounded to T at every store: gathers then need no conversion, which
// runs at a quarter of the rate.  Modifier 33 mixed (1,124 and 143 rows, dense
// 73): k_vtail 47 us, this 31; ten timesteps 67.2 -> 62.1 ms.  A thread per row
// (two rows of sixteen entries) needs the eight partial sums in registers too and
// spills: 80 us.
// CT_ROWS: nine rows a thread.  CT_SUM: what 160 KB of LDS hold beside the nine
// rows' partial sums.  CT_NC: aggregates of eight give 144 of 1,152 rows; beyond a
// third the matching has failed to shrink the level and nothing was measured.
constexpr int CT_ROWS = 1152, CT_NC = 384, CT_SUM = 2048;

template <typename T>
struct CtRows {
    static constexpr int R = CT_ROWS / 128, E = 2;
    static_assert(R == 9, "rows 0 to 7 are finished by the eight lanes, row 8 by lane 0");
    double v[R][E];
    unsigned cp[R];      // a row's two columns
    // bit r: this lane has a first / second entry of row r, the row has more
    unsigned one, two, longer;

    __device__ __forceinline__ void load(const VtLevel<T> &L, const int *rp)
    {
        const int n = L.A.n, lane8 = threadIdx.x & 7, g = threadIdx.x >> 3;
        one = two = longer = 0;
#pragma unroll
        for (int r = 0; r < R; r++) {
            cp[r] = 0;
            v[r][0] = v[r][1] = 0.0;
            if (128 * r >= n) continue;
            const int i = min(g + 128 * r, n - 1);
            const int beg = rp[i], end = rp[i + 1];
            longer |= (end - beg > 8 * E ? 1u : 0u) << r;
            const int k0 = beg + lane8, k1 = k0 + 8;
            const int q0 = k0 < end ? k0 : beg, q1 = k1 < end ? k1 : beg;
            one |= (k0 < end ? 1u : 0u) << r;
            two |= (k1 < end ? 1u : 0u) << r;
            v[r][0] = (double)L.A.csr[q0];
            v[r][1] = (double)L.A.csr[q1];
            cp[r] = (unsigned)L.A.col[q0] | (unsigned)L.A.col[q1] << 16;
        }
    }
    // f(r, i, this lane's part of (A src)_i) for every row of the thread
    template <typename F>
    __device__ __forceinline__ void parts(const VtLevel<T> &L, const int *rp, const double *src, F f) const
    {
        const int n = L.A.n, lane8 = threadIdx.x & 7, g = threadIdx.x >> 3;
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (128 * r >= n) continue;
            const int i = g + 128 * r;
            double acc = fma(v[r][0], src[cp[r] & 0xffffu], 0.0);
            if (!(one >> r & 1)) acc = 0.0;
            if (two >> r & 1) acc = fma(v[r][1], src[cp[r] >> 16], acc);
            if (longer >> r & 1) {
                const int ii = min(i, n - 1);
                for (int k = rp[ii] + 8 * E + lane8; k < rp[ii + 1]; k += 8)
                    acc = fma((double)L.A.csr[k], src[L.A.col[k]], acc);
            }
            f(r, i, acc);
        }
    }
    // f(i, (A src)_i), each row by one lane
    template <typename F>
    __device__ __forceinline__ void rows(const VtLevel<T> &L, const int *rp, const double *src, F f) const
    {
        const int n = L.A.n, lane8 = threadIdx.x & 7, g = threadIdx.x >> 3;
        double mine = 0.0, last = 0.0;
        parts(L, rp, src, [&](int r, int, double acc) {
            acc = lane8_sum(acc);
            if (r == 8) last = acc;
            else if (lane8 == r) mine = acc;
        });
        const int i = g + 128 * lane8;
        if (i < n) f(i, mine);
        if (lane8 == 0 && g + 1024 < n) f(g + 1024, last);
    }
};

template <typename T>
__global__ void __launch_bounds__(TAIL_THREADS) k_csr_tail(VtArgs<T> a, const KState *stop)
{
    if (stop && stop->all_done) return;
    __shared__ double xs[CT_SUM], alt[CT_ROWS], pl[CT_ROWS * 8];
    __shared__ T bl[CT_SUM], dl[CT_SUM];
    // row pointers, aggregates, their members and the members' ranges
    __shared__ int rps[CT_SUM + VT_LEVELS];
    __shared__ unsigned short ag[CT_SUM], am[CT_SUM], ap[CT_SUM + VT_LEVELS];
    __shared__ double bs[DENSE_MAX], xd[DENSE_MAX], part[TAIL_THREADS / DENSE_MAX][DENSE_MAX];
    const int tid = threadIdx.x, lane8 = tid & 7, g = tid >> 3, nu = a.nu;
    for (int l = 0; l < a.nl; l++)
        for (int i = tid; i <= a.lv[l].A.n; i += TAIL_THREADS) {
            const VtLevel<T> &L = a.lv[l];
            rps[L.rpo + i] = L.A.rp[i];
            if (i <= L.nc) ap[L.rpo + i] = (unsigned short)L.aptr[i];
            if (i < L.A.n) {
                dl[L.off + i] = L.dinv[i];
                ag[L.off + i] = (unsigned short)L.agg[i];
                am[L.off + i] = (unsigned short)L.amem[i];
            }
        }
    for (int i = tid; i < a.lv[0].A.n; i += TAIL_THREADS) bl[i] = a.b[i];
    __syncthreads();
    CtRows<T> M;
    for (int l = 0; l < a.nl; l++) {
        const VtLevel<T> &L = a.lv[l];
        const int n = L.A.n;
        double *x = xs + L.off;
        const T *b = bl + L.off;
        const int *rp = rps + L.rpo;
        const T *di = dl + L.off;
        const T w1 = (T)a.w[0], w2 = (T)a.w[nu >= 2 ? 1 : 0];
        // the buffer from which nu - 1 sweeps end in x
        double *cur = (nu - 1) & 1 ? alt : x, *oth = (nu - 1) & 1 ? x : alt;
        for (int i = tid; i < n; i += TAIL_THREADS) cur[i] = (double)vc_first(w1, di[i], b[i]);
        M.load(L, rp);
        __syncthreads();
        for (int k = 1; k < nu; k++) {
            const T omega = (T)a.w[k];
            if (k == 1)
                M.rows(L, rp, cur, [&](int i, double ax) { oth[i] = (double)vc_first2(w1, w2, di[i], b[i], ax); });
            else
                M.rows(L, rp, cur,
                       [&](int i, double ax) { oth[i] = (double)vc_jac((T)cur[i], omega, di[i], b[i], ax); });
            __syncthreads();
            double *sw = cur; cur = oth; oth = sw;
        }
        M.parts(L, rp, x, [&](int, int i, double acc) {
            if (i < n) pl[8 * i + lane8] = acc;
        });
        __syncthreads();
        const bool dense = l + 1 == a.nl;
        T *bc = dense ? nullptr : bl + a.lv[l + 1].off;
        for (int I0 = 0; I0 < L.nc; I0 += 128) {
            const int I = min(I0 + g, L.nc - 1);
            const int t0 = ap[L.rpo + I], cnt = ap[L.rpo + I + 1] - t0;
            double s = 0.0;
            for (int t = 0; t < cnt; t++) {
                const int i = am[L.off + t0 + t];
                if (lane8 == 0) s += (double)b[i];
                s -= pl[8 * i + lane8];
            }
            s = lane8_sum(s);
            if (lane8 == 0 && I0 + g < L.nc) { if (dense) bs[I] = (double)(T)s; else bc[I] = (T)s; }
        }
        __syncthreads();
    }
    {   // dense coarsest level, as k_dense_apply
        constexpr int PARTS = TAIL_THREADS / DENSE_MAX, PLEN = DENSE_MAX / PARTS;
        const int nd = a.nd;
        const int i = tid % DENSE_MAX, p = tid / DENSE_MAX;
        double sum = 0.0;
        if (i < nd) {
            const int j0 = p * PLEN;
#pragma unroll
            for (int jj = 0; jj < PLEN; jj++) {
                const int j = j0 + jj;
                if (j < nd) sum = fma(a.inv[(size_t)j * nd + i], bs[j], sum);
            }
        }
        part[p][i] = sum;
        __syncthreads();
        if (tid < nd) {
            double y = 0.0;
#pragma unroll
            for (int q = 0; q < PARTS; q++) y += part[q][tid];
            xd[tid] = (double)(T)y;
        }
        __syncthreads();
    }
    for (int l = a.nl - 1; l >= 0; l--) {
        const VtLevel<T> &L = a.lv[l];
        const int n = L.A.n;
        const double *xc = l + 1 == a.nl ? xd : xs + a.lv[l + 1].off;
        double *x = xs + L.off;
        const T *b = bl + L.off;
        const int *rp = rps + L.rpo;
        const T *di = dl + L.off;
        double *cur = nu & 1 ? alt : x, *oth = nu & 1 ? x : alt;
        for (int i = tid; i < n; i += TAIL_THREADS) cur[i] = (double)vc_prolong((T)x[i], a.cs, (T)xc[ag[L.off + i]]);
        if (l + 1 != a.nl) M.load(L, rp);   // the last level's entries are still there
        __syncthreads();
        for (int k = 0; k < nu; k++) {
            const T omega = (T)a.w[nu - 1 - k];
            const bool out = l == 0 && k == nu - 1;
            M.rows(L, rp, cur, [&](int i, double ax) {
                const T y = vc_jac((T)cur[i], omega, di[i], b[i], ax);
                if (out) a.x[i] = y;
                else oth[i] = (double)y;
            });
            __syncthreads();
            double *sw = cur; cur = oth; oth = sw;
        }
    }
}

// ----------------------------------------- FP16 fine-level smoothing --
// The FP32 V-cycle's fine-level passes on an FP16 copy of D^-1 A's six
// off-diagonals (entries in [-1, 0] for the pressure M-matrix) with the FP32
// inverse diagonal and diagonal: x' = x + w (D^-1 b - x - (D^-1 A)_off x),
// r = D (D^-1 b - x - (D^-1 A)_off x).  A row reads 12 bytes of matrix
// instead of 28.  The PCG's own product keeps the FP32 matrix, and the FP64
// refinement residual checks every step, so the rounding of the copy (5e-4
// relative) changes only the preconditioner.
struct HMat {
    int n;
    const _Float16 *h;
    const float *dinv, *diag;
    int off[6];
};

template <typename XF>
__device__ __forceinline__ float hmat_offx(const HMat &H, int i, XF X)
{
    float a[6];
    int j[6];
#pragma unroll
    for (int d = 0; d < 6; d++) {
        a[d] = (float)H.h[(size_t)d * H.n + i];
        j[d] = clampi(i + H.off[d], H.n);
    }
    float acc = 0.0f;
#pragma unroll
    for (int d = 0; d < 6; d++) acc += a[d] * X(j[d]);
    return acc;
}

__global__ void __launch_bounds__(BLOCK) k_jac_first2_h(HMat H, const float *b, float *xout, float w1, float w2,
                                                        int chunk, int two, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(H.n, r0 + chunk);
    for (int i = r0 + threadIdx.x; i < r1; i += BLOCK) {
        const float db = H.dinv[i] * b[i];
        const float x1 = w1 * db;
        if (!two) { xout[i] = x1; continue; }
        const float ax = hmat_offx(H, i, [&](int j) { return w1 * (H.dinv[j] * b[j]); });
        xout[i] = x1 + w2 * (db - x1 - ax);
    }
}

__global__ void __launch_bounds__(BLOCK) k_jac_h(HMat H, const float *b, const float *x, float *xout, float omega,
                                                 int chunk, const float *dotv, double *partials, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(H.n, r0 + chunk);
    double acc[1] = {0.0};
    for (int i = r0 + threadIdx.x; i < r1; i += BLOCK) {
        const float y = x[i];
        const float o = y + omega * (H.dinv[i] * b[i] - y - hmat_offx(H, i, [&](int j) { return x[j]; }));
        xout[i] = o;
        if (dotv) acc[0] += (double)dotv[i] * (double)o;
    }
    if (dotv) block_partials<1>(acc, partials, bb, gridDim.x);
}

__global__ void __launch_bounds__(BLOCK) k_resid_h(HMat H, const float *b, const float *x, float *r, int chunk,
                                                   const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(H.n, r0 + chunk);
    for (int i = r0 + threadIdx.x; i < r1; i += BLOCK)
        r[i] = H.diag[i] * (H.dinv[i] * b[i] - x[i] - hmat_offx(H, i, [&](int j) { return x[j]; }));
}

// ------------------------------------------------- box level passes --
// n / d for 0 <= n < 2^31 by multiply and shift (d >= 1): Granlund and
// Montgomery, Division by Invariant Integers using Multiplication, 1994
struct FastDiv {
    unsigned d, mul, sh;
};
static FastDiv fast_div(int d)
{
    FastDiv f;
    f.d = (unsigned)d;
    f.sh = 0;
    while ((1ull << f.sh) < (uint64_t)d) f.sh++;
    f.mul = (unsigned)(((1ull << 32) * ((1ull << f.sh) - d)) / d + 1);
    return f;
}
__device__ __forceinline__ int fdiv(int n, const FastDiv &f)
{
    return (int)(unsigned)(((uint64_t)__umulhi((unsigned)n, f.mul) + (unsigned)n) >> f.sh);
}

struct BoxWalk {
    BoxDims b;
    FastDiv dx, dxy;     // this level's row and plane length
    FastDiv cdx, cdxy;   // the next level's
};
static BoxWalk box_walk(const AmgLevel &L)
{
    BoxWalk w;
    w.b = box_dims(L);
    w.dx = fast_div(w.b.nx); w.dxy = fast_div(w.b.nx * w.b.ny);
    w.cdx = fast_div(w.b.cx); w.cdxy = fast_div(w.b.cx * w.b.cy);
    return w;
}

// Row i's residual b - A x, from a level's diagonals or the FP16 copy; the
// expressions of k_resid and k_resid_h.
template <int ND, typename T>
struct ResidDia {
    Mat<T> A;
    const T *b, *x;
    __device__ __forceinline__ double operator()(int i) const
    {
        constexpr bool SYM = ND < 0;
        constexpr int NA = SYM ? -ND : ND;
        double a[NA > 0 ? NA : 1], v[NA > 0 ? NA : 1];
#pragma unroll
        for (int d = 0; d < NA; d++) {
            a[d] = dia_at<SYM>(A, d, i);
            v[d] = (double)x[clampi(i + A.off[d], A.n)];
        }
        double acc = 0.0;
#pragma unroll
        for (int d = 0; d < NA; d++) acc = fma(a[d], v[d], acc);
        return (double)(T)((double)b[i] - acc);
    }
};
struct ResidH {
    HMat H;
    const float *b, *x;
    __device__ __forceinline__ double operator()(int i) const
    {
        return (double)(H.diag[i] * (H.dinv[i] * b[i] - x[i] - hmat_offx(H, i, [&](int j) { return x[j]; })));
    }
};

// bc[I] = sum of the residuals of coarse cell I's members.  Eight lanes per
// coarse cell, lane (i + 2 j + 4 k) its member at that corner: 64 lanes cover
// runs of 16 adjacent rows, the residual is never stored, and one launch takes
// the place of the residual and restriction passes (250,000 rows with the
// FP16 copy: 3.3 + 5.9 -> 4.9 us).
template <class R, typename T>
__global__ void __launch_bounds__(BLOCK) k_box_restrict(BoxWalk w, R resid, T *bc, const KState *stop)
{
    if (stop && stop->all_done) return;
    const BoxDims &b = w.b;
    const int I = xcd_block(blockIdx.x, gridDim.x) * (BLOCK / 8) + (threadIdx.x >> 3);
    const int lane8 = threadIdx.x & 7, i = lane8 & 1, j = (lane8 >> 1) & 1, k = lane8 >> 2;
    double s = 0.0;
    if (I < b.nc && i <= b.sx && j <= b.sy && k <= b.sz) {
        const int Z = fdiv(I, w.cdxy), q = I - Z * (b.cx * b.cy), Y = fdiv(q, w.cdx), X = q - Y * b.cx;
        const int x = (X << b.sx) + i, y = (Y << b.sy) + j, z = (Z << b.sz) + k;
        if (x < b.nx && y < b.ny && z < b.nz) s = resid(x + b.nx * (y + b.ny * z));
    }
    s = lane8_sum(s);
    if (lane8 == 0 && I < b.nc) bc[I] = (T)s;
}

// The same on a regular matched level, the members added in ascending order as
// k_restrict does.  A lane per x and coarse y, z: it forms the residuals of its four
// rows (64 adjacent ones per load), the even lane of a pair adds both lanes' in
// order.  4,194,304 rows, us: FP64 k_resid 31 + k_restrict 15 -> 32, the FP16 copy 33
// -> 19 (eight lanes a coarse cell, as above: 44 and 58; a thread a coarse cell: 68
// and 38).
template <class R, typename T>
__global__ void __launch_bounds__(BLOCK) k_reg_restrict(BoxWalk w, R resid, T *bc, const KState *stop)
{
    if (stop && stop->all_done) return;
    const BoxDims &b = w.b;
    const int t = xcd_block(blockIdx.x, gridDim.x) * BLOCK + threadIdx.x, I = t >> 1;
    if (I >= b.nc) return;   // both lanes of the pair
    const int Z = fdiv(I, w.cdxy), q = I - Z * (b.cx * b.cy), Y = fdiv(q, w.cdx), X = q - Y * b.cx;
    const int x = 2 * X + (t & 1), y = 2 * Y, z = 2 * Z;
    double r[4], o[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const bool in = x < b.nx && y + (m & 1) < b.ny && z + (m >> 1) < b.nz;
        const int i = min(x, b.nx - 1) + b.nx * (min(y + (m & 1), b.ny - 1) + b.ny * min(z + (m >> 1), b.nz - 1));
        const double v = resid(i);
        r[m] = in ? v : 0.0;   // adds +0 to a sum that starts at +0
    }
#pragma unroll
    for (int m = 0; m < 4; m++)
        o[m] = __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(r[m]), 0xB1, 0xf, 0xf, false),
                                __builtin_amdgcn_update_dpp(0, __double2loint(r[m]), 0xB1, 0xf, 0xf, false));
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < 4; m++) { s += r[m]; s += o[m]; }
    if (!(t & 1)) bc[I] = (T)s;
}

// The prolongation and the first post-smoothing sweep in one pass: every
// value the sweep reads is the prolonged x_j + cs xc[aggregate of j], the
// aggregate from j's coordinates (no index array), so the prolonged vector is
// neither written nor read again (250,000 rows with the FP16 copy: 2.9 + 3.5
// -> 4.1 us).
template <typename T>
struct BoxProlong {
    BoxWalk w;
    const T *x, *xc;
    T cs;
    // prolonged values at row i and at its neighbours -z -y -x +x +y +z (the
    // row itself where there is none: the matrix entry is zero)
    __device__ __forceinline__ T at(int i, T (&nb)[6]) const
    {
        const BoxDims &b = w.b;
        const int nxny = b.nx * b.ny;
        const int Z = fdiv(i, w.dxy), q = i - Z * nxny, Y = fdiv(q, w.dx), X = q - Y * b.nx;
        const int cxy = b.cx * b.cy;
        const int ax = X >> b.sx, ay = (Y >> b.sy) * b.cx, az = (Z >> b.sz) * cxy;
        int j[6], g[6];
        j[0] = Z > 0 ? i - nxny : i;        g[0] = ax + ay + (Z > 0 ? ((Z - 1) >> b.sz) * cxy : az);
        j[1] = Y > 0 ? i - b.nx : i;        g[1] = ax + (Y > 0 ? ((Y - 1) >> b.sy) * b.cx : ay) + az;
        j[2] = X > 0 ? i - 1 : i;           g[2] = (X > 0 ? (X - 1) >> b.sx : ax) + ay + az;
        j[3] = X + 1 < b.nx ? i + 1 : i;    g[3] = (X + 1 < b.nx ? (X + 1) >> b.sx : ax) + ay + az;
        j[4] = Y + 1 < b.ny ? i + b.nx : i; g[4] = ax + (Y + 1 < b.ny ? ((Y + 1) >> b.sy) * b.cx : ay) + az;
        j[5] = Z + 1 < b.nz ? i + nxny : i; g[5] = ax + ay + (Z + 1 < b.nz ? ((Z + 1) >> b.sz) * cxy : az);
#pragma unroll
        for (int d = 0; d < 6; d++) nb[d] = vc_prolong(x[j[d]], cs, xc[g[d]]);
        return vc_prolong(x[i], cs, xc[ax + ay + az]);
    }
};

template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_box_jac_prolong(BoxProlong<T> p, Mat<T> A, const T *dinv, const T *b,
                                                           T *xout, T omega, int chunk, const T *dotv,
                                                           double *partials, const KState *stop)
{
    if (stop && stop->all_done) return;
    constexpr bool SYM = ND < 0;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double acc[1] = {0.0};
    for (int i = r0 + (int)threadIdx.x; i < r1; i += BLOCK) {
        double a[7];
#pragma unroll
        for (int d = 0; d < 7; d++) a[d] = dia_at<SYM>(A, d, i);
        T nb[6];
        const T y = p.at(i, nb);
        double ax = 0.0;
#pragma unroll
        for (int d = 0; d < 7; d++) ax = fma(a[d], (double)(d < 3 ? nb[d] : d == 3 ? y : nb[d - 1]), ax);
        const T o = vc_jac(y, omega, dinv[i], b[i], ax);
        xout[i] = o;
        if (dotv) acc[0] += (double)dotv[i] * (double)o;
    }
    if (dotv) block_partials<1>(acc, partials, bb, gridDim.x);
}

__global__ void __launch_bounds__(BLOCK) k_box_jac_prolong_h(BoxProlong<float> p, HMat H, const float *b, float *xout,
                                                             float omega, int chunk, const float *dotv,
                                                             double *partials, const KState *stop)
{
    if (stop && stop->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(H.n, r0 + chunk);
    double acc[1] = {0.0};
    for (int i = r0 + (int)threadIdx.x; i < r1; i += BLOCK) {
        float a[6], nb[6];
#pragma unroll
        for (int d = 0; d < 6; d++) a[d] = (float)H.h[(size_t)d * H.n + i];
        const float y = p.at(i, nb);
        float off = 0.0f;
#pragma unroll
        for (int d = 0; d < 6; d++) off += a[d] * nb[d];
        const float o = y + omega * (H.dinv[i] * b[i] - y - off);
        xout[i] = o;
        if (dotv) acc[0] += (double)dotv[i] * (double)o;
    }
    if (dotv) block_partials<1>(acc, partials, bb, gridDim.x);
}

// ----------------------------------------------------- V-cycle tail --
// The small levels in seven-diagonal storage (box levels, or matched ones whose
// aggregates came out regular) and the dense coarsest one in one workgroup of
// 1024 threads.  Bound by the chain of passes, each a handful of values per row:
// a row's matrix entries, inverse diagonal, right-hand side and value stay in
// its thread's registers for the whole cycle (loaded at the start, all in
// flight together) and only x goes through LDS for the neighbours, so a sweep
// is seven LDS reads and two barriers instead of a launch (or, as in the
// earlier tail, a round of loads from L2).  LDS holds x as doubles also in the
// FP32 cycle: a value is converted once when stored, not by each of its seven
// readers (FP64 sums; the conversions run at a quarter of the rate).  Every row is formed by the
// expressions of the per-pass kernels in the same order, so the result is the
// same (amg_tail = 0 launches them).
// Rows: up to R0 x 1024 on the first level, 1024 and 512 below.  FP64
// takes R0 = 4 (more entries than registers beyond), FP32 5: 8,192 rows in
// eight a thread measured 52 us, its six launches with the tail of the next
// level 40.  FP64, 1,024 rows and a dense 128: 22 -> 11.8 us; 2,000 and 250
// rows: 38 -> 18 us.  FP32, 4,225 and 637 rows and a dense 112: 27 us, where
// the matched hierarchy's CSR levels of these sizes took 13 launches of 7 to
// 15 us.
constexpr int TAIL_LEVELS = 3;
template <typename T> constexpr int tail_rows() { return (sizeof(T) == 4 ? 5 : 4) * TAIL_THREADS; }
constexpr int tail_cap(int l) { return l <= 1 ? 1024 : 512; }   // rows of level l >= 1

template <typename T>
struct TailLevel {
    BoxDims b;                      // nx = 0: a matched level, its aggregation in the arrays
    Mat<T> A;
    const T *dinv;
    const int *agg, *aptr, *amem;
    int nc;
};

template <typename T>
struct TailArgs {
    TailLevel<T> lv[TAIL_LEVELS];
    int nl;                             // smoothed levels
    const T *b;                         // right-hand side and solution of the first
    T *x;
    const double *inv;                  // dense inverse, transposed
    int nd;                             // dense level size
    int nu;
    T cs;
    double w[8];
};

// The thread id as a value the compiler cannot trace: the row addresses of a
// pass are formed in it rather than kept in registers over the whole cycle
// (56 of them on a level of eight rows a thread, which then spilled).
__device__ __forceinline__ int tail_tid()
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// One level's rows of one thread: row r is tid + 1024 r.
template <int R, bool SYM, typename T>
struct TailRows {
    T a[R][7], di[R], b[R], x[R];
    __device__ __forceinline__ void load(const TailLevel<T> &L)
    {
        const int tid = tail_tid();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = tid + TAIL_THREADS * r;
            const bool in = i < L.A.n;
#pragma unroll
            for (int d = 0; d < 7; d++) a[r][d] = in ? (T)dia_at<SYM>(L.A, d, i) : (T)0;
            di[r] = in ? L.dinv[i] : (T)0;
        }
    }
    __device__ __forceinline__ double ax(const TailLevel<T> &L, const double *s, int r, int i) const
    {
        double acc = 0.0;
#pragma unroll
        for (int d = 0; d < 7; d++) {
            T av = a[r][d];
            if constexpr (sizeof(T) == 4) asm volatile("" : "+v"(av));   // converted here, not kept as a double
            acc = fma((double)av, s[clampi(i + L.A.off[d], L.A.n)], acc);
        }
        return acc;
    }
    __device__ __forceinline__ void put(const TailLevel<T> &L, double *s, const T (&v)[R]) const
    {
        const int tid = tail_tid();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = tid + TAIL_THREADS * r;
            if (i < L.A.n) s[i] = (double)v[r];
        }
    }
    // x <- x + omega D^-1 (b - A x), x also in s (which the caller's barrier
    // has made visible); leaves the new x in s
    __device__ __forceinline__ void sweep(const TailLevel<T> &L, double *s, T omega)
    {
        const int tid = tail_tid();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = tid + TAIL_THREADS * r;
            if (i < L.A.n) x[r] = vc_jac(x[r], omega, di[r], b[r], ax(L, s, r, i));
        }
        __syncthreads();
        put(L, s, x);
        __syncthreads();
    }
    // pre-smoothing from x = 0, then the residual into s
    __device__ __forceinline__ void down(const TailLevel<T> &L, double *s, const double *w, int nu)
    {
        const T w1 = (T)w[0], w2 = (T)w[nu >= 2 ? 1 : 0];
#pragma unroll
        for (int r = 0; r < R; r++) x[r] = vc_first(w1, di[r], b[r]);
        put(L, s, x);
        __syncthreads();
        if (nu >= 2) {
            const int tid = tail_tid();
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int i = tid + TAIL_THREADS * r;
                if (i < L.A.n) x[r] = vc_first2(w1, w2, di[r], b[r], ax(L, s, r, i));
            }
            __syncthreads();
            put(L, s, x);
            __syncthreads();
        }
        for (int k = 2; k < nu; k++) sweep(L, s, (T)w[k]);
        T res[R];
        const int tid = tail_tid();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = tid + TAIL_THREADS * r;
            res[r] = (i < L.A.n) ? (T)((double)b[r] - ax(L, s, r, i)) : (T)0;
        }
        __syncthreads();
        put(L, s, res);
        __syncthreads();
    }
    // prolongation from the next level's solution xc, post-smoothing
    __device__ __forceinline__ void up(const TailLevel<T> &L, double *s, const double *xc, T cs, const double *w, int nu)
    {
        const BoxDims &b_ = L.b;
        const int tid = tail_tid();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int i = tid + TAIL_THREADS * r;
            if (i < L.A.n) {
                int I;
                if (b_.nx) {
                    const int X = i % b_.nx, q = i / b_.nx, Y = q % b_.ny, Z = q / b_.ny;
                    I = (X >> b_.sx) + b_.cx * ((Y >> b_.sy) + b_.cy * (Z >> b_.sz));
                } else {
                    I = L.agg[i];
                }
                x[r] = vc_prolong(x[r], cs, (T)xc[I]);
            }
        }
        put(L, s, x);
        __syncthreads();
        for (int k = 0; k < nu; k++) sweep(L, s, (T)w[nu - 1 - k]);
    }
};

// The members of coarse row tid, found before the level's sweeps, and the sum
// of their residuals: a box level's in k_box_restrict's tree order, a matched
// level's in member order (k_resid_restrict_seq).
struct TailMembers {
    unsigned m[4];   // two 16-bit rows each, 0xffff: none
    template <typename T>
    __device__ __forceinline__ void load(const TailLevel<T> &L)
    {
        const int I = tail_tid();
        const BoxDims &b = L.b;
#pragma unroll
        for (int q = 0; q < 4; q++) m[q] = 0xffffffffu;
        if (I >= L.nc) return;
        if (b.nx) {
            const int X = I % b.cx, q = I / b.cx, Y = q % b.cy, Z = q / b.cy;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int i = e & 1, j = (e >> 1) & 1, k = e >> 2;
                const int x = (X << b.sx) + i, y = (Y << b.sy) + j, z = (Z << b.sz) + k;
                if (i <= b.sx && j <= b.sy && k <= b.sz && x < b.nx && y < b.ny && z < b.nz) put(e, x + b.nx * (y + b.ny * z));
            }
        } else {
            const int t0 = L.aptr[I], cnt = L.aptr[I + 1] - t0;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < cnt) put(e, L.amem[t0 + e]);
        }
    }
    __device__ __forceinline__ void put(int e, int i)
    {
        if (e & 1) m[e >> 1] = (m[e >> 1] & 0xffffu) | ((unsigned)i << 16);
        else m[e >> 1] = (m[e >> 1] & 0xffff0000u) | (unsigned)i;
    }
    __device__ __forceinline__ double sum(const double *s, bool tree) const
    {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const unsigned i = (e & 1) ? m[e >> 1] >> 16 : m[e >> 1] & 0xffffu;
            v[e] = i != 0xffffu ? s[i] : 0.0;
        }
        if (tree) return (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
        double t = 0.0;
#pragma unroll
        for (int e = 0; e < 8; e++) t += v[e];
        return t;
    }
};

template <int R0, bool SYM, typename T>
__global__ void __launch_bounds__(TAIL_THREADS) k_dia_tail(TailArgs<T> a, const KState *stop)
{
    if (stop && stop->all_done) return;
    __shared__ double s0[R0 * TAIL_THREADS], s1[tail_cap(1)], s2[tail_cap(2)];
    __shared__ double bs[DENSE_MAX];
    __shared__ double xd[DENSE_MAX];
    __shared__ double part[TAIL_THREADS / DENSE_MAX][DENSE_MAX];
    const int tid = threadIdx.x, nu = a.nu, nl = a.nl;
    TailRows<R0, SYM, T> r0;
    TailRows<1, SYM, T> r1, r2;
    r0.load(a.lv[0]);
#pragma unroll
    for (int r = 0; r < R0; r++) {
        const int i = tid + TAIL_THREADS * r;
        r0.b[r] = i < a.lv[0].A.n ? a.b[i] : (T)0;
    }
    TailMembers mem;   // of the level being left
    mem.load(a.lv[0]);
    if (nl > 1) r1.load(a.lv[1]);
    const double *rs = s0;   // the last smoothed level's residuals
    r0.down(a.lv[0], s0, a.w, nu);
    if (nl > 1) {
        r1.b[0] = (T)mem.sum(s0, a.lv[0].b.nx != 0);   // (zero beyond the level's rows)
        mem.load(a.lv[1]);
        r1.down(a.lv[1], s1, a.w, nu);
        rs = s1;
    }
    if (nl > 2) {
        r2.load(a.lv[2]);
        r2.b[0] = (T)mem.sum(s1, a.lv[1].b.nx != 0);
        mem.load(a.lv[2]);
        r2.down(a.lv[2], s2, a.w, nu);
        rs = s2;
    }
    {   // dense coarsest level, as k_dense_apply
        constexpr int PARTS = TAIL_THREADS / DENSE_MAX, PLEN = DENSE_MAX / PARTS;
        const int nd = a.nd;
        const int i = tid % DENSE_MAX, p = tid / DENSE_MAX;
        if (tid < nd) bs[tid] = (double)(T)mem.sum(rs, a.lv[nl - 1].b.nx != 0);
        __syncthreads();
        double sum = 0.0;
        if (i < nd) {
#pragma unroll
            for (int jj = 0; jj < PLEN; jj++) {
                const int j = p * PLEN + jj;
                if (j < nd) sum = fma(a.inv[(size_t)j * nd + i], bs[j], sum);
            }
        }
        part[p][i] = sum;
        __syncthreads();
        if (tid < nd) {
            double y = 0.0;
#pragma unroll
            for (int q = 0; q < PARTS; q++) y += part[q][tid];
            xd[tid] = (double)(T)y;
        }
        __syncthreads();
    }
    if (nl > 2) r2.up(a.lv[2], s2, xd, a.cs, a.w, nu);
    if (nl > 1) r1.up(a.lv[1], s1, nl > 2 ? s2 : xd, a.cs, a.w, nu);
    r0.up(a.lv[0], s0, nl > 1 ? s1 : xd, a.cs, a.w, nu);
#pragma unroll
    for (int r = 0; r < R0; r++) {
        const int i = tid + TAIL_THREADS * r;
        if (i < a.lv[0].A.n) a.x[i] = r0.x[r];
    }
}

// The cycle from level l down in one workgroup, when every level left fits.
template <typename T>
static int tail_launch(Ctx *c, size_t l, const T *b, T *x, int nu, const double *wts, const KState *stop, bool *done)
{
    *done = false;
    const size_t nl = c->amg.size() - 1 - l;
    if (!c->opt.amg_tail || l == 0 || nl == 0 || nl > (size_t)TAIL_LEVELS || nu > 8) return MC_OK;
    for (size_t k = 0; k < nl; k++) {
        AmgLevel &L = c->amg[l + k];
        if (nd_code(level_mat<T>(L)) != (sizeof(T) == 8 ? -7 : 7)) return MC_OK;
        if (L.n > (k ? tail_cap((int)k) : tail_rows<T>()) || L.nc > TAIL_THREADS) return MC_OK;
    }
    TailArgs<T> ta;
    memset(&ta, 0, sizeof(ta));
    ta.nl = (int)nl;
    for (size_t k = 0; k < nl; k++) {
        AmgLevel &L = c->amg[l + k];
        if (L.bx) ta.lv[k].b = box_dims(L);
        ta.lv[k].agg = L.agg; ta.lv[k].aptr = L.agg_ptr; ta.lv[k].amem = L.agg_members; ta.lv[k].nc = L.nc;
        ta.lv[k].A = level_mat<T>(L);
        ta.lv[k].dinv = lv_dinv<T>(L);
    }
    ta.b = b; ta.x = x;
    ta.inv = c->amg_dense; ta.nd = c->amg.back().n;
    ta.nu = nu; ta.cs = (T)c->opt.amg_cscale;
    for (int k = 0; k < 8; k++) ta.w[k] = wts[k];
    MC_TRY(dense_join(c));
    constexpr bool SYM = sizeof(T) == 8;   // the FP64 levels keep the upper diagonals
    const dim3 one(1), thr(TAIL_THREADS);
    const int n0 = c->amg[l].n;
    if (n0 <= TAIL_THREADS) hipLaunchKernelGGL((k_dia_tail<1, SYM, T>), one, thr, 0, c->stream, ta, stop);
    else if (n0 <= 2 * TAIL_THREADS) hipLaunchKernelGGL((k_dia_tail<2, SYM, T>), one, thr, 0, c->stream, ta, stop);
    else if (n0 <= 4 * TAIL_THREADS) hipLaunchKernelGGL((k_dia_tail<4, SYM, T>), one, thr, 0, c->stream, ta, stop);
    else if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((k_dia_tail<5, SYM, T>), one, thr, 0, c->stream, ta, stop);
    MC_LAUNCH_CHECK(c);
    c->tail_form[sizeof(T) == 4] = MC_TAIL_DIA;
    *done = true;
    return MC_OK;
}

// V-cycle on level l: x_l = M^-1 b_l.  On level 0 with ks != nullptr the
// last sweep also reduces (b, x) into the PCG's rho / beta.
template <typename T>
static int vcycle(Ctx *c, size_t l, const T *b, T *x, KState *ks, const KState *stop)
{
    AmgLevel &L = c->amg[l];
    double wts[8] = {};
    smoother_weights(c, std::max(1, std::min(c->opt.amg_nu, 8)), wts);
    const int nu = std::max(1, c->opt.amg_nu);
    {
        bool done = false;
        MC_TRY(tail_launch<T>(c, l, b, x, nu, wts, stop, &done));
        if (done) return MC_OK;
    }
    if (l >= 1 && l + 1 < c->amg.size() && c->opt.amg_tail && !L.bx) {
        // the rest of the cycle in one workgroup when every level left is
        // small and in seven-diagonal or CSR storage
        const size_t nl = c->amg.size() - 1 - l;
        bool ok = nl <= (size_t)VT_LEVELS && nu <= 8 && L.n <= VT_ROWS;
        bool csr = true;
        int sum = 0;
        for (size_t k = l; ok && k + 1 < c->amg.size(); k++) {
            const int code = nd_code(level_mat<T>(c->amg[k]));
            sum += c->amg[k].n;
            csr = csr && code == 0;
            ok = (code == 0 || code == (sizeof(T) == 8 ? -7 : 7)) && sum <= VT_SUM;
        }
        // CSR levels only: in registers, from the first level that fits
        // (the larger ones' launches are faster than k_vtail's passes: modifier 41, 2,154
        // rows, a timestep 7.8 -> 7.0 ms)
        if (csr) ok = ok && L.n <= CT_ROWS && L.nc <= CT_NC && sum <= CT_SUM;
        if (ok) {
            VtArgs<T> ta;
            memset(&ta, 0, sizeof(ta));
            ta.nl = (int)nl;
            int off = 0;
            for (size_t k = 0; k < nl; k++) {
                AmgLevel &Lk = c->amg[l + k];
                VtLevel<T> &t = ta.lv[k];
                t.A = level_mat<T>(Lk);
                t.dinv = lv_dinv<T>(Lk);
                t.agg = Lk.agg; t.aptr = Lk.agg_ptr; t.amem = Lk.agg_members; t.nc = Lk.nc;
                t.off = off;
                t.rpo = off + (int)k;   // n + 1 pointers a level
                off += Lk.n;
            }
            ta.b = b; ta.x = x;
            ta.inv = c->amg_dense; ta.nd = c->amg.back().n;
            ta.nu = nu; ta.cs = (T)c->opt.amg_cscale;
            for (int k = 0; k < 8; k++) ta.w[k] = wts[k];
            MC_TRY(dense_join(c));
            constexpr bool SYM = sizeof(T) == 8;   // FP64 seven-diagonal levels keep the upper diagonals
            if (csr) hipLaunchKernelGGL(k_csr_tail<T>, dim3(1), dim3(TAIL_THREADS), 0, c->stream, ta, stop);
            else hipLaunchKernelGGL((k_vtail<SYM, T>), dim3(1), dim3(TAIL_THREADS), 0, c->stream, ta, stop);
            MC_LAUNCH_CHECK(c);
            c->tail_form[sizeof(T) == 4] = csr ? MC_TAIL_CSR : MC_TAIL_MIXED;
            return MC_OK;
        }
    }
    if (l + 1 == c->amg.size()) {
        c->tail_form[sizeof(T) == 4] = MC_TAIL_NONE;
        MC_TRY(dense_join(c));
        hipLaunchKernelGGL(k_dense_apply<T>, dim3(1), dim3(1024), 0, c->stream, L.n, c->amg_dense, b, x, stop);
        if (ks) {  // one-level hierarchy: no smoothing sweep carries the (r, z) reduction
            const Grid g = grid_for(L.n);
            hipLaunchKernelGGL(k_rz<T>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, L.n, b, x, ks, c->red, g.chunk);
            if (!fold_on(c, g)) launch_finish<1>(c->stream, c->red, g.blocks, EpiRz{ks});
        }
        return MC_OK;
    }
    const Mat<T> A = level_mat<T>(L);
    const Grid g = l >= 1 && nd_code(A) == 0 ? grid_csr(L.n) : grid_for(L.n);
    T *dinv = lv_dinv<T>(L), *tmp = lv_t<T>(L);
    T *cur = x, *oth = tmp;
    // FP32 cycle on a level with the FP16 copy: its passes read that copy
    const bool half = sizeof(T) == 4 && L.hoff != nullptr && c->opt.amg_half;
    HMat H{};
    if (half) {
        H.n = L.n; H.h = L.hoff; H.dinv = L.dinv32; H.diag = L.diag32;
        for (int d = 0, q = 0; d < L.nd; d++) if (L.off[d] != 0) H.off[q++] = L.off[d];
    }
    if constexpr (sizeof(T) == 4) {
        if (half)
            hipLaunchKernelGGL(k_jac_first2_h, dim3(g.blocks), dim3(BLOCK), 0, c->stream, H, b, cur, (float)wts[0],
                               (float)wts[nu >= 2 ? 1 : 0], g.chunk, nu >= 2 ? 1 : 0, stop);
    }
    if (!half)
        MC_DISPATCH_ND(nd_code(A), (k_jac_first2<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, dinv, b, cur,
                       (T)wts[0], (T)wts[nu >= 2 ? 1 : 0], g.chunk, nu >= 2 ? 1 : 0, stop);
    for (int s = 2; s < nu; s++) {
        if constexpr (sizeof(T) == 4) {
            if (half)
                hipLaunchKernelGGL(k_jac_h, dim3(g.blocks), dim3(BLOCK), 0, c->stream, H, b, (const float *)cur, oth,
                                   (float)wts[s], g.chunk, (const float *)nullptr, (double *)nullptr, stop);
        }
        if (!half)
            MC_DISPATCH_ND(nd_code(A), (k_jac<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, dinv, b, cur,
                           oth, (T)wts[s], g.chunk, (const T *)nullptr, (double *)nullptr, stop);
        std::swap(cur, oth);
    }
    AmgLevel &Lc = c->amg[l + 1];
    T *bc = lv_b<T>(Lc), *xc = lv_x<T>(Lc);
    // below the finest level the residual and the restriction, and the
    // prolongation and the first post-smoothing sweep, share a launch
    constexpr int BND = sizeof(T) == 8 ? -7 : 7;   // the box levels' storage (level_mat)
    const bool reg = L.rx != 0 && nd_code(A) == BND && !(c->plain & MC_PLAIN_TRANSFERS);
    const bool box = L.bx != 0 || reg;
    const bool fuse = l >= 1 && !half;
    // below the finest level k_reg_restrict's four rows a lane pay from REG_ROWS on
    // (FP64, us against k_resid_restrict_seq: 65,536 rows 6.6 / 9, 8,192 rows 5.1 / 4)
    constexpr int REG_ROWS = 32768;
    if (box && !(reg && fuse && L.n < REG_ROWS)) {
        const BoxWalk w = box_walk(L);
        const dim3 gr(div_up(L.nc, BLOCK / 8));
        bool launched = false;
        if constexpr (sizeof(T) == 4) {
            if (half) {
                const ResidH rh{H, b, cur};
                if (reg) hipLaunchKernelGGL((k_reg_restrict<ResidH, float>), dim3(div_up(2 * L.nc, BLOCK)), dim3(BLOCK), 0,
                                            c->stream, w, rh, bc, stop);
                else hipLaunchKernelGGL((k_box_restrict<ResidH, float>), gr, dim3(BLOCK), 0, c->stream, w, rh, bc, stop);
                launched = true;
            }
        }
        if (!launched) {
            using RD = ResidDia<BND, T>;
            const RD rd{A, b, cur};
            if (reg) hipLaunchKernelGGL((k_reg_restrict<RD, T>), dim3(div_up(2 * L.nc, BLOCK)), dim3(BLOCK), 0, c->stream,
                                        w, rd, bc, stop);
            else hipLaunchKernelGGL((k_box_restrict<RD, T>), gr, dim3(BLOCK), 0, c->stream, w, rd, bc, stop);
        }
    } else if (fuse && A.nd) {
        MC_DISPATCH_ND(nd_code(A), (k_resid_restrict_seq<ND_, T>), dim3(div_up(L.nc, BLOCK / 8)), dim3(BLOCK), 0,
                       c->stream, A, L.nc, L.agg_ptr, L.agg_members, b, (const T *)cur, bc, stop);
    } else if (A.nd) {
        T *r = (cur == x) ? tmp : x;   // free until post-smoothing
        if constexpr (sizeof(T) == 4) {
            if (half)
                hipLaunchKernelGGL(k_resid_h, dim3(g.blocks), dim3(BLOCK), 0, c->stream, H, b, (const float *)cur, r,
                                   g.chunk, stop);
        }
        if (!half)
            MC_DISPATCH_ND(nd_code(A), (k_resid<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, b,
                           (const T *)cur, r, g.chunk, stop);
        hipLaunchKernelGGL(k_restrict<T>, dim3(div_up(L.nc, BLOCK)), dim3(BLOCK), 0, c->stream, L.nc, L.agg_ptr,
                           L.agg_members, (const T *)r, bc, stop);
    } else {
        hipLaunchKernelGGL(k_resid_restrict<T>, dim3(div_up(L.nc, BLOCK / 64)), dim3(BLOCK), 0, c->stream, A, L.nc,
                           L.agg_ptr, L.agg_members, b, (const T *)cur, bc, stop);
    }
    MC_TRY(vcycle<T>(c, l + 1, bc, xc, nullptr, stop));
    const T cs = (T)c->opt.amg_cscale;
    if (!fuse && !box)
        hipLaunchKernelGGL(k_prolong<T>, dim3(div_up(L.n, BLOCK)), dim3(BLOCK), 0, c->stream, L.n, L.agg,
                           (const T *)xc, cs, cur, stop);
    // post-smoothing: the last sweep writes x (and the fused dot on level 0)
    for (int s = 0; s < nu; s++) {
        const bool last = s == nu - 1;
        T *dst = last ? x : oth;
        if (dst == cur) dst = tmp;
        const T *dotv = (last && ks) ? b : nullptr;
        // A (FP16 copy: its six off-diagonals), dinv, b, x read, x' written
        const double jbytes = (l != 0 || !c->profile) ? 0.0
                              : half ? 28.0 * L.n : mat_bytes(A, L.nnz, sizeof(T)) + 4.0 * sizeof(T) * L.n;
        if (box && s == 0) {
            const BoxProlong<T> pr{box_walk(L), cur, xc, cs};
            const T om = (T)wts[nu - 1 - s];
            bool launched = false;
            if constexpr (sizeof(T) == 4) {
                if (half) {
                    hipLaunchKernelGGL(k_box_jac_prolong_h, dim3(g.blocks), dim3(BLOCK), 0, c->stream, pr, H, b, dst, om,
                                       g.chunk, dotv, c->red, stop);
                    launched = true;
                }
            }
            if (!launched) {
                hipLaunchKernelGGL((k_box_jac_prolong<BND, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, pr, A, dinv,
                                   b, dst, om, g.chunk, dotv, c->red, stop);
            }
        } else if (fuse && s == 0) {
            MC_DISPATCH_ND(nd_code(A), (k_jac_prolong<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, dinv, b,
                           (const T *)cur, L.agg, (const T *)xc, cs, dst, (T)wts[nu - 1 - s], g.chunk, stop);
        } else {
            KTimer kt(c, (l == 0) ? (sizeof(T) == 8 ? MC_KC_JAC64 : MC_KC_JAC32) : -1, jbytes);
            if constexpr (sizeof(T) == 4) {
                if (half)
                    hipLaunchKernelGGL(k_jac_h, dim3(g.blocks), dim3(BLOCK), 0, c->stream, H, b, (const float *)cur,
                                       dst, (float)wts[nu - 1 - s], g.chunk, dotv, c->red, stop);
            }
            if (!half)
                MC_DISPATCH_ND(nd_code(A), (k_jac<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, dinv, b,
                               cur, dst, (T)wts[nu - 1 - s], g.chunk, dotv, c->red, stop);
        }
        if (dotv && !fold_on(c, g)) launch_finish<1>(c->stream, c->red, g.blocks, EpiRz{ks});
        oth = cur;
        cur = dst;
    }
    if (cur != x) MC_HIP(c, hipMemcpyAsync(x, cur, (size_t)L.n * sizeof(T), hipMemcpyDeviceToDevice, c->stream));
    return MC_OK;
}

// Algorithmic bytes of one V-cycle as vcycle() runs it on the built
// hierarchy, each array counted once per pass.  Per level of n rows (T the
// value size, M one pass over its matrix, D its inverse diagonal):
//   first two sweeps from zero   M + D + 2Tn   (b read, x written)
//   each further sweep           M + D + 3Tn   (b, x read, x' written)
//   residual                     M + 3Tn       (+ the FP32 diagonal and D on the FP16 copy)
//   restriction                  4(n + nc + 1) + T(n + nc)
//   prolongation                 4n + T(nc + 2n)
// Below the finest level the residual and restriction share a pass (r is
// neither written nor read again: M + 2Tn + 4(n + nc + 1) + T nc) and the
// prolongation is folded into the first post-smoothing sweep (that sweep
// reads the aggregate ids and the coarse correction, 4n + T nc, and no
// prolonged vector is written or read).  Box levels and regular matched ones do
// the same on every level and read no aggregate ids.  On the FP16 copy M is its six
// off-diagonals (12n) and D the FP32 inverse diagonal; the dense coarsest
// solve reads its inverse (8 n^2) and b, writes x.
template <typename T>
static double vcycle_bytes(Ctx *c)
{
    const int nu = std::max(1, c->opt.amg_nu);
    const double t = (double)sizeof(T);
    double b = 0.0;
    for (size_t l = 0; l < c->amg.size(); l++) {
        AmgLevel &L = c->amg[l];
        const double n = L.n;
        if (l + 1 == c->amg.size()) {
            b += 8.0 * n * n + 2.0 * t * n;
            break;
        }
        const bool half = sizeof(T) == 4 && L.hoff != nullptr && c->opt.amg_half;
        const double M = half ? 12.0 * n : mat_bytes(level_mat<T>(L), L.nnz, sizeof(T));
        const double D = half ? 4.0 * n : t * n;
        b += (nu >= 2 ? M : 0.0) + D + 2.0 * t * n;
        b += (double)std::max(0, nu - 2) * (M + D + 3.0 * t * n);
        if (L.bx || (L.rx && nd_code(level_mat<T>(L)) == (sizeof(T) == 8 ? -7 : 7))) {
            b += M + (half ? 8.0 * n : 0.0) + 2.0 * t * n + t * L.nc;
            b += t * L.nc;
        } else if (l >= 1 && !half) {
            b += M + 2.0 * t * n + 4.0 * (n + L.nc + 1) + t * L.nc;
            b += 4.0 * n + t * L.nc;
        } else {
            b += M + (half ? 8.0 * n : 0.0) + 3.0 * t * n;
            b += 4.0 * (n + L.nc + 1) + t * (n + L.nc);
            b += 4.0 * n + t * (L.nc + 2.0 * n);
        }
        b += (double)nu * (M + D + 3.0 * t * n);
    }
    return b;
}

// ------------------------------------------------------------ PCG --
template <typename T>
struct PcgVecs {
    T *x, *r, *z, *p, *q, *p2;
};

// r = b - mean, x = 0, p = 0; partials of (r, r) and (b - mean, b - mean)
template <typename T>
__global__ void __launch_bounds__(BLOCK) k_pcg_init(int n, const T *b, const double *mean, PcgVecs<T> w,
                                                    double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = bb * chunk, i1 = min(n, i0 + chunk);
    double acc[2] = {0.0, 0.0};
    const double mu = mean ? *mean : 0.0;
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
        const T r = (T)((double)b[i] - mu);
        w.r[i] = r; w.x[i] = (T)0; w.p[i] = (T)0;
        acc[0] += (double)r * (double)r;
    }
    acc[1] = acc[0];
    block_partials<2>(acc, partials, bb, gridDim.x);
}

// from a given x: r = (b - mean) - A x, p = 0; same partials
template <int ND>
__global__ void __launch_bounds__(BLOCK) k_pcg_init_x0(Mat<double> A, const double *b, const double *mean,
                                                       PcgVecs<double> w, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double acc[2] = {0.0, 0.0};
    const double mu = *mean;
    const double *x = w.x;
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return x[j]; }, [&](int i, const double (&ax)[1]) {
        const double bt = b[i] - mu, r = bt - ax[0];
        w.r[i] = r; w.p[i] = 0.0;
        acc[0] += r * r;
        acc[1] += bt * bt;
    });
    block_partials<2>(acc, partials, bb, gridDim.x);
}

// tolerance from ||b - mean||, start from ||r||
struct EpiPcgInit {
    KState *ks;
    double rtol, atol;
    int maxit;
    __device__ void operator()(const double (&v)[2]) const
    {
        const double rn = sqrt(v[0]), bn = sqrt(v[1]);
        ks->bnorm[0] = bn; ks->rnorm[0] = rn;
        ks->tol[0] = fmax(rtol * bn, atol);
        ks->rho_old[0] = 0.0; ks->iters[0] = 0; ks->maxit = maxit;
        ks->done[0] = (rn <= ks->tol[0]) ? 1 : 0;
        ks->conv[0] = ks->done[0];
        ks->all_done = ks->done[0];
    }
};

// p_new = z + beta p_old ; q = A p_new ; alpha = rho / (p_new, q).  The
// product reads z + beta p_old at the neighbours, so the p update needs no
// pass of its own (p_old and p_new are separate buffers).
template <int ND, typename T>
__global__ void __launch_bounds__(BLOCK) k_pcg_pq(Mat<T> A, const T *z, const T *pold, T *pnew, T *q, KState *ks,
                                                  const double *fold, double *partials, int chunk)
{
    if (ks->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double be = fold ? 0.0 : ks->beta[0];
    if (fold) {   // EpiRz here, rho_old left to EpiPcgXr: no block reads what block 0 stores
        double v[1];
        fold_sums<1>(fold, gridDim.x, v);
        be = (ks->iters[0] == 0) ? 0.0 : v[0] / ks->rho_old[0];
        if (blockIdx.x == 0 && threadIdx.x == 0) { ks->rho[0] = v[0]; ks->beta[0] = be; }
    }
    const T beta = (T)be;
    double dsum[1] = {0.0};
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return (double)(z[j] + beta * pold[j]); },
                    [&](int r, const double (&ax)[1]) {
                        const T p = z[r] + beta * pold[r];
                        pnew[r] = p;
                        q[r] = (T)ax[0];
                        dsum[0] += (double)p * ax[0];
                    });
    block_partials<1>(dsum, partials, bb, gridDim.x);
}

struct EpiPcgAlpha {
    KState *ks;
    __device__ void operator()(const double (&v)[1]) const
    {
        if (!ks->all_done) ks->alpha[0] = ks->rho[0] / v[0];
    }
};

template <typename T>
__global__ void __launch_bounds__(BLOCK) k_pcg_xr(int n, T *x, T *r, const T *p, const T *q, const KState *ks,
                                                  const double *fold, double *partials, int chunk)
{
    if (ks->all_done) return;
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = bb * chunk, i1 = min(n, i0 + chunk);
    double a = fold ? 0.0 : ks->alpha[0];
    if (fold) {   // EpiPcgAlpha here
        double v[1];
        fold_sums<1>(fold, gridDim.x, v);
        a = ks->rho[0] / v[0];
    }
    const T al = (T)a;
    double acc[1] = {0.0};
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
        x[i] += al * p[i];
        const T rr = r[i] - al * q[i];
        r[i] = rr;
        acc[0] += (double)rr * (double)rr;
    }
    block_partials<1>(acc, partials, bb, gridDim.x);
}

struct EpiPcgXr {
    KState *ks;
    __device__ void operator()(const double (&v)[1]) const
    {
        if (ks->all_done) return;
        const double rn = sqrt(v[0]);
        ks->rho_old[0] = ks->rho[0];
        ks->rnorm[0] = rn;
        ks->iters[0] += 1;
        if (rn <= ks->tol[0]) { ks->done[0] = 1; ks->conv[0] = 1; }
        else if (ks->iters[0] >= ks->maxit || !(rn == rn)) ks->done[0] = 1;
        ks->all_done = ks->done[0];
    }
};

// One PCG iteration: z = M^-1 r (V-cycle, whose last sweep also forms rho and
// beta), p = z + beta p_old with q = A p (pa: p_old, pb: p), alpha, then x, r
// and ||r||; every step returns at once when the solve is done.
template <typename T>
static int pcg_iteration(Ctx *c, const Mat<T> &A, const Grid &g, PcgVecs<T> w, T *pa, T *pb, KState *ks,
                         double vbytes, const Pub &pub = Pub())
{
    const int n = c->N;
    const bool fold = fold_on(c, g);   // rho, beta and alpha formed by their consumers (fold_sums)
    double *red2 = fold ? c->red + RED_PARTIALS / 2 : c->red;
    {
        KTimer kt(c, MC_KC_VCYCLE, c->profile ? vcycle_bytes<T>(c) : 0.0);
        MC_TRY(vcycle<T>(c, 0, w.r, w.z, ks, ks));
    }
    {
        KTimer kt(c, sizeof(T) == 8 ? MC_KC_SPMV64 : MC_KC_SPMV32, vbytes);
        MC_DISPATCH_ND(nd_code(A), (k_pcg_pq<ND_, T>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, w.z, pa, pb, w.q,
                       ks, fold ? (const double *)c->red : nullptr, red2, g.chunk);
    }
    if (!fold) launch_finish<1>(c->stream, red2, g.blocks, EpiPcgAlpha{ks});
    hipLaunchKernelGGL(k_pcg_xr<T>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, w.x, w.r, pb, w.q, ks,
                       fold ? (const double *)red2 : nullptr, c->red, g.chunk);
    launch_finish<1>(c->stream, c->red, g.blocks, EpiPcgXr{ks}, pub);
    return MC_OK;
}

void graph_release(Ctx *c)
{
    for (auto &pr : c->pcg_graphs)
        for (auto &G : pr) {
            if (G.exec) (void)hipGraphExecDestroy(G.exec);
            G = Ctx::PcgGraph{};
        }
}

// The iteration above as a HIP graph: captured on first use (and again after
// the hierarchy, the options or the vectors changed), then replayed, so the
// GPU runs the V-cycle's ~30 small launches back to back instead of at the
// host's launch rate.  The capture holds kernel launches only (no memset or
// event nodes, no other stream: the coarsest inverse is joined first).
template <typename T>
static int pcg_graph(Ctx *c, const Mat<T> &A, const Grid &g, PcgVecs<T> w, T *pa, T *pb, KState *ks, double vbytes,
                     hipGraphExec_t *out)
{
    Ctx::PcgGraph &G = c->pcg_graphs[sizeof(T) == 8 ? 1 : 0][pa == w.p ? 0 : 1];
    const void *key[8] = {w.x, w.r, w.z, w.p, w.q, w.p2, ks, pa};
    bool hit = G.exec && G.gen == c->graph_gen;
    for (int k = 0; hit && k < 8; k++) hit = G.key[k] == key[k];
    if (!hit) {
        if (G.exec) (void)hipGraphExecDestroy(G.exec);
        G = Ctx::PcgGraph{};
        MC_TRY(dense_join(c));
        MC_HIP(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        const int rc = pcg_iteration<T>(c, A, g, w, pa, pb, ks, vbytes);
        hipGraph_t graph = nullptr;
        const hipError_t e = hipStreamEndCapture(c->stream, &graph);
        if (rc != MC_OK || e != hipSuccess) {
            if (graph) (void)hipGraphDestroy(graph);
            if (rc != MC_OK) return rc;
            c->err = std::string("PCG graph capture: ") + hipGetErrorString(e);
            return MC_ERR_HIP;
        }
        const hipError_t ei = hipGraphInstantiate(&G.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ei != hipSuccess) {
            G.exec = nullptr;
            c->err = std::string("PCG graph instantiation: ") + hipGetErrorString(ei);
            return MC_ERR_HIP;
        }
        G.gen = c->graph_gen;
        for (int k = 0; k < 8; k++) G.key[k] = key[k];
    }
    *out = G.exec;
    return MC_OK;
}

template <typename T>
static int pcg_core(Ctx *c, const T *b, bool project, PcgVecs<T> w, double rtol, double atol, int maxit, KState *ks,
                    KState *hs, int *iters_out, bool x0 = false)
{
    const int n = c->N;
    const Grid g = grid_for(n);
    const Mat<T> A = level_mat<T>(c->amg[0]);
    const double *mean = nullptr;
    if (project) {
        double *dm = c->dscal + 600;
        if constexpr (sizeof(T) == 8) {
            sum_scaled(c, (const double *)b, n, dm, 1.0 / (double)n);
            mean = dm;
        }
    }
    if constexpr (sizeof(T) == 8) {
        if (x0 && mean) {
            MC_DISPATCH_ND(nd_code(A), (k_pcg_init_x0<ND_>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A,
                           (const double *)b, mean, w, c->red, g.chunk);
        } else {
            hipLaunchKernelGGL(k_pcg_init<T>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, b, mean, w, c->red,
                               g.chunk);
        }
    } else {
        hipLaunchKernelGGL(k_pcg_init<T>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, b, mean, w, c->red, g.chunk);
    }
    launch_finish<2>(c->stream, c->red, g.blocks, EpiPcgInit{ks, rtol, atol, maxit});
    MC_LAUNCH_CHECK(c);
    // A; z and p_old read, p and q written
    const double vbytes = mat_bytes(A, c->nnz, sizeof(T)) + 4.0 * sizeof(T) * n;
    T *pa = w.p, *pb = w.p2;
    int it = 0, batch = 2;
    double rn_prev = -1.0;
    // the kernel classes an iteration would time: profiling them launches
    // kernel by kernel
    const unsigned timed = (1u << MC_KC_VCYCLE) | (1u << MC_KC_SPMV64) | (1u << MC_KC_SPMV32) |
                           (1u << MC_KC_JAC64) | (1u << MC_KC_JAC32);
    const bool graphs = c->opt.pcg_graph && !(c->profile & timed) && c->stream != nullptr;   // no capture on the null stream
    for (;;) {
        for (int j = 0; j < batch && it < maxit; j++, it++) {
            if (graphs) {
                hipGraphExec_t ge = nullptr;
                MC_TRY(pcg_graph<T>(c, A, g, w, pa, pb, ks, vbytes, &ge));
                MC_TRY(dense_join(c));
                MC_HIP(c, hipGraphLaunch(ge, c->stream));
            } else {
                const bool last = j == batch - 1 || it == maxit - 1;
                MC_TRY(pcg_iteration<T>(c, A, g, w, pa, pb, ks, vbytes,
                                        last ? make_pub(c, ks, 0, sizeof(KState)) : Pub()));
            }
            std::swap(pa, pb);
        }
        MC_LAUNCH_CHECK(c);
        MC_TRY(graphs ? poll_done(c, ks, hs) : wait_pub(c));
        c->st.host_polls++;
        if (hs->all_done || it >= maxit) break;
        const double rn = hs->rnorm[0] / std::max(hs->tol[0], 1e-300);
        batch = predict_batch(rn_prev, rn, batch, 1.0, 8);
        rn_prev = rn;
    }
    *iters_out = hs->iters[0];
    return MC_OK;
}

__global__ void k_sub_mean(int n, double *x, const double *mean)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] -= *mean;
}

static int project_mean_zero(Ctx *c, double *x)
{
    const int n = c->N;
    double *dm = c->dscal + 610;
    sum_scaled(c, x, n, dm, 1.0 / (double)n);
    hipLaunchKernelGGL(k_sub_mean, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n, x, dm);
    MC_LAUNCH_CHECK(c);
    return MC_OK;
}

int pcg_amg(Ctx *c, const double *vals, const double *b, double *x, double rtol, int maxit, double atol,
            mc_solve_status *st, bool x0)
{
    (void)vals;  // the hierarchy's level 0 holds these values
    KState *ks = (KState *)c->dscal;
    KState *hs = (KState *)c->hscal;
    PcgVecs<double> w{x, c->wk[0], c->wk[1], c->wk[2], c->wk[3], c->wk[5]};
    int iters = 0;
    MC_TRY(pcg_core<double>(c, b, true, w, rtol, atol, maxit, ks, hs, &iters, x0));
    // met at the zero start: x is all +0, already mean-zero
    c->p_zero = !x0 && iters == 0 && hs->conv[0];
    if (!c->p_zero) MC_TRY(project_mean_zero(c, x));
    if (st) {
        st->iterations = iters;
        st->converged = hs->conv[0];
        st->relres = hs->bnorm[0] > 0 ? hs->rnorm[0] / hs->bnorm[0] : 0.0;
        st->outer = 1;
        st->bnorm = hs->bnorm[0];
    }
    return MC_OK;
}

// ---------------------------------------------- mixed: FP32 inside FP64 IR --
template <int ND>
__global__ void __launch_bounds__(BLOCK) k_ir_resid(Mat<double> A, const double *b, const double *mean, const double *x,
                                                    double *r, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double dsum[1] = {0.0};
    const double mu = *mean;
    for_rows<ND, 1>(A, r0, r1, [&](int, int j) { return x[j]; }, [&](int row, const double (&ax)[1]) {
        const double rr = (b[row] - mu) - ax[0];
        r[row] = rr;
        dsum[0] += rr * rr;
    });
    block_partials<1>(dsum, partials, bb, gridDim.x);
}

// The first refinement residual of a solve started from zero: r = b - mean
// (the product A 0 adds +0.0, so these are the bits k_ir_resid gives for a
// matrix in diagonal storage, whose rows it visits in the same order) with x
// set to zero in the same pass; A and x are not read.
__global__ void __launch_bounds__(BLOCK) k_ir_resid0(int n, const double *b, const double *mean, double *x,
                                                     double *r, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(n, r0 + chunk);
    double dsum[1] = {0.0};
    const double mu = *mean;
    for (int row = r0 + threadIdx.x; row < r1; row += BLOCK) {
        const double rr = b[row] - mu;
        r[row] = rr;
        x[row] = 0.0;
        dsum[0] += rr * rr;
    }
    block_partials<1>(dsum, partials, bb, gridDim.x);
}

struct EpiSqrt {
    double *out;
    __device__ void operator()(const double (&v)[1]) const { *out = sqrt(v[0]); }
};

__global__ void k_to32_scaled(int n, const double *r, const double *nrm, float *r32)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double s = (*nrm > 0.0) ? 1.0 / *nrm : 0.0;
    r32[i] = (float)(r[i] * s);
}

__global__ void k_ir_update(int n, double *x, const float *e32, const double *nrm)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] += (double)e32[i] * *nrm;
}

__global__ void k_zero(int n, double *x)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0;
}

int mixed_ir_solve(Ctx *c, const double *vals, const double *b, double *x, double rtol, int maxit, double atol,
                   mc_solve_status *st, bool x0, double bnorm0, const IrStart *start)
{
    (void)vals;
    const int n = c->N;
    const Grid g = grid_for(n);
    KState *ks = (KState *)c->dscal;
    KState *hs = (KState *)c->hscal;
    double *rn = c->dscal + 621;
    const double *mean = c->dscal + 620;
    double *r = c->wk[4];
    float *r32 = c->wk32[0], *e32 = c->wk32[1];
    PcgVecs<float> w{e32, c->wk32[2], c->wk32[3], c->wk32[4], c->wk32[5], c->wk32[6]};
    const Mat<double> A = level_mat<double>(c->amg[0]);
    if (start) mean = start->mean;   // the deflation start's mean and first residual
    else sum_scaled(c, b, n, c->dscal + 620, 1.0 / (double)n);
    // diagonal storage: the first residual of a zero start skips A (same bits,
    // the same rows per thread); CSR rows are reduced in another order
    const bool fast0 = !x0 && nd_code(A) != 0;
    if (!x0 && !fast0) hipLaunchKernelGGL(k_zero, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n, x);
    double bnorm = x0 ? bnorm0 : -1.0, rnorm = 0.0;
    int total = 0, outer = 0;
    bool conv = false;
    const double inner = c->opt.mixed_inner_rtol > 0 ? c->opt.mixed_inner_rtol : 1e-5;
    const double rbytes = mat_bytes(A, c->nnz, 8) + 24.0 * n;   // A; b, x read, r written
    for (outer = 0; outer < 50; outer++) {
        const double *rnd = rn;   // ||r|| on the device, the scale of this step's FP32 system
        if (outer == 0 && start) {
            rnd = start->rn;
            rnorm = start->rnorm;
        } else {
            if (outer == 0 && fast0) {
                hipLaunchKernelGGL(k_ir_resid0, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, b, mean, x, r, c->red,
                                   g.chunk);
            } else {
                KTimer kt(c, MC_KC_IR_RESID, rbytes);
                MC_DISPATCH_ND(nd_code(A), (k_ir_resid<ND_>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, b, mean, x,
                               r, c->red, g.chunk);
            }
            launch_finish<1>(c->stream, c->red, g.blocks, EpiSqrt{rn}, make_pub(c, rn, 621, sizeof(double)));
            MC_LAUNCH_CHECK(c);
            MC_TRY(wait_pub(c));
            c->st.host_polls++;
            rnorm = c->hscal[621];
        }
        if (bnorm < 0) bnorm = rnorm;
        if (rnorm <= std::max(rtol * bnorm, atol) || !(rnorm == rnorm)) { conv = rnorm == rnorm; break; }
        if (total >= maxit) break;
        hipLaunchKernelGGL(k_to32_scaled, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n, r, rnd, r32);
        // the last refinement step needs only the remaining reduction
        const double need = std::max(rtol * bnorm, atol) / rnorm;
        int it = 0;
        MC_TRY(pcg_core<float>(c, r32, false, w, std::max(inner, 0.5 * need), 0.0, maxit - total, ks, hs, &it));
        total += it;
        hipLaunchKernelGGL(k_ir_update, dim3(div_up(n, 256)), dim3(256), 0, c->stream, n, x, e32, rnd);
        MC_LAUNCH_CHECK(c);
    }
    // met at the zero start: x is all +0, already mean-zero
    c->p_zero = !x0 && conv && total == 0;
    if (!c->p_zero) MC_TRY(project_mean_zero(c, x));
    if (st) {
        st->iterations = total;
        st->converged = conv ? 1 : 0;
        st->relres = bnorm > 0 ? rnorm / bnorm : 0.0;
        st->outer = outer;
        st->bnorm = bnorm;
    }
    return MC_OK;
}

// ------------------------------------------------ deflation-space start --
// A loop-1 pressure solve starts from the Galerkin projection of its solution
// onto the deflation space W = [g, x_1, ..., x_s]: g the learned net's guess
// (when the learned form uses it for this solve), x_1 .. x_s the last
// s = p_recycle loop-1 solutions (newest first), every vector mean-zero.
// x0 = W y with (W^T A W) y = W^T b is the vector of span W closest to the
// solution in the A-norm, so the error left to the PCG is A-orthogonal to W.
// The K x K system (K <= 5) is solved by Cholesky on one thread; a vector
// whose pivot falls to 1e-10 of its diagonal entry (numerically in the span
// of the earlier ones: successive solutions are nearly parallel), or is not a
// number (a net output with NaN / Inf fails every comparison), is dropped.
// The start is kept only if ||b - A x0|| < ||b - mean b||, else x0 = 0, so the
// solve never starts worse than the reference's zero start.  The PCG-AMG and
// its residual test are unchanged: W can change the iteration count, never
// the tolerance met.
constexpr int DEFL_W = DEFL_MAX + 1;   // the learned guess and the recycled solutions

struct DeflVecs {
    const double *w[DEFL_W];
    double *aw[DEFL_W];
};

template <int K>
constexpr int defl_nv() { return K * (K + 3) / 2 + 1; }   // E upper triangle, W^T b, sum b

// aw_k = A w_k for the K vectors in one pass over the matrix, with the block
// partials of (w_a, aw_c) for a <= c, (w_a, b) and sum b formed from the
// products' rows as they are made (each row read once, not again by a
// separate reduction pass)
template <int ND, int K>
__global__ void __launch_bounds__(BLOCK) k_defl_aw_dots(Mat<double> A, DeflVecs v, const double *b, double *partials,
                                                        int chunk)
{
    constexpr int NV = defl_nv<K>();
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = bb * chunk, r1 = min(A.n, r0 + chunk);
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) acc[q] = 0.0;
    for_rows<ND, K>(A, r0, r1, [&](int k, int j) { return v.w[k][j]; }, [&](int row, const double (&ax)[K]) {
        double w[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            v.aw[k][row] = ax[k];
            w[k] = v.w[k][row];
        }
        const double bi = b[row];
        int q = 0;
#pragma unroll
        for (int a = 0; a < K; a++)
#pragma unroll
            for (int c = a; c < K; c++) acc[q++] += w[a] * ax[c];
#pragma unroll
        for (int a = 0; a < K; a++) acc[q++] += w[a] * bi;
        acc[q] += bi;
    });
    block_partials<NV>(acc, partials, bb, gridDim.x);
}

// sc[0] = mean b, sc[1 .. K] = y, sc[K + 1] = vectors kept
template <int K>
struct EpiDefl {
    double *sc;
    double inv_n;
    __device__ void operator()(const double (&v)[defl_nv<K>()]) const
    {
        double E[K][K], f[K], L[K][K], z[K], y[K];
        bool keep[K];
        int q = 0;
        for (int a = 0; a < K; a++)
            for (int c = a; c < K; c++) { E[a][c] = v[q]; E[c][a] = v[q]; q++; }
        for (int a = 0; a < K; a++) f[a] = v[q++];
        sc[0] = v[q] * inv_n;
        int kept = 0;
        for (int j = 0; j < K; j++) {
            for (int i = 0; i < K; i++) L[i][j] = 0.0;
            double d = E[j][j];
            for (int k = 0; k < j; k++)
                if (keep[k]) d -= L[j][k] * L[j][k];
            keep[j] = E[j][j] > 0.0 && d > 1e-10 * E[j][j];
            if (!keep[j]) continue;
            kept++;
            L[j][j] = sqrt(d);
            for (int i = j + 1; i < K; i++) {
                double t = E[i][j];
                for (int k = 0; k < j; k++)
                    if (keep[k]) t -= L[i][k] * L[j][k];
                L[i][j] = t / L[j][j];
            }
        }
        for (int i = 0; i < K; i++) {
            z[i] = 0.0;
            if (!keep[i]) continue;
            double t = f[i];
            for (int k = 0; k < i; k++)
                if (keep[k]) t -= L[i][k] * z[k];
            z[i] = t / L[i][i];
        }
        for (int i = K - 1; i >= 0; i--) {
            y[i] = 0.0;
            if (!keep[i]) continue;
            double t = z[i];
            for (int k = i + 1; k < K; k++)
                if (keep[k]) t -= L[k][i] * y[k];
            y[i] = t / L[i][i];
        }
        for (int i = 0; i < K; i++) sc[1 + i] = y[i];
        sc[K + 1] = kept;
    }
};

// x = W y and r = (b - mean) - A W y (from the stored products), with the
// partials of ||b - mean||^2 and ||r||^2: the start, its residual (the first
// residual of the refinement that follows) and the two norms of its
// acceptance test in one pass.  A dropped vector has y_k = 0 and is skipped
// (it may hold NaN).  x and r are written whatever the test decides: a
// rejected start leaves the solve to set x = 0 itself.
template <int K>
__global__ void __launch_bounds__(BLOCK) k_defl_start(int n, DeflVecs v, const double *b, const double *sc, double *x,
                                                      double *r, double *partials, int chunk)
{
    const int bb = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = bb * chunk, i1 = min(n, i0 + chunk);
    double y[K];
#pragma unroll
    for (int k = 0; k < K; k++) y[k] = sc[1 + k];
    const double mu = sc[0];
    double acc[2] = {0.0, 0.0};
    for (int i = i0 + threadIdx.x; i < i1; i += BLOCK) {
        const double bt = b[i] - mu;
        double rr = bt, s = 0.0;
#pragma unroll
        for (int k = 0; k < K; k++)
            if (y[k] != 0.0) {
                rr -= y[k] * v.aw[k][i];
                s += y[k] * v.w[k][i];
            }
        x[i] = s;
        r[i] = rr;
        acc[0] += bt * bt;
        acc[1] += rr * rr;
    }
    block_partials<2>(acc, partials, bb, gridDim.x);
}

// sc[K + 2] = ||b - mean||, sc[K + 3] = ||r0||, sc[K + 4] = 1 if the start is kept
struct EpiDeflAccept {
    double *sc;
    int K;
    __device__ void operator()(const double (&v)[2]) const
    {
        const double bn = sqrt(v[0]), rn = sqrt(v[1]);
        sc[K + 2] = bn;
        sc[K + 3] = rn;
        sc[K + 4] = (sc[K + 1] > 0.0 && rn < bn) ? 1.0 : 0.0;
    }
};

// A grid for the deflation reductions: at most 21 partials per block.
static Grid defl_grid(int n)
{
    Grid g = grid_for(n);
    while (g.blocks > RED_PARTIALS / defl_nv<DEFL_W>() && g.chunk < (1 << 28)) {
        g.chunk *= 2;
        g.blocks = div_up(n, g.chunk);
    }
    return g;
}

static int defl_buffers(Ctx *c, int nrec)
{
    MemScope ms(c, MC_MEM_WORK);
    for (int k = 0; k < nrec; k++)
        if (!c->defl_x[k]) MC_TRY(dalloc(c, &c->defl_x[k], (size_t)c->N));
    for (int k = 0; k <= nrec; k++)
        if (!c->defl_aw[k]) MC_TRY(dalloc(c, &c->defl_aw[k], (size_t)c->N));
    return MC_OK;
}

template <int K>
static void defl_launch(Ctx *c, const DeflVecs &v, const double *b, double *x, double *r, double *sc)
{
    const int n = c->N;
    const Grid g = defl_grid(n);
    const Mat<double> A = level_mat<double>(c->amg[0]);
    MC_DISPATCH_ND(nd_code(A), (k_defl_aw_dots<ND_, K>), dim3(g.blocks), dim3(BLOCK), 0, c->stream, A, v, b, c->red,
                   g.chunk);
    launch_finish<defl_nv<K>()>(c->stream, c->red, g.blocks, EpiDefl<K>{sc, 1.0 / n});
    hipLaunchKernelGGL(k_defl_start<K>, dim3(g.blocks), dim3(BLOCK), 0, c->stream, n, v, b, (const double *)sc, x, r,
                       c->red, g.chunk);
    launch_finish<2>(c->stream, c->red, g.blocks, EpiDeflAccept{sc, K}, make_pub(c, sc, 640, (K + 5) * sizeof(double)));
}

// The start of a loop-1 solve: *used = the start is kept (x = W y, and *ir
// the refinement's first residual: r = b - mean b - A x in wk[4], its norm
// and the mean), *bnorm = ||b - mean b||; *guess = the learned guess is in W.
// A start not kept leaves x to the solve, which starts from zero.
static int deflation_start(Ctx *c, const double *b, double *x, bool want_guess, bool *used, double *bnorm,
                           bool *guess, IrStart *ir)
{
    *used = false;
    *guess = false;
    *bnorm = 0.0;
    const int n = c->N;
    const int nrec = (c->defl_cap == c->opt.p_recycle) ? std::min(c->opt.p_recycle, c->defl_count) : 0;
    if (c->opt.p_recycle > 0 || want_guess) MC_TRY(defl_buffers(c, std::max(c->opt.p_recycle, 0)));
    DeflVecs v{};
    int K = 0;
    if (want_guess && c->mpnn) {
        int ok = 0;
        double *gv = c->wk[6];
        MC_TRY(mpnn_guess(c, b, gv, &ok));
        if (ok) {
            MC_TRY(project_mean_zero(c, gv));
            v.w[K] = gv;
            v.aw[K] = c->defl_aw[K];
            K++;
            *guess = true;
        }
    }
    for (int k = 0; k < nrec; k++, K++) {
        v.w[K] = c->defl_x[(c->defl_head - k + c->defl_cap) % c->defl_cap];
        v.aw[K] = c->defl_aw[K];
    }
    if (K == 0) return MC_OK;
    double *sc = c->dscal + 640, *r = c->wk[4];
    switch (K) {
    case 1: defl_launch<1>(c, v, b, x, r, sc); break;
    case 2: defl_launch<2>(c, v, b, x, r, sc); break;
    case 3: defl_launch<3>(c, v, b, x, r, sc); break;
    case 4: defl_launch<4>(c, v, b, x, r, sc); break;
    default: defl_launch<5>(c, v, b, x, r, sc); break;
    }
    MC_LAUNCH_CHECK(c);
    MC_TRY(wait_pub(c));
    const double *h = c->hscal + 640;
    *used = h[K + 4] > 0.0;
    *bnorm = h[K + 2];
    // the guess is w[0]; a dropped vector (NaN / Inf output, or in the span
    // of the others) has coefficient exactly 0 and contributes nothing to x0
    if (*guess && h[1] == 0.0) *guess = false;
    if (*used) {
        ir->mean = sc;
        ir->rn = sc + K + 3;
        ir->rnorm = h[K + 3];
        const double ratio = h[K + 2] > 0.0 ? h[K + 3] / h[K + 2] : 0.0;
        c->st.p_defl_starts += 1;
        c->st.p_defl_ratio_sum += ratio;
        c->st.p_defl_vectors += (int64_t)h[K + 1];
        if (*guess) c->st.p_guess_ratio_sum += ratio;
    } else {
        *guess = false;
    }
    return MC_OK;
}

// A converged loop-1 solution (mean-zero) joins the recycled solutions: a
// ring of p_recycle slots (restarted when p_recycle changes).
static int defl_push(Ctx *c, const double *x)
{
    const int cap = c->opt.p_recycle;
    if (cap <= 0) return MC_OK;
    MC_TRY(defl_buffers(c, cap));
    if (c->defl_cap != cap) {
        c->defl_cap = cap;
        c->defl_count = 0;
        c->defl_head = cap - 1;
    }
    const int slot = (c->defl_head + 1) % cap;
    MC_HIP(c, hipMemcpyAsync(c->defl_x[slot], x, (size_t)c->N * 8, hipMemcpyDeviceToDevice, c->stream));
    c->defl_head = slot;
    c->defl_count = std::min(c->defl_count + 1, cap);
    return MC_OK;
}

static double ema(double old, double v) { return old < 0.0 ? v : 0.7 * old + 0.3 * v; }

int pressure_solve(Ctx *c, const double *b, double *x, mc_solve_status *st, double atol)
{
    const auto t0 = std::chrono::steady_clock::now();
    mc_solve_status s{};
    int rc;
    bool used = false, tried = false;
    double bn0 = 0.0;
    // a state set through the C-ABI can reach a solve before any assembly
    // built the hierarchy: build it from the stored pressure matrix
    if (!amg_current(c)) MC_TRY(amg_setup(c, c->PA_vals));
    // learned = 2: every loop-1 solve starts from the guess; learned = 1: only
    // while its measured saving (iterations x time per iteration) exceeds its
    // cost, re-checking the other choice after 16 solves, then after twice as
    // many each time a re-check confirms the choice (at most 1024)
    bool recheck = false, guess = false;
    IrStart ir{};
    if (c->opt.learned && c->mpnn && atol == 0.0) {
        tried = true;
        if (c->opt.learned == 1) {
            if (c->lg_it_on < 0.0) tried = true;
            else if (c->lg_it_off < 0.0) tried = false;
            else {
                recheck = c->lg_count - c->lg_last >= c->lg_period;
                tried = recheck ? !c->lg_on : c->lg_on;
            }
        }
    }
    // loop-1 solves (atol == 0) start from the deflation space when it holds
    // a vector; later loops solve the small non-orthogonal remainder from zero
    if (atol == 0.0 && (tried || c->opt.p_recycle > 0))
        MC_TRY(deflation_start(c, b, x, tried, &used, &bn0, &guess, &ir));
    const auto tg = std::chrono::steady_clock::now();
    if (c->opt.psolve == MC_PSOLVE_MIXED)
        rc = mixed_ir_solve(c, c->PA_vals, b, x, c->opt.p_rtol, c->opt.p_maxit, atol, &s, used, bn0,
                            used ? &ir : nullptr);
    else
        rc = pcg_amg(c, c->PA_vals, b, x, c->opt.p_rtol, c->opt.p_maxit, atol, &s, used);
    s.guess_used = guess ? 1 : 0;
    const auto t1 = std::chrono::steady_clock::now();
    c->st.p_solve_ms += std::chrono::duration<double, std::milli>(t1 - t0).count();
    if (rc) return rc;
    if (c->opt.learned && c->mpnn && atol == 0.0) {
        // the guess's cost: the start's time with it over the start's time
        // without it (the recycled vectors cost the same in both)
        const double solve_ms = std::chrono::duration<double, std::milli>(t1 - tg).count();
        const double start_ms = std::chrono::duration<double, std::milli>(tg - t0).count();
        if (s.iterations > 0) c->lg_iter_ms = ema(c->lg_iter_ms, solve_ms / s.iterations);
        if (tried) {
            c->lg_cost_ms = ema(c->lg_cost_ms, start_ms);
            c->lg_it_on = ema(c->lg_it_on, guess ? s.iterations : (c->lg_it_off < 0 ? s.iterations : c->lg_it_off));
        } else {
            c->lg_base_ms = ema(c->lg_base_ms, start_ms);
            c->lg_it_off = ema(c->lg_it_off, s.iterations);
        }
        const bool was_on = c->lg_on;
        if (c->lg_it_on >= 0.0 && c->lg_it_off >= 0.0)
            c->lg_on = (c->lg_it_off - c->lg_it_on) * c->lg_iter_ms > c->lg_cost_ms - std::max(c->lg_base_ms, 0.0);
        if (recheck) {
            c->lg_last = c->lg_count;
            c->lg_period = (c->lg_on == was_on) ? std::min(2 * c->lg_period, 1024) : 16;
        }
        c->lg_count++;
    }
    c->st.p_guesses += guess ? 1 : 0;
    if (c->mpnn) MC_TRY(mpnn_collect_pair(c, b, x));
    if (atol == 0.0 && s.converged) MC_TRY(defl_push(c, x));
    c->st.p_iters += s.iterations;
    c->st.p_solves += 1;
    c->st.p_outer += s.outer;
    c->st.last_p_relres = s.relres;
    {
        const double ref = std::max(s.bnorm, atol / c->opt.p_rtol);
        const double eff = ref > 0 ? s.relres * s.bnorm / ref : 0.0;
        c->st.p_relres_max = std::max(c->st.p_relres_max, eff);
    }
    if (st) *st = s;
    if (!s.converged) {
        c->err = "pressure solve did not converge";
        return MC_ERR_NOCONV;
    }
    return MC_OK;
}

// ------------------------------------------------------ copy probe --
// Streaming copy, the known-size kernel for HBM bandwidth and counter
// calibration: one 16-byte element per lane, one lane per element (a grid of
// n / 256 workgroups), streaming (non-temporal) loads and stores; every
// element is read once and written once.  Of the forms measured on the
// MI355X (several elements per lane at a 256-lane stride, grid-stride loops,
// plain or streaming accesses) this one moves the most bytes per second.
typedef double dvec2 __attribute__((ext_vector_type(2)));
__global__ void __launch_bounds__(256) k_copy_probe(int64_t n16, const dvec2 *__restrict__ src,
                                                   dvec2 *__restrict__ dst)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

int copy_probe(Ctx *c, int64_t bytes, int reps, double *ms_out)
{
    void *src = nullptr, *dst = nullptr;
    MC_HIP(c, hipMalloc(&src, (size_t)bytes));
    if (hipMalloc(&dst, (size_t)bytes) != hipSuccess) {
        (void)hipFree(src);
        c->err = "copy probe: hipMalloc failed";
        return MC_ERR_NOMEM;
    }
    int rc = MC_OK;
    hipEvent_t a = nullptr, b = nullptr;
    const int64_t n16 = bytes / 16;
    if (div_up(n16, 256) > INT32_MAX) {
        c->err = "copy probe: size beyond one launch";
        return MC_ERR_ARG;
    }
    const int blocks = div_up(n16, 256);
    if (hipMemsetAsync(src, 0, (size_t)bytes, c->stream) != hipSuccess || hipEventCreate(&a) != hipSuccess ||
        hipEventCreate(&b) != hipSuccess) {
        rc = MC_ERR_HIP;
    } else {
        hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, c->stream, n16, (const dvec2 *)src,
                           (dvec2 *)dst);   // untimed first touch
        (void)hipEventRecord(a, c->stream);
        for (int r = 0; r < reps; r++)
            hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, c->stream, n16, (const dvec2 *)src,
                               (dvec2 *)dst);
        (void)hipEventRecord(b, c->stream);
        float ms = 0.f;
        if (hipEventSynchronize(b) != hipSuccess || hipEventElapsedTime(&ms, a, b) != hipSuccess) rc = MC_ERR_HIP;
        *ms_out = (double)ms / reps;
    }
    if (rc) c->err = "copy probe: HIP error";
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    (void)hipFree(src);
    (void)hipFree(dst);
    return rc;
}

}  // namespace mc
