// lv_amg.hip -- multilevel preconditioner for the pressure system of find_pressure! (src/pressure.jl:89-224).
//
// No counterpart in the reference (it runs unpreconditioned MINRES, src/pressure.jl:219).  A
// one-ring preconditioner can shrink the condition number of the Voronoi Laplacian by a constant
// factor only; the smooth error modes need a coarse correction.
//
// Hierarchy (rebuilt for every assembled operator):
//   level 0: the particles and A itself (ELL, FP32);
//   level 1: the cells of a regular grid of width >= CELL_DR dr (2 dr: about 4 particles a cell)
//            over the boundary rectangle; every particle is aggregated into the cell holding it.
//            Cells of 4 dr (16 particles) coarsen faster but cost 20% more CG iterations on the
//            2048^2 benchmark steps (171 against 142 at 2 dr) for less work per cycle.  The Galerkin operator P^T A P of the
//            piecewise-constant P keeps the reference's difference form:
//              d_I = sum_{i in I} d_i,   c_IJ = sum_{i in I, j in J} c_ij,
//            stored as a 3x3 stencil (a coupling that would reach beyond the neighbouring cells,
//            only possible on strongly distorted meshes, is dropped from both sides, which keeps
//            the coarse operator positive semi-definite);
//   level l+1: 2 x 2 blocks of level-l cells, the same Galerkin rule (4 x 4 blocks coarsen too fast
//            for the V-cycle: on the 2048^2 benchmark system PCG needs ~60 iterations with them,
//            ~40 with 2 x 2);
//   the coarsest level (<= LV_AMG_DENSE_MAX cells) is inverted densely once per assembly.
// The small levels (from the first of at most LDS_MAX cells, or TAIL_MAX in a singular system) run inside
// one single-workgroup kernel per cycle (k_tail_lds): they are
// too small to fill the device, and one launch replaces two per level.  A singular system's cycle multiplies by
// the matrix of that kernel's W-visit instead (k_mat_mv).  Above them, levels
// 2 and up run in pairs, each pair as one down and one up kernel (k_st_down2, k_st_up2) that
// recompute a halo around each workgroup's tile instead of waiting for a second launch.
// Every sum is a gather in a fixed order (per-aggregate row lists are sorted), so the hierarchy
// and the preconditioner are deterministic.
//
// Cycle: symmetric V(1,1).  The fine smoother is the learned SPAI (M of lv_spai.hip, scaled so
// that the largest eigenvalue of M A is ~1.2, estimated by power iteration at set-up) or, without
// it, damped Jacobi (2/3 D^-1); the coarse smoothers are damped Jacobi.  The cycle is an SPD
// linear operator, so CG stays valid; it runs in FP32 inside the FP64 iterative refinement, where
// Jacobi-PCG remains the fallback and the FP64 residual remains the judge.
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "lv_amg.h"
#include "lv_ell.h"
#include "lv_reduce.h"

namespace {

constexpr int B = 256;
constexpr float OMEGA = 2.0f / 3.0f;  // damped Jacobi
constexpr float FINE_TARGET = 1.2f;   // lambda_max of the scaled learned smoother times A
constexpr int CF = 2;                 // coarse levels: CF x CF blocks of the finer level's cells
// Over-correction: the prolongated coarse correction is scaled by ALPHA_FINE into the fine level and
// by ALPHA_COARSE into a coarse level, except for corrections from the levels of at most TAIL_MAX
// cells (solved nearly exactly, where a scaling only overshoots).  The piecewise-constant
// prolongation leaves the coarse correction short in energy; the scaling keeps the cycle SPD for
// any factor >= 0 (I - a P B_c P^T A stays <= I in the A inner product when B_c is SPD) and cuts
// the PCG iterations on the 2048^2 benchmark system from 41 to ~34.
constexpr float ALPHA_FINE = 1.6f;
constexpr float ALPHA_COARSE = 1.4f;
constexpr int CF2 = CF * CF;
constexpr double CELL_DR = 2.0;  // level-1 cell width in units of dr
constexpr int RL = 4;            // lanes that restrict one level-1 cell (about 4 rows each)

// the sum of RL consecutive lanes by a fixed shuffle tree, in every one of them
__device__ __forceinline__ float sum_lanes(float s)
{
#pragma unroll
    for (int m = 1; m < RL; m <<= 1) s += __shfl_xor(s, m);
    return s;
}
__device__ __forceinline__ double sum_lanes(double s)
{
#pragma unroll
    for (int m = 1; m < RL; m <<= 1) s += __shfl_xor(s, m);
    return s;
}

inline dim3 g1(int64_t count) { return dim3((unsigned)std::max<int64_t>(1, (count + B - 1) / B)); }

// 3x3 stencil slots: k = 0..7 for the offsets (dx, dy), dx-major, skipping (0, 0)
__device__ __forceinline__ int slot_of(int dx, int dy)
{
    const int q = (dx + 1) * 3 + (dy + 1);
    return q > 4 ? q - 1 : q;
}
__device__ __forceinline__ void offset_of(int k, int &dx, int &dy)
{
    const int q = k >= 4 ? k + 1 : k;
    dx = q / 3 - 1;
    dy = q % 3 - 1;
}
// a cell offset on a periodic axis of K cells, folded into [-(K-1)/2, K/2]
__device__ __forceinline__ int fold(int d, int K, int per)
{
    if (!per) return d;
    d %= K;
    if (d > K / 2) d -= K;
    if (d < -((K - 1) / 2)) d += K;
    return d;
}
__device__ __forceinline__ int wrap(int i, int K, int per, bool &ok)
{
    if (per) {
        ok = true;
        return (i % K + K) % K;
    }
    ok = (i >= 0 && i < K);
    return i;
}

// ---- level 1: aggregation of the particles -----------------------------------------------------

__global__ __launch_bounds__(B) void k_agg_key(int n, const double *__restrict__ x, double x0, double y0, double hx,
                                               double hy, int Kx, int Ky, int *__restrict__ agg,
                                               int *__restrict__ cnt)
{
    const int i = blockIdx.x * B + threadIdx.x;
    const bool act = i < n;
    int a = 0;
    if (act) {
        int ix = (int)floor((x[i] - x0) / hx), iy = (int)floor((x[n + i] - y0) / hy);
        ix = ix < 0 ? 0 : (ix >= Kx ? Kx - 1 : ix);
        iy = iy < 0 ? 0 : (iy >= Ky ? Ky - 1 : iy);
        a = ix * Ky + iy;
        agg[i] = a;
    }
    (void)lv_run_atomic_add<1>(cnt, a, act);  // half the atomics, which bound this kernel and the next
}

// (the order of a cell's rows in list is then fixed by k_agg_sort; cnt is back at zero for the next set-up)
__global__ __launch_bounds__(B) void k_agg_fill(int n, const int *__restrict__ agg, const int *__restrict__ start,
                                                int *__restrict__ cnt, int *__restrict__ list)
{
    const int i = blockIdx.x * B + threadIdx.x;
    const bool act = i < n;
    const int a = act ? agg[i] : 0;
    const int p = lv_run_atomic_add<-1>(cnt, a, act);
    if (act) list[start[a] + p] = i;
}

// per cell: its rows sorted (a fixed order for every sum over a cell's rows, here and in the
// aggregate order)
__global__ __launch_bounds__(B) void k_agg_sort(int na, const int *__restrict__ start, int *__restrict__ list)
{
    const int I = blockIdx.x * B + threadIdx.x;
    if (I >= na) return;
    const int s0 = start[I], s1 = start[I + 1];
    for (int a = s0 + 1; a < s1; a++) {
        const int v = list[a];
        int b = a;
        while (b > s0 && list[b - 1] > v) {
            list[b] = list[b - 1];
            b--;
        }
        list[b] = v;
    }
}

// per cell, RL lanes: the Galerkin sums of d and of the couplings to the 8 neighbouring cells in
// FP64, lane q over the cell's sorted rows q, q + RL, ..., then the lanes' sums added by sum_lanes'
// fixed tree
__global__ __launch_bounds__(B) void k_coarse1(int na, int Kx, int Ky, int xper, int yper,
                                               const int *__restrict__ start, const int *__restrict__ list,
                                               const int *__restrict__ agg, int n, const int *__restrict__ deg,
                                               const int *__restrict__ ecol, const double *__restrict__ ev,
                                               const double *__restrict__ d64, float *__restrict__ dout,
                                               float *__restrict__ cout, float *__restrict__ dinv)
{
    const int t = blockIdx.x * B + threadIdx.x;
    const int I = t / RL, q = t % RL;
    const bool live = I < na;  // every lane takes part in the shuffles below
    const int Ic = live ? I : 0;
    const int s0 = start[Ic], s1 = live ? start[Ic + 1] : s0;
    const int Ix = Ic / Ky, Iy = Ic % Ky;
    double d = 0.0, c[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int a = s0 + q; a < s1; a += RL) {
        const int i = list[a];
        d += d64[i];
        const int dg = deg[i];
        for (int k = 0; k < dg; k++) {
            const size_t e = (size_t)k * n + i;
            const int J = agg[ecol[e]];
            if (J == Ic) continue;
            const int dx = fold(J / Ky - Ix, Kx, xper), dy = fold(J % Ky - Iy, Ky, yper);
            if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || (dx == 0 && dy == 0)) continue;
            c[slot_of(dx, dy)] += ev[e];
        }
    }
    d = sum_lanes(d);
#pragma unroll
    for (int k = 0; k < 8; k++) c[k] = sum_lanes(c[k]);
    if (!live || q != 0) return;
    if (s1 == s0) d = 1.0;  // an empty cell is a decoupled identity row
    double sum = d;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        cout[(size_t)k * na + I] = (float)c[k];
        sum += c[k];
    }
    dout[I] = (float)d;
    dinv[I] = sum > 0.0 ? (float)(1.0 / sum) : 1.0f;
}

// level l+1 from level l: CF x CF blocks of cells
__global__ __launch_bounds__(B) void k_coarsen(int Kxc, int Kyc, int Kxf, int Kyf, int xper, int yper,
                                               const float *__restrict__ df, const float *__restrict__ cf,
                                               float *__restrict__ dc, float *__restrict__ cc,
                                               float *__restrict__ dinv)
{
    const int P = blockIdx.x * B + threadIdx.x;
    const int nc = Kxc * Kyc, nf = Kxf * Kyf;
    if (P >= nc) return;
    const int PX = P / Kyc, PY = P % Kyc;
    double d = 0.0, c[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const int cx1 = std::min(CF * PX + CF, Kxf), cy1 = std::min(CF * PY + CF, Kyf);
    for (int cx = CF * PX; cx < cx1; cx++)
        for (int cy = CF * PY; cy < cy1; cy++) {
            const int f = cx * Kyf + cy;
            d += df[f];
            for (int k = 0; k < 8; k++) {
                const float ck = cf[(size_t)k * nf + f];
                if (ck == 0.0f) continue;
                int ox, oy;
                offset_of(k, ox, oy);
                bool okx, oky;
                const int nx = wrap(cx + ox, Kxf, xper, okx), ny = wrap(cy + oy, Kyf, yper, oky);
                if (!okx || !oky) continue;
                const int dx = fold(nx / CF - PX, Kxc, xper), dy = fold(ny / CF - PY, Kyc, yper);
                if (dx == 0 && dy == 0) continue;
                c[slot_of(dx, dy)] += ck;
            }
        }
    double sum = d;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        cc[(size_t)k * nc + P] = (float)c[k];
        sum += c[k];
    }
    dc[P] = (float)d;
    dinv[P] = sum > 0.0 ? (float)(1.0 / sum) : 1.0f;
}

// the coarsest level as a dense FP64 matrix (plus sigma/nc everywhere for a singular system, which
// makes it definite without changing its action on mean-free vectors), inverted in place in LDS by
// Gauss-Jordan in one workgroup (an SPD matrix needs no pivoting); the inverse is stored
// column-major in FP32.  In LDS the rows have the fixed stride DM, so that an entry's row and column
// are a shift and a mask of its index, and the 1024 lanes take DM * DM / 1024 entries each.
constexpr int DM = LV_AMG_DENSE_MAX, DTB = 1024;
static_assert(DM == 64 && (DM * DM) % DTB == 0, "dense level: 64 x 64 entries over the workgroup");
__global__ __launch_bounds__(DTB) void k_dense_inverse(int Kx, int Ky, int xper, int yper, const float *__restrict__ d,
                                                       const float *__restrict__ c, int singular,
                                                       float *__restrict__ inv)
{
    const int nc = Kx * Ky;
    __shared__ double M[DM * DM];
    __shared__ double colp[DM], rowdiag[DM];
    for (int t = threadIdx.x; t < DM * DM; t += DTB) M[t] = 0.0;
    __syncthreads();
    if (threadIdx.x < nc) {  // row I by lane I
        const int I = threadIdx.x, Ix = I / Ky, Iy = I % Ky;
        double diag = d[I];
        for (int k = 0; k < 8; k++) {
            const double ck = c[(size_t)k * nc + I];
            if (ck == 0.0) continue;
            int ox, oy;
            offset_of(k, ox, oy);
            bool okx, oky;
            const int jx = wrap(Ix + ox, Kx, xper, okx), jy = wrap(Iy + oy, Ky, yper, oky);
            if (!okx || !oky) continue;
            diag += ck;
            M[I * DM + jx * Ky + jy] -= ck;
        }
        M[I * DM + I] += diag;
        rowdiag[I] = diag;
    }
    __syncthreads();
    if (singular) {
        __shared__ double sig;
        if (threadIdx.x == 0) {
            double dsum = 0.0;
            for (int I = 0; I < nc; I++) dsum += rowdiag[I];
            sig = dsum / nc / nc;
        }
        __syncthreads();
        for (int t = threadIdx.x; t < DM * DM; t += DTB)
            if (t / DM < nc && t % DM < nc) M[t] += sig;
        __syncthreads();
    }
    // in place: after pivot p, row p holds row p of the partial inverse and column p the
    // eliminated multipliers
    for (int p = 0; p < nc; p++) {
        const double piv = M[p * DM + p];
        if (threadIdx.x < nc) colp[threadIdx.x] = M[threadIdx.x * DM + p];
        __syncthreads();
        if (threadIdx.x < nc) {
            const int j = threadIdx.x;
            M[p * DM + j] = (j == p ? 1.0 : M[p * DM + j]) / piv;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < DM * DM / DTB; q++) {
            const int t = threadIdx.x + q * DTB, i = t / DM, j = t % DM;
            if (i >= nc || j >= nc || i == p) continue;
            M[t] = (j == p ? 0.0 : M[t]) - colp[i] * M[p * DM + j];
        }
        __syncthreads();
    }
    for (int t = threadIdx.x; t < DM * DM; t += DTB) {
        const int i = t / DM, j = t % DM;
        if (i < nc && j < nc) inv[j * nc + i] = (float)M[t];
    }
}

// ---- fine level -----------------------------------------------------------------------------------
//
// The fine kernels read the operator through a row view (lv_ell.h): the operator's own ELL (FP32
// values, particle order) or the aggregate-order copy built at set-up (BF16 values, 16-bit column
// offsets), in which case every fine vector of the cycle is in the aggregate order too.

template <class V>
struct fine_ops {
    int n;
    V A;
    const float *diag, *dinv, *mval, *mdg;
    float scale, alpha;
};

// (A z)_i in the difference form with the first 8 slots unrolled and predicated
template <class V>
__device__ __forceinline__ float a_row(int i, const fine_ops<V> &F, const float *__restrict__ z)
{
    constexpr int U = 8;
    const int n = F.n;
    const float zi = z[i];
    float acc = F.diag[i] * zi;
    int c[U];
    float v[U], zj[U];
    const int d = lv_ell_head<U>(F.A, i, n, c, v);
#pragma unroll
    for (int k = 0; k < U; k++) zj[k] = z[c[k]];
#pragma unroll
    for (int k = 0; k < U; k++) acc += v[k] * (zi - zj[k]);
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        acc += F.A.value(e) * (zi - z[F.A.column(e, i, n)]);
    }
    return acc;
}

// (M r)_i of the learned preconditioner (on A's pattern, in the same order as the view), or D^-1 r
template <class V>
__device__ __forceinline__ float m_row(int i, const fine_ops<V> &F, const float *__restrict__ r)
{
    if (!F.mval) return F.dinv[i] * r[i];
    constexpr int U = 8;
    const int n = F.n;
    float acc = F.mdg[i] * r[i];
    int c[U];
    float v[U], rj[U];
    const int d = lv_ell_head_with<U>(F.A, F.mval, i, n, c, v);
#pragma unroll
    for (int k = 0; k < U; k++) rj[k] = r[c[k]];
#pragma unroll
    for (int k = 0; k < U; k++) acc += v[k] * rj[k];
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        acc += F.mval[e] * r[F.A.column(e, i, n)];
    }
    return acc;
}

// z = scale * M r
template <class V>
__global__ __launch_bounds__(B) void k_fine_pre(fine_ops<V> F, const float *__restrict__ r, float *__restrict__ z,
                                                const lv_cg_scalars *S)
{
    if (S && S->done) return;
    const int i = blockIdx.x * B + threadIdx.x;
    if (i >= F.n) return;
    z[i] = F.scale * m_row(i, F, r);
}

// t = r - A z
template <class V>
__global__ __launch_bounds__(B) void k_fine_resid(fine_ops<V> F, const float *__restrict__ r,
                                                  const float *__restrict__ z, float *__restrict__ t,
                                                  const lv_cg_scalars *S)
{
    if (S && S->done) return;
    const int i = blockIdx.x * B + threadIdx.x;
    if (i >= F.n) return;
    t[i] = r[i] - a_row(i, F, z);
}

// rc[I] = sum over the rows of cell I of t: RL lanes per cell read its (sorted) row list
// contiguously and reduce by a fixed shuffle tree; list null: the rows of cell I are
// start[I]..start[I+1]-1 themselves (aggregate order)
__global__ __launch_bounds__(B) void k_restrict1(int na, const int *__restrict__ start, const int *__restrict__ list,
                                                 const float *__restrict__ t, float *__restrict__ rc,
                                                 const lv_cg_scalars *S)
{
    if (S && S->done) return;
    const int tid = blockIdx.x * B + threadIdx.x;
    const int I = tid / RL, q = tid % RL;
    float s = 0.0f;
    if (I < na) {
        const int s1 = start[I + 1];
        if (list)
            for (int a = start[I] + q; a < s1; a += RL) s += t[list[a]];
        else
            for (int a = start[I] + q; a < s1; a += RL) s += t[a];
    }
    s = sum_lanes(s);
    if (q == 0 && I < na) rc[I] = s;
}

// Jacobi fine smoother, down, one row: z0 = w D^-1 r and t = r - A z0 (z0 of a neighbour is
// recomputed from its r); returns t, stores z0
template <class V>
__device__ __forceinline__ float down_row_j(const fine_ops<V> &F, int i, const float *__restrict__ r,
                                            float *__restrict__ z0)
{
    const int n = F.n;
    constexpr int U = 8;
    const float ri = r[i];
    const float zi = F.scale * F.dinv[i] * ri;
    float acc = F.diag[i] * zi;
    int c[U];
    float v[U];
    const int d = lv_ell_head<U>(F.A, i, n, c, v);
    float rj[U], dj[U];
#pragma unroll
    for (int k = 0; k < U; k++) {
        rj[k] = r[c[k]];
        dj[k] = F.dinv[c[k]];
    }
#pragma unroll
    for (int k = 0; k < U; k++) acc += v[k] * (zi - F.scale * dj[k] * rj[k]);
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        const int j = F.A.column(e, i, n);
        acc += F.A.value(e) * (zi - F.scale * F.dinv[j] * r[j]);
    }
    z0[i] = zi;
    return ri - acc;
}

template <class V>
__global__ __launch_bounds__(B) void k_fine_down_j(fine_ops<V> F, const float *__restrict__ r,
                                                   float *__restrict__ z0, float *__restrict__ t,
                                                   const lv_cg_scalars *S)
{
    if (S && S->done) return;
    const int i = blockIdx.x * B + threadIdx.x;
    if (i >= F.n) return;
    t[i] = down_row_j(F, i, r, z0);
}

// the convergence test of lv_cycle_head (k >= 0), every workgroup for itself and block 0 for the record; true
// when the solve has ended
__device__ __forceinline__ bool head_stops(const lv_cycle_head &H)
{
    double pp[1][LV_RED_PER], o[1];
    reduce_all_load<1>(H.part, H.nb, pp);
    const int dn = H.S->done;
    const double thr2 = H.S->thr2;
    reduce_all_pin<1>(pp);
    asm volatile("" ::"s"(dn), "s"(thr2));
    if (dn) return true;
    reduce_all_sum<1>(H.part, H.nb, pp, o);
    const bool conv = o[0] <= thr2;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (conv) {
            H.S->rr = o[0];
            H.S->iters = H.k + 1;
            H.S->done = 1;
            if (H.prog) __hip_atomic_store(&H.prog->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (H.prog) __hip_atomic_store(&H.prog->seen, H.k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return conv;
}

// The down pass and the restriction in one kernel, for the aggregate order (the rows of level-1
// cell I are start[I]..start[I+1]-1): block b owns the cells whose first row lies in
// [FUSE_ROWS b, FUSE_ROWS (b+1)) (blk[b].x..blk[b+1].x-1), keeps their residuals t in LDS and sums
// each cell's as k_restrict1 does (RL lanes, the same order and shuffle tree, so rc is the same).
// A block holds at most FUSE_ROWS - 1 + (largest cell) rows; set-up checks that this fits FUSE_CAP.
// With z0 given each thread takes FUSE_RPT rows (FUSE_ROWS a little under FUSE_RPT B), whose loads
// are in flight together.
constexpr int FUSE_RPT = 2;
constexpr int FUSE_ROWS = FUSE_RPT * 256 - 32;
constexpr int FUSE_CAP = 2048;

// t = r - A z0 for one row when z0 = w D^-1 r is already stored (the same values down_row_j forms)
template <class V>
__device__ __forceinline__ float down_row_z0(const fine_ops<V> &F, int i, const float *__restrict__ r,
                                             const float *__restrict__ z0)
{
    const int n = F.n;
    constexpr int U = 8;
    const float zi = z0[i];
    float acc = F.diag[i] * zi;
    int c[U];
    float v[U], zj[U];
    const int d = lv_ell_head<U>(F.A, i, n, c, v);
#pragma unroll
    for (int k = 0; k < U; k++) zj[k] = z0[c[k]];
#pragma unroll
    for (int k = 0; k < U; k++) acc += v[k] * (zi - zj[k]);
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        acc += F.A.value(e) * (zi - z0[F.A.column(e, i, n)]);
    }
    return r[i] - acc;
}

// the sums of a block's cells c0..c1-1 over their rows' residuals tl (first row R0); sa, sb, dv: the row-list
// bounds and level-1 diagonals of its first FUSE_RPT trips
__device__ __forceinline__ void fused_restrict(const float *tl, int c0, int c1, int R0, const int *__restrict__ start,
                                               int na, const int (&sa)[FUSE_RPT], const int (&sb)[FUSE_RPT],
                                               const float (&dv)[FUSE_RPT], float *__restrict__ rc,
                                               const float *__restrict__ dinv1, float *__restrict__ z1)
{
    const int lanes = (c1 - c0) * RL;
    // one trip of B lanes, RL per cell; the trip count is uniform, so every lane shuffles
    auto restrict_trip = [&](int base, int a0, int s1, float di) {
        const int idx = base + (int)threadIdx.x;
        const int I = c0 + idx / RL, q = idx % RL;
        float s = 0.0f;
        if (idx < lanes)
            for (int a = a0 + q; a < s1; a += RL) s += tl[a - R0];
        s = sum_lanes(s);
        if (q == 0 && idx < lanes) {
            rc[I] = s;
            if (z1) z1[I] = OMEGA * di * s;
        }
    };
#pragma unroll
    for (int p = 0; p < FUSE_RPT; p++)
        if (p * B < lanes) restrict_trip(p * B, sa[p], sb[p], dv[p]);
    for (int base = FUSE_RPT * B; base < lanes; base += B) {
        const int I = c0 + (base + (int)threadIdx.x) / RL;
        const int Ic = I < na ? I : na - 1;
        restrict_trip(base, start[Ic], start[Ic + 1], dinv1[Ic]);
    }
}

// With z1 (level 1 above the tail), each cell's pre-smoothed z1 = w D1^-1 rc is stored too, as
// level 1's down pass would form it.
//
// blk[b] = (first cell, first row) of block b, so the block's bounds take one round trip, with the
// done flag (S->done, or without a solve the zero pair blk[nbf + 1]).  The
// restriction's row-list bounds and level-1 diagonals for its first FUSE_RPT trips of B lanes (a
// block's cells have about as many lanes as rows) are loaded before the rows, not after the
// barrier: a block's life is a chain of dependent round trips, and the blocks on a CU take several
// turns.  A lane past the block's cells loads cell na - 1's and drops them; dinv1 (level 1's
// diagonal) is read whether or not z1 is stored.
// HEAD: first what the caller left to the cycle (lv_cycle_head), with the done flag; the workgroups all come
// to the same verdict, and block 0 records it.
template <class V, bool Z0, bool HEAD>
__global__ __launch_bounds__(B) void k_fine_down_jr(fine_ops<V> F, const float *__restrict__ r,
                                                    float *__restrict__ z0, const int *__restrict__ start,
                                                    const int2 *__restrict__ blk, int na, float *__restrict__ rc,
                                                    const float *__restrict__ dinv1, float *__restrict__ z1,
                                                    const int *__restrict__ done, lv_cycle_head H)
{
    __shared__ float tl[FUSE_CAP];
    const int b = lv_xcd_block(blockIdx.x, gridDim.x);
    const int2 p0 = blk[b], p1 = blk[b + 1];
    if constexpr (HEAD) {
        if (H.k < 0) {
            const int skip = H.dev && H.S->skip;
            if (blockIdx.x == 0) {
                double o[2];
                reduce_all<2>(H.part, H.nb, o);
                if (threadIdx.x == 0) {
                    H.S->thr2 = (H.dev ? H.S->itol2 : H.inner_tol2) * o[1];
                    H.S->iters = 0;
                    H.S->done = skip ? 1 : 0;
                }
            }
            if (skip) return;
        } else {
            // (the bounds in the same round trip as the head's loads)
            asm volatile("" ::"s"(p0.x), "s"(p0.y), "s"(p1.x), "s"(p1.y));
            if (head_stops(H)) return;
        }
    } else {
        const int dn = *done;
        // the bounds and the flag in one round trip: without this the bounds' loads sink below the test
        asm volatile("" ::"s"(p0.x), "s"(p0.y), "s"(p1.x), "s"(p1.y), "s"(dn));
        if (dn) return;
    }
    const int c0 = p0.x, c1 = p1.x, R0 = p0.y, R1 = p1.y;
    int sa[FUSE_RPT], sb[FUSE_RPT];
    float dv[FUSE_RPT];
#pragma unroll
    for (int p = 0; p < FUSE_RPT; p++) {
        const int I = c0 + (p * B + (int)threadIdx.x) / RL;
        const int Ic = I < na ? I : na - 1;
        sa[p] = start[Ic];
        sb[p] = start[Ic + 1];
        dv[p] = dinv1[Ic];
    }
    if constexpr (Z0) {
        // rows i0 + q B; all but the first are clamped into the block's rows so that every row's
        // loads are issued without a branch (a clamped duplicate is computed and dropped)
        for (int i0 = R0 + (int)threadIdx.x; i0 < R1; i0 += FUSE_RPT * B) {
            float t[FUSE_RPT];
#pragma unroll
            for (int q = 0; q < FUSE_RPT; q++) {
                const int i = i0 + q * B;
                t[q] = down_row_z0(F, i < R1 ? i : R1 - 1, r, z0);
            }
#pragma unroll
            for (int q = 0; q < FUSE_RPT; q++)
                if (i0 + q * B < R1) tl[i0 + q * B - R0] = t[q];
        }
    } else {
        for (int i = R0 + (int)threadIdx.x; i < R1; i += B) tl[i - R0] = down_row_j(F, i, r, z0);
    }
    __syncthreads();
    fused_restrict(tl, c0, c1, R0, start, na, sa, sb, dv, rc, dinv1, z1);
}

// k_fine_down_jr with the CG iteration's update in front of it (lv_cycle_update): every row's r - alpha q, and its
// neighbours' again for their z0, which k_cg_u's pass over the rows would have stored; the same values
// bit for bit.  One launch for two where launches bound the iteration (UPDATE_MAX).
template <class V>
__global__ __launch_bounds__(B) void k_fine_down_u(fine_ops<V> F, lv_cycle_update U, float *__restrict__ z0,
                                                   const int *__restrict__ start, const int2 *__restrict__ blk,
                                                   int na, float *__restrict__ rc, const float *__restrict__ dinv1,
                                                   float *__restrict__ z1)
{
    __shared__ float tl[FUSE_CAP];
    const int b = lv_xcd_block(blockIdx.x, gridDim.x);
    const int2 p0 = blk[b], p1 = blk[b + 1];
    double pp[1][LV_RED_PER], pq[1];
    reduce_all_load<1>(U.Ppq, U.nb, pp);
    const int dn = U.S->done;
    const double rzn = U.S->rz[U.par ^ 1];
    reduce_all_pin<1>(pp);
    asm volatile("" ::"s"(p0.x), "s"(p0.y), "s"(p1.x), "s"(p1.y), "s"(dn), "s"(rzn));
    if (dn) return;
    const int c0 = p0.x, c1 = p1.x, R0 = p0.y, R1 = p1.y;
    int sa[FUSE_RPT], sb[FUSE_RPT];
    float dv[FUSE_RPT];
#pragma unroll
    for (int p = 0; p < FUSE_RPT; p++) {
        const int I = c0 + (p * B + (int)threadIdx.x) / RL;
        const int Ic = I < na ? I : na - 1;
        sa[p] = start[Ic];
        sb[p] = start[Ic + 1];
        dv[p] = dinv1[Ic];
    }
    reduce_all_sum<1>(U.Ppq, U.nb, pp, pq);
    const double alpha = rzn / pq[0];
    const float a = (float)alpha;
    const int n = F.n;
    constexpr int W = 8;
    double rr = 0.0;
    for (int i0 = R0 + (int)threadIdx.x; i0 < R1; i0 += FUSE_RPT * B) {
        // (all rows' loads before the sums; a clamped duplicate is computed and dropped)
        int c[FUSE_RPT][W], d[FUSE_RPT];
        float v[FUSE_RPT][W], rj[FUSE_RPT][W], qj[FUSE_RPT][W], dj[FUSE_RPT][W];
        float ri[FUSE_RPT], qi[FUSE_RPT], di[FUSE_RPT], dg[FUSE_RPT], xi[FUSE_RPT], pi[FUSE_RPT];
#pragma unroll
        for (int h = 0; h < FUSE_RPT; h++) {
            const int i = i0 + h * B < R1 ? i0 + h * B : R1 - 1;
            ri[h] = U.r[i];
            qi[h] = U.q[i];
            di[h] = F.dinv[i];
            dg[h] = F.diag[i];
            xi[h] = U.x[i];
            pi[h] = U.p[i];
            d[h] = lv_ell_head<W>(F.A, i, n, c[h], v[h]);
        }
#pragma unroll
        for (int h = 0; h < FUSE_RPT; h++)
#pragma unroll
            for (int k = 0; k < W; k++) {
                rj[h][k] = U.r[c[h][k]];
                qj[h][k] = U.q[c[h][k]];
                dj[h][k] = F.dinv[c[h][k]];
            }
#pragma unroll
        for (int h = 0; h < FUSE_RPT; h++) {
            const int i = i0 + h * B;
            if (i >= R1) continue;
            const float rn = ri[h] - a * qi[h];
            const float zi = F.scale * di[h] * rn;
            float acc = dg[h] * zi;
#pragma unroll
            for (int k = 0; k < W; k++) acc += v[h][k] * (zi - F.scale * dj[h][k] * (rj[h][k] - a * qj[h][k]));
            for (int k = W; k < d[h]; k++) {
                const size_t e = (size_t)k * n + i;
                const int j = F.A.column(e, i, n);
                acc += F.A.value(e) * (zi - F.scale * F.dinv[j] * (U.r[j] - a * U.q[j]));
            }
            tl[i - R0] = rn - acc;
            U.x[i] = xi[h] + a * pi[h];
            U.r_out[i] = rn;
            z0[i] = zi;
            rr += (double)rn * (double)rn;
        }
    }
    const double w[1] = {rr};
    block_partials<1>(w, U.Pur, gridDim.x);  // (its barrier also stands between tl's rows and their sums)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        U.S->pq = pq[0];
        U.S->alpha = alpha;
    }
    fused_restrict(tl, c0, c1, R0, start, na, sa, sb, dv, rc, dinv1, z1);
}

// blk[b] = (the first cell I with start[I] >= FUSE_ROWS b, start[I]) for b = 0..nbf-1,
// blk[nbf] = (na, n) (start[na] = n, nbf = n / FUSE_ROWS + 1) and blk[nbf + 1] = (0, 0), the done flag
// of a cycle outside a solve.  Thread I writes the b in
// (start[I-1], start[I]] / FUSE_ROWS; flag[1] is set when a cell has more than FUSE_CAP - FUSE_ROWS
// rows.
__global__ __launch_bounds__(B) void k_fuse_blocks(int na, int nbf, const int *__restrict__ start,
                                                   int2 *__restrict__ blk, int *__restrict__ flag)
{
    const int I = blockIdx.x * B + threadIdx.x;
    if (I > na) return;
    const int sI = start[I];
    const int lo = I == 0 ? 0 : start[I - 1] / FUSE_ROWS + 1;
    const int hi = sI / FUSE_ROWS;
    for (int b = lo; b <= hi && b < nbf; b++) blk[b] = make_int2(I, sI);
    if (I == na) {
        blk[nbf] = make_int2(na, sI);
        blk[nbf + 1] = make_int2(0, 0);
    }
    if (I < na && start[I + 1] - sI > FUSE_CAP - FUSE_ROWS) atomicOr(flag + 1, 1);
}

// up: z1 = z0 + alpha P ec and t = r - A z1 in one pass (z1 of a neighbour from its z0 and its
// cell's ec)
template <class V>
__device__ __forceinline__ float up_row(const fine_ops<V> &F, int i, const float *__restrict__ z0,
                                        const int *__restrict__ agg, const float *__restrict__ ec,
                                        const float *__restrict__ r, float &z1)
{
    constexpr int U = 8;
    const int n = F.n;
    // three dependent stages (columns; their z0 and cells; the cells' corrections), each issued for
    // all of the first U slots before the next
    int c[U];
    float v[U];
    const int d = lv_ell_head<U>(F.A, i, n, c, v);
    float zj[U];
    int aj[U];
#pragma unroll
    for (int k = 0; k < U; k++) {
        zj[k] = z0[c[k]];
        aj[k] = agg[c[k]];
    }
    z1 = z0[i] + F.alpha * ec[agg[i]];
    float acc = F.diag[i] * z1;
#pragma unroll
    for (int k = 0; k < U; k++) acc += v[k] * (z1 - (zj[k] + F.alpha * ec[aj[k]]));
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        const int j = F.A.column(e, i, n);
        acc += F.A.value(e) * (z1 - (z0[j] + F.alpha * ec[agg[j]]));
    }
    return r[i] - acc;
}

// learned smoother, up: z = z1 and t = r - A z1 (the post-smoothing follows in k_fine_post)
template <class V>
__global__ __launch_bounds__(B) void k_fine_up(fine_ops<V> F, const float *__restrict__ r,
                                               const float *__restrict__ z0, const int *__restrict__ agg,
                                               const float *__restrict__ ec, float *__restrict__ z,
                                               float *__restrict__ t, const lv_cg_scalars *S)
{
    if (S && S->done) return;
    const int i = blockIdx.x * B + threadIdx.x;
    if (i >= F.n) return;
    float z1;
    const float ti = up_row(F, i, z0, agg, ec, r, z1);
    z[i] = z1;
    t[i] = ti;
}

// prolongation in place: z0 += alpha ec[cell of the row], four rows per thread with 16-byte loads
// and stores of agg and z0 (both start 256-byte aligned); the last thread takes the n % 4 rows
constexpr int PROLONG_RPT = 4;
__global__ __launch_bounds__(B) void k_prolong1(int n, const int *__restrict__ agg, const float *__restrict__ ec,
                                                float alpha, float *__restrict__ z0, const lv_cg_scalars *S)
{
    typedef int i4 __attribute__((ext_vector_type(4)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    if (S && S->done) return;
    const int i = PROLONG_RPT * (blockIdx.x * B + threadIdx.x);
    if (i + 3 < n) {
        const i4 a = *reinterpret_cast<const i4 *>(agg + i);
        f4 z = *reinterpret_cast<const f4 *>(z0 + i);
        z.x += alpha * ec[a.x];
        z.y += alpha * ec[a.y];
        z.z += alpha * ec[a.z];
        z.w += alpha * ec[a.w];
        *reinterpret_cast<f4 *>(z0 + i) = z;
    } else {
        for (int k = i; k < n; k++) z0[k] += alpha * ec[agg[k]];
    }
}

// Jacobi smoother, up (after k_prolong1): z = z1 + w D^-1 (r - A z1); partials r.z, r.r of the final z
template <class V>
__global__ __launch_bounds__(B) void k_fine_up_j(fine_ops<V> F, const float *__restrict__ r,
                                                 const float *__restrict__ z1, float *__restrict__ z,
                                                 double *__restrict__ Prr, const lv_cg_scalars *S)
{
    if (S && S->done) return;
    double v[2] = {0.0, 0.0};
    // (the compact overflow of lv_ell.h does not pay here: 49.4 against 48.5 us per launch at 2048^2)
    for (int i = lv_xcd_block(blockIdx.x, gridDim.x) * B + threadIdx.x; i < F.n; i += gridDim.x * B) {
        const float ti = r[i] - a_row(i, F, z1);
        const float zi = z1[i] + F.scale * F.dinv[i] * ti;
        z[i] = zi;
        const float ri = r[i];
        v[0] += (double)ri * (double)zi;
        v[1] += (double)ri * (double)ri;
    }
    if (Prr) block_partials<2>(v, Prr, gridDim.x);
}

// z += scale * M t; partials r.z, r.r of the final z (grid-stride over lv_nblocks(n) blocks)
template <class V>
__global__ __launch_bounds__(B) void k_fine_post(fine_ops<V> F, const float *__restrict__ r,
                                                 const float *__restrict__ t, float *__restrict__ z,
                                                 double *__restrict__ Prr, const lv_cg_scalars *S)
{
    if (S && S->done) return;
    double v[2] = {0.0, 0.0};
    for (int i = blockIdx.x * B + threadIdx.x; i < F.n; i += gridDim.x * B) {
        const float zi = z[i] + F.scale * m_row(i, F, t);
        z[i] = zi;
        const float ri = r[i];
        v[0] += (double)ri * (double)zi;
        v[1] += (double)ri * (double)ri;
    }
    if (Prr) block_partials<2>(v, Prr, gridDim.x);
}

// ---- coarse levels (3x3 stencil) ---------------------------------------------------------------

struct st_level {
    int Kx, Ky, xper, yper;
    const float *d, *c, *dinv;
    float alpha;  // factor on the correction prolongated into this level
};

// wrap(i, K, per) for i in [-1, K] (a cell index plus an offset of at most one): a compare and an
// add instead of two remainders
// (selects, not branches: a branch here splits the stencil kernels' loads into basic blocks that
// the compiler then waits between)
__device__ __forceinline__ int wrap_near(int i, int K, int per, bool &ok)
{
    const int w = i < 0 ? i + K : (i >= K ? i - K : i);
    ok = per || (i >= 0 && i < K);
    return per ? w : i;
}

// the 8 neighbour cells of (cx, cy) on level L and their couplings; a neighbour outside a
// non-periodic level gets coupling 0 and index f, so every load below is in bounds and all of them
// can be issued at once (the coupling slot is loaded whatever the neighbour, and then selected: a
// load under the condition would make the gathers wait for it).  With PJ, also each neighbour's
// parent on the next level (Kyc columns).
__device__ __forceinline__ void st_nbrs(const st_level &L, int cx, int cy, int f, float ck[8], int J[8],
                                        int *PJ = nullptr, int Kyc = 0)
{
    const int n = L.Kx * L.Ky;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        int ox, oy;
        offset_of(k, ox, oy);
        bool okx, oky;
        const int jx = wrap_near(cx + ox, L.Kx, L.xper, okx), jy = wrap_near(cy + oy, L.Ky, L.yper, oky);
        const bool ok = okx && oky;
        J[k] = ok ? jx * L.Ky + jy : f;
        const float c = L.c[(size_t)k * n + f];
        ck[k] = ok ? c : 0.0f;
        if (PJ) PJ[k] = ok ? (jx / CF) * Kyc + jy / CF : (cx / CF) * Kyc + cy / CF;
    }
}

// down, one lane: child q of parent P (CF2 lanes per parent): z_f = w D^-1 r_f and the child's
// residual t_f = r_f - (A z)_f, with the neighbours' z recomputed from their r (0 outside the level)
// (ZGIVEN: z = w D^-1 r of the level is already stored, the same values, and only gathered)
template <bool ZGIVEN = false>
__device__ __forceinline__ float st_down_lane(const st_level &L, int Kyc, int nc, int P, int q,
                                              const float *__restrict__ r, float *__restrict__ z)
{
    if (P >= nc) return 0.0f;
    const int Px = P / Kyc;
    const int cx = CF * Px + q / CF, cy = CF * (P - Px * Kyc) + q % CF;
    if (cx >= L.Kx || cy >= L.Ky) return 0.0f;
    const int f = cx * L.Ky + cy;
    float ck[8], zj[8];
    int J[8];
    st_nbrs(L, cx, cy, f, ck, J);
    const float rf = r[f];
    float zf;
    if (ZGIVEN) {
#pragma unroll
        for (int k = 0; k < 8; k++) zj[k] = z[J[k]];
        zf = z[f];
    } else {
        float rj[8], dj[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            rj[k] = r[J[k]];
            dj[k] = L.dinv[J[k]];
        }
#pragma unroll
        for (int k = 0; k < 8; k++) zj[k] = OMEGA * dj[k] * rj[k];
        zf = OMEGA * L.dinv[f] * rf;
    }
    float acc = L.d[f] * zf;
#pragma unroll
    for (int k = 0; k < 8; k++) acc += ck[k] * (zf - zj[k]);
    if (!ZGIVEN) z[f] = zf;
    return rf - acc;
}

// the children's residuals of CF2 consecutive lanes summed by a fixed shuffle tree (every lane of
// the wave takes part)
__device__ __forceinline__ float sum_children(float t)
{
#pragma unroll
    for (int m = 1; m < CF2; m <<= 1) t += __shfl_xor(t, m);
    return t;
}

// up, one cell: z1 = z + ec[parent] (neighbours' z1 recomputed), t = r - A z1, out = z1 + w D^-1 t
__device__ __forceinline__ float st_up_cell(const st_level &L, int Kyc, int f, const float *__restrict__ r,
                                            const float *__restrict__ z, const float *__restrict__ ec,
                                            float *__restrict__ out)
{
    const int cx = f / L.Ky, cy = f - cx * L.Ky;
    float ck[8], zj[8], ej[8];
    int J[8], PJ[8];
    st_nbrs(L, cx, cy, f, ck, J, PJ, Kyc);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        zj[k] = z[J[k]];
        ej[k] = L.alpha * ec[PJ[k]];
    }
    const float z1 = z[f] + L.alpha * ec[(cx / CF) * Kyc + cy / CF];
    float acc = L.d[f] * z1;
#pragma unroll
    for (int k = 0; k < 8; k++) acc += ck[k] * (z1 - (zj[k] + ej[k]));
    const float v = z1 + OMEGA * L.dinv[f] * (r[f] - acc);
    out[f] = v;
    return v;
}

// W-cycle, after the first visit of level L returned t: acc = t and r = r - A t (the right-hand
// side of the second visit)
__device__ __forceinline__ void st_wsave_cell(const st_level &L, int f, float *__restrict__ r,
                                              const float *__restrict__ t, float *__restrict__ acc)
{
    const int cx = f / L.Ky, cy = f - cx * L.Ky;
    float ck[8], tj[8];
    int J[8];
    st_nbrs(L, cx, cy, f, ck, J);
#pragma unroll
    for (int k = 0; k < 8; k++) tj[k] = t[J[k]];
    const float tf = t[f];
    float a = L.d[f] * tf;
#pragma unroll
    for (int k = 0; k < 8; k++) a += ck[k] * (tf - tj[k]);
    acc[f] = tf;
    r[f] -= a;
}

// down on level L: pre-smoothed z of L (given, or stored here) and the right-hand side rc of the
// next level
// (HEAD: after the down pass that made a CG update, with its convergence test)
template <bool ZGIVEN, bool HEAD>
__global__ __launch_bounds__(B) void k_st_down(st_level L, int Kyc, int nc, const float *__restrict__ r,
                                               float *__restrict__ z, float *__restrict__ rc, const lv_cg_scalars *S,
                                               lv_cycle_head H)
{
    if (HEAD) {
        if (head_stops(H)) return;
    } else if (S && S->done) {
        return;
    }
    // (workgroups in the XCD-aware order: the parent rows above and below a workgroup's, whose
    // children it gathers, are mostly on its own XCD)
    const int tid = lv_xcd_block(blockIdx.x, gridDim.x) * B + threadIdx.x;
    const int P = tid / CF2, q = tid % CF2;
    const float t = sum_children(st_down_lane<ZGIVEN>(L, Kyc, nc, P, q, r, z));
    if (q == 0 && P < nc) rc[P] = t;
}

// up on level L: the final correction out of L from the next level's correction ec.  PROLONG (level
// 1 in the aggregate order, whose cell f owns rows start[f]..start[f+1]-1): also the prolongation
// z0 += alpha0 out[f] of those rows, as k_prolong1 forms it
template <bool PROLONG>
__global__ __launch_bounds__(B) void k_st_up(st_level L, int Kyc, const float *__restrict__ r,
                                             const float *__restrict__ z, const float *__restrict__ ec,
                                             float *__restrict__ out, const lv_cg_scalars *S,
                                             const int *__restrict__ start, float alpha0, float *__restrict__ z0)
{
    if (S && S->done) return;
    const int f = lv_xcd_block(blockIdx.x, gridDim.x) * B + threadIdx.x;  // (as k_st_down)
    if (f >= L.Kx * L.Ky) return;
    // the prolongation's rows: bounds first, then the first PH rows' z0 loaded together (a row past
    // the cell's reloads its last, or row 0 for an empty cell at the end), so that the cell's rows
    // take one round trip after the stencil's loads instead of one each
    constexpr int PH = 4;
    int b0 = 0, e = 0;
    float zz[PH];
    if (PROLONG) {
        b0 = start[f];
        e = start[f + 1];
        const int last = e > 0 ? e - 1 : 0;
#pragma unroll
        for (int h = 0; h < PH; h++) zz[h] = z0[b0 + h < e ? b0 + h : last];
    }
    const float v = st_up_cell(L, Kyc, f, r, z, ec, out);
    if (PROLONG) {
        // (the rows' values in registers before the stores' branches, which would otherwise take
        // the first row's load with them)
        asm volatile("" : "+v"(zz[0]), "+v"(zz[1]), "+v"(zz[2]), "+v"(zz[3]));
        const float a = alpha0 * v;
#pragma unroll
        for (int h = 0; h < PH; h++)
            if (b0 + h < e) z0[b0 + h] = zz[h] + a;
        for (int i = b0 + PH; i < e; i++) z0[i] += a;
    }
}

// ---- two coarse levels in one kernel ------------------------------------------------------------
//
// Levels l and l+1 above the tail run their down passes as one kernel and their up passes as another.
// A block owns a tile of cells and recomputes in LDS what its stencils read from the cells around the
// tile (a halo), with the expressions and the order of st_down_lane, sum_children and st_up_cell, so
// every value is bit for bit the one the one-level kernels give.  Cells are addressed by unwrapped
// coordinates; the last cell of an odd periodic axis is its parent's only child, so that beyond the
// wrap children and parents lie one cell nearer than twice and half (child_near, parent_near; ODD: a
// periodic axis of level l or l+1 is odd.  The arithmetic costs a pair 1 us, so even ones go without).  Level
// l is at least PAIR_MIN_K cells wide on both axes, so the unwrapped coordinates of every region stay
// within one width of the level and one conditional add or subtract wraps them.  The down tile is small
// (PD = 4: 4 lanes of work per cell of level l+2) so that the small levels spread over many workgroups;
// 8 x 8 tiles left one wavefront per SIMD working through six halo cells a lane, no faster than two
// one-level kernels.

constexpr int PD = 4;   // down: a block owns PD x PD cells of level l+2
constexpr int PU = 16;  // up: a block owns PU x PU cells of level l, one a lane
constexpr int PAIR_MIN_K = 24;
static_assert(PAIR_MIN_K >= 4 * PD + 8 && PAIR_MIN_K >= PU + 8, "every region within one width of its level");

struct st_pair {
    st_level L0, L1;  // levels l and l+1
    int Kx2, Ky2;     // level l+2
};

// cell (x, y) of a Kx x Ky level, unwrapped within one width: its index, or 0 with ok false outside a
// non-periodic axis (so that every load below has a valid address and none waits behind a branch)
__device__ __forceinline__ int cell_of(int x, int y, int Kx, int Ky, int xper, int yper, bool &ok)
{
    bool okx, oky;
    x = wrap_near(x, Kx, xper, okx);
    y = wrap_near(y, Ky, yper, oky);
    ok = okx && oky;
    return ok ? x * Ky + y : 0;
}

// on an axis of K cells whose parents are Kc: the parent of cell x and the first child of parent X, all
// unwrapped within one width (outside a non-periodic axis: any nearby coordinate); and whether X has two children
template <bool ODD>
__device__ __forceinline__ int parent_near(int x, int K, int Kc, int per)
{
    if (!ODD) return x >> 1;
    const int d = per ? 2 * Kc - K : 0;
    return (x < 0 ? x - d : (x >= K ? x + d : x)) >> 1;
}
template <bool ODD>
__device__ __forceinline__ int child_near(int X, int K, int Kc, int per)
{
    if (!ODD) return 2 * X;
    const int d = per ? 2 * Kc - K : 0;
    return X < 0 ? 2 * X + d : (X >= Kc ? 2 * X - d : 2 * X);
}
template <bool ODD>
__device__ __forceinline__ bool two_children(int X, int K, int Kc, int per)
{
    return !ODD || !(per && (K & 1)) || !(X == Kc - 1 || X == -1);
}

// the couplings of cell f = (x, y) (unwrapped) of level L and the mask of its neighbours inside the
// level; a neighbour outside gets coupling 0 (st_nbrs)
__device__ __forceinline__ unsigned st_coefs(const st_level &L, int x, int y, int f, float ck[8])
{
    const int n = L.Kx * L.Ky;
    unsigned ok = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        int ox, oy;
        offset_of(k, ox, oy);
        const bool in = (L.xper || (x + ox >= 0 && x + ox < L.Kx)) && (L.yper || (y + oy >= 0 && y + oy < L.Ky));
        ok |= (unsigned)in << k;
        const float c = L.c[(size_t)k * n + f];
        ck[k] = in ? c : 0.0f;
    }
    return ok;
}

// the residual r - A z of one cell from the z of its 3 x 3 neighbourhood in an LDS region of row
// length SR (zc at offset 0), as st_down_lane forms it
template <int SR>
__device__ __forceinline__ float st_resid_lds(float rf, float d, const float ck[8], unsigned ok,
                                              const float *__restrict__ zc)
{
    const float zf = zc[0];
    float acc = d * zf;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        int ox, oy;
        offset_of(k, ox, oy);
        const float zj = ((ok >> k) & 1) ? zc[ox * SR + oy] : zf;
        acc += ck[k] * (zf - zj);
    }
    return rf - acc;
}

// down on levels l and l+1: the pre-smoothed z of both, the right-hand side r1 of level l+1 and r2
// of level l+2, as k_st_down<false> on level l and then on level l+1.  Regions of a block (level,
// first cell relative to its tile's first cell, side): A (l, -3, 4PD+6) z and r, B (l, -2, 4PD+4)
// the residual, C (l+1, -1, 2PD+2) r and z, D (l+1, 0, 2PD) the residual.
template <bool ODD>
__global__ __launch_bounds__(B) void k_st_down2(st_pair Q, const float *__restrict__ r0, float *__restrict__ z0,
                                                float *__restrict__ r1, float *__restrict__ z1,
                                                float *__restrict__ r2, const lv_cg_scalars *S)
{
    constexpr int SA = 4 * PD + 6, SB = 4 * PD + 4, SC = 2 * PD + 2, SD = 2 * PD;
    constexpr int NA = SA * SA, NB = SB * SB, NC = SC * SC;
    constexpr int IA = (NA + B - 1) / B, IB = (NB + B - 1) / B, IC = (NC + B - 1) / B;
    static_assert(SD * SD <= B, "region D: at most one cell a lane");
    __shared__ float zA[NA], rA[NA], tB[NB], rC[NC], zC[NC], tD[SD * SD];
    if (S && S->done) return;
    const st_level &L0 = Q.L0, &L1 = Q.L1;
    const int qx = blockIdx.x * PD, qy = blockIdx.y * PD;  // the tile's first cell on level l+2
    const int ax = 4 * qx - 3, ay = 4 * qy - 3, cx = 2 * qx - 1, cy = 2 * qy - 1;
    const int tid = threadIdx.x;
    // every global load first, unconditionally (fA..: -1 outside the level or past the region)
    int fA[IA], fB[IB], fC[IC];
    float ra[IA], da[IA], dB[IB], cB[IB][8], dvC[IC], cD[8];
    unsigned okB[IB];
#pragma unroll
    for (int i = 0; i < IA; i++) {
        const int s = tid + i * B, sa = s < NA ? s : NA - 1;  // lanes past the region load a cell of it
        bool ok;
        const int f = cell_of(ax + sa / SA, ay + sa % SA, L0.Kx, L0.Ky, L0.xper, L0.yper, ok);
        ra[i] = r0[f];
        da[i] = L0.dinv[f];
        fA[i] = (ok && s < NA) ? f : -1;
    }
#pragma unroll
    for (int i = 0; i < IB; i++) {
        const int s = tid + i * B, sb = s < NB ? s : NB - 1, x = ax + 1 + sb / SB, y = ay + 1 + sb % SB;
        bool ok;
        const int f = cell_of(x, y, L0.Kx, L0.Ky, L0.xper, L0.yper, ok);
        dB[i] = L0.d[f];
        okB[i] = st_coefs(L0, x, y, f, cB[i]);
        fB[i] = (ok && s < NB) ? f : -1;
    }
#pragma unroll
    for (int i = 0; i < IC; i++) {
        const int s = tid + i * B, sc = s < NC ? s : NC - 1;
        bool ok;
        const int f = cell_of(cx + sc / SC, cy + sc % SC, L1.Kx, L1.Ky, L1.xper, L1.yper, ok);
        dvC[i] = L1.dinv[f];
        fC[i] = (ok && s < NC) ? f : -1;
    }
    const int td = tid < SD * SD ? tid : 0, dxs = td / SD, dys = td % SD, Xd = cx + 1 + dxs, Yd = cy + 1 + dys;
    bool okd;
    int fD = cell_of(Xd, Yd, L1.Kx, L1.Ky, L1.xper, L1.yper, okd);
    const float dD = L1.d[fD];
    const unsigned okD = st_coefs(L1, Xd, Yd, fD, cD);
    fD = (okd && tid < SD * SD && Xd < L1.Kx && Yd < L1.Ky) ? fD : -1;  // (none beyond the wrap)
    // A: z = w D^-1 r of level l
#pragma unroll
    for (int i = 0; i < IA; i++) {
        const int s = tid + i * B;
        if (s < NA) {
            zA[s] = fA[i] >= 0 ? OMEGA * da[i] * ra[i] : 0.0f;
            rA[s] = fA[i] >= 0 ? ra[i] : 0.0f;
        }
    }
    __syncthreads();
    // B: the residual of level l; the tile's own cells store their z
#pragma unroll
    for (int i = 0; i < IB; i++) {
        const int s = tid + i * B;
        if (s >= NB) continue;
        const int sx = s / SB, sy = s % SB;
        if (fB[i] < 0) {
            tB[s] = 0.0f;
            continue;
        }
        const int a = (sx + 1) * SA + sy + 1;
        tB[s] = st_resid_lds<SA>(rA[a], dB[i], cB[i], okB[i], zA + a);
        const int x = ax + 1 + sx, y = ay + 1 + sy;
        if (sx >= 2 && sx < 4 * PD + 2 && sy >= 2 && sy < 4 * PD + 2 && x < L0.Kx && y < L0.Ky) z0[fB[i]] = zA[a];
    }
    __syncthreads();
    // C: r of level l+1, the sum of its children's residuals in sum_children's order, and its z
#pragma unroll
    for (int i = 0; i < IC; i++) {
        const int s = tid + i * B;
        if (s >= NC) continue;
        const int sx = s / SC, sy = s % SC;
        if (fC[i] < 0) {
            rC[s] = 0.0f;
            zC[s] = 0.0f;
            continue;
        }
        const int X = cx + sx, Y = cy + sy;
        const int b = (child_near<ODD>(X, L0.Kx, L1.Kx, L0.xper) - (ax + 1)) * SB +
                      (child_near<ODD>(Y, L0.Ky, L1.Ky, L0.yper) - (ay + 1));
        const bool x2 = two_children<ODD>(X, L0.Kx, L1.Kx, L0.xper), y2 = two_children<ODD>(Y, L0.Ky, L1.Ky, L0.yper);
        const float r = (tB[b] + (y2 ? tB[b + 1] : 0.0f)) +
                        ((x2 ? tB[b + SB] : 0.0f) + (x2 && y2 ? tB[b + SB + 1] : 0.0f));
        rC[s] = r;
        zC[s] = OMEGA * dvC[i] * r;
        if (sx >= 1 && sx < 2 * PD + 1 && sy >= 1 && sy < 2 * PD + 1 && X < L1.Kx && Y < L1.Ky) r1[fC[i]] = r;
    }
    __syncthreads();
    // D: the residual of level l+1 on the tile's children; they store their z
    if (tid < SD * SD) {
        const int c = (dxs + 1) * SC + dys + 1;
        tD[tid] = fD >= 0 ? st_resid_lds<SC>(rC[c], dD, cD, okD, zC + c) : 0.0f;
        if (fD >= 0) z1[fD] = zC[c];
    }
    __syncthreads();
    // E: r of level l+2
    if (tid < PD * PD) {
        const int sx = tid / PD, sy = tid % PD, X = qx + sx, Y = qy + sy;
        if (X < Q.Kx2 && Y < Q.Ky2) {
            const int b = 2 * sx * SD + 2 * sy;
            r2[X * Q.Ky2 + Y] = (tD[b] + tD[b + 1]) + (tD[b + SD] + tD[b + SD + 1]);
        }
    }
}

// up on levels l+1 and l: the final correction t0 of level l from the final correction t2 of level
// l+2, as k_st_up<false> on level l+1 and then on level l (level l+1's own correction stays in LDS).
// Regions of a block (level, first cell relative to the tile's, side): Z0 (l, -1, PU+2) z, V (l+1,
// -1, PU/2+2) the correction, Z1 (l+1, -2, PU/2+4) z, E t2 of level l+2 (-1, PU/4+2; odd: -2, PU/4+4).
template <bool ODD>
__global__ __launch_bounds__(B) void k_st_up2(st_pair Q, const float *__restrict__ r0, const float *__restrict__ z0,
                                              const float *__restrict__ r1, const float *__restrict__ z1,
                                              const float *__restrict__ t2, float *__restrict__ t0,
                                              const lv_cg_scalars *S)
{
    constexpr int SZ0 = PU + 2, SV = PU / 2 + 2, SZ1 = PU / 2 + 4, EH = ODD ? 2 : 1,
                  SE = PU / 4 + 2 * EH;
    constexpr int NZ0 = SZ0 * SZ0, IZ0 = (NZ0 + B - 1) / B;
    static_assert(PU * PU == B && SZ1 * SZ1 <= B && SV * SV <= B, "one cell of each region a lane");
    __shared__ float zl[NZ0], vm[SV * SV], zm[SZ1 * SZ1], e2[SE * SE];
    if (S && S->done) return;
    const st_level &L0 = Q.L0, &L1 = Q.L1;
    const int x0 = blockIdx.x * PU, y0 = blockIdx.y * PU;  // the tile's first cell on level l
    const int vx = x0 / 2 - 1, vy = y0 / 2 - 1, ex = x0 / 4 - EH, ey = y0 / 4 - EH;
    const int tid = threadIdx.x;
    // every global load first, unconditionally (from cell 0 outside a level or a region)
    float zv[IZ0];
#pragma unroll
    for (int i = 0; i < IZ0; i++) {
        const int s = tid + i * B, sz = s < NZ0 ? s : NZ0 - 1;  // lanes past the region load a cell of it
        bool ok;
        const int f = cell_of(x0 - 1 + sz / SZ0, y0 - 1 + sz % SZ0, L0.Kx, L0.Ky, L0.xper, L0.yper, ok);
        const float v = z0[f];
        zv[i] = ok ? v : 0.0f;
    }
    bool okm, oke;
    const int tm = tid < SZ1 * SZ1 ? tid : 0, te = tid < SE * SE ? tid : 0;
    const int fm = cell_of(vx - 1 + tm / SZ1, vy - 1 + tm % SZ1, L1.Kx, L1.Ky, L1.xper, L1.yper, okm);
    const int fe = cell_of(ex + te / SE, ey + te % SE, Q.Kx2, Q.Ky2, L1.xper, L1.yper, oke);
    const float zm_ = z1[fm], ev_ = t2[fe];
    const float zmv = okm ? zm_ : 0.0f, ev = oke ? ev_ : 0.0f;
    const int tv = tid < SV * SV ? tid : 0, vxs = tv / SV, vys = tv % SV, Xv = vx + vxs, Yv = vy + vys;
    bool okv;
    int fV = cell_of(Xv, Yv, L1.Kx, L1.Ky, L1.xper, L1.yper, okv);
    float cV[8];
    const float dV = L1.d[fV], dvV = L1.dinv[fV], rV = r1[fV];
    const unsigned okV = st_coefs(L1, Xv, Yv, fV, cV);
    fV = (okv && tid < SV * SV) ? fV : -1;
    const int txs = tid / PU, tys = tid % PU, x = x0 + txs, y = y0 + tys;
    const bool own = x < L0.Kx && y < L0.Ky;
    const int f = own ? x * L0.Ky + y : 0;
    float cT[8];
    const float dT = L0.d[f], dvT = L0.dinv[f], rT = r0[f];
    const unsigned okT = st_coefs(L0, x, y, f, cT);
#pragma unroll
    for (int i = 0; i < IZ0; i++)
        if (tid + i * B < NZ0) zl[tid + i * B] = zv[i];
    if (tid < SZ1 * SZ1) zm[tid] = zmv;
    if (tid < SE * SE) e2[tid] = ev;
    __syncthreads();
    // V: level l+1's final correction (st_up_cell with ec = t2)
    if (tid < SV * SV) {
        float v = 0.0f;
        if (fV >= 0) {
            const float a = L1.alpha;
            const int zc = (vxs + 1) * SZ1 + vys + 1;
            auto pe_of = [&](int X, int Y) {
                return e2[(parent_near<ODD>(X, L1.Kx, Q.Kx2, L1.xper) - ex) * SE + parent_near<ODD>(Y, L1.Ky, Q.Ky2, L1.yper) - ey];
            };
            const float pe = pe_of(Xv, Yv);
            const float z1c = zm[zc] + a * pe;
            float acc = dV * z1c;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                int ox, oy;
                offset_of(k, ox, oy);
                const bool in = (okV >> k) & 1;
                const float zj = in ? zm[zc + ox * SZ1 + oy] : zm[zc];
                const float ej = a * (in ? pe_of(Xv + ox, Yv + oy) : pe);
                acc += cV[k] * (z1c - (zj + ej));
            }
            v = z1c + OMEGA * dvV * (rV - acc);
        }
        vm[tid] = v;
    }
    __syncthreads();
    // the tile: level l's final correction (st_up_cell with ec = level l+1's)
    if (own) {
        const float a = L0.alpha;
        const int zc = (txs + 1) * SZ0 + tys + 1;
        auto pv_of = [&](int X, int Y) {
            return vm[(parent_near<ODD>(X, L0.Kx, L1.Kx, L0.xper) - vx) * SV + parent_near<ODD>(Y, L0.Ky, L1.Ky, L0.yper) - vy];
        };
        const float pv = pv_of(x, y);
        const float z1c = zl[zc] + a * pv;
        float acc = dT * z1c;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            int ox, oy;
            offset_of(k, ox, oy);
            const bool in = (okT >> k) & 1;
            const float zj = in ? zl[zc + ox * SZ0 + oy] : zl[zc];
            const float ej = a * (in ? pv_of(x + ox, y + oy) : pv);
            acc += cT[k] * (z1c - (zj + ej));
        }
        t0[f] = z1c + OMEGA * dvT * (rT - acc);
    }
}

// The small levels of the cycle in one workgroup: a program of operations on levels first..last
// (last: the dense one), built at set-up for a V- or W-cycle, each operation followed by a barrier
// (the levels' vectors stay in global memory, which the barrier makes visible across the
// workgroup).  Reads the right-hand side of level first, writes its final correction.
constexpr int TB = 1024;
constexpr int TAIL_MAX = 1024;  // levels of at most this many cells run in the tail
// A singular system's cycle multiplies by the matrix of its first level of at most MAT_MAX cells: 26 MB, what
// the eight L2s hold, so that a small system's cycles find it there.  An iteration with the matrix and with the level's two
// stencil launches and the next level's matrix: 22.4 and 25.5 us at 33 x 33 cells, 22.1 and 25.7 at 45 x 45, 23.6
// and 25.7 at 50 x 50, 23.8 and 25.8 at 53 x 53, 26.6 and 25.5 at 56 x 56, 30.2 and 25.4 at 64 x 64, and the set-up
// 20 to 60 us more: the two cross just above the line.
constexpr int MAT_MAX = 2560;
// A nonsingular system, whose tail is visited once a cycle, starts it at its first level of at most LDS_MAX
// cells (33 x 33 cells: 11.0 us with them, 9.0 and two launches of 3.3 without).  An iteration at 132^2 to 144^2
// particles, 33 x 33 to 36 x 36 cells on level 2, takes 34.2 to 35.1 us with them and 37.1 to 38 without; as level 1 (66^2
// to 70^2 particles) 31 to 32 either way, since the down pass then makes no CG update.  The LDS would hold 38 x 38
// cells; the level above, 65 x 65 with its couplings in registers, cost 17 us more, so that one keeps its launches.
constexpr int LDS_MAX = 1280;
constexpr int LV_DESC = 16;  // ints of a level's descriptor (tail_descriptors)
constexpr int LV_CELL = 12;  // floats of a cell's constants in the LDS image: c[8], d, 1 / (d + sum c), two unused
enum tail_op { OP_DOWN = 0, OP_DENSE = 1, OP_UP = 2, OP_WSAVE = 3, OP_WADD = 4 };
constexpr int OP_SHIFT = 5;  // an operation is op << OP_SHIFT | level
static_assert(LV_AMG_MAXLEV < (1 << OP_SHIFT), "levels fit the operation code");
struct tail_levels {
    int first, last, xper, yper;
    int Kx[LV_AMG_MAXLEV + 1], Ky[LV_AMG_MAXLEV + 1];
    float alpha[LV_AMG_MAXLEV + 1];
    const float *d[LV_AMG_MAXLEV + 1], *c[LV_AMG_MAXLEV + 1], *dinv[LV_AMG_MAXLEV + 1];
    float *r[LV_AMG_MAXLEV + 1], *z[LV_AMG_MAXLEV + 1], *t[LV_AMG_MAXLEV + 1], *acc[LV_AMG_MAXLEV + 1];
};

// The tail levels in LDS, offsets in floats: a level's constants (LV_CELL floats a cell), then the dense
// inverse; then, zeroed and filled by the program, z and t with a halo of one cell around the level (its periodic
// neighbours, or zeros outside it), and r and the W-cycle's accumulator.  With the constants of a cell in three
// 16-byte reads and the neighbours at fixed offsets, an operation has next to no index arithmetic, which is what
// a single workgroup has to spend its instructions on otherwise (the same program with slot-major
// couplings, neighbour indices and the neighbours' z recomputed from r and D^-1: 10.1 us at 16 x 32 cells and
// 11.9 at 32 x 32, against 7.0 and 9.7).
constexpr int TAIL_LDS = 35 * 1024;
struct tail_layout {
    int k[LV_AMG_MAXLEV + 1], r[LV_AMG_MAXLEV + 1], z[LV_AMG_MAXLEV + 1], t[LV_AMG_MAXLEV + 1],
        acc[LV_AMG_MAXLEV + 1];
    int inv, coef, total;  // [0, coef): the constants, then the work vectors
};

// Columns of the W-visited tail's matrix (k_tail_lds<true>) where the levels do not fit the LDS: strips one cell
// wide, with halos three times their cells.  The program on arrays in global memory, a copy of them (stride floats)
// for each column, each operation followed by a barrier that makes its writes visible to the workgroup.  (Run
// in every cycle on the levels' own arrays it made a singular solve on 4000 x 4 particles 4.15 ms, with the matrix
// from here 0.74.)
__global__ __launch_bounds__(TB) void k_tail_columns(tail_levels T, const int *__restrict__ prog, int nprog,
                                                     const float *__restrict__ inv, int stride, float *__restrict__ mat,
                                                     int ld)
{
    const size_t at = (size_t)blockIdx.x * stride;
    auto R = [&](int l) { return T.r[l] + at; };
    auto Z = [&](int l) { return T.z[l] + at; };
    auto E = [&](int l) { return T.t[l] + at; };
    auto A = [&](int l) { return T.acc[l] + at; };
    const int n0 = T.Kx[T.first] * T.Ky[T.first];
    for (int f = threadIdx.x; f < n0; f += TB) R(T.first)[f] = f == (int)blockIdx.x ? 1.0f : 0.0f;
    __syncthreads();
    for (int pc = 0; pc < nprog; pc++) {
        const int code = prog[pc];
        const int op = code >> OP_SHIFT, l = code & ((1 << OP_SHIFT) - 1);
        const st_level L{T.Kx[l], T.Ky[l], T.xper, T.yper, T.d[l], T.c[l], T.dinv[l], T.alpha[l]};
        const int n = T.Kx[l] * T.Ky[l];
        if (op == OP_DOWN) {
            const int Kyc = T.Ky[l + 1], nc = T.Kx[l + 1] * T.Ky[l + 1];
            for (int base = 0; base < nc * CF2; base += TB) {  // uniform trip count: every lane shuffles
                const int tid = base + threadIdx.x;
                const int P = tid / CF2, q = tid % CF2;
                const float t = sum_children(st_down_lane(L, Kyc, nc, P, q, R(l), Z(l)));
                if (q == 0 && P < nc) R(l + 1)[P] = t;
            }
        } else if (op == OP_DENSE) {
            // t = inv r: 16 lanes per row (LV_AMG_DENSE_MAX * 16 == TB)
            const int i = threadIdx.x >> 4, q = threadIdx.x & 15;
            float acc = 0.0f;
            if (i < n)
                for (int j = q; j < n; j += 16) acc += inv[j * n + i] * R(l)[j];
            acc += __shfl_xor(acc, 1);
            acc += __shfl_xor(acc, 2);
            acc += __shfl_xor(acc, 4);
            acc += __shfl_xor(acc, 8);
            if (q == 0 && i < n) E(l)[i] = acc;
        } else if (op == OP_UP) {
            for (int f = threadIdx.x; f < n; f += TB) st_up_cell(L, T.Ky[l + 1], f, R(l), Z(l), E(l + 1), E(l));
        } else if (op == OP_WSAVE) {
            for (int f = threadIdx.x; f < n; f += TB) st_wsave_cell(L, f, R(l), E(l), A(l));
        } else {  // OP_WADD
            for (int f = threadIdx.x; f < n; f += TB) E(l)[f] += A(l)[f];
        }
        __syncthreads();
    }
    float *row = mat + (size_t)blockIdx.x * ld;
    for (int f = threadIdx.x; f < ld; f += TB) row[f] = f < n0 ? E(T.first)[f] : 0.0f;
}

// a / K with rK = 1 / K in FP32, for 0 <= a < 8192: (a + 1/2) / K is at least 1 / (2 K) from an integer, a
// relative 6e-5, and the product is off by 2e-7 at most
__device__ __forceinline__ int div_small(int a, float rK) { return (int)(((float)a + 0.5f) * rK); }

// a level in LDS
struct tail_lev {
    int Kx, Ky, n, ld;
    float rKy, alpha;
    const float *k;          // constants
    float *r, *z, *t, *acc;  // z and t with halo, leading dimension ld = Ky + 2
};
__device__ __forceinline__ tail_lev tail_level(float *lds, const int *D)
{
    return tail_lev{D[0], D[1], D[2], D[1] + 2, __int_as_float(D[4]), __int_as_float(D[3]), lds + D[5], lds + D[6],
                    lds + D[7], lds + D[8], lds + D[9]};
}
struct tail_cell {
    float c[8], d, dinv;
};
__device__ __forceinline__ tail_cell tail_consts(const tail_lev &L, int f)
{
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4 *k = reinterpret_cast<const f4 *>(L.k + f * LV_CELL);
    const f4 a = k[0], b = k[1], e = k[2];
    return tail_cell{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, e.x, e.y};
}
// v into cell (cx, cy) of the haloed array a, and into the halo cells that stand for it on periodic axes
__device__ __forceinline__ void tail_put(float *a, const tail_lev &L, int xper, int yper, int cx, int cy, float v)
{
    const int ld = L.ld;
    a[(cx + 1) * ld + cy + 1] = v;
    const bool x0 = xper && cx == 0, x1 = xper && cx == L.Kx - 1, y0 = yper && cy == 0, y1 = yper && cy == L.Ky - 1;
    if (!(x0 || x1 || y0 || y1)) return;
    auto column = [&](int px) {
        if (y0) a[px * ld + L.Ky + 1] = v;
        if (y1) a[px * ld] = v;
    };
    column(cx + 1);
    if (x0) {
        a[(L.Kx + 1) * ld + cy + 1] = v;
        column(L.Kx + 1);
    }
    if (x1) {
        a[cy + 1] = v;
        column(0);
    }
}
// the neighbours of the haloed array's entry at p, in slot order
__device__ __forceinline__ void tail_nbrs(const float *a, int p, int ld, float (&v)[8])
{
    v[0] = a[p - ld - 1];
    v[1] = a[p - ld];
    v[2] = a[p - ld + 1];
    v[3] = a[p - 1];
    v[4] = a[p + 1];
    v[5] = a[p + ld - 1];
    v[6] = a[p + ld];
    v[7] = a[p + ld + 1];
}

// One operation in LDS, the arithmetic of st_down_lane, st_up_cell and st_wsave_cell (L: its level, C: the next).  A
// right-hand side is stored with its level's pre-smoothed z = w D^-1 r.  (A neighbour outside a level has
// coupling 0 there, by construction, and a zero in the halo.)
__device__ __forceinline__ void tail_step(int op, const tail_lev &L, const tail_lev &C, bool dense_next, const float *inv,
                                          int xper, int yper)
{
    if (op == OP_DOWN) {
        for (int base = 0; base < C.n * CF2; base += TB) {  // uniform trip count: every lane shuffles
            const int tid = base + threadIdx.x;
            const int P = tid / CF2, q = tid % CF2, Px = div_small(P, C.rKy), Py = P - Px * C.Ky;
            const int cx = CF * Px + q / CF, cy = CF * Py + q % CF;
            float t = 0.0f;
            if (P < C.n && cx < L.Kx && cy < L.Ky) {
                const int f = cx * L.Ky + cy, p = (cx + 1) * L.ld + cy + 1;
                const tail_cell k = tail_consts(L, f);
                float zj[8];
                tail_nbrs(L.z, p, L.ld, zj);
                const float zf = L.z[p];
                float acc = k.d * zf;
#pragma unroll
                for (int e = 0; e < 8; e++) acc += k.c[e] * (zf - zj[e]);
                t = L.r[f] - acc;
            }
            t = sum_children(t);
            if (q == 0 && P < C.n) {
                C.r[P] = t;
                if (!dense_next) tail_put(C.z, C, xper, yper, Px, Py, OMEGA * C.k[P * LV_CELL + 9] * t);
            }
        }
    } else if (op == OP_DENSE) {
        // t = inv r: 16 lanes per row (LV_AMG_DENSE_MAX * 16 == TB)
        const int n = L.n, i = threadIdx.x >> 4, q = threadIdx.x & 15;
        float acc = 0.0f;
        if (i < n)
            for (int j = q; j < n; j += 16) acc += inv[j * n + i] * L.r[j];
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        acc += __shfl_xor(acc, 4);
        acc += __shfl_xor(acc, 8);
        if (q == 0 && i < n) {
            const int cx = div_small(i, L.rKy);
            tail_put(L.t, L, xper, yper, cx, i - cx * L.Ky, acc);
        }
    } else if (op == OP_UP) {
        for (int f = threadIdx.x; f < L.n; f += TB) {
            const int cx = div_small(f, L.rKy), cy = f - cx * L.Ky, p = (cx + 1) * L.ld + cy + 1;
            const tail_cell k = tail_consts(L, f);
            float zj[8];
            tail_nbrs(L.z, p, L.ld, zj);
            // the parents of the neighbours on each side: the cell's own, or the next one (with the halo, at
            // the ends of the level too; a last cell without a sibling has the next parent on its right)
            const int Px = cx / CF + 1, Py = cy / CF + 1;
            const int xl = (cx % CF ? Px : Px - 1) * C.ld, xr = (cx % CF || cx + 1 == L.Kx ? Px + 1 : Px) * C.ld;
            const int yl = cy % CF ? Py : Py - 1, yr = cy % CF || cy + 1 == L.Ky ? Py + 1 : Py;
            const int xo = Px * C.ld;
            const float a = L.alpha;
            const float ej[8] = {a * C.t[xl + yl], a * C.t[xl + Py], a * C.t[xl + yr], a * C.t[xo + yl],
                                 a * C.t[xo + yr], a * C.t[xr + yl], a * C.t[xr + Py], a * C.t[xr + yr]};
            const float z1 = L.z[p] + a * C.t[xo + Py];
            float acc = k.d * z1;
#pragma unroll
            for (int e = 0; e < 8; e++) acc += k.c[e] * (z1 - (zj[e] + ej[e]));
            tail_put(L.t, L, xper, yper, cx, cy, z1 + OMEGA * k.dinv * (L.r[f] - acc));
        }
    } else if (op == OP_WSAVE) {
        for (int f = threadIdx.x; f < L.n; f += TB) {
            const int cx = div_small(f, L.rKy), cy = f - cx * L.Ky, p = (cx + 1) * L.ld + cy + 1;
            const tail_cell k = tail_consts(L, f);
            float tj[8];
            tail_nbrs(L.t, p, L.ld, tj);
            const float tf = L.t[p];
            float acc = k.d * tf;
#pragma unroll
            for (int e = 0; e < 8; e++) acc += k.c[e] * (tf - tj[e]);
            L.acc[f] = tf;
            const float r = L.r[f] - acc;
            L.r[f] = r;
            tail_put(L.z, L, xper, yper, cx, cy, OMEGA * k.dinv * r);
        }
    } else {  // OP_WADD
        for (int f = threadIdx.x; f < L.n; f += TB) {
            const int cx = div_small(f, L.rKy), cy = f - cx * L.Ky;
            tail_put(L.t, L, xper, yper, cx, cy, L.t[(cx + 1) * L.ld + cy + 1] + L.acc[f]);
        }
    }
}

// The same program with the tail levels in LDS: the couplings, the dense inverse, the program
// and the right-hand side of the first level are copied in, every operation then reads and
// writes LDS only, and the final correction of the first level is copied out.
// The constant arrays come from img (k_tail_pack's image of them in this layout) by one flat copy
// whose loads are all issued before the done flag is tested and the first LDS store is made; a copy
// loop per array would wait for a global round trip per iteration.
//
// The W-visited tail as a matrix (COLS).  A visit is a linear, symmetric operator on the right-hand side of the
// tail's first level: for a singular system set-up applies the program to every unit vector, one workgroup a
// column (the right-hand side is that of cell blockIdx.x, and the correction becomes row blockIdx.x of mat, of
// leading dimension ld: the operator is symmetric), and each cycle multiplies by the matrix (k_mat_mv).  The
// W-visit is a serial chain of about 30 operations on one CU, 25-29 us a cycle whatever the rest of the device
// does; the product reads at most 4 MB spread over the device in one round trip, 2.7-4.7 us, and the columns
// take 60 us once per set-up (25 x 25 cells, 3 turns of the device).  A nonsingular system keeps the
// program: its V-visit takes 7-11 us, and its solves keep their iterates bit for bit (velocities near rest
// are small differences of pressures, and would show another rounding of the cycle magnified).
struct tail_lds_args {
    const int *desc, *prog;  // the levels' descriptors (LV_DESC ints each), the operations
    int nprog;
    const float *img;
    int coef, total, first, last, n0, xper, yper, inv;
    const float *r, *dinv;  // right-hand side, 1 / (d + sum c) and correction of level `first`
    float *t;
};

template <bool COLS>
__global__ __launch_bounds__(TB) void k_tail_lds(tail_lds_args T, const lv_cg_scalars *S, float *__restrict__ mat, int ld)
{
    __shared__ __align__(16) float lds[TAIL_LDS];
    __shared__ int lprog[LV_AMG_MAXPROG], desc[(LV_AMG_MAXLEV + 1) * LV_DESC];
    constexpr int PER4 = (TAIL_LDS / 4 + TB - 1) / TB;  // float4s per lane
    const int n4 = T.coef / 4, t = threadIdx.x;
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4 *img4 = reinterpret_cast<const f4 *>(T.img);
    f4 v[PER4];
#pragma unroll
    for (int q = 0; q < PER4; q++)
        if (q * TB + t < n4) v[q] = img4[q * TB + t];
    const int pr = t < T.nprog ? T.prog[t] : 0;  // nprog <= LV_AMG_MAXPROG <= TB
    const int de = t < (LV_AMG_MAXLEV + 1) * LV_DESC ? T.desc[t] : 0;
    float r0[2], v0[2];  // n0 <= LDS_MAX <= 2 TB
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int f = h * TB + t;
        r0[h] = f < T.n0 ? (COLS ? (f == (int)blockIdx.x ? 1.0f : 0.0f) : T.r[f]) : 0.0f;
        v0[h] = f < T.n0 ? T.dinv[f] : 0.0f;
    }
    if (S && S->done) return;  // tested after the loads above are issued (they read valid arrays)
    f4 *lds4 = reinterpret_cast<f4 *>(lds);
#pragma unroll
    for (int q = 0; q < PER4; q++)
        if (q * TB + t < n4) lds4[q * TB + t] = v[q];
    for (int f = T.coef + t; f < T.total; f += TB) lds[f] = 0.0f;
    if (t < T.nprog) lprog[t] = pr;
    if (t < (LV_AMG_MAXLEV + 1) * LV_DESC) desc[t] = de;
    __syncthreads();
    const tail_lev L0 = tail_level(lds, desc + T.first * LV_DESC);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int f = h * TB + t;
        if (f >= T.n0) continue;
        L0.r[f] = r0[h];
        const int cx = div_small(f, L0.rKy);
        if (T.first < T.last) tail_put(L0.z, L0, T.xper, T.yper, cx, f - cx * L0.Ky, OMEGA * v0[h] * r0[h]);
    }
    __syncthreads();
    for (int pc = 0; pc < T.nprog; pc++) {
        const int code = lprog[pc];
        const int op = code >> OP_SHIFT, l = code & ((1 << OP_SHIFT) - 1);
        const int *D = desc + l * LV_DESC;
        tail_step(op, tail_level(lds, D), tail_level(lds, D + (l < T.last ? LV_DESC : 0)), l + 1 == T.last, lds + T.inv,
                  T.xper, T.yper);
        __syncthreads();
    }
    float *row = COLS ? mat + (size_t)blockIdx.x * ld : T.t;
    for (int f = t; f < (COLS ? ld : T.n0); f += TB) {
        const int cx = div_small(f, L0.rKy);
        row[f] = f < T.n0 ? L0.t[(cx + 1) * L0.ld + (f - cx * L0.Ky) + 1] : 0.0f;
    }
}

// The matrix of level L from that of the next level (nc cells, leading dimension ldc): row j is the
// V-visit of the unit vector of cell j, EXT_ROWS to a workgroup, which loads each cell's couplings once
// for all of them.  The right-hand side a unit vector leaves the next level has a handful of entries, at the parents of
// its 3 x 3 neighbourhood, so that level's correction is a sum of as many rows of its matrix.  At 50 x 50
// cells (level 1 of 100^2 particles) it takes 41 us once per set-up (99 with a row a workgroup and the whole down
// pass for each) and the product 5.1 us, against the 11 us of the two stencil launches, the product and
// the prolongation that it replaces in each cycle.
constexpr int EXT_ROWS = 4;
__global__ __launch_bounds__(B) void k_mat_extend(st_level L, int Kyc, int nc, const float *__restrict__ matc, int ldc,
                                                  float *__restrict__ mat, int ld)
{
    __shared__ float ec[EXT_ROWS][TAIL_MAX], cv[EXT_ROWS][9], rv[EXT_ROWS][9];
    __shared__ int cp[EXT_ROWS][9], rp[EXT_ROWS][9], rcnt[EXT_ROWS];
    const int n = L.Kx * L.Ky, R0 = blockIdx.x * EXT_ROWS, t = threadIdx.x;
    static_assert(EXT_ROWS * 9 * CF2 <= B, "a lane a child");
    {  // the parents of the unit cell's 3 x 3 neighbourhood, a lane for each of their children
        const int k = min(t / (9 * CF2), EXT_ROWS - 1), c9 = t / CF2 % 9, q = t % CF2;
        const int R = min(R0 + k, n - 1), cx = R / L.Ky, cy = R - cx * L.Ky;
        bool okx, oky;
        const int jx = wrap_near(cx + c9 / 3 - 1, L.Kx, L.xper, okx), jy = wrap_near(cy + c9 % 3 - 1, L.Ky, L.yper, oky);
        const int P = okx && oky ? (jx / CF) * Kyc + jy / CF : nc;
        const int Px = P / Kyc, x = CF * Px + q / CF, y = CF * (P - Px * Kyc) + q % CF;
        float v = 0.0f;
        if (P < nc && x < L.Kx && y < L.Ky) {  // as st_down_lane
            const int f = x * L.Ky + y;
            float ck[8];
            int J[8];
            st_nbrs(L, x, y, f, ck, J);
            const float rf = f == R ? 1.0f : 0.0f, zf = OMEGA * L.dinv[f] * rf;
            float acc = L.d[f] * zf;
#pragma unroll
            for (int m = 0; m < 8; m++) acc += ck[m] * (zf - OMEGA * L.dinv[J[m]] * (J[m] == R ? 1.0f : 0.0f));
            v = rf - acc;
        }
        v = sum_children(v);
        if (q == 0 && t < EXT_ROWS * 9 * CF2) {
            cp[k][c9] = P;
            cv[k][c9] = v;
        }
    }
    __syncthreads();
    if (t < EXT_ROWS) {  // the nonzero ones in order, each once
        int m = 0;
        for (int last = -1;; m++) {
            int best = nc, at = 0;
            for (int q = 0; q < 9; q++)
                if (cp[t][q] > last && cp[t][q] < best && cv[t][q] != 0.0f) {
                    best = cp[t][q];
                    at = q;
                }
            if (best == nc) break;
            rp[t][m] = best;
            rv[t][m] = cv[t][at];
            last = best;
        }
        rcnt[t] = m;
    }
    __syncthreads();
    for (int i = t; i < nc; i += B)
#pragma unroll
        for (int k = 0; k < EXT_ROWS; k++) {
            float a = 0.0f;
            for (int q = 0; q < rcnt[k]; q++) a += rv[k][q] * matc[(size_t)rp[k][q] * ldc + i];
            ec[k][i] = a;
        }
    __syncthreads();
    float zr[EXT_ROWS];
#pragma unroll
    for (int k = 0; k < EXT_ROWS; k++) zr[k] = OMEGA * L.dinv[min(R0 + k, n - 1)] * 1.0f;
    for (int f = t; f < ld; f += B) {  // as st_up_cell
        float ck[8], d = 0.0f, di = 0.0f;
        int J[8], PJ[8], Pf = 0;
        if (f < n) {
            const int cx = f / L.Ky, cy = f - cx * L.Ky;
            st_nbrs(L, cx, cy, f, ck, J, PJ, Kyc);
            Pf = (cx / CF) * Kyc + cy / CF;
            d = L.d[f];
            di = L.dinv[f];
        }
#pragma unroll
        for (int k = 0; k < EXT_ROWS; k++) {
            const int R = R0 + k;
            if (R >= n) break;
            float v = 0.0f;
            if (f < n) {
                const float z1 = (f == R ? zr[k] : 0.0f) + L.alpha * ec[k][Pf];
                float acc = d * z1;
#pragma unroll
                for (int m = 0; m < 8; m++)
                    acc += ck[m] * (z1 - ((J[m] == R ? zr[k] : 0.0f) + L.alpha * ec[k][PJ[m]]));
                v = z1 + OMEGA * di * ((f == R ? 1.0f : 0.0f) - acc);
            }
            mat[(size_t)R * ld + f] = v;
        }
    }
}

// t = mat r for the matrix level (n cells, at most 256 PER): a wavefront a row, every load of the row and
// of r issued before the done flag is tested.  r is allocated to a multiple of 4; the entries past n are
// dropped.  PROLONG (level 1 in the aggregate order): also the prolongation of each cell's correction into
// its rows of z0, as k_prolong1 forms it.
// (HEAD as in k_st_down)
template <int PER, bool PROLONG, bool HEAD>
__global__ __launch_bounds__(B) void k_mat_mv(int n, int ld, const float *__restrict__ mat, const float *__restrict__ r,
                                              float *__restrict__ t, const lv_cg_scalars *S,
                                              const int *__restrict__ start, float alpha0, float *__restrict__ z0,
                                              lv_cycle_head H)
{
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, row = blockIdx.x * (B / 64) + (threadIdx.x >> 6);
    const int rw = row < n ? row : n - 1;
    const f4 *m4 = reinterpret_cast<const f4 *>(mat + (size_t)rw * ld);
    const f4 *r4 = reinterpret_cast<const f4 *>(r);
    f4 m[PER], x[PER];
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int k = q * 64 + lane, kk = 4 * k < ld ? k : 0;
        m[q] = m4[kk];
        x[q] = r4[kk];
    }
    const int b0 = PROLONG ? start[rw] : 0, e = PROLONG ? start[rw + 1] : 0;
    if (HEAD) {
        if (head_stops(H)) return;
    } else if (S && S->done) {
        return;
    }
    float a = 0.0f;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int k = 4 * (q * 64 + lane);
#pragma unroll
        for (int c = 0; c < 4; c++) a += k + c < n ? m[q][c] * x[q][c] : 0.0f;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
    if (row >= n) return;
    if (lane == 0) t[row] = a;
    if (PROLONG)
        for (int i = b0 + lane; i < e; i += 64) z0[i] += alpha0 * a;
}
static_assert(B == 256 && FUSE_ROWS + 64 <= FUSE_CAP, "fused blocks fit their LDS rows");
static_assert(LV_AMG_DENSE_MAX * 16 == TB, "the dense solve of the tail maps 16 lanes to a row");
static_assert(TAIL_MAX <= LDS_MAX && LDS_MAX <= 2 * TB && LV_AMG_MAXPROG <= TB && LDS_MAX * CF2 <= 8192 &&
                  (LV_AMG_MAXLEV + 1) * LV_DESC <= TB,
              "right-hand side entries, operations and descriptors per lane, and indices that div_small divides");
static_assert(TAIL_LDS % 4 == 0, "the LDS image is copied as float4");

// the program and the levels' descriptors, by value in the launch: two copies from pageable memory would
// each hold the host up
struct tail_tables {
    uint8_t prog[LV_AMG_MAXPROG];
    int desc[(LV_AMG_MAXLEV + 1) * LV_DESC];
};
static_assert((OP_WADD << OP_SHIFT | LV_AMG_MAXLEV) < 256, "an operation fits a byte");
__global__ __launch_bounds__(TB) void k_tail_put(tail_tables H, int nprog, int *__restrict__ prog, int *__restrict__ desc)
{
    const int t = threadIdx.x;
    if (t < nprog) prog[t] = H.prog[t];
    if (t < (LV_AMG_MAXLEV + 1) * LV_DESC) desc[t] = H.desc[t];
}

// the tail levels' constants and the dense inverse into img in the LDS layout
__global__ __launch_bounds__(B) void k_tail_pack(tail_levels T, tail_layout Y, const float *__restrict__ inv,
                                                 float *__restrict__ img)
{
    const int stride = gridDim.x * B;
    for (int l = T.first; l < T.last; l++) {
        const int n = T.Kx[l] * T.Ky[l];
        for (int f = blockIdx.x * B + threadIdx.x; f < LV_CELL * n; f += stride) {
            const int i = f / LV_CELL, k = f - i * LV_CELL;
            img[Y.k[l] + f] = k < 8 ? T.c[l][(size_t)k * n + i] : k == 8 ? T.d[l][i] : k == 9 ? T.dinv[l][i] : 0.0f;
        }
    }
    const int nd = T.Kx[T.last] * T.Ky[T.last];
    for (int f = blockIdx.x * B + threadIdx.x; f < ((nd * nd + 3) & ~3); f += stride)
        img[Y.inv + f] = f < nd * nd ? inv[f] : 0.0f;
}

// ---- power iteration for the scale of the learned fine smoother ----------------------------------

// +-1 probe hashed from the particle index (list: the particle of each row in the aggregate order)
__global__ __launch_bounds__(B) void k_pw_init(int n, const int *__restrict__ list, float *__restrict__ v)
{
    const int p = blockIdx.x * B + threadIdx.x;
    if (p >= n) return;
    const int i = list ? list[p] : p;
    uint64_t z = 0x5EED5EEDull + ((uint64_t)i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    v[p] = (z >> 63) ? 1.0f : -1.0f;
}

// u = M (A v) computed row-wise through the work vector t = A v: two launches
template <class V>
__global__ __launch_bounds__(B) void k_pw_av(fine_ops<V> F, const float *__restrict__ v, float *__restrict__ t)
{
    const int i = blockIdx.x * B + threadIdx.x;
    if (i < F.n) t[i] = a_row(i, F, v);
}
// u = M t; partials |u|^2, |v|^2
template <class V>
__global__ __launch_bounds__(B) void k_pw_mt(fine_ops<V> F, const float *__restrict__ t,
                                             const float *__restrict__ v, float *__restrict__ u,
                                             double *__restrict__ part)
{
    double s[2] = {0.0, 0.0};
    for (int i = blockIdx.x * B + threadIdx.x; i < F.n; i += gridDim.x * B) {
        const float ui = m_row(i, F, t);
        u[i] = ui;
        s[0] += (double)ui * (double)ui;
        s[1] += (double)v[i] * (double)v[i];
    }
    block_partials<2>(s, part, gridDim.x);
}
__global__ __launch_bounds__(B) void k_pw_norm(const double *__restrict__ part, int nb, double *__restrict__ out)
{
    double o[2];
    reduce_all<2>(part, nb, o);
    if (threadIdx.x == 0) {
        out[0] = o[0];
        out[1] = o[1];
    }
}
// v = u / |u|
__global__ __launch_bounds__(B) void k_pw_scale(int n, const float *__restrict__ u, const double *__restrict__ nrm,
                                                float *__restrict__ v)
{
    const int i = blockIdx.x * B + threadIdx.x;
    if (i < n) v[i] = (float)((double)u[i] / sqrt(nrm[0]));
}

// ---- the aggregate order -----------------------------------------------------------------------

// iperm[list[p]] = p and the level-1 cell of row p
__global__ __launch_bounds__(B) void k_perm_index(int n, const int *__restrict__ list, const int *__restrict__ agg,
                                                  int *__restrict__ iperm, int *__restrict__ aggp)
{
    const int p = blockIdx.x * B + threadIdx.x;
    if (p >= n) return;
    const int i = list[p];
    iperm[i] = p;
    aggp[p] = agg[i];
}

// row p of the aggregate order from row list[p] of the operator (same slot order): degree, column
// offsets taken modulo n into [-n/2, n/2], FP32 and BF16 couplings, d, D^-1, and the learned M;
// slots LV_OVF_BASE.. (offsets, FP32 couplings) also into the compact overflow of p's 64-row group
// when the group has at most ocap overflow slots (lv_ell.h); *flag is raised when an offset needs
// more than 16 bits
__global__ __launch_bounds__(B) void k_perm_ell(int n, const int *__restrict__ list, const int *__restrict__ iperm,
                                                const int *__restrict__ deg, const int *__restrict__ ecol,
                                                const float *__restrict__ ev, const float *__restrict__ diag,
                                                const float *__restrict__ dinv, const float *__restrict__ mval,
                                                const float *__restrict__ mdg, uint8_t *__restrict__ pdeg,
                                                int16_t *__restrict__ poff, float *__restrict__ pev32,
                                                uint16_t *__restrict__ pev16, float *__restrict__ pdiag,
                                                float *__restrict__ pdinv, float *__restrict__ pmval,
                                                float *__restrict__ pmdg, int *__restrict__ flag,
                                                int16_t *__restrict__ ooff, float *__restrict__ oev32, int ocap)
{
    const int p = blockIdx.x * B + threadIdx.x;
    // everything of row i loaded as soon as i is known, unconditionally (a lane past n takes row
    // list[n-1] and drops it): the degree, the diagonals and the first U slots' columns and
    // couplings; then their rows' new positions gathered together (a slot past the degree reads
    // the allocated slot, and its column is taken as the row's own so that the gather stays in
    // bounds; neither is used)
    const int i = list[p < n ? p : n - 1];
    constexpr int U = 8;
    const int di = deg[i];
    const float dgi = diag[i], dvi = dinv[i];
    int cj[U];
    float vj[U];
#pragma unroll
    for (int k = 0; k < U; k++) {
        const size_t e = (size_t)k * n + i;
        cj[k] = ecol[e];
        vj[k] = ev[e];
    }
    const int d = p < n ? di : 0;
    const lv_ovf_pos q = lv_ovf_prefix(d);  // the block's wavefronts are whole 64-row groups
    if (p >= n) return;
    const bool compact = ocap > 0 && q.tot <= ocap;
    const size_t g0 = (size_t)(p >> 6) * LV_OVF_CAP;
    pdeg[p] = (uint8_t)d;
    pdiag[p] = dgi;
    pdinv[p] = dvi;
    if (mdg) pmdg[p] = mdg[i];
    bool wide = false;
    int pj[U];
#pragma unroll
    for (int k = 0; k < U; k++) pj[k] = k < d ? cj[k] : i;
#pragma unroll
    for (int k = 0; k < U; k++) pj[k] = iperm[pj[k]];
    auto put = [&](int k, int col_new, float v) {
        const size_t e = (size_t)k * n + i, ep = (size_t)k * n + p;
        int off = col_new - p;
        if (off > n / 2) off -= n;
        if (off < -(n / 2)) off += n;
        wide |= (off < -32768 || off > 32767);
        poff[ep] = (int16_t)off;
        pev32[ep] = v;
        pev16[ep] = lv_bf16_bits(v);
        if (mval) pmval[ep] = mval[e];
        if (compact && k >= LV_OVF_BASE) {
            const size_t eo = g0 + (size_t)(q.pos + (k - LV_OVF_BASE));
            ooff[eo] = (int16_t)off;
            oev32[eo] = v;
        }
    };
#pragma unroll
    for (int k = 0; k < U; k++)
        if (k < d) put(k, pj[k], vj[k]);
    for (int k = U; k < d; k++) {
        const size_t e = (size_t)k * n + i;
        put(k, iperm[ecol[e]], ev[e]);
    }
    if (wide) atomicOr(flag, 1);
}

}  // namespace

#define AMG_CHECK(expr)                  \
    do {                                 \
        hipError_t _e = (expr);          \
        if (_e != hipSuccess) return _e; \
    } while (0)

template <typename T>
static hipError_t grow(T **p, size_t *cap, size_t want)
{
    if (*cap >= want && *p) return hipSuccess;
    if (*p) AMG_CHECK(hipFree(*p));
    *p = nullptr;
    *cap = 0;
    AMG_CHECK(hipMalloc((void **)p, sizeof(T) * (want ? want : 1)));
    *cap = want;
    return hipSuccess;
}

hipError_t lv_amg_init(lv_amg *G)
{
    memset(G, 0, sizeof(*G));
    AMG_CHECK(hipMalloc(&G->dense_inv, sizeof(float) * LV_AMG_DENSE_MAX * LV_AMG_DENSE_MAX));
    AMG_CHECK(hipMalloc(&G->tail_img, sizeof(float) * TAIL_LDS));
    AMG_CHECK(hipMalloc(&G->pw, sizeof(double) * (2 * LV_NBMAX + 2)));
    AMG_CHECK(hipMalloc(&G->prog, sizeof(int) * LV_AMG_MAXPROG));
    AMG_CHECK(hipMalloc(&G->desc, sizeof(int) * (LV_AMG_MAXLEV + 1) * LV_DESC));
    AMG_CHECK(hipMalloc(&G->pflag, 2 * sizeof(int)));
    AMG_CHECK(hipMemset(G->pflag, 0, 2 * sizeof(int)));
    return hipSuccess;
}

void lv_amg_free(lv_amg *G)
{
    void *ptrs[] = {G->agg, G->cnt, G->start, G->list, G->scan_tmp, G->t0, G->z0, G->dense_inv, G->tail_img, G->tail_mat, G->ext_mat, G->tail_work,
                    G->pw, G->pv, G->pu, G->prog, G->desc, G->iperm, G->aggp, G->pdeg, G->poff, G->pev32, G->pev16,
                    G->pdiag32, G->pdinv32, G->pmval, G->pmdg, G->pflag, G->bfirst, G->ooff, G->oev32};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    lv_mail_free(&G->mail);
    for (int l = 0; l <= LV_AMG_MAXLEV; l++) {
        lv_amg_level &L = G->lev[l];
        void *q[] = {L.d, L.c, L.dinv, L.r, L.z, L.t, L.acc};
        for (void *p : q)
            if (p) (void)hipFree(p);
    }
    memset(G, 0, sizeof(*G));
}

static hipError_t level_alloc(lv_amg_level &L, int Kx, int Ky)
{
    L.Kx = Kx;
    L.Ky = Ky;
    L.n = Kx * Ky;
    if (L.cap < (size_t)L.n) {
        void *q[] = {L.d, L.c, L.dinv, L.r, L.z, L.t, L.acc};
        L.d = L.c = L.dinv = L.r = L.z = L.t = L.acc = nullptr;
        L.cap = 0;
        for (void *p : q)
            if (p) AMG_CHECK(hipFree(p));
        const size_t m = (size_t)L.n;
        AMG_CHECK(hipMalloc(&L.d, sizeof(float) * m));
        AMG_CHECK(hipMalloc(&L.c, sizeof(float) * 8 * m));
        AMG_CHECK(hipMalloc(&L.dinv, sizeof(float) * m));
        AMG_CHECK(hipMalloc(&L.r, sizeof(float) * ((m + 3) & ~(size_t)3)));  // read as float4 by k_mat_mv
        AMG_CHECK(hipMalloc(&L.z, sizeof(float) * m));
        AMG_CHECK(hipMalloc(&L.t, sizeof(float) * m));
        AMG_CHECK(hipMalloc(&L.acc, sizeof(float) * m));
        L.cap = m;
    }
    return hipSuccess;
}

static fine_ops<lv_ell_own<float>> fine_own(const lv_amg *G, const lv_pressure_system &A)
{
    fine_ops<lv_ell_own<float>> F;
    F.n = G->n0;
    F.A = lv_ell_own<float>{A.deg, A.ecol, A.ev32};
    F.diag = A.diag32;
    F.dinv = A.dinv32;
    F.mval = G->fine_learned ? G->mval : nullptr;
    F.mdg = G->fine_learned ? G->mdg : nullptr;
    F.scale = G->fine_scale;
    F.alpha = G->fine_alpha;
    return F;
}

// the aggregate order with the couplings in V's precision (BF16 for the cycle, FP32 for the power
// iteration of the smoother scale)
template <class V, typename VAL>
static fine_ops<V> fine_agg(const lv_amg *G, const VAL *val)
{
    fine_ops<V> F;
    F.n = G->n0;
    F.A = V{G->pdeg, G->poff, val};
    if constexpr (std::is_same<VAL, float>::value) {  // the compact overflow holds the FP32 couplings
        F.A.ocol = G->ooff;
        F.A.oval = G->oev32;
        F.A.ocap = G->ovf_cap;
    }
    F.diag = G->pdiag32;
    F.dinv = G->pdinv32;
    F.mval = G->fine_learned ? G->pmval : nullptr;
    F.mdg = G->fine_learned ? G->pmdg : nullptr;
    F.scale = G->fine_scale;
    F.alpha = G->fine_alpha;
    return F;
}

// 10 steps of power iteration on M A (fine view F): the largest eigenvalue's estimate, 0 if none
template <class V>
static hipError_t power_lambda(lv_amg *G, const fine_ops<V> &Fo, const int *list, double *lam, hipStream_t s)
{
    const int n = G->n0;
    const int nb = lv_nblocks(n);
    double *part = G->pw, *nrm = G->pw + 2 * LV_NBMAX;
    hipLaunchKernelGGL(k_pw_init, g1(n), dim3(B), 0, s, n, list, G->pv);
    double h[2] = {0.0, 0.0};
    for (int it = 0; it < 10; it++) {
        hipLaunchKernelGGL(k_pw_av<V>, g1(n), dim3(B), 0, s, Fo, (const float *)G->pv, G->t0);
        hipLaunchKernelGGL(k_pw_mt<V>, dim3(nb), dim3(B), 0, s, Fo, (const float *)G->t0, (const float *)G->pv,
                           G->pu, part);
        hipLaunchKernelGGL(k_pw_norm, dim3(1), dim3(B), 0, s, (const double *)part, nb, nrm);
        hipLaunchKernelGGL(k_pw_scale, g1(n), dim3(B), 0, s, n, (const float *)G->pu, (const double *)nrm, G->pv);
    }
    AMG_CHECK(hipMemcpyAsync(h, nrm, sizeof(h), hipMemcpyDeviceToHost, s));
    AMG_CHECK(hipStreamSynchronize(s));
    *lam = (h[1] > 0.0) ? sqrt(h[0] / h[1]) : 0.0;
    return hipSuccess;
}

// the operations of the single-workgroup kernel for the visit of level l (last: the dense level);
// with W, every coarse level below l is visited twice, the second time on the residual the first
// correction leaves (OP_WSAVE), the two corrections summed (OP_WADD).  false if the program would
// not fit.
static bool tail_visit(int l, int last, bool W, int *prog, int &np)
{
    auto emit = [&](int op, int lev) {
        if (np >= LV_AMG_MAXPROG) return false;
        prog[np++] = (op << OP_SHIFT) | lev;
        return true;
    };
    if (l == last) return emit(OP_DENSE, l);
    if (!emit(OP_DOWN, l) || !tail_visit(l + 1, last, W, prog, np)) return false;
    if (W && l + 1 < last)
        if (!emit(OP_WSAVE, l + 1) || !tail_visit(l + 1, last, W, prog, np) || !emit(OP_WADD, l + 1)) return false;
    return emit(OP_UP, l);
}

// the program of the tail: the visit of its first level, itself W-visited when W
static int tail_program(int first, int last, bool W, int *prog)
{
    int np = 0;
    bool ok = tail_visit(first, last, W, prog, np);
    if (ok && W && first < last) {
        ok = np < LV_AMG_MAXPROG;
        if (ok) prog[np++] = (OP_WSAVE << OP_SHIFT) | first;
        ok = ok && tail_visit(first, last, W, prog, np) && np < LV_AMG_MAXPROG;
        if (ok) prog[np++] = (OP_WADD << OP_SHIFT) | first;
    }
    if (ok) return np;
    np = 0;
    tail_visit(first, last, false, prog, np);
    return np;
}

// the levels lk..nlev of the single-workgroup kernel
static tail_levels tail_levels_of(const lv_amg *G)
{
    tail_levels T;
    memset(&T, 0, sizeof(T));
    T.first = G->lk;
    T.last = G->nlev;
    T.xper = G->xper;
    T.yper = G->yper;
    for (int l = G->lk; l <= G->nlev; l++) {
        const lv_amg_level &L = G->lev[l];
        T.Kx[l] = L.Kx;
        T.Ky[l] = L.Ky;
        T.alpha[l] = L.alpha;
        T.acc[l] = L.acc;
        T.d[l] = L.d;
        T.c[l] = L.c;
        T.dinv[l] = L.dinv;
        T.r[l] = L.r;
        T.z[l] = L.z;
        T.t[l] = L.t;
    }
    return T;
}

// their LDS layout
static tail_layout tail_layout_of(const lv_amg *G)
{
    tail_layout Y;
    memset(&Y, 0, sizeof(Y));
    int off = 0;
    auto put = [&off](int count) {
        const int o = off;
        off += (count + 3) & ~3;
        return o;
    };
    for (int l = G->lk; l < G->nlev; l++) Y.k[l] = put(LV_CELL * G->lev[l].n);
    Y.inv = put(G->lev[G->nlev].n * G->lev[G->nlev].n);
    Y.coef = off;
    for (int l = G->lk; l <= G->nlev; l++) {
        const lv_amg_level &L = G->lev[l];
        const int halo = (L.Kx + 2) * (L.Ky + 2);
        Y.r[l] = put(L.n);
        Y.t[l] = put(halo);
        if (l < G->nlev) Y.z[l] = put(halo);
        if (l < G->nlev && G->wcycle) Y.acc[l] = put(L.n);
    }
    Y.total = off;
    return Y;
}

// the levels' descriptors for the LDS kernel
static void tail_descriptors(const lv_amg *G, const tail_layout &Y, int *D)
{
    auto bits = [](float f) {
        int i;
        memcpy(&i, &f, sizeof(i));
        return i;
    };
    memset(D, 0, sizeof(int) * (LV_AMG_MAXLEV + 1) * LV_DESC);
    for (int l = G->lk; l <= G->nlev; l++) {
        const lv_amg_level &L = G->lev[l];
        const int v[10] = {L.Kx,    L.Ky,   L.n,    bits(L.alpha), bits(1.0f / (float)L.Ky), Y.k[l], Y.r[l],
                           Y.z[l], Y.t[l], Y.acc[l]};
        memcpy(D + l * LV_DESC, v, sizeof(v));
    }
}

static tail_lds_args tail_args_of(const lv_amg *G)
{
    const lv_amg_level &L = G->lev[G->lk];
    return tail_lds_args{G->desc,  G->prog, G->nprog, G->tail_img, G->tail_coef, G->tail_total, G->lk, G->nlev,
                         L.n, G->xper, G->yper, G->tail_inv, L.r, L.dinv, L.t};
}

hipError_t lv_amg_setup(lv_amg *G, const lv_grid_params &g, const double *x, const lv_pressure_system &A, int n,
                        const float *mval, const float *mdg, int layout, hipStream_t s)
{
    if (!G->mail.host) AMG_CHECK(lv_mail_init(&G->mail));
    G->n0 = n;
    G->xper = g.xperiodic;
    G->yper = g.yperiodic;
    const double Lx = g.bxmax0 - g.bxmin0, Ly = g.bxmax1 - g.bxmin1;
    const int Kx = std::max(1, (int)floor(Lx / (CELL_DR * g.dr))), Ky = std::max(1, (int)floor(Ly / (CELL_DR * g.dr)));
    const int na = Kx * Ky;
    G->na = na;
    AMG_CHECK(grow(&G->agg, &G->cap_agg, (size_t)n));
    AMG_CHECK(grow(&G->list, &G->cap_list, (size_t)n));
    AMG_CHECK(grow(&G->t0, &G->cap_t0, (size_t)n));
    AMG_CHECK(grow(&G->z0, &G->cap_z0, (size_t)n));
    const size_t cap_cnt = G->cap_cnt;
    AMG_CHECK(grow(&G->cnt, &G->cap_cnt, (size_t)na + 1));
    if (G->cap_cnt != cap_cnt || G->midway) AMG_CHECK(hipMemsetAsync(G->cnt, 0, sizeof(int) * G->cap_cnt, s));
    if (G->midway) AMG_CHECK(hipMemsetAsync(G->pflag, 0, 2 * sizeof(int), s));
    G->midway = 1;
    AMG_CHECK(grow(&G->start, &G->cap_start, (size_t)na + 1));
    AMG_CHECK(grow((char **)&G->scan_tmp, &G->cap_scan, lv_scan_temp_bytes((int64_t)na + 1)));
    hipLaunchKernelGGL(k_agg_key, g1(n), dim3(B), 0, s, n, x, g.bxmin0, g.bxmin1, Lx / Kx, Ly / Ky, Kx, Ky, G->agg,
                       G->cnt);
    AMG_CHECK(lv_exclusive_scan_i32(G->cnt, G->start, (int64_t)na + 1, nullptr, G->scan_tmp, s));
    AMG_CHECK(lv_fail_here(&G->fail_at, LV_FAIL_AMG_COUNTS));
    hipLaunchKernelGGL(k_agg_fill, g1(n), dim3(B), 0, s, n, (const int *)G->agg, (const int *)G->start, G->cnt,
                       G->list);
    AMG_CHECK(level_alloc(G->lev[1], Kx, Ky));
    hipLaunchKernelGGL(k_agg_sort, g1(na), dim3(B), 0, s, na, (const int *)G->start, G->list);
    // fine smoother
    G->fine_learned = (mval && mdg) ? 1 : 0;
    G->mval = mval;
    G->mdg = mdg;
    G->fine_scale = OMEGA;
    // the aggregate order: the rows of each level-1 cell consecutive (list, sorted within a cell)
    G->perm_ok = 0;
    G->nbfuse = 0;
    G->z0_in = 0;
    const bool aggregate = layout == 0 || layout >= 2;
    const int nbf = n / FUSE_ROWS + 1;
    if (aggregate) {
        const size_t m = (size_t)LV_MAXE * n;
        AMG_CHECK(grow(&G->iperm, &G->cap_iperm, (size_t)n));
        AMG_CHECK(grow(&G->aggp, &G->cap_aggp, (size_t)n));
        AMG_CHECK(grow(&G->pdeg, &G->cap_pdeg, (size_t)n));
        AMG_CHECK(grow(&G->poff, &G->cap_poff, m));
        AMG_CHECK(grow(&G->pev32, &G->cap_pev32, m));
        AMG_CHECK(grow(&G->pev16, &G->cap_pev16, m));
        const size_t mo = ((size_t)n / 64 + 1) * LV_OVF_CAP;
        AMG_CHECK(grow(&G->ooff, &G->cap_ooff, mo));
        AMG_CHECK(grow(&G->oev32, &G->cap_oev32, mo));
        // (below 65536 rows launches, not the padding, set the kernels' time: no compact copy)
        G->ovf_cap = (layout == 0 && n >= 65536) ? LV_OVF_CAP : layout == 3 ? 16 : 0;
        AMG_CHECK(grow(&G->pdiag32, &G->cap_pdiag32, (size_t)n));
        AMG_CHECK(grow(&G->pdinv32, &G->cap_pdinv32, (size_t)n));
        if (G->fine_learned) {
            AMG_CHECK(grow(&G->pmval, &G->cap_pmval, m));
            AMG_CHECK(grow(&G->pmdg, &G->cap_pmdg, (size_t)n));
        }
        hipLaunchKernelGGL(k_perm_index, g1(n), dim3(B), 0, s, n, (const int *)G->list, (const int *)G->agg, G->iperm,
                           G->aggp);
        hipLaunchKernelGGL(k_perm_ell, g1(n), dim3(B), 0, s, n, (const int *)G->list, (const int *)G->iperm,
                           (const int *)A.deg, (const int *)A.ecol, (const float *)A.ev32, (const float *)A.diag32,
                           (const float *)A.dinv32, G->fine_learned ? mval : nullptr,
                           G->fine_learned ? mdg : nullptr, G->pdeg, G->poff, G->pev32, G->pev16, G->pdiag32,
                           G->pdinv32, G->pmval, G->pmdg, G->pflag, G->ooff, G->oev32, G->ovf_cap);
        // the blocks of the fused down pass (Jacobi smoother)
        AMG_CHECK(grow(&G->bfirst, &G->cap_bfirst, 2 * ((size_t)nbf + 2)));
        hipLaunchKernelGGL(k_fuse_blocks, g1((int64_t)na + 1), dim3(B), 0, s, na, nbf, (const int *)G->start,
                           reinterpret_cast<int2 *>(G->bfirst), G->pflag);
        AMG_CHECK(lv_fail_here(&G->fail_at, LV_FAIL_AMG_LEVELS));
        AMG_CHECK(lv_mail_post(&G->mail, G->pflag, 2, 2, s));  // read when the coarse levels are launched
    }
    hipLaunchKernelGGL(k_coarse1, g1((int64_t)na * RL), dim3(B), 0, s, na, Kx, Ky, G->xper, G->yper,
                       (const int *)G->start, (const int *)G->list,
                       (const int *)G->agg, n, (const int *)A.deg, (const int *)A.ecol, (const double *)A.ev64,
                       (const double *)A.diag64, G->lev[1].d, G->lev[1].c, G->lev[1].dinv);
    int l = 1;
    while (G->lev[l].n > LV_AMG_DENSE_MAX && l < LV_AMG_MAXLEV) {
        const lv_amg_level &F = G->lev[l];
        AMG_CHECK(level_alloc(G->lev[l + 1], (F.Kx + CF - 1) / CF, (F.Ky + CF - 1) / CF));
        lv_amg_level &C = G->lev[l + 1];
        hipLaunchKernelGGL(k_coarsen, g1(C.n), dim3(B), 0, s, C.Kx, C.Ky, F.Kx, F.Ky, G->xper, G->yper,
                           (const float *)F.d, (const float *)F.c, C.d, C.c, C.dinv);
        l++;
    }
    if (G->lev[l].n > LV_AMG_DENSE_MAX) return hipErrorInvalidValue;
    G->nlev = l;
    // over-correction factors, the tail's first level and its program (a W-cycle for a singular
    // system, whose coarse levels carry no compressibility term to damp the smooth error)
    G->fine_alpha = G->lev[1].n > TAIL_MAX ? ALPHA_FINE : 1.0f;
    for (int k = 1; k <= G->nlev; k++)
        G->lev[k].alpha = (k < G->nlev && G->lev[k + 1].n > TAIL_MAX) ? ALPHA_COARSE : 1.0f;
    int lt = G->nlev;
    while (lt > 1 && G->lev[lt - 1].n <= TAIL_MAX) lt--;
    G->wcycle = A.singular ? 1 : 0;
    // the first level of the single-workgroup kernel: a singular system W-visits the levels of at most TAIL_MAX
    // cells, a nonsingular one may start a level earlier, or where its levels first fit (strips one cell wide)
    G->lk = lt;
    if (!G->wcycle) {
        while (G->lk > 1 && G->lev[G->lk - 1].n <= LDS_MAX) G->lk--;
        while (G->lk < G->nlev && tail_layout_of(G).total > TAIL_LDS) G->lk++;
    }
    const int lk = G->lk;
    G->nprog = tail_program(lk, G->nlev, G->wcycle != 0, G->hprog);
    const tail_layout Y = tail_layout_of(G);
    G->tail_coef = Y.coef;
    G->tail_inv = Y.inv;
    G->tail_total = Y.total;
    // a singular system's tail as a matrix, and the level above it when it is small
    const bool mat = G->wcycle;
    G->lmat = mat && lk > 1 && G->lev[lk - 1].n <= MAT_MAX ? lk - 1 : lk;
    G->mat_ld = mat ? (G->lev[G->lmat].n + 3) & ~3 : 0;
    // pairs of levels above the tail that run as one kernel each way, from the tail upwards (the
    // smallest levels gain most): level l at least PAIR_MIN_K wide
    memset(G->pair, 0, sizeof(G->pair));
    for (int k = G->lmat - 2; k >= 2;) {
        const lv_amg_level &L = G->lev[k];
        const bool ok = L.Kx >= PAIR_MIN_K && L.Ky >= PAIR_MIN_K;
        const bool odd = (G->xper && L.Kx % 4 != 0) || (G->yper && L.Ky % 4 != 0);
        G->pair[k] = ok ? (odd ? 2 : 1) : 0;
        k -= ok ? 2 : 1;
    }
    tail_tables H;
    for (int k = 0; k < G->nprog; k++) H.prog[k] = (uint8_t)G->hprog[k];
    tail_descriptors(G, Y, H.desc);
    hipLaunchKernelGGL(k_tail_put, dim3(1), dim3(TB), 0, s, H, G->nprog, G->prog, G->desc);
    const lv_amg_level &D = G->lev[l];
    hipLaunchKernelGGL(k_dense_inverse, dim3(1), dim3(DTB), 0, s, D.Kx, D.Ky, G->xper, G->yper, (const float *)D.d,
                       (const float *)D.c, A.singular, G->dense_inv);
    const bool lds = Y.total <= TAIL_LDS;
    if (lds)
        hipLaunchKernelGGL(k_tail_pack, dim3(64), dim3(B), 0, s, tail_levels_of(G), Y, (const float *)G->dense_inv,
                           G->tail_img);
    if (mat) {
        const int nt = G->lev[lk].n, ldt = (nt + 3) & ~3;
        AMG_CHECK(grow(&G->tail_mat, &G->cap_tail_mat, (size_t)nt * ldt));
        if (lds) {
            hipLaunchKernelGGL(k_tail_lds<true>, dim3(nt), dim3(TB), 0, s, tail_args_of(G),
                               (const lv_cg_scalars *)nullptr, G->tail_mat, ldt);
        } else {
            tail_levels T = tail_levels_of(G);
            size_t stride = 0;
            for (int k = lk; k <= G->nlev; k++) stride += 4 * (size_t)G->lev[k].n;
            AMG_CHECK(grow(&G->tail_work, &G->cap_tail_work, stride * nt));
            float *w = G->tail_work;
            for (int k = lk; k <= G->nlev; k++)
                for (float **p : {&T.r[k], &T.z[k], &T.t[k], &T.acc[k]}) {
                    *p = w;
                    w += G->lev[k].n;
                }
            hipLaunchKernelGGL(k_tail_columns, dim3(nt), dim3(TB), 0, s, T, (const int *)G->prog, G->nprog,
                               (const float *)G->dense_inv, (int)stride, G->tail_mat, ldt);
        }
        G->mat = G->tail_mat;
        if (G->lmat < lk) {
            const lv_amg_level &L = G->lev[G->lmat];
            AMG_CHECK(grow(&G->ext_mat, &G->cap_ext_mat, (size_t)L.n * G->mat_ld));
            hipLaunchKernelGGL(k_mat_extend, dim3((L.n + EXT_ROWS - 1) / EXT_ROWS), dim3(B), 0, s,
                               st_level{L.Kx, L.Ky, G->xper, G->yper, L.d, L.c, L.dinv, L.alpha}, G->lev[lk].Ky, nt,
                               (const float *)G->tail_mat, ldt, G->ext_mat, G->mat_ld);
            G->mat = G->ext_mat;
        }
    }
    if (aggregate) {
        int flags[2];
        AMG_CHECK(lv_mail_await(&G->mail, flags, 2, s));
        G->perm_ok = flags[0] ? 0 : 1;
        G->nbfuse = (G->perm_ok && !flags[1]) ? nbf : 0;
        G->z0_in = (G->nbfuse > 0 && !G->fine_learned) ? 1 : 0;
    }
    // the learned smoother's scale: lambda_max(M A) -> FINE_TARGET
    if (G->fine_learned) {
        AMG_CHECK(grow(&G->pv, &G->cap_pv, (size_t)n));
        AMG_CHECK(grow(&G->pu, &G->cap_pu, (size_t)n));
        G->fine_scale = 1.0f;
        double lam = 0.0;
        if (G->perm_ok)
            AMG_CHECK(power_lambda(G, fine_agg<lv_ell_agg32>(G, (const float *)G->pev32), G->list, &lam, s));
        else
            AMG_CHECK(power_lambda(G, fine_own(G, A), nullptr, &lam, s));
        G->fine_scale = (lam > 0.0 && lam == lam) ? (float)(FINE_TARGET / lam) : 0.0f;
        if (!(G->fine_scale > 0.0f)) {  // no usable estimate: damped Jacobi
            G->fine_learned = 0;
            G->fine_scale = OMEGA;
        }
    }
    AMG_CHECK(hipGetLastError());
    G->midway = 0;
    return hipSuccess;
}

// levels l and l+1 for the pair kernels
static st_pair st_pair_of(const lv_amg *G, int l)
{
    const lv_amg_level &A = G->lev[l], &C = G->lev[l + 1], &C2 = G->lev[l + 2];
    return st_pair{st_level{A.Kx, A.Ky, G->xper, G->yper, A.d, A.c, A.dinv, A.alpha},
                   st_level{C.Kx, C.Ky, G->xper, G->yper, C.d, C.c, C.dinv, C.alpha}, C2.Kx, C2.Ky};
}

// the cycle on a fine view F; agg: level-1 cell of each fine row; list: the fine rows of each cell
// (null when they are consecutive)
template <class V>
static hipError_t vcycle(const lv_amg *G, const fine_ops<V> &F, const int *agg, const int *list, const float *r,
                         float *z, double *Prr, const lv_cg_scalars *S, hipStream_t s, bool z0_ready,
                         const lv_cycle_head *head, const lv_cycle_update *update)
{
    const int n = G->n0;
    const lv_amg_level &L1 = G->lev[1];
    const bool pairs = !G->level_kernels;
    const int lt = G->lmat;  // the levels below it have kernels of their own
    bool z1_given = false;  // the fused down pass stored level 1's pre-smoothed z
    // level 0, down: z0 (in G->z0) and its residual t (in G->t0), restricted to level 1
    if (G->fine_learned) {
        hipLaunchKernelGGL(k_fine_pre<V>, g1(n), dim3(B), 0, s, F, r, G->z0, S);
        hipLaunchKernelGGL(k_fine_resid<V>, g1(n), dim3(B), 0, s, F, r, (const float *)G->z0, G->t0, S);
        hipLaunchKernelGGL(k_restrict1, g1((int64_t)G->na * RL), dim3(B), 0, s, G->na, (const int *)G->start, list,
                           (const float *)G->t0, L1.r, S);
    } else if (!list && G->nbfuse > 0) {
        // level 1 above the tail: its pre-smoothed z stored here, gathered by its down pass
        z1_given = lt > 1;
        float *z1 = z1_given ? L1.z : nullptr;
        const int *done = S ? &S->done : G->bfirst + 2 * (G->nbfuse + 1);
#define LV_DOWN_JR(Z0, HEAD)                                                                                     \
    hipLaunchKernelGGL((k_fine_down_jr<V, Z0, HEAD>), dim3(G->nbfuse), dim3(B), 0, s, F, r, G->z0,                 \
                       (const int *)G->start, reinterpret_cast<const int2 *>(G->bfirst), G->na, L1.r,              \
                       (const float *)L1.dinv, z1, done, head ? *head : lv_cycle_head{})
        const bool z0_in = z0_ready && G->z0_in;
        if (update)
            hipLaunchKernelGGL(k_fine_down_u<V>, dim3(G->nbfuse), dim3(B), 0, s, F, *update, G->z0, (const int *)G->start,
                               reinterpret_cast<const int2 *>(G->bfirst), G->na, L1.r, (const float *)L1.dinv, z1);
        else if (z0_in && head) LV_DOWN_JR(true, true);
        else if (z0_in) LV_DOWN_JR(true, false);
        else if (head) LV_DOWN_JR(false, true);
        else LV_DOWN_JR(false, false);
#undef LV_DOWN_JR
    } else {
        hipLaunchKernelGGL(k_fine_down_j<V>, g1(n), dim3(B), 0, s, F, r, G->z0, G->t0, S);
        hipLaunchKernelGGL(k_restrict1, g1((int64_t)G->na * RL), dim3(B), 0, s, G->na, (const int *)G->start, list,
                           (const float *)G->t0, L1.r, S);
    }
    // coarse levels above the tail, down: each level's pre-smoothed z and the next level's
    // right-hand side
    for (int l = 1; l < lt; l++) {
        const lv_amg_level &L = G->lev[l], &C = G->lev[l + 1];
        const st_level sl{L.Kx, L.Ky, G->xper, G->yper, L.d, L.c, L.dinv, L.alpha};
        if (pairs && G->pair[l]) {
            const lv_amg_level &C2 = G->lev[l + 2];
            const st_pair q = st_pair_of(G, l);
            hipLaunchKernelGGL(G->pair[l] == 2 ? k_st_down2<true> : k_st_down2<false>,
                               dim3((C2.Kx + PD - 1) / PD, (C2.Ky + PD - 1) / PD), dim3(B), 0, s, q,
                               (const float *)L.r, L.z, C.r, C.z, C2.r, S);
            l++;
            continue;
        }
        auto down = l > 1 || !z1_given ? k_st_down<false, false> : update ? k_st_down<true, true> : k_st_down<true, false>;
        hipLaunchKernelGGL(down, g1((int64_t)C.n * CF2), dim3(B), 0, s, sl, C.Ky, C.n, (const float *)L.r, L.z, C.r, S,
                           update ? *head : lv_cycle_head{});
    }
    // the tail: levels lt..nlev down, dense, and up, or the matrix of that; the final correction of level
    // lt in its t.  Then the coarse levels above it, up: each level's final correction in t; level 1 in the
    // aggregate order with the Jacobi smoother also prolongates into z0.
    const lv_amg_level &LT = G->lev[lt];
    const bool prolong_in_up = (lt > 1 || G->mat_ld) && !G->fine_learned && list == nullptr;
    if (G->mat_ld) {
        const bool pr = lt == 1 && prolong_in_up;
        const bool hd = update && lt == 1;  // (the update comes with pr there)
        constexpr int PT = TAIL_MAX / 256, PM = MAT_MAX / 256;
        auto kern = LT.n <= TAIL_MAX ? (hd   ? k_mat_mv<PT, true, true>
                                        : pr ? k_mat_mv<PT, true, false>
                                             : k_mat_mv<PT, false, false>)
                                     : (hd   ? k_mat_mv<PM, true, true>
                                        : pr ? k_mat_mv<PM, true, false>
                                             : k_mat_mv<PM, false, false>);
        hipLaunchKernelGGL(kern, dim3((LT.n + B / 64 - 1) / (B / 64)), dim3(B), 0, s, LT.n, G->mat_ld,
                           (const float *)G->mat, (const float *)LT.r, LT.t, S,
                           pr ? (const int *)G->start : (const int *)nullptr, G->fine_alpha, G->z0,
                           hd ? *head : lv_cycle_head{});
    } else
        hipLaunchKernelGGL(k_tail_lds<false>, dim3(1), dim3(TB), 0, s, tail_args_of(G), S, (float *)nullptr, 0);
    for (int l = lt - 1; l >= 1; l--) {
        if (pairs && l >= 3 && G->pair[l - 1]) {
            const lv_amg_level &L = G->lev[l - 1], &C = G->lev[l], &C2 = G->lev[l + 1];
            hipLaunchKernelGGL(G->pair[l - 1] == 2 ? k_st_up2<true> : k_st_up2<false>,
                               dim3((L.Kx + PU - 1) / PU, (L.Ky + PU - 1) / PU), dim3(B), 0, s,
                               st_pair_of(G, l - 1), (const float *)L.r, (const float *)L.z, (const float *)C.r,
                               (const float *)C.z, (const float *)C2.t, L.t, S);
            l--;
            continue;
        }
        const lv_amg_level &L = G->lev[l], &C = G->lev[l + 1];
        const st_level sl{L.Kx, L.Ky, G->xper, G->yper, L.d, L.c, L.dinv, L.alpha};
        if (l == 1 && prolong_in_up)
            hipLaunchKernelGGL(k_st_up<true>, g1(L.n), dim3(B), 0, s, sl, C.Ky, (const float *)L.r,
                               (const float *)L.z, (const float *)C.t, L.t, S, (const int *)G->start, G->fine_alpha,
                               G->z0);
        else
            hipLaunchKernelGGL(k_st_up<false>, g1(L.n), dim3(B), 0, s, sl, C.Ky, (const float *)L.r,
                               (const float *)L.z, (const float *)C.t, L.t, S, (const int *)nullptr, 0.0f,
                               (float *)nullptr);
    }
    // level 0, up: prolongation, residual and post-smoothing; partials of r.z, r.r
    if (G->fine_learned) {
        hipLaunchKernelGGL(k_fine_up<V>, g1(n), dim3(B), 0, s, F, r, (const float *)G->z0, agg, (const float *)L1.t,
                           z, G->t0, S);
        hipLaunchKernelGGL(k_fine_post<V>, dim3(lv_nblocks(n)), dim3(B), 0, s, F, r, (const float *)G->t0, z, Prr, S);
    } else {
        if (!prolong_in_up)
            hipLaunchKernelGGL(k_prolong1, g1((n + PROLONG_RPT - 1) / PROLONG_RPT), dim3(B), 0, s, n, agg,
                               (const float *)L1.t, G->fine_alpha, G->z0, S);
        if constexpr (std::is_same<V, lv_ell_agg16>::value) {
            if (n > LV_NT_ROWS) {
                typedef decltype(lv_ell_streamed(F.A)) VS;
                const fine_ops<VS> FS{F.n, lv_ell_streamed(F.A), F.diag, F.dinv, F.mval, F.mdg, F.scale, F.alpha};
                hipLaunchKernelGGL(k_fine_up_j<VS>, dim3(lv_nblocks(n)), dim3(B), 0, s, FS, r, (const float *)G->z0, z,
                                   Prr, S);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL(k_fine_up_j<V>, dim3(lv_nblocks(n)), dim3(B), 0, s, F, r, (const float *)G->z0, z, Prr, S);
    }
    return hipGetLastError();
}

hipError_t lv_amg_vcycle(const lv_amg *G, const lv_pressure_system &A, const float *r, float *z, double *Prr,
                         const lv_cg_scalars *S, hipStream_t s, bool z0_ready, const lv_cycle_head *head,
                         const lv_cycle_update *update)
{
    if (G->perm_ok)
        return vcycle(G, fine_agg<lv_ell_agg16>(G, (const uint16_t *)G->pev16), (const int *)G->aggp,
                      (const int *)nullptr, r, z, Prr, S, s, z0_ready, head, update);
    return vcycle(G, fine_own(G, A), (const int *)G->agg, (const int *)G->list, r, z, Prr, S, s, false, nullptr, nullptr);
}

// The test in the down pass adds 0.5 us to it at 131,072 and 265,225 rows and 1.0 at 1,000,000, for a launch of 2.6 us
// and its gap; at 4,194,304 rows 8.2 for a launch of 4.8.  The line (2 M rows) lies between, in what the workgroups
// read together.
static constexpr int64_t HEAD_MAX = 1ll << 23;
bool lv_amg_takes_head(const lv_amg *G, int nb)
{
    return G->perm_ok && !G->fine_learned && G->nbfuse > 0 && (int64_t)G->nbfuse * nb <= HEAD_MAX;
}

// With the update in the down pass an iteration's part up to level 1's own takes 12.1 us for 14.5 (and a gap
// between launches less) at 10,000 rows, 11.8 for 13.7 at 131,072, 14.9 for 16.1 at 265,225, and 28.7 for 28.0 at
// 1,000,000, where the neighbours' second and third gather count; a sweep that has converged pays for one down pass.
static constexpr int UPDATE_MAX = 1 << 19;
bool lv_amg_takes_update(const lv_amg *G)
{
    // (the kernel behind the down pass makes the convergence test: a stencil level, or the matrix as level 1)
    return G->perm_ok && G->z0_in && G->n0 <= UPDATE_MAX && G->nbfuse <= 2 * LV_NBMAX && (G->lmat > 1 || G->mat_ld);
}
