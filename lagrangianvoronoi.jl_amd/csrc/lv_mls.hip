// lv_mls.hip -- nearest_polygon (src/voronoigrid.jl:154-178), movingls with the Gaussian kernel
// (src/movingls.jl:41-96) and point_value (:140-145), a group of G lanes per query or per polygon.
//
// The walks go over the cell list of the last remesh (periodic images included, as the reference's
// cells hold them), each candidate taken at its own seed position q.x:
//   * nearest_polygon measures |q.x - x|^2 without a minimum image, walks the magic path in order and
//     stops at the first node whose rr exceeds the best distance found.  A group takes G nodes at a
//     time, one per lane, and an exclusive prefix minimum over the lanes tells which of them the
//     sequential walk would have reached, so index and ties are the sequential walk's;
//   * movingls takes y = p.x + get_arrow(q.x, p.x) and, in the reference, stops at the first node with
//     rr > h (it compares the squared node bound with h itself).  Only candidates with |y - p.x| < h
//     contribute, and a cell with rr > h^2 holds none unless it lists one of them a second time through
//     another periodic image, which takes a period shorter than r_max + h and two cells.  The host
//     therefore limits the walk to rr <= h^2 (with a margin for rounding: on a regular lattice, seeds
//     at the distance h exactly are the rule) where the periods are longer than that, and keeps the
//     reference's bound where they are not (mls_walk_limit).  At h = 2 dr that is 21 cells instead of
//     the 100 and more within r_max.
// What bounds them is the chain of dependent loads of a walk (path node, cell bounds, positions, values)
// and FP64 work, not bytes.  One thread per query or polygon and the whole walk took 2152 us for 200,003
// point_values on 512^2 seeds and 260 us for 317 x 251 quadratic expansions at h = 3 dr; these take 152 us
// and 46 us with 4 lanes each (2 lanes 207 and 145 us, 8 lanes 154 and 62, 16 lanes 183 and 93).
// The cells of a grid row within the bound are consecutive, and so are their candidates in the cell
// list, which carries each label's position next to it: a group reads row by row, its lanes taking
// consecutive candidates.  The sums a = sum w (f(q) - f(p)) dx and R = sum w dx dx^T (symmetric: one
// triangle) accumulate per lane in FP64 and are added over the group in a fixed order; the 2x2 system is
// solved by Cramer's rule, the 5x5 and 9x9 ones by Gaussian elimination with partial pivoting.
#include "lv_internal.h"

namespace {

constexpr int B = 256;

struct mls_args {
    lv_grid_params g;
    const double *x;
    int n;
    const int *cell_start, *cell_labels;
    const double *cell_x;  // positions of the cell list's items, two planes of stride ldx
    int64_t ldx;
    const int *path_i;
    const double *path_rr;
};

// sum of v over the G lanes of a group (G a power of two, at most 64), the same in every lane
template <int G>
__device__ __forceinline__ double group_sum(double v)
{
#pragma unroll
    for (int o = 1; o < G; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// the bits of a group's lanes in a ballot of its wavefront
template <int G>
__device__ __forceinline__ unsigned long long group_bits(unsigned long long m)
{
    const int at = (threadIdx.x & 63) & ~(G - 1);
    return (m >> at) & ((G == 64) ? ~0ull : ((1ull << G) - 1));
}

// nearest_polygon by a group of G lanes (lane l of it): the index of the nearest seed, -1 if the path
// prefix ends before the search does; the same in every lane
template <int G>
__device__ int nearest(const mls_args &A, int l, double q1, double q2)
{
    const lv_grid_params &g = A.g;
    int k1, k2;
    lv_findkey(g, q1, q2, k1, k2);
    if (k1 < 0) return -1;
    double best = __builtin_inf();
    int ib = -1;
    for (int base = 0; base < g.npath; base += G) {
        const int k = base + l;
        double lb = __builtin_inf(), rrk = __builtin_inf();
        int lj = -1;
        if (k < g.npath) {
            rrk = A.path_rr[k];
            const int c1 = k1 + A.path_i[2 * k], c2 = k2 + A.path_i[2 * k + 1];
            if (!(rrk > best) && c1 >= 1 && c1 <= g.n1 && c2 >= 1 && c2 <= g.n2) {
                const int c = (c1 - 1) + (c2 - 1) * g.n1;
                const int s1 = A.cell_start[c + 1];
                for (int s = A.cell_start[c]; s < s1; s++) {
                    const double a = A.cell_x[s] - q1, b = A.cell_x[A.ldx + s] - q2;
                    const double rr = a * a + b * b;
                    if (rr < lb) {
                        lb = rr;
                        lj = s;
                    }
                }
            }
        }
        // eb: the best distance the sequential walk holds when it comes to this lane's node
        double pm = lb;  // inclusive prefix minimum
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const double t = __shfl_up(pm, o, G);
            if (l >= o) pm = fmin(pm, t);
        }
        double eb = __shfl_up(pm, 1, G);
        eb = (l == 0) ? best : fmin(best, eb);
        const bool reached = k < g.npath && !(rrk > eb);
        if (!reached) lb = __builtin_inf();
        double m = lb;
#pragma unroll
        for (int o = 1; o < G; o <<= 1) m = fmin(m, __shfl_xor(m, o, G));
        if (m < best) {
            // the first lane (path order) that holds the minimum
            const unsigned long long at = group_bits<G>(__ballot(lb == m));
            best = m;
            ib = __shfl(lj, __ffsll((long long)at) - 1, G);
        }
        if (group_bits<G>(__ballot(k < g.npath && !reached)) != 0) return ib < 0 ? -1 : A.cell_labels[ib];
    }
    if (g.has_next && !(g.next_rr > best)) return -1;  // the walk would go on
    return ib < 0 ? -1 : A.cell_labels[ib];
}

template <int N>
__device__ __forceinline__ void power_vector(double d1, double d2, double (&p)[N])
{
    p[0] = d1;
    p[1] = d2;
    if (N >= 5) {
        p[2] = d1 * d1;
        p[3] = d1 * d2;
        p[4] = d2 * d2;
    }
    if (N >= 9) {
        p[5] = (d1 * d1) * d1;
        p[6] = (d1 * d1) * d2;
        p[7] = (d1 * d2) * d2;
        p[8] = (d2 * d2) * d2;
    }
}

// movingls(T, grid, p, fun; h) for polygon i and the scalar field f by a group of G lanes: the N Taylor
// coefficients, the same in every lane.  The walk takes the cells with rr <= lim (mls_walk_limit).
//
// With LIST, a lane first collects the candidates within h (about a quarter of the cells') in its LDS
// column and works them off when the column is full and at the end: the weight and the sums (an exp and
// N + N (N + 1) / 2 multiply-adds) then run for nearly full wavefronts, not once per candidate that any
// of its lanes keeps.  (For point_value, whose sums are five numbers, the list costs more than it saves:
// 165 against 152 us.)
constexpr int LCAP = 12;

template <int N, int G, bool LIST>
__device__ __forceinline__ void movingls_at(const mls_args &A, int l, const double *__restrict__ f, double h,
                                            double lim, int i, double (&a)[N], int (*list)[B])
{
    const lv_grid_params &g = A.g;
    const double x1 = A.x[i], x2 = A.x[A.n + i];
    const double fp = f[i];
    constexpr int NT = N * (N + 1) / 2;
    double T[NT];
#pragma unroll
    for (int r = 0; r < N; r++) a[r] = 0.0;
#pragma unroll
    for (int r = 0; r < NT; r++) T[r] = 0.0;
    // gaussian_kernel(h, r) = exp(-0.5 (r/h)^2) / sqrt(2 pi h^2), src/movingls.jl:22-24
    const double norm = sqrt((2.0 * 3.141592653589793) * (h * h));
    const double hh = h * h * (1.0 + 1e-12);
    auto offset = [&](int s, double &y1, double &y2, double &rr) {
        lv_arrow_target(g, A.cell_x[s], A.cell_x[A.ldx + s], x1, x2, y1, y2);
        const double e1 = x1 - y1, e2 = x2 - y2;
        rr = e1 * e1 + e2 * e2;
    };
    auto add = [&](int s) {
        double y1, y2, rr;
        offset(s, y1, y2, rr);
        const double r = sqrt(rr);
        if ((x1 == y1 && x2 == y2) || !(r < h)) return;
        const double q = r / h;
        const double w = exp(-0.5 * (q * q)) / norm;
        const double df = f[A.cell_labels[s]] - fp;
        double dx[N];
        power_vector<N>(y1 - x1, y2 - x2, dx);
        int o = 0;
#pragma unroll
        for (int q = 0; q < N; q++) {
            a[q] += (w * df) * dx[q];
            const double wd = w * dx[q];
#pragma unroll
            for (int t = q; t < N; t++) T[o++] += wd * dx[t];
        }
    };
    int cnt = 0;
    int k1, k2;
    lv_findkey(g, x1, x2, k1, k2);
    const double gh = g.h * g.h;
    int K = 0;  // rows of cells on each side that the bound reaches
    while (K + 1 < g.n2 && gh * (double)((long long)K * K) <= lim) K++;
    for (int d0 = -K; d0 <= K; d0 += G) {
        // lane r of the group takes the item range of row d0 + r: the cells |i1| - 1 <= a with
        // h^2 (a^2 + b^2) <= lim
        int s0 = 0, s1 = 0;
        const int d = d0 + l;
        const int c2 = k2 + d;
        if (d <= K && c2 >= 1 && c2 <= g.n2) {
            const long long b = d < 0 ? -d - 1 : (d > 0 ? d - 1 : 0);
            long long w = (long long)sqrt(fmax(0.0, lim / gh - (double)(b * b)));
            while (gh * (double)((w + 1) * (w + 1) + b * b) <= lim) w++;
            while (w >= 0 && gh * (double)(w * w + b * b) > lim) w--;
            if (w >= 0) {
                const int lo = (int)max(1ll, k1 - (w + 1)), hi = (int)min((long long)g.n1, k1 + (w + 1));
                if (lo <= hi) {
                    const int c = (c2 - 1) * g.n1 - 1;
                    s0 = A.cell_start[c + lo];
                    s1 = A.cell_start[c + hi + 1];
                }
            }
        }
        const int rows = min(G, K - d0 + 1);
        for (int r = 0; r < rows; r++) {
            const int e = __shfl(s1, r, G);
            for (int s = __shfl(s0, r, G) + l; s < e; s += G) {
                double y1, y2, rr;
                offset(s, y1, y2, rr);
                if (!(rr < hh)) continue;
                if (LIST) {
                    list[cnt++][threadIdx.x] = s;
                    if (cnt == LCAP) {
                        for (int q = 0; q < LCAP; q++) add(list[q][threadIdx.x]);
                        cnt = 0;
                    }
                } else {
                    add(s);
                }
            }
        }
    }
    if (LIST)
        for (int q = 0; q < cnt; q++) add(list[q][threadIdx.x]);
#pragma unroll
    for (int r = 0; r < N; r++) a[r] = group_sum<G>(a[r]);
#pragma unroll
    for (int r = 0; r < NT; r++) T[r] = group_sum<G>(T[r]);
    double R[N][N];
    {
        int o = 0;
#pragma unroll
        for (int q = 0; q < N; q++)
#pragma unroll
            for (int t = q; t < N; t++) {
                R[q][t] = T[o];
                R[t][q] = T[o++];
            }
    }
    if (N == 2) {
        const double det = R[0][0] * R[1][1] - R[0][1] * R[1][0];
        const double b0 = a[0], b1 = a[1];
        a[0] = (R[1][1] * b0 - R[0][1] * b1) / det;
        a[1] = (R[0][0] * b1 - R[1][0] * b0) / det;
        return;
    }
    // Gaussian elimination with partial pivoting
#pragma unroll
    for (int p = 0; p < N; p++) {
        int m = p;
        double best = fabs(R[p][p]);
#pragma unroll
        for (int r = p + 1; r < N; r++)
            if (fabs(R[r][p]) > best) {
                best = fabs(R[r][p]);
                m = r;
            }
#pragma unroll
        for (int r = p + 1; r < N; r++)
            if (r == m) {
#pragma unroll
                for (int c = 0; c < N; c++) {
                    const double t = R[p][c];
                    R[p][c] = R[r][c];
                    R[r][c] = t;
                }
                const double t = a[p];
                a[p] = a[r];
                a[r] = t;
            }
#pragma unroll
        for (int r = p + 1; r < N; r++) {
            const double l = R[r][p] / R[p][p];
#pragma unroll
            for (int c = p; c < N; c++) R[r][c] -= l * R[p][c];
            a[r] -= l * a[p];
        }
    }
#pragma unroll
    for (int p = N - 1; p >= 0; p--) {
        double s = a[p];
#pragma unroll
        for (int c = p + 1; c < N; c++) s -= R[p][c] * a[c];
        a[p] = s / R[p][p];
    }
}

template <int N, int G>
__global__ __launch_bounds__(B) void k_movingls(mls_args A, const double *__restrict__ f, double h, double lim,
                                                double *__restrict__ out)
{
    __shared__ int list[LCAP][B];
    const int i = blockIdx.x * (B / G) + threadIdx.x / G, l = threadIdx.x & (G - 1);
    if (i >= A.n) return;  // whole groups
    double a[N];
    movingls_at<N, G, true>(A, l, f, h, lim, i, a, list);
#pragma unroll
    for (int q = 0; q < N; q++)
        if (q % G == l) out[(size_t)i * N + q] = a[q];
}

template <int G>
__global__ __launch_bounds__(B) void k_nearest(mls_args A, int m, const double *__restrict__ q, int *__restrict__ idx)
{
    const int t = blockIdx.x * (B / G) + threadIdx.x / G, l = threadIdx.x & (G - 1);
    if (t >= m) return;  // whole groups
    const int p = nearest<G>(A, l, q[t], q[m + t]);
    if (l == 0) idx[t] = p;
}

// point_value(grid, x, fun) = fun(p) + dot(L, x - p.x) with p the nearest polygon and L its linear
// expansion at h = grid.h; NaN where the nearest polygon is not found
template <int G>
__global__ __launch_bounds__(B) void k_point_value(mls_args A, int m, const double *__restrict__ q,
                                                   const double *__restrict__ f, double h, double lim,
                                                   double *__restrict__ out)
{
    const int t = blockIdx.x * (B / G) + threadIdx.x / G, l = threadIdx.x & (G - 1);
    if (t >= m) return;  // whole groups
    const double q1 = q[t], q2 = q[m + t];
    const int p = nearest<G>(A, l, q1, q2);
    if (p < 0) {
        if (l == 0) out[t] = __builtin_nan("");
        return;
    }
    double L[2];
    movingls_at<2, G, false>(A, l, f, h, lim, p, L, nullptr);
    if (l == 0) out[t] = f[p] + (L[0] * (q1 - A.x[p]) + L[1] * (q2 - A.x[A.n + p]));
}

template <int G>
inline dim3 groups_for(int m)
{
    constexpr int per = B / G;
    return dim3((unsigned)((m + per - 1) / per > 0 ? (m + per - 1) / per : 1));
}

// The bound on rr of movingls' walk at kernel width h: the reference's min(h, rr_max), cut to h^2 where
// no candidate beyond can contribute.  A cell with rr > h^2 lists a seed within h only at another
// periodic image of it than the nearest one, i.e. at least a period less h away along that axis, while
// the walk reaches at most r_max and two cells.
double mls_walk_limit(const lv_grid_params &g, double h)
{
    const double full = h < g.rr_max ? h : g.rr_max;
    const double cut = h * h * (1.0 + 1e-9);
    const double reach = (g.r_max + 2.0 * g.h) * (1.0 + 1e-9);
    if ((g.xperiodic && !(g.xperiod - h > reach)) || (g.yperiodic && !(g.yperiod - h > reach))) return full;
    return cut < full ? cut : full;
}

// From this many queries on, four lanes each: sixteen lanes shorten a query's chain of dependent loads,
// which is what a small call waits for (100 queries: 9.5 us), but repeat more of its scalar work (200,003
// queries: 183 us against 152).  Calls with sixteen and with four: 38 and 46 us at 100 points, 57 and 65 at 8,000, 73 and 85
// at 16,000, 111 and 110 at 32,000, 131 and 127 at 40,000, 185 and 171 at 64,000.
constexpr int MANY_QUERIES = 32768;

}  // namespace

hipError_t lv_launch_movingls(const lv_grid_params &g, const double *x, int n, const int *cell_start,
                              const int *cell_labels, const double *cell_x, int64_t ldx, const int *path_i,
                              const double *path_rr, int order, const double *f, double h, double *out, hipStream_t s)
{
    const mls_args A{g, x, n, cell_start, cell_labels, cell_x, ldx, path_i, path_rr};
    if (n <= 0) return hipSuccess;
    const double lim = mls_walk_limit(g, h);
    if (order == 1) hipLaunchKernelGGL((k_movingls<2, 4>), groups_for<4>(n), dim3(B), 0, s, A, f, h, lim, out);
    else if (order == 2) hipLaunchKernelGGL((k_movingls<5, 4>), groups_for<4>(n), dim3(B), 0, s, A, f, h, lim, out);
    else if (order == 3) hipLaunchKernelGGL((k_movingls<9, 4>), groups_for<4>(n), dim3(B), 0, s, A, f, h, lim, out);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t lv_launch_nearest(const lv_grid_params &g, const double *x, int n, const int *cell_start,
                             const int *cell_labels, const double *cell_x, int64_t ldx, const int *path_i,
                             const double *path_rr, int m, const double *q, int *idx, hipStream_t s)
{
    const mls_args A{g, x, n, cell_start, cell_labels, cell_x, ldx, path_i, path_rr};
    if (m <= 0) return hipSuccess;
    if (m < MANY_QUERIES) hipLaunchKernelGGL(k_nearest<16>, groups_for<16>(m), dim3(B), 0, s, A, m, q, idx);
    else hipLaunchKernelGGL(k_nearest<4>, groups_for<4>(m), dim3(B), 0, s, A, m, q, idx);
    return hipGetLastError();
}

hipError_t lv_launch_point_value(const lv_grid_params &g, const double *x, int n, const int *cell_start,
                                 const int *cell_labels, const double *cell_x, int64_t ldx, const int *path_i,
                                 const double *path_rr, int m, const double *q, const double *f, double h, double *out,
                                 hipStream_t s)
{
    const mls_args A{g, x, n, cell_start, cell_labels, cell_x, ldx, path_i, path_rr};
    if (m <= 0) return hipSuccess;
    const double lim = mls_walk_limit(g, h);
    if (m < MANY_QUERIES)
        hipLaunchKernelGGL(k_point_value<16>, groups_for<16>(m), dim3(B), 0, s, A, m, q, f, h, lim, out);
    else hipLaunchKernelGGL(k_point_value<4>, groups_for<4>(m), dim3(B), 0, s, A, m, q, f, h, lim, out);
    return hipGetLastError();
}
