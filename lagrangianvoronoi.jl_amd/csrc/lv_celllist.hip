// lv_celllist.hip -- cell-list rebuild: CellList insert!/insert_periodic! (src/neighborlist.jl:47-67,
// src/voronoigrid.jl:130-147) as a counting sort over the cells.
//
// The reference pushes label i (and up to 8 periodic images) into FastVector cells in label order,
// so each cell holds its labels in ascending order.  Here the images of every seed are counted per
// cell with atomics, the counts are scanned, every image takes a slot of its cell (again by an
// atomic, so in no fixed order) and is then ranked among the few labels of its cell: the rank is its
// place, so the list is the reference's whatever order the atomics ran in.
//
// Bound by launches below some 10^5 seeds, by the atomics above.  Six launches (four up to 16384
// cells) and nothing that the host waits for; a radix sort of the cell ids took 16 to 21 launches and a read of the
// item count in the middle.
#include "lv_internal.h"

#include <climits>

namespace {

constexpr int B = 256;

// In-grid images of seed x in insert_periodic! order; returns how many, writes their cell ids.
// the keys of a seed and of its periodic images, in the order insert_periodic! visits them.  An
// image's coordinate is x1, x1 + P or x1 - P (and x2, x2 + Q or x2 - Q; the reference's
// zero-weighted terms add 0.0, which changes no floor), so the exact divisions of findkey are made
// once per distinct coordinate: 6 instead of 18
__device__ __forceinline__ bool lv_key_axis(double x, double origin, double h, int nmax, int &i)
{
    const double f = floor((x - origin) / h);
    if (!(f == f) || f < -2.0e9 || f > 2.0e9) return false;
    i = (int)f + 1;
    return i >= 1 && i <= nmax;
}

__device__ __forceinline__ int seed_images(const lv_grid_params &g, double x1, double x2, int *cells)
{
    const double P = g.xperiod, Q = g.yperiod;
    int ix[3], iy[3];
    bool ox[3], oy[3];
    ox[0] = lv_key_axis(x1, g.origin0, g.h, g.n1, ix[0]);
    oy[0] = lv_key_axis(x2, g.origin1, g.h, g.n2, iy[0]);
    ox[1] = ox[2] = oy[1] = oy[2] = false;
    if (g.xperiodic) {
        ox[1] = lv_key_axis(x1 + P * 1.0, g.origin0, g.h, g.n1, ix[1]);
        ox[2] = lv_key_axis(x1 - P * 1.0, g.origin0, g.h, g.n1, ix[2]);
    }
    if (g.yperiodic) {
        oy[1] = lv_key_axis(x2 + Q * 1.0, g.origin1, g.h, g.n2, iy[1]);
        oy[2] = lv_key_axis(x2 - Q * 1.0, g.origin1, g.h, g.n2, iy[2]);
    }
    // (a, b): the image's x and y variants, in the order of the reference's image list
    int pa[9], pb[9], k = 0;
    pa[k] = 0; pb[k] = 0; k++;
    if (g.xperiodic) {
        pa[k] = 1; pb[k] = 0; k++;
        pa[k] = 2; pb[k] = 0; k++;
    }
    if (g.yperiodic) {
        pa[k] = 0; pb[k] = 1; k++;
        pa[k] = 0; pb[k] = 2; k++;
    }
    if (g.xperiodic && g.yperiodic) {
        pa[k] = 1; pb[k] = 1; k++;
        pa[k] = 1; pb[k] = 2; k++;
        pa[k] = 2; pb[k] = 1; k++;
        pa[k] = 2; pb[k] = 2; k++;
    }
    int m = 0;
    for (int j = 0; j < k; j++)
        if (ox[pa[j]] && oy[pb[j]]) cells[m++] = (ix[pa[j]] - 1) + (iy[pb[j]] - 1) * g.n1;
    return m;
}

// cnt[c] += images in cell c.  Consecutive seeds mostly share a cell, so one atomic serves a run of
// them; the periodic images, few, take one each.
__global__ __launch_bounds__(B) void k_img_count(lv_grid_params g, int n, const double *__restrict__ x,
                                                 int *__restrict__ cnt)
{
    const int i = blockIdx.x * B + threadIdx.x;
    int cells[9];
    const int m = i < n ? seed_images(g, x[i], x[n + i], cells) : 0;
    (void)lv_run_atomic_add<1>(cnt, m > 0 ? cells[0] : 0, m > 0);
    for (int j = 1; j < m; j++) atomicAdd(&cnt[cells[j]], 1);
}

// every image into a slot of its cell; leaves cnt at zero for the next build
__global__ __launch_bounds__(B) void k_img_fill(lv_grid_params g, int n, const double *__restrict__ x,
                                                int *__restrict__ cnt, const int *__restrict__ cell_start,
                                                int2 *__restrict__ items, int64_t cap)
{
    const int i = blockIdx.x * B + threadIdx.x;
    int cells[9];
    const int m = i < n ? seed_images(g, x[i], x[n + i], cells) : 0;
    int slot = lv_run_atomic_add<-1>(cnt, m > 0 ? cells[0] : 0, m > 0);
    for (int j = 0; j < m; j++) {
        if (j > 0) slot = atomicAdd(&cnt[cells[j]], -1) - 1;
        const int64_t o = (int64_t)cell_start[cells[j]] + slot;
        if (o < cap) items[o] = make_int2(cells[j], i);
    }
}

// Every item to its place: the labels of its cell that are smaller (two images of one seed in one
// cell are alike and go by slot).  A thread per item, so that a crowded cell is ranked by as many
// threads as it has items.  The seed's position goes along, so the clipper reads candidate label and
// position from one run (cell_x holds two planes of stride cap).
__global__ __launch_bounds__(B) void k_cell_rank(const int *__restrict__ nitems, const int2 *__restrict__ items,
                                                 const int *__restrict__ cell_start, int *__restrict__ cell_labels,
                                                 double *__restrict__ cell_x, const double *__restrict__ x, int n,
                                                 int64_t cap)
{
    const int p = blockIdx.x * B + threadIdx.x;
    const int m = *nitems;
    if (p >= m || p >= cap) return;
    const int2 it = items[p];
    const int s0 = cell_start[it.x], s1 = cell_start[it.x + 1];
    int at = s0;
    for (int q = s0; q < s1; q++) {
        const int l = items[q].y;
        at += (l < it.y) || (l == it.y && q < p);
    }
    cell_labels[at] = it.y;
    cell_x[at] = x[it.y];
    cell_x[cap + at] = x[n + it.y];
}

__global__ void k_fill_i32(int *p, int64_t n, int v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace

// temp layout: [cnt: ncells + 1 ints, zero between builds][scan temp][items: max_items int2]
static size_t cell_cnt_bytes(int64_t ncells) { return ((size_t)(ncells + 1) * 4 + 255) & ~(size_t)255; }
static size_t cell_scan_bytes(int64_t ncells) { return (lv_scan_temp_bytes(ncells + 1) + 255) & ~(size_t)255; }

size_t lv_celllist_temp_bytes(int64_t max_items, int64_t ncells)
{
    return cell_cnt_bytes(ncells) + cell_scan_bytes(ncells) + (size_t)max_items * sizeof(int2);
}

hipError_t lv_celllist_temp_init(void *temp, int64_t ncells, hipStream_t s)
{
    const int64_t k = ncells + 1;
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((k + 255) / 256)), dim3(256), 0, s, (int *)temp, k, 0);
    return hipGetLastError();
}

// The cell list of n seeds, built in two parts without waiting for either.  The first counts: cell_start, and in
// d_nitems the item count.  If that exceeds max_items the list is cut off there (cell_start never points beyond
// it): the caller, who reads the count with its next flags, throws it away and builds again with more room.
hipError_t lv_count_cells(const lv_grid_params &g, int n, const double *x, int *cell_start, int64_t max_items,
                          int *d_nitems, void *temp, hipStream_t s)
{
    const int64_t ncells = (int64_t)g.n1 * g.n2;
    int *cnt = (int *)temp;
    void *scan_tmp = (char *)temp + cell_cnt_bytes(ncells);
    if (n > 0) hipLaunchKernelGGL(k_img_count, dim3((n + B - 1) / B), dim3(B), 0, s, g, n, x, cnt);
    return lv_exclusive_scan_i32(cnt, cell_start, ncells + 1, d_nitems, scan_tmp, s,
                                 (int)(max_items < INT_MAX ? max_items : INT_MAX));
}

// The second fills, and leaves the counters at zero.
hipError_t lv_fill_cells(const lv_grid_params &g, int n, const double *x, const int *cell_start, int *cell_labels,
                         double *cell_x, int64_t max_items, const int *d_nitems, void *temp, hipStream_t s)
{
    const int64_t ncells = (int64_t)g.n1 * g.n2;
    int *cnt = (int *)temp;
    int2 *items = (int2 *)((char *)temp + cell_cnt_bytes(ncells) + cell_scan_bytes(ncells));
    if (n > 0) {
        hipLaunchKernelGGL(k_img_fill, dim3((n + B - 1) / B), dim3(B), 0, s, g, n, x, cnt, cell_start,
                           items, max_items);
        hipLaunchKernelGGL(k_cell_rank, dim3((unsigned)((max_items + B - 1) / B)), dim3(B), 0, s,
                           d_nitems, (const int2 *)items, cell_start, cell_labels, cell_x, x, n, max_items);
    }
    return hipGetLastError();
}
