// lv_clip.hip -- Voronoi polygon construction by half-plane clipping: the cutting loop of remesh!
// (src/voronoigrid.jl:53-81, 89-108), voronoicut!(p, y, label) (src/polygon.jl:51-97), influence_rr
// (:101-107), sort_edges! (src/IO.jl:35-48) and the area/centroid read-outs (src/polygon.jl:114-122,
// 201-219), fused into one kernel.
//
// What bounds clipping is not bytes but chains of dependent FP64 operations and loads, and, once the device is
// full, the number of instructions.  Two ways to run it:
//   * a group of G = 16 lanes owns a seed, each lane one edge slot of its polygon in registers: a cut
//     evaluates every edge at once, and 16 candidates are loaded and tested at once.  The shortest
//     chain, for few seeds (lv_launch_clip), and for those that outgrow the other way's slots;
//   * one thread owns a seed, its polygon in LDS as five slot-major planes (v1x, v1y, v2x, v2y, label),
//     so lane t of the block addresses bank-conflict-free 8-byte words, and mirrored in registers for the
//     tests.  The fewest instructions, for many seeds.  Each polygon has CAP = 8 slots (18 KB per 64-seed
//     block, which holds a CU at 8 wavefronts), or 10 while the device holds them all at once (WIDE_MAX);
//     a seed whose polygon outgrows them (0.4% at a 2048^2 jittered lattice with eight, where no polygon
//     passes 10 edges while it is clipped) is queued and clipped again from the start by a group, so the
//     result is the same either way.
//
// The edge list keeps the reference's storage semantics exactly: cut edges are rewritten in place,
// deleted edges are replaced by the last edge (FastVector deleteat!, src/fastvector.jl:44-50) and
// re-tested, and the new edge is pushed last.  Every edge is tested once, in its original state, so a
// group tests all of them together; the deletions are then replayed on bit masks, which gives the
// order in which the sequential loop meets the edges (its last two crossings make the new edge) and the
// places the survivors move to.  With the same candidate order (magic path, then each cell's labels ascending) and
// IEEE FP64 without contraction, every vertex, label and edge position equals the reference's bit
// for bit.  Candidates come from the sorted cell list, which carries each label's seed position next
// to it.
#include "lv_internal.h"

namespace {

constexpr int GB = 256;             // lanes per block of the groups' kernel
constexpr int G = LV_MAXE;          // lanes of a group: one per edge slot
static_assert(G == 16, "a group is a row of 16 lanes");
constexpr int RETRY_BLOCKS = 1024;  // blocks over the queue (grid-stride)
constexpr int LCAP = 64;            // candidates of a group listed in LDS at a time
constexpr int CB = 64;              // seeds per block (one wavefront) with a thread per seed
constexpr double SIGNUM_EPS = 2.0 * 2.220446049250313e-16;  // 2*eps(Float64), src/polygon.jl:2

struct clip_lds {
    int s[GB / G][LCAP];              // candidates of a group: cell-list item,
    unsigned char q[GB / G][LCAP];    // and which of the current nodes it belongs to
    double term[GB / G][3][G];        // area and centroid terms by edge position
};

// The move in front of this remesh was refused (a NaN velocity), which the host learns with the remesh's own
// flags: the polygons, areas and centroids stay those of the last remesh.  err: as the kernel found it.
__device__ __forceinline__ bool move_refused(int err) { return err == LV_E_NAN_VELOCITY; }

__device__ __forceinline__ int signum(double v)
{
    if (v < -SIGNUM_EPS) return -1;
    if (v > SIGNUM_EPS) return 1;
    return 0;
}

// ---- a group of lanes per seed --------------------------------------------------------------------

// a group's lanes in a ballot of its wavefront
__device__ __forceinline__ unsigned group_ballot(bool p)
{
    return (unsigned)(__ballot(p) >> ((threadIdx.x & 63) & ~(G - 1))) & ((1u << G) - 1u);
}
// LDS written by a group's lanes, read by its other lanes: the wavefront's LDS operations are in order
__device__ __forceinline__ void lds_visible()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the polygon of a group: lane l holds edge l (l < len)
struct group_poly {
    double v1x, v1y, v2x, v2y;
    int lab, len;
};

// max of v and the value ROT lanes on in the row of 16 lanes (a register move, not the LDS crossbar)
template <int ROT>
__device__ __forceinline__ double row_max(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + ROT, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + ROT, 0xf, 0xf, true);
    return fmax(v, __hiloint2double(hi, lo));
}

__device__ __forceinline__ double group_influence_rr(const group_poly &P, int l, double x1, double x2)
{
    const double a = P.v1x - x1, b = P.v1y - x2;
    const double r = 4.0 * (a * a + b * b);
    const double m = (l < P.len && r > 0.0) ? r : 0.0;
    return row_max<1>(row_max<2>(row_max<4>(row_max<8>(m))));
}

// voronoicut!(p, y, label): 1 if an edge was added, 0 if not, -1 on overflow
__device__ __forceinline__ int group_cut(group_poly &P, int l, double x1, double x2, double y1, double y2, int label)
{
    const double d1 = y1 - x1, d2 = y2 - x2;
    const double m1 = 0.5 * (y1 + x1), m2 = 0.5 * (y2 + x2);
    const double c = d1 * m1 + d2 * m2;
    const double f1 = (d1 * P.v1x + d2 * P.v1y) - c;
    const double f2 = (d1 * P.v2x + d2 * P.v2y) - c;
    const int s1 = signum(f1), s2 = signum(f2);
    const int s12 = s1 + s2;
    const bool on = l < P.len;
    const bool cross = on && (0 <= s12 && s12 <= 1) && ((s1 | s2) != 0);
    const unsigned C = group_ballot(cross), D = group_ballot(on && 1 <= s12);
    if ((C | D) == 0) return 0;
    double X1 = 0.0, X2 = 0.0;
    if (cross) {
        const double e1x = P.v1x, e1y = P.v1y, e2x = P.v2x, e2y = P.v2y;
        const double tt = 1.0 / (f1 - f2);
        X1 = tt * (f1 * e2x - f2 * e1x);
        X2 = tt * (f1 * e2y - f2 * e1y);
        if (s1 == 0) { X1 = e1x; X2 = e1y; }
        if (s2 == 0) { X1 = e2x; X2 = e2y; }
        if (s1 == 1) { P.v1x = X1; P.v1y = X2; }
        else { P.v2x = X1; P.v2y = X2; }
    }
    // the deletions, in ascending position h: the last edge moves into h and is tested there, until one
    // stays.  key orders the edges as the loop meets them; src is the edge that ends up in this lane.
    int key = l * 32, src = l, L = P.len;
    for (unsigned rem = D; rem != 0;) {
        const int h = __ffs((int)rem) - 1;
        if (h >= L) break;
        int t = 0;
        for (;;) {
            L--;
            if (L <= h) break;
            t++;
            if (l == L) key = h * 32 + t;
            if (!((D >> L) & 1u)) {
                if (l == h) src = L;
                break;
            }
        }
        rem &= rem - 1;
    }
    double Xl1 = 0.0, Xl2 = 0.0, Y1 = 0.0, Y2 = 0.0;
    const bool two = (C & (C - 1)) != 0;
    if (two) {  // the last crossing and the one before it
        int a = __ffs((int)C) - 1, ka = __shfl(key, a, G), b = -1, kb = -1;
        for (unsigned rem = C & (C - 1); rem != 0; rem &= rem - 1) {
            const int e = __ffs((int)rem) - 1, ke = __shfl(key, e, G);
            if (ke > ka) {
                b = a;
                kb = ka;
                a = e;
                ka = ke;
            } else if (ke > kb) {
                b = e;
                kb = ke;
            }
        }
        Xl1 = __shfl(X1, a, G);
        Xl2 = __shfl(X2, a, G);
        Y1 = __shfl(X1, b, G);
        Y2 = __shfl(X2, b, G);
    }
    if (group_ballot(src != l) != 0) {
        P.v1x = __shfl(P.v1x, src, G);
        P.v1y = __shfl(P.v1y, src, G);
        P.v2x = __shfl(P.v2x, src, G);
        P.v2y = __shfl(P.v2y, src, G);
        P.lab = __shfl(P.lab, src, G);
    }
    P.len = L;
    if (!two || (isnan(Y1) && isnan(Y2)) || !(Xl1 != Y1 || Xl2 != Y2)) return 0;
    if (L >= G) return -1;
    if (l == L) {
        const double cr = (Y1 - Xl1) * (x2 - Xl2) - (Y2 - Xl2) * (x1 - Xl1);  // cross2(Y - X, x - X)
        const bool inv = cr > 0.0;                                             // invert(e), src/IO.jl:5-7
        P.v1x = inv ? Y1 : Xl1;
        P.v1y = inv ? Y2 : Xl2;
        P.v2x = inv ? Xl1 : Y1;
        P.v2y = inv ? Xl2 : Y2;
        P.lab = label;
    }
    P.len = L + 1;
    return 1;
}

// one seed's polygon, clipped by lane l of its group (gi: the group's place in the block)
__device__ __forceinline__ void group_clip_seed(const lv_grid_params &g, int n, int i, int l, int gi,
                                          const double *__restrict__ x, const int *__restrict__ cell_start,
                                          const int *__restrict__ cell_labels, const double *__restrict__ cell_x, int m,
                                          const int *__restrict__ path_i, const double *__restrict__ path_rr,
                                          int *__restrict__ ne, double *__restrict__ ev, int *__restrict__ el, int ld,
                                          double *__restrict__ area, double *__restrict__ cent, int *__restrict__ err,
                                          clip_lds &S)
{
    const double x1 = x[i], x2 = x[n + i];
    group_poly P;
    // reset!(p, cropping_rect), src/polygon.jl:37-47: DOWN(B->A), LEFT(A->D), UP(D->C), RIGHT(C->B)
    P.v1x = (l == 0 || l == 3) ? g.cmax0 : g.cmin0;
    P.v1y = (l == 2 || l == 3) ? g.cmax1 : g.cmin1;
    P.v2x = (l == 2 || l == 3) ? g.cmax0 : g.cmin0;
    P.v2y = (l == 1 || l == 2) ? g.cmax1 : g.cmin1;
    P.lab = l == 0 ? -3 : l == 1 ? -4 : l == 2 ? -1 : -2;
    P.len = 4;
    double prr = group_influence_rr(P, l, x1, x2);
    int k1, k2;
    lv_findkey(g, x1, x2, k1, k2);
    int status = LV_OK;
    // The magic path, G nodes at a time: lane l takes node kb + l, and the nodes' candidates are listed in
    // order.  The walk ends at the first node whose rr exceeds the polygon's influence, which a node's
    // first candidate within reach, or the end of the nodes, brings to light: nodes that have no
    // candidate within reach change nothing, and rr never decreases along the path.
    for (int kb = 0;; kb += G) {
        if (kb >= g.npath) {
            if (g.has_next && !(g.next_rr > prr)) status = LV_E_MESH_DESTROYED;  // src/voronoigrid.jl:63-65
            break;
        }
        const int k = kb + l;
        double rrk = __builtin_inf();
        int s0 = 0, s1 = 0;
        if (k < g.npath) {
            rrk = path_rr[k];
            const int c1 = k1 + path_i[2 * k], c2 = k2 + path_i[2 * k + 1];
            if (c1 >= 1 && c1 <= g.n1 && c2 >= 1 && c2 <= g.n2) {
                const int c = (c1 - 1) + (c2 - 1) * g.n1;
                s0 = cell_start[c];
                s1 = cell_start[c + 1];
            }
        }
        if (__shfl(rrk, 0, G) > prr) break;
        int pre = s1 - s0;  // inclusive prefix of the nodes' candidate counts
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const int t = __shfl_up(pre, o, G);
            if (l >= o) pre += t;
        }
        const int total = __shfl(pre, G - 1, G);
        pre -= s1 - s0;
        int node = -1;  // the node the walk is in
        bool stop = false;
        for (int c0 = 0; c0 < total && !stop; c0 += LCAP) {
            lds_visible();
            // (of each node only what falls into these LCAP: going through all of it for every LCAP made a seed's work
            // quadratic in its candidates: 8,000 seeds in one cell 46 ms, 0.76 this way)
            const int first = max(0, c0 - pre), end = min(s1 - s0, c0 + LCAP - pre);
            for (int t = first; t < end; t++) {
                S.s[gi][pre + t - c0] = s0 + t;
                S.q[gi][pre + t - c0] = (unsigned char)l;
            }
            lds_visible();
            const int cnt = min(LCAP, total - c0);
            // each batch's candidates are loaded while the one before it is worked off
            int qn = 0, jn = 0;
            double u1 = 0.0, u2 = 0.0;
            auto load = [&](int t0) {
                const int t = min(t0 + l, cnt - 1);
                const int s = S.s[gi][t];
                qn = S.q[gi][t];
                jn = cell_labels[s];
                u1 = cell_x[s];
                u2 = cell_x[m + s];
            };
            load(0);
            for (int t0 = 0; t0 < cnt && !stop; t0 += G) {
                const int q = qn, j = jn;
                const double rrq = __shfl(rrk, q, G);
                double y1, y2;
                lv_arrow_target(g, u1, u2, x1, x2, y1, y2);
                if (t0 + G < cnt) load(t0 + G);
                const double a = x1 - y1, b = x2 - y2;
                const double dd = a * a + b * b;
                const bool ok = t0 + l < cnt && !(x1 == y1 && x2 == y2);
                unsigned pend = group_ballot(ok && !(dd > prr));
                while (pend != 0) {
                    const int e = __ffs((int)pend) - 1;
                    const int qe = __shfl(q, e, G);
                    if (qe != node) {
                        node = qe;
                        if (__shfl(rrq, e, G) > prr) {
                            stop = true;
                            break;
                        }
                    }
                    const int r = group_cut(P, l, x1, x2, __shfl(y1, e, G), __shfl(y2, e, G), __shfl(j, e, G));
                    pend &= pend - 1;
                    if (r < 0) {
                        status = LV_E_POLY_OVERFLOW;
                        stop = true;
                        break;
                    }
                    if (r > 0) {
                        prr = group_influence_rr(P, l, x1, x2);
                        pend = group_ballot(ok && !(dd > prr)) & ~((2u << e) - 1u);
                    }
                }
            }
        }
        if (stop || __shfl(rrk, min(G, g.npath - kb) - 1, G) > prr) break;
    }
    if (status != LV_OK) {
        if (l == 0) {
            atomicCAS(err, 0, status);
            ne[i] = 0;
            area[i] = 0.0;
            cent[i] = 0.0;
            cent[n + i] = 0.0;
        }
        return;
    }
    // sort_edges!, src/IO.jl:35-48: pos is the position of this lane's edge
    const int len = P.len;
    int pos = l < len ? l : 64;
    for (int a = 0; a < len; a++) {
        const int cur = __ffs((int)group_ballot(pos == a)) - 1;
        const double lx = __shfl(P.v2x, cur, G), ly = __shfl(P.v2y, cur, G);
        unsigned M = group_ballot(l < len && pos > a && lx == P.v1x && ly == P.v1y);
        if (M == 0) continue;
        int b = __ffs((int)M) - 1, pb = __shfl(pos, b, G);
        for (M &= M - 1; M != 0; M &= M - 1) {  // several edges start there: the first by position
            const int e = __ffs((int)M) - 1, pe = __shfl(pos, e, G);
            if (pe < pb) {
                b = e;
                pb = pe;
            }
        }
        if (pos == a + 1) pos = pb;
        if (l == b) pos = a + 1;
    }
    // area(p) and centroid(p) in edge order, src/polygon.jl:114-122, 201-219: lanes 0, 1 and 2 add a
    // quantity each
    if (l < len) {
        const double p1 = P.v1x - x1, p2 = P.v1y - x2, q1 = P.v2x - x1, q2 = P.v2y - x2;
        const double h = 0.5 * fabs(p1 * q2 - p2 * q1);
        S.term[gi][0][pos] = h;
        S.term[gi][1][pos] = (h * ((x1 + P.v1x) + P.v2x)) / 3.0;
        S.term[gi][2][pos] = (h * ((x2 + P.v1y) + P.v2y)) / 3.0;
        ev[(size_t)(0 * LV_MAXE + pos) * ld + i] = P.v1x;
        ev[(size_t)(1 * LV_MAXE + pos) * ld + i] = P.v1y;
        ev[(size_t)(2 * LV_MAXE + pos) * ld + i] = P.v2x;
        ev[(size_t)(3 * LV_MAXE + pos) * ld + i] = P.v2y;
        el[(size_t)pos * ld + i] = P.lab;
    }
    lds_visible();
    double sum = 0.0;
    if (l < 3)
        for (int k = 0; k < len; k++) sum += S.term[gi][l][k];
    const double A = __shfl(sum, 0, G);
    if (l == 0) {
        ne[i] = len;
        area[i] = A;
    } else if (l < 3) {
        cent[(size_t)(l - 1) * n + i] = sum / A;
    }
    lds_visible();  // (a group that goes on to another seed writes the terms again)
}

// ---- a thread per seed ----------------------------------------------------------------------------

template <int CAP>
struct lds_poly {
    double v1x[CAP][CB], v1y[CAP][CB], v2x[CAP][CB], v2y[CAP][CB];
    int lab[CAP][CB];
};

// the slots in registers, read again whenever a cut changed them
template <int CAP>
struct reg_poly {
    double v1x[CAP], v1y[CAP], v2x[CAP], v2y[CAP];
};

template <int CAP>
__device__ __forceinline__ double load_slots(reg_poly<CAP> &R, const lds_poly<CAP> &P, int t, int len, double x1, double x2)
{
    double rr = 0.0;  // influence_rr
#pragma unroll
    for (int k = 0; k < CAP; k++) {
        R.v1x[k] = P.v1x[k][t];
        R.v1y[k] = P.v1y[k][t];
        R.v2x[k] = P.v2x[k][t];
        R.v2y[k] = P.v2y[k][t];
        const double a = R.v1x[k] - x1, b = R.v1y[k] - x2;
        const double r = 4.0 * (a * a + b * b);
        if (k < len && r > rr) rr = r;
    }
    return rr;
}

// voronoicut!(p, y, label): 1 if an edge was added, 0 if not, -1 on overflow.  First the ends of all edges
// against the bisector, from registers and side by side.  Then only the edges that it crosses or removes
// are taken up, in the order and with the moves of a walk over the slots (a removed edge's slot takes the
// last edge, which is looked at there).  Bound by instruction issue: some lane of a wavefront cuts at nearly
// every candidate, so a pre-test of the corners alone costs more than it spares (1.86 ms against 1.76 at
// 4,194,304 seeds of 0.1 dr of jitter), and lanes that each run ahead to their next cut take 3.4 to 5.6:
// they no longer go through the path together.  A walk over the slots from LDS, edge by edge, took 2.35.
template <int CAP>
__device__ __forceinline__ int cut(lds_poly<CAP> &P, const reg_poly<CAP> &R, int t, int &len, double x1, double x2, double y1,
                                   double y2, int label, bool &changed)
{
    const double d1 = y1 - x1, d2 = y2 - x2;
    const double m1 = 0.5 * (y1 + x1), m2 = 0.5 * (y2 + x2);
    const double c = d1 * m1 + d2 * m2;
    unsigned cross = 0, rem = 0;
#pragma unroll
    for (int k = 0; k < CAP; k++) {
        const double f1 = (d1 * R.v1x[k] + d2 * R.v1y[k]) - c;
        const double f2 = (d1 * R.v2x[k] + d2 * R.v2y[k]) - c;
        const bool p1 = f1 > SIGNUM_EPS, p2 = f2 > SIGNUM_EPS;
        if (p1 != p2) cross |= 1u << k;
        if ((p1 || p2) && !(f1 < -SIGNUM_EPS) && !(f2 < -SIGNUM_EPS)) rem |= 1u << k;
    }
    unsigned act = (cross | rem) & ((1u << len) - 1u);
    changed = act != 0;
    if (!changed) return 0;
    const double qnan = __builtin_nan("");
    double X1 = qnan, X2 = qnan, Y1 = qnan, Y2 = qnan;
    do {
        const int i = __ffs((int)act) - 1;
        if ((cross >> i) & 1u) {
            const double e1x = P.v1x[i][t], e1y = P.v1y[i][t], e2x = P.v2x[i][t], e2y = P.v2y[i][t];
            const double f1 = (d1 * e1x + d2 * e1y) - c;
            const double f2 = (d1 * e2x + d2 * e2y) - c;
            const int s1 = signum(f1), s2 = signum(f2);
            Y1 = X1;
            Y2 = X2;
            const double tt = 1.0 / (f1 - f2);
            X1 = tt * (f1 * e2x - f2 * e1x);
            X2 = tt * (f1 * e2y - f2 * e1y);
            if (s1 == 0) { X1 = e1x; X2 = e1y; }
            if (s2 == 0) { X1 = e2x; X2 = e2y; }
            if (s1 == 1) { P.v1x[i][t] = X1; P.v1y[i][t] = X2; }
            else { P.v2x[i][t] = X1; P.v2y[i][t] = X2; }
        }
        if ((rem >> i) & 1u) {
            const int last = --len;
            if (last > i) {
                P.v1x[i][t] = P.v1x[last][t];
                P.v1y[i][t] = P.v1y[last][t];
                P.v2x[i][t] = P.v2x[last][t];
                P.v2y[i][t] = P.v2y[last][t];
                P.lab[i][t] = P.lab[last][t];
            }
            cross = (cross & ~(1u << i)) | (((cross >> last) & 1u) << i);
            rem = (rem & ~(1u << i)) | (((rem >> last) & 1u) << i);
            act = (cross | rem) & ((1u << len) - 1u) & (~0u << i);
        } else {
            act &= act - 1u;
        }
    } while (act != 0);
    if (!(isnan(Y1) && isnan(Y2)) && (X1 != Y1 || X2 != Y2)) {
        if (len >= CAP) return -1;
        const double cr = (Y1 - X1) * (x2 - X2) - (Y2 - X2) * (x1 - X1);  // cross2(Y - X, x - X)
        if (cr > 0.0) {  // invert(e), src/IO.jl:5-7
            P.v1x[len][t] = Y1; P.v1y[len][t] = Y2; P.v2x[len][t] = X1; P.v2y[len][t] = X2;
        } else {
            P.v1x[len][t] = X1; P.v1y[len][t] = X2; P.v2x[len][t] = Y1; P.v2y[len][t] = Y2;
        }
        P.lab[len][t] = label;
        len++;
        return 1;
    }
    return 0;
}

template <int CAP>
__device__ __forceinline__ void swap_slots(lds_poly<CAP> &P, int t, int a, int b)
{
    double tx;
    tx = P.v1x[a][t]; P.v1x[a][t] = P.v1x[b][t]; P.v1x[b][t] = tx;
    tx = P.v1y[a][t]; P.v1y[a][t] = P.v1y[b][t]; P.v1y[b][t] = tx;
    tx = P.v2x[a][t]; P.v2x[a][t] = P.v2x[b][t]; P.v2x[b][t] = tx;
    tx = P.v2y[a][t]; P.v2y[a][t] = P.v2y[b][t]; P.v2y[b][t] = tx;
    int tl = P.lab[a][t]; P.lab[a][t] = P.lab[b][t]; P.lab[b][t] = tl;
}

// the candidates of the walk's node k (none, and a valid index, beyond the grid and the path's end)
__device__ __forceinline__ void path_node(const lv_grid_params &g, const int *__restrict__ path_i, int k, int k1,
                                          int k2, const int *__restrict__ cell_start, int &s0, int &s1)
{
    s0 = s1 = 0;
    if (k >= g.npath) return;
    const int c1 = k1 + path_i[2 * k], c2 = k2 + path_i[2 * k + 1];
    if (c1 < 1 || c1 > g.n1 || c2 < 1 || c2 > g.n2) return;
    const int c = (c1 - 1) + (c2 - 1) * g.n1;
    s0 = cell_start[c];
    s1 = cell_start[c + 1];
}

// one seed's polygon, clipped in P's LDS slots; false when it outgrew them
template <int CAP>
__device__ bool clip_seed(const lv_grid_params &g, int n, int i, const double *__restrict__ x,
                          const int *__restrict__ cell_start, const int *__restrict__ cell_labels,
                          const double *__restrict__ cell_x, int m, const int *__restrict__ path_i,
                          const double *__restrict__ path_rr, int *__restrict__ ne, double *__restrict__ ev,
                          int *__restrict__ el, int ld, double *__restrict__ area, double *__restrict__ cent,
                          int *__restrict__ err, lds_poly<CAP> &P, int t)
{
    const double x1 = x[i], x2 = x[n + i];

    // reset!(p, cropping_rect), src/polygon.jl:37-47: DOWN(B->A), LEFT(A->D), UP(D->C), RIGHT(C->B)
    {
        const double Ax = g.cmin0, Ay = g.cmin1, Cx = g.cmax0, Cy = g.cmax1;
        const double Bx = Cx, By = Ay, Dx = Ax, Dy = Cy;
        P.v1x[0][t] = Bx; P.v1y[0][t] = By; P.v2x[0][t] = Ax; P.v2y[0][t] = Ay; P.lab[0][t] = -3;
        P.v1x[1][t] = Ax; P.v1y[1][t] = Ay; P.v2x[1][t] = Dx; P.v2y[1][t] = Dy; P.lab[1][t] = -4;
        P.v1x[2][t] = Dx; P.v1y[2][t] = Dy; P.v2x[2][t] = Cx; P.v2y[2][t] = Cy; P.lab[2][t] = -1;
        P.v1x[3][t] = Cx; P.v1y[3][t] = Cy; P.v2x[3][t] = Bx; P.v2y[3][t] = By; P.lab[3][t] = -2;
    }
    int len = 4;
    reg_poly<CAP> R;
    double prr = load_slots(R, P, t, len, x1, x2);
    int k1, k2;
    lv_findkey(g, x1, x2, k1, k2);
    int status = LV_OK;
    // node k's candidates: cell_start two nodes ahead of their use, a position one candidate ahead (the
    // first of the next node; a position beyond the items, at most one, is in cell_x's room)
    int s0, s1, n0, n1, f0, f1;
    path_node(g, path_i, 0, k1, k2, cell_start, s0, s1);
    path_node(g, path_i, 1, k1, k2, cell_start, n0, n1);
    double c1 = cell_x[s0], c2 = cell_x[m + s0];
    for (int k = 0;; k++) {
        if (k == g.npath) {
            if (g.has_next && !(g.next_rr > prr)) status = LV_E_MESH_DESTROYED;  // src/voronoigrid.jl:63-65
            break;
        }
        if (path_rr[k] > prr) break;
        path_node(g, path_i, k + 2, k1, k2, cell_start, f0, f1);
        for (int s = s0; s < s1; s++) {
            const int sn = s + 1 < s1 ? s + 1 : n0;
            const double y1c = c1, y2c = c2;
            c1 = cell_x[sn];
            c2 = cell_x[m + sn];
            double y1, y2;
            lv_arrow_target(g, y1c, y2c, x1, x2, y1, y2);
            const double a = x1 - y1, b = x2 - y2;
            if ((x1 == y1 && x2 == y2) || (a * a + b * b > prr)) continue;
            bool changed;
            const int r = cut(P, R, t, len, x1, x2, y1, y2, cell_labels[s], changed);
            if (r < 0) {
                status = LV_E_POLY_OVERFLOW;
                break;
            }
            if (changed) {
                const double rr = load_slots(R, P, t, len, x1, x2);
                if (r) prr = rr;
            }
        }
        if (status != LV_OK) break;
        if (s0 >= s1) {
            c1 = cell_x[n0];
            c2 = cell_x[m + n0];
        }
        s0 = n0; s1 = n1;
        n0 = f0; n1 = f1;
    }
    if (status == LV_E_POLY_OVERFLOW) return false;
    if (status != LV_OK) {
        atomicCAS(err, 0, status);
        ne[i] = 0;
        area[i] = 0.0;
        cent[i] = 0.0;
        cent[n + i] = 0.0;
        return true;
    }
    // sort_edges!, src/IO.jl:35-48
    for (int a = 0; a < len; a++) {
        const double lx = P.v2x[a][t], ly = P.v2y[a][t];
        for (int b = a + 1; b < len; b++) {
            if (lx == P.v1x[b][t] && ly == P.v1y[b][t]) {
                if (b != a + 1) swap_slots(P, t, a + 1, b);
                break;
            }
        }
    }
    // area(p) and centroid(p) in edge order, src/polygon.jl:114-122, 201-219
    double A = 0.0, Ac = 0.0, cx = 0.0, cy = 0.0;
    for (int k = 0; k < len; k++) {
        const double v1x = P.v1x[k][t], v1y = P.v1y[k][t], v2x = P.v2x[k][t], v2y = P.v2y[k][t];
        const double p1 = v1x - x1, p2 = v1y - x2, q1 = v2x - x1, q2 = v2y - x2;
        const double h = 0.5 * fabs(p1 * q2 - p2 * q1);
        A += h;
        Ac += h;
        cx += (h * ((x1 + v1x) + v2x)) / 3.0;
        cy += (h * ((x2 + v1y) + v2y)) / 3.0;
        ev[(size_t)(0 * LV_MAXE + k) * ld + i] = v1x;
        ev[(size_t)(1 * LV_MAXE + k) * ld + i] = v1y;
        ev[(size_t)(2 * LV_MAXE + k) * ld + i] = v2x;
        ev[(size_t)(3 * LV_MAXE + k) * ld + i] = v2y;
        el[(size_t)k * ld + i] = P.lab[k][t];
    }
    ne[i] = len;
    area[i] = A;
    cent[i] = cx / Ac;
    cent[n + i] = cy / Ac;
    return true;
}

constexpr int CHUNK = 4 * CB;

// The seed of this lane.  Some lane of a wavefront cuts at nearly every candidate unless its seeds see
// alike candidates in alike order, and that depends on where in its cell a seed sits: on a lattice of two
// seeds to a cell side neighbours take turns.  So the four wavefronts of a chunk of consecutive seeds share
// them by NB x NB parts of the cell.  Each of the four orders the chunk for itself (only an order: the
// mesh does not depend on it).  At 4,194,304 seeds 2.03 -> 1.76 ms on a lattice of 0.1 dr of jitter and 3.26 ->
// 2.98 with 0.45 dr; 4 x 4 parts 1.83 and 3.02.
template <int NB>
__device__ __forceinline__ int clip_seed_of(const lv_grid_params &g, int n, int chunk, int part,
                                            const double *__restrict__ x, unsigned char *ord)
{
    const int t = threadIdx.x;
    int key[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int i = chunk * CHUNK + r * CB + t;
        key[r] = NB * NB;
        if (i < n) {
            const double fx = (x[i] - g.origin0) / g.h, fy = (x[n + i] - g.origin1) / g.h;
            const int bx = (int)(NB * (fx - floor(fx))), by = (int)(NB * (fy - floor(fy)));
            key[r] = (bx & (NB - 1)) * NB + ((by ^ (bx & 1 ? NB - 1 : 0)) & (NB - 1));
        }
    }
    const unsigned long long lt = (1ull << t) - 1ull;
    int off = 0;
    for (int b = 0; b <= NB * NB; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const unsigned long long M = __ballot(key[r] == b);
            if (key[r] == b) ord[off + __popcll(M & lt)] = (unsigned char)(r * CB + t);
            off += __popcll(M);
        }
    lds_visible();
    return chunk * CHUNK + ord[part * CB + t];
}

// The chunk a workgroup works on and its part of it.  Workgroups are dispatched round-robin over the 8
// XCDs, so workgroup b runs on XCD b mod 8: 32 workgroups take 8 chunks, the four parts of a chunk on one
// XCD, whose L2 joins their stores.  The clipping work per seed varies across the domain, and mapped
// straight each XCD would get every 8th chunk, on a lattice whose rows span a multiple of 8 chunks the same
// few column strips of the domain in every row: XCDs with the costly strips ran up to 28% longer while the
// others idled for the last third of the launch.  Rotating each group by a hash of its index (the top 3 bits of a
// multiplicative hash, so that no period of the domain lines up with it) gives every XCD an even share
// of every column.
__device__ __forceinline__ void clip_chunk(int b, int &chunk, int &part)
{
    const unsigned q = (unsigned)b >> 5;
    const unsigned rot = (q * 2654435761u) >> 29;
    chunk = (int)((q << 3) | ((b + rot) & 7));
    part = (b >> 3) & 3;
}

// every seed with CAP slots; the ones that outgrow them go to the queue retry[1..retry[0]]
template <int CAP>
__global__ __launch_bounds__(CB) void k_clip(lv_grid_params g, int n, const double *__restrict__ x,
                                             const int *__restrict__ cell_start, const int *__restrict__ cell_labels,
                                             const double *__restrict__ cell_x, int m, const int *__restrict__ path_i,
                                             const double *__restrict__ path_rr, int *__restrict__ ne,
                                             double *__restrict__ ev, int *__restrict__ el, int ld,
                                             double *__restrict__ area, double *__restrict__ cent,
                                             int *__restrict__ err, int *__restrict__ retry)
{
    __shared__ lds_poly<CAP> P;
    __shared__ unsigned char ord[CHUNK];
    const int t = threadIdx.x;
    const int before = *err;
    int chunk, part;
    clip_chunk(blockIdx.x, chunk, part);
    if (chunk * CHUNK >= n) return;
    const int i = clip_seed_of<2>(g, n, chunk, part, x, ord);
    if (i >= n || move_refused(before)) return;  // no block-wide barriers below
    if (!clip_seed(g, n, i, x, cell_start, cell_labels, cell_x, m, path_i, path_rr, ne, ev, el, ld, area, cent, err, P, t))
        retry[1 + atomicAdd(&retry[0], 1)] = i;
}

// the queued seeds (queue[1..queue[0]], grid-stride), or all n of them without a queue
__global__ __launch_bounds__(GB) void k_clip_group(lv_grid_params g, int n, const double *__restrict__ x,
                                                   const int *__restrict__ cell_start,
                                                   const int *__restrict__ cell_labels,
                                                   const double *__restrict__ cell_x, int m,
                                                   const int *__restrict__ path_i,
                                                   const double *__restrict__ path_rr, int *__restrict__ ne,
                                                   double *__restrict__ ev, int *__restrict__ el, int ld,
                                                   double *__restrict__ area, double *__restrict__ cent,
                                                   int *__restrict__ err, const int *__restrict__ queue)
{
    __shared__ clip_lds S;
    const int l = threadIdx.x & (G - 1), gi = threadIdx.x / G;
    const int before = *err;
    const int cnt = queue ? queue[0] : n;
    if (move_refused(before)) return;
    for (int q = blockIdx.x * (GB / G) + gi; q < cnt; q += gridDim.x * (GB / G))
        group_clip_seed(g, n, queue ? queue[1 + q] : q, l, gi, x, cell_start, cell_labels, cell_x, m, path_i, path_rr, ne,
                        ev, el, ld, area, cent, err, S);
}

// Up to this many seeds, a group of lanes each.  On lattices of 0.1 dr of jitter clipping takes 34 us with
// groups and 62 us with a thread per seed (and the queue's launch) at 1,024 seeds, 43 and 71 at 10,000,
// 77 and 76 at 25,600, 107 and 79 at 40,000; with 0.45 dr of jitter 40 and 97, 52 and 131, 89 and 114, 103 and 113 at
// 32,400, and 123 and 152 at 40,000: the line lies between where the two cross.
constexpr int GROUP_MAX = 32768;

// Up to this many, a thread per seed with ten slots: a CU holds 6 of its 64-seed blocks (23 KB), all blocks are
// resident at once and hardly a polygon goes to the queue (70 us for 96 with eight slots at 65,536 seeds,
// 92 for 117 at 96,100; with 0.45 dr of jitter 113 for 144 and 162 for 169).  Above it the residency counts: 138
// for 118 at 122,500 and 189 for 168 at 262,144.
constexpr int WIDE_MAX = 6 * 256 * CB;

}  // namespace

hipError_t lv_launch_clip(const lv_grid_params &g, int n, const double *x, const int *cell_start,
                          const int *cell_labels, const double *cell_x, const int *path_i, const double *path_rr,
                          int *ne, double *ev, int *el, int ld, double *area, double *cent, int *err, int *retry,
                          hipStream_t s, int m)
{
    if (n <= 0) return hipSuccess;
    const int groups = (n + GB / G - 1) / (GB / G);
    const bool all = n <= GROUP_MAX;
    if (!all) {
        hipError_t e = hipMemsetAsync(retry, 0, sizeof(int), s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(n <= WIDE_MAX ? k_clip<10> : k_clip<8>, dim3((n + 8 * CHUNK - 1) / (8 * CHUNK) * 32),
                           dim3(CB), 0, s, g, n, x, cell_start, cell_labels, cell_x, m,
                           path_i, path_rr, ne, ev, el, ld, area, cent, err, retry);
    }
    hipLaunchKernelGGL(k_clip_group, dim3(all ? groups : std::min(RETRY_BLOCKS, groups)), dim3(GB), 0, s, g, n, x,
                       cell_start, cell_labels, cell_x, m, path_i, path_rr, ne, ev, el, ld, area, cent, err,
                       all ? (const int *)nullptr : (const int *)retry);
    return hipGetLastError();
}
