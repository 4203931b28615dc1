// RKPM on gfx950: reproducing-kernel functions with element-as-cell strain smoothing
// over a Tet4 or Hex8 background mesh (one- and two-pass force), and finite-element
// strain smoothing on Tet4 (the same cells with the element's own shape functions).
//
// Set-up (once, Total Lagrangian):
//   max edge length     src/MaxEdgeLengthProcessor.cpp:36-60
//   kernel radius       src/NeighborSearchProcessor.cpp:154-185 (r = scale * l; scale 1 -> 1 + 1e-6)
//   ball search         include/NeighborSearchProcessor.h:196-317, src/NeighborSearchProcessor.cpp:185-240,
//                       include/NeighborSelectorFunctor.h:63-99 — here a uniform cell list (cell edge =
//                       largest radius) replaces STK's LBVH; each point keeps its 40 nearest accepted
//                       candidates by (tweaked d^2, id) in LDS
//   RK functions        include/FunctionCreationProcessor.h:85-130,
//                       include/ShapeFunctionsFunctorReproducingKernel.h:190-257 (4x4 moment matrix
//                       inverted by complete-pivoting LU in registers)
//   cell node lists     include/SmoothedCellDataProcessor.h:407-539 (first-seen union)
//   cell derivatives    include/SmoothedCellDataProcessor.h:542-675, include/QuadratureSmoothed.h:32-62
//   RK mass             src/MassUtils.cpp:79-112 via FunctionEvaluationProcessor::ScatterValues
//   two-pass cells      include/SmoothedCellDataProcessor.h:474-486, :637-648 (the element's own
//                       nodes, derivative (B_k V)/V)
// Per step, element cells (both methods; src/Solvers/Explicit.cpp:148-186):
//   gather kernel       FunctionEvaluationProcessor::ComputeValues (include/FunctionEvaluationProcessor.h:
//                       70-117): u = Phi d
//   element tiles       include/ComputeInternalForceSmoothedCell.h:86-117, :186-224, :325-349 on u, the
//                       cell of an element being the element (tile.hip, force mode)
//   scatter kernel      ScatterValues (:130-181) as a gather over reverse neighbor lists (points that
//                       list the node, ascending), fused with the central-difference node update
//                       (small meshes: gather and scatter in the tile's and the node's launch)
// Nodal smoothing cells on a thex mesh (each tet split into four hexes):
//   active nodes        include/MeshLabelerProcessor.h:227-330 (each hex's node of lowest
//                       caller id; exactly one per hex), cells and subcells :690-827 (one cell
//                       per active node: the hexes around it; subdomains 0: every hex a
//                       subcell, 1: the cell one subcell); internal nodes are renumbered with
//                       the active ones first, so nodes with degrees of freedom are a prefix
//   max edge length     edges to inactive nodes doubled (src/MaxEdgeLengthProcessor.cpp:54-55)
//   search              query points: every node; candidates: the active nodes
//   subcell CSR         include/SmoothedCellDataProcessor.h:407-675 over the hexes of a subcell
//   F-bar force         include/ComputeInternalForceSmoothedCell.h:120-413 (subcell J, cell
//                       J-bar, stress of F-bar, dual pressure, un-barred stress), used when a
//                       cell has more subcells than one (:458-459)
// Per step, nodal cells: one kernel over cell tiles (forces to the tiles' node slots) and one over
// the nodes (slots in ascending tile order, node update).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <numeric>
#include <thread>
#include <vector>

#include "element.hpp"
#include "internal.hpp"
#include "workers.hpp"

namespace aphip {

namespace {

constexpr int kSearchBlock = 64;
constexpr int kFusedNodes = 12000;  // element cells: two launches a step (rk_fused)
constexpr int kCellBlock = 64;

__device__ __forceinline__ void ld3(const double *p, int64_t i, double *o) {
    o[0] = p[3 * i];
    o[1] = p[3 * i + 1];
    o[2] = p[3 * i + 2];
}

__device__ __forceinline__ void st3(double *p, int64_t i, const double *o) {
    p[3 * i] = o[0];
    p[3 * i + 1] = o[1];
    p[3 * i + 2] = o[2];
}

// |a - b|^2 with a fixed fused order (the oracle evaluates the same expression)
__device__ __forceinline__ double dist2(const double *a, const double *b) {
    const double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
    return __fma_rn(dz, dz, __fma_rn(dy, dy, dx * dx));
}

template <int NPE>
__global__ __launch_bounds__(256) void k_max_edge(int64_t nn, const int32_t *node_start, const int32_t *node_inc,
                                                  const int32_t *conn, const double *X, double scale, int64_t n_active,
                                                  double *radius) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    double xi[3];
    ld3(X, i, xi);
    double l = 0.0;
    for (int32_t t = node_start[i]; t < node_start[i + 1]; ++t) {
        const int64_t e = node_inc[t] / NPE;
#pragma unroll
        for (int k = 0; k < NPE; ++k) {
            double xj[3];
            const int32_t j = conn[NPE * e + k];
            ld3(X, j, xj);
            // an edge to a node without degrees of freedom counts twice (nodes j >= n_active)
            l = fmax(l, sqrt(dist2(xi, xj)) * (j >= n_active ? 2.0 : 1.0));
        }
    }
    radius[i] = l * scale;
}

struct Grid {
    double lo[3];
    double cell;
    int nb[3];
};

__device__ __forceinline__ int bin_coord(double x, double lo, double cell, int nb) {
    int b = (int)floor((x - lo) / cell);
    return b < 0 ? 0 : (b >= nb ? nb - 1 : b);
}

__global__ __launch_bounds__(256) void k_bin_count(int64_t nn, const double *X, Grid G, int32_t *bin_of,
                                                   int32_t *count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    const int bx = bin_coord(X[3 * i], G.lo[0], G.cell, G.nb[0]);
    const int by = bin_coord(X[3 * i + 1], G.lo[1], G.cell, G.nb[1]);
    const int bz = bin_coord(X[3 * i + 2], G.lo[2], G.cell, G.nb[2]);
    const int b = (bz * G.nb[1] + by) * G.nb[0] + bx;
    bin_of[i] = b;
    atomicAdd(&count[b], 1);
}

// order inside a bin is irrelevant: accepted candidates are ranked by (d^2, id)
__global__ __launch_bounds__(256) void k_bin_fill(int64_t nn, const int32_t *bin_of, const int32_t *bstart,
                                                  int32_t *fill, int32_t *items) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    const int b = bin_of[i];
    items[bstart[b] + atomicAdd(&fill[b], 1)] = (int32_t)i;
}

struct SearchArgs {
    int64_t nn;
    const double *X;
    const double *radius;
    const int32_t *caller_id;
    Grid G;
    const int32_t *bstart;
    const int32_t *items;
    int32_t *num;
    int32_t *nbr;
    int32_t *ncand;
};

__device__ __forceinline__ bool before(double da, int ia, double db, int ib) {
    return da < db || (da == db && ia < ib);
}

__global__ __launch_bounds__(kSearchBlock) void k_search(SearchArgs A) {
    __shared__ double sd[kMaxNbr * kSearchBlock];
    __shared__ int32_t sk[kMaxNbr * kSearchBlock];  // ranking key: caller id
    __shared__ int32_t sn[kMaxNbr * kSearchBlock];  // internal id
    const int tid = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * kSearchBlock + tid;
    if (i >= A.nn) return;
    double xi[3];
    ld3(A.X, i, xi);
    const int bx = bin_coord(xi[0], A.G.lo[0], A.G.cell, A.G.nb[0]);
    const int by = bin_coord(xi[1], A.G.lo[1], A.G.cell, A.G.nb[1]);
    const int bz = bin_coord(xi[2], A.G.lo[2], A.G.cell, A.G.nb[2]);
    int cnt = 0, seen = 0;
    for (int z = bz - 1; z <= bz + 1; ++z) {
        if (z < 0 || z >= A.G.nb[2]) continue;
        for (int y = by - 1; y <= by + 1; ++y) {
            if (y < 0 || y >= A.G.nb[1]) continue;
            for (int x = bx - 1; x <= bx + 1; ++x) {
                if (x < 0 || x >= A.G.nb[0]) continue;
                const int b = (z * A.G.nb[1] + y) * A.G.nb[0] + x;
                for (int p = A.bstart[b]; p < A.bstart[b + 1]; ++p) {
                    const int32_t j = A.items[p];
                    double xj[3];
                    ld3(A.X, j, xj);
                    const double rj = A.radius[j];
                    // the sphere of neighbor j contains point i
                    if (!(dist2(xj, xi) <= rj * rj)) continue;
                    ++seen;
                    // ranking distance with the neighbor coordinates tweaked by (1+1e-6, 1+1e-7, 1+1e-8)
                    const double tw[3] = {xj[0] * (1 + 1.0e-6), xj[1] * (1 + 1.0e-7), xj[2] * (1 + 1.0e-8)};
                    const double d2 = dist2(tw, xi);
                    const int32_t key = A.caller_id[j];
                    if (cnt == kMaxNbr && !before(d2, key, sd[(kMaxNbr - 1) * kSearchBlock + tid],
                                                  sk[(kMaxNbr - 1) * kSearchBlock + tid]))
                        continue;
                    int pos = cnt < kMaxNbr ? cnt : kMaxNbr - 1;
                    while (pos > 0 && before(d2, key, sd[(pos - 1) * kSearchBlock + tid], sk[(pos - 1) * kSearchBlock + tid])) {
                        sd[pos * kSearchBlock + tid] = sd[(pos - 1) * kSearchBlock + tid];
                        sk[pos * kSearchBlock + tid] = sk[(pos - 1) * kSearchBlock + tid];
                        sn[pos * kSearchBlock + tid] = sn[(pos - 1) * kSearchBlock + tid];
                        --pos;
                    }
                    sd[pos * kSearchBlock + tid] = d2;
                    sk[pos * kSearchBlock + tid] = key;
                    sn[pos * kSearchBlock + tid] = j;
                    if (cnt < kMaxNbr) ++cnt;
                }
            }
        }
    }
    A.num[i] = cnt;
    A.ncand[i] = seen;
    for (int k = 0; k < kMaxNbr; ++k) A.nbr[i * kMaxNbr + k] = k < cnt ? sn[k * kSearchBlock + tid] : -1;
}

// Cubic B-spline kernel, include/MathUtils.h:321-330
__device__ __forceinline__ double kernel_value(const double *d, double R) {
    const double q = sqrt(__fma_rn(d[2], d[2], __fma_rn(d[1], d[1], d[0] * d[0]))) / R;
    if (q < 0.5) return 1.0 + 6.0 * q * q * (-1.0 + q);
    if (q < 1.0) return 2.0 * (1.0 + q * (-3.0 + 3.0 * q - 1.0 * q * q));
    return 0.0;
}

__device__ __forceinline__ void swap_d(double &a, double &b) {
    const double t = a;
    a = b;
    b = t;
}

// Row 0 of the inverse of the symmetric 4x4 moment matrix by LU with complete
// pivoting (the published FullPivLU algorithm of Eigen 3.4, which InvertMatrix uses on
// CPU builds, include/MathUtils.h:307-319): first maximum in column-major scan,
// rank threshold |max pivot| * eps * 4, unknowns beyond the rank set to zero.
// All indices are compile-time after unrolling, so the matrix stays in registers.
// Returns the Frobenius norm of the full inverse.
__device__ double inverse4_row0(double (&a)[4][4], double (&row0)[4]) {
    int prow[4] = {0, 1, 2, 3}, pcol[4] = {0, 1, 2, 3};
    int nonzero = 4;
    double maxpiv = 0.0;
    bool stop = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!stop) {
            double big = -1.0;
            int bi = k, bj = k;
#pragma unroll
            for (int j = k; j < 4; ++j)
#pragma unroll
                for (int i = k; i < 4; ++i) {
                    const double v = fabs(a[i][j]);
                    if (v > big) {
                        big = v;
                        bi = i;
                        bj = j;
                    }
                }
            if (big == 0.0) {
                nonzero = k;
                stop = true;
            } else {
                maxpiv = fmax(maxpiv, big);
#pragma unroll
                for (int r = k + 1; r < 4; ++r)
                    if (bi == r) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) swap_d(a[k][j], a[r][j]);
                        const int tmp = prow[k];
                        prow[k] = prow[r];
                        prow[r] = tmp;
                    }
#pragma unroll
                for (int r = k + 1; r < 4; ++r)
                    if (bj == r) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) swap_d(a[i][k], a[i][r]);
                        const int tmp = pcol[k];
                        pcol[k] = pcol[r];
                        pcol[r] = tmp;
                    }
                const double piv = a[k][k];
#pragma unroll
                for (int i = k + 1; i < 4; ++i) a[i][k] /= piv;
#pragma unroll
                for (int i = k + 1; i < 4; ++i)
#pragma unroll
                    for (int j = k + 1; j < 4; ++j) a[i][j] -= a[i][k] * a[k][j];
            }
        }
    }
    const double thr = maxpiv * (2.220446049250313e-16 * 4.0);
    int rank = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < nonzero && fabs(a[i][i]) > thr) ++rank;
    double fro = 0.0;
#pragma unroll
    for (int col = 0; col < 4; ++col) row0[col] = 0.0;
    if (rank == 0) return 0.0;
#pragma unroll
    for (int col = 0; col < 4; ++col) {
        double cv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) cv[i] = (prow[i] == col) ? 1.0 : 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < i; ++j) cv[i] -= a[i][j] * cv[j];
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            if (i < rank) {
#pragma unroll
                for (int j = i + 1; j < 4; ++j)
                    if (j < rank) cv[i] -= a[i][j] * cv[j];
                cv[i] /= a[i][i];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double x = i < rank ? cv[i] : 0.0;
            fro += x * x;
            if (pcol[i] == 0) row0[col] = x;
        }
    }
    return sqrt(fro);
}

__global__ __launch_bounds__(128) void k_rk_phi(int64_t nn, const double *X, const double *radius, const int32_t *num,
                                                const int32_t *nbr, double *phi) {
    const int64_t i = (int64_t)blockIdx.x * 128 + threadIdx.x;
    if (i >= nn) return;
    const int n = num[i];
    double *ph = phi + i * kMaxNbr;
    for (int k = 0; k < kMaxNbr; ++k) ph[k] = 0.0;
    if (n == 0) return;
    if (n == 1) {
        ph[0] = 1.0;
        return;
    }
    double xi[3];
    ld3(X, i, xi);
    double M[4][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
    double wsum = 0.0;
    for (int k = 0; k < n; ++k) {
        const int32_t j = nbr[i * kMaxNbr + k];
        double xj[3];
        ld3(X, j, xj);
        const double d[3] = {xi[0] - xj[0], xi[1] - xj[1], xi[2] - xj[2]};
        const double w = kernel_value(d, radius[j]);
        if (w == 0.0) continue;
        const double Hb[4] = {1.0, d[0], d[1], d[2]};
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) M[a][b] += (w * Hb[a]) * Hb[b];
        wsum += w;
    }
    double r0[4];
    const double fro = inverse4_row0(M, r0);
    const bool shepard = fro < 1e-15;
    for (int k = 0; k < n; ++k) {
        const int32_t j = nbr[i * kMaxNbr + k];
        double xj[3];
        ld3(X, j, xj);
        const double d[3] = {xi[0] - xj[0], xi[1] - xj[1], xi[2] - xj[2]};
        const double w = kernel_value(d, radius[j]);
        if (shepard) {
            ph[k] = w / wsum;
        } else if (w != 0.0) {
            ph[k] = (r0[0] + r0[1] * d[0] + r0[2] * d[1] + r0[3] * d[2]) * w;
        }
    }
}

// First-seen union of the neighbor lists of a cell's NPE nodes, in LDS.
template <int NPE>
__device__ __forceinline__ int cell_union(const int32_t *en, const int32_t *num, const int32_t *nbr, int32_t *list,
                                          int stride) {
    int len = 0;
    for (int k = 0; k < NPE; ++k) {
        const int32_t a = en[k];
        const int na = num[a];
        for (int l = 0; l < na; ++l) {
            const int32_t j = nbr[(int64_t)a * kMaxNbr + l];
            bool found = false;
            for (int t = 0; t < len; ++t)
                if (list[t * stride] == j) {
                    found = true;
                    break;
                }
            if (!found) list[(len++) * stride] = j;
        }
    }
    return len;
}

// cells per block of the set-up kernels: each thread keeps its union list of up to
// NPE * kMaxNbr entries in LDS (40 KB per block either way)
template <int NPE>
constexpr int cell_block() { return NPE == 4 ? kCellBlock : kCellBlock / 2; }

template <int NPE>
__global__ __launch_bounds__(cell_block<NPE>()) void k_cell_count(int64_t ne, const int32_t *conn, const int32_t *num,
                                                                  const int32_t *nbr, int32_t *len_out) {
    constexpr int BLK = cell_block<NPE>();
    __shared__ int32_t list[NPE * kMaxNbr * BLK];
    const int64_t e = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (e >= ne) return;
    int32_t en[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) en[k] = conn[NPE * e + k];
    len_out[e] = cell_union<NPE>(en, num, nbr, list + threadIdx.x, BLK);
}

struct CellFillArgs {
    int64_t ne;
    const int32_t *conn;
    const double *X;
    const int32_t *num;
    const int32_t *nbr;
    const double *phi;
    const int64_t *start;
    int32_t *nodes;
    double *dphi;
    double *volume;
};

template <int NPE>
__global__ __launch_bounds__(cell_block<NPE>()) void k_cell_fill(CellFillArgs A) {
    constexpr int BLK = cell_block<NPE>();
    __shared__ int32_t list[NPE * kMaxNbr * BLK];
    const int tid = threadIdx.x;
    const int64_t e = (int64_t)blockIdx.x * BLK + tid;
    if (e >= A.ne) return;
    int32_t en[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) en[k] = A.conn[NPE * e + k];
    int32_t *my = list + tid;
    const int len = cell_union<NPE>(en, A.num, A.nbr, my, BLK);
    const int64_t s0 = A.start[e];
    double X[NPE][3], B[NPE][3], V;
#pragma unroll
    for (int k = 0; k < NPE; ++k) ld3(A.X, en[k], X[k]);
    smoothed_cell<NPE>(X, B, V);
    double *dp = A.dphi + 3 * s0;
    for (int t = 0; t < len; ++t) {
        A.nodes[s0 + t] = my[t * BLK];
        dp[3 * t] = dp[3 * t + 1] = dp[3 * t + 2] = 0.0;
    }
    // grad phi_J = sum_k B_k V phi_{k,J} / V_sub (SmoothedCellDataProcessor.h:623-662)
#pragma unroll
    for (int k = 0; k < NPE; ++k) {
        const int32_t a = en[k];
        const int na = A.num[a];
        for (int l = 0; l < na; ++l) {
            const int32_t j = A.nbr[(int64_t)a * kMaxNbr + l];
            const double fv = A.phi[(int64_t)a * kMaxNbr + l];
            int t = 0;
            while (my[t * BLK] != j) ++t;
#pragma unroll
            for (int m = 0; m < 3; ++m) dp[3 * t + m] += B[k][m] * V * fv;
        }
    }
    for (int t = 0; t < len; ++t) {
        dp[3 * t] /= V;
        dp[3 * t + 1] /= V;
        dp[3 * t + 2] /= V;
    }
    A.volume[e] = V;
}

// Two-pass cells: entry 4e + k is node k of element e with derivative (B_k V) / V.
template <int NPE>
__global__ __launch_bounds__(256) void k_cell_two_pass(int64_t ne, const int32_t *conn, const double *X,
                                                       int32_t *nodes, double *dphi, double *volume) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= ne) return;
    int32_t en[NPE];
#pragma unroll
    for (int k = 0; k < NPE; ++k) en[k] = conn[NPE * e + k];
    double Xe[NPE][3], B[NPE][3], V;
#pragma unroll
    for (int k = 0; k < NPE; ++k) ld3(X, en[k], Xe[k]);
    smoothed_cell<NPE>(Xe, B, V);
#pragma unroll
    for (int k = 0; k < NPE; ++k) {
        nodes[NPE * e + k] = en[k];
#pragma unroll
        for (int m = 0; m < 3; ++m) dphi[3 * (NPE * e + k) + m] = (B[k][m] * V) / V;
    }
    volume[e] = V;
}

__global__ __launch_bounds__(256) void k_identity_functions(int64_t nn, int32_t *num, int32_t *nbr, double *phi) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    num[i] = 1;
    // the whole row: the node itself with value 1, the unused entries -1 / 0
    for (int k = 0; k < kMaxNbr; ++k) {
        nbr[i * kMaxNbr + k] = k == 0 ? (int32_t)i : -1;
        phi[i * kMaxNbr + k] = k == 0 ? 1.0 : 0.0;
    }
}

// ---- smoothed-cell force step --------------------------------------------
// The derivative of a smoothed cell is a product, grad phi_J = sum_k B_k phi_J(x_k) over the
// nodes k of its elements, and so are the cell's gradient and force:
//   H = sum_J d_J (x) grad phi_J = sum_k (Phi d)_k (x) B_k,
//   f = -sum_c V_c P_c grad phi^T = Phi^T (-sum_c V_c P_c B_k^T).
// Element cells (one- and two-pass method alike) therefore apply the factors: a gather
// u = Phi d over the nodes' neighbor rows, the cell force on u by the element tile plan (the
// cell of a Tet4 is the element itself with its own gradient), and a scatter Phi^T over the
// reverse neighbor lists.  Applying the product instead (the CSR of about 77 derivatives a
// Tet4 cell at kernel scale 1.5, 26 B each, in wave-sized cell tiles) took 0.92 ms a step on
// the 64^3-node lattice where the factors take 0.2 ms; the CSR is kept for aphip_rk_get_cells.
// Nodal cells (several hexes each, F-bar over their subcells) run on cell tiles over the CSR.
// Lanes in groups stride over a node's (or cell's) entries, accumulate their share of the sum
// and combine the partial sums with a xor butterfly; addition is commutative, so every lane
// ends with the same bits.
constexpr int kCellLanes = 16;
constexpr int kSlotLanes = 8;  // lanes per node of the nodal cells' slot sum

// lanes per node of the two-pass gather (u = Phi d)
constexpr int kGsLanes = 8;
constexpr int kNumXcd = 8;

// Consecutive logical blocks go to the same XCD (the dispatcher places block b on
// XCD b % 8), so neighbouring cells / nodes share that XCD's L2 for their gathers.
// The grid is padded to a multiple of 8 so the map is a bijection.
__device__ __forceinline__ int64_t xcd_block(int64_t nblocks_padded) {
    const int64_t b = blockIdx.x;
    const int64_t per = nblocks_padded / kNumXcd;
    return (b % kNumXcd) * per + b / kNumXcd;
}

template <int LANES>
__device__ __forceinline__ double group_sum(double x) {
#pragma unroll
    for (int s = LANES / 2; s >= 1; s >>= 1) x += __shfl_xor(x, s, LANES);
    return x;
}

struct RkNodeArgs {
    int64_t nn, nblocks;
    const double *mass;
    const uint8_t *fixed;
    double *f, *a, *v, *u;
    double dt;
    // mode 2, 1: another step of the same call follows with the same dt.  The node then
    // also takes that step's predictor (u and v are what k_predict would leave) and stores
    // neither f nor a, which that step overwrites unread
    int more;
    int raw;  // mode 2: the step's predictor has not been taken yet
};

// Node i's force f is complete: store it and finish the node (MODE 0: force only,
// 1: a = f/m, 2: central-difference corrector).
template <int MODE>
__device__ __forceinline__ void rk_finish(const RkNodeArgs &A, int64_t i, const double (&f)[3]) {
    if constexpr (MODE == 2) {
        double u[3], vh[3], a1[3], v1[3];
        ld3(A.v, i, vh);
        const unsigned fx = A.fixed ? A.fixed[i] : 0u;
        if (A.more || A.raw) ld3(A.u, i, u);
        if (A.raw) {
            double v0[3] = {vh[0], vh[1], vh[2]}, a0[3], u0[3] = {u[0], u[1], u[2]};
            ld3(A.a, i, a0);
            cd_predict(u0, v0, a0, fx, A.dt, vh, u);
            if (!A.more) st3(A.u, i, u);
        }
        cd_correct(f, A.mass[i], fx, A.dt, vh, a1, v1);
        if (A.more) {
            double u1[3];
            cd_predict(u, v1, a1, fx, A.dt, vh, u1);
            st3(A.u, i, u1);
            st3(A.v, i, vh);
        } else {
            st3(A.f, i, f);
            st3(A.a, i, a1);
            st3(A.v, i, v1);
        }
    } else {
        st3(A.f, i, f);
        if constexpr (MODE == 1) {
            const double m = A.mass[i];
            const double a1[3] = {f[0] / m, f[1] / m, f[2] / m};
            st3(A.a, i, a1);
        }
    }
}

// ---- nodal cells on cell tiles -------------------------------------------
// A tile is a run of consecutive (Morton-ordered) cells; its node set is the sorted
// union of their node lists and every entry carries its node's index in that set
// (uint16).  One wave per tile:
//   A. stages u of the tile's nodes in LDS and clears one force row per tile node,
//   B. takes 64 / LPC cells at a time, LPC lanes per cell: each lane loads its
//      entries (lane j: j, j + LPC, ...; the first K stay in registers), sums its
//      share of H = sum_t u_node(t) (x) grad phi_t from the staged u, the group
//      combines the shares with a xor butterfly and every lane of the group
//      evaluates the stress; the lanes then add the entry forces -V P grad phi_t of
//      their registered entries into the LDS rows of the entries' nodes,
//   C. writes the tile's rows to its slots (tile-major, coalesced).
// Each entry's grad phi is read from HBM once per step: the reference's per-entry
// atomic scatter (include/ComputeInternalForceSmoothedCell.h:312-351) becomes LDS
// adds of one wave, in program order, and a node pass that sums each node's slots in
// ascending tile order and finishes the node.  Both are fixed orders, so the result
// is the same bits on every run.
struct RkTileArgs {
    int64_t ncells, ntiles, nblocks;
    int maxtn;
    const int64_t *start;
    const uint16_t *lidx;     // [nnz] entry -> index in its tile's node set
    const double *dphi;
    const double *volume;
    const double *u;
    const int32_t *t_nstart;  // [ntiles + 1] offsets of the tile node sets
    const int32_t *t_node;    // [total] internal node ids, ascending within a tile
    const int64_t *t_cstart;  // [ntiles + 1] first cell of each tile
    double *slots;            // [total * 3] tile force rows, tile-major
    double *H, *P;
    const double *state_n;
    double *state_np1;
    MatParams mat;
    const double *elem_lambda, *elem_mu;
    const double *Hn, *Pn;
    double rate_dt;
    int keep;  // 0: an inner step, H and P are not stored
    // raw: u is predicted on the way (the nodes below n_dof; dt is rate_dt)
    int raw;
    int64_t n_dof;
    const double *v, *a;
    const uint8_t *fixed;
};

// u of the tile's nodes tb .. tb + tn - 1 to U, by blockDim threads, in batches of kStage rows a
// thread, every load of a batch issued before its first LDS write (a load and its write per
// iteration would cost a latency each).
__device__ __forceinline__ void stage_tile_u(const RkTileArgs &A, int tb, int tn, double *U) {
    constexpr int kStage = 4;
    const int nt = blockDim.x;
    for (int l0 = threadIdx.x; l0 < tn; l0 += nt * kStage) {
        int64_t gi[kStage];
#pragma unroll
        for (int r = 0; r < kStage; ++r) gi[r] = A.t_node[tb + min(l0 + nt * r, tn - 1)];
        double ur[kStage][3];
#pragma unroll
        for (int r = 0; r < kStage; ++r) ld3(A.u, gi[r], ur[r]);
        if (A.raw) {
#pragma unroll
            for (int r = 0; r < kStage; ++r) {
                double v[3], a[3], vh[3], u1[3];
                ld3(A.v, gi[r], v);
                ld3(A.a, gi[r], a);
                cd_predict(ur[r], v, a, A.fixed ? A.fixed[gi[r]] : 0u, A.rate_dt, vh, u1);
#pragma unroll
                for (int d = 0; d < 3; ++d) ur[r][d] = gi[r] < A.n_dof ? u1[d] : ur[r][d];
            }
        }
#pragma unroll
        for (int r = 0; r < kStage; ++r)
            if (l0 + nt * r < tn) st3(U, l0 + nt * r, ur[r]);
    }
}

template <int KIND, int LPC, int K>
__global__ __launch_bounds__(64) void k_rk_tile(RkTileArgs A) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) double rk_lds[];
    double *U = rk_lds;
    double *F = rk_lds + 3 * (size_t)A.maxtn;
    const int64_t t = xcd_block(A.nblocks);
    if (t >= A.ntiles) return;
    const int lane = threadIdx.x;
    const int tb = A.t_nstart[t], tn = A.t_nstart[t + 1] - tb;
    stage_tile_u(A, tb, tn, U);
    for (int k = lane; k < 3 * tn; k += 64) F[k] = 0.0;
    __syncthreads();
    constexpr int G = 64 / LPC;
    const int grp = lane / LPC, j = lane % LPC;
    const int64_t c0 = A.t_cstart[t], c1 = A.t_cstart[t + 1];
    for (int64_t cb = c0; cb < c1; cb += G) {
        const int64_t c_raw = cb + grp;
        const bool live = c_raw < c1;
        const int64_t c = live ? c_raw : c1 - 1;  // idle groups recompute the tile's last cell, store nothing
        const int64_t t0 = A.start[c], t1 = A.start[c + 1];
        double H[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, P[9];
        double gr[K][3] = {};
        int li[K] = {};
        if (t1 > t0) {
#pragma unroll
            for (int r = 0; r < K; ++r) {
                const int64_t e = min(t0 + j + r * LPC, t1 - 1);
                li[r] = A.lidx[e];
                ld3(A.dphi, e, gr[r]);
            }
#pragma unroll
            for (int r = 0; r < K; ++r) {
                const bool in = t0 + j + r * LPC < t1;
#pragma unroll
                for (int b = 0; b < 3; ++b) gr[r][b] = in ? gr[r][b] : 0.0;
                double uj[3];
                ld3(U, li[r], uj);
#pragma unroll
                for (int a = 0; a < 3; ++a)
#pragma unroll
                    for (int b = 0; b < 3; ++b) H[3 * a + b] = __fma_rn(uj[a], gr[r][b], H[3 * a + b]);
            }
        }
        for (int64_t e = t0 + j + K * LPC; e < t1; e += LPC) {  // entries past the registered ones
            double uj[3], g[3];
            ld3(U, A.lidx[e], uj);
            ld3(A.dphi, e, g);
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) H[3 * a + b] = __fma_rn(uj[a], g[b], H[3 * a + b]);
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) H[i] = group_sum<LPC>(H[i]);
        MatParams m = A.mat;
        if (A.elem_lambda) {
            m.lambda = A.elem_lambda[c];
            m.mu = A.elem_mu[c];
        }
        double snp1 = 0.0, aux = 0.0;
        const double sn = load_state<KIND>(A.state_n, c), sn2 = load_state2<KIND>(A.state_n, c);
        RateIn rin;
        load_rate<KIND>(rin, A.Hn, A.Pn, A.ncells, c, A.rate_dt);
        stress<KIND>(H, m, sn, snp1, aux, P, &rin, sn2);
        snp1 = cell_damage_marker<KIND>(snp1, m);
        if (live && j == 0) {
            store_state<KIND>(A.state_np1, c, snp1, aux);
            // plain stores: one lane per cell writes H and P, a sparse stream that
            // measured 2 % faster through the L2 than as non-temporal stores
            if (A.keep) {
#pragma unroll
                for (int i = 0; i < 9; ++i) {
                    A.H[i * A.ncells + c] = H[i];
                    A.P[i * A.ncells + c] = P[i];
                }
            }
        }
        if (!live) continue;
        const double mv = -A.volume[c];
#pragma unroll
        for (int r = 0; r < K; ++r) {
            if (t0 + j + r * LPC < t1) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const double fa = mv * dot3(P[3 * a], gr[r][0], P[3 * a + 1], gr[r][1], P[3 * a + 2], gr[r][2]);
                    __hip_atomic_fetch_add(F + 3 * li[r] + a, fa, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
        }
        for (int64_t e = t0 + j + K * LPC; e < t1; e += LPC) {
            double g[3];
            ld3(A.dphi, e, g);
            const int lr = A.lidx[e];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double fa = mv * dot3(P[3 * a], g[0], P[3 * a + 1], g[1], P[3 * a + 2], g[2]);
                __hip_atomic_fetch_add(F + 3 * lr + a, fa, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    __syncthreads();
    double *dst = A.slots + 3 * (int64_t)tb;
    for (int k = lane; k < 3 * tn; k += 64) dst[k] = F[k];
}

// F-bar on cell tiles (ComputeInternalForceSmoothedCell.h:120-413): a tile holds whole
// nodal cells, so every pass of the F-bar force runs inside one workgroup with the subcell
// rows in LDS: (1) subcell H (LPC lanes per subcell, butterfly) and J = DetApIm1(H) + 1;
// (2) one lane per subcell: J-bar of its cell (the cell's J_k V_k summed in order over
// V_cell, :120-175), H-bar = H cbrt(J-bar / J) + (cbrt(.) - 1) I unless the ratio is
// within 3 eps of 1, the stress of H-bar (:177-213) and the subcell's term of the dual
// pressure; (3) one lane per subcell: the dual pressure (the cell's terms in order) and
// the un-barred P = P-bar s + (p - s / (3 J) P-bar : F) J F^-T (UnBarStress, :215-309);
// (4) the entry forces -V P grad phi added into LDS rows as in k_rk_tile, one set of rows per
// wave (a wave's adds are in program order), and the waves' rows summed in wave order.
// The entries are read twice, in (1) and (4).  A tile is one nodal cell of some twenty subcells;
// bound by latency and by the entries' loads (26 B each).  Loading a lane's entries together
// and summing J-bar from volumes in LDS (not one global load after the other) took the kernel
// from 31 to 24.6 us on 41k subcells, and 20 steps with three streams in turn from 400 to 303;
// holding the entries in registers from (1) to (4) (152 VGPRs: 422 us) or loading the next
// subcell's ahead (316 us) did not pay.
constexpr int kFbarSubRow = 29;  // LDS doubles per subcell: H 9, J 1, P-bar 9, dual term 1, P 9

struct FbarTileArgs {
    RkTileArgs T;
    const int32_t *t_fstart;     // [ntiles + 1] first nodal cell of each tile
    const int64_t *fcell_sub;    // [n_fcells + 1] subcell range of each nodal cell
    const double *fcell_volume;  // [n_fcells]
    const int32_t *sub_fcell;    // [ncells] nodal cell of each subcell
    int maxsub;                  // most subcells in one tile
};

template <int KIND, int LPC>
__global__ __launch_bounds__(256) void k_fbar_tile(FbarTileArgs B) {
#pragma clang fp contract(off)
    constexpr double kEps = 2.2204460492503131e-16;
    const RkTileArgs &A = B.T;
    extern __shared__ __align__(16) double rk_lds[];
    const int tid = threadIdx.x, nt = blockDim.x, nw = nt / 64;
    double *U = rk_lds;
    double *F = U + 3 * (size_t)A.maxtn;         // a set of rows per wave
    double *SH = F + 3 * (size_t)A.maxtn * nw;   // [maxsub * 9]
    double *SJ = SH + 9 * (size_t)B.maxsub;
    double *SPb = SJ + B.maxsub;                 // [maxsub * 9]
    double *SD = SPb + 9 * (size_t)B.maxsub;
    // [maxsub * 9] P; before (3) its place 0 holds the subcell's volume, 1 and 2 J-bar and cbrt
    double *SP = SD + B.maxsub;
    const int64_t t = xcd_block(A.nblocks);
    if (t >= A.ntiles) return;
    const int tb = A.t_nstart[t], tn = A.t_nstart[t + 1] - tb;
    const int64_t c0 = A.t_cstart[t], c1 = A.t_cstart[t + 1];
    const int grp = tid / LPC, j = tid % LPC, G = nt / LPC;
    // a subcell's entries, K per lane in flight together (those past the end weighted by zero)
    constexpr int K = LPC == 4 ? 1 : 5;
    auto entries = [&](int64_t e0, int64_t e1, int (&li)[K], double (&g)[K][3]) {
#pragma unroll
        for (int r = 0; r < K; ++r) {
            const int64_t e = min(e0 + r * LPC, e1 - 1);
            li[r] = A.lidx[e];
            ld3(A.dphi, e, g[r]);
        }
    };
    stage_tile_u(A, tb, tn, U);
    for (int k = tid; k < 3 * A.maxtn * nw; k += nt) F[k] = 0.0;
    for (int64_t s = c0 + tid; s < c1; s += nt) SP[9 * (int)(s - c0)] = A.volume[s];
    __syncthreads();
    // (1) subcell H and J
    for (int64_t cb = c0; cb < c1; cb += G) {
        const int64_t c = cb + grp;
        const bool live = c < c1;  // (a lane group is live or idle as a whole)
        if (!live) break;
        double H[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        const int64_t s0 = A.start[c], s1 = A.start[c + 1];
        for (int64_t e = s0 + j; e < s1; e += K * LPC) {
            int li[K];
            double g[K][3];
            entries(e, s1, li, g);
#pragma unroll
            for (int r = 0; r < K; ++r) {
                const bool in = e + r * LPC < s1;
                double uj[3];
                ld3(U, li[r], uj);
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const double gb = in ? g[r][b] : 0.0;
#pragma unroll
                    for (int a = 0; a < 3; ++a) H[3 * a + b] = __fma_rn(uj[a], gb, H[3 * a + b]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) H[i] = group_sum<LPC>(H[i]);
        if (j == 0) {
            const int sl = (int)(c - c0);
#pragma unroll
            for (int i = 0; i < 9; ++i) SH[9 * sl + i] = H[i];
            if (A.keep) {
#pragma unroll
                for (int i = 0; i < 9; ++i) store_once(A.H + i * A.ncells + c, H[i]);
            }
            SJ[sl] = det_ap_im1(H) + 1.0;
        }
    }
    __syncthreads();
    // (2) H-bar, its stress, the dual-pressure term
    for (int64_t s = c0 + tid; s < c1; s += nt) {
        const int sl = (int)(s - c0);
        const int64_t r = B.sub_fcell[s];
        const int k0 = (int)(B.fcell_sub[r] - c0), k1 = (int)(B.fcell_sub[r + 1] - c0);
        double jbar = 0.0;
        for (int k = k0; k < k1; ++k) jbar = jbar + SJ[k] * SP[9 * k];
        jbar = jbar / B.fcell_volume[r];
        double H[9], Hb[9], Pb[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) H[i] = SH[9 * sl + i];
        const double ratio = jbar / SJ[sl];
        const double js = cbrt(ratio);
        const bool same = fabs(ratio - 1.0) < 3.0 * kEps;
#pragma unroll
        for (int i = 0; i < 9; ++i) Hb[i] = same ? H[i] : H[i] * js;
        const double add = same ? 0.0 : js - 1.0;
        if (!same) {
            Hb[0] += add;
            Hb[4] += add;
            Hb[8] += add;
        }
        double snp1 = 0.0, aux = 0.0;
        const double sn = load_state<KIND>(A.state_n, s);
        stress<KIND>(Hb, A.mat, sn, snp1, aux, Pb);
        store_state<KIND>(A.state_np1, s, snp1, aux);
#pragma unroll
        for (int i = 0; i < 9; ++i) SPb[9 * sl + i] = Pb[i];
        const double djb = js / (3.0 * jbar);
        double ph = 0.0;
#pragma unroll
        for (int i = 0; i < 9; ++i) ph += Pb[i] * H[i];
        const double tr = Pb[0] + Pb[4] + Pb[8];
        SD[sl] = djb * SP[9 * sl] * (ph + tr);
        SP[9 * sl + 1] = js;
    }
    __syncthreads();
    // (3) the dual pressure and the un-barred stress
    for (int64_t s = c0 + tid; s < c1; s += nt) {
        const int sl = (int)(s - c0);
        const int64_t r = B.sub_fcell[s];
        const int k0 = (int)(B.fcell_sub[r] - c0), k1 = (int)(B.fcell_sub[r + 1] - c0);
        double dual = 0.0;
        for (int k = k0; k < k1; ++k) dual += SD[k];
        dual = dual / B.fcell_volume[r];
        const double Js = SJ[sl], js = SP[9 * sl + 1];
        double Fm[9], Fi[9], Pb[9], pf = 0.0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            Fm[i] = SH[9 * sl + i];
            Pb[i] = SPb[9 * sl + i];
        }
        Fm[0] += 1.0;
        Fm[4] += 1.0;
        Fm[8] += 1.0;
#pragma unroll
        for (int i = 0; i < 9; ++i) pf += Pb[i] * Fm[i];
        const double djj = -js / (3.0 * Js);
        const double scalar = (dual + djj * pf) * Js;
        inverse3(Fm, Fi);
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const double p = Pb[3 * a + b] * js + scalar * Fi[3 * b + a];
                SP[9 * sl + 3 * a + b] = p;
                if (A.keep) store_once(A.P + (3 * a + b) * A.ncells + s, p);
            }
    }
    __syncthreads();
    // (4) entry forces
    double *Fw = F + 3 * (size_t)A.maxtn * (tid / 64);
    for (int64_t cb = c0; cb < c1; cb += G) {
        const int64_t c = cb + grp;
        if (c >= c1) break;
        const int sl = (int)(c - c0);
        double P[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) P[i] = SP[9 * sl + i];
        const double mv = -A.volume[c];
        const int64_t s0 = A.start[c], s1 = A.start[c + 1];
        for (int64_t e = s0 + j; e < s1; e += K * LPC) {
            int li[K];
            double g[K][3];
            entries(e, s1, li, g);
#pragma unroll
            for (int r = 0; r < K; ++r) {
                if (e + r * LPC < s1) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const double fa = mv * dot3(P[3 * a], g[r][0], P[3 * a + 1], g[r][1], P[3 * a + 2], g[r][2]);
                        __hip_atomic_fetch_add(Fw + 3 * li[r] + a, fa, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
            }
        }
    }
    __syncthreads();
    double *dst = A.slots + 3 * (int64_t)tb;
    for (int k = tid; k < 3 * tn; k += nt) {
        double f = F[k];
        for (int q = 1; q < nw; ++q) f += F[3 * (size_t)A.maxtn * q + k];
        dst[k] = f;
    }
}

struct RkSlotNodeArgs {
    RkNodeArgs out;
    const int64_t *nslot_start;  // [n + 1] slot range of each node
    const int32_t *nslot;        // slots (tile-node positions) of each node, ascending tile
    const double *slots;
};

// f_i = sum of node i's tile rows in ascending tile order (lanes stride over them,
// then the butterfly), then the node update.
template <int MODE, int LANES>
__global__ __launch_bounds__(256) void k_rk_slot_nodes(RkSlotNodeArgs A) {
#pragma clang fp contract(off)
    const int l = threadIdx.x & (LANES - 1);
    const int64_t i_raw = xcd_block(A.out.nblocks) * (256 / LANES) + (threadIdx.x / LANES);
    const bool live = i_raw < A.out.nn;
    const int64_t i = live ? i_raw : A.out.nn - 1;
    double f[3] = {0.0, 0.0, 0.0};
    const int64_t s0 = A.nslot_start[i], s1 = A.nslot_start[i + 1];
    for (int64_t s = s0 + l; s < s1; s += LANES) {
        double r[3];
        ld3(A.slots, A.nslot[s], r);
        f[0] += r[0];
        f[1] += r[1];
        f[2] += r[2];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) f[d] = group_sum<LANES>(f[d]);
    if (!live || l != 0) return;
    rk_finish<MODE>(A.out, i, f);
}

// ---- two-pass method: gather before, scatter after the cell force -----------
struct RkGatherArgs {
    int64_t nn, nblocks;
    const int32_t *num, *nbr;
    const double *phi;
    const double *src;  // coefficients [nn * 3]
    double *dst;        // physical values [nn * 3]
    int copy_lonely;    // two-pass: a node without neighbors copies its coefficient (one-pass: zero)
    // RAW: the coefficients are predicted on the way
    const double *v, *a;
    const uint8_t *fixed;
    double dt;
};

// dst_i = sum_k phi_ik src_(nbr_ik): LANES lanes per node, lane l takes entries
// l, l + LANES, ... of the node's row (contiguous across the lanes), the partial
// sums are combined by the xor butterfly.
// (8 lanes, five entries each for a full row of 40: 3 % faster than 16 lanes.)
template <int LANES, bool RAW>
__global__ __launch_bounds__(256) void k_rk_gather(RkGatherArgs A) {
    auto coefficient = [&](int64_t j, double (&x)[3]) {
        if constexpr (RAW) {
            double u[3], v[3], a[3], vh[3];
            ld3(A.src, j, u);
            ld3(A.v, j, v);
            ld3(A.a, j, a);
            cd_predict(u, v, a, A.fixed ? A.fixed[j] : 0u, A.dt, vh, x);
        } else {
            ld3(A.src, j, x);
        }
    };
    constexpr int R = (kMaxNbr + LANES - 1) / LANES;
    const int l = threadIdx.x & (LANES - 1);
    const int64_t i_raw = xcd_block(A.nblocks) * (256 / LANES) + (threadIdx.x / LANES);
    const bool live = i_raw < A.nn;
    const int64_t i = live ? i_raw : A.nn - 1;
    const int n = A.num[i];
    const int64_t row = i * kMaxNbr;
    int32_t j[R];
    double w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = l + r * LANES;
        const int kk = max(min(k, n - 1), 0);  // inside the row; entries past n are weighted by zero
        const int32_t jl = A.nbr[row + kk];
        const double wl = A.phi[row + kk];
        j[r] = n > 0 ? jl : (int32_t)i;
        w[r] = k < n ? wl : 0.0;
    }
    double s[3] = {0.0, 0.0, 0.0};
    double x[R][3];
#pragma unroll
    for (int r = 0; r < R; ++r) coefficient(j[r], x[r]);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int d = 0; d < 3; ++d) s[d] += x[r][d] * w[r];
#pragma unroll
    for (int d = 0; d < 3; ++d) s[d] = group_sum<LANES>(s[d]);
    if (!live || l != 0) return;
    if (n == 0 && A.copy_lonely) coefficient(i, s);
    A.dst[3 * i] = s[0];
    A.dst[3 * i + 1] = s[1];
    A.dst[3 * i + 2] = s[2];
}

struct RkScatterArgs {
    RkNodeArgs out;          // force and node update of the coefficients
    const int32_t *num;
    const int64_t *rstart;   // [nn + 1] reverse neighbor lists
    const int32_t *rsrc;     // points i listing the node, ascending
    const double *rphi;      // phi_iJ of each reverse entry
    const double *src;       // local (physical) force [nn * 3]
    int copy_lonely;         // two-pass: a node without neighbors takes src_J
    // SLOTS: the local force of the nodes from first_shared on is the sum of their slots
    // bstart[j - first_shared] .. (ascending, as the shared-node pass adds them)
    const int32_t *bstart;
    const double *bpart;
    int64_t first_shared;
    double *local;  // also store the shared nodes' local force, or null
};

// f_J = sum over points i that list J of phi_iJ src_i (the transpose of the
// gather), LANES lanes per node over its contiguous reverse entries, NB per lane at a
// time (16 x 3: a reverse list of about 40 entries in one round with little padding;
// 6 % faster than 16 x 4, and than 8 x 5), then the node update.
template <int MODE, int LANES, int NB, bool SLOTS = false>
__global__ __launch_bounds__(256) void k_rk_scatter(RkScatterArgs A) {
    // local force of NB nodes
    auto local = [&](auto &src, auto &x) {
        constexpr int M = sizeof(src) / sizeof(src[0]);
        if constexpr (!SLOTS) {
#pragma unroll
            for (int r = 0; r < M; ++r) ld3(A.src, src[r], x[r]);
        } else {
            const double *p[M];
            int left[M], most = 1;
#pragma unroll
            for (int r = 0; r < M; ++r) {
                p[r] = A.src + 3 * (int64_t)src[r];
                left[r] = 1;
                if (const int64_t b = src[r] - A.first_shared; b >= 0) {
                    const int32_t s0 = A.bstart[b];
                    left[r] = A.bstart[b + 1] - s0;
                    if (left[r] > 0) p[r] = A.bpart + 3 * (int64_t)s0;  // (a node of no element has no slot)
                }
                most = max(most, left[r]);
                x[r][0] = x[r][1] = x[r][2] = 0.0;
            }
            constexpr int Q = 2;
            for (int q = 0; q < most; q += Q) {
                double y[M][Q][3];
#pragma unroll
                for (int r = 0; r < M; ++r)
#pragma unroll
                    for (int k = 0; k < Q; ++k) ld3(p[r], max(min(q + k, left[r] - 1), 0), y[r][k]);
#pragma unroll
                for (int r = 0; r < M; ++r)
#pragma unroll
                    for (int k = 0; k < Q; ++k)
#pragma unroll
                        for (int d = 0; d < 3; ++d) x[r][d] += q + k < left[r] ? y[r][k][d] : 0.0;
            }
        }
    };
    const int l = threadIdx.x & (LANES - 1);
    const int64_t i_raw = xcd_block(A.out.nblocks) * (256 / LANES) + (threadIdx.x / LANES);
    const bool live = i_raw < A.out.nn;
    const int64_t i = live ? i_raw : A.out.nn - 1;
    double f[3] = {0.0, 0.0, 0.0};
    const int64_t t0 = A.rstart[i], t1 = A.rstart[i + 1];
    for (int64_t tb = t0 + l; tb < t1; tb += NB * LANES) {
        int32_t src[NB];
        double w[NB], x[NB][3];
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const int64_t t = min(tb + r * LANES, t1 - 1);
            src[r] = A.rsrc[t];
            w[r] = tb + r * LANES < t1 ? A.rphi[t] : 0.0;
        }
        local(src, x);
#pragma unroll
        for (int r = 0; r < NB; ++r)
#pragma unroll
            for (int d = 0; d < 3; ++d) f[d] += x[r][d] * w[r];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) f[d] = group_sum<LANES>(f[d]);
    if (!live || l != 0) return;
    const bool lonely = A.copy_lonely && A.num[i] == 0;
    if (lonely || (SLOTS && A.local && i >= A.first_shared)) {
        const int32_t self[1] = {(int32_t)i};
        double x[1][3];
        local(self, x);
        if (SLOTS && A.local && i >= A.first_shared) st3(A.local, i, x[0]);
        if (lonely) {
#pragma unroll
            for (int d = 0; d < 3; ++d) f[d] = x[0][d];
        }
    }
    rk_finish<MODE>(A.out, i, f);
}

// mass_from_elements: rho V / NPE from every cell touching the node, ascending cell
template <int NPE>
__global__ __launch_bounds__(256) void k_rk_mfe(int64_t nn, const int32_t *node_start, const int32_t *node_inc,
                                                const double *vol, double rho, double *mfe) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nn) return;
    double m = 0.0;
    for (int32_t t = node_start[i]; t < node_start[i + 1]; ++t) m += (vol[node_inc[t] / NPE] * rho) / NPE;
    mfe[i] = m;
}

// m_J = sum over points i that list J of phi_iJ * mfe_i, ascending i (ScatterValues)
__global__ __launch_bounds__(256) void k_rk_mass(int64_t nn, const int32_t *num, const int64_t *rstart,
                                                 const int32_t *rsrc, const double *rphi, const double *mfe,
                                                 double *mass) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= nn) return;
    if (num[j] == 0) {
        mass[j] = mfe[j];
        return;
    }
    double m = 0.0;
    for (int64_t t = rstart[j]; t < rstart[j + 1]; ++t) m += mfe[rsrc[t]] * rphi[t];
    mass[j] = m;
}

inline dim3 grid1(int64_t n, int block) { return dim3((unsigned)((n + block - 1) / block)); }

// blocks of 256 / lanes groups for n groups, padded to a multiple of the XCD count
inline int64_t padded_groups(int64_t n, int lanes = kCellLanes) {
    const int64_t per = 256 / lanes, nb = (n + per - 1) / per;
    return ((nb + kNumXcd - 1) / kNumXcd) * kNumXcd;
}

// counts -> exclusive prefix (host) -> device start array of n+1 entries
template <typename T>
void scan_counts(Ctx &c, const DevBuf<int32_t> &counts, int64_t n, DevBuf<T> &start, int64_t *total) {
    std::vector<int32_t> h(n);
    counts.download(h.data(), n, c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    std::vector<T> s(n + 1, 0);
    for (int64_t i = 0; i < n; ++i) s[i + 1] = s[i] + (T)h[i];
    start.upload(s.data(), s.size(), c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    if (total) *total = (int64_t)s[n];
}

}  // namespace

void fe_smoothing_setup(Ctx &c);
void rk_cells_and_order(Ctx &c, bool two_pass, bool elem_cells);
void rk_cells_order(Ctx &c);

// Nodal cells of a thex mesh (MeshLabelerProcessor.h:227-330, :690-827): marks each hex's
// node of lowest caller id active, checks that every hex then holds exactly one active
// node, renumbers the internal nodes with the active ones first (c.n_dof of them) and
// records, per cell (active node, ascending caller id) its hexes in ascending caller
// element id; with subdomains 0 every hex is a subcell, with 1 the whole cell.  Returns
// the subcells as element lists (sub_start / sub_elems, internal element ids).
static void nodal_label(Ctx &c, int subdomains, std::vector<int64_t> &sub_start, std::vector<int32_t> &sub_elems) {
    CellData &D = c.cells;
    const int64_t nn = c.nn, ne = c.ne;
    APHIP_REQUIRE(c.etype == APHIP_HEX8,
                  "Nodal integration will only work correctly when being built from hexahedral elements. Use 'thex' "
                  "to divide a tetrahedral mesh into hexahedral elements.");
    APHIP_REQUIRE(subdomains == 0 || subdomains == 1, "nodal smoothing cells take subdomains 0 or 1");
    std::vector<uint8_t> act(nn, 0);
    for (int64_t e = 0; e < ne; ++e) {
        int best = 0;
        for (int k = 1; k < 8; ++k)
            if (c.node_iperm[c.conn_h[8 * e + k]] < c.node_iperm[c.conn_h[8 * e + best]]) best = k;
        act[c.conn_h[8 * e + best]] = 1;
    }
    for (int64_t e = 0; e < ne; ++e) {
        int n = 0;
        for (int k = 0; k < 8; ++k) n += act[c.conn_h[8 * e + k]];
        APHIP_REQUIRE(n == 1, "Nodal integration requires exactly one active node per element. Found " +
                                  std::to_string(n) + " active nodes in element " +
                                  std::to_string(c.elem_iperm[e]) + ".");
    }
    // active nodes first, each group in its current (Morton) order
    std::vector<int32_t> old_of_new;
    old_of_new.reserve(nn);
    for (int64_t i = 0; i < nn; ++i)
        if (act[i]) old_of_new.push_back((int32_t)i);
    const int64_t n_act = (int64_t)old_of_new.size();
    for (int64_t i = 0; i < nn; ++i)
        if (!act[i]) old_of_new.push_back((int32_t)i);
    renumber_nodes(c, old_of_new);
    c.tiles.reset();  // the tile plan's node groups are void after the renumbering
    c.patch.reset();
    c.n_dof = n_act;
    // cells: active nodes by caller id; hexes by caller element id
    std::vector<int32_t> act_nodes(n_act);
    std::iota(act_nodes.begin(), act_nodes.end(), 0);
    std::sort(act_nodes.begin(), act_nodes.end(),
              [&](int32_t x, int32_t y) { return c.node_iperm[x] < c.node_iperm[y]; });
    std::vector<int32_t> cell_of_node(n_act);
    for (int64_t r = 0; r < n_act; ++r) cell_of_node[act_nodes[r]] = (int32_t)r;
    std::vector<int32_t> hexes(ne);
    std::iota(hexes.begin(), hexes.end(), 0);
    std::vector<int32_t> hex_cell(ne);
    for (int64_t e = 0; e < ne; ++e)
        for (int k = 0; k < 8; ++k)
            if (c.conn_h[8 * e + k] < n_act) hex_cell[e] = cell_of_node[c.conn_h[8 * e + k]];
    std::sort(hexes.begin(), hexes.end(), [&](int32_t x, int32_t y) {
        return hex_cell[x] != hex_cell[y] ? hex_cell[x] < hex_cell[y] : c.elem_iperm[x] < c.elem_iperm[y];
    });
    D.n_fcells = n_act;
    std::vector<int64_t> cell_start(n_act + 1, 0);
    for (int64_t e = 0; e < ne; ++e) cell_start[hex_cell[e] + 1]++;
    for (int64_t r = 0; r < n_act; ++r) cell_start[r + 1] += cell_start[r];
    sub_elems = hexes;
    if (subdomains == 0) {
        sub_start.resize(ne + 1);
        std::iota(sub_start.begin(), sub_start.end(), 0);
        D.fcell_sub_h = cell_start;
    } else {
        sub_start = cell_start;
        D.fcell_sub_h.resize(n_act + 1);
        std::iota(D.fcell_sub_h.begin(), D.fcell_sub_h.end(), 0);
    }
}

// Subcell node lists (first-seen union of the neighbors of the nodes of the subcell's
// hexes, in hex order) and derivatives sum_e sum_k B_k V_e phi / V_sub
// (SmoothedCellDataProcessor.h:407-675), built on the host from the device's neighbor
// lists and functions; cell volumes are the sums of their hexes' volumes.
static void nodal_subcells(Ctx &c, const std::vector<int64_t> &sub_start, const std::vector<int32_t> &sub_elems) {
    CellData &D = c.cells;
    const int64_t nn = c.nn, ne = c.ne, ns = (int64_t)sub_start.size() - 1;
    std::vector<int32_t> hn(nn), hb(nn * kMaxNbr);
    std::vector<double> hp(nn * kMaxNbr), hX(3 * nn);
    D.num_nbr.download(hn.data(), nn, c.stream);
    D.nbr.download(hb.data(), hb.size(), c.stream);
    D.phi.download(hp.data(), hp.size(), c.stream);
    c.X.download(hX.data(), hX.size(), c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    std::vector<int64_t> start(ns + 1, 0);
    std::vector<int32_t> nodes;
    std::vector<double> dphi, vsub(ns, 0.0), evol(ne, 0.0);
    std::vector<int64_t> stamp(nn, -1);
    std::vector<int32_t> pos(nn, 0);
    D.sub_of_elem.assign(ne, -1);
    D.sub_first_elem.assign(ns, -1);
    for (int64_t sc = 0; sc < ns; ++sc) {
        const int64_t t0 = (int64_t)nodes.size();
        start[sc] = t0;
        for (int64_t q = sub_start[sc]; q < sub_start[sc + 1]; ++q) {
            const int32_t e = sub_elems[q];
            D.sub_of_elem[e] = (int32_t)sc;
            if (q == sub_start[sc]) D.sub_first_elem[sc] = e;
            for (int k = 0; k < 8; ++k) {
                const int32_t a = c.conn_h[8 * (int64_t)e + k];
                for (int l = 0; l < hn[a]; ++l) {
                    const int32_t j = hb[(int64_t)a * kMaxNbr + l];
                    if (stamp[j] != sc) {
                        stamp[j] = sc;
                        pos[j] = (int32_t)((int64_t)nodes.size() - t0);
                        nodes.push_back(j);
                    }
                }
            }
        }
        dphi.resize(3 * nodes.size(), 0.0);
        double vs = 0.0;
        for (int64_t q = sub_start[sc]; q < sub_start[sc + 1]; ++q) {
            const int32_t e = sub_elems[q];
            double Xe[8][3], B[8][3], V;
            for (int k = 0; k < 8; ++k)
                for (int d = 0; d < 3; ++d) Xe[k][d] = hX[3 * (int64_t)c.conn_h[8 * (int64_t)e + k] + d];
            smoothed_hex8(Xe, B, V);
            evol[e] = V;
            vs += V;
            for (int k = 0; k < 8; ++k) {
                const int32_t a = c.conn_h[8 * (int64_t)e + k];
                for (int l = 0; l < hn[a]; ++l) {
                    const int32_t j = hb[(int64_t)a * kMaxNbr + l];
                    const double fv = hp[(int64_t)a * kMaxNbr + l];
                    double *dp = &dphi[3 * (t0 + pos[j])];
                    for (int m = 0; m < 3; ++m) dp[m] += B[k][m] * V * fv;
                }
            }
        }
        for (size_t t = 3 * t0; t < dphi.size(); ++t) dphi[t] /= vs;
        vsub[sc] = vs;
    }
    start[ns] = (int64_t)nodes.size();
    D.ncells = ns;
    D.nnz = start[ns];
    APHIP_REQUIRE(D.nnz < (int64_t)INT32_MAX, "too many cell entries for int32 incidences");
    D.start.upload(start.data(), start.size(), c.stream);
    D.nodes.upload(nodes.data(), std::max<size_t>(nodes.size(), 1), c.stream);
    D.dphi.upload(dphi.data(), std::max<size_t>(dphi.size(), 1), c.stream);
    D.volume.upload(vsub.data(), std::max<int64_t>(ns, 1), c.stream);
    D.evol.upload(evol.data(), std::max<int64_t>(ne, 1), c.stream);
    // nodal cells: subcell ranges and volumes (sum of the cell's hex volumes, in order)
    std::vector<double> vcell(D.n_fcells, 0.0);
    for (int64_t r = 0; r < D.n_fcells; ++r)
        for (int64_t sc = D.fcell_sub_h[r]; sc < D.fcell_sub_h[r + 1]; ++sc)
            for (int64_t q = sub_start[sc]; q < sub_start[sc + 1]; ++q) vcell[r] += evol[sub_elems[q]];
    D.fcell_sub.upload(D.fcell_sub_h.data(), D.fcell_sub_h.size(), c.stream);
    D.fcell_volume.upload(vcell.data(), std::max<int64_t>(D.n_fcells, 1), c.stream);
    if (D.fbar) {
        std::vector<int32_t> sc_of(std::max<int64_t>(ns, 1), 0);
        for (int64_t r = 0; r < D.n_fcells; ++r)
            for (int64_t sc = D.fcell_sub_h[r]; sc < D.fcell_sub_h[r + 1]; ++sc) sc_of[sc] = (int32_t)r;
        D.sub_fcell.upload(sc_of.data(), sc_of.size(), c.stream);
    }
    APHIP_HIP(hipStreamSynchronize(c.stream));
}

// The element cells' force runs on the element tile plan, one element per thread: built
// here when the context has none (APHIP_FLAG_TWO_PASS, a nodal set-up before this one) or
// has the eight-lanes-per-Hex8 shape.  64 elements always fit a CU's LDS.  RKPM cells on Tet4
// take smaller tiles than the mesh's default unless the caller set them: 256 elements on the
// small meshes, where a workgroup of 1024 keeps its CU's issue slots busy four times as long
// (alone, 10 steps of 16k cells in two launches: 291 -> 218 us), else 512, whose workgroups
// leave room for a second one on the CU (10 steps of 750k cells: 742 -> 719 us).
static void ensure_element_tiles(Ctx &c, bool fe_cells) {
    auto fits = [&] {
        return c.tiles.ready && c.tiles.threads == c.tiles.te && c.tiles.cell_lds_bytes <= 160 * 1024;
    };
    int te0 = c.npe == 4 ? 1024 : 128;
    if (c.npe == 4 && !fe_cells && !c.tiles.by_user) te0 = c.nn <= kFusedNodes ? 256 : 512;
    if (c.ne == 0 || (fits() && c.tiles.te <= te0)) return;
    for (int te = te0;; te /= 2) {
        try {
            tile_build(c, te, te);
            if (fits()) return;
        } catch (const Error &e) {
            if (te <= 64 || e.code != APHIP_ERR_INVALID) throw;
        }
    }
}

void rk_setup(Ctx &c, double scale, bool two_pass, bool fe_cells, int nodal_subdomains, bool fbar) {
    CellData &D = c.cells;
    D.reset();
    c.n_dof = c.nn;
    const int64_t nn = c.nn;
    if (nodal_subdomains < 0) ensure_element_tiles(c, fe_cells);  // (renumbers the nodes: before anything refers to them)
    if (fe_cells) {
        fe_smoothing_setup(c);
        return;
    }
    if (scale == 1.0) scale += 1.0e-6;  // src/NeighborSearchProcessor.cpp:161-163
    const bool nodal = nodal_subdomains >= 0;
    std::vector<int64_t> sub_start;
    std::vector<int32_t> sub_elems;
    if (nodal) {
        nodal_label(c, nodal_subdomains, sub_start, sub_elems);
        D.nodal = true;
        // F-bar only where a cell holds more than one subcell (ComputeInternalForceSmoothedCell.h:458-459)
        D.fbar = fbar && (int64_t)sub_start.size() - 1 != D.n_fcells;
    }
    const int64_t n_act = c.n_dof;  // search candidates: the nodes with degrees of freedom

    // kernel radius from the max edge length
    D.radius.alloc(nn);
    const bool hex = c.etype == APHIP_HEX8;  // Hex8 background: ElementReproducingKernelHex8
    hipLaunchKernelGGL(hex ? k_max_edge<8> : k_max_edge<4>, grid1(nn, 256), dim3(256), 0, c.stream, nn, c.node_start.p,
                       c.node_inc.p, c.conn.p, c.X.p, scale, n_act, D.radius.p);
    APHIP_HIP(hipGetLastError());

    // uniform cell list of the candidates with cell edge = their largest radius
    std::vector<double> hX(3 * nn), hr(nn);
    c.X.download(hX.data(), hX.size(), c.stream);
    D.radius.download(hr.data(), hr.size(), c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    Grid G;
    double hi[3];
    for (int d = 0; d < 3; ++d) {
        G.lo[d] = INFINITY;
        hi[d] = -INFINITY;
    }
    double rmax = 0.0;
    for (int64_t i = 0; i < nn; ++i) {
        for (int d = 0; d < 3; ++d) {
            G.lo[d] = std::min(G.lo[d], hX[3 * i + d]);
            hi[d] = std::max(hi[d], hX[3 * i + d]);
        }
        if (i < n_act) rmax = std::max(rmax, hr[i]);
    }
    double ext = 0.0;
    for (int d = 0; d < 3; ++d) ext = std::max(ext, hi[d] - G.lo[d]);
    G.cell = rmax > 0.0 ? rmax : (ext > 0.0 ? ext : 1.0);
    // keep the grid modest; a coarser cell only adds candidates, never drops one
    while (true) {
        int64_t tot = 1;
        for (int d = 0; d < 3; ++d) {
            G.nb[d] = (int)std::floor((hi[d] - G.lo[d]) / G.cell) + 1;
            tot *= G.nb[d];
        }
        if (tot <= (int64_t)1 << 24) break;
        G.cell *= 1.26;
    }
    const int64_t nbins = (int64_t)G.nb[0] * G.nb[1] * G.nb[2];
    DevBuf<int32_t> bin_of, bcount, bstart, bfill, items;
    bin_of.alloc(std::max<int64_t>(n_act, 1));
    bcount.alloc(nbins);
    bcount.zero(c.stream);
    hipLaunchKernelGGL(k_bin_count, grid1(n_act, 256), dim3(256), 0, c.stream, n_act, c.X.p, G, bin_of.p, bcount.p);
    APHIP_HIP(hipGetLastError());
    scan_counts(c, bcount, nbins, bstart, nullptr);
    bfill.alloc(nbins);
    bfill.zero(c.stream);
    items.alloc(std::max<int64_t>(n_act, 1));
    hipLaunchKernelGGL(k_bin_fill, grid1(n_act, 256), dim3(256), 0, c.stream, n_act, bin_of.p, bstart.p, bfill.p,
                       items.p);
    APHIP_HIP(hipGetLastError());

    // ball search of every node among the candidates, ranked by caller ids for ties
    DevBuf<int32_t> ncand;
    D.num_nbr.alloc(nn);
    D.nbr.alloc(nn * kMaxNbr);
    ncand.alloc(nn);
    SearchArgs S{nn, c.X.p, D.radius.p, c.d_node_iperm.p, G, bstart.p, items.p, D.num_nbr.p, D.nbr.p, ncand.p};
    hipLaunchKernelGGL(k_search, grid1(nn, kSearchBlock), dim3(kSearchBlock), 0, c.stream, S);
    APHIP_HIP(hipGetLastError());
    {
        std::vector<int32_t> hn(nn), hc(nn);
        D.num_nbr.download(hn.data(), nn, c.stream);
        ncand.download(hc.data(), nn, c.stream);
        APHIP_HIP(hipStreamSynchronize(c.stream));
        int64_t tr = 0;
        for (int64_t i = 0; i < nn; ++i) tr += hc[i] - hn[i];
        D.n_truncated = tr;
    }

    // RK function values
    D.phi.alloc(nn * kMaxNbr);
    hipLaunchKernelGGL(k_rk_phi, grid1(nn, 128), dim3(128), 0, c.stream, nn, c.X.p, D.radius.p, D.num_nbr.p, D.nbr.p,
                       D.phi.p);
    APHIP_HIP(hipGetLastError());

    if (nodal) {
        nodal_subcells(c, sub_start, sub_elems);
        rk_cells_order(c);
    } else {
        rk_cells_and_order(c, two_pass, two_pass);
    }
}

// Finite-element strain smoothing with element cells (ElementSmoothedTetrahedron4,
// include/ElementSmoothedTetrahedron4.h): the element's own shape functions, i.e. every
// node its own only "neighbor" with value 1, and the cells of the element's nodes with
// derivative (B_k V) / V (SmoothedCellDataProcessor.h:623-668 with unit function values).
// Phi is the identity, so a step is the fused element tile step; the mass scatter is the
// identity too.
void fe_smoothing_setup(Ctx &c) {
    CellData &D = c.cells;
    D.fe = true;
    const int64_t nn = c.nn;
    D.radius.alloc(nn);
    D.radius.zero(c.stream);
    D.num_nbr.alloc(nn);
    D.nbr.alloc(nn * kMaxNbr);
    D.phi.alloc(nn * kMaxNbr);
    hipLaunchKernelGGL(k_identity_functions, grid1(nn, 256), dim3(256), 0, c.stream, nn, D.num_nbr.p, D.nbr.p,
                       D.phi.p);
    APHIP_HIP(hipGetLastError());
    D.n_truncated = 0;
    rk_cells_and_order(c, false, true);
}

// Cells (element-node cells when elem_cells) and reverse neighbor lists; two_pass selects
// the reference's force method, which fixes what a node without neighbors contributes and
// whether the physical displacement and local force can be read.
void rk_cells_and_order(Ctx &c, bool two_pass, bool elem_cells) {
    CellData &D = c.cells;
    const int64_t nn = c.nn, ne = c.ne;
    const bool hex = c.etype == APHIP_HEX8;
    const int npe = hex ? 8 : 4;
    // smoothed cells: counts, offsets, lists and derivatives
    D.two_pass = two_pass;
    if (elem_cells) {
        // the element's own nodes (SmoothedCellDataProcessor.h:474-486, :637-648)
        D.nnz = npe * ne;
        APHIP_REQUIRE(D.nnz < (int64_t)INT32_MAX, "too many cell entries for int32 incidences");
        std::vector<int64_t> hs(ne + 1);
        for (int64_t e = 0; e <= ne; ++e) hs[e] = npe * e;
        D.start.upload(hs.data(), hs.size(), c.stream);
        D.nodes.alloc(std::max<int64_t>(D.nnz, 1));
        D.dphi.alloc(3 * std::max<int64_t>(D.nnz, 1));
        D.volume.alloc(std::max<int64_t>(ne, 1));
        if (ne) {
            hipLaunchKernelGGL(hex ? k_cell_two_pass<8> : k_cell_two_pass<4>, grid1(ne, 256), dim3(256), 0, c.stream, ne, c.conn.p, c.X.p,
                               D.nodes.p, D.dphi.p, D.volume.p);
            APHIP_HIP(hipGetLastError());
        }
    } else {
        DevBuf<int32_t> clen;
        clen.alloc(std::max<int64_t>(ne, 1));
        if (ne) {
            const int blk = hex ? cell_block<8>() : cell_block<4>();
            hipLaunchKernelGGL(hex ? k_cell_count<8> : k_cell_count<4>, grid1(ne, blk), dim3(blk), 0, c.stream, ne, c.conn.p,
                               D.num_nbr.p, D.nbr.p, clen.p);
            APHIP_HIP(hipGetLastError());
        }
        scan_counts(c, clen, ne, D.start, &D.nnz);
        APHIP_REQUIRE(D.nnz < (int64_t)INT32_MAX, "too many cell entries for int32 incidences");
        D.nodes.alloc(std::max<int64_t>(D.nnz, 1));
        D.dphi.alloc(3 * std::max<int64_t>(D.nnz, 1));
        D.volume.alloc(std::max<int64_t>(ne, 1));
        if (ne) {
            CellFillArgs F{ne, c.conn.p, c.X.p, D.num_nbr.p, D.nbr.p, D.phi.p, D.start.p, D.nodes.p, D.dphi.p,
                           D.volume.p};
            const int blk = hex ? cell_block<8>() : cell_block<4>();
            hipLaunchKernelGGL(hex ? k_cell_fill<8> : k_cell_fill<4>, grid1(ne, blk), dim3(blk), 0, c.stream, F);
            APHIP_HIP(hipGetLastError());
        }
    }

    D.u_phys.alloc(3 * nn);
    D.u_phys.zero(c.stream);
    D.f_local.alloc(3 * nn);
    D.f_local.zero(c.stream);
    D.ncells = ne;
    rk_cells_order(c);
}

// LDS of one tile-kernel workgroup (u and force rows of the tile nodes; F-bar also the
// subcell rows) is kept to 64 KiB so that several tiles share a CU.
constexpr int64_t kTileLdsMax = 64 * 1024;

static int64_t tile_lds(int maxtn, int maxsub, bool fbar) {
    return 48 * (int64_t)std::max(maxtn, 1) + (fbar ? 8 * (int64_t)kFbarSubRow * std::max(maxsub, 1) : 0);
}

// Cell tiles of the nodal cells: runs of tile_cells consecutive cells, the sorted
// union of their node lists, every entry's index in it, and every node's slots (its
// positions in the tile-major node sets, ascending tile).  The tile size starts at 64
// cells (256 for cells of at most four entries), is halved while the mesh gives fewer
// than 2048 tiles (F-bar, whose tiles do several passes over their subcells: 8192; on a
// thex mesh of 192,000 subcells 16 instead of 64 subcells per tile took the step from
// 0.131 to 0.121 ms), and then until every tile's node set fits the LDS budget.  The lanes
// per cell follow the longest cell list (4 up to 4 entries, 8 up to 96, else 16).
// APHIP_RK_TILE_CELLS and APHIP_RK_TILE_LANES override the two choices.
static void rk_tile_plan(Ctx &c) {
    CellData &D = c.cells;
    const int64_t nc = D.ncells, nnz = D.nnz, nn = c.nn;
    std::vector<int64_t> hs(nc + 1, 0);
    std::vector<int32_t> hn(std::max<int64_t>(nnz, 1));
    D.start.download(hs.data(), nc + 1, c.stream);
    if (nnz) D.nodes.download(hn.data(), nnz, c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    int64_t maxlen = 0;
    for (int64_t k = 0; k < nc; ++k) maxlen = std::max(maxlen, hs[k + 1] - hs[k]);
    D.tile_lpc = maxlen <= 4 ? 4 : (maxlen <= 96 ? 8 : 16);
    if (const char *env = std::getenv("APHIP_RK_TILE_LANES")) {
        const int v = std::atoi(env);
        if (v == 4 || v == 8 || v == 16) D.tile_lpc = v;
    }
    int tc = D.tile_lpc == 4 ? 256 : 64;
    // small meshes: at least 2048 tiles (eight waves per CU; F-bar 8192) while a tile keeps 8 cells
    const int64_t min_tiles = D.fbar ? 8192 : 2048;
    while (tc > 8 && (nc + tc - 1) / tc < min_tiles) tc /= 2;
    if (const char *env = std::getenv("APHIP_RK_TILE_CELLS")) {
        const int v = std::atoi(env);
        if (v >= 1 && v <= 4096) tc = v;
    }
    const int nthreads = (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    std::vector<uint16_t> lidx(std::max<int64_t>(nnz, 1));
    std::vector<std::vector<int32_t>> sets;
    int64_t nt = 0;
    int maxtn = 0, maxsub = 0;
    std::vector<int64_t> cst;  // first cell of each tile
    std::vector<int32_t> fst;  // F-bar: first nodal cell of each tile
    while (true) {
        cst.clear();
        fst.clear();
        if (D.fbar) {
            // whole nodal cells, as many as fit tc subcells (a larger cell gets a tile alone)
            const std::vector<int64_t> &fs = D.fcell_sub_h;
            for (int64_t r = 0; r < D.n_fcells;) {
                cst.push_back(fs[r]);
                fst.push_back((int32_t)r);
                int64_t r1 = r + 1;
                while (r1 < D.n_fcells && fs[r1 + 1] - fs[r] <= tc) ++r1;
                r = r1;
            }
            cst.push_back(nc);
            fst.push_back((int32_t)D.n_fcells);
        } else {
            for (int64_t k = 0; k < nc; k += tc) cst.push_back(k);
            cst.push_back(nc);
        }
        nt = (int64_t)cst.size() - 1;
        maxsub = 0;
        for (int64_t t = 0; t < nt; ++t) maxsub = std::max<int64_t>(maxsub, cst[t + 1] - cst[t]);
        sets.assign(nt, {});
        std::vector<int> tile_max(std::max<int64_t>(nt, 1), 0);
        std::atomic<int64_t> next{0};
        auto work = [&] {
            std::vector<int32_t> loc(nn, 0);
            for (int64_t t; (t = next++) < nt;) {
                const int64_t e0 = hs[cst[t]], e1 = hs[cst[t + 1]];
                std::vector<int32_t> &u = sets[t];
                u.assign(hn.begin() + e0, hn.begin() + e1);
                std::sort(u.begin(), u.end());
                u.erase(std::unique(u.begin(), u.end()), u.end());
                tile_max[t] = (int)u.size();
                if (u.size() > 65535) continue;  // too large: the caller halves the tile
                for (size_t k = 0; k < u.size(); ++k) loc[u[k]] = (int32_t)k;
                for (int64_t e = e0; e < e1; ++e) lidx[e] = (uint16_t)loc[hn[e]];
            }
        };
        run_workers(nthreads, work);
        maxtn = *std::max_element(tile_max.begin(), tile_max.end());
        if (tile_lds(maxtn, maxsub, D.fbar) <= kTileLdsMax || tc == 1) break;
        tc = std::max(1, tc / 2);
    }
    APHIP_REQUIRE(tile_lds(maxtn, maxsub, D.fbar) <= kTileLdsMax,
                  "a smoothing cell names too many nodes (or a nodal cell holds too many subcells) for the tile kernels");
    std::vector<int32_t> tstart(nt + 1, 0);
    for (int64_t t = 0; t < nt; ++t) {
        APHIP_REQUIRE((int64_t)tstart[t] + (int64_t)sets[t].size() < (int64_t)INT32_MAX, "too many tile nodes");
        tstart[t + 1] = tstart[t] + (int32_t)sets[t].size();
    }
    const int64_t total = tstart[nt];
    std::vector<int32_t> tnode(std::max<int64_t>(total, 1));
    std::vector<int64_t> sstart(nn + 1, 0);
    for (int64_t t = 0; t < nt; ++t) {
        std::copy(sets[t].begin(), sets[t].end(), tnode.begin() + tstart[t]);
        for (int32_t g : sets[t]) sstart[g + 1]++;
    }
    for (int64_t i = 0; i < nn; ++i) sstart[i + 1] += sstart[i];
    std::vector<int32_t> nslot(std::max<int64_t>(total, 1));
    {
        std::vector<int64_t> fill(sstart.begin(), sstart.end() - 1);
        for (int64_t k = 0; k < total; ++k) nslot[fill[tnode[k]]++] = (int32_t)k;  // tiles in ascending order
    }
    sets.clear();
    D.tile_cells = tc;
    D.tile_maxtn = maxtn;
    D.tile_maxsub = maxsub;
    D.ntiles = nt;
    D.tile_total = total;
    D.t_cstart.upload(cst.data(), cst.size(), c.stream);
    if (D.fbar) D.t_fstart.upload(fst.data(), fst.size(), c.stream);
    D.lidx.upload(lidx.data(), lidx.size(), c.stream);
    D.t_nstart.upload(tstart.data(), tstart.size(), c.stream);
    D.t_node.upload(tnode.data(), tnode.size(), c.stream);
    D.nslot_start.upload(sstart.data(), sstart.size(), c.stream);
    D.nslot.upload(nslot.data(), nslot.size(), c.stream);
    D.slots.alloc(3 * std::max<int64_t>(total, 1));
    D.slots.zero(c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
}

// Reverse neighbor lists (after the cell CSR) and, for nodal cells, the cell tiles.
void rk_cells_order(Ctx &c) {
    CellData &D = c.cells;
    const int64_t nn = c.nn;
    // reverse neighbor lists: for node J the points i that list it, ascending i,
    // with phi_iJ (the mass scatter and the two-pass force scatter)
    {
        std::vector<int32_t> hn(nn), hb(nn * kMaxNbr);
        std::vector<double> hp(nn * kMaxNbr);
        D.num_nbr.download(hn.data(), nn, c.stream);
        D.nbr.download(hb.data(), hb.size(), c.stream);
        D.phi.download(hp.data(), hp.size(), c.stream);
        APHIP_HIP(hipStreamSynchronize(c.stream));
        std::vector<int64_t> rstart(nn + 1, 0);
        for (int64_t i = 0; i < nn; ++i)
            for (int l = 0; l < hn[i]; ++l) rstart[hb[i * kMaxNbr + l] + 1]++;
        for (int64_t j = 0; j < nn; ++j) rstart[j + 1] += rstart[j];
        const int64_t nrev = std::max<int64_t>(rstart[nn], 1);
        std::vector<int32_t> rsrc(nrev, 0);
        std::vector<double> rphi(nrev, 0.0);
        std::vector<int64_t> fill(rstart.begin(), rstart.end() - 1);
        for (int64_t i = 0; i < nn; ++i)
            for (int l = 0; l < hn[i]; ++l) {
                const int64_t t = fill[hb[i * kMaxNbr + l]]++;
                rsrc[t] = (int32_t)i;
                rphi[t] = hp[i * kMaxNbr + l];
            }
        D.rstart.upload(rstart.data(), rstart.size(), c.stream);
        D.rsrc.upload(rsrc.data(), rsrc.size(), c.stream);
        D.rphi.upload(rphi.data(), rphi.size(), c.stream);
        APHIP_HIP(hipStreamSynchronize(c.stream));
    }

    if (D.nodal) rk_tile_plan(c);  // nodal cells run on cell tiles, element cells on the element tile plan
    APHIP_HIP(hipStreamSynchronize(c.stream));
    D.ready = true;
}

template <int KIND>
static void launch_rk_tile(const RkTileArgs &T, int lpc, dim3 g, size_t lds, hipStream_t s) {
    if (lpc == 4) hipLaunchKernelGGL((k_rk_tile<KIND, 4, 1>), g, dim3(64), lds, s, T);
    else if (lpc == 8) hipLaunchKernelGGL((k_rk_tile<KIND, 8, 12>), g, dim3(64), lds, s, T);
    else hipLaunchKernelGGL((k_rk_tile<KIND, 16, 8>), g, dim3(64), lds, s, T);
}

static RkTileArgs rk_tile_args(Ctx &c, bool keep, bool raw) {
    CellData &D = c.cells;
    const int64_t nbt = ((D.ntiles + kNumXcd - 1) / kNumXcd) * kNumXcd;
    return RkTileArgs{D.ncells, D.ntiles, nbt, D.tile_maxtn, D.start.p, D.lidx.p, D.dphi.p,
                      D.volume.p, c.u.p, D.t_nstart.p, D.t_node.p, D.t_cstart.p, D.slots.p, c.Hnp1().p, c.Pnp1().p,
                      c.state[1 - c.state_np1].p, c.state[c.state_np1].p, c.mat.params(),
                      c.has_fields ? c.elem_lambda.p : nullptr, c.has_fields ? c.elem_mu.p : nullptr,
                      c.mat.rate_form() ? c.Hn().p : nullptr, c.mat.rate_form() ? c.Pn().p : nullptr, c.rate_dt,
                      keep || c.mat.rate_form(), raw, c.n_dof, c.v.p, c.a.p, c.has_fixed ? c.fixed.p : nullptr};
}

template <int KIND>
static void launch_fbar_tile(const FbarTileArgs &B, int lpc, dim3 g, int threads, size_t lds, hipStream_t s) {
    if (lpc == 4) hipLaunchKernelGGL((k_fbar_tile<KIND, 4>), g, dim3(threads), lds, s, B);
    else if (lpc == 8) hipLaunchKernelGGL((k_fbar_tile<KIND, 8>), g, dim3(threads), lds, s, B);
    else hipLaunchKernelGGL((k_fbar_tile<KIND, 16>), g, dim3(threads), lds, s, B);
}

static void rk_fbar_tiles(Ctx &c, bool keep, bool raw) {
    CellData &D = c.cells;
    if (D.ntiles == 0) return;
    const FbarTileArgs B{rk_tile_args(c, keep, raw), D.t_fstart.p, D.fcell_sub.p, D.fcell_volume.p, D.sub_fcell.p,
                         std::max(D.tile_maxsub, 1)};
    const dim3 g((unsigned)B.T.nblocks);
    const int lpc = D.tile_lpc;
    // Meshes of few tiles: as many waves as give every subcell of the largest tile a lane group, up
    // to four and to what the LDS budget leaves for their rows (10 steps of 719 tiles in turn, 1 /
    // 3 waves: 91 / 83 us; 20 steps of 2183 tiles: 303 / 381 us)
    size_t lds = (size_t)tile_lds(D.tile_maxtn, D.tile_maxsub, true);
    const size_t row = 24 * (size_t)std::max(D.tile_maxtn, 1);
    int waves = 1;
    while (D.ntiles <= 1024 && waves < 4 && waves * 64 / lpc < D.tile_maxsub && lds + row <= (size_t)kTileLdsMax) {
        ++waves;
        lds += row;
    }
    switch (c.mat.kind) {
        case APHIP_LINEAR_ELASTIC: launch_fbar_tile<APHIP_LINEAR_ELASTIC>(B, lpc, g, 64 * waves, lds, c.stream); break;
        case APHIP_NEO_HOOKEAN: launch_fbar_tile<APHIP_NEO_HOOKEAN>(B, lpc, g, 64 * waves, lds, c.stream); break;
        case APHIP_J2: launch_fbar_tile<APHIP_J2>(B, lpc, g, 64 * waves, lds, c.stream); break;
        case APHIP_SVK: launch_fbar_tile<APHIP_SVK>(B, lpc, g, 64 * waves, lds, c.stream); break;
        default: throw Error(APHIP_ERR_UNSUPPORTED, "F-bar takes the linear elastic, neo-Hookean, J2 and SVK materials");
    }
    APHIP_HIP(hipGetLastError());
}

static void rk_tile_force(Ctx &c, bool keep, bool raw) {
    CellData &D = c.cells;
    if (D.ntiles == 0) return;
    const RkTileArgs T = rk_tile_args(c, keep, raw);
    const dim3 g((unsigned)T.nblocks);
    const size_t lds = 48 * (size_t)std::max(D.tile_maxtn, 1);
    const int lpc = D.tile_lpc;
    switch (c.mat.kind) {
        case APHIP_LINEAR_ELASTIC: launch_rk_tile<APHIP_LINEAR_ELASTIC>(T, lpc, g, lds, c.stream); break;
        case APHIP_NEO_HOOKEAN: launch_rk_tile<APHIP_NEO_HOOKEAN>(T, lpc, g, lds, c.stream); break;
        case APHIP_J2: launch_rk_tile<APHIP_J2>(T, lpc, g, lds, c.stream); break;
        case APHIP_SVK: launch_rk_tile<APHIP_SVK>(T, lpc, g, lds, c.stream); break;
        case APHIP_NEO_HOOKEAN_DAMAGE: launch_rk_tile<APHIP_NEO_HOOKEAN_DAMAGE>(T, lpc, g, lds, c.stream); break;
        case APHIP_POWER_LAW_CREEP: launch_rk_tile<APHIP_POWER_LAW_CREEP>(T, lpc, g, lds, c.stream); break;
        case APHIP_DRUCKER_PRAGER: launch_rk_tile<APHIP_DRUCKER_PRAGER>(T, lpc, g, lds, c.stream); break;
        default: throw Error(APHIP_ERR_INVALID, "material not set");
    }
    APHIP_HIP(hipGetLastError());
}

// Small meshes: fewer launches a step.  The passes take the first step's predictor themselves,
// the scatter sums the shared nodes' slots itself (once for each list that holds them), and Tet4
// tiles gather u = Phi d as they stage their nodes (a shared node's row in each of its tiles): two
// launches a step, whose added work stays below the launches saved up to about 12k nodes.  10
// one-pass steps at kernel scale 1.3 with three streams in turn, four launches / two: 343 nodes
// 161 / 105 us, 9261 162 / 118, 19683 164 / 201.  Hex8 cells keep the gather pass (their tile
// workgroups of two waves take longer over it than a launch costs: 9261 nodes 113 / 166 us).
bool rk_fused(const Ctx &c) {
    const CellData &D = c.cells;
    return D.ready && !D.nodal && !D.fbar && D.ncells > 0 && !c.node_dt.p && c.n_dof == c.nn &&
           !c.tiles.orphans && c.nn <= kFusedNodes;
}

bool rk_takes_predictor(const Ctx &c) { return rk_fused(c) || (c.cells.ready && c.cells.nodal && !c.node_dt.p); }

void rk_cell_force(Ctx &c, bool keep, bool raw, bool keep_local) {
    CellData &D = c.cells;
    if (D.ncells == 0) return;  // no cells: f_local stays zero
    if (D.fbar) {
        rk_fbar_tiles(c, keep, raw);
        return;
    }
    if (D.nodal) {
        rk_tile_force(c, keep, raw);
        return;
    }
    // physical displacement = Phi d (ExplicitSolver::ComputeForce, Explicit.cpp:148-152), then
    // the element tiles
    const bool fused = rk_fused(c);
    if (fused && c.npe == 4) {
        const PhiRows phi{D.num_nbr.p, D.nbr.p, D.phi.p, D.two_pass, raw, keep_local ? D.u_phys.p : nullptr,
                          c.tiles.bstart.p};
        TileRun run;
        run.phi = &phi;
        run.park = true;
        run.f_out = D.f_local.p;
        run.keep = keep;
        const bool prof = c.prof.enabled;  // timed as this force pass, not as tile launches
        c.prof.enabled = false;
        tile_run(c, c.rate_dt, 0, run);
        c.prof.enabled = prof;
        return;
    }
    const int64_t nbg = padded_groups(c.nn, kGsLanes);
    const RkGatherArgs G{c.nn, nbg, D.num_nbr.p, D.nbr.p, D.phi.p, c.u.p, D.u_phys.p, D.two_pass,
                         c.v.p, c.a.p, c.has_fixed ? c.fixed.p : nullptr, c.rate_dt};
    if (raw) hipLaunchKernelGGL((k_rk_gather<kGsLanes, true>), dim3((unsigned)nbg), dim3(256), 0, c.stream, G);
    else hipLaunchKernelGGL((k_rk_gather<kGsLanes, false>), dim3((unsigned)nbg), dim3(256), 0, c.stream, G);
    APHIP_HIP(hipGetLastError());
    const bool prof = c.prof.enabled;  // timed as this force pass, not as tile launches
    c.prof.enabled = false;
    TileRun run;
    run.u_in = D.u_phys.p;
    run.f_out = D.f_local.p;
    run.keep = keep;
    run.park = fused;
    tile_run(c, 0.0, 0, run);
    c.prof.enabled = prof;
}

void rk_node_update(Ctx &c, double dt, int mode, bool more, bool raw, bool keep) {
    CellData &D = c.cells;
    // nodes with degrees of freedom only (nodal cells put them first; the others keep
    // their values, as the reference's integrator runs over the active part)
    const int lanes = D.nodal ? kSlotLanes : kCellLanes;
    const int64_t nb = padded_groups(c.n_dof, lanes);
    const dim3 g((unsigned)nb);
    const RkNodeArgs A{c.n_dof, nb, c.mass.p, c.has_fixed ? c.fixed.p : nullptr, c.f.p, c.a.p, c.v.p, c.u.p, dt, more,
                       raw};
    if (D.nodal) {
        const RkSlotNodeArgs N{A, D.nslot_start.p, D.nslot.p, D.slots.p};
        if (mode == 0) hipLaunchKernelGGL((k_rk_slot_nodes<0, kSlotLanes>), g, dim3(256), 0, c.stream, N);
        else if (mode == 1) hipLaunchKernelGGL((k_rk_slot_nodes<1, kSlotLanes>), g, dim3(256), 0, c.stream, N);
        else hipLaunchKernelGGL((k_rk_slot_nodes<2, kSlotLanes>), g, dim3(256), 0, c.stream, N);
    } else {  // f = Phi^T f_local with the node update (ScatterValues, Explicit.cpp:181-186)
        const RkScatterArgs S{A, D.num_nbr.p, D.rstart.p, D.rsrc.p, D.rphi.p, D.f_local.p, D.two_pass,
                              c.tiles.bstart.p, c.tiles.bpart.p, c.tiles.n_interior, mode != 2 || keep ? D.f_local.p : nullptr};
        constexpr int NB = (kMaxNbr + kCellLanes - 1) / kCellLanes;
        if (rk_fused(c)) {
            if (mode == 0) hipLaunchKernelGGL((k_rk_scatter<0, kCellLanes, NB, true>), g, dim3(256), 0, c.stream, S);
            else if (mode == 1) hipLaunchKernelGGL((k_rk_scatter<1, kCellLanes, NB, true>), g, dim3(256), 0, c.stream, S);
            else hipLaunchKernelGGL((k_rk_scatter<2, kCellLanes, NB, true>), g, dim3(256), 0, c.stream, S);
        } else if (mode == 0) hipLaunchKernelGGL((k_rk_scatter<0, kCellLanes, NB>), g, dim3(256), 0, c.stream, S);
        else if (mode == 1) hipLaunchKernelGGL((k_rk_scatter<1, kCellLanes, NB>), g, dim3(256), 0, c.stream, S);
        else hipLaunchKernelGGL((k_rk_scatter<2, kCellLanes, NB>), g, dim3(256), 0, c.stream, S);
    }
    APHIP_HIP(hipGetLastError());
}

void rk_mass(Ctx &c, double *total) {
    CellData &D = c.cells;
    const int64_t nn = c.nn;
    DevBuf<double> mfe;
    mfe.alloc(nn);
    hipLaunchKernelGGL(c.etype == APHIP_HEX8 ? k_rk_mfe<8> : k_rk_mfe<4>, grid1(nn, 256), dim3(256), 0, c.stream, nn, c.node_start.p, c.node_inc.p,
                       D.nodal ? D.evol.p : D.volume.p, c.mat.density, mfe.p);
    APHIP_HIP(hipGetLastError());
    c.mass.alloc(nn);
    hipLaunchKernelGGL(k_rk_mass, grid1(nn, 256), dim3(256), 0, c.stream, nn, D.num_nbr.p, D.rstart.p, D.rsrc.p,
                       D.rphi.p, mfe.p, c.mass.p);
    APHIP_HIP(hipGetLastError());
    std::vector<double> hm(nn);
    c.mass.download(hm.data(), nn, c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    double tot = 0.0;
    for (double x : hm) tot += x;
    if (total) *total = tot;
}

}  // namespace aphip
