// Fused element-tile step for gfx950: one workgroup owns a Morton-contiguous tile
// of elements (one element per thread) and, in one launch,
//   A. stages the tile's nodes in LDS (reference coordinates and the predicted
//      displacement u + dt (v + dt/2 a) of the central-difference step) together
//      with the tile's local CSR, masses and boundary flags,
//   B. evaluates every element of the tile (B, H, P, stress update, -B P^T w) and
//      writes its force partials to LDS,
//   C. sums each tile node's partials through the local CSR in ascending element
//      order (deterministic; no atomics) and finishes the nodes that only this
//      tile touches (a = f/m, BCs, v = v1/2 + dt/2 a, writes u, v, a, f).
// Nodes shared with other tiles leave their tile sum in a slot of a per-node
// contiguous slot list; a second, much smaller launch adds each shared node's
// slots in ascending tile order and finishes it.  This replaces the reference's
// per-element atomic scatter (include/ComputeInternalForceGaussian.h:127-130,
// include/Field.h:235-246) and its separate node loops (src/Solvers/Explicit.cpp:405-452).
//
// Node numbering (set by the plan): the interior nodes of tile t are the
// contiguous range [int_base[t], int_base[t] + ninterior[t]); all shared nodes
// follow as one contiguous range [n_interior, n_nodes).  Interior nodes are
// therefore read and written without indirection, and the shared-node pass is
// coalesced.
#include <algorithm>
#include <vector>

#include "element.hpp"
#include "internal.hpp"

namespace aphip {

namespace {

constexpr int kNumXcd = 8;

__device__ __forceinline__ int64_t xcd_tile(int64_t nblocks_padded) {
    const int64_t b = blockIdx.x;
    const int64_t per = nblocks_padded / kNumXcd;
    return (b % kNumXcd) * per + b / kNumXcd;
}

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

struct TileArgs {
    const double *X;
    double *u, *v, *a, *f;
    const double *mass;
    const uint8_t *fixed;
    const int32_t *tn_start;
    const int32_t *tile_e0;
    const int32_t *tn_ninterior;
    const int32_t *int_base;
    const int32_t *tn_node;
    const uint32_t *tn_csr;
    const int32_t *tn_bdst;
    const uint16_t *lcsr;
    const uint16_t *lconn;
    const int32_t *tnp_node;  // fixed-stride copies of tn_node / tn_csr / tn_bdst / lconn
    const uint32_t *tnp_csr;
    const int32_t *tnp_bdst;
    const uint16_t *lconn_p;
    int tpad;
    // k_hex_tile's forms (TilePlan::hx_*): corners as 3 x local node; per round and node row the
    // first eight entries as force-row offsets (padded with the zero row) and the further
    // batches (first << 16) | count in hx_more, from hx_base[tile * rounds + round] on
    const uint16_t *hx_conn;
    const uint4 *hx_first, *hx_more;
    const uint32_t *hx_csr;
    const int32_t *hx_base;
    double *hx_part;  // several rounds: [ntiles * tpad * 3] the rows' sums so far
    int hx_rounds;
    double *bpart;
    double *H, *P;
    const double *Hn, *Pn;  // rate-form materials: H and P of the previous step
    double rate_dt;         // and the increment of this evaluation
    const double *state_n;
    double *state_np1;
    MatParams mat;
    const double *elem_lambda, *elem_mu;
    const double *node_dt;  // per-node increment (ensembles) or null
    const double *zero;     // 8 zero doubles: stands in for an absent optional array
    const int32_t *meta;    // [ntiles * 8] packed per-tile scalars (TileMeta)
    double gauss_a;
    int64_t ne, ntiles, nblocks;
    int64_t nn, nslot;      // nodes; shared-node slots (bpart holds 3 doubles each)
    int te, maxtn;
    int max_nint;  // most interior nodes in one tile (Hex8: LDS rows of the corrector data)
    double dt;
    // mode 2, steps of one call: pred: u and v hold this step's predicted displacement and
    // v1/2 (else predicted here from u, v, a); more: leave the next step's there, and no a
    int pred, more;
    int64_t first_shared;
    // 0: an inner step of one call, whose H, P and f the next step overwrites unread
    int keep;
    int keep_h;  // H alone (the updated formulation reads it in the next step)
    // updated / semi-Lagrangian steps (X: the configuration integrated over): the increments
    // written, the next coordinates (updated), 1 when the increments accumulate (semi)
    double *dinc, *xnp1;
    int semi;
    int cell_marker;  // smoothed cells turn a new failure's marker into the maximum damage
    PhiRows phi;      // GATHER
};

// LDS carve-up (bytes), sized on the host (tile_lds_bytes) from the tile's rows.  X and U (the
// predicted displacement) are kept for every tile node; v_half, m, dt and the fixed mask for
// max_nint rows (Hex8: the interior nodes, the only ones the kernel finishes; Tet4: every
// tile node); F holds nf doubles: the element forces of one round or the Hex8 element rows.
// LEAN: a Hex8 tile in rounds, which reads m, dt, the mask and the entries from global memory when
// it needs them (the freed LDS saves rounds: 76,800 Hex8 in bars of three, tiles of 256, 58 to
// 61 us a step in four rounds, 47 to 51 in two).
struct TileLds {
    double *X, *U, *V, *F, *M, *DT;
    uint32_t *csr;
    int32_t *bdst;
    uint16_t *ent;
    uint8_t *fx;
};

// Rows between the slot blocks of the element-force rows: te_round + pad with
// stride = 4 (mod 32), so that the 24-byte rows of one element's slots start 24 banks
// apart (mod 64): the 4 or 8 slots of an element, which the nodes of that element
// read at the same time in the gather, never share a bank.
__host__ __device__ __forceinline__ int f_stride(int te_round) { return te_round + ((4 - te_round) & 31); }

__host__ __device__ __forceinline__ TileLds carve(char *base, int maxtn, int max_nint, int nent, size_t nf,
                                                  bool lean = false) {
    TileLds L;
    const int fin = lean ? 0 : max_nint;
    L.X = reinterpret_cast<double *>(base);
    L.U = L.X + 3 * maxtn;
    L.V = L.U + 3 * maxtn;
    L.M = L.V + 3 * max_nint;
    L.DT = L.M + fin;
    L.F = L.DT + fin;
    L.csr = reinterpret_cast<uint32_t *>(L.F + nf);
    L.bdst = reinterpret_cast<int32_t *>(L.csr + (lean ? 0 : maxtn));
    // (16-byte aligned: entries are read eight at a time)
    L.ent = reinterpret_cast<uint16_t *>((reinterpret_cast<uintptr_t>(L.bdst + maxtn) + 15) & ~(uintptr_t)15);
    L.fx = reinterpret_cast<uint8_t *>(L.ent + nent);
    return L;
}

// F doubles of a tile: Tet4 one round of slot-major force rows, smoothed Hex8 cells two rounds
// of half the tile (half the rows: twice the workgroups fit a CU), Gauss Hex8 kHexRow a row and
// a zero row
__host__ __device__ __forceinline__ size_t tile_f_doubles(int npe, int te, bool cell) {
    return npe == 4 ? 12 * (size_t)f_stride(te) : cell ? 24 * (size_t)f_stride(te / 2) : kHexRow * (size_t)te + 4;
}

// Entries of a Hex8 tile kept in LDS: eight a row, or none in rounds.
__host__ __device__ __forceinline__ int hex_entries(int maxtn, int rounds) { return rounds == 1 ? 8 * maxtn : 0; }

// nent: entries kept in LDS; lean: as carve's
__host__ inline size_t tile_lds_bytes(int maxtn, int max_nint, int te, int npe, int nent, bool cell, bool lean = false) {
    return sizeof(double) * (6 * (size_t)maxtn + (lean ? 3 : 5) * (size_t)max_nint + tile_f_doubles(npe, te, cell)) +
           (lean ? 4 : 8) * (size_t)maxtn + 2 * (size_t)nent + (lean ? 0 : (size_t)max_nint) + 16 + 16;
}

// Materials whose Hex8 kernel needs more than the 128 VGPRs of four waves per SIMD (it would
// spill 117 for creep, 78 for Drucker-Prager, 10 for damage).
template <int KIND, bool UL = false>
constexpr bool hex_wide() {
    return UL || rate_form<KIND>() || KIND == APHIP_NEO_HOOKEAN_DAMAGE;
}
// Workgroup of the Hex8 kernel: eight lanes per element, at most 512 lanes up to 128 elements
// (two passes: two workgroups fit a CU) and in rounds, else 1024 (wide materials 512).
template <int KIND, bool UL = false>
__host__ int hex_threads(int te, int rounds) {
    return std::min(te <= 128 || rounds > 1 || hex_wide<KIND, UL>() ? 512 : 1024, 8 * (te / rounds));
}

// Optional arrays are read without branches: an absent array is replaced by the
// zero buffer at index 0 (a uniform select), and the value is then selected.  A
// load under a branch ends a basic block, and at the join the compiler waits for
// every outstanding memory operation of the wave, stores included.
__device__ __forceinline__ unsigned load_fixed(const TileArgs &A, int64_t g) {
    const uint8_t *p = A.fixed ? A.fixed : reinterpret_cast<const uint8_t *>(A.zero);
    return p[A.fixed ? g : 0];
}

__device__ __forceinline__ double load_node_dt(const TileArgs &A, int64_t g) {
    const double *p = A.node_dt ? A.node_dt : A.zero;
    const double d = p[A.node_dt ? g : 0];
    return A.node_dt ? d : A.dt;
}

__device__ __forceinline__ void load_elem_lame(const TileArgs &A, int64_t e, MatParams &m) {
    const double *pl = A.elem_lambda ? A.elem_lambda : A.zero;
    const double *pm = A.elem_lambda ? A.elem_mu : A.zero;
    const int64_t i = A.elem_lambda ? e : 0;
    const double l = pl[i], mu = pm[i];
    m.lambda = A.elem_lambda ? l : m.lambda;
    m.mu = A.elem_lambda ? mu : m.mu;
}

// MODE 2 staging of a node: v1/2 and what the element gradients are taken of, the predicted
// displacement or (UL, u then being the semi-Lagrangian increments so far) the increment
// since the configuration integrated over.
template <bool UL>
__device__ __forceinline__ void stage_predict(const TileArgs &A, const double *u, const double *v, const double *a,
                                              unsigned fx, double dt, double *vh, double *u1) {
#pragma clang fp contract(off)
    cd_predict(u, v, a, fx, dt, vh, u1);
    if constexpr (UL) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double inc = dt * vh[d];
            u1[d] = A.semi ? u[d] + inc : inc;
        }
    }
}

// U rows of tile t's nodes: Phi u, eight lanes a node, each with its share of the row (the
// entries past the row weighted by zero), combined by a xor butterfly.
__device__ __forceinline__ void stage_phi(const TileArgs &A, const TileLds &L, int64_t t, int tn) {
    constexpr int LANES = 8, R = (kMaxNbr + LANES - 1) / LANES;
    const int l = threadIdx.x & (LANES - 1), step = blockDim.x / LANES;
    const int rounds = (tn + step - 1) / step;
    for (int r0 = 0; r0 < rounds; ++r0) {
        const int ln_raw = r0 * step + (int)threadIdx.x / LANES, ln = min(ln_raw, tn - 1);
        const int64_t i = A.tnp_node[t * (int64_t)A.tpad + ln];
        const int n = A.phi.num[i];
        const int64_t row = i * kMaxNbr;
        int32_t j[R];
        double w[R], x[R][3], s[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < R; ++r) {
            // (a row holds kMaxNbr places: loaded without waiting for its length)
            const int k = l + r * LANES, kk = min(k, kMaxNbr - 1);
            const int32_t jl = A.phi.nbr[row + kk];
            const double wl = A.phi.phi[row + kk];
            j[r] = k < n ? jl : (int32_t)i;
            w[r] = k < n ? wl : 0.0;
        }
        if (n == 0 && A.phi.copy_lonely && l == 0) w[0] = 1.0;
        if (A.phi.raw) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                double u[3], v[3], a[3], vh[3];
                ld3(A.u, j[r], u);
                ld3(A.v, j[r], v);
                ld3(A.a, j[r], a);
                cd_predict(u, v, a, load_fixed(A, j[r]), A.dt, vh, x[r]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) ld3(A.u, j[r], x[r]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int d = 0; d < 3; ++d) s[d] += x[r][d] * w[r];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = LANES / 2; m >= 1; m >>= 1) s[d] += __shfl_xor(s[d], m, LANES);
        if (l == 0 && ln_raw < tn) {
            st3(L.U, ln, s);
            if (A.phi.out) {
                const int32_t slot = A.tnp_bdst[t * (int64_t)A.tpad + ln];
                if (slot < 0 || slot == A.phi.bstart[i - A.first_shared]) st3(A.phi.out, i, s);
            }
        }
    }
}

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt at their maxima: not waited on).  At a
// point where no store is outstanding this costs nothing beyond the loads' latency.
__device__ __forceinline__ void wait_vmem_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// Updated / semi-Lagrangian node update (ExplicitTimeIntegrator.h:193-226): with the step's
// increment inc = dt v1/2, u += inc; updated: x_{n+1} = x_n + inc and the increment itself is
// kept; semi: the accumulated increment acc.
__device__ __forceinline__ void ul_store1(double *u, double *dinc, double *xnp1, int semi, int64_t k, double dt,
                                          double vh, double x, double acc) {
#pragma clang fp contract(off)
    const double inc = dt * vh;
    u[k] = u[k] + inc;
    dinc[k] = semi ? acc : inc;
    if (!semi) xnp1[k] = x + inc;
}

// Node ln's force f is complete: an interior node is finished and written (MODE 0: f;
// 1: f and a = f/m; 2: the corrector); a shared node parks f in its slot for the
// shared-node pass.
template <int MODE, bool UL = false, bool LEAN = false>
__device__ __forceinline__ void finish_node(const TileArgs &A, const TileLds &L, int ln, int nint, int64_t ibase,
                                            const double (&f)[3]) {
    if (ln < nint) {
        const int64_t g = ibase + ln;
        if (MODE != 2 || A.keep) st3(A.f, g, f);
        const double mm = MODE == 0 ? 1.0 : LEAN ? A.mass[g] : L.M[ln];
        if constexpr (MODE == 1) {
            const double acc[3] = {f[0] / mm, f[1] / mm, f[2] / mm};
            st3(A.a, g, acc);
        } else if constexpr (MODE == 2) {
            double vh[3], u1[3], a1[3], v1[3];
            const unsigned fx = LEAN ? load_fixed(A, g) : L.fx[ln];
            const double nd = LEAN ? load_node_dt(A, g) : L.DT[ln];
            ld3(L.V, ln, vh);
            ld3(L.U, ln, u1);
            cd_correct(f, mm, fx, nd, vh, a1, v1);
            if constexpr (UL) {
                double x[3];
                ld3(L.X, ln, x);
#pragma unroll
                for (int d = 0; d < 3; ++d) ul_store1(A.u, A.dinc, A.xnp1, A.semi, 3 * g + d, A.dt, vh[d], x[d], u1[d]);
            } else if (A.more) {
                double u2[3], v2[3];
                cd_predict(u1, v1, a1, fx, nd, v2, u2);
                st3(A.u, g, u2);
                st3(A.v, g, v2);
                return;
            } else {
                st3(A.u, g, u1);
            }
            st3(A.v, g, v1);
            st3(A.a, g, a1);
        }
    } else {
        st3(A.bpart, L.bdst[ln], f);
    }
}

// MODE 0: force only; 1: force + a = f/m (initial); 2: full central-difference step.
// One element per thread: Tet4 (NPE 4), or smoothed Hex8 cells (NPE 8, MODE 0); the 2x2x2 Gauss
// Hex8 has k_hex_tile.
// UL: updated / semi-Lagrangian step.  GATHER: the displacement staged is Phi u.
template <int NPE, int KIND, int MODE, bool UL = false, bool GATHER = false>
__global__ __launch_bounds__(NPE == 4 ? 1024 : 256, NPE == 8 ? 2 : 1) void k_tile(TileArgs A) {
    static_assert(!GATHER || (NPE == 4 && MODE == 0), "Tet4 in force mode");
    static_assert(NPE == 4 || MODE == 0, "smoothed Hex8 cells are evaluated in force mode");
    extern __shared__ __align__(16) char lds_raw[];
    const int64_t t = xcd_tile(A.nblocks);
    if (t >= A.ntiles) return;
    // Smoothed Hex8 cells pass their forces through LDS in two rounds (24 doubles per element
    // otherwise keep a 128-element tile at one wave per SIMD); Tet4 tiles in one.
    constexpr int ROUNDS = NPE == 8 ? 2 : 1;
    const TileLds L = carve(lds_raw, A.maxtn, NPE == 4 ? A.maxtn : A.max_nint, A.te * NPE,
                            tile_f_doubles(NPE, A.te, true));
    const int tid = threadIdx.x;
    const int le = tid;
    int lc[NPE];
    // (le < te always; the fixed-stride copy needs no per-tile scalar)
    const int64_t ep = t * (int64_t)A.te + le;
    if constexpr (NPE == 4) {
        const ushort4 c = reinterpret_cast<const ushort4 *>(A.lconn_p)[ep];
        lc[0] = c.x; lc[1] = c.y; lc[2] = c.z; lc[3] = c.w;
    } else {
        const ushort4 c0 = reinterpret_cast<const ushort4 *>(A.lconn_p)[2 * ep];
        const ushort4 c1 = reinterpret_cast<const ushort4 *>(A.lconn_p)[2 * ep + 1];
        lc[0] = c0.x; lc[1] = c0.y; lc[2] = c0.z; lc[3] = c0.w;
        lc[4] = c1.x; lc[5] = c1.y; lc[6] = c1.z; lc[7] = c1.w;
    }

    // A: tile CSR entries and node data into LDS.  Every global load of the stage is
    // issued before the first LDS write: the CSR words and the tile-node indices
    // together, then the node data of the first NPT node rows of each thread.  (A load
    // followed by its LDS write in a loop waits for that load, and vmcnt counts in
    // order, so each iteration would add a full memory latency.)
    constexpr int EW = NPE == 4 ? 2 : 4;  // CSR words per thread: nent / 2 <= EW x blockDim
    constexpr int NPT = NPE == 4 ? 1 : 2; // node rows per thread loaded together
    const int nw = A.te * NPE / 2;  // words of a full tile; a partial tile reads zeros past its end
    const uint32_t *ent_src = reinterpret_cast<const uint32_t *>(A.lcsr) + t * (int64_t)nw;
    uint32_t ew[EW];
#pragma unroll
    for (int r = 0; r < EW; ++r) ew[r] = ent_src[min(tid + r * (int)blockDim.x, nw - 1)];
    int64_t gq[NPT];
    uint32_t csrq[NPT];
    int32_t bdq[NPT];
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
        // all loads unconditional (tn_node also lists the interior nodes, as ibase + ln)
        const int64_t row = t * (int64_t)A.tpad + min(tid + q * (int)blockDim.x, A.tpad - 1);
        gq[q] = A.tnp_node[row];
        csrq[q] = A.tnp_csr[row];
        bdq[q] = A.tnp_bdst[row];
    }
    double xq[NPT][3], uq[NPT][3], vq[NPT][3], aq[NPT][3], mq[NPT], dq[NPT];
    unsigned fq[NPT];
    bool pq[NPT];  // shared row of a predicted state: X and u only
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
        const int64_t g = gq[q];
        pq[q] = MODE == 2 && !UL && A.pred && bdq[q] >= 0;
        ld3(A.X, g, xq[q]);
        ld3(UL ? A.dinc : A.u, g, uq[q]);
        mq[q] = 1.0;
        dq[q] = A.dt;
        fq[q] = 0u;
#pragma unroll
        for (int d = 0; d < 3; ++d) vq[q][d] = aq[q][d] = 0.0;
        if (!pq[q]) {
            fq[q] = load_fixed(A, g);
            if constexpr (MODE >= 1) mq[q] = A.mass[g];
            if constexpr (MODE == 2) {
                ld3(A.v, g, vq[q]);
                if (UL || !A.pred) ld3(A.a, g, aq[q]);
                dq[q] = load_node_dt(A, g);
            }
        }
    }
    // per-tile scalars, read after the staging loads are out (their addresses need none)
    const int tb = A.tn_start[t];
    const int tn = A.tn_start[t + 1] - tb;
    const int nint = A.tn_ninterior[t];
    const int64_t ibase = A.int_base[t];
    const int64_t te0 = A.tile_e0[t];
    const int nel = A.tile_e0[t + 1] - (int)te0;
    const int64_t e = te0 + le;
    const bool has_elem = le < nel;
    const int64_t ec = te0 + min(le, nel - 1);  // clamped: the loads below need no branch
    MatParams m = A.mat;
    double sn = 0.0;
    load_elem_lame(A, ec, m);
    double sn2 = 0.0;
    if constexpr (NPE == 4) {
        sn = load_state<KIND>(A.state_n, ec);
        sn2 = load_state2<KIND>(A.state_n, ec);
    }
    RateIn rin;
    load_rate<KIND, UL>(rin, A.Hn, A.Pn, A.ne, ec, A.rate_dt);

    {
        uint32_t *dst = reinterpret_cast<uint32_t *>(L.ent);
#pragma unroll
        for (int r = 0; r < EW; ++r) {
            const int i = tid + r * (int)blockDim.x;
            if (i < nw) dst[i] = ew[r];
        }
    }
    // Hex8 keeps the corrector data of interior nodes only (the only ones it finishes);
    // Tet4 writes it for every node (measured faster with its 512-element tiles).
    // (the corrector data written for a shared row are never read)
    auto stage = [&](int ln, uint32_t csr, int32_t bdst, const double *x, const double *u, const double *v,
                     const double *a, unsigned fx, double mm, double nd) {
        L.csr[ln] = csr;
        L.bdst[ln] = bdst;
        st3(L.X, ln, x);
        const bool interior = NPE == 4 || ln < nint;
        if (interior) {
            L.fx[ln] = (uint8_t)fx;
            L.M[ln] = mm;
            L.DT[ln] = nd;
        }
        if constexpr (MODE == 2) {
            double vh[3] = {v[0], v[1], v[2]}, u1[3] = {u[0], u[1], u[2]};
            if (UL || !A.pred) stage_predict<UL>(A, u, v, a, fx, nd, vh, u1);
            st3(L.U, ln, u1);
            if (interior) st3(L.V, ln, vh);
        } else if constexpr (!GATHER) {
            st3(L.U, ln, u);
        }
    };
#pragma unroll
    for (int q = 0; q < NPT; ++q) {
        const int ln = tid + q * (int)blockDim.x;
        if (ln < tn) stage(ln, csrq[q], bdq[q], xq[q], uq[q], vq[q], aq[q], fq[q], mq[q], dq[q]);
    }
    // rows past NPT x blockDim (tiles with unusually many nodes)
    for (int ln = tid + NPT * (int)blockDim.x; ln < tn; ln += blockDim.x) {
        const int64_t g = A.tn_node[tb + ln];
        double x[3], u[3], v[3], a[3];
        ld3(A.X, g, x);
        ld3(UL ? A.dinc : A.u, g, u);
        const unsigned fx = load_fixed(A, g);
        double mm = 1.0, nd = A.dt;
        if constexpr (MODE >= 1) mm = A.mass[g];
        if constexpr (MODE == 2) {
            ld3(A.v, g, v);
            ld3(A.a, g, a);
            nd = load_node_dt(A, g);
        }
        stage(ln, A.tn_csr[tb + ln], A.tn_bdst[tb + ln], x, u, v, a, fx, mm, nd);
    }
    if constexpr (GATHER) stage_phi(A, L, t, tn);
    // Every load of the wave completes here, on every path (a wave whose lanes all
    // skip the staging loop still has its element prefetch in flight).  Otherwise the
    // join after the element phase merges a path with pending loads into the path
    // with the H / P stores, and the first register reuse in the gather waits for
    // vmcnt(0): for every store of the wave.
    wait_vmem_loads();
    __syncthreads();

    // B: one element per thread.  The element's nodal forces stay in registers until their
    // round's LDS pass.
    double fe[NPE][3];
    // Tet4: the element phase stores H and keeps P for the start of the gather phase.
    // The 144 B per element of H and P, all issued during the element phase, leave a CU
    // faster than the memory takes them while many CUs are in that phase; split between
    // the two phases they overlap the gather (tile kernel 274 -> 250 us on the 6M-tet
    // block; H and P both after the barrier: 277 us; P after the gather: 256 us).  Hex8
    // tiles, whose element phase is arithmetic-bound, measured the same either way.
    double pdef[NPE == 4 ? 9 : 1];
    const int te_round = ROUNDS == 1 ? A.te : A.te / ROUNDS;
    const int my_round = ROUNDS == 1 ? 0 : le / te_round;
    // LDS row of entry (element j of the round, slot k): slot-major with padded slot blocks, so
    // a wave's writes of one slot are consecutive 24-byte rows (no bank conflicts;
    // element-major rows 96 bytes apart hit 16 of the 64 banks) and the slots of one element
    // sit in distinct banks for the gather.
    const int fs = f_stride(te_round);
    auto frow = [fs](int j, int k) { return k * fs + j; };
    if (has_elem) {
        double X[NPE][3], U[NPE][3];
#pragma unroll
        for (int k = 0; k < NPE; ++k) {
            ld3(L.X, lc[k], X[k]);
            ld3(L.U, lc[k], U[k]);
        }
        double H[9], P[9];
        if constexpr (NPE == 4) {
            double snp1 = 0.0, aux = 0.0;
            tet4_element<KIND, UL>(X, U, m, sn, snp1, aux, H, P, fe, &rin, sn2);
            if (A.cell_marker) snp1 = cell_damage_marker<KIND>(snp1, m);
            store_state<KIND>(A.state_np1, e, snp1, aux);
        } else {
            const int64_t so = state_width<KIND>() * e;
            hex8_cell<KIND>(X, U, m, state_width<KIND>() ? A.state_n + so : nullptr,
                            state_width<KIND>() ? A.state_np1 + so : nullptr, H, P, fe, &rin);
        }
        if constexpr (NPE == 4) {
#pragma unroll
            for (int i = 0; i < 9; ++i) pdef[i] = P[i];
        }
        if (A.keep_h) {
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                store_once(A.H + i * A.ne + e, H[i]);
                if constexpr (NPE != 4) store_once(A.P + i * A.ne + e, P[i]);
            }
        }
        if (my_round == 0) {
#pragma unroll
            for (int k = 0; k < NPE; ++k) st3(L.F, frow(le, k), fe[k]);
        }
    }
    __syncthreads();
    if constexpr (NPE == 4) {
        if (has_elem && A.keep) {
#pragma unroll
            for (int i = 0; i < 9; ++i) store_once(A.P + i * A.ne + e, pdef[i]);
        }
    }

    // C: deterministic per-node gather from LDS (each node's entries in ascending order:
    // round r adds the entries of elements [r, r + 1) x te / ROUNDS, a contiguous run of
    // the node's sorted list, so the sum is the same sequence for every round count);
    // then finish interior nodes and park shared-node sums.
    if constexpr (ROUNDS == 1) {
        for (int ln = tid; ln < tn; ln += blockDim.x) {
            const uint32_t pk = L.csr[ln];
            const int st = (int)(pk >> 16), cnt = (int)(pk & 0xffffu);
            double f[3] = {0.0, 0.0, 0.0};
            for (int j = 0; j < cnt; ++j) {
                const int s = L.ent[st + j];
                const int rw = 3 * frow(s / NPE, s % NPE);
                f[0] += L.F[rw];
                f[1] += L.F[rw + 1];
                f[2] += L.F[rw + 2];
            }
            finish_node<MODE, UL>(A, L, ln, nint, ibase, f);
        }
        return;
    }
    // Several rounds: a thread owns the tile nodes tid + q * blockDim (maxtn <= NPE x te
    // <= NPE x blockDim) and keeps their partial sums in registers between rounds.
    double acc[NPE][3];
    int jpos[NPE];
#pragma unroll
    for (int q = 0; q < NPE; ++q) {
        acc[q][0] = acc[q][1] = acc[q][2] = 0.0;
        jpos[q] = 0;
    }
    for (int r = 0; r < ROUNDS; ++r) {
        if (r > 0) {
            __syncthreads();  // the previous round's gather is done with F
            if (has_elem && my_round == r) {
#pragma unroll
                for (int k = 0; k < NPE; ++k) st3(L.F, frow(le - r * te_round, k), fe[k]);
            }
            __syncthreads();
        }
        const int off = r * te_round * NPE, lim = off + te_round * NPE;
#pragma unroll
        for (int q = 0; q < NPE; ++q) {
            const int ln = tid + q * (int)blockDim.x;
            if (ln < tn) {
                const uint32_t pk = L.csr[ln];
                const int st = (int)(pk >> 16), cnt = (int)(pk & 0xffffu);
                int j = jpos[q];
                for (; j < cnt; ++j) {
                    const int s = L.ent[st + j];
                    if (s >= lim) break;
                    const int rw = 3 * frow((s - off) / NPE, (s - off) % NPE);
                    acc[q][0] += L.F[rw];
                    acc[q][1] += L.F[rw + 1];
                    acc[q][2] += L.F[rw + 2];
                }
                jpos[q] = j;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NPE; ++q) {
        const int ln = tid + q * (int)blockDim.x;
        if (ln < tn) finish_node<MODE>(A, L, ln, nint, ibase, acc[q]);
    }
}

// Gauss Hex8 tile step: the phases of k_tile with eight lanes per element (hex8_lanes).  Bound
// by VALU issue (340 FP64 and about 230 other instructions a Gauss point; 77 % of the issue
// slots busy on the uneven ensemble).  One element per thread held 246 VGPRs, two waves per
// SIMD, and gave a 128-element tile two waves in all; the lanes' kernel fits the 128 VGPRs of
// four waves per SIMD (the wide materials two).  20^3 Hex8, a step: 21.6 -> 12.5 us alone; the
// 1.3M-Hex8 ensemble, where issue slots alone count, 0.20 ms of tile kernel either way.  The
// elements' forces and, before them, the modes share the element's LDS row; a tile whose rows
// do not fit the LDS passes them through in rounds (MULTI), between which a node's thread keeps
// its row's sum in global memory: the same sequence for every number of rounds.
template <int KIND, bool PER_QP, int MODE, bool MULTI, bool UL = false>
__global__ __launch_bounds__((MULTI || hex_wide<KIND, UL>()) ? 512 : 1024, (MULTI || hex_wide<KIND, UL>()) ? 2 : 4) void k_hex_tile(TileArgs A) {
    extern __shared__ __align__(16) char lds_raw[];
    const int64_t t = xcd_tile(A.nblocks);
    if (t >= A.ntiles) return;
    const int rounds = MULTI ? A.hx_rounds : 1, rw = A.te / rounds;
    const TileLds L = carve(lds_raw, A.maxtn, A.max_nint, hex_entries(A.maxtn, rounds), tile_f_doubles(8, rw, false), MULTI);
    const int tid = threadIdx.x, nt = blockDim.x;
    // A: every global load of the stage before the first LDS write (see k_tile)
    constexpr int PASSES = hex_wide<KIND, UL>() ? 4 : 2;  // te <= PASSES * blockDim / 8
    const uint4 *conn = reinterpret_cast<const uint4 *>(A.hx_conn) + t * (int64_t)A.te;
    uint4 cq[PASSES];
    if constexpr (!MULTI) {
#pragma unroll
        for (int q = 0; q < PASSES; ++q) cq[q] = conn[min((tid + q * nt) >> 3, rw - 1)];
    }
    const int wave0 = tid & ~63;  // waves past the last node row load none
    double x0[3], u0[3], v0[3], a0[3], m0 = 1.0, d0 = A.dt;
    unsigned f0 = 0u;
    int32_t bd0 = 0;
    uint4 en0{};
    uint32_t csr0 = 0;
    if (wave0 < A.tpad) {
        const int64_t row = t * (int64_t)A.tpad + min(tid, A.tpad - 1);
        const int64_t g0 = A.tnp_node[row];
        bd0 = A.tnp_bdst[row];
        if constexpr (!MULTI) {
            en0 = A.hx_first[row];
            csr0 = A.hx_csr[row];
        }
        ld3(A.X, g0, x0);
        ld3(UL ? A.dinc : A.u, g0, u0);
#pragma unroll
        for (int d = 0; d < 3; ++d) v0[d] = a0[d] = 0.0;
        if (!(MODE == 2 && !UL && A.pred && bd0 >= 0)) {  // (a shared row of a predicted state: X and u only)
            f0 = load_fixed(A, g0);
            if constexpr (MODE >= 1) m0 = A.mass[g0];
            if constexpr (MODE == 2) {
                ld3(A.v, g0, v0);
                if (UL || !A.pred) ld3(A.a, g0, a0);
                d0 = load_node_dt(A, g0);
            }
        }
    }
    const int tn = A.tn_start[t + 1] - A.tn_start[t];
    const int nint = A.tn_ninterior[t];
    const int64_t ibase = A.int_base[t];
    const int64_t te0 = A.tile_e0[t];
    const int nel = A.tile_e0[t + 1] - (int)te0;
    if (tid < 3) L.F[kHexRow * rw + tid] = 0.0;  // the row of padding entries
    auto stage = [&](int ln, uint4 en, uint32_t csr, int32_t bdst, const double *x, const double *u, const double *v,
                     const double *a, unsigned fx, double mm, double nd) {
        if constexpr (!MULTI) {
            reinterpret_cast<uint4 *>(L.ent)[ln] = en;
            L.csr[ln] = csr;
        }
        L.bdst[ln] = bdst;
        st3(L.X, ln, x);
        if (!MULTI && ln < nint) {
            L.fx[ln] = (uint8_t)fx;
            L.M[ln] = mm;
            L.DT[ln] = nd;
        }
        if constexpr (MODE == 2) {
            double vh[3] = {v[0], v[1], v[2]}, u1[3] = {u[0], u[1], u[2]};
            if (UL || !A.pred) stage_predict<UL>(A, u, v, a, fx, nd, vh, u1);
            st3(L.U, ln, u1);
            if (ln < nint) st3(L.V, ln, vh);
        } else {
            st3(L.U, ln, u);
        }
    };
    if (tid < tn) stage(tid, en0, csr0, bd0, x0, u0, v0, a0, f0, m0, d0);
    for (int ln = tid + nt; ln < tn; ln += nt) {  // tiles with more nodes than threads
        const int64_t row = t * (int64_t)A.tpad + ln, g = A.tnp_node[row];
        double x[3], u[3], v[3], a[3], mm = 1.0, nd = A.dt;
        ld3(A.X, g, x);
        ld3(UL ? A.dinc : A.u, g, u);
        const unsigned fx = load_fixed(A, g);
        if constexpr (MODE >= 1) mm = A.mass[g];
        if constexpr (MODE == 2) {
            ld3(A.v, g, v);
            ld3(A.a, g, a);
            nd = load_node_dt(A, g);
        }
        stage(ln, MULTI ? uint4{} : A.hx_first[row], MULTI ? 0u : A.hx_csr[row], A.tnp_bdst[row], x, u, v, a, fx, mm,
              nd);
    }
    __syncthreads();

    // node sums: eight entries' rows in flight (padding entries add zero), in ascending order
    auto add8 = [&](const uint4 &w, double (&f)[3]) {
        const unsigned en[8] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16,
                                w.z & 0xffffu, w.z >> 16, w.w & 0xffffu, w.w >> 16};
        double r[8][3];
#pragma unroll
        for (int k = 0; k < 8; ++k) ld3(L.F + en[k], 0, r[k]);
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int d = 0; d < 3; ++d) f[d] += r[k][d];
    };
    auto add_more = [&](uint32_t csr, int32_t base, double (&f)[3]) {
        for (uint32_t k = 0; k < (csr & 0xffffu); ++k) add8(A.hx_more[base + (csr >> 16) + k], f);
    };
    for (int r = 0; r < rounds; ++r) {
        // B: eight lanes per element; a group of eight is active or idle together
        auto element = [&](int lr, const uint4 &cw) {
            const int le = r * rw + lr;
            const int64_t e = te0 + le;
            MatParams m = A.mat;
            {  // (a uniform base and a 32-bit lane offset)
                const double *pl = A.elem_lambda ? A.elem_lambda + te0 : A.zero;
                const double *pm = A.elem_lambda ? A.elem_mu + te0 : A.zero;
                const unsigned i = A.elem_lambda ? (unsigned)le : 0u;
                const double lam = pl[i], mu = pm[i];
                m.lambda = A.elem_lambda ? lam : m.lambda;
                m.mu = A.elem_lambda ? mu : m.mu;
            }
            RateIn rin;
            load_rate<KIND, UL>(rin, A.Hn, A.Pn, A.ne, e, A.rate_dt);
            const uint32_t cn[4] = {cw.x, cw.y, cw.z, cw.w};
            const int64_t so = state_width<KIND>() * (PER_QP ? e * 8 : e);
            double H[9], P[9];
            const bool last = hex8_lanes<KIND, PER_QP, MULTI, UL>(tid & 7, cn, L.X, L.U, L.F + kHexRow * lr, m, A.gauss_a,
                                                       state_width<KIND>() ? A.state_n + so : nullptr,
                                                       state_width<KIND>() ? A.state_np1 + so : nullptr, H, P, &rin);
            if (last && A.keep_h) {
#pragma unroll
                for (int i = 0; i < 9; ++i) {
                    store_once(A.H + i * A.ne + e, H[i]);
                    if (A.keep) store_once(A.P + i * A.ne + e, P[i]);
                }
            }
        };
        if constexpr (!MULTI) {
#pragma unroll
            for (int q = 0; q < PASSES; ++q) {
                const int lr = (tid + q * nt) >> 3;
                if (lr >= rw || lr >= nel) break;
                element(lr, cq[q]);
            }
        } else {
#pragma unroll 1
            for (int lr = tid >> 3; lr < min(rw, nel - r * rw); lr += nt >> 3) element(lr, conn[r * rw + lr]);
        }
        __syncthreads();
        // C: gather
        if constexpr (!MULTI) {
            for (int ln = tid; ln < tn; ln += nt) {
                double f[3] = {0.0, 0.0, 0.0};
                add8(reinterpret_cast<const uint4 *>(L.ent)[ln], f);
                const uint32_t csr = L.csr[ln];
                if (csr & 0xffffu) add_more(csr, A.hx_base[t], f);
                finish_node<MODE, UL>(A, L, ln, nint, ibase, f);
            }
        } else {
            const int64_t tr = t * (int64_t)rounds + r;
            for (int ln = tid; ln < tn; ln += nt) {
                double f[3] = {0.0, 0.0, 0.0};
                const int64_t row = t * (int64_t)A.tpad + ln;
                if (r > 0) ld3(A.hx_part, row, f);
                add8(A.hx_first[tr * A.tpad + ln], f);
                const uint32_t csr = A.hx_csr[tr * A.tpad + ln];
                if (csr & 0xffffu) add_more(csr, A.hx_base[tr], f);
                if (r + 1 < rounds) st3(A.hx_part, row, f);
                else finish_node<MODE, UL, true>(A, L, ln, nint, ibase, f);
            }
            if (r + 1 < rounds) __syncthreads();
        }
    }
}

// ---- persistent, software-pipelined Tet4 step -------------------------------
// Same arithmetic and summation order as k_tile<4, KIND, 2>, so the
// results are bitwise identical.  A block owns the tile sequence
//   tbeg(xcd) + kx, + bx, + 2 bx, ...   (xcd = block % 8, kx = block / 8)
// inside the Morton range of its XCD and overlaps the global loads of the next
// tiles with the work of the current one: while tile j is evaluated, the node
// data of tile j+1, the node slots of tile j+2 and the scalars of tile j+3 are in
// flight.  Node staging is double-buffered in LDS and tile j+1 is committed to the
// idle buffer after tile j's element arithmetic but before tile j's H / P stores.
// gfx9 counts loads and stores on one in-order counter, so this order lets the
// wait for the prefetched data leave the fresh stores in flight.  Every global
// access in the loop is unconditional (idle lanes use clamped loads and dropped
// buffer stores): a memory instruction under a branch would make the compiler's
// wait counts conservative at the join, and a conservative count drains the stores.
// Requires one element per thread and at most one tile node per thread.

// Per-tile scalars, packed so that one 32-byte load brings all of them.
struct TileMeta {
    int tb, tn, nint, nel;  // first tile-node slot, tile nodes, interior nodes, elements
    int ibase, e0, pad0, pad1;  // first interior node id, first element
};

__device__ __forceinline__ TileMeta load_meta(const TileArgs &A, int64_t t) {
    const int4 *p = reinterpret_cast<const int4 *>(A.meta + 8 * t);
    const int4 a = p[0], b = p[1];
    return TileMeta{a.x, a.y, a.z, a.w, b.x, b.y, 0, 0};
}

// Raw buffer stores (stride 0): a store whose offset lies past the resource's
// num_records is discarded by the hardware's range check, which turns a
// per-lane condition into an unconditional instruction with no memory traffic.
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
constexpr uint32_t kDropOffset = 0x80000000u;  // beyond every resource (all are < 2 GiB)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void *p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

// aux: cache policy (2 = nt, the non-temporal hint used for the H / P stream)
template <int AUX = 0>
__device__ __forceinline__ void bstore(__amdgpu_buffer_rsrc_t r, uint32_t off, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), r, off, 0, AUX);
}

__device__ __forceinline__ void bstore3(__amdgpu_buffer_rsrc_t r, uint32_t off, const double *v) {
    bstore(r, off, v[0]);
    bstore(r, off + 8, v[1]);
    bstore(r, off + 16, v[2]);
}

struct StageIdx {  // per-thread node slot of a tile
    int g;
    uint32_t csr;
    int bdst;
};

struct StageData {  // one thread's share of a tile, from global memory
    TileMeta mt;
    uint32_t csr;
    int bdst;
    double x[3], u[3], v[3], a[3];
    double m, ndt, lam, mu, sn;
    unsigned fx;
    ushort4 lc;
    uint32_t w0, w1;
};

// One staging buffer: the tile's nodes and elements as the element and node phases read them.
struct StageLds {
    double *X, *U, *V, *M, *DT, *LAM, *MU, *SN;
    uint32_t *csr;
    int32_t *bdst;
    ushort4 *lc;
    uint32_t *ent;  // the tile's CSR entries (u16 pairs)
    uint8_t *fx;
};

__host__ __device__ inline size_t stage_bytes(int te, int maxtn) {
    const size_t d = 8 * (11 * (size_t)maxtn + 3 * (size_t)te);  // X U V M DT LAM MU SN
    const size_t w = 4 * (2 * (size_t)maxtn) + 8 * (size_t)te + 8 * (size_t)te;  // csr bdst lc ent
    return (d + w + (size_t)maxtn + 15) & ~(size_t)15;
}

__host__ __device__ inline size_t stream_lds_bytes(int te, int maxtn) {
    return 96 * (size_t)te + 2 * stage_bytes(te, maxtn);
}

__device__ __forceinline__ StageLds stage_carve(char *base, int te, int maxtn) {
    StageLds S;
    S.X = reinterpret_cast<double *>(base);
    S.U = S.X + 3 * maxtn;
    S.V = S.U + 3 * maxtn;
    S.M = S.V + 3 * maxtn;
    S.DT = S.M + maxtn;
    S.LAM = S.DT + maxtn;
    S.MU = S.LAM + te;
    S.SN = S.MU + te;
    S.lc = reinterpret_cast<ushort4 *>(S.SN + te);
    S.ent = reinterpret_cast<uint32_t *>(S.lc + te);
    S.csr = S.ent + 2 * te;
    S.bdst = reinterpret_cast<int32_t *>(S.csr + maxtn);
    S.fx = reinterpret_cast<uint8_t *>(S.bdst + maxtn);
    return S;
}

__device__ __forceinline__ void stage_idx(const TileArgs &A, const TileMeta &mt, int tid, StageIdx &s) {
    const int slot = mt.tb + min(tid, mt.tn - 1);  // clamped: no branch around the loads
    s.g = A.tn_node[slot];
    s.csr = A.tn_csr[slot];
    s.bdst = A.tn_bdst[slot];
}

// Optional per-node increment and per-element moduli are read from the zero buffer
// when absent and added to the uniform value, so the loaded value is used on both
// paths and the compiler keeps the loads unconditional.
template <int KIND>
__device__ __forceinline__ void stage_data(const TileArgs &A, int64_t t, const TileMeta &mt, int tid,
                                           const StageIdx &si, StageData &d) {
    d.mt = mt;
    d.csr = si.csr;
    d.bdst = si.bdst;
    const int64_t g = si.g;
    ld3(A.X, g, d.x);
    ld3(A.u, g, d.u);
    ld3(A.v, g, d.v);
    ld3(A.a, g, d.a);
    d.fx = load_fixed(A, g);
    d.m = A.mass[g];
    const double *pd = A.node_dt ? A.node_dt : A.zero;
    d.ndt = pd[A.node_dt ? g : 0] + (A.node_dt ? 0.0 : A.dt);
    const int64_t e = (int64_t)mt.e0 + min(tid, mt.nel - 1);
    d.lc = reinterpret_cast<const ushort4 *>(A.lconn)[e];
    const int64_t ie = A.elem_lambda ? e : 0;
    const double *pl = A.elem_lambda ? A.elem_lambda : A.zero;
    const double *pm = A.elem_lambda ? A.elem_mu : A.zero;
    d.lam = pl[ie] + (A.elem_lambda ? 0.0 : A.mat.lambda);
    d.mu = pm[ie] + (A.elem_lambda ? 0.0 : A.mat.mu);
    d.sn = 0.0;
    if constexpr (KIND == APHIP_J2) d.sn = A.state_n[e];
    // the tile's CSR entries: te * 4 u16 = 2 words per thread
    const uint32_t *src = reinterpret_cast<const uint32_t *>(A.lcsr + t * (int64_t)(A.te * 4));
    d.w0 = src[tid];
    d.w1 = src[tid + A.te];
}

// Writes one thread's share of a staged tile into an LDS buffer (predictor applied).
__device__ __forceinline__ void stage_commit(const StageData &d, const StageLds &S, int tid, int te) {
    if (tid < d.mt.tn) {
        S.csr[tid] = d.csr;
        S.bdst[tid] = d.bdst;
        st3(S.X, tid, d.x);
        S.fx[tid] = (uint8_t)d.fx;
        S.M[tid] = d.m;
        S.DT[tid] = d.ndt;
        double vh[3], u1[3];
        cd_predict(d.u, d.v, d.a, d.fx, d.ndt, vh, u1);
        st3(S.U, tid, u1);
        st3(S.V, tid, vh);
    }
    S.lc[tid] = d.lc;
    S.LAM[tid] = d.lam;
    S.MU[tid] = d.mu;
    S.SN[tid] = d.sn;
    S.ent[tid] = d.w0;
    S.ent[tid + te] = d.w1;
}

template <int KIND>
__global__ __launch_bounds__(256) void k_tile_stream(TileArgs A, int nblk) {
    extern __shared__ __align__(16) char lds_raw[];
    const int te = A.te;
    double *F = reinterpret_cast<double *>(lds_raw);
    const size_t sb = stage_bytes(te, A.maxtn);
    const StageLds S0 = stage_carve(lds_raw + 96 * (size_t)te, te, A.maxtn);
    const StageLds S1 = stage_carve(lds_raw + 96 * (size_t)te + sb, te, A.maxtn);
    const int tid = threadIdx.x;
    const int xcd = blockIdx.x % kNumXcd, kx = blockIdx.x / kNumXcd;
    const int bx = nblk / kNumXcd;
    const int64_t per = (A.ntiles + kNumXcd - 1) / kNumXcd;
    const int64_t tend = min(A.ntiles, (int64_t)(xcd + 1) * per);
    int64_t t = (int64_t)xcd * per + kx;
    if (t >= tend) return;
    // every prefetch is unconditional, on tile ids clamped to the block's range: a
    // branch around a load would make the compiler wait for it at the join
    const int64_t tlast = tend - 1;
    // (an inner step's H, P and f stores are dropped by empty resources)
    const int64_t hp_bytes = A.keep ? 72 * A.ne : 0;
    const __amdgpu_buffer_rsrc_t rH = buffer_rsrc(A.H, hp_bytes), rP = buffer_rsrc(A.P, hp_bytes);
    const __amdgpu_buffer_rsrc_t rS = buffer_rsrc(A.state_np1, KIND == APHIP_J2 ? 8 * A.ne : 0);
    const __amdgpu_buffer_rsrc_t rF = buffer_rsrc(A.f, A.keep ? 24 * A.nn : 0), rU = buffer_rsrc(A.u, 24 * A.nn);
    const __amdgpu_buffer_rsrc_t rV = buffer_rsrc(A.v, 24 * A.nn), rA = buffer_rsrc(A.a, 24 * A.nn);
    const __amdgpu_buffer_rsrc_t rB = buffer_rsrc(A.bpart, 24 * A.nslot);

    StageIdx si;
    StageData d;
    {
        const TileMeta m0 = load_meta(A, t);
        stage_idx(A, m0, tid, si);
        stage_data<KIND>(A, t, m0, tid, si, d);
        stage_commit(d, S0, tid, te);
    }
    TileMeta m1 = load_meta(A, min(t + bx, tlast));
    stage_idx(A, m1, tid, si);
    TileMeta m2 = load_meta(A, min(t + 2 * bx, tlast));
    TileMeta c = d.mt;  // the tile in the current buffer
    bool odd = false;
    __syncthreads();

    // One tile; returns false after the block's last tile.  The first call is peeled
    // off the loop so that the loop header merges two identical states and the
    // compiler's wait counts for the in-flight prefetch stay exact.
    auto tile = [&]() __attribute__((always_inline)) -> bool {
        const StageLds &S = odd ? S1 : S0;
        const StageLds &Sn = odd ? S0 : S1;
        const int64_t t1 = t + bx;
        // prefetch (data of t1, slots of t2, scalars of t3)
        stage_data<KIND>(A, min(t1, tlast), m1, tid, si, d);
        stage_idx(A, m2, tid, si);
        m1 = m2;
        m2 = load_meta(A, min(t + 3 * bx, tlast));
        // keep the scheduler from sinking the prefetch towards its use
        __builtin_amdgcn_sched_barrier(0);
        // B: element (every lane computes; the stores of lanes past the last element are dropped)
        const bool has_elem = tid < c.nel;
        const int64_t e = (int64_t)c.e0 + tid;
        {
            const ushort4 q = S.lc[tid];
            const int lc[4] = {q.x, q.y, q.z, q.w};
            MatParams m = A.mat;
            m.lambda = S.LAM[tid];
            m.mu = S.MU[tid];
            double X[4][3], U[4][3], fe[4][3];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                ld3(S.X, lc[k], X[k]);
                ld3(S.U, lc[k], U[k]);
            }
            static_assert(state_width<KIND>() <= 1, "the pipelined kernel keeps one state value per element");
            double H[9], P[9], snp1 = 0.0, aux = 0.0;
            tet4_element<KIND>(X, U, m, S.SN[tid], snp1, aux, H, P, fe);
#pragma unroll
            for (int k = 0; k < 4; ++k) st3(F, tid * 4 + k, fe[k]);
            // commit the prefetched tile before this tile's stores are issued
            stage_commit(d, Sn, tid, te);
            const uint32_t oe = has_elem ? (uint32_t)(8 * e) : kDropOffset;
            const uint32_t oi = (uint32_t)(8 * A.ne);
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                bstore<2>(rH, oe + i * oi, H[i]);
                bstore<2>(rP, oe + i * oi, P[i]);
            }
            if constexpr (KIND == APHIP_J2) bstore<2>(rS, oe, snp1);
        }
        __syncthreads();

        // C: gather and finish (same order as k_tile).  Stores are unconditional; those
        // of lanes past the tile's nodes, and the u, v, a of a shared node (finished by
        // the shared-node pass), are dropped.
        {
            const bool live = tid < c.tn, interior = tid < c.nint;
            const int ln = min(tid, c.tn - 1);
            const uint32_t pk = S.csr[ln];
            const int st = (int)(pk >> 16), cnt = (int)(pk & 0xffffu);
            const uint16_t *ent = reinterpret_cast<const uint16_t *>(S.ent);
            double f[3] = {0.0, 0.0, 0.0};
            for (int j = 0; j < cnt; ++j) {
                const int s = ent[st + j];
                f[0] += F[3 * s];
                f[1] += F[3 * s + 1];
                f[2] += F[3 * s + 2];
            }
            double vh[3], u1[3], a1[3], v1[3];
            ld3(S.V, ln, vh);
            ld3(S.U, ln, u1);
            cd_correct(f, S.M[ln], S.fx[ln], S.DT[ln], vh, a1, v1);
            const int64_t g = (int64_t)c.ibase + tid;
            const uint32_t og = (live && interior) ? (uint32_t)(24 * g) : kDropOffset;
            const uint32_t ob = (live && !interior) ? (uint32_t)(24 * (int64_t)S.bdst[ln]) : kDropOffset;
            bstore3(rF, og, f);
            bstore3(rB, ob, f);
            bstore3(rU, og, u1);
            bstore3(rV, og, v1);
            bstore3(rA, og, a1);
        }
        if (t1 >= tend) return false;
        c = d.mt;
        odd = !odd;
        t = t1;
        __syncthreads();
        return true;
    };
    if (tile())
        while (tile()) {
        }
}

struct BoundArgs {
    int64_t nb;
    int64_t first;  // global id of the first shared node
    const int32_t *bstart;
    const double *bpart;
    double *u, *v, *a, *f;
    const double *mass;
    const uint8_t *fixed;
    const double *node_dt;
    const double *zero;  // 8 zero doubles: stands in for an absent optional array
    double dt;
    int pred, more;  // as in TileArgs
    int keep;       // 0: an inner step, f is not stored
    // updated / semi-Lagrangian: the configuration integrated over, and as in TileArgs
    const double *xn;
    double *dinc, *xnp1;
    int semi;
};

// One thread per component of a node: a wave's accesses to u, v, a, f and (the slots of
// consecutive nodes being consecutive) to the slots are contiguous runs.  Bound by memory; one
// thread per node, three strided accesses each, took 36 us where this took 34.8 (6M Tet4 in tiles of
// 512: memory-bound there, 73k Tet4: 14.1 -> 12.2 us a step alone), and 23.1 once the steps of a call left
// the next predictor in u and v instead of u, v, a and a copy of the predicted displacement.
constexpr int kBoundNodes = 64;  // nodes per workgroup
template <int MODE, bool UL = false>
__global__ __launch_bounds__(3 * kBoundNodes) void k_boundary(BoundArgs A) {
#pragma clang fp contract(off)
    const int64_t b_raw = (int64_t)blockIdx.x * kBoundNodes + threadIdx.x / 3;
    const int d = threadIdx.x % 3;
    const bool live = b_raw < A.nb;
    const int64_t b = live ? b_raw : A.nb - 1;  // idle lanes redo the last node and store nothing
    const int64_t g = A.first + b, k = 3 * g + d;
    const int32_t s0 = A.bstart[b], s1 = A.bstart[b + 1];
    // node data first: independent of the slot sums, so its loads overlap them
    double u = 0.0, v = 0.0, a = 0.0, m = 1.0, dt = A.dt;
    bool fx = false;
    if constexpr (MODE >= 1) m = A.mass[g];
    if constexpr (MODE == 2) {
        u = A.u[k];
        v = A.v[k];
        if (UL || !A.pred) a = A.a[k];
        const uint8_t *pf = A.fixed ? A.fixed : reinterpret_cast<const uint8_t *>(A.zero);
        const double *pd = A.node_dt ? A.node_dt : A.zero;
        const unsigned f8 = pf[A.fixed ? g : 0];
        const double d8 = pd[A.node_dt ? g : 0];
        fx = A.fixed && (f8 & (1u << d));
        dt = A.node_dt ? d8 : A.dt;
    }
    // slot sums in ascending tile order, four slots' loads at a time (clamped; an
    // absent slot adds zero)
    double f = 0.0;
    for (int32_t sb = s0; sb < s1; sb += 4) {
        double p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = A.bpart[3 * (int64_t)min(sb + r, s1 - 1) + d];
#pragma unroll
        for (int r = 0; r < 4; ++r) f += sb + r < s1 ? p[r] : 0.0;
    }
    if (!live) return;
    if (MODE != 2 || A.keep) A.f[k] = f;
    if constexpr (MODE == 1) {
        A.a[k] = f / m;
    } else if constexpr (MODE == 2) {
        double vh = v, u1 = u, a1, v1;
        if (UL || !A.pred) cd_predict1(u, v, a, fx, dt, vh, u1);
        cd_correct1(f, m, fx, dt, vh, a1, v1);
        if constexpr (UL) ul_store1(A.u, A.dinc, A.xnp1, A.semi, k, dt, vh, A.xn[k], A.dinc[k] + dt * vh);
        if (!UL && A.more) {
            double vh2, u2;
            cd_predict1(u1, v1, a1, fx, dt, vh2, u2);
            A.u[k] = u2;
            A.v[k] = vh2;
        } else {
            if constexpr (!UL) A.u[k] = u1;
            A.v[k] = v1;
            A.a[k] = a1;
        }
    }
}

inline int64_t padded(int64_t n) { return ((n + kNumXcd - 1) / kNumXcd) * kNumXcd; }

template <int NPE, int KIND, bool PER_QP, int MODE>
void launch_tile(Ctx &c, const TileArgs &A) {
    const TilePlan &P = c.tiles;
    auto go = [&](auto kern, int threads, size_t lds) {
        allow_lds(c, (const void *)kern, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)A.nblocks), dim3(threads), lds, c.stream, A);
    };
    if constexpr (MODE == 2) {
        if (c.formulation != APHIP_TOTAL_LAGRANGIAN) {
            if constexpr (NPE == 4) go(k_tile<4, KIND, 2, true>, P.threads, P.lds_bytes);
            else go(k_hex_tile<KIND, PER_QP, 2, false, true>, hex_threads<KIND, true>(P.te, 1), P.lds_bytes);
            return;
        }
    }
    if constexpr (NPE == 4) {
        if constexpr (MODE == 0) {
            if (A.phi.num) {
                go(k_tile<4, KIND, 0, false, true>, P.threads, P.lds_bytes);
                return;
            }
        }
        go(k_tile<4, KIND, MODE>, P.threads, P.lds_bytes);
    } else {
        if constexpr (MODE == 0 && !PER_QP) {
            if (c.cells.ready) {
                go(k_tile<8, KIND, 0>, P.te, P.cell_lds_bytes);
                return;
            }
        }
        if (P.hx_rounds == 1) go(k_hex_tile<KIND, PER_QP, MODE, false>, hex_threads<KIND>(P.te, 1), P.lds_bytes);
        else go(k_hex_tile<KIND, PER_QP, MODE, true>, hex_threads<KIND>(P.te, P.hx_rounds), P.lds_bytes);
    }
}

template <int KIND>
void launch_stream(Ctx &c, const TileArgs &A) {
    auto kern = k_tile_stream<KIND>;
    TilePlan &P = c.tiles;
    const size_t lds = stream_lds_bytes(P.te, P.maxtn);
    int &grid = P.stream_grid[KIND];
    if (grid == 0) {
        allow_lds(c, (const void *)kern, lds);
        int per_cu = 0, cus = 0;
        APHIP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, P.threads, lds));
        APHIP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c.device));
        const int64_t want = std::max<int64_t>(1, std::min<int64_t>((P.ntiles + kNumXcd - 1) / kNumXcd,
                                                                   (int64_t)std::max(per_cu, 1) * cus / kNumXcd));
        grid = (int)(want * kNumXcd);
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(P.threads), lds, c.stream, A, grid);
}

bool stream_eligible(const Ctx &c) {
    const TilePlan &P = c.tiles;
    // buffer-store offsets are 32-bit and must stay below the drop offset (2 GiB)
    const int64_t lim = (int64_t)1 << 31;
    return P.use_stream && c.npe == 4 && P.te == P.threads && P.threads <= 256 && P.maxtn <= P.threads &&
           stream_lds_bytes(P.te, P.maxtn) <= 160 * 1024 && 72 * c.ne < lim && 24 * c.nn < lim &&
           24 * P.nslot < lim;
}

bool stream_kind(int kind) {
    return kind == APHIP_LINEAR_ELASTIC || kind == APHIP_NEO_HOOKEAN || kind == APHIP_J2 || kind == APHIP_SVK;
}

template <int NPE, int MODE>
void dispatch_kind(Ctx &c, const TileArgs &A) {
    if constexpr (NPE == 4 && MODE == 2) {
        if (stream_eligible(c) && c.formulation == APHIP_TOTAL_LAGRANGIAN) {
            switch (c.mat.kind) {
                case APHIP_LINEAR_ELASTIC: launch_stream<APHIP_LINEAR_ELASTIC>(c, A); return;
                case APHIP_NEO_HOOKEAN: launch_stream<APHIP_NEO_HOOKEAN>(c, A); return;
                case APHIP_J2: launch_stream<APHIP_J2>(c, A); return;
                case APHIP_SVK: launch_stream<APHIP_SVK>(c, A); return;
                default: break;
            }
        }
    }
    const bool pq = c.mat.state_per_qp && NPE == 8;
    switch (c.mat.kind) {
        case APHIP_LINEAR_ELASTIC: launch_tile<NPE, APHIP_LINEAR_ELASTIC, false, MODE>(c, A); break;
        case APHIP_NEO_HOOKEAN: launch_tile<NPE, APHIP_NEO_HOOKEAN, false, MODE>(c, A); break;
        case APHIP_J2:
            if (pq) launch_tile<NPE, APHIP_J2, true, MODE>(c, A);
            else launch_tile<NPE, APHIP_J2, false, MODE>(c, A);
            break;
        case APHIP_SVK: launch_tile<NPE, APHIP_SVK, false, MODE>(c, A); break;
        case APHIP_NEO_HOOKEAN_DAMAGE:
            if (pq) launch_tile<NPE, APHIP_NEO_HOOKEAN_DAMAGE, true, MODE>(c, A);
            else launch_tile<NPE, APHIP_NEO_HOOKEAN_DAMAGE, false, MODE>(c, A);
            break;
        case APHIP_POWER_LAW_CREEP:
            if (pq) launch_tile<NPE, APHIP_POWER_LAW_CREEP, true, MODE>(c, A);
            else launch_tile<NPE, APHIP_POWER_LAW_CREEP, false, MODE>(c, A);
            break;
        case APHIP_DRUCKER_PRAGER:
            if (pq) launch_tile<NPE, APHIP_DRUCKER_PRAGER, true, MODE>(c, A);
            else launch_tile<NPE, APHIP_DRUCKER_PRAGER, false, MODE>(c, A);
            break;
        default: throw Error(APHIP_ERR_INVALID, "material not set");
    }
}

}  // namespace

// Builds the tile plan for the current internal connectivity and renumbers the
// nodes so that interior nodes are contiguous per tile and shared nodes follow.
void tile_build(Ctx &c, int te, int threads) {
    const int npe = c.npe;
    const int64_t ne = c.ne, nn = c.nn;
    APHIP_REQUIRE(!c.cells.ready, "tiling applies to the Gaussian element path");
    c.graph_reset();
    if (npe == 4) {
        APHIP_REQUIRE(te == threads && (threads == 64 || threads == 128 || threads == 256 || threads == 512 ||
                                        threads == 1024),
                      "Tet4 tiles: one element per thread, 64, 128, 256, 512 or 1024 threads");
    } else {
        const bool per_elem = te == threads && (threads == 64 || threads == 128 || threads == 256);
        const bool per_qp = threads == 8 * te && (te == 8 || te == 16 || te == 32 || te == 64);
        APHIP_REQUIRE(per_elem || per_qp,
                      "Hex8 tiles: one element per thread (64, 128 or 256) or eight lanes per element (8..64 elements)");
    }
    const std::vector<int32_t> &ci = c.conn_h;
    // tiles: consecutive chunks of te elements inside each element block
    std::vector<int32_t> te0v;
    for (size_t sg = 0; sg + 1 < c.elem_seg.size(); ++sg)
        for (int64_t e = c.elem_seg[sg]; e < c.elem_seg[sg + 1]; e += te) te0v.push_back((int32_t)e);
    const int64_t nt = (int64_t)te0v.size();
    te0v.push_back((int32_t)ne);

    // 1. node set of every tile and the number of tiles touching each node
    std::vector<int32_t> ntouch(nn, 0), stamp(nn, -1);
    std::vector<int32_t> tstart(nt + 1, 0), tnodes;
    tnodes.reserve((size_t)(ne * npe / 3 + 16));
    std::vector<int32_t> tmp;
    for (int64_t t = 0; t < nt; ++t) {
        tmp.clear();
        const int64_t e0 = te0v[t], e1 = te0v[t + 1];
        for (int64_t e = e0; e < e1; ++e)
            for (int k = 0; k < npe; ++k) {
                const int32_t n = ci[e * npe + k];
                if (stamp[n] != (int32_t)t) {
                    stamp[n] = (int32_t)t;
                    tmp.push_back(n);
                    ntouch[n]++;
                }
            }
        std::sort(tmp.begin(), tmp.end());
        tnodes.insert(tnodes.end(), tmp.begin(), tmp.end());
        APHIP_REQUIRE(tnodes.size() < (size_t)INT32_MAX, "tile node count overflow");
        tstart[t + 1] = (int32_t)tnodes.size();
    }

    // 2. new numbering: interior nodes tile by tile, then every other node in old order
    std::vector<int32_t> new_of_old(nn, -1), int_base(nt), ninterior(nt);
    int32_t next = 0;
    for (int64_t t = 0; t < nt; ++t) {
        int_base[t] = next;
        for (int32_t i = tstart[t]; i < tstart[t + 1]; ++i)
            if (ntouch[tnodes[i]] == 1) new_of_old[tnodes[i]] = next++;
        ninterior[t] = next - int_base[t];
    }
    const int64_t n_interior = next;
    for (int64_t n = 0; n < nn; ++n)
        if (new_of_old[n] < 0) new_of_old[n] = next++;
    const int64_t nb = nn - n_interior;

    // 3. tile node lists in new ids (interior first, each part ascending), local conn and CSR
    for (auto &x : tnodes) x = new_of_old[x];
    int maxtn = 0;
    std::vector<int32_t> loc(nn, -1);
    std::vector<uint16_t> lconn((size_t)ne * npe), lcsr((size_t)nt * te * npe, 0);
    std::vector<uint32_t> tcsr(tnodes.size());
    std::vector<int32_t> cnt, fillp;
    for (int64_t t = 0; t < nt; ++t) {
        auto b = tnodes.begin() + tstart[t], en = tnodes.begin() + tstart[t + 1];
        const int tn = (int)(en - b);
        APHIP_REQUIRE(tn <= 65535, "tile has more than 65535 nodes");
        maxtn = std::max(maxtn, tn);
        std::sort(b, en);  // interior ids are < n_interior, so they come first
        for (int i = 0; i < tn; ++i) loc[*(b + i)] = i;
        cnt.assign(tn, 0);
        const int64_t e0 = te0v[t], e1 = te0v[t + 1];
        for (int64_t e = e0; e < e1; ++e)
            for (int k = 0; k < npe; ++k) {
                const int ln = loc[new_of_old[ci[e * npe + k]]];
                lconn[e * npe + k] = (uint16_t)ln;
                cnt[ln]++;
            }
        fillp.assign(tn, 0);
        int run = 0;
        for (int ln = 0; ln < tn; ++ln) {
            fillp[ln] = run;
            tcsr[tstart[t] + ln] = ((uint32_t)run << 16) | (uint32_t)cnt[ln];
            run += cnt[ln];
        }
        uint16_t *dst = &lcsr[(size_t)t * te * npe];
        for (int64_t e = e0; e < e1; ++e)
            for (int k = 0; k < npe; ++k) {
                const int ln = loc[new_of_old[ci[e * npe + k]]];
                dst[fillp[ln]++] = (uint16_t)((e - e0) * npe + k);
            }
    }

    // 4. shared-node slots: contiguous per node, ascending tile order
    std::vector<int32_t> bstart(nb + 1, 0), tbdst(tnodes.size(), -1);
    for (int64_t t = 0; t < nt; ++t)
        for (int32_t i = tstart[t] + ninterior[t]; i < tstart[t + 1]; ++i) bstart[tnodes[i] - n_interior + 1]++;
    for (int64_t b = 0; b < nb; ++b) bstart[b + 1] += bstart[b];
    std::vector<int32_t> bfill(bstart.begin(), bstart.end() - 1);
    for (int64_t t = 0; t < nt; ++t)
        for (int32_t i = tstart[t] + ninterior[t]; i < tstart[t + 1]; ++i)
            tbdst[i] = bfill[tnodes[i] - n_interior]++;

    // 5. renumber the context's nodes, then upload the plan
    std::vector<int32_t> old_of_new(nn);
    for (int64_t n = 0; n < nn; ++n) old_of_new[new_of_old[n]] = (int32_t)n;
    renumber_nodes(c, old_of_new);

    TilePlan &P = c.tiles;
    P.te = te;
    P.threads = threads;
    P.ntiles = nt;
    P.maxtn = maxtn;
    P.nb = nb;
    P.n_interior = n_interior;
    P.by_user = false;
    P.orphans = false;
    for (int64_t b = 0; b < nb; ++b) P.orphans |= bstart[b] == bstart[b + 1];
    P.total_tile_nodes = (int64_t)tnodes.size();
    P.tn_start.upload(tstart.data(), tstart.size(), c.stream);
    P.tile_e0.upload(te0v.data(), te0v.size(), c.stream);
    P.tn_ninterior.upload(ninterior.data(), ninterior.size(), c.stream);
    P.int_base.upload(int_base.data(), int_base.size(), c.stream);
    P.tn_node.upload(tnodes.data(), tnodes.size(), c.stream);
    P.tn_csr.upload(tcsr.data(), tcsr.size(), c.stream);
    P.tn_bdst.upload(tbdst.data(), tbdst.size(), c.stream);
    P.lcsr.upload(lcsr.data(), lcsr.size(), c.stream);
    P.lconn.upload(lconn.data(), lconn.size(), c.stream);
    {  // fixed-stride copies for the tile kernel
        P.tpad = std::max(maxtn, 1);
        std::vector<int32_t> pn((size_t)nt * P.tpad), pb((size_t)nt * P.tpad);
        std::vector<uint32_t> pc((size_t)nt * P.tpad);
        std::vector<uint16_t> pl((size_t)nt * te * npe);
        for (int64_t t = 0; t < nt; ++t) {
            const int tn = tstart[t + 1] - tstart[t];
            for (int r = 0; r < P.tpad; ++r) {
                const int32_t i = tstart[t] + std::min(r, tn - 1);
                pn[(size_t)t * P.tpad + r] = tnodes[i];
                pc[(size_t)t * P.tpad + r] = tcsr[i];
                pb[(size_t)t * P.tpad + r] = tbdst[i];
            }
            const int64_t e0 = te0v[t], nel = te0v[t + 1] - e0;
            for (int le = 0; le < te; ++le)
                for (int k = 0; k < npe; ++k)
                    pl[((size_t)t * te + le) * npe + k] = lconn[(e0 + std::min<int64_t>(le, nel - 1)) * npe + k];
        }
        P.tnp_node.upload(pn.data(), pn.size(), c.stream);
        P.tnp_csr.upload(pc.data(), pc.size(), c.stream);
        P.tnp_bdst.upload(pb.data(), pb.size(), c.stream);
        P.lconn_p.upload(pl.data(), pl.size(), c.stream);
        if (npe == 8) {  // k_hex_tile's forms
            std::vector<uint16_t> hc(pl.size());
            for (size_t i = 0; i < pl.size(); ++i) hc[i] = (uint16_t)(3 * (int)pl[i]);
            P.hx_conn.upload(hc.data(), hc.size(), c.stream);
            // one round unless the rows do not fit the LDS beside the tile's nodes
            int max_int = 0;
            for (int64_t t = 0; t < nt; ++t) max_int = std::max(max_int, ninterior[t]);
            auto lds_of = [&](int r) { return tile_lds_bytes(maxtn, max_int, te / r, 8, hex_entries(maxtn, r), false, r > 1); };
            int R = 1;
            while (te / R > 16 && lds_of(R) > 160 * 1024) R *= 2;
            const int rw = te / R;
            P.hx_rounds = R;
            P.lds_bytes = lds_of(R);
            std::vector<uint16_t> first((size_t)nt * R * P.tpad * 8, (uint16_t)(kHexRow * rw)), more;
            std::vector<uint32_t> hcsr((size_t)nt * R * P.tpad, 0);
            std::vector<int32_t> base((size_t)nt * R, 0);
            for (int64_t t = 0; t < nt; ++t)
                for (int r = 0; r < R; ++r) {
                    const int64_t tr = t * R + r;
                    base[tr] = (int32_t)(more.size() / 8);
                    for (int ln = 0; ln < tstart[t + 1] - tstart[t]; ++ln) {
                        const uint32_t pk = tcsr[tstart[t] + ln];
                        const uint16_t *es = &lcsr[(size_t)t * te * npe + (pk >> 16)];
                        int k = 0, n = 0, cnt = (int)(pk & 0xffffu);
                        while (k < cnt && es[k] < r * rw * 8) ++k;
                        const uint32_t m0 = (uint32_t)(more.size() / 8 - base[tr]);
                        for (; k < cnt && es[k] < (r + 1) * rw * 8; ++k, ++n) {
                            const int s = es[k] - r * rw * 8;
                            const uint16_t off = (uint16_t)(kHexRow * (s / 8) + 3 * (s % 8));
                            if (n < 8) {
                                first[((size_t)tr * P.tpad + ln) * 8 + n] = off;
                            } else {
                                if (n % 8 == 0) more.resize(more.size() + 8, (uint16_t)(kHexRow * rw));
                                more[more.size() - 8 + n % 8] = off;
                            }
                        }
                        hcsr[(size_t)tr * P.tpad + ln] = (m0 << 16) | (n > 8 ? (uint32_t)(n - 1) / 8 : 0u);
                    }
                }
            APHIP_REQUIRE(more.size() / 8 < (size_t)INT32_MAX, "too many tile entries");
            P.hx_first.upload(reinterpret_cast<const uint4 *>(first.data()), first.size() / 8, c.stream);
            P.hx_more.upload(reinterpret_cast<const uint4 *>(more.data()), more.size() / 8, c.stream);
            P.hx_csr.upload(hcsr.data(), hcsr.size(), c.stream);
            P.hx_base.upload(base.data(), base.size(), c.stream);
            P.hx_part.alloc(R > 1 ? 3 * (size_t)nt * P.tpad : 0);
        }
    }
    P.nslot = bstart[nb];
    P.bpart.alloc(3 * std::max<int64_t>(1, (int64_t)bstart[nb]));
    P.bstart.upload(bstart.data(), bstart.size(), c.stream);
    P.zero.alloc(8);
    P.zero.zero(c.stream);
    {
        std::vector<int32_t> meta((size_t)nt * 8, 0);
        for (int64_t t = 0; t < nt; ++t) {
            int32_t *m = &meta[(size_t)t * 8];
            m[0] = tstart[t];
            m[1] = tstart[t + 1] - tstart[t];
            m[2] = ninterior[t];
            m[3] = te0v[t + 1] - te0v[t];
            m[4] = int_base[t];
            m[5] = te0v[t];
        }
        P.meta.upload(meta.data(), meta.size(), c.stream);
    }
    // LDS: X, U, V (3 doubles each) + mass + increment per node, partials, csr/bdst per node, entries, flags
    int max_nint = 0;
    for (int64_t t = 0; t < nt; ++t) max_nint = std::max(max_nint, ninterior[t]);
    P.max_nint = npe == 4 ? maxtn : max_nint;  // LDS rows of the corrector data (the kernel's choice)
    if (npe == 4) P.lds_bytes = tile_lds_bytes(P.maxtn, P.max_nint, te, npe, te * npe, false);
    P.cell_lds_bytes = tile_lds_bytes(P.maxtn, P.max_nint, te, npe, te * npe, true);
    // (smoothed Hex8 cells check their own at launch)
    APHIP_REQUIRE(P.lds_bytes <= 160 * 1024, "tile needs more LDS than a CU has; use a smaller tile");
    for (const bool cell : {false, true}) {  // the kernels' carve-up must end inside the allocation
        const int R = npe == 8 && !cell ? P.hx_rounds : 1;
        const int nent = npe == 8 && !cell ? hex_entries(P.maxtn, R) : te * npe;
        const TileLds L = carve(nullptr, P.maxtn, P.max_nint, nent, tile_f_doubles(npe, te / R, cell), R > 1);
        APHIP_REQUIRE((size_t)(reinterpret_cast<const char *>(L.fx + (R > 1 ? 0 : P.max_nint)) - static_cast<const char *>(nullptr)) <=
                          (cell ? P.cell_lds_bytes : P.lds_bytes),
                      "tile LDS layout exceeds its allocation");
    }
    // the one-element-per-thread gather covers npe x te nodes; its staging loads te * npe / 2
    // CSR words with at most 2 (Tet4) or 4 (Hex8 cells) per thread.
    APHIP_REQUIRE(maxtn <= npe * te, "tile has more nodes than its gather covers");
    P.use_stream = (c.flags & APHIP_FLAG_PIPELINED) != 0;
    for (int &g : P.stream_grid) g = 0;  // sized (and LDS attribute set) at the first launch
    P.ready = true;
    c.patch.reset();
    APHIP_HIP(hipStreamSynchronize(c.stream));
}

void tile_run(Ctx &c, double dt, int mode, const TileRun &run) {
    TilePlan &P = c.tiles;
    APHIP_REQUIRE(P.ready, "tile plan not built");
    APHIP_REQUIRE(mode == 0 || (run.u_in == nullptr && run.f_out == nullptr && !run.phi && !run.park),
                  "displacement / force arrays only in force mode");
    APHIP_REQUIRE(mode == 2 || !(run.pred_in || run.pred_out), "predicted displacements only in step mode");
    // (the pipelined kernel predicts from u, v and a in every step)
    const bool chain = !(c.npe == 4 && stream_eligible(c) && stream_kind(c.mat.kind));
    const bool pred_in = run.pred_in && chain, pred_out = run.pred_out && chain;
    // smoothed Hex8 cells have a B of their own (a smoothed Tet4's is its gradient)
    const bool cells8 = c.npe == 8 && c.cells.ready;
    APHIP_REQUIRE(!run.phi || c.npe == 4, "Phi rows are staged by Tet4 tiles");
    APHIP_REQUIRE(!cells8 || (mode == 0 && P.threads == P.te), "Hex8 cells: force mode, one cell per thread");
    if (c.ne == 0) return;
    const bool ul = c.formulation != APHIP_TOTAL_LAGRANGIAN;
    APHIP_REQUIRE(!ul || (mode == 2 && !pred_in && !pred_out && P.hx_rounds == 1), "updated formulation: step mode");
    TileArgs A;
    A.X = ul ? c.xcn().p : c.X.p;
    A.u = run.u_in ? const_cast<double *>(run.u_in) : c.u.p;
    A.v = c.v.p;
    A.a = c.a.p;
    A.f = run.f_out ? run.f_out : c.f.p;
    A.mass = c.mass.p;
    A.fixed = c.has_fixed ? c.fixed.p : nullptr;
    A.tn_start = P.tn_start.p;
    A.tile_e0 = P.tile_e0.p;
    A.tn_ninterior = P.tn_ninterior.p;
    A.int_base = P.int_base.p;
    A.tn_node = P.tn_node.p;
    A.tn_csr = P.tn_csr.p;
    A.tn_bdst = P.tn_bdst.p;
    A.lcsr = P.lcsr.p;
    A.lconn = P.lconn.p;
    A.tnp_node = P.tnp_node.p;
    A.tnp_csr = P.tnp_csr.p;
    A.tnp_bdst = P.tnp_bdst.p;
    A.lconn_p = P.lconn_p.p;
    A.tpad = P.tpad;
    A.hx_conn = P.hx_conn.p;
    A.hx_first = P.hx_first.p;
    A.hx_more = P.hx_more.p;
    A.hx_csr = P.hx_csr.p;
    A.hx_base = P.hx_base.p;
    A.hx_part = P.hx_part.p;
    A.hx_rounds = P.hx_rounds;
    A.bpart = P.bpart.p;
    A.H = c.Hnp1().p;
    A.P = c.Pnp1().p;
    A.Hn = c.formulation == APHIP_SEMI_LAGRANGIAN ? c.Href.p : c.h_pair() ? c.Hn().p : nullptr;
    A.Pn = c.mat.rate_form() ? c.Pn().p : nullptr;
    A.rate_dt = mode == 2 ? dt : c.rate_dt;
    A.state_n = c.state[1 - c.state_np1].p;
    A.state_np1 = c.state[c.state_np1].p;
    A.mat = c.mat.params();
    A.elem_lambda = c.has_fields ? c.elem_lambda.p : nullptr;
    A.elem_mu = c.has_fields ? c.elem_mu.p : nullptr;
    A.node_dt = c.node_dt.p;
    A.zero = P.zero.p;
    A.meta = P.meta.p;
    A.gauss_a = 1.0 / std::sqrt(3.0);
    A.ne = c.ne;
    A.nn = c.nn;
    A.nslot = P.nslot;
    A.ntiles = P.ntiles;
    A.nblocks = padded(P.ntiles);
    A.te = P.te;
    A.maxtn = P.maxtn;
    A.max_nint = P.max_nint;
    A.dt = dt;
    A.pred = pred_in;
    A.more = pred_out;
    A.first_shared = P.n_interior;
    A.cell_marker = c.cells.ready;
    A.phi = run.phi ? *run.phi : PhiRows{};
    A.dinc = c.dinc.p;
    A.xnp1 = c.formulation == APHIP_UPDATED_LAGRANGIAN ? c.xcnp1().p : nullptr;
    A.semi = c.formulation == APHIP_SEMI_LAGRANGIAN;
    A.keep = run.keep || c.mat.rate_form();  // (the rate-form materials read the previous H and P)
    A.keep_h = A.keep || c.h_pair();
    prof_begin(c, 1);
    if (c.npe == 4) {
        if (mode == 0) dispatch_kind<4, 0>(c, A);
        else if (mode == 1) dispatch_kind<4, 1>(c, A);
        else dispatch_kind<4, 2>(c, A);
    } else {
        if (mode == 0) dispatch_kind<8, 0>(c, A);
        else if (mode == 1) dispatch_kind<8, 1>(c, A);
        else dispatch_kind<8, 2>(c, A);
    }
    APHIP_HIP(hipGetLastError());
    prof_end(c, 1);
    if (P.nb > 0 && !run.park) {
        BoundArgs B{P.nb, P.n_interior, P.bstart.p, P.bpart.p, c.u.p, c.v.p, c.a.p, A.f, c.mass.p,
                    c.has_fixed ? c.fixed.p : nullptr, c.node_dt.p, P.zero.p, dt,
                    A.pred, A.more, A.keep,
                    A.X, A.dinc, A.xnp1, A.semi};
        const dim3 grid((unsigned)((P.nb + kBoundNodes - 1) / kBoundNodes)), block(3 * kBoundNodes);
        prof_begin(c, 2);
        if (mode == 0) hipLaunchKernelGGL(k_boundary<0>, grid, block, 0, c.stream, B);
        else if (mode == 1) hipLaunchKernelGGL(k_boundary<1>, grid, block, 0, c.stream, B);
        else if (ul) hipLaunchKernelGGL((k_boundary<2, true>), grid, block, 0, c.stream, B);
        else hipLaunchKernelGGL(k_boundary<2>, grid, block, 0, c.stream, B);
        APHIP_HIP(hipGetLastError());
        prof_end(c, 2);
    }
}

}  // namespace aphip
