// Internal context and helpers of the aperi-hip library (host side).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <stdexcept>
#include <algorithm>
#include <string>
#include <vector>

#include "aperi_hip.h"
#include "device_math.hpp"
#include "exodus_format.hpp"

namespace aphip {

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define APHIP_HIP(x)                                                                                  \
    do {                                                                                              \
        hipError_t e_ = (x);                                                                          \
        if (e_ != hipSuccess)                                                                         \
            throw ::aphip::Error(APHIP_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_));      \
    } while (0)

#define APHIP_REQUIRE(cond, msg)                                                                      \
    do {                                                                                              \
        if (!(cond)) throw ::aphip::Error(APHIP_ERR_INVALID, msg);                                    \
    } while (0)

// Owning device buffer.
template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    ~DevBuf() { release(); }
    void alloc(size_t count) {
        if (count == n && p) return;
        release();
        if (count == 0) return;
        if (hipMalloc(reinterpret_cast<void **>(&p), sizeof(T) * count) != hipSuccess) {
            p = nullptr;
            throw Error(APHIP_ERR_ALLOC, "hipMalloc of " + std::to_string(sizeof(T) * count) + " bytes failed");
        }
        n = count;
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void zero(hipStream_t s) {
        if (p) APHIP_HIP(hipMemsetAsync(p, 0, sizeof(T) * n, s));
    }
    void upload(const T *h, size_t count, hipStream_t s) {
        alloc(count);
        if (count) APHIP_HIP(hipMemcpyAsync(p, h, sizeof(T) * count, hipMemcpyHostToDevice, s));
    }
    void download(T *h, size_t count, hipStream_t s) const {
        if (count) APHIP_HIP(hipMemcpyAsync(h, p, sizeof(T) * count, hipMemcpyDeviceToHost, s));
    }
};

// Host memory that the device writes to.
template <typename T>
struct PinnedBuf {
    T *p = nullptr;
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf &) = delete;
    PinnedBuf &operator=(const PinnedBuf &) = delete;
    ~PinnedBuf() {
        if (p) (void)hipHostFree(p);
    }
    void alloc(size_t count) {
        if (p) return;
        if (hipHostMalloc(reinterpret_cast<void **>(&p), sizeof(T) * count, hipHostMallocDefault) != hipSuccess) {
            p = nullptr;
            throw Error(APHIP_ERR_ALLOC, "hipHostMalloc of " + std::to_string(sizeof(T) * count) + " bytes failed");
        }
    }
};

// Material constants resolved on the host (Lame form).
struct MaterialConst {
    int kind = -1;
    double density = 0.0;
    double lambda = 0.0, mu = 0.0;
    double yield_stress = 0.0, hardening = 0.0;
    double E = 0.0, nu = 0.0;
    int state_per_qp = 0;
    // neo-Hookean with damage (increment and maximum already clamped to [0, 1])
    double I1_critical = 0.0, I1_failure = 0.0, alpha = 0.0, max_damage = 0.0, max_damage_increment = 0.0;
    // power-law creep and Drucker-Prager: bulk modulus; creep rate factor A exp(-m / T), exponent
    double bulk = 0.0, creep_rate = 0.0, creep_n = 0.0;
    double dp_A1 = 0.0, dp_A2 = 0.0, dp_A2G = 0.0;
    MatParams params() const {
        return MatParams{lambda, mu,     yield_stress, hardening, I1_critical, I1_failure, alpha, max_damage,
                         max_damage_increment, bulk, creep_rate, creep_n, dp_A1, dp_A2, dp_A2G};
    }
    // reads the previous displacement gradient and stress (velocity gradient, old stress)
    bool rate_form() const { return kind == APHIP_POWER_LAW_CREEP || kind == APHIP_DRUCKER_PRAGER; }
    // state values per evaluation point
    int state_width() const {
        return kind == APHIP_J2 ? 1 : (kind == APHIP_NEO_HOOKEAN_DAMAGE || rate_form()) ? 2 : 0;
    }
};

// Checkpointed forward run for the adjoint (adjoint.hip).
struct AdjointData {
    bool ready = false;
    double dt = 0.0;
    int n_steps = 0, interval = 0;
    std::vector<DevBuf<double> *> ckpt;  // (u, v, a) at steps 0, K, 2K, ...; 9 doubles per node
    DevBuf<double> final_state;          // (u, v, a) at the last step
    DevBuf<double> seg_u;                // u of one segment's steps, K x 3 x nn
    int seg_held = -1;                   // the segment it holds (the last one after a forward run);
                                         // -1: none, or recorded with another model (model_changed)
    DevBuf<double> ub, vb, ab;           // adjoint node state
    DevBuf<double> vb1, ab1;             // on patches: the vb, ab that the next launch writes
    DevBuf<double> lam_bar, mu_bar;      // per-element parameter adjoints
    void reset() {
        for (auto *b : ckpt) delete b;
        ckpt.clear();
        final_state.release();
        seg_u.release();
        seg_held = -1;
        ub.release(); vb.release(); ab.release(); vb1.release(); ab1.release(); lam_bar.release(); mu_bar.release();
        ready = false;
    }
    ~AdjointData() { reset(); }
};

// Smoothed-cell (RKPM) data in internal numbering.
struct CellData {
    bool ready = false;
    int64_t nnz = 0;
    int64_t n_truncated = 0;
    DevBuf<int32_t> num_nbr;    // [nn]
    DevBuf<int32_t> nbr;        // [nn * 40] internal ids, -1 padded
    DevBuf<double> phi;         // [nn * 40]
    DevBuf<double> radius;      // [nn]
    DevBuf<int64_t> start;      // [ne + 1] cell entry ranges
    DevBuf<int32_t> nodes;      // [nnz] internal node ids
    DevBuf<double> dphi;        // [nnz * 3]
    DevBuf<double> volume;      // [ne]
    DevBuf<int64_t> rstart;     // [nn + 1] reverse neighbor lists: points i that list node J
    DevBuf<int32_t> rsrc;       // [nrev] i, ascending per node
    DevBuf<double> rphi;        // [nrev] phi_iJ
    int64_t ncells = 0;         // cells of the CSR above: the elements, or the subcells of nodal cells
    // nodal smoothing cells on a thex mesh: the CSR cells above are subcells, grouped into
    // one cell per active node; nodes with degrees of freedom come first (Ctx::n_dof)
    bool nodal = false;
    bool fbar = false;              // F-bar over the subcells of each cell
    int64_t n_fcells = 0;           // nodal cells
    DevBuf<int64_t> fcell_sub;      // [n_fcells + 1] subcell range of each nodal cell
    DevBuf<double> fcell_volume;    // [n_fcells]
    DevBuf<int32_t> sub_fcell;      // [ncells] F-bar: nodal cell of each subcell
    DevBuf<double> evol;            // [ne] smoothed volume of every element (nodal cells)
    std::vector<int32_t> sub_of_elem;     // [ne] subcell of each internal element (nodal cells)
    std::vector<int32_t> sub_first_elem;  // [ncells] first internal element of each subcell
    std::vector<int64_t> fcell_sub_h;     // host copy of fcell_sub
    // two-pass method: cells list the element's own nodes, u_phys and f_local can be read
    bool two_pass = false;
    // finite-element strain smoothing: Phi is the identity, the step is the element tiles' own
    bool fe = false;
    // element cells (one-pass too): the cell force acts on u_phys = Phi d and f = Phi^T f_local
    DevBuf<double> u_phys;      // [nn * 3] physical displacement of the last evaluation
    DevBuf<double> f_local;     // [nn * 3] cell force before the scatter
    // nodal cells on cell tiles (runs of consecutive cells, one wave each)
    int tile_cells = 0;             // cells per tile
    int tile_maxtn = 0;             // largest tile node set
    int tile_lpc = 8;               // lanes per cell of the tile kernel
    int64_t ntiles = 0, tile_total = 0;
    DevBuf<uint16_t> lidx;          // [nnz] entry -> index in its tile's node set
    int tile_maxsub = 0;            // most cells in one tile
    DevBuf<int64_t> t_cstart;       // [ntiles + 1] first cell of each tile
    DevBuf<int32_t> t_fstart;       // F-bar: [ntiles + 1] first nodal cell of each tile
    DevBuf<int32_t> t_nstart;       // [ntiles + 1]
    DevBuf<int32_t> t_node;         // [tile_total] internal node ids, ascending per tile
    DevBuf<int64_t> nslot_start;    // [nn + 1] slot range of each node
    DevBuf<int32_t> nslot;          // [tile_total] slots of each node, ascending tile
    DevBuf<double> slots;           // [tile_total * 3] tile force rows
    void reset() {
        ready = false;
        two_pass = false;
        fe = false;
        tile_cells = tile_maxtn = 0;
        ntiles = tile_total = 0;
        lidx.release(); t_nstart.release(); t_node.release(); nslot_start.release(); nslot.release(); slots.release();
        t_cstart.release(); t_fstart.release();
        tile_maxsub = 0;
        rstart.release(); rsrc.release(); rphi.release(); u_phys.release(); f_local.release();
        nnz = n_truncated = 0;
        ncells = n_fcells = 0;
        nodal = fbar = false;
        fcell_sub.release(); fcell_volume.release(); evol.release(); sub_fcell.release();
        sub_of_elem.clear(); sub_first_elem.clear(); fcell_sub_h.clear();
        num_nbr.release(); nbr.release(); phi.release(); radius.release(); start.release();
        nodes.release(); dphi.release(); volume.release();
    }
};

// Element-tile plan of the fused step (tile.hip), internal numbering.  The plan
// renumbers nodes: interior nodes of each tile are contiguous, shared nodes follow.
struct TilePlan {
    bool by_user = false;  // shape set by aphip_set_tiling or aphip_autotune
    bool orphans = false;  // some node belongs to no element
    bool ready = false;
    int te = 0;                       // elements per tile (= threads)
    int threads = 0;                  // workgroup size
    int64_t ntiles = 0;
    int maxtn = 0;                    // most nodes in one tile
    int max_nint = 0;                 // most interior nodes in one tile
    int64_t nb = 0;                   // shared nodes (finished by the second launch)
    int64_t n_interior = 0;           // first shared node id
    int64_t total_tile_nodes = 0;
    int64_t nslot = 0;                // shared-node slots (tile sums parked for the second launch)
    size_t lds_bytes = 0;
    int stream_grid[4] = {0, 0, 0, 0};  // persistent Tet4 step grid per material kind (0 = not sized yet)
    bool use_stream = false;           // persistent pipelined Tet4 step (APHIP_FLAG_PIPELINED)
    DevBuf<int32_t> tn_start;         // [ntiles + 1] offsets into the tile-node arrays
    DevBuf<int32_t> tile_e0;          // [ntiles + 1] first element of each tile
    DevBuf<int32_t> tn_ninterior;     // [ntiles] interior nodes come first in each tile
    DevBuf<int32_t> int_base;         // [ntiles] id of the tile's first interior node
    DevBuf<int32_t> tn_node;          // [total] global node id
    DevBuf<uint32_t> tn_csr;          // [total] (local CSR start << 16) | count
    DevBuf<int32_t> tn_bdst;          // [total] slot of a shared node's tile sum (-1 interior)
    DevBuf<uint16_t> lcsr;            // [ntiles * te * npe] local element * npe + slot
    DevBuf<uint16_t> lconn;           // [ne * npe] local node of each element slot
    DevBuf<double> bpart;             // [slots * 3] tile sums of shared nodes
    DevBuf<int32_t> bstart;           // [nb + 1] slot range of each shared node
    DevBuf<double> zero;              // [8] zeros: stands in for absent optional arrays
    DevBuf<int32_t> meta;             // [ntiles * 8] packed per-tile scalars of the pipelined step
    // the tile kernel's copies at a fixed stride per tile (rows past a tile's end repeat
    // its last row), so their addresses need no per-tile scalar
    int tpad = 0;                     // node rows per tile (= maxtn)
    DevBuf<int32_t> tnp_node;         // [ntiles * tpad]
    DevBuf<uint32_t> tnp_csr;         // [ntiles * tpad]
    DevBuf<int32_t> tnp_bdst;         // [ntiles * tpad]
    DevBuf<uint16_t> lconn_p;         // [ntiles * te * npe]
    // the Gauss Hex8 kernel's forms of the corners and the entries (k_hex_tile)
    int hx_rounds = 1;                // LDS rounds of a tile's elements
    DevBuf<uint16_t> hx_conn;         // [ntiles * te * 8] 3 x local node
    DevBuf<uint4> hx_first, hx_more;  // [ntiles * rounds * tpad] first eight entries of a row; the rest
    DevBuf<uint32_t> hx_csr;          // [ntiles * rounds * tpad] (first further batch << 16) | batches
    DevBuf<int32_t> hx_base;          // [ntiles * rounds] origin of the batches in hx_more
    DevBuf<double> hx_part;           // several rounds: [ntiles * tpad * 3] the rows' sums so far
    size_t cell_lds_bytes = 0;        // LDS of the smoothed Hex8 cell kernel
    void reset() {
        ready = false;
        te = threads = maxtn = max_nint = 0;
        ntiles = nb = n_interior = total_tile_nodes = nslot = 0;
        lds_bytes = 0;
        for (int &g : stream_grid) g = 0;
        tn_start.release(); tile_e0.release(); tn_ninterior.release(); int_base.release(); tn_node.release(); tn_csr.release();
        tn_bdst.release(); lcsr.release(); lconn.release(); bpart.release(); bstart.release();
        zero.release(); meta.release();
        tpad = 0;
        tnp_node.release(); tnp_csr.release(); tnp_bdst.release(); lconn_p.release();
        hx_conn.release(); hx_first.release(); hx_more.release(); hx_csr.release(); hx_base.release(); hx_part.release();
        hx_rounds = 1;
        cell_lds_bytes = 0;
    }
};

// Node patches of the small-mesh step (patch.hip), internal numbering.
struct PatchPlan {
    static constexpr int kRings = 4;  // most rings of a plan
    bool ready = false;
    bool tried = false;               // built, or found not to apply, for the current tile plan
    int rings = 0;                    // rings of this plan: most steps per launch
    int threads = 0;
    int64_t npatch = 0;
    int npad = 0, cpad = 0, epad = 0, entpad = 0;  // row counts of the padded lists below
    size_t lds_bytes = 0;
    DevBuf<unsigned char> lists;      // the lists below
    const int32_t *meta = nullptr, *node = nullptr, *elem = nullptr;  // [npatch * 16 / npad / epad]
    const uint32_t *csr = nullptr;                                    // [npatch * cpad]
    const uint16_t *conn = nullptr, *ent = nullptr;                   // [npatch * epad * npe / entpad]
    DevBuf<double> u, v, a;           // [nn * 3] the buffers the next launch writes
    void reset() {
        ready = tried = false;
        rings = threads = npad = cpad = epad = entpad = 0;
        npatch = 0;
        lds_bytes = 0;
        lists.release();
        meta = node = elem = nullptr;
        csr = nullptr;
        conn = ent = nullptr;
        u.release(); v.release(); a.release();
    }
};

struct Profile {
    bool enabled = false;
    std::vector<hipEvent_t> ev;   // pairs (start, stop) tagged by which
    std::vector<int> tag;
    int64_t launches[3] = {0, 0, 0};
    double ms[3] = {0, 0, 0};
};

// Specimens collected between aphip_batch_begin / aphip_batch_end (caller numbering).
struct BatchBuild {
    bool open = false;
    int etype = -1;
    int kind = -1;
    std::vector<double> X;
    std::vector<int32_t> conn;
    std::vector<int64_t> node_seg{0}, elem_seg{0};
    std::vector<aphip_material_params> params;
    std::vector<double> dt;
};

struct Ctx {
    int device = 0;
    hipStream_t stream = nullptr;

    // mesh
    int etype = -1;
    int npe = 0;
    int64_t nn = 0, ne = 0;
    int64_t n_dof = 0;                // nodes with degrees of freedom: internal ids 0 .. n_dof - 1
    std::vector<int32_t> node_perm;   // caller -> internal
    std::vector<int32_t> node_iperm;  // internal -> caller
    std::vector<int32_t> elem_perm;   // caller -> internal
    std::vector<int32_t> elem_iperm;  // internal -> caller
    std::vector<int32_t> conn_h;      // internal connectivity (host copy, for tile plans)
    std::vector<int64_t> elem_seg{0}; // element blocks (specimens); tiles never cross them
    int flags = 0;
    BatchBuild batch;
    int64_t n_specimens = 0;
    std::vector<int64_t> spec_node_seg, spec_elem_seg;  // caller-numbering ranges per specimen

    DevBuf<int32_t> d_node_iperm, d_elem_iperm;  // device copies of node_iperm / elem_iperm
    DevBuf<int32_t> d_count;             // one counter (validation of device-side field input)

    DevBuf<double> X, u, v, a, f, mass;  // node vectors AoS n x 3 (mass n)
    DevBuf<uint8_t> fixed;               // bit d set = DOF d held at zero
    DevBuf<int32_t> conn;                // AoS ne x npe, internal node ids
    DevBuf<double> H, P;                 // SoA 9 x ne
    DevBuf<double> H1, P1;               // rate-form materials: the second of the N / NP1 pairs
    DevBuf<double> state[2];             // material state (N / NP1)
    int state_np1 = 1;                   // index of the NP1 state buffer
    double rate_dt = 0.0;                // increment for force-only evaluations of rate-form materials
    int formulation = APHIP_TOTAL_LAGRANGIAN;
    DevBuf<double> xc[2];                // updated Lagrangian: current coordinates (N / NP1 with the state);
                                         // semi-Lagrangian: xc[0] is the reference configuration
    DevBuf<double> dinc;                 // the step's displacement increments (semi: accumulated)
    DevBuf<double> Href;                 // semi-Lagrangian: reference displacement gradient (SoA 9 x ne)
    int64_t semi_interval = 1, steps_done = 0;
    DevBuf<double> &xcn() { return formulation == APHIP_SEMI_LAGRANGIAN ? xc[0] : xc[1 - state_np1]; }
    DevBuf<double> &xcnp1() { return xc[state_np1]; }
    // H of the previous step is read by the rate-form materials and the updated formulation
    bool h_pair() const { return mat.rate_form() || formulation == APHIP_UPDATED_LAGRANGIAN; }
    // H and P of the current evaluation (NP1) and of the previous step (N); the pairs
    // swap with the state buffers
    DevBuf<double> &Hnp1() { return h_pair() && state_np1 == 0 ? H1 : H; }
    DevBuf<double> &Pnp1() { return mat.rate_form() && state_np1 == 0 ? P1 : P; }
    DevBuf<double> &Hn() { return state_np1 == 0 ? H : H1; }
    DevBuf<double> &Pn() { return state_np1 == 0 ? P : P1; }
    DevBuf<double> volume;               // ne
    DevBuf<int32_t> node_start;          // nn + 1
    DevBuf<int32_t> node_inc;            // ne * npe: element * npe + slot, ascending element
    DevBuf<double> partial;              // ne * npe * 3 element force partials

    MaterialConst mat;
    bool has_fields = false;             // per-element lambda / mu
    DevBuf<double> elem_lambda, elem_mu;
    DevBuf<double> elem_rho;             // per-element density (ensembles), else mat.density
    DevBuf<double> elem_E, elem_nu;      // per-element E / nu (internal order) when fields are set
    DevBuf<double> stage;                // E and nu, or their adjoints, in caller order (field.hip)
    DevBuf<double> node_dt;              // per-node time increment (ensembles), else the step argument

    // captured step sequences (aphip_set_graph)
    bool graph_enabled = false;
    hipGraphExec_t graph_exec = nullptr;
    double graph_dt = 0.0;
    int graph_parity = -1;
    int graph_steps = 0;
    void graph_reset() {
        if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
        graph_exec = nullptr;
        graph_steps = 0;
    }
    bool has_mass = false;
    bool has_fixed = false;
    bool all_fixed = false;              // every DOF of every node is fixed

    std::unique_ptr<exo::Writer> results;  // open Exodus II results file, if any

    // power method: the eigenvector of the last call, the next call's start vector; the
    // per-node max edge length, computed on the first call after the mesh is set (it
    // depends on X and the connectivity only; a node renumbering permutes it); the work
    // buffers of the allocating entry point, kept between its calls
    std::vector<const void *> big_lds;   // kernels that may take a CU's whole LDS (allow_lds)
    DevBuf<double> pm_eig;               // 3 nn, internal numbering, allocated with the mesh
    double pm_norm = 1.0;                // by which pm_eig is still to be divided
    PinnedBuf<double> pm_total;          // the norm's square, written by the device; allocated with the mesh
    DevBuf<double> pm_l;                 // nn, internal numbering, allocated with the mesh
    DevBuf<double> pm_work[8];
    bool pm_eig_valid = false;
    bool pm_l_valid = false;

    CellData cells;
    TilePlan tiles;
    PatchPlan patch;
    AdjointData adj;
    Profile prof;

    // Material, fields, mass or constraints were set: captured sequences hold their old values, and
    // recorded displacements of a segment are recomputed from its checkpoint with the new ones
    void model_changed() {
        graph_reset();
        adj.seg_held = -1;
    }

    int64_t state_count() const {
        return mat.state_width() * ne * ((etype == APHIP_HEX8 && mat.state_per_qp) ? 8 : 1);
    }
};

void set_last_error(const std::string &msg);

// ---- kernels (fem.hip) ----
void fem_element_force(Ctx &c);
void fem_predict(Ctx &c, double dt);
// semi-Lagrangian reference update: x_ref += increment, increment = 0, H_ref = H
void fem_semi_update(Ctx &c);
// mode 0: f only; 1: f and a = f/m (initial); 2: f, a, BC, v += dt/2 a (step corrector)
void fem_node_update(Ctx &c, double dt, int mode);
void fem_volumes(Ctx &c);
void fem_lumped_mass(Ctx &c, double rho);

// ---- fused tile step (tile.hip) ----
void tile_build(Ctx &c, int te, int threads);
// Reorders the internal nodes (old_of_new[i] = current id of new node i) and every
// node-indexed array of the context (capi.hip).
void renumber_nodes(Ctx &c, const std::vector<int32_t> &old_of_new);
// One tiled pass (MODE 0 force only, 1 force and a = f/m, 2 the full step).
constexpr int kMaxNbr = 40;  // neighbors of a node (include/Constants.h:15)

// Rows of Phi, by which a force evaluation takes the displacements it stages.
struct PhiRows {
    const int32_t *num, *nbr;  // neighbors of a node, kMaxNbr to a row
    const double *phi;
    int copy_lonely;  // a node without neighbors takes its own coefficient (else zero)
    int raw;          // the coefficients are predicted on the way (central difference, dt)
    double *out;      // also store Phi u, or null; a shared node's by the tile of its first slot
    const int32_t *bstart;
};
struct TileRun {
    // MODE 0: displacement read and force written when not the context's u and f (RKPM
    // element cells: physical displacement in, local force out)
    const double *u_in = nullptr;
    double *f_out = nullptr;
    // MODE 0, Tet4: the displacement staged is Phi u of the context's u
    const PhiRows *phi = nullptr;
    // MODE 0: the shared nodes' partial sums stay in their slots, no shared-node pass
    bool park = false;
    // MODE 2: u and v hold the step's predicted displacement and v1/2 (the previous step ran
    // with pred_out and the same dt in this same call); pred_out: leave the next step's there
    bool pred_in = false, pred_out = false;
    // false: H, P (and in MODE 2 f) of this evaluation are not stored: an inner step of one
    // call, whose values the next step overwrites before anything can read them, or a force
    // evaluation whose stress nobody reads (ignored for the rate-form materials)
    bool keep = true;
};
void tile_run(Ctx &c, double dt, int mode, const TileRun &run = TileRun());

// A launch of kern with more than 64 KiB of dynamic LDS needs an attribute of the kernel: set
// once per context and kernel, to all of a CU's LDS (contexts of several threads launch the same
// kernels with different sizes).
inline void allow_lds(Ctx &c, const void *kern, size_t lds) {
    constexpr size_t kCuLds = 160 * 1024;
    if (lds <= 65536 || (lds <= kCuLds && std::find(c.big_lds.begin(), c.big_lds.end(), kern) != c.big_lds.end())) return;
    APHIP_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)std::max(lds, kCuLds)));
    c.big_lds.push_back(kern);
}

// ---- small-mesh step on node patches (patch.hip) ----
// Whether this context's total-Lagrangian steps run on patches (builds the plan on first use:
// aphip_initialize or aphip_set_tiling, or the first step without them).
bool patch_eligible(Ctx &c);
int patch_steps(const Ctx &c, int left);
// `steps` steps in one launch (the state buffers' roles were swapped once by the caller);
// keep: store H, P and f of the last one; u_rec: store its displacement there as well
void patch_run(Ctx &c, double dt, int steps, bool keep, double *u_rec = nullptr);
// whether the mesh has a plan (built on first use), for passes with conditions of their own
bool patch_planned(Ctx &c);

// ---- adjoint (adjoint.hip) ----
void adjoint_forward(Ctx &c, double dt, int n_steps, int interval);
void adjoint_backward(Ctx &c, const double *ub_T, const double *vb_T, double *E_bar, double *nu_bar,
                      double *v0_bar);
void force_vjp(Ctx &c, const double *f_bar, double *u_bar, double *E_bar, double *nu_bar);
// keep: as tile_run's, for every step but the last of a call
void step_once_tiles(Ctx &c, double dt, bool keep);

// ---- RK (rk.hip) ----
// nodal_subdomains >= 0: nodal smoothing cells of a thex mesh (0: every hex a subcell,
// 1: every cell one subcell), with F-bar over the subcells when fbar
void rk_setup(Ctx &c, double scale, bool two_pass, bool fe_cells = false, int nodal_subdomains = -1,
              bool fbar = false);
// keep = false: H and P may be left unwritten (see TileRun)
// keep_local = false: an inner step, Phi u may be left unwritten
void rk_cell_force(Ctx &c, bool keep, bool raw = false, bool keep_local = true);
// more (mode 2): another step of the same call with the same dt follows; its predictor is
// taken here and fem_predict is not called for it
// raw: the step's predictor has not been taken; both passes take it (rk_takes_predictor).
// keep = false: an inner step, the local force may be left unwritten
void rk_node_update(Ctx &c, double dt, int mode, bool more, bool raw = false, bool keep = true);
bool rk_fused(const Ctx &c);
bool rk_takes_predictor(const Ctx &c);
void rk_mass(Ctx &c, double *total);

// ---- profiling helpers (capi.hip) ----
void prof_begin(Ctx &c, int which);
void prof_end(Ctx &c, int which);

// ---- power-method stable increment (power.hip) ----
void pm_max_edge(Ctx &c, double *l);
void pm_start(Ctx &c, const int32_t *caller_id, uint64_t seed, double eps, const double *l, double *v);
// u = u_in + v / norm l eps (partial: as for the pm_next that follows)
void pm_perturb(Ctx &c, const double *u_in, const double *v, double norm, const double *l, double eps, double *u,
                double *partial);
// doubles of the partial-sum buffer pm_next needs (one per block of nodes, plus their count)
int64_t pm_partials(const Ctx &c);
// v = (f - f0) / (l eps m), returns |v|_2 (partial: pm_partials(c) doubles); parked: the shared
// nodes' f stands in the tile plan's slots
double pm_next(Ctx &c, const double *f, bool parked, const double *f0, const double *l, double eps, double *v,
               double *partial);

// ---- field transfer with caller device arrays (field.hip) ----
// dst[i, :] = src[iperm[i], :] / dst[iperm[i], :] = src[i, :], w doubles per entity
void field_gather_rows(Ctx &c, int64_t n, int w, const int32_t *iperm, const double *src, double *dst);
void material_fields_from_host(Ctx &c, const double *E, const double *nu);
void parameter_gradients_to_host(Ctx &c, const double *lam_bar, const double *mu_bar, double *E_bar, double *nu_bar);
void field_scatter_rows(Ctx &c, int64_t n, int w, const int32_t *iperm, const double *src, double *dst);
// SoA 9 x ne tensor planes -> caller row-major n_elem x 9
void field_scatter_tensor(Ctx &c, const double *planes, double *dst);
// caller-numbered nodal mass into c.mass; returns how many values are not positive
int32_t field_gather_mass(Ctx &c, const double *src);

// ---- copy yardstick (probe.hip): device milliseconds per copy of nbytes ----
double bandwidth_probe(int device, int64_t nbytes, int reps);

}  // namespace aphip
