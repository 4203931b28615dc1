// Small meshes: several central-difference steps of a node patch per launch.
//
// A mesh of some thousand elements fills a few of the tile plan's workgroups and leaves most of
// the chip idle, and a step is two dependent launches (about 3.4 us of host time each, 12 us of
// device time a step on 6,174 Tet4).  Here a workgroup owns a patch of neighbouring nodes and
// recomputes what it needs from its neighbours instead of exchanging it: with K rings,
//   N_0 = the owned nodes, E_r = the elements around N_{r-1}, N_r = the nodes of E_r
// (E_1 also holds the elements the patch owns, a run of the element order; a node belongs to
// the patch of its lowest element),
// it stages N_k (k <= K), and step s = 1..k evaluates E_{k-s+1} and finishes N_{k-s} in LDS;
// after the last step it writes its owned nodes, and, of the elements it owns, the state (and H
// and P if the call ends here).  No workgroup waits for another and nothing is exchanged: u, v
// and a are read from one set of buffers and written to another, which the host exchanges.
//
// The price is the elements evaluated by several patches, so the plan is for small meshes only
// (the rule is at patch_build).  What bounds it is latency: the launch, two dependent loads,
// and per step the element's arithmetic and LDS reads (6,174 SVK Tet4, 50 steps in one call:
// 338 -> about 115 us with three meshes in turn, 595 -> 290 us alone; 49,392 Tet4, one step a
// call: 7.6 -> 5.2 us a step in turn, 14 -> 11 us alone; 8,000 neo-Hookean Hex8, 50 steps:
// 276 -> 216 us in turn, 626 -> 550 us alone).  Results are the tile path's, bit for bit: the element
// arithmetic is the same and a node's sum is grouped by the plan's tiles (partial sums of the
// node's elements in ascending order, added in ascending tile order).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <memory>
#include <thread>
#include <vector>

#include "patch.hpp"
#include "workers.hpp"

namespace aphip {

namespace {

constexpr int kNumXcd = 8;
constexpr int kRings = PatchPlan::kRings;

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

struct PatchArgs {
    const double *X;
    const double *u, *v, *a;     // state read
    double *u1, *v1, *a1, *f;    // state written (other buffers)
    double *u_rec;               // the displacement once more, or null
    const double *mass;
    const uint8_t *fixed;
    const double *zero;          // 8 zero doubles: stands in for an absent optional array
    const int32_t *meta;         // [npatch * 16] nodes per ring at 0, elements per ring at 8 (owned: at 8)
    const int32_t *node;         // [npatch * npad] node ids, ring by ring
    const uint32_t *csr;         // [npatch * cpad] (start << 16) | count of the nodes N_{K-1}
    const int32_t *elem;         // [npatch * epad] element ids, owned ones first, ring by ring
    const uint16_t *conn;        // [npatch * epad * npe] local nodes (Hex8: 3 x local node)
    const uint16_t *ent;         // [npatch * entpad] offset of the entry's force row / 3 (| kNewTile)
    double *H, *P;
    const double *state_n;
    double *state_np1;
    MatParams mat;
    const double *elem_lambda, *elem_mu;
    double gauss_a;
    double dt;
    int64_t ne, npatch, nblocks;
    int npad, cpad, epad, entpad;
    int steps, keep;
};

// LDS carve-up (bytes), sized on the host with the same function
struct PatchLds {
    double *X, *U, *V, *M, *S, *F;
    uint32_t *csr;
    uint16_t *conn, *ent;
    uint8_t *fx;
    size_t bytes;
};

__host__ __device__ __forceinline__ PatchLds carve(char *base, int npe, int npad, int cpad, int epad, int entpad) {
    PatchLds L;
    char *p = base;
    auto take = [&](size_t n) {
        char *q = p;
        p += (n + 15) & ~(size_t)15;
        return q;
    };
    L.X = reinterpret_cast<double *>(take(24 * (size_t)npad));
    L.U = reinterpret_cast<double *>(take(24 * (size_t)npad));
    L.V = reinterpret_cast<double *>(take(24 * (size_t)npad));
    L.M = reinterpret_cast<double *>(take(8 * (size_t)cpad));
    L.S = reinterpret_cast<double *>(take(8 * (size_t)epad));
    L.F = reinterpret_cast<double *>(take(npe == 4 ? 96 * (size_t)patch_stride(epad) : 8 * kHexRow * (size_t)epad));
    L.csr = reinterpret_cast<uint32_t *>(take(4 * (size_t)cpad));
    L.conn = reinterpret_cast<uint16_t *>(take(2 * (size_t)npe * epad));
    L.ent = reinterpret_cast<uint16_t *>(take(2 * (size_t)entpad));
    L.fx = reinterpret_cast<uint8_t *>(take((size_t)npad));
    L.bytes = (size_t)(p - base);
    return L;
}

template <int NPE, int KIND>
__global__ __launch_bounds__(NPE == 4 ? 1024 : 512, NPE == 4 ? 1 : 3) void k_patch(PatchArgs A) {
    extern __shared__ __align__(16) char lds_raw[];
    const int64_t b = blockIdx.x;
    const int64_t p = (b % kNumXcd) * (A.nblocks / kNumXcd) + b / kNumXcd;  // neighbours share an XCD's L2
    if (p >= A.npatch) return;
    const PatchLds L = carve(lds_raw, NPE, A.npad, A.cpad, A.epad, A.entpad);
    const int tid = threadIdx.x, nt = blockDim.x;
    // the first row of every list needs the patch id alone (the lists are padded to a fixed
    // stride, rows past the end repeat the last one), so that staging is two memory latencies
    const int32_t *node = A.node + p * A.npad;
    const int32_t *elem = A.elem + p * A.epad;
    const int32_t *meta = A.meta + 16 * p;
    const int nN = meta[A.steps], nE = meta[8 + A.steps], nC = meta[A.steps - 1], nown = meta[8];
    for (int i = tid; i < A.npad; i += nt) {
        const int64_t g = node[i];
        double x[3], u[3], v[3], a[3], vh[3], up[3];
        ld3(A.X, g, x);
        ld3(A.u, g, u);
        ld3(A.v, g, v);
        ld3(A.a, g, a);
        const uint8_t *pf = A.fixed ? A.fixed : reinterpret_cast<const uint8_t *>(A.zero);
        const unsigned f8 = pf[A.fixed ? g : 0], fx = A.fixed ? f8 : 0u;
        const double m = A.mass[g];
        cd_predict(u, v, a, fx, A.dt, vh, up);
        if (i < nN) {
            st3(L.X, i, x);
            st3(L.U, i, up);
            st3(L.V, i, vh);
            L.fx[i] = (uint8_t)fx;
            if (i < A.cpad) L.M[i] = m;
        }
    }
    for (int i = tid; i < A.cpad; i += nt) L.csr[i] = A.csr[p * A.cpad + i];
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(A.ent + p * A.entpad);
        uint4 *dst = reinterpret_cast<uint4 *>(L.ent);
        for (int i = tid; i < A.entpad / kBatch; i += nt) dst[i] = src[i];
    }
    for (int i = tid; i < A.epad; i += nt) {
#pragma unroll
        for (int k = 0; k < NPE / 4; ++k)
            reinterpret_cast<ushort4 *>(L.conn)[NPE / 4 * i + k] =
                reinterpret_cast<const ushort4 *>(A.conn + p * A.epad * NPE)[NPE / 4 * i + k];
        if constexpr (state_width<KIND>() > 0) L.S[i] = load_state<KIND>(A.state_n, elem[i]);
    }
    __syncthreads();
    const int fs = patch_stride(A.epad);
    int ne_now = nE, nn_now = nC;
    for (int s = 1;; ++s) {
        const bool last = s == A.steps;
        if constexpr (NPE == 8) {  // eight lanes per element
            for (int le = tid >> 3; le < ne_now; le += nt >> 3) {
                const uint4 c = reinterpret_cast<const uint4 *>(L.conn)[le];
                const uint32_t cn[4] = {c.x, c.y, c.z, c.w};
                MatParams m = A.mat;
                if (A.elem_lambda) {
                    const int64_t e = elem[le];
                    m.lambda = A.elem_lambda[e];
                    m.mu = A.elem_mu[e];
                }
                double H[9], P[9];
                if (hex8_lanes<KIND, false>(tid & 7, cn, L.X, L.U, L.F + kHexRow * le, m, A.gauss_a, L.S + le, L.S + le,
                                            H, P) &&
                    last && le < nown) {
                    const int64_t e = elem[le];
                    if constexpr (state_width<KIND>() > 0) A.state_np1[e] = L.S[le];
                    if (A.keep) {
#pragma unroll
                        for (int i = 0; i < 9; ++i) {
                            store_once(A.H + i * A.ne + e, H[i]);
                            store_once(A.P + i * A.ne + e, P[i]);
                        }
                    }
                }
            }
        } else {
            for (int le = tid; le < ne_now; le += nt) {
                const ushort4 c = reinterpret_cast<const ushort4 *>(L.conn)[le];
                const int lc[4] = {c.x, c.y, c.z, c.w};
                double X[NPE][3], U[NPE][3], fe[NPE][3], H[9], P[9];
#pragma unroll
                for (int k = 0; k < NPE; ++k) {
                    ld3(L.X, lc[k], X[k]);
                    ld3(L.U, lc[k], U[k]);
                }
                MatParams m = A.mat;
                if (A.elem_lambda) {
                    const int64_t e = elem[le];
                    m.lambda = A.elem_lambda[e];
                    m.mu = A.elem_mu[e];
                }
                double sn = 0.0, snp1 = 0.0, aux = 0.0;
                if constexpr (state_width<KIND>() > 0) sn = L.S[le];
                tet4_element<KIND>(X, U, m, sn, snp1, aux, H, P, fe);
#pragma unroll
                for (int k = 0; k < NPE; ++k) st3(L.F, k * fs + le, fe[k]);
                if (last) {
                    if (le < nown && (A.keep || state_width<KIND>() > 0)) {
                        const int64_t e = elem[le];
                        store_state<KIND>(A.state_np1, e, snp1, aux);
                        if (A.keep) {
#pragma unroll
                            for (int i = 0; i < 9; ++i) {
                                store_once(A.H + i * A.ne + e, H[i]);
                                store_once(A.P + i * A.ne + e, P[i]);
                            }
                        }
                    }
                } else if constexpr (state_width<KIND>() > 0) {
                    L.S[le] = snp1;
                }
            }
        }
        __syncthreads();
        // four lanes per node, one per component (the fourth idles)
        for (int t4 = tid; t4 < 4 * nn_now; t4 += nt) {
            const int ln = t4 >> 2, d = t4 & 3;
            if (d == 3) continue;
            const double f = patch_sum(L.F + d, L.ent, L.csr[ln]);
            const bool fx = L.fx[ln] & (1u << d);
            double a1, v1;
            const double u1 = L.U[3 * ln + d];
            cd_correct1(f, L.M[ln], fx, A.dt, L.V[3 * ln + d], a1, v1);
            if (last) {
                const int64_t g = 3 * (int64_t)node[ln] + d;
                A.u1[g] = u1;
                if (A.u_rec) A.u_rec[g] = u1;
                A.v1[g] = v1;
                A.a1[g] = a1;
                if (A.keep) A.f[g] = f;
            } else {
                cd_predict1(u1, v1, a1, fx, A.dt, L.V[3 * ln + d], L.U[3 * ln + d]);
            }
        }
        if (last) return;
        __syncthreads();
        ne_now = meta[8 + A.steps - s];
        nn_now = meta[A.steps - s - 1];
    }
}

static_assert(state_width<APHIP_J2>() == 1, "patches keep one state value per element");

template <int NPE>
void launch(Ctx &c, const PatchArgs &A) {
    const PatchPlan &P = c.patch;
    auto go = [&](auto kern) {
        allow_lds(c, (const void *)kern, P.lds_bytes);
        hipLaunchKernelGGL(kern, dim3((unsigned)A.nblocks), dim3(P.threads), P.lds_bytes, c.stream, A);
        APHIP_HIP(hipGetLastError());
    };
    switch (c.mat.kind) {
        case APHIP_LINEAR_ELASTIC: go(k_patch<NPE, APHIP_LINEAR_ELASTIC>); break;
        case APHIP_NEO_HOOKEAN: go(k_patch<NPE, APHIP_NEO_HOOKEAN>); break;
        case APHIP_J2: go(k_patch<NPE, APHIP_J2>); break;
        case APHIP_SVK: go(k_patch<NPE, APHIP_SVK>); break;
        default: throw Error(APHIP_ERR_INVALID, "material without a patch kernel");
    }
}

}  // namespace

// Steps that the next launch of a call with `left` steps to go takes.  A material with state
// ends a call with a launch of one step: the N buffer must hold the state before the last step.
int patch_steps(const Ctx &c, int left) {
    const int k = std::min(left, c.patch.rings);
    return c.mat.state_width() > 0 && left > 1 && k == left ? left - 1 : k;
}

// Plan of K rings and runs of `target` owned elements for the current tile plan and numbering;
// false when a patch's rows do not fit a CU's LDS (or the lists' 16-bit fields).
static bool patch_plan(Ctx &c, int K, int64_t target) {
    PatchPlan &P = c.patch;
    const int64_t nn = c.nn, ne = c.ne;
    const int npe = c.npe, sh = npe == 4 ? 2 : 3;
    const std::vector<int32_t> &conn = c.conn_h;
    // node -> (element, slot), ascending
    std::vector<int32_t> start(nn + 1, 0), inc((size_t)ne * npe);
    for (int64_t t = 0; t < ne * npe; ++t) start[conn[t] + 1]++;
    for (int64_t i = 0; i < nn; ++i) start[i + 1] += start[i];
    {
        std::vector<int32_t> fill(start.begin(), start.end() - 1);
        for (int64_t t = 0; t < ne * npe; ++t) inc[fill[conn[t]]++] = (int32_t)t;
    }
    // patch of every node: that of its lowest element; nodes of no element go round
    const int64_t np = (ne + target - 1) / target;
    std::vector<std::vector<int32_t>> own(np);
    for (int64_t i = 0; i < nn; ++i)
        own[start[i] < start[i + 1] ? (inc[start[i]] >> sh) / target : i % np].push_back((int32_t)i);
    // tile of every element (the grouping of the sums)
    const int te = c.tiles.te;
    struct Patch {
        std::vector<int32_t> nodes, elems;
        int nn[kRings + 1] = {0}, ne[kRings + 1] = {0};
        std::vector<uint32_t> csr;
        std::vector<uint16_t> conn, ent;
    };
    std::vector<Patch> pt(np);
    std::atomic<bool> fits{true};
    std::atomic<int64_t> next{0};
    auto work = [&] {
        std::vector<int32_t> nloc(nn, -1), eloc(ne, -1);
        for (int64_t p; (p = next++) < np;) {
            Patch &q = pt[p];
            q.nodes = own[p];
            for (int64_t e = p * target; e < std::min(ne, (p + 1) * target); ++e) {
                eloc[e] = 0;
                q.elems.push_back((int32_t)e);
            }
            q.ne[0] = (int)q.elems.size();
            q.elems.reserve(4 * target);
            q.nodes.reserve(4 * target);
            q.conn.reserve(4 * npe * target);
            q.ent.reserve(2 * npe * target);
            for (size_t i = 0; i < q.nodes.size(); ++i) nloc[q.nodes[i]] = (int32_t)i;
            q.nn[0] = (int)q.nodes.size();
            size_t n_from = 0;
            for (int r = 1; r <= K; ++r) {
                const size_t n_to = q.nodes.size(), e_from = q.elems.size(), e_new = r == 1 ? 0 : e_from;
                for (size_t i = n_from; i < n_to; ++i)
                    for (int32_t t = start[q.nodes[i]]; t < start[q.nodes[i] + 1]; ++t) {
                        const int32_t e = inc[t] >> sh;
                        if (eloc[e] < 0) {
                            eloc[e] = 0;
                            q.elems.push_back(e);
                        }
                    }
                std::sort(q.elems.begin() + e_from, q.elems.end());
                for (size_t i = e_new; i < q.elems.size(); ++i) {  // ring 1: the owned elements too
                    eloc[q.elems[i]] = (int32_t)i;
                    for (int k = 0; k < npe; ++k) {
                        const int32_t n = conn[(int64_t)q.elems[i] * npe + k];
                        if (nloc[n] < 0) {
                            nloc[n] = 0;
                            q.nodes.push_back(n);
                        }
                    }
                }
                std::sort(q.nodes.begin() + n_to, q.nodes.end());
                for (size_t i = n_to; i < q.nodes.size(); ++i) nloc[q.nodes[i]] = (int32_t)i;
                n_from = n_to;
                q.nn[r] = (int)q.nodes.size();
                q.ne[r] = (int)q.elems.size();
            }
            for (int i = 0; i < q.nn[K - 1]; ++i) {
                const size_t s0 = q.ent.size();
                int32_t tile = -1;
                for (int32_t t = start[q.nodes[i]]; t < start[q.nodes[i] + 1]; ++t) {
                    const int32_t e = inc[t] >> sh, k = inc[t] & (npe - 1);
                    const bool fresh = tile >= 0 && e / te != tile;
                    tile = e / te;
                    // (local element and slot; the force row once the row stride is known)
                    q.ent.push_back((uint16_t)(eloc[e] * npe + k) | (fresh ? kNewTile : 0));
                }
                const size_t cnt = q.ent.size() - s0;
                if (s0 / kBatch > 0xffff || cnt > 0xffff) fits = false;
                q.csr.push_back((uint32_t)((s0 / kBatch) << 16) | (uint32_t)cnt);
                while (q.ent.size() % kBatch) q.ent.push_back(0);
            }
            for (int32_t e : q.elems)
                for (int k = 0; k < npe; ++k) q.conn.push_back((uint16_t)nloc[conn[(int64_t)e * npe + k]]);
            if (force_row(npe, (int)q.elems.size(), (int)q.elems.size(), npe) > 0x7fff || 3 * q.nodes.size() > 0xffff)
                fits = false;
            for (int32_t n : q.nodes) nloc[n] = -1;
            for (int32_t e : q.elems) eloc[e] = -1;
        }
    };
    auto parallel = [&](int most, auto &fn) {  // (a thread costs some 20 us)
        next = 0;
        run_workers((int)std::min<int64_t>({most, (int64_t)std::thread::hardware_concurrency(), np / 6}), fn);
    };
    parallel(16, work);
    if (!fits) return false;
    size_t npad = 1, cpad = 1, epad = 1, entpad = kBatch;
    for (const Patch &q : pt) {
        npad = std::max(npad, q.nodes.size());
        cpad = std::max(cpad, q.csr.size());
        epad = std::max(epad, q.elems.size());
        entpad = std::max(entpad, q.ent.size());
    }
    if (force_row(npe, (int)epad, (int)epad, npe) > 0x7fff) return false;
    const size_t lds = carve(nullptr, npe, (int)npad, (int)cpad, (int)epad, (int)entpad).bytes;
    if (lds > 160 * 1024) return false;
    // the six lists (each on a 16-byte boundary) in one allocation and one copy
    size_t total = 0;
    auto put = [&](size_t bytes) {
        const size_t at = total;
        total += (bytes + 15) & ~(size_t)15;
        return at;
    };
    const size_t o_meta = put(64 * np), o_node = put(4 * np * npad), o_csr = put(4 * np * cpad),
                 o_elem = put(4 * np * epad), o_conn = put(2 * np * epad * npe), o_ent = put(2 * np * entpad);
    std::unique_ptr<unsigned char[]> bytes(new unsigned char[total]);
    auto pack = [&] {
        for (int64_t p; (p = next++) < np;) {
            const Patch &q = pt[p];
            int32_t *meta = reinterpret_cast<int32_t *>(bytes.get() + o_meta) + 16 * p;
            int32_t *node = reinterpret_cast<int32_t *>(bytes.get() + o_node) + p * npad;
            uint32_t *csr = reinterpret_cast<uint32_t *>(bytes.get() + o_csr) + p * cpad;
            int32_t *elem = reinterpret_cast<int32_t *>(bytes.get() + o_elem) + p * epad;
            uint16_t *lconn = reinterpret_cast<uint16_t *>(bytes.get() + o_conn) + p * epad * npe;
            uint16_t *ent = reinterpret_cast<uint16_t *>(bytes.get() + o_ent) + p * entpad;
            std::fill(meta, meta + 16, 0);
            for (int r = 0; r <= K; ++r) {
                meta[r] = q.nn[r];
                meta[8 + r] = q.ne[r];
            }
            for (size_t i = 0; i < npad; ++i) node[i] = q.nodes[std::min(i, q.nodes.size() - 1)];
            for (size_t i = 0; i < cpad; ++i) csr[i] = i < q.csr.size() ? q.csr[i] : 0;
            for (size_t i = 0; i < entpad; ++i) {
                const int le = i < q.ent.size() ? q.ent[i] & ~kNewTile : 0;
                ent[i] = i < q.ent.size() ? (uint16_t)force_row(npe, (int)epad, le >> sh, le & (npe - 1)) | (q.ent[i] & kNewTile) : 0;
            }
            for (size_t i = 0; i < epad; ++i) {
                const size_t j = std::min(i, q.elems.size() - 1);
                elem[i] = q.elems[j];
                for (int k = 0; k < npe; ++k) lconn[i * npe + k] = (uint16_t)((npe == 8 ? 3 : 1) * q.conn[j * npe + k]);
            }
        }
    };
    parallel(4, pack);
    P.u.alloc(3 * nn);
    P.v.alloc(3 * nn);
    P.a.alloc(3 * nn);
    P.lists.upload(bytes.get(), total, c.stream);
    P.meta = reinterpret_cast<const int32_t *>(P.lists.p + o_meta);
    P.node = reinterpret_cast<const int32_t *>(P.lists.p + o_node);
    P.csr = reinterpret_cast<const uint32_t *>(P.lists.p + o_csr);
    P.elem = reinterpret_cast<const int32_t *>(P.lists.p + o_elem);
    P.conn = reinterpret_cast<const uint16_t *>(P.lists.p + o_conn);
    P.ent = reinterpret_cast<const uint16_t *>(P.lists.p + o_ent);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    P.rings = K;
    P.npatch = np;
    P.npad = (int)npad;
    P.cpad = (int)cpad;
    P.epad = (int)epad;
    P.entpad = (int)entpad;
    P.lds_bytes = lds;
    // Tet4: one element per thread where 1024 reach; Hex8 (eight lanes per element) 256, so that
    // several patches share a CU (8,000 Hex8, 50 steps: 216 us in turn, 312 us with 512)
    P.threads = npe == 4 ? std::max(128, std::min(1024, (int)(epad + 63) / 64 * 64)) : 256;
    P.ready = true;
    return true;
}

// Plan for the current tile plan; none when the mesh is too large for it.
static void patch_build(Ctx &c) {
    PatchPlan &P = c.patch;
    P.tried = true;
    const int64_t ne = c.ne;
    const int npe = c.npe;
    // The lines, from calls of 20 steps on n^3 x 6 Tet4 lattices (neo-Hookean; us a call, three
    // meshes in turn / one alone; T the tile path, k x s: k rings, s owned elements):
    //     750 T 71/177  2x64 59/149          24,576 T 119/275  1x128 70/174  2x128 88/169
    //   3,072 T 169/294 2x64 46/137  1x64 95/203   48,000 T 168/280  1x256 114/211  1x128 119/229
    //  10,368 T 120/264 2x128 54/165 2x64 69/146   93,750 T 167/288  1x256 209/344
    // n^3 Hex8 (the tile path costs 163-175 in turn from launches alone, on this host):
    //     125 T 96/192  2x8 59/171  1x16 94/181    8,000 T 175/286  1x32 103/248  1x64 138/336
    //   1,000 T 172/265 1x16 93/178 2x8 74/216    17,576 T 168/337  1x32 153/322
    //   2,744 T 175/267 1x16 97/181 1x32 92/211   32,768 T 163/292  1x64 231/340
    // 64 or 128 owned Tet4 where two rings fit (both measured again; a second ring of 128 that does not
    // fit leaves one):
    //     4,374 2x64 60/141 2x128 72/160     7,986 2x64 60/142 2x128 96/174 (one ring)
    //     6,000 2x64 60/143 2x128 60/156    10,368 2x64 66/140 2x128 59/154
    // A second ring pays while the chip idles (it evaluates some four times the elements), the
    // whole scheme until the elements evaluated twice cost what a launch does.  That line, in us a
    // step against the tile path as it is now (the T above are of its 1024-element tiles):
    //   48,000 Tet4 T 6.2/13.1 patches 5.5/9.2    63,888 Tet4 T 6.1/13.0 patches 7.1/9.3
    //   13,824 Hex8 T 6.5/13.1 patches 6.2/12.7   19,683 Hex8 T 6.5/13.2 patches 8.4/15.6
    if (ne == 0 || ne > (npe == 4 ? 54000 : 15000) || c.tiles.threads != c.tiles.te || c.elem_seg.size() != 2) return;
    const int K = ne <= (npe == 4 ? 16000 : 500) ? 2 : 1;
    const int64_t target = npe == 4 ? (ne <= 9000 ? 64 : ne <= 32000 ? 128 : 256) : (ne <= 500 ? 8 : ne <= 4000 ? 16 : 32);
    // without the memory for a plan the steps stay on the tiles
    auto none = [&] {
        (void)hipGetLastError();
        P.reset();
        P.tried = true;
    };
    try {
        for (int k = K; k >= 1 && !patch_plan(c, k, target); --k) {  // (some mesh shapes have larger second rings)
        }
    } catch (const Error &e) {
        if (e.code != APHIP_ERR_ALLOC) throw;
        none();
    } catch (const std::bad_alloc &) {
        none();
    }
}

bool patch_planned(Ctx &c) {
    if (c.tiles.ready && !c.patch.tried) patch_build(c);
    return c.patch.ready;
}

bool patch_eligible(Ctx &c) {
    return !c.node_dt.p && !c.tiles.use_stream && !c.mat.state_per_qp &&
           (c.mat.kind == APHIP_LINEAR_ELASTIC || c.mat.kind == APHIP_NEO_HOOKEAN || c.mat.kind == APHIP_J2 ||
            c.mat.kind == APHIP_SVK) &&
           patch_planned(c);  // (last: builds the plan, 0.6 to 2 ms of host time)
}

void patch_run(Ctx &c, double dt, int steps, bool keep, double *u_rec) {
    PatchPlan &P = c.patch;
    APHIP_REQUIRE(P.ready && steps >= 1 && steps <= P.rings, "patch plan does not cover these steps");
    PatchArgs A;
    A.X = c.X.p;
    A.u = c.u.p;
    A.v = c.v.p;
    A.a = c.a.p;
    A.u1 = P.u.p;
    A.v1 = P.v.p;
    A.a1 = P.a.p;
    A.u_rec = u_rec;
    A.f = c.f.p;
    A.mass = c.mass.p;
    A.fixed = c.has_fixed ? c.fixed.p : nullptr;
    A.zero = c.tiles.zero.p;
    A.meta = P.meta;
    A.node = P.node;
    A.csr = P.csr;
    A.elem = P.elem;
    A.conn = P.conn;
    A.ent = P.ent;
    A.H = c.H.p;
    A.P = c.P.p;
    A.state_n = c.state[1 - c.state_np1].p;
    A.state_np1 = c.state[c.state_np1].p;
    A.mat = c.mat.params();
    A.elem_lambda = c.has_fields ? c.elem_lambda.p : nullptr;
    A.elem_mu = c.has_fields ? c.elem_mu.p : nullptr;
    A.gauss_a = 1.0 / std::sqrt(3.0);
    A.dt = dt;
    A.ne = c.ne;
    A.npatch = P.npatch;
    A.nblocks = ((P.npatch + kNumXcd - 1) / kNumXcd) * kNumXcd;
    A.npad = P.npad;
    A.cpad = P.cpad;
    A.epad = P.epad;
    A.entpad = P.entpad;
    A.steps = steps;
    A.keep = keep;
    if (c.npe == 4) launch<4>(c, A);
    else launch<8>(c, A);
    std::swap(c.u.p, P.u.p);
    std::swap(c.v.p, P.v.p);
    std::swap(c.a.p, P.a.p);
}

}  // namespace aphip
