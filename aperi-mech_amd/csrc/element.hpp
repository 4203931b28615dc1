// Per-element force math shared by the element kernels (fem.hip, tile.hip).
//
//   Tet4 1-point: B from the constant derivatives, w = detJ / 6
//     (include/ShapeFunctionsFunctorTet4.h:27-35, include/QuadratureGaussian.h:17-38,
//      include/ElementTetrahedron4.h:125-127)
//   Hex8 2x2x2: Gauss points in the order of include/ElementHexahedron8.h:107-115, w = detJ;
//     per point H = (u^T dN) J^-1 and f_k -= dN_k (w J^-1 P^T), i.e. -B P^T w without
//     forming B (include/ComputeInternalForceGaussian.h:85-124)
//   Stored H / P are those of the last Gauss point (ComputeInternalForceGaussian.h:89, :99-107).
#pragma once

#include "device_math.hpp"

namespace aphip {

// Central-difference node updates shared by every kernel that finishes a node, so
// a node finished in the tile kernel and one finished in the boundary pass see
// bit-identical arithmetic.
//   predictor  v1/2 = v + dt/2 a, velocity BC, u1 = u + dt v1/2  (ExplicitTimeIntegrator.h:116-126, :348-357)
//   corrector  a = f/m, acceleration BC, v = v1/2 + dt/2 a       (ExplicitTimeIntegrator.h:267-276, :308-318)
APHIP_DEV void cd_predict1(double u, double v, double a, bool fixed, double dt, double &vh, double &u1) {
#pragma clang fp contract(off)
    double w = __fma_rn(0.5 * dt, a, v);
    if (fixed) w = 0.0;
    vh = w;
    u1 = __fma_rn(dt, w, u);
}

APHIP_DEV void cd_correct1(double f, double m, bool fixed, double dt, double vh, double &a1, double &v1) {
#pragma clang fp contract(off)
    double acc = f / m;
    if (fixed) acc = 0.0;
    a1 = acc;
    v1 = __fma_rn(0.5 * dt, acc, vh);
}

APHIP_DEV void cd_predict(const double *u, const double *v, const double *a, unsigned fixed, double dt, double *vh,
                          double *u1) {
#pragma unroll
    for (int d = 0; d < 3; ++d) cd_predict1(u[d], v[d], a[d], fixed & (1u << d), dt, vh[d], u1[d]);
}

APHIP_DEV void cd_correct(const double *f, double m, unsigned fixed, double dt, const double *vh, double *a1,
                          double *v1) {
#pragma unroll
    for (int d = 0; d < 3; ++d) cd_correct1(f[d], m, fixed & (1u << d), dt, vh[d], a1[d], v1[d]);
}

// H, P and the state are written once per step and not read again in it: a
// non-temporal store keeps that stream (144 B per element) from evicting the node
// data that neighbouring tiles re-read from L2.
APHIP_DEV void store_once(double *p, double v) { __builtin_nontemporal_store(v, p); }

// Tet4: fe[k][j] = -(B_k . P_j) w; sn, snp1, aux, r as for stress<KIND>.  UL: X are the
// start-of-step coordinates, U the step's displacement increments, r->Hn the element's
// previous displacement gradient (updated Lagrangian).
template <int KIND, bool UL = false>
APHIP_DEV void tet4_element(const double (&X)[4][3], const double (&U)[4][3], const MatParams &m, double sn,
                            double &snp1, double &aux, double *H, double *P, double (&fe)[4][3],
                            const RateIn *r = nullptr, double sn2 = 0.0) {
#pragma clang fp contract(off)
    double J[9], Ji[9];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        J[3 * i + 0] = X[1][i] - X[0][i];
        J[3 * i + 1] = X[2][i] - X[0][i];
        J[3 * i + 2] = X[3][i] - X[0][i];
    }
    const double det = inverse3(J, Ji);
    const double w = (1.0 / 6.0) * det;
    double B[4][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        B[1][j] = Ji[j];
        B[2][j] = Ji[3 + j];
        B[3][j] = Ji[6 + j];
        B[0][j] = ((-Ji[j]) - Ji[3 + j]) - Ji[6 + j];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            H[3 * i + j] = dot4(U[0][i], B[0][j], U[1][i], B[1][j], U[2][i], B[2][j], U[3][i], B[3][j]);
    if constexpr (UL) ul_gradient(H, r->Hn);
    stress<KIND>(H, m, sn, snp1, aux, P, r, sn2);
    double Pf[9];
    if constexpr (UL) {
        ul_force_stress(P, r->Hn, Pf);
    } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) Pf[i] = P[i];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            fe[k][j] = -(dot3(B[k][0], Pf[3 * j], B[k][1], Pf[3 * j + 1], B[k][2], Pf[3 * j + 2]) * w);
}

APHIP_DEV void hex8_sign(int k, int &s0, int &s1, int &s2) {
    s0 = (k == 1 || k == 2 || k == 5 || k == 6) ? 1 : -1;
    s1 = (k == 2 || k == 3 || k == 6 || k == 7) ? 1 : -1;
    s2 = (k >= 4) ? 1 : -1;
}

// Hex8 2x2x2 in modal form.  A trilinear field is a combination of the eight
// corner modes 1, s0, s1, s2, s0 s1, s0 s2, s1 s2, s0 s1 s2 (s_d = the corner's sign
// along parametric axis d); its Walsh-Hadamard transform over the corners gives the
// mode coefficients, and at a Gauss point p = (p0, p1, p2)
//   8 dX/dxi0 = M[s0] + p1 M[s0s1] + p2 M[s0s2] + p1 p2 M[s0s1s2]   (and cyclically),
// which replaces the 8-corner sums of J and grad u by 3 multiply-adds per entry.
// The nodal force f_k = -sum_q dN_k(q) Q_q is accumulated in the same seven modes
// and returned to the corners by one inverse transform.  The 1/8 of the shape function
// derivatives is carried as exact powers of two (J and grad u scaled by 8, the force by
// 1/512), and w J^-1 = det J J^-1 is the adjugate.
// Gauss points in the order of include/ElementHexahedron8.h:107-115, w = detJ;
// stored H / P are those of the last point (ComputeInternalForceGaussian.h:89, :99-107).

// corner k (hex8_sign order) -> binary index b0 + 2 b1 + 4 b2 with b_d = (s_d + 1) / 2
APHIP_DEV constexpr int hex8_bin(int k) { return k == 2 ? 3 : k == 3 ? 2 : k == 6 ? 7 : k == 7 ? 6 : k; }

// w[S] = sum over corners of prod_{d in S} s_d * v; S a bitmask of axes (w[0] unused)
APHIP_DEV void hex8_modes(const double (&v)[8], double (&w)[8]) {
#pragma clang fp contract(off)
#pragma unroll
    for (int k = 0; k < 8; ++k) w[hex8_bin(k)] = v[k];
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (!(i & h)) {
                const double a = w[i], b = w[i | h];
                w[i] = b + a;
                w[i | h] = b - a;
            }
}

// v_k = sum_S prod_{d in S} s_d(k) r[S], with r[0] = 0
APHIP_DEV void hex8_corners(const double (&r)[8], double (&v)[8]) {
#pragma clang fp contract(off)
    double w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = r[i];
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (!(i & h)) {
                const double a = w[i], b = w[i | h];
                w[i] = a - b;
                w[i | h] = a + b;
            }
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = w[hex8_bin(k)];
}

// 8 d(field_i)/dxi at Gauss point (p0, p1, p2); p01 = p0 p1 etc.
APHIP_DEV void hex8_grad(const double (&w)[8], double p0, double p1, double p2, double p01, double p02, double p12,
                         double (&g)[3]) {
#pragma clang fp contract(off)
    g[0] = __fma_rn(p12, w[7], __fma_rn(p2, w[5], __fma_rn(p1, w[3], w[1])));
    g[1] = __fma_rn(p02, w[7], __fma_rn(p2, w[6], __fma_rn(p0, w[3], w[2])));
    g[2] = __fma_rn(p01, w[7], __fma_rn(p1, w[6], __fma_rn(p0, w[5], w[4])));
}

// state_n / state_np1 point at the element's state slot(s) (per_qp: 8 slots), each
// state_width<KIND>() values wide.  r: the element's H_n, P_n (those of its last Gauss
// point in the previous step, like the reference's element fields) for every point.
template <int KIND, bool PER_QP, bool UL = false>
APHIP_DEV void hex8_element(const double (&X)[8][3], const double (&U)[8][3], const MatParams &m, double ga,
                            const double *state_n, double *state_np1, double *H, double *P, double (&fe)[8][3],
                            const RateIn *r = nullptr) {
#pragma clang fp contract(off)
    double XM[3][8], UM[3][8];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        double vx[8], vu[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            vx[k] = X[k][i];
            vu[k] = U[k][i];
        }
        hex8_modes(vx, XM[i]);
        hex8_modes(vu, UM[i]);
    }
    // force modes r[j][S] (S = 1..7)
    double R[3][8];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int S = 0; S < 8; ++S) R[j][S] = 0.0;
    const double ga2 = ga * ga;
    double sn = 0.0, sn2 = 0.0;
    if constexpr (!PER_QP) {
        sn = load_state<KIND>(state_n, 0);
        sn2 = load_state2<KIND>(state_n, 0);
    }
#pragma unroll 1
    for (int q = 0; q < 8; ++q) {
        int sq0, sq1, sq2;
        hex8_sign(q, sq0, sq1, sq2);
        const double p0 = sq0 * ga, p1 = sq1 * ga, p2 = sq2 * ga;
        const double p01 = (sq0 * sq1) * ga2, p02 = (sq0 * sq2) * ga2, p12 = (sq1 * sq2) * ga2;
        double J[9], G[9];  // 8 J, 8 grad u (row i = component, column = parametric axis)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            double gx[3], gu[3];
            hex8_grad(XM[i], p0, p1, p2, p01, p02, p12, gx);
            hex8_grad(UM[i], p0, p1, p2, p01, p02, p12, gu);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                J[3 * i + d] = gx[d];
                G[3 * i + d] = gu[d];
            }
        }
        double Ad[9];  // adj(8 J): w J^-1 up to exact powers of two
        const double id = 1.0 / adjugate3(J, Ad);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                H[3 * i + j] = dot3(G[3 * i], Ad[j], G[3 * i + 1], Ad[3 + j], G[3 * i + 2], Ad[6 + j]) * id;
        double snp1 = 0.0, aux = 0.0;
        if constexpr (PER_QP) {
            sn = load_state<KIND>(state_n, q);
            sn2 = load_state2<KIND>(state_n, q);
        }
        if constexpr (UL) ul_gradient(H, r->Hn);
        stress<KIND>(H, m, sn, snp1, aux, P, r, sn2);
        if constexpr (PER_QP) store_state<KIND>(state_np1, q, snp1, aux);
        else if (q == 7) store_state<KIND>(state_np1, 0, snp1, aux);
        double Pf[9];
        if constexpr (UL) {
            ul_force_stress(P, r->Hn, Pf);
        } else {
#pragma unroll
            for (int i = 0; i < 9; ++i) Pf[i] = P[i];
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            // Q[n] = (w J^-1 P^T)[n][j] up to exact powers of two: the force of axis n's derivative
            double Q[3];
#pragma unroll
            for (int n = 0; n < 3; ++n) Q[n] = dot3(Ad[3 * n], Pf[3 * j], Ad[3 * n + 1], Pf[3 * j + 1], Ad[3 * n + 2], Pf[3 * j + 2]);
            R[j][1] += Q[0];
            R[j][2] += Q[1];
            R[j][4] += Q[2];
            R[j][3] = __fma_rn(p1, Q[0], __fma_rn(p0, Q[1], R[j][3]));
            R[j][5] = __fma_rn(p2, Q[0], __fma_rn(p0, Q[2], R[j][5]));
            R[j][6] = __fma_rn(p2, Q[1], __fma_rn(p1, Q[2], R[j][6]));
            R[j][7] = __fma_rn(p12, Q[0], __fma_rn(p02, Q[1], __fma_rn(p01, Q[2], R[j][7])));
        }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        double v[8];
        hex8_corners(R[j], v);
#pragma unroll
        for (int k = 0; k < 8; ++k) fe[k][j] = v[k] * (-1.0 / 512.0);  // (exact: -w det^-1 of the scaled J)
    }
}

// Hex8 with one lane per Gauss point, in the modal form of hex8_element.  Eight lanes share
// an element: one field's corner values per lane (six of the eight) go through the transform
// and its seven modes into the element's LDS row, every lane evaluates its Gauss point from
// the row, and the three vectors Q_n of the force are summed over the points, combined into
// the modes and returned to the corners by transforms across the lanes (DPP moves, no LDS).
//
// A lane's label x = (x0, x1, x2) says which point (axis a at + if x_a), mode (the axes with
// x_a) and corner (s_a = + if x_a) it holds.  Labels are chosen so that the partner along every
// axis is one DPP move away: axis 0 lane ^ 1, axis 1 lane ^ 2, axis 2 lane ^ 7 (the mirror in a
// half row; xor 4 is not a DPP pattern), i.e. x2 = bit 2, x1 = bit 1 ^ x2, x0 = bit 0 ^ x2.
constexpr int kHexRow = 42;  // doubles of an element's LDS row: 6 fields x 7 modes, then 8 x 3 forces

template <int CTRL>
APHIP_DEV double dpp_move(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// the value of the partner lane along axis a
template <int AXIS>
APHIP_DEV double hex8_partner(double v) {
    constexpr int ctrl = AXIS == 0 ? 0xb1 /* quad_perm 1,0,3,2 */ : AXIS == 1 ? 0x4e /* 2,3,0,1 */ : 0x141 /* half-row mirror */;
    return dpp_move<ctrl>(v);
}

APHIP_DEV int hex8_lane_label(int lane) {
    const int x2 = (lane >> 2) & 1, x1 = ((lane >> 1) & 1) ^ x2, x0 = (lane & 1) ^ x2;
    return x0 | (x1 << 1) | (x2 << 2);
}

// One field's modes to the seven doubles of out (src: the field's component of node 0).
APHIP_DEV void hex8_field_modes(const uint32_t (&cn)[4], const double *src, double ga, double *out) {
#pragma clang fp contract(off)
    double v[8], w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = src[k & 1 ? cn[k >> 1] >> 16 : cn[k >> 1] & 0xffffu];
    hex8_modes(v, w);
    // a mode of |S| axes is only ever used times ga^(|S| - 1) and signs
    w[3] *= ga;
    w[5] *= ga;
    w[6] *= ga;
    w[7] *= ga * ga;
#pragma unroll
    for (int S = 1; S < 8; ++S) out[S - 1] = w[S];
}

// The lanes' nodal vectors of a stress-like P: scale sum over the points and axes n of the
// derivative along n of a corner's function times (Ad P^T)_n, to out of every lane's corner.
APHIP_DEV void hex8_to_corners(int x, bool b0, bool b1, bool b2, double s0, double s1, double s2, double ga, double scale,
                               const double *Ad, const double *P, double *out) {
#pragma clang fp contract(off)
    // W_nj[x] = sum over the points of sign_(x without n)(point) Q_nj by butterflies: lane x keeps
    // pattern x of the other axes, along axis n both partners take the plain sum
    double W[3][3];
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double v = dot3(Ad[3 * n], P[3 * j], Ad[3 * n + 1], P[3 * j + 1], Ad[3 * n + 2], P[3 * j + 2]);
            v = n == 0 ? v + hex8_partner<0>(v) : __fma_rn(s0, hex8_partner<0>(v), v);
            v = n == 1 ? v + hex8_partner<1>(v) : __fma_rn(s1, hex8_partner<1>(v), v);
            W[n][j] = n == 2 ? v + hex8_partner<2>(v) : __fma_rn(s2, hex8_partner<2>(v), v);
        }
    // mode x: R_xj = c sum_{n in x} W_nj, c = ga^(|x| - 1); then to the corners
    const int nx = (x & 1) + ((x >> 1) & 1) + (x >> 2);
    const double c = (nx == 3 ? ga * ga : nx == 2 ? ga : 1.0) * scale;
    const double c0 = b0 ? c : 0.0, c1 = b1 ? c : 0.0, c2 = b2 ? c : 0.0;
    double f[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        double v = __fma_rn(c2, W[2][j], __fma_rn(c1, W[1][j], c0 * W[0][j]));
        v = __fma_rn(-s0, hex8_partner<0>(v), v);
        v = __fma_rn(-s1, hex8_partner<1>(v), v);
        f[j] = __fma_rn(-s2, hex8_partner<2>(v), v);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) out[j] = f[j];
}

// lane: 0..7 within the element (all eight active); cn: the offsets (3 x local node) of corners
// 2 i and 2 i + 1 in cn[i]; sX, sU: 3 doubles per local node; row: the element's kHexRow doubles, on
// return the corner forces (corner k at 3 k).  H, P and the state of the last point are valid
// in the lane for which the function returns true; with PER_QP every lane stores its state.
// LEAN: the lane's signs are derived again after the stress update instead of held across it
// (12 VGPRs less, for callers that would spill).
// UL: updated / semi-Lagrangian, as hex8_element's.
template <int KIND, bool PER_QP, bool LEAN = false, bool UL = false>
APHIP_DEV bool hex8_lanes(int lane, const uint32_t (&cn)[4], const double *sX, const double *sU, double *row,
                          const MatParams &m, double ga, const double *state_n, double *state_np1, double *H,
                          double *P, const RateIn *r = nullptr) {
#pragma clang fp contract(off)
    int x = hex8_lane_label(lane);
    bool b0 = x & 1, b1 = x & 2, b2 = x & 4;
    const int q = x == 2 ? 3 : x == 3 ? 2 : x == 6 ? 7 : x == 7 ? 6 : x;  // point (and corner) index
    if (lane < 6) hex8_field_modes(cn, (lane < 3 ? sX : sU) + (lane < 3 ? lane : lane - 3), ga, row + 7 * lane);
    __builtin_amdgcn_wave_barrier();  // (LDS operations of a wave stay in order)
    double s0 = b0 ? -1.0 : 1.0, s1 = b1 ? -1.0 : 1.0, s2 = b2 ? -1.0 : 1.0;
    const double s01 = s0 * s1, s02 = s0 * s2, s12 = s1 * s2;
    double J[9], G[9];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        double wx[8], wu[8], g[3];
        wx[0] = wu[0] = 0.0;
#pragma unroll
        for (int S = 1; S < 8; ++S) {
            wx[S] = row[7 * i + S - 1];
            wu[S] = row[7 * (i + 3) + S - 1];
        }
        hex8_grad(wx, -s0, -s1, -s2, s01, s02, s12, g);
        J[3 * i] = g[0];
        J[3 * i + 1] = g[1];
        J[3 * i + 2] = g[2];
        hex8_grad(wu, -s0, -s1, -s2, s01, s02, s12, g);
        G[3 * i] = g[0];
        G[3 * i + 1] = g[1];
        G[3 * i + 2] = g[2];
    }
    // w J^-1 = adj(J) up to exact powers of two, so the force takes the adjugate itself
    double Ad[9];
    const double id = 1.0 / adjugate3(J, Ad);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            H[3 * i + j] = dot3(G[3 * i], Ad[j], G[3 * i + 1], Ad[3 + j], G[3 * i + 2], Ad[6 + j]) * id;
    const bool last = q == 7;
    double snp1 = 0.0, aux = 0.0;
    const double sn = load_state<KIND>(state_n, PER_QP ? q : 0), sn2 = load_state2<KIND>(state_n, PER_QP ? q : 0);
    if constexpr (UL) ul_gradient(H, r->Hn);
    stress<KIND>(H, m, sn, snp1, aux, P, r, sn2);
    if constexpr (PER_QP) store_state<KIND>(state_np1, q, snp1, aux);
    else if (last) store_state<KIND>(state_np1, 0, snp1, aux);
    double Pf[9];
    if constexpr (UL) {
        ul_force_stress(P, r->Hn, Pf);
    } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) Pf[i] = P[i];
    }
    if constexpr (LEAN) {
        asm volatile("" : "+v"(x));  // (a value the compiler cannot match with the earlier one)
        b0 = x & 1;
        b1 = x & 2;
        b2 = x & 4;
        s0 = b0 ? -1.0 : 1.0;
        s1 = b1 ? -1.0 : 1.0;
        s2 = b2 ? -1.0 : 1.0;
    }
    hex8_to_corners(x, b0, b1, b2, s0, s1, s2, ga, -1.0 / 512.0, Ad, Pf, row + 3 * q);  // (exact: -w det^-1)
    return last;
}

// Smoothed Tet4 B and volume from the faces (include/QuadratureSmoothed.h:32-62)
__host__ __device__ inline void smoothed_tet4(const double (&X)[4][3], double (&B)[4][3], double &V) {
    const int faces[4][3] = {{0, 1, 3}, {1, 2, 3}, {0, 3, 2}, {0, 2, 1}};
    double vol = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) B[k][0] = B[k][1] = B[k][2] = 0.0;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        double e1[3], e2[3], n[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            e1[d] = X[faces[f][1]][d] - X[faces[f][0]][d];
            e2[d] = X[faces[f][2]][d] - X[faces[f][0]][d];
        }
        n[0] = (e1[1] * e2[2] - e1[2] * e2[1]) / 2.0;
        n[1] = (e1[2] * e2[0] - e1[0] * e2[2]) / 2.0;
        n[2] = (e1[0] * e2[1] - e1[1] * e2[0]) / 2.0;
        const double *x0 = X[faces[f][0]];
        vol += x0[0] * n[0] + x0[1] * n[1] + x0[2] * n[2];
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
            for (int d = 0; d < 3; ++d) B[faces[f][l]][d] += n[d] / 3.0;
    }
    vol /= 3.0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) B[k][d] /= vol;
    V = vol;
}

// Smoothed Hex8 B and volume from the faces, each split into four triangles about
// its centroid (include/QuadratureSmoothed.h:96-150)
__host__ __device__ inline void smoothed_hex8(const double (&X)[8][3], double (&B)[8][3], double &V) {
    const int faces[6][4] = {{0, 1, 5, 4}, {1, 2, 6, 5}, {2, 3, 7, 6}, {0, 4, 7, 3}, {0, 3, 2, 1}, {4, 5, 6, 7}};
    double vol = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) B[k][0] = B[k][1] = B[k][2] = 0.0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        double mid[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int d = 0; d < 3; ++d) mid[d] += X[faces[f][k]][d];
#pragma unroll
        for (int d = 0; d < 3; ++d) mid[d] /= 4.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int km1 = (k + 3) & 3;
            double e1[3], e2[3], n[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                e1[d] = X[faces[f][km1]][d] - mid[d];
                e2[d] = X[faces[f][k]][d] - mid[d];
            }
            n[0] = (e1[1] * e2[2] - e1[2] * e2[1]) / 2.0;
            n[1] = (e1[2] * e2[0] - e1[0] * e2[2]) / 2.0;
            n[2] = (e1[0] * e2[1] - e1[1] * e2[0]) / 2.0;
            vol += mid[0] * n[0] + mid[1] * n[1] + mid[2] * n[2];
#pragma unroll
            for (int l = 0; l < 4; ++l) {
                const double cw = (l == k || l == km1) ? 5.0 / 12.0 : 1.0 / 12.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) B[faces[f][l]][d] += n[d] * cw;
            }
        }
    }
    vol /= 3.0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) B[k][d] /= vol;
    V = vol;
}

template <int NPE>
__host__ __device__ __forceinline__ void smoothed_cell(const double (&X)[NPE][3], double (&B)[NPE][3], double &V) {
    if constexpr (NPE == 4) smoothed_tet4(X, B, V);
    else smoothed_hex8(X, B, V);
}

// Smoothed Hex8 cell (one subcell per hex, include/ComputeInternalForceSmoothedCell.h:86-117,
// :186-224, :325-349): H = sum_k u_k (x) B_k and fe[k] = -V P B_k with the face-smoothed B,
// recomputed from the coordinates (192 B a cell less to read, some 600 flops).
template <int KIND>
APHIP_DEV void hex8_cell(const double (&X)[8][3], const double (&U)[8][3], const MatParams &m, const double *state_n,
                         double *state_np1, double *H, double *P, double (&fe)[8][3], const RateIn *r = nullptr) {
#pragma clang fp contract(off)
    double B[8][3], V;
    smoothed_hex8(X, B, V);
#pragma unroll
    for (int i = 0; i < 9; ++i) H[i] = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) H[3 * i + j] = __fma_rn(U[k][i], B[k][j], H[3 * i + j]);
    double snp1 = 0.0, aux = 0.0;
    stress<KIND>(H, m, load_state<KIND>(state_n, 0), snp1, aux, P, r, load_state2<KIND>(state_n, 0));
    store_state<KIND>(state_np1, 0, cell_damage_marker<KIND>(snp1, m), aux);
    const double mv = -V;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < 3; ++i)
            fe[k][i] = mv * dot3(P[3 * i], B[k][0], P[3 * i + 1], B[k][1], P[3 * i + 2], B[k][2]);
}

}  // namespace aphip
