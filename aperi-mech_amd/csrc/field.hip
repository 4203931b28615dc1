// Field transfer between caller-owned device arrays (caller numbering, the reference's
// field layout: node vectors n x w row-major, element tensors n_elem x 9 row-major,
// element state n_elem x w) and the context's internal arrays (Morton numbering; node
// vectors AoS, tensors SoA 9 x n_elem).  One thread per value; the internal side is read or
// written contiguously, the caller side a row at a time through the permutation.
#include "internal.hpp"

namespace aphip {

namespace {

constexpr int kBlock = 256;

inline dim3 blocks(int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

// dst[i, :] = src[iperm[i], :]  (caller -> internal, w values per entity), one thread per
// value: the internal side is contiguous across the lanes and a row of the caller's side is
// one run of w lanes.  W: the row width known at compile time (3: node vectors), 0: w.
template <int W>
__global__ __launch_bounds__(kBlock) void k_gather_rows(int64_t n, int w_any, const int32_t *iperm, const double *src,
                                                        double *dst) {
    const int w = W ? W : w_any;
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= n * w) return;
    const int64_t i = t / w;
    dst[t] = src[(int64_t)iperm[i] * w + (t - i * w)];
}

// dst[iperm[i], :] = src[i, :]  (internal -> caller), lanes as in k_gather_rows
template <int W>
__global__ __launch_bounds__(kBlock) void k_scatter_rows(int64_t n, int w_any, const int32_t *iperm, const double *src,
                                                         double *dst) {
    const int w = W ? W : w_any;
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= n * w) return;
    const int64_t i = t / w;
    dst[(int64_t)iperm[i] * w + (t - i * w)] = src[t];
}

// dst[iperm[e], k] = planes[k, e]  (SoA tensor -> caller row-major).  Bound by HBM (144 B per
// element).  A block transposes its 256 elements in LDS: the planes are read 64 consecutive
// doubles at a time and every 72-byte row is written by nine consecutive lanes; the rows of
// elements that are neighbours in the caller's order mostly fall into one block, whose stores
// then fill whole lines.  (One thread writing its nine values 72 bytes from the next lane's
// took 758 us for 6M elements, 1.1 TB/s; this takes about 240 us, 3.6 TB/s.)
__global__ __launch_bounds__(kBlock) void k_scatter_tensor(int64_t ne, const int32_t *iperm, const double *planes,
                                                           double *dst) {
    __shared__ double row[9 * kBlock];
    __shared__ int32_t to[kBlock];
    const int tid = threadIdx.x;
    const int64_t e0 = (int64_t)blockIdx.x * kBlock;
    const int64_t e = min(e0 + tid, ne - 1);  // lanes past the end repeat the last element
    double v[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] = planes[k * ne + e];
    to[tid] = iperm[e];
#pragma unroll
    for (int k = 0; k < 9; ++k) row[9 * tid + k] = v[k];
    __syncthreads();
    const int n9 = 9 * (int)min((int64_t)kBlock, ne - e0);
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        const int t = r * kBlock + tid, j = t / 9;
        if (t < n9) dst[9 * (int64_t)to[j] + (t - 9 * j)] = row[t];
    }
}

// Per-element E and nu (caller order) to internal order, and their Lame constants
// (lambda = E nu / ((1 + nu) (1 - 2 nu)), mu = E / (2 (1 + nu))).
__global__ __launch_bounds__(kBlock) void k_lame(int64_t ne, const int32_t *iperm, const double *E, const double *nu,
                                                 double *E_i, double *nu_i, double *lambda, double *mu) {
#pragma clang fp contract(off)
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= ne) return;
    const int64_t s = iperm[e];
    const double Ee = E[s], n = nu[s];
    E_i[e] = Ee;
    nu_i[e] = n;
    mu[e] = Ee / (2 * (1 + n));
    lambda[e] = (Ee * n) / ((1 + n) * (1 - 2 * n));
}

// Adjoints of E and nu, caller order, from those of lambda and mu (E, nu: per element, or null
// and the material's).
__global__ __launch_bounds__(kBlock) void k_parameter_gradients(int64_t ne, const int32_t *iperm, const double *lam_bar,
                                                                const double *mu_bar, const double *E_i,
                                                                const double *nu_i, double E0, double nu0,
                                                                double *E_bar, double *nu_bar) {
#pragma clang fp contract(off)
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= ne) return;
    const double E = E_i ? E_i[e] : E0, nu = E_i ? nu_i[e] : nu0;
    const double q = (1 + nu) * (1 - 2 * nu);
    const double dl_dE = nu / q, dm_dE = 1.0 / (2 * (1 + nu));
    const double dl_dnu = E * (1 + 2 * nu * nu) / (q * q), dm_dnu = -E / (2 * (1 + nu) * (1 + nu));
    const int64_t ce = iperm[e];
    E_bar[ce] = lam_bar[e] * dl_dE + mu_bar[e] * dm_dE;
    nu_bar[ce] = lam_bar[e] * dl_dnu + mu_bar[e] * dm_dnu;
}

// dst[i] = src[iperm[i]] and a count of the values that are not positive (nodal mass)
__global__ __launch_bounds__(kBlock) void k_gather_positive(int64_t n, const int32_t *iperm, const double *src,
                                                            double *dst, int32_t *n_bad) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double x = src[iperm[i]];
    dst[i] = x;
    if (!(x > 0.0)) atomicAdd(n_bad, 1);
}

}  // namespace

void field_gather_rows(Ctx &c, int64_t n, int w, const int32_t *iperm, const double *src, double *dst) {
    if (n == 0) return;
    if (w == 3) hipLaunchKernelGGL(k_gather_rows<3>, blocks(n * w), dim3(kBlock), 0, c.stream, n, w, iperm, src, dst);
    else hipLaunchKernelGGL(k_gather_rows<0>, blocks(n * w), dim3(kBlock), 0, c.stream, n, w, iperm, src, dst);
    APHIP_HIP(hipGetLastError());
}

void field_scatter_rows(Ctx &c, int64_t n, int w, const int32_t *iperm, const double *src, double *dst) {
    if (n == 0) return;
    if (w == 3) hipLaunchKernelGGL(k_scatter_rows<3>, blocks(n * w), dim3(kBlock), 0, c.stream, n, w, iperm, src, dst);
    else hipLaunchKernelGGL(k_scatter_rows<0>, blocks(n * w), dim3(kBlock), 0, c.stream, n, w, iperm, src, dst);
    APHIP_HIP(hipGetLastError());
}

// Both pass the caller-ordered host arrays through the staging buffer; the permutation and the
// divisions run on the device (48,000 Tet4: the two took 0.16 ms of host loops).
static double *staging(Ctx &c) {
    c.stage.alloc(2 * (size_t)c.ne);
    return c.stage.p;
}

void material_fields_from_host(Ctx &c, const double *E, const double *nu) {
    for (DevBuf<double> *b : {&c.elem_E, &c.elem_nu, &c.elem_lambda, &c.elem_mu}) b->alloc(c.ne);
    if (c.ne == 0) return;
    double *s = staging(c);
    APHIP_HIP(hipMemcpyAsync(s, E, sizeof(double) * c.ne, hipMemcpyHostToDevice, c.stream));
    APHIP_HIP(hipMemcpyAsync(s + c.ne, nu, sizeof(double) * c.ne, hipMemcpyHostToDevice, c.stream));
    hipLaunchKernelGGL(k_lame, blocks(c.ne), dim3(kBlock), 0, c.stream, c.ne, c.d_elem_iperm.p, s, s + c.ne, c.elem_E.p,
                       c.elem_nu.p, c.elem_lambda.p, c.elem_mu.p);
    APHIP_HIP(hipGetLastError());
    APHIP_HIP(hipStreamSynchronize(c.stream));
}

void parameter_gradients_to_host(Ctx &c, const double *lam_bar, const double *mu_bar, double *E_bar, double *nu_bar) {
    if (c.ne == 0) return;
    double *s = staging(c);
    const bool fields = c.has_fields && c.elem_E.p;
    hipLaunchKernelGGL(k_parameter_gradients, blocks(c.ne), dim3(kBlock), 0, c.stream, c.ne, c.d_elem_iperm.p, lam_bar,
                       mu_bar, fields ? c.elem_E.p : nullptr, fields ? c.elem_nu.p : nullptr, c.mat.E, c.mat.nu, s,
                       s + c.ne);
    APHIP_HIP(hipGetLastError());
    if (E_bar) APHIP_HIP(hipMemcpyAsync(E_bar, s, sizeof(double) * c.ne, hipMemcpyDeviceToHost, c.stream));
    if (nu_bar) APHIP_HIP(hipMemcpyAsync(nu_bar, s + c.ne, sizeof(double) * c.ne, hipMemcpyDeviceToHost, c.stream));
    APHIP_HIP(hipStreamSynchronize(c.stream));
}

void field_scatter_tensor(Ctx &c, const double *planes, double *dst) {
    if (c.ne == 0) return;
    hipLaunchKernelGGL(k_scatter_tensor, blocks(c.ne), dim3(kBlock), 0, c.stream, c.ne, c.d_elem_iperm.p, planes,
                       dst);
    APHIP_HIP(hipGetLastError());
}

int32_t field_gather_mass(Ctx &c, const double *src) {
    c.d_count.zero(c.stream);
    hipLaunchKernelGGL(k_gather_positive, blocks(c.nn), dim3(kBlock), 0, c.stream, c.nn, c.d_node_iperm.p, src,
                       c.mass.p, c.d_count.p);
    APHIP_HIP(hipGetLastError());
    int32_t bad = 0;
    c.d_count.download(&bad, 1, c.stream);
    APHIP_HIP(hipStreamSynchronize(c.stream));
    return bad;
}

}  // namespace aphip
