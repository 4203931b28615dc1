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
