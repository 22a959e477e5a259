// Dense FP64 inverse of a multigrid hierarchy's coarsest level (at most 1024 cells),
// assembled and inverted on the device.
//
// The inverse is a blocked in-place Gauss-Jordan elimination with 32 x 32 pivot blocks.
// Per block two launches: k_gj_panel inverts the pivot block (every workgroup for itself:
// 32 rank-1 steps in registers, the pivot row and column exchanged through LDS, one barrier
// a step) and forms one 32-column tile of the scaled pivot rows; k_gj_update applies the
// rank-32 update to the other rows in 64 x 64 tiles held 4 x 4 per thread. The chain of n
// pivots bounds it, not the 2 n^3 operations: at n = 1000, 32 x (12.5 us panel + 10.1 us
// update) = 0.72 ms. The diagonal
// pivots of a symmetric matrix are all positive exactly when it is positive definite, which
// every level of a Laplacian with a non-negative shift is; a pivot that is not positive
// sets a flag, and the level is then inverted on the host with row exchanges, as an
// indefinite operator needs. On a 640 x 400 variable-coefficient equation (coarsest level
// 40 x 25, rebuilt at every solve) the host elimination took 240 ms of a 252 ms solve; the
// solve now takes 2.6 ms.
#include <algorithm>
#include <cmath>

#include "gmg.hpp"

namespace opf {
namespace {

constexpr int kPB = 32;  // pivot block
constexpr int kTU = 64;  // update tile

// the coarsest level's operator as the assembly reads it
struct CoarseOp {
    int n[3], dim, N;
    int per[3];
    double alpha[3][2];
    bool var;
    double a[3], sigma;       // constant mode
    const double* af[3];      // variable mode
    const double* sg;
};

__device__ __forceinline__ double coarse_face(const CoarseOp& o, int d, int i, int j, int k) {
    return o.var ? o.af[d][face_index(d, i, j, k, o.n[0], o.n[1])] : o.a[d];
}

// diagonal of cell c; row (when given) receives the neighbours' entries
__device__ double coarse_row(const CoarseOp& o, int c, double* row) {
    const int p[3] = {c % o.n[0], (c / o.n[0]) % o.n[1], c / (o.n[0] * o.n[1])};
    double D = o.var ? o.sg[c] : o.sigma;
    for (int d = 0; d < o.dim; ++d)
        for (int s = 0; s < 2; ++s) {
            int f[3] = {p[0], p[1], p[2]}, q[3] = {p[0], p[1], p[2]};
            f[d] += s;
            q[d] += s == 0 ? -1 : 1;
            const double a = coarse_face(o, d, f[0], f[1], f[2]);
            if ((q[d] < 0 || q[d] >= o.n[d]) && !o.per[d]) {
                D += a * (1.0 - o.alpha[d][s]);
                continue;
            }
            q[d] = q[d] < 0 ? o.n[d] - 1 : q[d] >= o.n[d] ? 0 : q[d];
            D += a;
            if (row) row[q[0] + o.n[0] * (q[1] + o.n[1] * q[2])] -= a;
        }
    return D;
}

// mean diagonal / N: added to every entry of a singular operator, it lifts the constant
// vector's eigenvalue off zero
__global__ __launch_bounds__(1024) void k_coarse_shift(CoarseOp o, double* __restrict__ dm) {
    __shared__ double sh[16];
    double s = 0;
    for (int c = threadIdx.x; c < o.N; c += 1024) s += coarse_row(o, c, nullptr);
    for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        s = 0;
        for (int w = 0; w < 16; ++w) s += sh[w];
        *dm = s / ((double)o.N * o.N);
    }
}

// one workgroup per row
__global__ __launch_bounds__(256) void k_coarse_fill(CoarseOp o, const double* __restrict__ dm, double* __restrict__ A) {
    double* row = A + (size_t)blockIdx.x * o.N;
    const double v = dm ? *dm : 0.0;
    for (int c = threadIdx.x; c < o.N; c += 256) row[c] = v;
    __syncthreads();
    if (threadIdx.x == 0) row[blockIdx.x] += coarse_row(o, blockIdx.x, row);
}

// 1 / v to about one unit in the last place (v_rcp_f64 and two Newton steps): the pivots'
// reciprocals are on the chain, where an IEEE division is twice as long
__device__ __forceinline__ double quick_rcp(double v) {
    double y = __builtin_amdgcn_rcp(v);
    y = __builtin_fma(__builtin_fma(-v, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-v, y, 1.0), y, y);
}

// pivot block k0: R (kPB x n) = the scaled pivot rows, the inverted pivot block in the
// pivot's own columns; C (n x kPB) = the pivot columns as they were. One barrier a pivot:
// the row and column buffers alternate, and a buffer is written again only after the next
// pivot's barrier.
__global__ __launch_bounds__(256) void k_gj_panel(const double* __restrict__ A, int n, int k0, double* __restrict__ R,
                                                  double* __restrict__ C, int* __restrict__ flag) {
    __shared__ double prow[2][kPB], pcol[2][kPB], P[kPB][kPB + 2], T[kPB][kPB + 2];
    const int bs = min(kPB, n - k0), j0 = blockIdx.x * kPB;
    const int t = threadIdx.x, r = t >> 3, g = t & 7, c0 = g * 4;  // this thread: row r, columns c0 .. c0 + 3
    double a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = c0 + q;
        a[q] = r < bs && c < bs ? A[(size_t)(k0 + r) * n + k0 + c] : (r == c ? 1.0 : 0.0);
        T[r][c] = r < bs && j0 + c < n ? A[(size_t)(k0 + r) * n + j0 + c] : 0.0;
        if (j0 + r < n) C[(size_t)(j0 + r) * kPB + c] = c < bs ? A[(size_t)(j0 + r) * n + k0 + c] : 0.0;
    }
    bool bad = false;
    for (int m = 0; m < kPB / 4; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // pivot p, held in register q of the threads with g = m
            const int p = 4 * m + q;
            double* pr = prow[q & 1];
            double* pc = pcol[q & 1];
            if (r == p) {
#pragma unroll
                for (int w = 0; w < 4; ++w) pr[c0 + w] = a[w];
            }
            if (g == m) pc[r] = a[q];
            __syncthreads();
            const double piv = pr[p], inv = quick_rcp(piv);
            bad |= !(piv > 0.0) || !isfinite(inv);
            const bool own = r == p;
            const double f = own ? -inv : pc[r] * inv;  // the pivot's row is scaled: a' = a / piv
#pragma unroll
            for (int w = 0; w < 4; ++w) a[w] = __builtin_fma(-f, pr[c0 + w], own ? 0.0 : a[w]);
            if (g == m) a[q] = own ? inv : -f;
        }
    if (bad && t == 0 && blockIdx.x == 0) *flag = 1;
    if (j0 == k0) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (j0 + c0 + q < n) R[(size_t)r * n + j0 + c0 + q] = a[q];
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) P[r][c0 + q] = a[q];
    __syncthreads();
    double s[4] = {0, 0, 0, 0};
#pragma unroll 8
    for (int m = 0; m < kPB; ++m) {
        const double pm = P[r][m];
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = __builtin_fma(pm, T[m][c0 + q], s[q]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (j0 + c0 + q < n) R[(size_t)r * n + j0 + c0 + q] = s[q];
}

// rows of the pivot block become R; every other row loses (its pivot columns) x R, with
// its pivot columns taken as zero first. The tile's own entries are loaded first, so that
// they arrive while the panels are staged.
__global__ __launch_bounds__(256) void k_gj_update(double* __restrict__ A, int n, int k0, const double* __restrict__ R,
                                                   const double* __restrict__ C) {
    __shared__ double sc[kPB][kTU + 2], sr[kPB][kTU + 2];
    const int bs = min(kPB, n - k0), i0 = blockIdx.y * kTU, j0 = blockIdx.x * kTU, t = threadIdx.x;
    const int ti = (t >> 4) * 4, tj = t & 15;  // rows ti .. ti + 3, columns tj + 16 y
    double acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const int i = min(i0 + ti + x, n - 1), j = min(j0 + tj + 16 * y, n - 1);
            acc[x][y] = A[(size_t)i * n + j];
        }
#pragma unroll
    for (int w = 0; w < kPB * kTU / 256; ++w) {
        const int e = t + 256 * w;
        const int ci = e / kPB, cm = e % kPB;  // C is kPB wide
        sc[cm][ci] = i0 + ci < n ? C[(size_t)(i0 + ci) * kPB + cm] : 0.0;
        const int rm = e / kTU, rj = e % kTU;
        sr[rm][rj] = rm < bs && j0 + rj < n ? R[(size_t)rm * n + j0 + rj] : 0.0;
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        const int j = j0 + tj + 16 * y;
        const bool zero = j >= k0 && j < k0 + bs;
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[x][y] = zero ? 0.0 : acc[x][y];
    }
    __syncthreads();
#pragma unroll 4
    for (int m = 0; m < kPB; ++m) {
        double u[4], v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) u[q] = -sc[m][ti + q], v[q] = sr[m][tj + 16 * q];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = __builtin_fma(u[x], v[y], acc[x][y]);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const int i = i0 + ti + x;
        if (i >= n) continue;
        const bool prow = i >= k0 && i < k0 + bs;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const int j = j0 + tj + 16 * y;
            if (j < n) A[(size_t)i * n + j] = prow ? sr[i - k0][tj + 16 * y] : acc[x][y];
        }
    }
}

// Gauss-Jordan inverse with partial pivoting (host)
bool invert_pivoting(std::vector<double>& A, int n, std::vector<double>& inv) {
    inv.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; ++i) inv[(size_t)i * n + i] = 1.0;
    for (int c = 0; c < n; ++c) {
        int p = c;
        for (int r = c + 1; r < n; ++r)
            if (std::fabs(A[(size_t)r * n + c]) > std::fabs(A[(size_t)p * n + c])) p = r;
        if (A[(size_t)p * n + c] == 0.0) return false;
        if (p != c)
            for (int k = 0; k < n; ++k) {
                std::swap(A[(size_t)p * n + k], A[(size_t)c * n + k]);
                std::swap(inv[(size_t)p * n + k], inv[(size_t)c * n + k]);
            }
        double d = 1.0 / A[(size_t)c * n + c];
        for (int k = 0; k < n; ++k) {
            A[(size_t)c * n + k] *= d;
            inv[(size_t)c * n + k] *= d;
        }
        for (int r = 0; r < n; ++r) {
            if (r == c) continue;
            double f = A[(size_t)r * n + c];
            if (f == 0.0) continue;
            for (int k = 0; k < n; ++k) {
                A[(size_t)r * n + k] -= f * A[(size_t)c * n + k];
                inv[(size_t)r * n + k] -= f * inv[(size_t)c * n + k];
            }
        }
    }
    return true;
}

}  // namespace

int coarse_inverse_dev(hipStream_t st, Hierarchy& H) {
    const GLevelHost& L = H.host.back();
    const GLevelDev& D = H.dev.back();
    const int n = (int)L.N;
    CoarseOp o{};
    for (int d = 0; d < 3; ++d) {
        o.n[d] = L.n[d];
        o.per[d] = H.per[d];
        o.a[d] = L.a[d];
        o.af[d] = D.af64[d];
        for (int s = 0; s < 2; ++s) o.alpha[d][s] = H.alpha[d][s];
    }
    o.dim = H.dim;
    o.N = n;
    o.var = L.var;
    o.sigma = L.sigma;
    o.sg = D.sg64;
    // scratch kept with the hierarchy: R, C, the shift and the flag
    const size_t panel = (size_t)kPB * n;
    if (!H.cinv) {
        OPF_HIP(hipMalloc((void**)&H.cinv, sizeof(double) * n * n));
        OPF_HIP(hipMalloc((void**)&H.cwork, sizeof(double) * (2 * panel + 2)));
        H.cN = n;
        H.bytes += sizeof(double) * ((size_t)n * n + 2 * panel + 2);
    }
    double *R = H.cwork, *C = R + panel, *dm = C + panel;
    int* flag = (int*)(dm + 1);
    auto assemble = [&] {
        if (H.singular) hipLaunchKernelGGL(k_coarse_shift, dim3(1), dim3(1024), 0, st, o, dm);
        hipLaunchKernelGGL(k_coarse_fill, dim3(n), dim3(256), 0, st, o, H.singular ? (const double*)dm : nullptr, H.cinv);
    };
    int bad = 0;
    OPF_HIP(hipMemsetAsync(flag, 0, sizeof(int), st));
    assemble();
    const unsigned panels = (unsigned)((n + kPB - 1) / kPB), tiles = (unsigned)((n + kTU - 1) / kTU);
    for (int k0 = 0; k0 < n; k0 += kPB) {
        hipLaunchKernelGGL(k_gj_panel, dim3(panels), dim3(256), 0, st, (const double*)H.cinv, n, k0, R, C, flag);
        hipLaunchKernelGGL(k_gj_update, dim3(tiles, tiles), dim3(256), 0, st, H.cinv, n, k0, (const double*)R,
                           (const double*)C);
    }
    OPF_HIP(hipGetLastError());
    OPF_HIP(hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, st));
    OPF_HIP(hipStreamSynchronize(st));
    if (!bad) return OPF_OK;
    std::vector<double> A((size_t)n * n), inv;
    assemble();
    OPF_HIP(hipMemcpyAsync(A.data(), H.cinv, sizeof(double) * A.size(), hipMemcpyDeviceToHost, st));
    OPF_HIP(hipStreamSynchronize(st));
    OPF_CHECK(invert_pivoting(A, n, inv), OPF_ERR_ARG, "gmg: singular coarsest operator");
    OPF_HIP(hipMemcpyAsync(H.cinv, inv.data(), sizeof(double) * inv.size(), hipMemcpyHostToDevice, st));
    OPF_HIP(hipStreamSynchronize(st));
    return OPF_OK;
}

}  // namespace opf
