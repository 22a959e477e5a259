// Dense FP64 inverse of a multigrid hierarchy's coarsest level (at most 1024 cells),
// assembled and inverted on the device.
//
// The inverse is a blocked Gauss-Jordan elimination with 32 x 32 pivot blocks, one launch a
// block. A workgroup of k_gj_step owns a 64 x 64 tile: it scales its part of the pivot rows by the
// inverted pivot block and subtracts (its part of the pivot columns) x (those rows), both on the
// matrix cores (FP64 16 x 16 x 4), reading one buffer and writing the other, so that no workgroup
// waits for another. Workgroup 0 has no tile: it forms the next pivot block for itself from the same
// buffer and inverts it with its 256 threads, four pivots a round and one barrier a round, while the
// others update. n = 1000: 32 launches of 11.3 us; a panel launch in which every workgroup inverted the
// pivot block and an update launch on the vector pipes took 12.9 + 10.4 us and a gap more; with the
// block formed and inverted by the workgroup of its tile, after its update, 15.3. The inverse is as
// far from one in 80 bits as the host's elimination with row exchanges is (1000 cells with a coefficient
// over two powers of ten: 3e-15 of its largest entry both).
// The diagonal pivots of a symmetric matrix are all positive exactly when it is positive
// definite, which every level of a Laplacian with a non-negative shift is; a pivot that is not
// positive sets a flag, and the level is then inverted on the host with row exchanges, as an
// indefinite operator needs. On a 640 x 400 variable-coefficient equation (coarsest level
// 40 x 25, rebuilt at every solve) the host elimination took 240 ms of a 252 ms solve.
#include <algorithm>
#include <cmath>
#include <utility>

#include "gmg.hpp"

namespace opf {
namespace {

constexpr int kPB = 32;  // pivot block
constexpr int kTU = 64;  // tile of a workgroup

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

// In-place inverse of the symmetric kPB x kPB matrix M by one workgroup of 256: thread t has columns
// 4 (t / 32) .. of row t % 32. Four pivots a round: their columns are exchanged through LDS (their
// rows are the columns, negated for the pivots already taken, as elimination in place leaves a
// symmetric matrix), every thread inverts their 4 x 4 block by halves and subtracts a rank-4 update.
// The round's chain of latencies bounds it: with one pivot a round 12 us a block, with four by one
// wave 6, now 3.5. One barrier a round: the buffers alternate. xch: kXch values. False when a leading
// minor of a pivot block is not positive.
constexpr int kXch = 16 * kPB;
__device__ __forceinline__ bool invert_block(double (*M)[kPB + 2], double* xch) {
    const int r = threadIdx.x & 31, g = threadIdx.x >> 5;
    double a[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) a[w] = M[r][4 * g + w];
    bool ok = true;
#pragma unroll 1
    for (int m = 0; m < kPB / 4; ++m) {
        const int p = 4 * m;
        const bool own = r >= p && r < p + 4;
        double *col = xch + (m & 1) * 8 * kPB, *rows = col + 4 * kPB;  // col[4 r + k], rows[kPB k + c]
        if (g == m) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                col[4 * r + k] = a[k];
                rows[kPB * k + r] = r < p ? -a[k] : a[k];
            }
        }
        __syncthreads();
        // V = the inverse of [[P, Q], [Q^T, S]] (2 x 2 blocks, P and S symmetric)
        const double* b = col + 4 * p;
        const double p0 = b[0], p1 = b[4], p2 = b[5], q0 = b[8], q1 = b[12], q2 = b[9], q3 = b[13];
        const double dp = p0 * p2 - p1 * p1, ip = quick_rcp(dp);
        const double i0 = p2 * ip, i1 = -p1 * ip, i2 = p0 * ip;                     // P^-1
        const double u0 = i0 * q0 + i1 * q2, u1 = i0 * q1 + i1 * q3;                // U = P^-1 Q
        const double u2 = i1 * q0 + i2 * q2, u3 = i1 * q1 + i2 * q3;
        const double s0 = b[10] - (q0 * u0 + q2 * u2), s1 = b[14] - (q1 * u0 + q3 * u2);
        const double s2 = b[15] - (q1 * u1 + q3 * u3);                              // S - Q^T U
        const double ds = s0 * s2 - s1 * s1, is = quick_rcp(ds);
        const double j0 = s2 * is, j1 = -s1 * is, j2 = s0 * is;
        ok &= p0 > 0.0 && dp > 0.0 && s0 > 0.0 && ds > 0.0 && isfinite(ip) && isfinite(is);
        const double v0 = -(u0 * j0 + u1 * j1), v1 = -(u0 * j1 + u1 * j2);          // -U (..)^-1
        const double v2 = -(u2 * j0 + u3 * j1), v3 = -(u2 * j1 + u3 * j2);
        const double w0 = i0 - (v0 * u0 + v1 * u1), w1 = i1 - (v0 * u2 + v1 * u3), w2 = i2 - (v2 * u2 + v3 * u3);
        // a row of the block becomes V times the pivot rows: its factors are those of -1 in its place
        double c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = own ? (r == p + k ? -1.0 : 0.0) : col[4 * r + k];
        const double f[4] = {c[0] * w0 + c[1] * w1 + c[2] * v0 + c[3] * v1, c[0] * w1 + c[1] * w2 + c[2] * v2 + c[3] * v3,
                             c[0] * v0 + c[1] * v2 + c[2] * j0 + c[3] * j1, c[0] * v1 + c[1] * v3 + c[2] * j1 + c[3] * j2};
        const double keep = own ? 0.0 : 1.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            double n = keep * a[w];
#pragma unroll
            for (int k = 0; k < 4; ++k) n = __builtin_fma(-f[k], rows[kPB * k + 4 * g + w], n);
            a[w] = g == m ? -f[w] : n;
        }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) M[r][4 * g + w] = a[w];
    __syncthreads();
    return ok;
}

// the first pivot block's inverse
__global__ __launch_bounds__(256) void k_gj_first(const double* __restrict__ A, int n, double* __restrict__ D,
                                                  int* __restrict__ flag) {
    __shared__ double M[kPB][kPB + 2];
    __shared__ __attribute__((aligned(16))) double xch[kXch];
#pragma unroll
    for (int u = 0; u < kPB * kPB / 256; ++u) {
        const int e = threadIdx.x + 256 * u, r = e / kPB, c = e % kPB;
        const double v = A[(size_t)min(r, n - 1) * n + min(c, n - 1)];
        M[r][c] = r < n && c < n ? v : (r == c ? 1.0 : 0.0);
    }
    __syncthreads();
    if (!invert_block(M, xch) && threadIdx.x == 0) *flag = 1;
#pragma unroll
    for (int u = 0; u < kPB * kPB / 256; ++u) {
        const int e = threadIdx.x + 256 * u;
        D[e] = M[e / kPB][e % kPB];
    }
}

typedef double f64x4 __attribute__((ext_vector_type(4)));
// v_mfma_f64_16x16x4: lane l brings row (column) l % 16 of the factors at depth l / 16 and holds
// column l % 16, rows l / 16 + 4 q of the product.
// The next pivot block's inverse, by the first workgroup of a step, which forms the block for itself
// instead of waiting for its tile: the block less (its pivot columns) x (scaled pivot rows).
__device__ __forceinline__ void next_block(const double* __restrict__ A, int n, int k0, const double* __restrict__ D,
                                           double* __restrict__ Dn, int* __restrict__ flag, double (*sc)[kTU + 2],
                                           double (*sr)[kTU + 2], double (*sd)[kPB + 2], double* xch) {
    const int k1 = k0 + kPB, t = threadIdx.x, w = t >> 6, lane = t & 63, lo = lane & 15, hi = lane >> 4;
    const int x = 16 * (w >> 1), y = 16 * (w & 1);  // this wave's quarter of the block
    auto at = [&](int i, int j) { return A[(size_t)min(i, n - 1) * n + min(j, n - 1)]; };
    f64x4 acc, s = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int i = k1 + x + hi + 4 * q, j = k1 + y + lo;
        const double v = at(i, j);
        acc[q] = i < n && j < n ? v : (i == j ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < kPB * kPB / 256; ++u) {  // k1 < n: the pivot block at k0 is whole
        const int e = t + 256 * u, r = e / kPB, c = e % kPB;
        const double cv = at(k1 + r, k0 + c), rv = at(k0 + r, k1 + c);
        sc[c][r] = k1 + r < n ? -cv : 0.0;
        sr[r][c] = k1 + c < n ? rv : 0.0;
        sd[c][r] = D[e];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kPB; m += 4)
        s = __builtin_amdgcn_mfma_f64_16x16x4f64(sd[m + hi][x + lo], sr[m + hi][y + lo], s, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) sr[x + hi + 4 * q][y + lo] = s[q];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kPB; m += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sc[m + hi][x + lo], sr[m + hi][y + lo], acc, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 4; ++q) sd[x + hi + 4 * q][y + lo] = acc[q];
    __syncthreads();
    if (!invert_block(sd, xch) && t == 0) *flag = 1;
#pragma unroll
    for (int u = 0; u < kPB * kPB / 256; ++u) {
        const int e = t + 256 * u;
        Dn[e] = sd[e / kPB][e % kPB];
    }
}

// Pivot block k0 with inverse D: B = A after its elimination (workgroups 1 ..: a tile each), Dn =
// the inverse of the next pivot block (workgroup 0).
__global__ __launch_bounds__(256) void k_gj_step(const double* __restrict__ A, double* __restrict__ B, int n, int k0,
                                                 const double* __restrict__ D, double* __restrict__ Dn,
                                                 int* __restrict__ flag) {
    __shared__ double sc[kPB][kTU + 2];   // -(pivot columns), by depth
    __shared__ double sr[kPB][kTU + 2];   // pivot rows, then scaled
    __shared__ double sd[kPB][kPB + 2];   // D transposed
    __shared__ __attribute__((aligned(16))) double xch[kXch];
    if (blockIdx.x == 0) {
        if (k0 + kPB < n) next_block(A, n, k0, D, Dn, flag, sc, sr, sd, xch);
        return;
    }
    const int tiles = (n + kTU - 1) / kTU, tile = blockIdx.x - 1;
    const int bs = min(kPB, n - k0), i0 = tile / tiles * kTU, j0 = tile % tiles * kTU, t = threadIdx.x;
    const int w = t >> 6, lane = t & 63, lo = lane & 15, hi = lane >> 4;
    f64x4 acc[4];  // rows i0 + 16 w + hi + 4 q, columns j0 + 16 y + lo: the pivot's columns from zero
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = i0 + 16 * w + hi + 4 * q, j = j0 + 16 * y + lo;
            const double v = A[(size_t)min(i, n - 1) * n + min(j, n - 1)];
            acc[y][q] = i < n && j < n && !(j >= k0 && j < k0 + bs) ? v : 0.0;
        }
#pragma unroll
    for (int u = 0; u < kPB * kTU / 256; ++u) {
        const int e = t + 256 * u;
        const int ci = e / kPB, cm = e % kPB;
        const double c = A[(size_t)min(i0 + ci, n - 1) * n + min(k0 + cm, n - 1)];
        sc[cm][ci] = i0 + ci < n && cm < bs ? -c : 0.0;
        const int rm = e / kTU, rj = e % kTU, j = j0 + rj;
        const double r = A[(size_t)min(k0 + rm, n - 1) * n + min(j, n - 1)];
        // the pivot's own columns become its inverse: D times the identity
        sr[rm][rj] = j >= k0 && j < k0 + kPB ? (rm == j - k0 && rm < bs ? 1.0 : 0.0) : rm < bs && j < n ? r : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kPB * kPB / 256; ++u) {
        const int e = t + 256 * u;
        sd[e % kPB][e / kPB] = D[e];
    }
    __syncthreads();
    {  // wave w scales columns 16 w .. of the pivot rows
        f64x4 s[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
        for (int m = 0; m < kPB; m += 4) {
            const double b = sr[m + hi][16 * w + lo];
#pragma unroll
            for (int x = 0; x < 2; ++x)
                s[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(sd[m + hi][16 * x + lo], b, s[x], 0, 0, 0);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int q = 0; q < 4; ++q) sr[16 * x + hi + 4 * q][16 * w + lo] = s[x][q];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kPB; m += 4) {
        const double a = sc[m + hi][16 * w + lo];
#pragma unroll
        for (int y = 0; y < 4; ++y)
            acc[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, sr[m + hi][16 * y + lo], acc[y], 0, 0, 0);
    }
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = i0 + 16 * w + hi + 4 * q, j = j0 + 16 * y + lo;
            if (i < n && j < n) B[(size_t)i * n + j] = i >= k0 && i < k0 + bs ? sr[i - k0][16 * y + lo] : acc[y][q];
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

// the second buffer, two pivot blocks, the shift and the flag
static size_t scratch_count(int n) { return (size_t)n * n + 2 * kPB * kPB + 2; }

void coarse_scratch_free(Hierarchy& H) {
    if (!H.cwork) return;
    hipFree(H.cwork);
    H.cwork = nullptr;
    H.bytes -= sizeof(double) * scratch_count(H.cN);
}

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
    const size_t nn = (size_t)n * n;
    H.cN = n;
    for (auto [buf, count] : {std::pair{&H.cinv, nn}, std::pair{&H.cwork, scratch_count(n)}}) {
        if (*buf) continue;
        OPF_HIP(hipMalloc((void**)buf, sizeof(double) * count));
        H.bytes += sizeof(double) * count;
    }
    double *D0 = H.cwork + nn, *dm = D0 + 2 * kPB * kPB;
    int* flag = (int*)(dm + 1);
    // the buffers alternate from one pivot block to the next and end on cinv
    const int blocks = (n + kPB - 1) / kPB;
    double* buf[2] = {blocks & 1 ? H.cwork : H.cinv, blocks & 1 ? H.cinv : H.cwork};
    auto assemble = [&] {
        if (H.singular) hipLaunchKernelGGL(k_coarse_shift, dim3(1), dim3(1024), 0, st, o, dm);
        hipLaunchKernelGGL(k_coarse_fill, dim3(n), dim3(256), 0, st, o, H.singular ? (const double*)dm : nullptr, buf[0]);
    };
    int bad = 0;
    OPF_HIP(hipMemsetAsync(flag, 0, sizeof(int), st));
    assemble();
    const unsigned tiles = (unsigned)((n + kTU - 1) / kTU);
    hipLaunchKernelGGL(k_gj_first, dim3(1), dim3(256), 0, st, (const double*)buf[0], n, D0, flag);
    for (int q = 0; q < blocks; ++q)
        hipLaunchKernelGGL(k_gj_step, dim3(tiles * tiles + 1), dim3(256), 0, st, (const double*)buf[q & 1], buf[~q & 1], n,
                           q * kPB, (const double*)(D0 + (q & 1) * kPB * kPB), D0 + (~q & 1) * kPB * kPB, flag);
    OPF_HIP(hipGetLastError());
    OPF_HIP(hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, st));
    OPF_HIP(hipStreamSynchronize(st));
    if (!bad) return OPF_OK;
    std::vector<double> A((size_t)n * n), inv;
    assemble();
    OPF_HIP(hipMemcpyAsync(A.data(), buf[0], sizeof(double) * A.size(), hipMemcpyDeviceToHost, st));
    OPF_HIP(hipStreamSynchronize(st));
    OPF_CHECK(invert_pivoting(A, n, inv), OPF_ERR_ARG, "gmg: singular coarsest operator");
    OPF_HIP(hipMemcpyAsync(H.cinv, inv.data(), sizeof(double) * inv.size(), hipMemcpyHostToDevice, st));
    OPF_HIP(hipStreamSynchronize(st));
    return OPF_OK;
}

}  // namespace opf
