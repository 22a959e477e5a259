// FTCS heat update fast path:  u = u + coef * (d2x(u) + d2y(u) [+ d2z(u)])
// (examples/FTCS2D/FTCS-OMP.cpp:26, D2SecondOrderCentered.hpp:160-171,
//  FieldAssigner.hpp:26-86). A launch reads u^n and writes u^{n+k}; the field is
// complete, its ghosts as updatePadding leaves them, after the call. On a uniform
// mesh the reference's dx_l = dx_r = dx_c = h exactly, so D2 = ((r-c)/h - (c-l)/h)/h;
// the divisions are replaced by cheaper operations that give the same bits (below).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "constdiv.hpp"
#include "fastdiv.hpp"
#include "opf_internal.hpp"

using namespace opf;

namespace {

template <typename T>
struct FtcsArgs {
    int n[3];       // interior cells
    int e0, e1;     // storage extents (n+2)
    T coef;
    T coefh;        // coef / h^2 (FTCS_FACTORED: exact, h a power of two)
    T hh[3];        // 1/h (FTCS_MUL, FTCS_FACTORED) or h (FTCS_DIV)
    int per[3];
    int rtype[3][2];  // ghost rule per dim/side: RULE_*
    T rc1[3][2], rc2[3][2], rc3[3][2];
    ConstDivisor cd[3];     // FTCS_CDIV: the spacings
    ConstDivisor gd[3][2];  // RULE_CDIV: the divisors of the ghost rules
    int gform;              // RULE_MUL when no side needs a division, else RULE_DIV
};
// v -> (rc1 v - rc2) / rc3 (Dirichlet) by division, by the multiplication with rc3's exact
// reciprocal (rc3 a power of two: the same real number rounded once), or by const_div;
// v + rc1 (Neumann)
enum { RULE_NONE = 0, RULE_DIV = 1, RULE_ADD = 2, RULE_MUL = 3, RULE_CDIV = 4 };

// Arithmetic modes of the update (all give the reference's bits):
//  FTCS_DIV      D2 = ((r-c)/h - (c-l)/h)/h per dimension, as D2SecondOrderCentered computes it;
//  FTCS_MUL      h a power of two: the divisions become multiplications by 1/h (exact);
//  FTCS_FACTORED h a power of two and equal in every dimension. Scaling by a power of two
//                commutes with rounding (no overflow: |u| h^-2 below the largest finite
//                value), so ((r-c)*k - (c-l)*k)*k = ((r-c) - (c-l)) * k^2 exactly, the sum
//                over dimensions keeps the common factor k^2, and coef * (k^2 S) =
//                (coef k^2) * S with coef k^2 exact: u + coefh * (Dx + Dy [+ Dz]) with
//                D = (r-c) - (c-l) -- 10 operations per 3-D cell instead of 19.
//  FTCS_CDIV     any h: the divisions by h through its reciprocal (constdiv.hpp), where every
//                value is in the range that needs; elsewhere FTCS_DIV's divisions.
enum { FTCS_DIV = 0, FTCS_MUL = 1, FTCS_FACTORED = 2, FTCS_CDIV = 3 };

// x / h of dim d in an arithmetic mode
template <typename T, int MODE>
__device__ __forceinline__ T over_h(T x, const FtcsArgs<T>& a, int d) {
    if constexpr (MODE == FTCS_FACTORED) return x;
    else if constexpr (MODE == FTCS_MUL) return x * a.hh[d];
    else if constexpr (MODE == FTCS_CDIV) return const_div(x, a.cd[d]);
    else return x / a.hh[d];
}

template <typename T, int MODE>
__device__ __forceinline__ T d2(T l, T c, T r, T hh) {
    if constexpr (MODE != FTCS_DIV) return ((r - c) * hh - (c - l) * hh) * hh;
    else return ((r - c) / hh - (c - l) / hh) / hh;
}

// u^{n+1} at one cell of a 3-D field from its value and its x / y / z neighbours
template <typename T, int MODE>
__device__ __forceinline__ T ftcs3(T c, T xl, T xr, T yl, T yr, T zl, T zr, const FtcsArgs<T>& a) {
    if constexpr (MODE == FTCS_FACTORED) {
        T s = ((xr - c) - (c - xl)) + ((yr - c) - (c - yl));
        s = s + ((zr - c) - (c - zl));
        return c + a.coefh * s;
    } else {
        T s = d2<T, MODE>(xl, c, xr, a.hh[0]) + d2<T, MODE>(yl, c, yr, a.hh[1]);
        s = s + d2<T, MODE>(zl, c, zr, a.hh[2]);
        return c + a.coef * s;
    }
}

template <typename T>
__device__ __forceinline__ T rule(const FtcsArgs<T>& a, int d, int s, T v) {
    const int t = a.rtype[d][s];
    if (t == RULE_ADD) return v + a.rc1[d][s];
    if (t == RULE_NONE) return v;
    const T x = a.rc1[d][s] * v - a.rc2[d][s];
    if (t == RULE_MUL) return x * a.rc3[d][s];
    return x / a.rc3[d][s];
}

// The ghost rules of a launch in one form, (c1 v - c2) over c3 with c1 = c3 = 1 where the rule only
// adds (both exact): over c3 a multiplication by its exact reciprocal, a const_div or a division.
// One straight line for every side, so that the lanes of a wave take theirs together.
template <typename T>
struct SideRule {
    T c1, c2, c3;
    ConstDivisor cd;
};
template <typename T>
__device__ __forceinline__ SideRule<T> side_rule(const FtcsArgs<T>& a, int d, int s) {
    const int t = a.rtype[d][s];
    SideRule<T> r{T(1), T(0), T(1), {}};
    if (t == RULE_ADD) r.c2 = -a.rc1[d][s];
    if (t == RULE_DIV || t == RULE_MUL || t == RULE_CDIV) r.c1 = a.rc1[d][s], r.c2 = a.rc2[d][s], r.c3 = a.rc3[d][s];
    if (t == RULE_CDIV) r.cd = a.gd[d][s];
    return r;
}
// again: RULE_CDIV met a value outside const_div's range
template <int FORM, typename T>
__device__ __forceinline__ T ghost_value(T c1, T c2, T c3, double h, double y, T v, bool& again) {
    const T x = c1 * v - c2;
    if constexpr (FORM == RULE_MUL) return x * c3;
    else if constexpr (FORM == RULE_DIV) return x / c3;
    else {
        const T q = const_div(x, ConstDivisor{h, y});
        if constexpr (sizeof(T) == 4) again |= div_subnormal(q);
        else again |= div_key(v) < kDivLow;
        return c3 < T(0) ? -q : q;  // h = |c3|
    }
}

// the value of the next / previous lane of the wave (0 in the last / first lane)
template <int CTRL>
__device__ __forceinline__ int dpp32(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
    if constexpr (sizeof(T) == 4) return __int_as_float(dpp32<CTRL>(__float_as_int(v)));
    else return __hiloint2double(dpp32<CTRL>(__double2hiint(v)), dpp32<CTRL>(__double2loint(v)));
}
// c ? x : y of two loaded values (a conditional between array elements would pick an address and
// put the array in memory)
template <typename T>
__device__ __forceinline__ T pick(bool c, T x, T y) {
    return c ? x : y;
}
template <typename T>
__device__ __forceinline__ T lane_next(T v) { return dpp<0x130>(v); }
template <typename T>
__device__ __forceinline__ T lane_prev(T v) { return dpp<0x138>(v); }

// 2-D steps in registers. A workgroup holds a region of 64 XW x NW RW cells: lane l of a wave
// the XW neighbouring cells l XW .. in x, wave w the RW rows w RW .., so that y neighbours are
// registers, x neighbours are registers or one lane away (DPP, no LDS), and only the first and
// last row of each wave pass through LDS, with one barrier a step. It advances the region nt
// steps and writes the tx x ty tile in its middle; the values at distance < s from an open region
// edge are stale after s steps, which never reaches the tile. A difference of neighbours, and its
// quotient by h, is formed once and serves both cells. On a non-periodic side the region starts
// at, or contains, the ghost layer, which is refilled after every step from the fresh cells with
// the BC rules, x first, then y (the corner composition of updatePadding); the rows are placed so
// that a y ghost and its source cell belong to one wave. Periodic sides read wrapped cells. The
// tile's ghost images are written with it, so the output field is complete.
// Per cell and step the operations and their order are those of D2 in the reference, so the bits
// are too. FP64 issue bounds the large grids (7 operations and 2 lane moves a cell and step, 19 and
// 2 with const_div, over the share of the region that is tile), the barrier and the launch the
// small ones. Against LDS tiles of the values (32 x 32, 4 steps; 8 x 8, 5 steps): 256^2 Dirichlet
// 1.61 -> 0.75 us a step, 1500 x 1100 with const_div 12.3 -> 4.5 (0.13 -> 0.37 T cell-updates/s),
// 4096^2 periodic 42 -> 10.1 (0.40 -> 1.66 T/s).
template <typename T, int MODE, int XW, int RW, int NW>
__global__ __launch_bounds__(64 * NW) void ftcs2d_strip_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                               FtcsArgs<T> a, int nt, int tx, int ty) {
    static_assert(XW <= 2, "the ghost columns are a lane's first or second");
    constexpr int WX = 64 * XW, WY = RW * NW;
    __shared__ T edge[2][NW][2][XW][64];  // first and last row of every wave, double-buffered
    const int n0 = a.n[0], n1 = a.n[1];
    const int tilesx = (n0 + tx - 1) / tx;
    const int tb = (int)xcd_block(blockIdx.x, gridDim.x);  // x-neighbouring tiles share an XCD's L2
    const int x0 = (tb % tilesx) * tx, y0 = (tb / tilesx) * ty;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // region origin; non-periodic sides: x from the ghost column on, y from the ghost row or up to it
    int lox = x0 - nt, loy = y0 - nt;
    if (!a.per[0]) lox = max(lox, -1);
    if (!a.per[1]) {
        loy = max(loy, -1);
        if (loy + WY > n1 + 1) {
            loy = n1 + 1 - WY;  // the upper ghost row is the last of the last wave
            if (loy < -1) loy = (n1 + 1) % RW == 0 ? -2 : -1;  // both ghost rows inside
        }
    }
    const int gx0 = lox + lane * XW, gy0 = loy + w * RW;
    T u[RW][XW];
    {
        int ox[XW];
#pragma unroll
        for (int k = 0; k < XW; ++k) {
            int gx = gx0 + k;
            if (a.per[0]) gx = ((gx % n0) + n0) % n0;
            ox[k] = min(max(gx, -1), n0) + 1;
        }
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            int gy = gy0 + r;
            if (a.per[1]) gy = ((gy % n1) + n1) % n1;
            const T* row = in + (long long)a.e0 * (min(max(gy, -1), n1) + 1);
#pragma unroll
            for (int k = 0; k < XW; ++k) u[r][k] = row[ox[k]];
        }
    }
    // the ghosts of this wave: columns (uniform over the workgroup), rows (of this wave)
    const bool xlo = !a.per[0] && lox <= -1, xhi = !a.per[0] && lox + WX > n0;
    const int rlo = a.per[1] ? -1 : -1 - gy0, rhi = a.per[1] ? -1 : n1 - gy0;
    const bool ylo = rlo >= 0 && rlo < RW, yhi = rhi >= 0 && rhi < RW;
    const bool ghosts = xlo || xhi || ylo || yhi;
    constexpr int FORM = MODE == FTCS_CDIV ? RULE_CDIV : MODE == FTCS_DIV ? RULE_DIV : RULE_MUL;
    // x rule of this lane's column (a lane holds at most one ghost column of each side)
    const bool hilane = gx0 + XW > n0;
    const SideRule<T> rl = side_rule(a, 0, 0), rh = side_rule(a, 0, 1), ryl = side_rule(a, 1, 0), ryh = side_rule(a, 1, 1);
    const T xc1 = hilane ? rh.c1 : rl.c1, xc2 = hilane ? rh.c2 : rl.c2, xc3 = hilane ? rh.c3 : rl.c3;
    const double xh = hilane ? rh.cd.h : rl.cd.h, xy = hilane ? rh.cd.y : rl.cd.y;
    // refills the ghosts of v; true when RULE_CDIV met a value out of its range (v is unchanged then)
    auto refill = [&](auto F, T(&v)[RW][XW]) __attribute__((always_inline)) -> bool {
        constexpr int FM = decltype(F)::value;
        bool again = false;
        if (xlo || xhi) {
            // the lower ghost is a lane's first column, its source the next one; the upper ghost's
            // source the previous column
            T g[RW][XW];
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const T nx = XW > 1 ? v[r][XW > 1 ? 1 : 0] : lane_next(v[r][0]);
                const T pv = lane_prev(v[r][XW - 1]);
                g[r][0] = ghost_value<FM>(xc1, xc2, xc3, xh, xy, hilane ? pv : nx, again);
                if constexpr (XW > 1) g[r][1] = ghost_value<FM>(xc1, xc2, xc3, xh, xy, v[r][0], again);
            }
            if (FM == RULE_CDIV && __any(again)) return true;
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                v[r][0] = pick(gx0 == -1 || gx0 == n0, g[r][0], v[r][0]);
                if constexpr (XW > 1) v[r][1] = pick(gx0 + 1 == n0, g[r][1], v[r][1]);
            }
        }
        if (ylo) {
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                T src = v[1][k];
#pragma unroll
                for (int r = 1; r + 1 < RW; ++r) src = pick(r == rlo, v[r + 1][k], src);
                T g = ghost_value<FM>(ryl.c1, ryl.c2, ryl.c3, ryl.cd.h, ryl.cd.y, src, again);
                if (FM == RULE_CDIV && __any(again)) g = ghost_value<RULE_DIV>(ryl.c1, ryl.c2, ryl.c3, 1., 1., src, again);
#pragma unroll
                for (int r = 0; r + 1 < RW; ++r) v[r][k] = pick(r == rlo, g, v[r][k]);
            }
        }
        if (yhi) {
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                T src = v[0][k];
#pragma unroll
                for (int r = 2; r < RW; ++r) src = pick(r == rhi, v[r - 1][k], src);
                T g = ghost_value<FM>(ryh.c1, ryh.c2, ryh.c3, ryh.cd.h, ryh.cd.y, src, again);
                if (FM == RULE_CDIV && __any(again)) g = ghost_value<RULE_DIV>(ryh.c1, ryh.c2, ryh.c3, 1., 1., src, again);
#pragma unroll
                for (int r = 1; r < RW; ++r) v[r][k] = pick(r == rhi, g, v[r][k]);
            }
        }
        return false;
    };
    bool slow = false;  // FTCS_CDIV, FP64: a value outside the range for the whole launch
    if constexpr (MODE == FTCS_CDIV && sizeof(T) == 8) {
        bool bad = false;
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) bad |= div_unsafe(u[r][k]);
        slow = __syncthreads_or(bad);
    }
    for (int s = 0; s < nt; ++s) {
        auto& e = edge[s & 1];
        if constexpr (NW > 1) {
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                e[w][0][k][lane] = u[0][k];
                e[w][1][k][lane] = u[RW - 1][k];
            }
        }
        T v[RW][XW];  // the second x differences, then the new values
        // returns whether a float quotient was subnormal
        auto xpart = [&](auto M) __attribute__((always_inline)) -> bool {
            constexpr int MD = decltype(M)::value;
            bool sub = false;
            auto quo = [&](T x) __attribute__((always_inline)) -> T {
                const T q = over_h<T, MD>(x, a, 0);
                if constexpr (MD == FTCS_CDIV && sizeof(T) == 4) sub |= div_subnormal(q);
                return q;
            };
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                T qx[XW];
#pragma unroll
                for (int k = 0; k < XW; ++k) {
                    const T right = k + 1 < XW ? u[r][k + 1 < XW ? k + 1 : 0] : lane_next(u[r][0]);
                    qx[k] = quo(right - u[r][k]);
                }
                const T left = lane_prev(qx[XW - 1]);
#pragma unroll
                for (int k = 0; k < XW; ++k) v[r][k] = quo(qx[k] - (k > 0 ? qx[k > 0 ? k - 1 : 0] : left));
            }
            return sub;
        };
        T dn[XW], up[XW];  // the rows before the first and after the last
        auto ypart = [&](auto M) __attribute__((always_inline)) -> bool {
            constexpr int MD = decltype(M)::value;
            bool sub = false;
            auto quo = [&](T x) __attribute__((always_inline)) -> T {
                const T q = over_h<T, MD>(x, a, 1);
                if constexpr (MD == FTCS_CDIV && sizeof(T) == 4) sub |= div_subnormal(q);
                return q;
            };
            T qy[XW];
#pragma unroll
            for (int k = 0; k < XW; ++k) qy[k] = quo(u[0][k] - dn[k]);
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int k = 0; k < XW; ++k) {
                    const T qn = quo((r + 1 < RW ? u[r + 1 < RW ? r + 1 : 0][k] : up[k]) - u[r][k]);
                    const T dy = quo(qn - qy[k]);
                    qy[k] = qn;
                    v[r][k] = u[r][k] + (MD == FTCS_FACTORED ? a.coefh : a.coef) * (v[r][k] + dy);
                }
            return sub;
        };
        bool sub = xpart(std::integral_constant<int, MODE>{});  // needs no other wave: while the rows are on their way
        if constexpr (NW > 1) {
            __syncthreads();
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                dn[k] = e[max(w - 1, 0)][1][k][lane];
                up[k] = e[min(w + 1, NW - 1)][0][k][lane];
            }
        } else {
#pragma unroll
            for (int k = 0; k < XW; ++k) dn[k] = u[0][k], up[k] = u[RW - 1][k];
        }
        bool again = slow;
        if constexpr (MODE == FTCS_CDIV && sizeof(T) == 8) {
            unsigned m = 0xffffffffu;
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                m = min(m, min(div_key(dn[k]), div_key(up[k])));
#pragma unroll
                for (int r = 0; r < RW; ++r) m = min(m, div_key(u[r][k]));
            }
            again |= __any(m < kDivLow);
        }
        if (!again) sub |= ypart(std::integral_constant<int, MODE>{});
        if constexpr (MODE == FTCS_CDIV) {
            if (sizeof(T) == 4) again = __any(sub);
            if (again) {
                xpart(std::integral_constant<int, FTCS_DIV>{});
                ypart(std::integral_constant<int, FTCS_DIV>{});
            }
        }
        if (ghosts) {
            bool done = false;
            if (FORM == RULE_MUL && a.gform == RULE_MUL) done = !refill(std::integral_constant<int, RULE_MUL>{}, v);
            else if (FORM == RULE_CDIV && !again) done = !refill(std::integral_constant<int, RULE_CDIV>{}, v);
            if (!done) refill(std::integral_constant<int, RULE_DIV>{}, v);
        }
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) u[r][k] = v[r][k];
    }
    // the tile with the ghost positions beyond it: its own columns and, on non-periodic sides, the
    // ghost columns; periodic images of the first and last column and row
    const int x1 = min(x0 + tx, n0), y1 = min(y0 + ty, n1);
    const int xa = !a.per[0] && x0 == 0 ? -1 : x0, xb = !a.per[0] && x1 == n0 ? n0 + 1 : x1;
    const int ya = !a.per[1] && y0 == 0 ? -1 : y0, yb = !a.per[1] && y1 == n1 ? n1 + 1 : y1;
    const bool imlo = a.per[0] && x1 == n0, imhi = a.per[0] && x0 == 0;  // images at -1 and at n
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int gy = gy0 + r;
        if (gy < ya || gy >= yb) continue;
        auto put = [&](int y) __attribute__((always_inline)) {
            T* row = out + (long long)a.e0 * (y + 1) + 1;
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                const int gx = gx0 + k;
                if (gx >= xa && gx < xb) row[gx] = u[r][k];
                if (imlo && gx == n0 - 1) row[-1] = u[r][k];
                if (imhi && gx == 0) row[n0] = u[r][k];
            }
        };
        put(gy);
        if (a.per[1]) {
            if (gy == n1 - 1) put(-1);
            if (gy == 0) put(n1);
        }
    }
}

// 3-D single step, LDS-tiled: a 64 x NTY workgroup owns a 64 x (NTY * RY) x-y
// tile (each thread RY rows) and marches ZC planes in z. The current plane of
// the tile and its one-cell x/y halo sit in LDS (double-buffered, one barrier
// per plane); each thread keeps its cells' z-1 / z / z+1 values in registers
// and loads plane k+2 while plane k is computed. The input's ghost layer
// supplies the halo of boundary tiles, so loads never wrap; the kernel writes
// interior cells only and the host loop refills the output's ghosts before
// they are read. Per cell: d2x + d2y, then + d2z, then u + coef * s -- the
// arithmetic every FTCS kernel here uses, so all give the same bits.
// Launch shape swept at 512^3 on MI355X (64 x 8 threads, 2 rows each, 8 planes).
constexpr int FT3_TX = 64, FT3_NTY = 8, FT3_RY = 2, FT3_TY = FT3_NTY * FT3_RY, FT3_ZC = 8;

template <typename T, int MODE, int ZC, int NTY, int RY>
__global__ __launch_bounds__(64 * NTY) void ftcs3d_lds_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                              FtcsArgs<T> a) {
    constexpr int TY = NTY * RY;
    static_assert(128 + 2 * TY <= 64 * NTY, "one halo element per thread at most");
    __shared__ T lds[2][TY + 2][FT3_TX + 2];
    const int tx = threadIdx.x, ty = threadIdx.y, t = ty * 64 + tx;
    // tile of this block: the flat id through xcd_block, so that each XCD's L2 holds a
    // contiguous slab whose x / y halo lines its own tiles share
    const uint32_t L = xcd_block(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                                 gridDim.x * gridDim.y * gridDim.z);
    const int x0 = (int)(L % gridDim.x) * FT3_TX, y0 = (int)((L / gridDim.x) % gridDim.y) * TY,
              k0 = (int)(L / (gridDim.x * gridDim.y)) * ZC;
    const int kend = min(k0 + ZC, a.n[2]);
    const long long sy = a.e0, sz = (long long)a.e0 * a.e1;
    const int i = x0 + tx;
    // storage index of (x, y, k) (ghost layer at -1 and n)
    auto at = [&](int x, int y, int k) { return (long long)(x + 1) + sy * (y + 1) + sz * (k + 1); };
    // valid storage positions: interior and the ghost layer
    auto ok = [&](int x, int y) { return x >= -1 && x <= a.n[0] && y >= -1 && y <= a.n[1]; };
    // this thread's halo element: rows y0 - 1 and y0 + TY (threads 0..127), then the
    // columns x0 - 1 and x0 + TX over the tile's rows; corners are not read
    int hx = 0, hy = 0, hlx = 0, hly = 0;
    if (t < 128) {
        hx = x0 + (t & 63);
        hy = t < 64 ? y0 - 1 : y0 + TY;
        hlx = (t & 63) + 1;
        hly = t < 64 ? 0 : TY + 1;
    } else if (t < 128 + 2 * TY) {
        const int q = t - 128, side = q / TY, r = q % TY;
        hx = side == 0 ? x0 - 1 : x0 + FT3_TX;
        hy = y0 + r;
        hlx = side == 0 ? 0 : FT3_TX + 1;
        hly = r + 1;
    }
    const bool hl = t < 128 + 2 * TY && ok(hx, hy);
    bool own[RY];
    T zm[RY], zc[RY], zp[RY], zq[RY];
    T hp = T(0), hq = T(0);
#pragma unroll
    for (int r = 0; r < RY; ++r) {
        const int j = y0 + ty * RY + r;
        own[r] = ok(i, j);
        zm[r] = own[r] ? in[at(i, j, k0 - 1)] : T(0);
        zc[r] = own[r] ? in[at(i, j, k0)] : T(0);
        zp[r] = own[r] ? in[at(i, j, k0 + 1)] : T(0);  // k0 + 1 <= n[2]: the ghost plane at most
        lds[0][ty * RY + r + 1][tx + 1] = zc[r];
    }
    if (hl) {
        lds[0][hly][hlx] = in[at(hx, hy, k0)];
        hp = in[at(hx, hy, k0 + 1)];
    }
    __syncthreads();
    int cur = 0;
    for (int k = k0; k < kend; ++k) {
        // plane k + 2 is loaded one step ahead of its use (only while a next step needs it)
        if (k + 1 < kend) {
#pragma unroll
            for (int r = 0; r < RY; ++r) zq[r] = own[r] ? in[at(i, y0 + ty * RY + r, k + 2)] : T(0);
            if (hl) hq = in[at(hx, hy, k + 2)];
        }
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int ly = ty * RY + r + 1, j = y0 + ly - 1;
            if (i >= a.n[0] || j >= a.n[1]) continue;
            const T c = zc[r];
            out[at(i, j, k)] = ftcs3<T, MODE>(c, lds[cur][ly][tx], lds[cur][ly][tx + 2], lds[cur][ly - 1][tx + 1],
                                              lds[cur][ly + 1][tx + 1], zm[r], zp[r], a);
        }
        const int nxt = cur ^ 1;
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            lds[nxt][ty * RY + r + 1][tx + 1] = zp[r];
            zm[r] = zc[r];
            zc[r] = zp[r];
            zp[r] = zq[r];
        }
        if (hl) lds[nxt][hly][hlx] = hp;
        hp = hq;
        __syncthreads();
        cur = nxt;
    }
}

// 3-D temporal blocking, K steps per launch. A workgroup owns a TX x TY column
// of the x-y plane and the z chunk [z0, z0 + zc) and streams the planes of u^n
// with a K-cell halo in x and y. Every thread owns fixed positions of the
// (TX+2K) x (TY+2K) region and keeps, for each, the last three planes of
// levels 0 .. K-1 (u^n .. u^{n+K-1}) in registers, so the centre and the z
// neighbours never go through LDS; LDS holds only the current plane of each
// level (double-buffered), read for the x and y neighbours. Step zz stores
// level-0 plane zz and computes level L at plane zz - L (L = 1 .. K) on the
// region shrunk by L cells; level K is exactly the tile and goes straight to
// global memory. One barrier per step separates a step's LDS writes from the
// next step's reads (levels read the plane the level below wrote one step
// earlier). Level-0 planes are loaded three planes ahead; the unroll by 3 keeps
// the history slots static; every load is unconditional so the compiler keeps
// counted load waits.
// Periodic dimensions wrap the halo to interior cells (the input's ghosts are
// never read). Dirichlet / Neumann dimensions (ALLPER = false) clamp the halo to
// the ghost layer: level 0 reads the input's ghosts (refilled by the host before
// the launch), and the ghosts of the intermediate levels 1 .. K-1 are rebuilt
// from the level's fresh boundary cells with the BC rules, as updatePadding
// does after every step: x / y face ghosts in LDS at the start of the next step
// (one extra barrier, only in workgroups whose region reaches such a side), z
// ghost planes in the register history when the level computes plane 0 or
// reaches plane n. The 7-point stencil reads face ghosts only, so edge and
// corner ghosts are never needed; region cells beyond the ghost layer hold
// values that never reach a valid cell. The output's ghosts are left stale and
// refilled by the host loop before anything reads them. Per cell and step the
// arithmetic is that of ftcs3d_lds_kernel, so the result has the same bits as K
// single steps.
template <typename T, int MODE, int TX, int TY, int NT, int K, bool XCD, bool ALLPER>
__global__ __launch_bounds__(NT) void ftcs3d_tb_kernel(const T* __restrict__ in, T* __restrict__ out, FtcsArgs<T> a,
                                                       int zc) {
    static_assert(K >= 2, "one step per launch is ftcs3d_lds_kernel");
    constexpr int RX = TX + 2 * K, RY = TY + 2 * K, RP = RX * RY;
    constexpr int NL = (RP + NT - 1) / NT;
    constexpr int PF = 3;
    __shared__ T lds[K][2][NL * NT];  // current plane of levels 0 .. K-1
    const int tilesx = (a.n[0] + TX - 1) / TX, tilesy = (a.n[1] + TY - 1) / TY;
    int b = XCD ? (int)xcd_block(blockIdx.x, gridDim.x) : (int)blockIdx.x;  // neighbouring tiles share an XCD's L2
    const int x0 = (b % tilesx) * TX;
    b /= tilesx;
    const int y0 = (b % tilesy) * TY;
    const int z0 = (b / tilesy) * zc;
    const int z1 = min(z0 + zc, a.n[2]);
    const long long sz = (long long)a.e0 * a.e1;
    const int tid = threadIdx.x;
    // this thread's region positions: input offset, region coordinates, output offset;
    // gh: 0 interior, 1 / 2 the low / high x face ghost, 3 / 4 the low / high y face ghost
    int off[NL], lxm[NL], lym[NL], gh[NL];
    bool valid[NL], inr[NL];
    long long oo[NL];
#pragma unroll
    for (int m = 0; m < NL; ++m) {
        const int e = tid + m * NT;
        valid[m] = e < RP;
        const int ee = valid[m] ? e : 0;
        const int lx = ee % RX, ly = ee / RX;
        lxm[m] = lx;
        lym[m] = ly;
        int gx = x0 - K + lx, gy = y0 - K + ly;
        gh[m] = 0;
        if (ALLPER || a.per[0]) gx = (gx % a.n[0] + a.n[0]) % a.n[0];
        if (ALLPER || a.per[1]) gy = (gy % a.n[1] + a.n[1]) % a.n[1];
        if (!ALLPER) {
            const bool inx = gx >= 0 && gx < a.n[0], iny = gy >= 0 && gy < a.n[1];
            if (iny && (gx == -1 || gx == a.n[0])) gh[m] = gx < 0 ? 1 : 2;
            if (inx && (gy == -1 || gy == a.n[1])) gh[m] = gy < 0 ? 3 : 4;
            gx = min(max(gx, -1), a.n[0]);  // clamped: inside the storage
            gy = min(max(gy, -1), a.n[1]);
        }
        off[m] = (gx + 1) + a.e0 * (gy + 1);
        const int i = x0 + lx - K, j = y0 + ly - K;
        inr[m] = i < a.n[0] && j < a.n[1];
        oo[m] = (long long)(i + 1) + (long long)a.e0 * (j + 1);
    }
    // position m takes part in level L (region shrunk by L cells)
    auto at_level = [&](int m, int L) {
        return valid[m] && lxm[m] >= L && lxm[m] <= RX - 1 - L && lym[m] >= L && lym[m] <= RY - 1 - L;
    };
    // the region reaches a non-periodic x / y side: face ghosts to rebuild (uniform over the block)
    const bool edge = !ALLPER && ((!a.per[0] && (x0 - K < 0 || x0 + TX + K > a.n[0])) ||
                                  (!a.per[1] && (y0 - K < 0 || y0 + TY + K > a.n[1])));
    const bool zper = ALLPER || a.per[2];
    const int zb = z0 - K, ze = z1 + K;  // level-0 planes zb .. ze - 1
    T pre[PF][NL], hist[K][NL][3];       // history slot of plane p: (p - zb) % 3
    auto load = [&](T(&r)[NL], int z) {
        if (zper) z = (z % a.n[2] + a.n[2]) % a.n[2];
        else z = min(max(z, -1), a.n[2]);
        const T* p = in + sz * (z + 1);
#pragma unroll
        for (int m = 0; m < NL; ++m) r[m] = p[off[m]];
    };
#pragma unroll
    for (int u = 0; u < PF; ++u) load(pre[u], min(zb + u, ze - 1));
    for (int zz0 = zb; zz0 < ze; zz0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int zz = zz0 + u;  // (zz - zb) % 3 == u
            if (zz >= ze) break;     // uniform over the block
            __syncthreads();
            T* w0 = lds[0][zz & 1];
#pragma unroll
            for (int m = 0; m < NL; ++m) {
                hist[0][m][u] = pre[u][m];
                w0[tid + m * NT] = pre[u][m];
            }
            load(pre[u], min(zz + PF, ze - 1));
            if (!ALLPER && edge) {
                // face ghosts of the planes levels 1 .. K-1 wrote in the last step, from their
                // boundary cells (read after the barrier above), before the next level reads them
#pragma unroll
                for (int L = 1; L < K; ++L) {
                    if (zz - 1 < z0 - K + 2 * L) continue;  // level L had no plane yet (uniform)
                    T* P = lds[L][(zz - 1 - L) & 1];
#pragma unroll
                    for (int m = 0; m < NL; ++m) {
                        if (!gh[m] || !at_level(m, L)) continue;
                        const int e = tid + m * NT;
                        const int g = gh[m];
                        const int nb = g == 1 ? e + 1 : g == 2 ? e - 1 : g == 3 ? e + RX : e - RX;
                        P[e] = rule(a, g <= 2 ? 0 : 1, (g - 1) & 1, P[nb]);
                    }
                }
                __syncthreads();
            }
#pragma unroll
            for (int L = 1; L <= K; ++L) {
                if (zz < z0 - K + 2 * L) break;  // plane zz - L of level L not computable yet (uniform)
                // level L-1 planes zz-L+1, zz-L, zz-L-1 sit in slots sp, sc, sm
                const int sp = ((u - L + 1) % 3 + 3) % 3, sc = ((u - L) % 3 + 3) % 3, sm = ((u - L - 1) % 3 + 3) % 3;
                const T* P = lds[L - 1][(zz - L) & 1];
                const int pz = zz - L;  // the plane level L computes
#pragma unroll
                for (int m = 0; m < NL; ++m) {
                    if (L < K ? !at_level(m, L) : !(at_level(m, K) && inr[m])) continue;
                    const int e = tid + m * NT;
                    const T c = hist[L - 1][m][sc];
                    T v = ftcs3<T, MODE>(c, P[e - 1], P[e + 1], P[e - RX], P[e + RX], hist[L - 1][m][sm],
                                         hist[L - 1][m][sp], a);
                    if (L < K) {
                        if (!zper && pz == a.n[2]) v = rule(a, 2, 1, hist[L][m][sm]);  // ghost plane n
                        hist[L][m][sc] = v;
                        if (!zper && pz == 0) hist[L][m][sm] = rule(a, 2, 0, v);  // ghost plane -1
                        lds[L][(zz - L) & 1][e] = v;
                    } else {
                        out[sz * (zz - K + 1) + oo[m]] = v;
                    }
                }
            }
        }
    }
}

// Launches of the 2-D kernel: the region (cells in x per lane, rows per wave, waves), the steps per
// launch and the tile that is left of the region. Per step a launch costs
//   S2_LAUNCH / nt + max(alone, tiles / CUs * shared)
// with the measured time of one step of one workgroup when it has a CU to itself (alone: the
// barrier and the waves' latency) and when several share one (shared: instruction issue), about
// 1.8 times that with const_div. More steps a launch save launches and lose tile. FP64, us per
// step: 256^2 periodic 64 x 32 region with 12 steps 0.65 (64 x 64, 24 steps: 0.71); 700^2 64 x 64,
// 10 steps 2.0 (64 x 32, 6: 2.1); 4096^2 128 x 64, 10 steps 10.1 (64 x 64: 14.0, 64 x 32: 19.8).
// With const_div the 128 x 64 region holds too few waves (117 registers): 2000^2 7.7 against 7.3.
constexpr int S2_XW[3] = {1, 1, 2}, S2_RW[3] = {4, 8, 8}, S2_NW[3] = {8, 8, 8};
constexpr double S2_ALONE[3] = {0.33, 0.55, 1.3}, S2_SHARED[3] = {0.31, 0.49, 0.74}, S2_LAUNCH = 4.2;
constexpr int S2_MOST = 128;  // steps a launch takes at most (the range const_div is given, div_range)
struct Strip2d {
    int cfg = 0;
    int nt = 1, tx = 1, ty = 1;  // steps, tile
};

Strip2d strip_plan(const int n[3], const int per[3], int nsteps, int tblock, bool div, int cus) {
    Strip2d best;
    double cost = 0;
    for (int c = 0; c < (div ? 2 : 3); ++c) {
        const int wx = 64 * S2_XW[c], wy = S2_RW[c] * S2_NW[c];
        const bool allx = !per[0] && n[0] + 2 <= wx, ally = !per[1] && n[1] + 3 <= wy;  // no halo in that dim
        const int most = std::min(nsteps, allx && ally ? S2_MOST : (ally ? wx : allx ? wy : std::min(wx, wy)) / 2 - 2);
        // 1 (when asked for), else 2, 3 .. 12, 24, .. and the most
        for (int nt = tblock == 1 ? 1 : std::min(2, most);;) {
            const int tx = allx ? n[0] : wx - 2 * nt, ty = ally ? n[1] : wy - 2 * nt;
            const double tiles = (double)((n[0] + tx - 1) / tx) * ((n[1] + ty - 1) / ty);
            const double t = S2_LAUNCH / nt +
                             (div ? 1.8 : 1.0) * std::max(S2_ALONE[c], tiles / cus * S2_SHARED[c]);
            if (cost == 0 || t < cost) {
                cost = t;
                best.cfg = c;
                best.nt = nt;
            }
            if (tblock == 1 || nt >= most) break;
            nt = std::min(most, nt < 12 ? nt + 1 : 2 * nt);
        }
    }
    // the steps spread evenly over that many launches
    const int launches = (nsteps + best.nt - 1) / best.nt;
    best.nt = (nsteps + launches - 1) / launches;
    const int wx = 64 * S2_XW[best.cfg], wy = S2_RW[best.cfg] * S2_NW[best.cfg];
    best.tx = !per[0] && n[0] + 2 <= wx ? n[0] : wx - 2 * best.nt;
    best.ty = !per[1] && n[1] + 3 <= wy ? n[1] : wy - 2 * best.nt;
    return best;
}

// 3-D blocked launch shape per precision (swept at 512^3 on MI355X): TX x TY
// columns, NT threads, K steps per launch (a remainder of two steps takes one K = 2
// launch of the same tile, one step the single-step kernel); the z chunk is chosen per
// launch (ftcs_t)
template <typename T>
struct Ftcs3dCfg;
template <>
struct Ftcs3dCfg<double> {
    static constexpr int TX = 64, TY = 32, NT = 1024, K = 3;
    static constexpr bool XCD = true;
};
template <>
struct Ftcs3dCfg<float> {
    static constexpr int TX = 128, TY = 32, NT = 1024, K = 3;
    static constexpr bool XCD = true;
};

// Steps the next launch of a 3-D field advances. tblock = 1 forces single steps.
int launch_steps3(int dtype, long long plane, int remaining, int tblock) {
    const int k3 = dtype == OPF_F64 ? Ftcs3dCfg<double>::K : Ftcs3dCfg<float>::K;
    return tblock != 1 && plane < (1LL << 31) && remaining >= 2 ? std::min(k3, remaining) : 1;
}

bool is_pow2(double h) {
    if (!(h > 0)) return false;
    int e;
    double m = std::frexp(h, &e);
    return m == 0.5;
}

// ext_spare: null = the field's own second buffer (allocated on first use);
// otherwise a caller-provided device buffer of at least f->nbytes used as the
// second time level, with the result copied back into f->data at the end.
template <typename T>
int ftcs_t(opf_field* f, double coef, int nsteps, int tblock, void* ext_spare = nullptr) {
    const opf_field_desc& d = f->d;
    const opf_mesh* m = f->mesh;
    FtcsArgs<T> a{};
    bool pow2 = true;
    for (int q = 0; q < 3; ++q) {
        a.n[q] = q < d.dim ? d.local_end[q] - d.local_start[q] : 1;
        a.per[q] = 0;
    }
    a.e0 = d.extent[0];
    a.e1 = d.extent[1];
    a.coef = (T)coef;
    GhostInfo gi;
    OPF_TRY(build_ghost_info(f, &gi));
    for (int q = 0; q < d.dim; ++q) {
        OPF_CHECK(d.loc[q] == OPF_LOC_CENTER, OPF_ERR_UNSUPPORTED, "ftcs: centre location required");
        OPF_CHECK(d.padding == 1 && d.ext[q][0] == 1 && d.ext[q][1] == 1, OPF_ERR_UNSUPPORTED,
                  "ftcs: padding = ext = 1 required");
        OPF_CHECK(m->uniform[q], OPF_ERR_UNSUPPORTED, "ftcs: uniform mesh required");
        OPF_CHECK(d.assign_start[q] == d.local_start[q] && d.assign_end[q] == d.local_end[q] && d.local_start[q] == 0,
                  OPF_ERR_UNSUPPORTED, "ftcs: assignable range must be the whole interior");
        a.per[q] = gi.per[q];
        for (int s = 0; s < 2; ++s) {
            int t = d.bc_type[q][s];
            OPF_CHECK(t == OPF_BC_DIRC || t == OPF_BC_NEUM || t == OPF_BC_PERIODIC, OPF_ERR_UNSUPPORTED,
                      "ftcs: bc %d unsupported", t);
            const GhostRule& r = gi.rule[q][s][0];
            a.rtype[q][s] = r.type == 1 ? RULE_DIV : r.type == 2 ? RULE_ADD : RULE_NONE;
            a.rc1[q][s] = (T)r.c1;
            a.rc2[q][s] = (T)r.c2;
            a.rc3[q][s] = (T)r.c3;
        }
        double h = m->h[q];
        // D2 on a uniform mesh: dx_l = (h+h)*0.5 = h, dx_r = h, dx_c = h exactly
        pow2 &= is_pow2(h);
        a.hh[q] = (T)h;
    }
    bool same = true;
    for (int q = 1; q < d.dim; ++q) same &= m->h[q] == m->h[0];
    int mode = !pow2 ? FTCS_DIV : same ? FTCS_FACTORED : FTCS_MUL;
    if (mode == FTCS_DIV && d.dim == 2) {
        bool ok = std::is_same<T, float>::value || div_range(m->h, d.dim, coef, S2_MOST);
        for (int q = 0; q < d.dim; ++q) {
            a.cd[q].h = (double)a.hh[q];
            a.cd[q].y = 1.0 / a.cd[q].h;
            for (int s = 0; s < 2; ++s) {  // a boundary's constant is 0 or well inside the range
                const GhostRule& r = gi.rule[q][s][0];
                const double c = std::fabs(r.type == 1 ? r.c2 / r.c3 : r.type == 2 ? r.c1 : 0.0);
                ok &= c == 0.0 || (c >= 0x1p-400 && c <= 0x1p400);
            }
        }
        if (ok) mode = FTCS_CDIV;
    }
    // the Dirichlet rules' divisors, in the form the arithmetic mode takes: reciprocals when every
    // one of them is a power of two
    bool rpow2 = mode != FTCS_CDIV;
    for (int q = 0; q < d.dim; ++q)
        for (int s = 0; s < 2; ++s) {
            const double c3 = std::fabs((double)a.rc3[q][s]);
            if (a.rtype[q][s] == RULE_DIV) rpow2 &= is_pow2(c3) && c3 >= 0x1p-100 && c3 <= 0x1p100;
        }
    a.gform = rpow2 ? RULE_MUL : RULE_DIV;
    for (int q = 0; q < d.dim; ++q)
        for (int s = 0; s < 2; ++s) {
            if (a.rtype[q][s] != RULE_DIV) continue;
            if (rpow2) {
                a.rtype[q][s] = RULE_MUL;
                a.rc3[q][s] = T(1) / a.rc3[q][s];
            } else if (mode == FTCS_CDIV) {
                a.rtype[q][s] = RULE_CDIV;
                a.gd[q][s].h = std::fabs((double)a.rc3[q][s]);
                a.gd[q][s].y = 1.0 / a.gd[q][s].h;
            }
        }
    if (pow2) {
        for (int q = 0; q < d.dim; ++q) a.hh[q] = (T)(1.0 / m->h[q]);
        const T k2 = a.hh[0] * a.hh[0];  // exact: a power of two
        a.coefh = a.coef * k2;            // exact: a power-of-two scaling of the rounded coef
    }
    hipStream_t st = f->ctx->stream;
    void* cur = f->data;  // time level the next launch reads
    void* nxt = nullptr;  // time level it writes
    if (ext_spare) {
        // every cell the kernels do not write keeps the field's value
        OPF_HIP(hipMemcpyAsync(ext_spare, f->data, f->nbytes, hipMemcpyDeviceToDevice, st));
        nxt = ext_spare;
    } else {
        if (!f->spare) {
            OPF_HIP(hipMalloc(&f->spare, f->nbytes));
            f->spare_valid = false;
        }
        if (!f->spare_valid) {
            OPF_HIP(hipMemcpyAsync(f->spare, f->data, f->nbytes, hipMemcpyDeviceToDevice, st));
            f->spare_valid = true;
        }
        nxt = f->spare;
    }
    const Strip2d p2 = d.dim == 2 ? strip_plan(a.n, a.per, nsteps, tblock, !pow2, f->ctx->cus) : Strip2d{};
    bool ghosts_stale = false;  // the 3-D blocked kernel writes interior cells only
    for (int it = 0; it < nsteps;) {
        const T* in = (const T*)cur;
        T* out = (T*)nxt;
        const int k = d.dim == 2 ? std::min(p2.nt, nsteps - it)
                                 : launch_steps3(d.dtype, (long long)a.e0 * a.e1, nsteps - it, tblock);
        if (ghosts_stale && !(d.dim == 3 && k > 1 && a.per[0] && a.per[1] && a.per[2])) {
            OPF_TRY(launch_ghost_fill(f, cur));
            ghosts_stale = false;
        }
        // launches the kernel instantiated for the arithmetic mode
        auto by_mode = [&](auto launch) {
            if (mode == FTCS_FACTORED) launch(std::integral_constant<int, FTCS_FACTORED>{});
            else if (mode == FTCS_MUL) launch(std::integral_constant<int, FTCS_MUL>{});
            else launch(std::integral_constant<int, FTCS_DIV>{});
        };
        if (d.dim == 2) {
            const unsigned tiles = (unsigned)(((a.n[0] + p2.tx - 1) / p2.tx) * ((a.n[1] + p2.ty - 1) / p2.ty));
            auto launch2 = [&](auto M) {
                constexpr int MD = decltype(M)::value;
                auto with = [&](auto C) {
                    constexpr int c = decltype(C)::value;
                    hipLaunchKernelGGL((ftcs2d_strip_kernel<T, MD, S2_XW[c], S2_RW[c], S2_NW[c]>), dim3(tiles),
                                       dim3(64 * S2_NW[c]), 0, st, in, out, a, k, p2.tx, p2.ty);
                };
                if (p2.cfg == 0) with(std::integral_constant<int, 0>{});
                else if (p2.cfg == 1) with(std::integral_constant<int, 1>{});
                else if constexpr (MD != FTCS_CDIV && MD != FTCS_DIV) with(std::integral_constant<int, 2>{});
            };
            if (mode == FTCS_CDIV) launch2(std::integral_constant<int, FTCS_CDIV>{});
            else by_mode(launch2);
        } else if (d.dim == 3 && k > 1) {
            using C3 = Ftcs3dCfg<T>;
            const bool allper = a.per[0] && a.per[1] && a.per[2];
            // z chunk: periodic fields take the longest (each chunk recomputes 2K halo
            // planes) that still gives every CU a workgroup (one 147 KB workgroup fills a
            // CU). 512^3 FP64: 256 planes, 256 workgroups, one round: 750 -> 800 G
            // cell-updates/s against 64-plane chunks (four rounds); FP32 (128-wide tiles)
            // 128 planes: 1515 -> 1610. With Dirichlet / Neumann sides the workgroups that
            // rebuild ghosts take longer, and 64-plane chunks (more workgroups than CUs,
            // balanced by the dispatcher) stay faster (512^3 FP64: 376 vs 330 G/s)
            const int tiles = ((a.n[0] + C3::TX - 1) / C3::TX) * ((a.n[1] + C3::TY - 1) / C3::TY);
            int zc = allper ? 256 : 64;
            while (zc > 16 && (long long)tiles * ((a.n[2] + zc - 1) / zc) < f->ctx->cus) zc /= 2;
            const int nb = tiles * ((a.n[2] + zc - 1) / zc);
            static_assert(C3::K == 3, "remainder launches assume K = 3");
            by_mode([&](auto M) {
                constexpr int MD = decltype(M)::value;
                if (k == C3::K && allper)
                    hipLaunchKernelGGL((ftcs3d_tb_kernel<T, MD, C3::TX, C3::TY, C3::NT, C3::K, C3::XCD, true>),
                                       dim3(nb), dim3(C3::NT), 0, st, in, out, a, zc);
                else if (k == C3::K)
                    hipLaunchKernelGGL((ftcs3d_tb_kernel<T, MD, C3::TX, C3::TY, C3::NT, C3::K, C3::XCD, false>),
                                       dim3(nb), dim3(C3::NT), 0, st, in, out, a, zc);
                else if (allper)
                    hipLaunchKernelGGL((ftcs3d_tb_kernel<T, MD, C3::TX, C3::TY, C3::NT, 2, C3::XCD, true>),
                                       dim3(nb), dim3(C3::NT), 0, st, in, out, a, zc);
                else
                    hipLaunchKernelGGL((ftcs3d_tb_kernel<T, MD, C3::TX, C3::TY, C3::NT, 2, C3::XCD, false>),
                                       dim3(nb), dim3(C3::NT), 0, st, in, out, a, zc);
            });
            ghosts_stale = true;
        } else if (d.dim == 3) {
            dim3 grid((a.n[0] + FT3_TX - 1) / FT3_TX, (a.n[1] + FT3_TY - 1) / FT3_TY, (a.n[2] + FT3_ZC - 1) / FT3_ZC);
            by_mode([&](auto M) {
                hipLaunchKernelGGL((ftcs3d_lds_kernel<T, decltype(M)::value, FT3_ZC, FT3_NTY, FT3_RY>), grid,
                                   dim3(64, FT3_NTY), 0, st, in, out, a);
            });
            ghosts_stale = true;
        } else {
            set_error("ftcs: dim %d not supported by the fast path", d.dim);
            return OPF_ERR_UNSUPPORTED;
        }
        it += k;
        std::swap(cur, nxt);
    }
    if (ghosts_stale) OPF_TRY(launch_ghost_fill(f, cur));
    OPF_HIP(hipGetLastError());
    if (ext_spare) {
        if (cur != f->data) OPF_HIP(hipMemcpyAsync(f->data, cur, f->nbytes, hipMemcpyDeviceToDevice, st));
    } else {
        f->data = cur;
        f->spare = nxt;
    }
    return OPF_OK;
}

}  // namespace

extern "C" int opf_ftcs(opf_field* u, double coef, int nsteps) {
    OPF_CHECK(u && nsteps >= 0, OPF_ERR_ARG, "opf_ftcs: bad args");
    if (nsteps == 0) return OPF_OK;
    return u->d.dtype == OPF_F64 ? ftcs_t<double>(u, coef, nsteps, 0) : ftcs_t<float>(u, coef, nsteps, 0);
}

extern "C" int opf_ftcs_noalloc(opf_field* u, double coef, int nsteps) {
    OPF_CHECK(u && nsteps >= 0, OPF_ERR_ARG, "opf_ftcs_noalloc: bad args");
    OPF_CHECK(u->nbytes <= (size_t)OPF_FTCS_NOALLOC_MAX_BYTES, OPF_ERR_NOMEM,
              "opf_ftcs_noalloc: field storage of %zu bytes exceeds the %zu-byte device scratch", u->nbytes,
              (size_t)OPF_FTCS_NOALLOC_MAX_BYTES);
    OPF_CHECK(u->ctx->noalloc_scratch, OPF_ERR_HIP, "opf_ftcs_noalloc: no scratch address for device %d",
              u->ctx->device);
    if (nsteps == 0) return OPF_OK;
    void* s = u->ctx->noalloc_scratch;
    return u->d.dtype == OPF_F64 ? ftcs_t<double>(u, coef, nsteps, 0, s) : ftcs_t<float>(u, coef, nsteps, 0, s);
}

extern "C" int opf_ftcs_plan(const opf_field* u, int nsteps, int tblock, int* launches, int* max_steps) {
    OPF_CHECK(u && nsteps >= 0 && tblock >= 0 && launches && max_steps, OPF_ERR_ARG, "opf_ftcs_plan: bad args");
    const opf_field_desc& d = u->d;
    int n[3] = {1, 1, 1}, per[3] = {0, 0, 0};
    for (int q = 0; q < d.dim; ++q) {
        n[q] = d.local_end[q] - d.local_start[q];
        per[q] = d.bc_type[q][0] == OPF_BC_PERIODIC;
    }
    *launches = 0;
    *max_steps = 0;
    bool pow2 = true;
    for (int q = 0; q < d.dim; ++q) pow2 &= is_pow2(u->mesh->h[q]);
    const int nt = d.dim == 2 && nsteps > 0 ? strip_plan(n, per, nsteps, tblock, !pow2, u->ctx->cus).nt : 0;
    for (int it = 0; it < nsteps;) {
        const int k = d.dim == 2 ? std::min(nt, nsteps - it)
                                 : launch_steps3(d.dtype, (long long)d.extent[0] * d.extent[1], nsteps - it, tblock);
        ++*launches;
        *max_steps = std::max(*max_steps, k);
        it += k;
    }
    return OPF_OK;
}

extern "C" int opf_ftcs_blocked(opf_field* u, double coef, int nsteps, int tblock) {
    OPF_CHECK(u && nsteps >= 0 && tblock >= 0, OPF_ERR_ARG, "opf_ftcs_blocked: bad args");
    if (nsteps == 0) return OPF_OK;
    return u->d.dtype == OPF_F64 ? ftcs_t<double>(u, coef, nsteps, tblock) : ftcs_t<float>(u, coef, nsteps, tblock);
}
