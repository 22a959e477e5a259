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
    int divide;             // FTCS_CDIV: every division by h as a division
    unsigned low;           // FTCS_CDIV: the least div_key of a value in the range
    int stale;              // 3-D: the input's ghosts are not filled
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
//  FTCS_CDIV     any h: FTCS_DIV's divisions through the reciprocal of h (constdiv.hpp) where the
//                values are in the range that needs, as divisions elsewhere (FtcsArgs::divide: all).
enum { FTCS_DIV = 0, FTCS_MUL = 1, FTCS_FACTORED = 2, FTCS_CDIV = 3 };

// x / h of dim d in an arithmetic mode
template <typename T, int MODE>
__device__ __forceinline__ T over_h(T x, const FtcsArgs<T>& a, int d) {
    if constexpr (MODE == FTCS_FACTORED) return x;
    else if constexpr (MODE == FTCS_MUL) return x * a.hh[d];
    else if constexpr (MODE == FTCS_CDIV) return const_div(x, a.cd[d]);
    else return x / a.hh[d];
}

// The ghost rules of a launch in one form, (c1 v - c2) over c3 with c1 = c3 = 1 where the rule only
// adds (both exact): over c3 a multiplication by its exact reciprocal, a const_div or a division.
// One straight line for every side, so that the lanes of a wave take theirs together.
template <typename T>
struct SideRule {
    T c1, c2, c3;
    double h, y;  // |c3| and its reciprocal (RULE_CDIV)
};
template <typename T>
__device__ __forceinline__ SideRule<T> side_rule(const FtcsArgs<T>& a, int d, int s) {
    const int t = a.rtype[d][s];
    SideRule<T> r{T(1), T(0), T(1), 1.0, 1.0};
    if (t == RULE_ADD) r.c2 = -a.rc1[d][s];
    if (t == RULE_DIV || t == RULE_MUL || t == RULE_CDIV) r.c1 = a.rc1[d][s], r.c2 = a.rc2[d][s], r.c3 = a.rc3[d][s];
    if (t == RULE_CDIV) r.h = a.gd[d][s].h, r.y = a.gd[d][s].y;
    return r;
}
// again: RULE_CDIV met a value outside const_div's range
template <int FORM, typename T>
__device__ __forceinline__ T ghost_value(const SideRule<T>& s, T v, unsigned low, bool& again) {
    const T x = s.c1 * v - s.c2;
    if constexpr (FORM == RULE_MUL) return x * s.c3;
    else if constexpr (FORM == RULE_DIV) return x / s.c3;
    else {
        const T q = const_div(x, ConstDivisor{s.h, s.y});
        again |= div_key(v) < low;
        return s.c3 < T(0) ? -q : q;  // h = |c3|
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

// a wave-uniform value in scalar registers
__device__ __forceinline__ float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
__device__ __forceinline__ double uniform(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
template <bool HOIST, typename T>
__device__ __forceinline__ SideRule<T> uniform_side(const SideRule<T>* s) {
    int here = 0;
    if constexpr (!HOIST) asm volatile("" : "+s"(here));  // read at each use, see stage_sides
    s += here;
    return {uniform(s->c1), uniform(s->c2), uniform(s->c3), uniform(s->h), uniform(s->y)};
}

// the rules of a field's sides in LDS, x lower, x upper, y lower, ..: in 3-D read where a workgroup
// has ghosts to refill, they would otherwise hold 40 scalar registers through every loop; 2-D has
// the registers (HOIST)
template <typename T>
__device__ __forceinline__ void stage_sides(const FtcsArgs<T>& a, SideRule<T>* side, int dim) {
    if ((int)threadIdx.x < 2 * dim) side[threadIdx.x] = side_rule(a, threadIdx.x >> 1, threadIdx.x & 1);
    __syncthreads();
}

// The ghost cells of a wave's part of a region (XW cells a lane from column gx0, RW rows from row
// gy0; the region spans width columns from lox) and their refill from fresh cells: x, then y.
template <typename T, int XW, int RW, bool HOIST>
struct StripGhosts {
    static_assert(XW <= 2, "the ghost columns are a lane's first or second");
    bool xlo, xhi, ylo, yhi, any;  // uniform over the wave
    bool lo, hi0, hi1;             // this lane: its first column is the lower ghost; its first, second the upper
    int rlo, rhi;                  // ghost rows
    const SideRule<T>* side;       // x lower, x upper, y lower, y upper
    unsigned low;                  // FtcsArgs::low

    __device__ __forceinline__ StripGhosts(const FtcsArgs<T>& a, const SideRule<T>* sides, int lox, int width, int gx0,
                                           int gy0)
        : side(sides), low(a.low) {
        const int n0 = a.n[0], n1 = a.n[1];
        xlo = !a.per[0] && lox <= -1;
        xhi = !a.per[0] && lox + width > n0;
        rlo = a.per[1] ? -1 : -1 - gy0;
        rhi = a.per[1] ? -1 : n1 - gy0;
        ylo = rlo >= 0 && rlo < RW;
        yhi = rhi >= 0 && rhi < RW;
        any = xlo || xhi || ylo || yhi;
        lo = gx0 == -1;
        hi0 = gx0 == n0;
        hi1 = gx0 + 1 == n0;
    }
    // true when RULE_CDIV met a value out of its range: the fill is then done again by division
    template <int FM>
    __device__ __forceinline__ bool refill(T (&v)[RW][XW]) const {
        bool again = false;
        if (xlo) {
            const SideRule<T> s = uniform_side<HOIST>(side);
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const T src = XW > 1 ? v[r][XW > 1 ? 1 : 0] : lane_next(v[r][0]);
                v[r][0] = pick(lo, ghost_value<FM>(s, src, low, again), v[r][0]);
            }
        }
        if (xhi) {
            const SideRule<T> s = uniform_side<HOIST>(side + 1);
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const T prev = lane_prev(v[r][XW - 1]);
                if constexpr (XW > 1) v[r][1] = pick(hi1, ghost_value<FM>(s, v[r][0], low, again), v[r][1]);
                v[r][0] = pick(hi0, ghost_value<FM>(s, prev, low, again), v[r][0]);
            }
        }
        if (ylo) {
            const SideRule<T> s = uniform_side<HOIST>(side + 2);
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                T src = v[1][k];
#pragma unroll
                for (int r = 1; r + 1 < RW; ++r) src = pick(r == rlo, v[r + 1][k], src);
                const T g = ghost_value<FM>(s, src, low, again);
#pragma unroll
                for (int r = 0; r + 1 < RW; ++r) v[r][k] = pick(r == rlo, g, v[r][k]);
            }
        }
        if (yhi) {
            const SideRule<T> s = uniform_side<HOIST>(side + 3);
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                T src = v[0][k];
#pragma unroll
                for (int r = 2; r < RW; ++r) src = pick(r == rhi, v[r - 1][k], src);
                const T g = ghost_value<FM>(s, src, low, again);
#pragma unroll
                for (int r = 1; r < RW; ++r) v[r][k] = pick(r == rhi, g, v[r][k]);
            }
        }
        return FM == RULE_CDIV && __any(again);
    }
    // mul: every rule multiplies; slow: no const_div
    template <int FORM>
    __device__ __forceinline__ void fill(T (&v)[RW][XW], bool mul, bool slow) const {
        if (FORM == RULE_MUL && mul) refill<RULE_MUL>(v);
        else if (FORM != RULE_CDIV || slow || refill<RULE_CDIV>(v)) refill<RULE_DIV>(v);
    }
};

// First row of a region of WY rows for the tile from row y0 with nt rows of halo, on a side that is
// not periodic: from the ghost row on, or up to it as the last row of the last wave; both ghost rows
// inside, each in one wave with the row beside it.
template <int RW, int WY>
__device__ __forceinline__ int strip_rows(int y0, int nt, int n1) {
    int lo = max(y0 - nt, -1);
    if (lo + WY > n1 + 1) {
        lo = n1 + 1 - WY;
        if (lo < -1) lo = (n1 + 1) % RW == 0 ? -2 : -1;
    }
    return lo;
}

// a ghost plane from the plane beside it
template <int FORM, typename T, int RW, int XW>
__device__ __forceinline__ void strip_ghost_plane(const SideRule<T>* side, const T (&src)[RW][XW], T (&dst)[RW][XW],
                                                  bool mul, bool slow, unsigned low) {
    const SideRule<T> r = uniform_side<false>(side);
    auto fill = [&](auto F) __attribute__((always_inline)) -> bool {
        constexpr int FM = decltype(F)::value;
        bool again = false;
#pragma unroll
        for (int j = 0; j < RW; ++j)
#pragma unroll
            for (int k = 0; k < XW; ++k)
                dst[j][k] = ghost_value<FM>(r, src[j][k], low, again);
        return FM == RULE_CDIV && __any(again);
    };
    if (FORM == RULE_MUL && mul) fill(std::integral_constant<int, RULE_MUL>{});
    else if (FORM != RULE_CDIV || slow || fill(std::integral_constant<int, RULE_CDIV>{}))
        fill(std::integral_constant<int, RULE_DIV>{});
}

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
// 4096^2 periodic 42 -> 11.0 (0.40 -> 1.53 T/s).
template <typename T, int MODE, int XW, int RW, int NW>
__global__ __launch_bounds__(64 * NW) void ftcs2d_strip_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                               FtcsArgs<T> a, int nt, int tx, int ty) {
    constexpr int WX = 64 * XW, WY = RW * NW;
    __shared__ T edge[2][NW][2][XW][64];  // first and last row of every wave, double-buffered
    const int n0 = a.n[0], n1 = a.n[1];
    const int tilesx = (n0 + tx - 1) / tx;
    const int tb = (int)xcd_block(blockIdx.x, gridDim.x);  // x-neighbouring tiles share an XCD's L2
    const int x0 = (tb % tilesx) * tx, y0 = (tb / tilesx) * ty;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lox = a.per[0] ? x0 - nt : max(x0 - nt, -1);
    const int loy = a.per[1] ? y0 - nt : strip_rows<RW, WY>(y0, nt, n1);
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
    constexpr int FORM = MODE == FTCS_CDIV ? RULE_CDIV : RULE_MUL;
    __shared__ SideRule<T> side[4];
    stage_sides(a, side, 2);
    const StripGhosts<T, XW, RW, true> gh(a, side, lox, WX, gx0, gy0);
    bool slow = MODE == FTCS_CDIV && a.divide;  // FP64: or a value outside the range for the whole launch
    if constexpr (MODE == FTCS_CDIV && sizeof(T) == 8) {
        bool bad = false;
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) bad |= div_unsafe(u[r][k]);
        slow |= (bool)__syncthreads_or(bad);
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
        auto xpart = [&](auto M) __attribute__((always_inline)) {
            constexpr int MD = decltype(M)::value;
            auto quo = [&](T x) __attribute__((always_inline)) -> T { return over_h<T, MD>(x, a, 0); };
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
        };
        T dn[XW], up[XW];  // the rows before the first and after the last
        auto ypart = [&](auto M) __attribute__((always_inline)) {
            constexpr int MD = decltype(M)::value;
            auto quo = [&](T x) __attribute__((always_inline)) -> T { return over_h<T, MD>(x, a, 1); };
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
        };
        xpart(std::integral_constant<int, MODE>{});  // needs no other wave: while the rows are on their way
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
        if constexpr (MODE == FTCS_CDIV) {
            unsigned m = 0xffffffffu;
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                m = min(m, min(div_key(dn[k]), div_key(up[k])));
#pragma unroll
                for (int r = 0; r < RW; ++r) m = min(m, div_key(u[r][k]));
            }
            again |= __any(m < a.low);
        }
        if (!again) ypart(std::integral_constant<int, MODE>{});
        if constexpr (MODE == FTCS_CDIV) {
            if (again) {
                xpart(std::integral_constant<int, FTCS_DIV>{});
                ypart(std::integral_constant<int, FTCS_DIV>{});
            }
        }
        if (gh.any) gh.template fill<FORM>(v, a.gform == RULE_MUL, again);
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

// 3-D steps in registers, K per launch: the 2-D kernel's region (64 XW x NW RW cells of a plane,
// RW rows a wave) marching through the planes of a z chunk. Stage s of the pipeline takes the
// planes of level s (u^{n+s}) as they appear and gives those of level s + 1 one plane later. Per
// level a cell holds its value, the quotient of its last z difference and d2x + d2y, so that a new
// plane costs one difference in z, and the update follows from registers alone:
//   level s + 1 at plane p - 1 from level s at p - 1 (held) and at p (new), straight into stage
//   s + 1 as its plane p - 1, and so on; level K goes to memory.
// Then each wave's first and last rows of every level's new plane pass through LDS (one barrier a
// plane), and d2x + d2y of those planes is formed for the next one. One plane
// of level 0 is in flight. Periodic sides wrap the halo; on the others the region starts at, or contains, the
// ghost layer: level 0 reads the input's ghosts, those of the other levels are refilled in
// registers when a plane appears (x, then y), and the ghost planes in z are the rules of the planes
// beside them. The output's ghosts are left stale: the host loop refills them before a launch that
// reads them and at the end (a launch of three steps that refilled them itself would gain nothing,
// 196 against 187 us a step at 512^3 FP64 Dirichlet: the workgroups at the sides are the last to
// end); a single step refills its input in registers (128^3 17.9 -> 13.2 us). Per cell and step the
// operations and their order are those of D2 in the reference.
// A plane step takes 2.5 us of a workgroup that has its CU to itself, 1.4 of it FP64, lane moves and
// LDS instructions of the three levels, the rest the waves' wait at the barrier and for the rows of
// their neighbours. FP32 has the registers for two planes a round, which saves the moves of the held
// planes (512^3 98 -> 86 us a step); FP64 spills with two. us a step, against LDS tiles of the values
// that marched with one step (ghosts filled by a launch per step; periodic FACTORED: two steps):
// 512^3 FP64 periodic 180 -> 152, Dirichlet 355 -> 187, 128^3 Dirichlet 30 -> 14.3, 300 x 260 x 220
// FP32 Dirichlet 59 -> 23.
template <typename T, int MODE, int XW, int RW, int NW, int K, bool ALLPER>
__global__ __launch_bounds__(64 * NW) void ftcs3d_strip_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                               FtcsArgs<T> a, int tx, int ty, int zc) {
    constexpr int WX = 64 * XW, WY = RW * NW;
    constexpr bool D64 = sizeof(T) == 8;
    constexpr int FORM = MODE == FTCS_CDIV ? RULE_CDIV : RULE_MUL;
    __shared__ T edge[2][K][NW][2][XW][64];  // first and last row of every wave and level, double-buffered
    __shared__ int wild;                     // FTCS_CDIV, FP64: a value outside the range has been read
    const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2];
    const int tilesx = (n0 + tx - 1) / tx, tilesy = (n1 + ty - 1) / ty;
    int b = (int)xcd_block(blockIdx.x, gridDim.x);  // neighbouring tiles share an XCD's L2
    const int x0 = (b % tilesx) * tx;
    b /= tilesx;
    const int y0 = (b % tilesy) * ty;
    const int z0 = (b / tilesy) * zc, z1 = min(z0 + zc, n2);
    const int lane = threadIdx.x & 63, w_ = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool xper = ALLPER || a.per[0], yper = ALLPER || a.per[1], zper = ALLPER || a.per[2];
    const int lox = xper ? x0 - K : max(x0 - K, -1);
    const int loy = yper ? y0 - K : strip_rows<RW, WY>(y0, K, n1);
    const int gx0 = lox + lane * XW, gy0 = loy + w_ * RW;
    __shared__ SideRule<T> side[6];
    stage_sides(a, side, 3);
    const StripGhosts<T, XW, RW, false> gh(a, side, lox, WX, gx0, gy0);
    const long long sz = (long long)a.e0 * a.e1;
    const int st = K > 1 || ALLPER ? 0 : a.stale;  // read no ghosts
    int ox[XW];  // storage offsets of this lane's columns and this wave's rows
    long long oy[RW];
#pragma unroll
    for (int k = 0; k < XW; ++k) {
        int gx = gx0 + k;
        if (xper) gx = ((gx % n0) + n0) % n0;
        ox[k] = min(max(gx, -1 + st), n0 - st) + 1;
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        int gy = gy0 + r;
        if (yper) gy = ((gy % n1) + n1) % n1;
        oy[r] = (long long)a.e0 * (min(max(gy, -1 + st), n1 - st) + 1);
    }
    // planes of level 0 from ta; level K's plane t - K appears at t
    const int ta = zper ? z0 - K : max(z0 - K, -1 + st), tb = z1 + K;
    const int zw = zper ? ((ta % n2) + n2) % n2 : max(ta, -1 + st);
    const T* from = in + sz * (zw + 1);  // the next plane to load
    const T* const wrap = in + sz * (n2 + 1);
    const T* const last = wrap - sz * st;
    T pre[RW][XW], u[K][RW][XW], qz[K][RW][XW], sx[K][RW][XW];
#pragma unroll
    for (int s = 0; s < K; ++s)
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) u[s][r][k] = qz[s][r][k] = sx[s][r][k] = T(0);
    int odd[K] = {};  // FTCS_CDIV: bit q: plane t - s - q of this wave holds a value under the range
    bool slow = MODE == FTCS_CDIV && a.divide;
    if (MODE == FTCS_CDIV && D64) {
        if (threadIdx.x == 0) wild = slow;
        __syncthreads();
    }
    auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) pre[r][k] = (from + oy[r])[ox[k]];
        // periodic: plane 0 after plane n2 - 1; else the last plane (the ghost plane) again
        from += sz;
        if (zper && from == wrap) from = in + sz;
        if (!zper && from > last) from = last;
    };
    load();
    const T coef = MODE == FTCS_FACTORED ? a.coefh : a.coef;
    auto plane = [&](int t) __attribute__((always_inline)) {
        T w[RW][XW];  // the plane that appears
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int k = 0; k < XW; ++k) w[r][k] = pre[r][k];
        load();
        if constexpr (MODE == FTCS_CDIV && D64) {
            bool bad = false;
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int k = 0; k < XW; ++k) bad |= div_unsafe(w[r][k]);
            if (__any(bad)) slow = true, wild = 1;
        }
        if (K == 1 && !ALLPER && st && gh.any) gh.template fill<FORM>(w, a.gform == RULE_MUL, slow);
#pragma unroll
        for (int s = 0; s < K; ++s) {
            if (!zper && (s > 0 || (K == 1 && st))) {  // ghost planes of level s: n2 from the last plane, -1 before the first
                if (t - s == n2) strip_ghost_plane<FORM>(side + 5, u[s], w, a.gform == RULE_MUL, slow, a.low);
                if (t - s == 0) strip_ghost_plane<FORM>(side + 4, w, u[s], a.gform == RULE_MUL, slow, a.low);
            }
            T qn[RW][XW], v[RW][XW];
            auto zpart = [&](auto M) __attribute__((always_inline)) {
                constexpr int MD = decltype(M)::value;
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int k = 0; k < XW; ++k) {
                        qn[r][k] = over_h<T, MD>(w[r][k] - u[s][r][k], a, 2);
                        const T dz = over_h<T, MD>(qn[r][k] - qz[s][r][k], a, 2);
                        v[r][k] = u[s][r][k] + coef * (sx[s][r][k] + dz);
                    }
            };
            bool again = slow;
            if constexpr (MODE == FTCS_CDIV) {
                unsigned m = 0xffffffffu;
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int k = 0; k < XW; ++k) m = min(m, div_key(w[r][k]));
                odd[s] = (odd[s] << 1 | (__any(m < a.low) ? 1 : 0)) & 7;
                again |= odd[s] != 0;
            }
            if (!again) zpart(std::integral_constant<int, MODE>{});
            if constexpr (MODE == FTCS_CDIV) {
                if (again) zpart(std::integral_constant<int, FTCS_DIV>{});
            }
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int k = 0; k < XW; ++k) {
                    u[s][r][k] = w[r][k];
                    qz[s][r][k] = qn[r][k];
                    w[r][k] = v[r][k];
                }
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                edge[t & 1][s][w_][0][k][lane] = u[s][0][k];
                edge[t & 1][s][w_][1][k][lane] = u[s][RW - 1][k];
            }
            if (!ALLPER && s + 1 < K && gh.any) gh.template fill<FORM>(w, a.gform == RULE_MUL, again);
        }
        if (t - K >= z0) {  // level K of plane t - K
            T* to = out + sz * (t - K + 1);
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const int gy = gy0 + r;
                if (gy < y0 || gy >= min(y0 + ty, n1)) continue;
#pragma unroll
                for (int k = 0; k < XW; ++k) {
                    const int gx = gx0 + k;
                    if (gx >= x0 && gx < min(x0 + tx, n0)) (to + (long long)a.e0 * (gy + 1) + 1)[gx] = w[r][k];
                }
            }
        }
        __syncthreads();
        if constexpr (MODE == FTCS_CDIV && D64) slow = __builtin_amdgcn_readfirstlane(wild) != 0;
#pragma unroll
        for (int s = 0; s < K; ++s) {
            T dn[XW], up[XW];
#pragma unroll
            for (int k = 0; k < XW; ++k) {
                dn[k] = edge[t & 1][s][max(w_ - 1, 0)][1][k][lane];
                up[k] = edge[t & 1][s][min(w_ + 1, NW - 1)][0][k][lane];
            }
            auto xypart = [&](auto M) __attribute__((always_inline)) {
                constexpr int MD = decltype(M)::value;
                auto quo = [&](T x, int d) __attribute__((always_inline)) -> T { return over_h<T, MD>(x, a, d); };
                T qy[XW];
#pragma unroll
                for (int k = 0; k < XW; ++k) qy[k] = quo(u[s][0][k] - dn[k], 1);
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    T qx[XW];
#pragma unroll
                    for (int k = 0; k < XW; ++k) {
                        const T right = k + 1 < XW ? u[s][r][k + 1 < XW ? k + 1 : 0] : lane_next(u[s][r][0]);
                        qx[k] = quo(right - u[s][r][k], 0);
                    }
                    const T left = lane_prev(qx[XW - 1]);
#pragma unroll
                    for (int k = 0; k < XW; ++k) {
                        const T qn = quo((r + 1 < RW ? u[s][r + 1 < RW ? r + 1 : 0][k] : up[k]) - u[s][r][k], 1);
                        const T dx = quo(qx[k] - (k > 0 ? qx[k > 0 ? k - 1 : 0] : left), 0);
                        sx[s][r][k] = dx + quo(qn - qy[k], 1);
                        qy[k] = qn;
                    }
                }
            };
            bool again = slow;
            if constexpr (MODE == FTCS_CDIV) {
                unsigned m = 0xffffffffu;
#pragma unroll
                for (int k = 0; k < XW; ++k) m = min(m, min(div_key(dn[k]), div_key(up[k])));
                again |= (odd[s] & 1) != 0 || __any(m < a.low);
            }
            if (!again) xypart(std::integral_constant<int, MODE>{});
            if constexpr (MODE == FTCS_CDIV) {
                if (again) xypart(std::integral_constant<int, FTCS_DIV>{});
            }
        }
    };
    for (int t = ta; t < tb; ++t) {
        plane(t);
        if (!D64) {  // two planes a round: the held planes change registers by name, not by moves
            if (++t >= tb) break;
            plane(t);
        }
    }
}

// Launches of the 2-D kernel: the region (cells in x per lane, rows per wave, waves), the steps per
// launch and the tile that is left of the region. Per step a launch costs
//   S2_LAUNCH / nt + max(alone, tiles / CUs * shared + traffic / nt)
// with the measured time of one step of one workgroup when it has a CU to itself (alone: the
// barrier and the waves' latency) and when several share one (shared: instruction issue), about
// 1.8 times that with const_div, and the regions read and tiles written at the rate of the last-level
// cache or of memory, where both time levels are past the L2s (on a grid within them shared has it).
// More steps a launch save launches and traffic and lose tile. FP64, us per step: 256^2 64 x 32 region
// with 12 steps 0.80 (64 x 64, 20 steps: 1.00); 700^2, const_div, 64 x 64, 10 steps 1.89 (64 x 32, 6:
// 1.99); 4096^2 periodic 128 x 64, 10 steps 10.0 (64 x 64, 8: 12.5). With const_div the 128 x 64 region
// holds too few waves (117 registers): 2000^2, 4 steps, 7.7 against 7.3.
// What the rule takes, without the traffic -> with it, and the best of a sweep over regions and 2 to 24
// steps: 4096^2 FP64 17.4 -> 11.0, best 10.0; 8192^2 125.7 -> 42.6, 40.8; 16384^2 510 -> 170, 161; 8192^2
// FP32 64.7 -> 28.4, 25.9; const_div 3000^2 16.3 -> 12.1, 12.1; 8000^2 112 -> 82, 82.
constexpr int S2_XW[3] = {1, 1, 2}, S2_RW[3] = {4, 8, 8}, S2_NW[3] = {8, 8, 8};
constexpr double S2_ALONE[3] = {0.33, 0.55, 1.3}, S2_SHARED[3] = {0.31, 0.49, 0.74}, S2_LAUNCH = 4.2;
constexpr double S2_L2 = 32 << 20, S2_LLC = 256 << 20;  // bytes
constexpr double S2_LLC_RATE = 9.6e6, S2_HBM_RATE = 5.6e6;  // bytes a us, measured on these launches
constexpr double S2_F32 = 0.65;  // shared of FP32, where the traffic is counted apart
constexpr int S2_MOST = 128;  // steps a launch takes at most (the range const_div is given, div_range)
struct Strip2d {
    int cfg = 0;
    int nt = 1, tx = 1, ty = 1;  // steps, tile
};

// vsize: bytes of a value
Strip2d strip_plan(const int n[3], const int per[3], int nsteps, int tblock, bool div, int cus, size_t vsize) {
    Strip2d best;
    double cost = 0;
    const double level = (double)n[0] * n[1] * vsize;
    const bool past = 2 * level > S2_L2;
    const double rate = 2 * level <= S2_LLC ? S2_LLC_RATE : S2_HBM_RATE, issue = vsize == 4 ? S2_F32 : 1.0;
    for (int c = 0; c < (div ? 2 : 3); ++c) {
        const int wx = 64 * S2_XW[c], wy = S2_RW[c] * S2_NW[c];
        const bool allx = !per[0] && n[0] + 2 <= wx, ally = !per[1] && n[1] + 3 <= wy;  // no halo in that dim
        const int most = std::min(nsteps, allx && ally ? S2_MOST : (ally ? wx : allx ? wy : std::min(wx, wy)) / 2 - 2);
        // 1 (when asked for), else 2, 3 .. 12, 24, .. and the most
        for (int nt = tblock == 1 ? 1 : std::min(2, most);;) {
            const int tx = allx ? n[0] : wx - 2 * nt, ty = ally ? n[1] : wy - 2 * nt;
            const double tiles = (double)((n[0] + tx - 1) / tx) * ((n[1] + ty - 1) / ty);
            const double f = div ? 1.8 : 1.0, shared = f * tiles / cus * S2_SHARED[c];
            const double busy = past ? shared * issue + (tiles * wx * wy * vsize + level) / (rate * nt) : shared;
            const double t = S2_LAUNCH / nt + std::max(f * S2_ALONE[c], busy);
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

// Launches of the 3-D kernel: 64 x 64 cells of a plane in 16 waves of 4 rows, three steps a launch
// (a remainder of two or one takes a launch of its own). Swept at 512^3 FP64 periodic: 8 waves of 8
// rows 151 us a step, 128 x 32 cells 202, against 146; four steps fit 64 x 48 cells (162: 130 tiles
// fill the chip badly) and spill in 64 x 64.
constexpr int S3_XW = 1, S3_RW = 4, S3_NW = 16, S3_K = 3;
// Single steps take half the waves and two workgroups a CU while the field and its second buffer
// stay in the 256 MB last-level cache, where a workgroup's latency bounds them: 128^3 FP64 Dirichlet
// 14.9 -> 13.2 us, 64^3 9.4 -> 7.4; beyond, the larger region reads less halo (512^3 FP64 609 -> 485).
constexpr size_t S3_CACHE = (size_t)256 << 20;

// Steps the next launch of a 3-D field advances. tblock = 1 forces single steps.
// The last four are two and two.
int launch_steps3(int remaining, int tblock) { return tblock == 1 ? 1 : remaining == 4 ? 2 : std::min(S3_K, remaining); }

// Planes per workgroup: a chunk of zc planes costs zc + 2 K plane steps and one workgroup fills a CU,
// so the cost is that times the rounds the workgroups take; 512^3 FP64 periodic (81 tiles): 171
// planes, one round of 243, 146 us a step; 128 planes, two rounds, 211; 86, two rounds, 170.
int chunk_planes(int tiles, int n2, int k, int cus) {
    int best = n2;
    long long cost = 0;
    for (int c = 1; c == 1 || n2 / c >= 2; ++c) {
        const int zc = (n2 + c - 1) / c;
        const long long wgs = (long long)tiles * ((n2 + zc - 1) / zc);
        const long long t = ((wgs + cus - 1) / cus) * (zc + 2 * k);
        if (c == 1 || t < cost) best = zc, cost = t;
        if (wgs > 16LL * cus) break;
    }
    return best;
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
    const int mode = !pow2 ? FTCS_CDIV : same ? FTCS_FACTORED : FTCS_MUL;
    if (mode == FTCS_CDIV) {
        constexpr bool f64 = std::is_same<T, double>::value;
        bool ok = div_range(m->h, d.dim, coef, S2_MOST, f64);
        a.low = div_low(m->h, d.dim, f64);
        for (int q = 0; q < d.dim; ++q) {
            a.cd[q].h = (double)a.hh[q];
            a.cd[q].y = 1.0 / a.cd[q].h;
            for (int s = 0; s < 2; ++s) {
                const GhostRule& r = gi.rule[q][s][0];
                ok &= div_side(r.type == 1 ? r.c2 / r.c3 : r.type == 2 ? r.c1 : 0.0, m->h, d.dim, f64);
            }
        }
        a.divide = !ok;
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
    const Strip2d p2 = d.dim == 2 ? strip_plan(a.n, a.per, nsteps, tblock, !pow2, f->ctx->cus, sizeof(T)) : Strip2d{};
    bool ghosts_stale = false;  // the 3-D blocked kernel writes interior cells only
    for (int it = 0; it < nsteps;) {
        const T* in = (const T*)cur;
        T* out = (T*)nxt;
        const int k = d.dim == 2 ? std::min(p2.nt, nsteps - it)
                                 : launch_steps3(nsteps - it, tblock);
        const bool allper = a.per[0] && a.per[1] && a.per[2];
        // launches the kernel instantiated for the arithmetic mode
        auto by_mode = [&](auto launch) {
            if (mode == FTCS_FACTORED) launch(std::integral_constant<int, FTCS_FACTORED>{});
            else if (mode == FTCS_MUL) launch(std::integral_constant<int, FTCS_MUL>{});
            else launch(std::integral_constant<int, FTCS_CDIV>{});
        };
        if (d.dim == 2) {
            const unsigned tiles = (unsigned)(((a.n[0] + p2.tx - 1) / p2.tx) * ((a.n[1] + p2.ty - 1) / p2.ty));
            by_mode([&](auto M) {
                constexpr int MD = decltype(M)::value;
                auto with = [&](auto C) {
                    constexpr int c = decltype(C)::value;
                    hipLaunchKernelGGL((ftcs2d_strip_kernel<T, MD, S2_XW[c], S2_RW[c], S2_NW[c]>), dim3(tiles),
                                       dim3(64 * S2_NW[c]), 0, st, in, out, a, k, p2.tx, p2.ty);
                };
                if (p2.cfg == 0) with(std::integral_constant<int, 0>{});
                else if (p2.cfg == 1) with(std::integral_constant<int, 1>{});
                else if constexpr (MD != FTCS_CDIV) with(std::integral_constant<int, 2>{});
            });
        } else if (d.dim == 3) {
            const bool small = k == 1 && 2 * f->nbytes <= S3_CACHE;
            const int wx = 64 * S3_XW, wy = S3_RW * (small ? S3_NW / 2 : S3_NW);
            const int tx = !a.per[0] && a.n[0] + 2 <= wx ? a.n[0] : wx - 2 * k;
            const int ty = !a.per[1] && a.n[1] + 3 <= wy ? a.n[1] : wy - 2 * k;
            const int tiles = ((a.n[0] + tx - 1) / tx) * ((a.n[1] + ty - 1) / ty);
            const int zc = chunk_planes(tiles, a.n[2], k, f->ctx->cus * (small ? 2 : 1));
            const unsigned nb = (unsigned)tiles * ((a.n[2] + zc - 1) / zc);
            if (k > 1 && ghosts_stale && !allper) OPF_TRY(launch_ghost_fill(f, cur));
            a.stale = k == 1 && ghosts_stale && !allper;
            by_mode([&](auto M) {
                constexpr int MD = decltype(M)::value;
                auto with = [&](auto K_, auto W_) {
                    constexpr int K = decltype(K_)::value, W = decltype(W_)::value;
                    if (allper)
                        hipLaunchKernelGGL((ftcs3d_strip_kernel<T, MD, S3_XW, S3_RW, W, K, true>), dim3(nb),
                                           dim3(64 * W), 0, st, in, out, a, tx, ty, zc);
                    else
                        hipLaunchKernelGGL((ftcs3d_strip_kernel<T, MD, S3_XW, S3_RW, W, K, false>), dim3(nb),
                                           dim3(64 * W), 0, st, in, out, a, tx, ty, zc);
                };
                static_assert(S3_K == 3, "a launch of each remainder");
                using Whole = std::integral_constant<int, S3_NW>;
                if (k == 3) with(std::integral_constant<int, 3>{}, Whole{});
                else if (k == 2) with(std::integral_constant<int, 2>{}, Whole{});
                else if (!small) with(std::integral_constant<int, 1>{}, Whole{});
                else with(std::integral_constant<int, 1>{}, std::integral_constant<int, S3_NW / 2>{});
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
    const int nt = d.dim == 2 && nsteps > 0 ? strip_plan(n, per, nsteps, tblock, !pow2, u->ctx->cus, dtype_size(d.dtype)).nt : 0;
    for (int it = 0; it < nsteps;) {
        const int k = d.dim == 2 ? std::min(nt, nsteps - it)
                                 : launch_steps3(nsteps - it, tblock);
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
