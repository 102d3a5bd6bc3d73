// mac_tile_kernels.h -- the smoothing legs of the cell-centred V-cycle, one
// launch each.
//
// A leg of a level was one launch per colour (zero, 4 colours, residual,
// restriction down; prolongation, 4 colours up).  On levels of 64^3 cells and
// below each launch cost 3-5 us of launch and latency for a fraction of that
// work; on larger ones every colour streamed all coefficients and both colours
// of x again (48 bytes per cell and colour in FP64).  Here a workgroup holds a
// tile of x with a halo in LDS, runs every colour of the leg on it (the halo
// shrinks by one cell per colour, recomputed by each tile), forms the residual
// and restricts it, and writes x and the coarse right-hand side once.  b and the
// coefficients come from the caches for each update (x 2-3 per cell).  The
// per-cell arithmetic and its order are those of one launch per colour, and the
// results are the same bit for bit, whichever tiles a level takes.
//   8 x 8 x 8 tiles: many workgroups with short stages (small levels);
//   16 x 16 x 8 tiles: 2.05 updates per cell and sweep pair instead of 4.2.
// Bound by the latency of the stages (5 barriers) on small levels, by the L2
// reads of the coefficients on large ones.
#pragma once

#include "mac_kernels.h"
#include "nodal_mg.h"

namespace mgx {

#pragma clang fp contract(on)  // as in mac_kernels.h

enum { MT_ZERO = 0, MT_X = 1, MT_PROLONG = 2 };  // x starts from 0, xin, xin + parent's xc

template <class T>
struct MacTileArgs {
    MGeomK g, gc;
    MCoef<T> c;
    const T *bx, *by, *bz, *a, *b;
    const T* xin;
    const T* xc;   // MT_PROLONG: the coarse correction
    T* xout;
    T* bc;         // REST: coarse right-hand side
    int gx, gy, gz;
};

// (L x) and its diagonal at a cell whose x and neighbours lie in LDS (p points
// at the cell, strides 1, sy, sz); the terms in mac_apply_cell's order
template <class T>
__device__ __forceinline__ T mac_apply_lds(const MGeomK& g, const MCoef<T>& c, const T* __restrict__ bx,
                                           const T* __restrict__ by, const T* __restrict__ bz,
                                           const T* __restrict__ acoef, const T* p, int sy, int sz, int i,
                                           int j, int k, T& diag) {
    const int pos[3] = {i, j, k}, st[3] = {1, sy, sz};
    const long f0 = i + (long)(g.n[0] + 1) * (j + (long)g.n[1] * k);
    const long f1 = i + (long)g.n[0] * (j + (long)(g.n[1] + 1) * k);
    const long f2 = cidx(g, i, j, k);
    const T bl[3] = {bx[f0], by[f1], bz[f2]};
    const T bh[3] = {bx[f0 + 1], by[f1 + g.n[0]], bz[f2 + (long)g.n[0] * g.n[1]]};
    const T pc = p[0];
    T acc = 0, dg = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (pos[d] > 0 || g.per[d]) {
            const T w = c.ih2[d] * bl[d];
            acc += w * (p[-st[d]] - pc);
            dg -= w;
        } else if (g.dlo[d]) {
            const T w = 2 * c.ih2[d] * bl[d];
            acc -= w * pc;
            dg -= w;
        }
        if (pos[d] + 1 < g.n[d] || g.per[d]) {
            const T w = c.ih2[d] * bh[d];
            acc += w * (p[st[d]] - pc);
            dg -= w;
        } else if (g.dhi[d]) {
            const T w = 2 * c.ih2[d] * bh[d];
            acc -= w * pc;
            dg -= w;
        }
    }
    if (acoef) {
        const T av = acoef[f2];
        acc -= av * pc;
        dg -= av;
    }
    diag = dg;
    return acc;
}

// one colour on the cells within M of the output tile
template <class T, int TX, int TY, int TZ, int H, int M, bool FIRST, int NT>
__device__ __forceinline__ void mac_tile_colour(const MacTileArgs<T>& a, T* xs, const int* px, const int* py,
                                                const int* pz, int color) {
    constexpr int LX = TX + 2 * H, LY = TY + 2 * H, S0 = H - M;
    constexpr int RX = (TX + 2 * M) / 2, RY = TY + 2 * M, RZ = TZ + 2 * M;
    for (int e = threadIdx.x; e < RX * RY * RZ; e += NT) {
        const int q = e % RX, r = e / RX, tj = S0 + r % RY, tk = S0 + r / RY;
        // tile origins are even, so the parity of a cell is that of its tile indices - 3 H
        const int ti = S0 + 2 * q + ((S0 + color + H + tj + tk) & 1);
        const int i = px[ti], j = py[tj], k = pz[tk];
        if (i < 0 || j < 0 || k < 0) continue;
        T* p = xs + ti + LX * (tj + LY * tk);
        T dg, acc;
        if (FIRST) {
            // x is 0 all over the tile: no neighbours (some lie outside it)
            T z[3] = {0, 0, 0};
            acc = mac_apply_lds<T>(a.g, a.c, a.bx, a.by, a.bz, a.a, z + 1, 0, 0, i, j, k, dg);
        } else {
            acc = mac_apply_lds<T>(a.g, a.c, a.bx, a.by, a.bz, a.a, p, LX, LX * LY, i, j, k, dg);
        }
        if (dg != (T)0) p[0] += (a.b[cidx(a.g, i, j, k)] - acc) / dg;
    }
    __syncthreads();
}

// NSW red-black sweeps (0..2) of a level from SRC, then (REST) the residual's
// cell average onto the coarse level
template <class T, int TX, int TY, int TZ, int NSW, int SRC, bool REST>
static __global__ void __launch_bounds__(512) mac_tile_kernel(MacTileArgs<T> a) {
    constexpr int NT = 512;
    constexpr int HN = 2 * NSW + (REST ? 1 : 0) - (SRC == MT_ZERO && NSW > 0 ? 1 : 0);
    constexpr int H = HN > 1 ? HN : 1;
    constexpr int LX = TX + 2 * H, LY = TY + 2 * H, LZ = TZ + 2 * H;
    __shared__ T xs[LX * LY * LZ];
    __shared__ int px[LX], py[LY], pz[LZ];  // domain indices of the tile's columns, -1 outside
    const MGeomK& g = a.g;
    const int tid = threadIdx.x;
    const int lb = xcd_order(blockIdx.x, a.gx * a.gy * a.gz, 4096);
    const int x0 = TX * (lb % a.gx), y0 = TY * ((lb / a.gx) % a.gy), z0 = TZ * (lb / (a.gx * a.gy));
    auto fill = [&](int* p, int len, int o, int d) {
        for (int e = tid; e < len; e += NT) {
            int v = o - H + e;
            if (g.per[d]) v = ((v % g.n[d]) + g.n[d]) % g.n[d];
            p[e] = v < 0 || v >= g.n[d] ? -1 : v;
        }
    };
    fill(px, LX, x0, 0);
    fill(py, LY, y0, 1);
    fill(pz, LZ, z0, 2);
    if (SRC == MT_ZERO)
        for (int e = tid; e < LX * LY * LZ; e += NT) xs[e] = (T)0;
    __syncthreads();
    if (SRC != MT_ZERO) {
        for (int e = tid; e < LX * LY * LZ; e += NT) {
            const int i = px[e % LX], j = py[(e / LX) % LY], k = pz[e / (LX * LY)];
            T v = 0;
            if (i >= 0 && j >= 0 && k >= 0) {
                v = a.xin[cidx(g, i, j, k)];
                if (SRC == MT_PROLONG) v += a.xc[cidx(a.gc, i >> 1, j >> 1, k >> 1)];
            }
            xs[e] = v;
        }
        __syncthreads();
    }
    constexpr int R = REST ? 1 : 0;
    if constexpr (NSW >= 1) {
        mac_tile_colour<T, TX, TY, TZ, H, 2 * NSW - 1 + R, SRC == MT_ZERO, NT>(a, xs, px, py, pz, 0);
        mac_tile_colour<T, TX, TY, TZ, H, 2 * NSW - 2 + R, false, NT>(a, xs, px, py, pz, 1);
    }
    if constexpr (NSW >= 2) {
        mac_tile_colour<T, TX, TY, TZ, H, 1 + R, false, NT>(a, xs, px, py, pz, 0);
        mac_tile_colour<T, TX, TY, TZ, H, R, false, NT>(a, xs, px, py, pz, 1);
    }
    for (int e = tid; e < TX * TY * TZ; e += NT) {
        const int ti = e % TX, tj = (e / TX) % TY, tk = e / (TX * TY);
        const int i = x0 + ti, j = y0 + tj, k = z0 + tk;
        if (i < g.n[0] && j < g.n[1] && k < g.n[2])
            a.xout[cidx(g, i, j, k)] = xs[ti + H + LX * (tj + H + LY * (tk + H))];
    }
    if (REST) {
        // residuals by all threads, then (over the tile of x) their averages
        constexpr int NR = (TX * TY * TZ + NT - 1) / NT, CX = TX / 2, CY = TY / 2, CZ = TZ / 2;
        T rv[NR];
#pragma unroll
        for (int m = 0; m < NR; ++m) {
            const int e = tid + NT * m, ti = e % TX, tj = (e / TX) % TY, tk = e / (TX * TY);
            const int i = x0 + ti, j = y0 + tj, k = z0 + tk;
            rv[m] = 0;
            if (e < TX * TY * TZ && i < g.n[0] && j < g.n[1] && k < g.n[2]) {
                T dg;
                rv[m] = a.b[cidx(g, i, j, k)] -
                        mac_apply_lds<T>(g, a.c, a.bx, a.by, a.bz, a.a,
                                         xs + (ti + H) + LX * ((tj + H) + LY * (tk + H)), LX, LX * LY, i, j, k, dg);
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < NR; ++m)
            if (tid + NT * m < TX * TY * TZ) xs[tid + NT * m] = rv[m];
        __syncthreads();
        for (int e = tid; e < CX * CY * CZ; e += NT) {
            const int ci = e % CX, cj = (e / CX) % CY, ck = e / (CX * CY);
            const int I = x0 / 2 + ci, J = y0 / 2 + cj, K = z0 / 2 + ck;
            if (I >= a.gc.n[0] || J >= a.gc.n[1] || K >= a.gc.n[2]) continue;
            T s = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                s += xs[2 * ci + (q & 1) + TX * (2 * cj + ((q >> 1) & 1) + TY * (2 * ck + (q >> 2)))];
            a.bc[cidx(a.gc, I, J, K)] = (T)0.125 * s;
        }
    }
}

// The same leg on 8 x 8 x 8 tiles with each cell's coefficients in registers:
// a thread owns up to SL cells of each colour (halo included), loads their
// coefficients once, all of them in flight together, and every colour then
// touches LDS only.  Neighbours outside the domain hold 0 in LDS, so a
// Dirichlet face is a doubled coefficient and a Neumann face a zero one (the
// same products as mac_apply_cell's).
template <class T, int NSW, int SRC, bool REST>
static __global__ void __launch_bounds__(512) mac_reg_tile_kernel(MacTileArgs<T> a) {
    constexpr int NT = 512, TX = 8, R = REST ? 1 : 0;
    constexpr int HN = 2 * NSW + R - (SRC == MT_ZERO && NSW > 0 ? 1 : 0);
    constexpr int H = HN > 1 ? HN : 1, LX = TX + 2 * H, NC = LX * LX * LX / 2, SL = (NC + NT - 1) / NT;
    constexpr int SX = 1, SY = LX, SZ = LX * LX;
    __shared__ T xs[LX * LX * LX];
    __shared__ T rs[REST ? TX * TX * TX : 1];
    __shared__ int pos[3][LX];  // domain indices of the tile's columns, -1 outside
    const MGeomK& g = a.g;
    const int tid = threadIdx.x;
    const int lb = xcd_remap(blockIdx.x, a.gx * a.gy * a.gz);
    const int x0 = TX * (lb % a.gx), y0 = TX * ((lb / a.gx) % a.gy), z0 = TX * (lb / (a.gx * a.gy));
    if (tid < 3 * LX) {
        const int d = tid / LX, e = tid % LX;
        int v = (d == 0 ? x0 : (d == 1 ? y0 : z0)) - H + e;
        if (g.per[d]) v = ((v % g.n[d]) + g.n[d]) % g.n[d];
        pos[d][e] = v < 0 || v >= g.n[d] ? -1 : v;
    }
    __syncthreads();
    struct Cell {
        T t[6], b, dg, av;
        int off, depth;  // LDS index; layers outside the output tile (large: never updated)
    };
    Cell cell[2][SL];
#pragma unroll
    for (int col = 0; col < 2; ++col)
#pragma unroll
        for (int m = 0; m < SL; ++m) {
            Cell& c = cell[col][m];
            const int e = tid + NT * m;
            c.off = 0;
            c.depth = 1 << 20;
            if (e >= NC) continue;
            const int q = e % (LX / 2), r = e / (LX / 2), tj = r % LX, tk = r / LX;
            // tile origins are even, so the parity of a cell is that of its tile indices - 3 H
            const int ti = 2 * q + ((col + H + tj + tk) & 1);
            c.off = ti + LX * (tj + LX * tk);
            const int i = pos[0][ti], j = pos[1][tj], k = pos[2][tk];
            const bool in = i >= 0 && j >= 0 && k >= 0;
            T x = 0;
            if (SRC != MT_ZERO && in) {
                x = a.xin[cidx(g, i, j, k)];
                if (SRC == MT_PROLONG) x += a.xc[cidx(a.gc, i >> 1, j >> 1, k >> 1)];
            }
            xs[c.off] = x;
            auto out = [](int v) { return max(max(H - v, v - (H + TX - 1)), 0); };
            const int depth = max(max(out(ti), out(tj)), out(tk));
            // the layers this colour's first update reaches (REST: the tile itself)
            constexpr int reach0 = NSW > 0 ? 2 * NSW - 1 + R : 0, reach1 = NSW > 0 ? 2 * NSW - 2 + R : 0;
            if (in && (NSW > 0 || REST) && depth <= (col == 0 ? reach0 : reach1)) {
                const long f0 = i + (long)(g.n[0] + 1) * (j + (long)g.n[1] * k);
                const long f1 = i + (long)g.n[0] * (j + (long)(g.n[1] + 1) * k);
                const long f2 = cidx(g, i, j, k);
                const T bl[3] = {a.bx[f0], a.by[f1], a.bz[f2]};
                const T bh[3] = {a.bx[f0 + 1], a.by[f1 + g.n[0]], a.bz[f2 + (long)g.n[0] * g.n[1]]};
                const int p[3] = {i, j, k};
                c.b = a.b[f2];
                c.av = a.a ? a.a[f2] : (T)0;
                T dg = 0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    T lo = a.c.ih2[d] * bl[d], hi = a.c.ih2[d] * bh[d];
                    if (!(p[d] > 0 || g.per[d])) lo = g.dlo[d] ? 2 * lo : (T)0;
                    if (!(p[d] + 1 < g.n[d] || g.per[d])) hi = g.dhi[d] ? 2 * hi : (T)0;
                    c.t[2 * d] = lo;
                    c.t[2 * d + 1] = hi;
                    dg -= lo;
                    dg -= hi;
                }
                if (a.a) dg -= c.av;
                c.dg = dg;
                c.depth = depth;
            }
        }
    __syncthreads();
    auto resid = [&](const Cell& c, T pc) {
        const T* p = xs + c.off;
        T acc = 0;
        acc += c.t[0] * (p[-SX] - pc);
        acc += c.t[1] * (p[SX] - pc);
        acc += c.t[2] * (p[-SY] - pc);
        acc += c.t[3] * (p[SY] - pc);
        acc += c.t[4] * (p[-SZ] - pc);
        acc += c.t[5] * (p[SZ] - pc);
        if (a.a) acc -= c.av * pc;
        return c.b - acc;
    };
    // from zero the first colour sees no neighbours (and reaches the tile's edge)
    auto colour = [&](int col, int reach, bool first) {
#pragma unroll
        for (int m = 0; m < SL; ++m) {
            const Cell& c = cell[col][m];
            if (c.depth <= reach && c.dg != (T)0) {
                const T pc = first ? (T)0 : xs[c.off];
                xs[c.off] = pc + (first ? c.b : resid(c, pc)) / c.dg;
            }
        }
        __syncthreads();
    };
#pragma unroll
    for (int q = 0; q < NSW; ++q) {
        colour(0, 2 * (NSW - q) - 1 + R, SRC == MT_ZERO && q == 0);
        colour(1, 2 * (NSW - q) - 2 + R, false);
    }
    {
        // 512 output cells, one per thread
        const int ti = tid % TX, tj = (tid / TX) % TX, tk = tid / (TX * TX);
        const int i = x0 + ti, j = y0 + tj, k = z0 + tk;
        if (i < g.n[0] && j < g.n[1] && k < g.n[2])
            a.xout[cidx(g, i, j, k)] = xs[ti + H + LX * (tj + H + LX * (tk + H))];
    }
    if (REST) {
#pragma unroll
        for (int col = 0; col < 2; ++col)
#pragma unroll
            for (int m = 0; m < SL; ++m) {
                const Cell& c = cell[col][m];
                if (c.depth == 0) {
                    const int ti = c.off % LX - H, tj = (c.off / LX) % LX - H, tk = c.off / (LX * LX) - H;
                    rs[ti + TX * (tj + TX * tk)] = resid(c, xs[c.off]);
                }
            }
        __syncthreads();
        constexpr int CX = TX / 2;
        if (tid < CX * CX * CX) {
            const int ci = tid % CX, cj = (tid / CX) % CX, ck = tid / (CX * CX);
            const int I = x0 / 2 + ci, J = y0 / 2 + cj, K = z0 / 2 + ck;
            if (I < a.gc.n[0] && J < a.gc.n[1] && K < a.gc.n[2]) {
                T s = 0;
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    s += rs[2 * ci + (q & 1) + TX * (2 * cj + ((q >> 1) & 1) + TX * (2 * ck + (q >> 2)))];
                a.bc[cidx(a.gc, I, J, K)] = (T)0.125 * s;
            }
        }
    }
}

#pragma clang fp contract(fast)

template <class T, int NSW, int SRC, bool REST>
inline void mac_tile_launch(MacTileArgs<T> a, const MacTiles& tiles, hipStream_t s) {
    const long n = (long)a.g.n[0] * a.g.n[1] * a.g.n[2];
    a.gz = (a.g.n[2] + 7) / 8;
    if constexpr (NSW > 0)
        if (n > tiles.big) {
            a.gx = (a.g.n[0] + 15) / 16;
            a.gy = (a.g.n[1] + 15) / 16;
            mac_tile_kernel<T, 16, 16, 8, NSW, SRC, REST><<<a.gx * a.gy * a.gz, 512, 0, s>>>(a);
            return;
        }
    a.gx = (a.g.n[0] + 7) / 8;
    a.gy = (a.g.n[1] + 7) / 8;
    if constexpr (NSW > 0)
        if (n > tiles.reg) {
            mac_tile_kernel<T, 8, 8, 8, NSW, SRC, REST><<<a.gx * a.gy * a.gz, 512, 0, s>>>(a);
            return;
        }
    mac_reg_tile_kernel<T, NSW, SRC, REST><<<a.gx * a.gy * a.gz, 512, 0, s>>>(a);
}

template <class T, int NSW>
inline void mac_tile_leg(const MacTileArgs<T>& a, int src, bool rest, const MacTiles& tiles, hipStream_t s) {
    if (src == MT_ZERO) {
        if (rest) mac_tile_launch<T, NSW, MT_ZERO, true>(a, tiles, s);
        else mac_tile_launch<T, NSW, MT_ZERO, false>(a, tiles, s);
    } else if (src == MT_X) {
        if (rest) mac_tile_launch<T, NSW, MT_X, true>(a, tiles, s);
        else mac_tile_launch<T, NSW, MT_X, false>(a, tiles, s);
    } else {
        mac_tile_launch<T, NSW, MT_PROLONG, false>(a, tiles, s);
    }
}

// Launches of the down and the up leg, at most 2 sweeps each: the fewest with an
// even sum, after which the iterate is back in the buffer it started from (128^3
// cells with 3 + 3 sweeps: 2 + 2 launches)
inline void mac_leg_launches(int nu1, int nu2, int& down, int& up) {
    down = std::max(1, (nu1 + 1) / 2);
    up = std::max(1, (nu2 + 1) / 2);
    if ((down + up) % 2) ++(up > down ? up : down);  // that leg has 3 sweeps or more
}

// nu sweeps as m launches, alternating between the buffers (the first reads xa
// unless src is MT_ZERO)
template <class T>
inline void mac_tile_sweeps(MacTileArgs<T> a, int src, T* xa, T* xb, int nu, int m, bool rest,
                            const MacTiles& tiles, hipStream_t s) {
    for (int q = 0; q < m; ++q) {
        const int sw = std::min(2, nu - (m - 1 - q));  // leave at least one per later launch
        nu -= std::max(sw, 0);
        a.xin = q % 2 == 0 ? xa : xb;
        a.xout = q % 2 == 0 ? xb : xa;
        const int from = q == 0 ? src : MT_X;
        const bool r = rest && q == m - 1;
        if (sw >= 2) mac_tile_leg<T, 2>(a, from, r, tiles, s);
        else if (sw == 1) mac_tile_leg<T, 1>(a, from, r, tiles, s);
        else mac_tile_leg<T, 0>(a, from, r, tiles, s);
    }
}

}  // namespace mgx
