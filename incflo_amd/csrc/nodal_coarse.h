// nodal_coarse.h -- several coarse levels of the nodal V-cycle in one workgroup.
#pragma once

#include "bottom_kernels.h"

namespace mgx {

// ---- coarse levels: the whole V-cycle below a size threshold in one workgroup ----
// The levels are small enough that one workgroup sweeps each of them in a few
// microseconds, so running smoothing, residual, restriction, prolongation and
// the BiCGStab bottom solve back to back with workgroup barriers replaces
// about 7 launches per level.  Same operations, same order, as the per-level
// kernels.
constexpr int kMaxCoarse = 8;

template <class T>
struct CoarseLevel {
    KGeom g;
    Coef<T> c;
    T omega;
    const T* sig;
    T* b;
    T* x;
    T* x2;
    T* r;
    const unsigned char* m;  // overset mask (global memory), null without one
};

template <class T>
struct CoarseArgs {
    CoarseLevel<T> L[kMaxCoarse];
    int nl;           // levels in this launch (the last one is the bottom)
    int nu1, nu2;
    Coef<double> cb;  // bottom operator coefficients (double)
    BottomArgs bottom;
};

template <class T>
__device__ __forceinline__ void node_of(const KGeom& g, int id, int& i, int& j, int& k) {
    const int q = id / g.nn[0];
    i = id - q * g.nn[0];
    j = q % g.nn[1];
    k = q / g.nn[1];
}

// L x at node (i,j,k) with direct loads; also returns the sum of the 8 cell coefficients.
template <class T>
__device__ __forceinline__ T apply_node_T(const KGeom& g, const Coef<T>& c, const T* sig,
                                          const T* x, int i, int j, int k, T& ssum) {
    return apply_node_nbhd<T, T, T>(g, c, sig, x, i, j, k, ssum);
}

// Bytes of dynamic LDS the coarse kernel needs for levels L[0..nl-1]: every
// level's sigma, b, x, x2 and r (r shares x2's storage) and the bottom
// solver's multiplied vector.
template <class T>
inline size_t coarse_lds_bytes(const KGeom* g, int nl) {
    size_t b = 0;
    for (int l = 0; l < nl; ++l) {
        const size_t nn = (size_t)g[l].nn[0] * g[l].nn[1] * g[l].nn[2];
        const size_t ns = (size_t)g[l].sg[0] * g[l].sg[1] * g[l].sg[2];
        b += ((ns + 3 * nn) * sizeof(T) + 15) / 16 * 16;
    }
    const size_t nb = (size_t)g[nl - 1].nn[0] * g[nl - 1].nn[1] * g[nl - 1].nn[2];
    return b + nb * sizeof(double);
}

// The whole coarse hierarchy lives in LDS for the duration of the launch:
// sigma and the top level's rhs are copied in, the top level's correction is
// copied out; everything in between never touches global memory.
template <class T>
static __global__ void __launch_bounds__(512) coarse_vcycle_kernel(const CoarseArgs<T> a) {
    __shared__ BottomRed red;
    __shared__ CoarseLevel<T> sl[kMaxCoarse];  // level descriptors with LDS pointers
    __shared__ double* swork;
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, nt = blockDim.x;
    if (tid == 0) {
        size_t off = 0;
        for (int l = 0; l < a.nl; ++l) {
            CoarseLevel<T> lv = a.L[l];
            const int nn = lv.g.nn[0] * lv.g.nn[1] * lv.g.nn[2];
            const int ns = lv.g.sg[0] * lv.g.sg[1] * lv.g.sg[2];
            T* base = reinterpret_cast<T*>(lds + off);
            lv.sig = base;
            lv.b = base + ns;
            lv.x = base + ns + nn;
            lv.x2 = base + ns + 2 * nn;
            lv.r = lv.x2;  // the residual is formed after smoothing, when x2 is free
            sl[l] = lv;
            off += ((size_t)(ns + 3 * nn) * sizeof(T) + 15) / 16 * 16;
        }
        swork = reinterpret_cast<double*>(lds + off);
    }
    __syncthreads();
    for (int l = 0; l < a.nl; ++l) {
        const int ns = sl[l].g.sg[0] * sl[l].g.sg[1] * sl[l].g.sg[2];
        T* dst = const_cast<T*>(sl[l].sig);
        const T* src = a.L[l].sig;
        for (int id = tid; id < ns; id += nt) dst[id] = src[id];
    }
    {
        const int nn = sl[0].g.nn[0] * sl[0].g.nn[1] * sl[0].g.nn[2];
        for (int id = tid; id < nn; id += nt) sl[0].b[id] = a.L[0].b[id];
    }
    __syncthreads();
    T* top_x_global = a.L[0].x;
    unsigned swmask = 0u;  // bit l: level l's current iterate is in x2
    auto cur = [&](int l) { return ((swmask >> l) & 1u) ? sl[l].x2 : sl[l].x; };
    auto oth = [&](int l) { return ((swmask >> l) & 1u) ? sl[l].x : sl[l].x2; };
    auto jacobi = [&](int l) {
        const CoarseLevel<T>& lv = sl[l];
        const int n = lv.g.nn[0] * lv.g.nn[1] * lv.g.nn[2];
        const T* xin = cur(l);
        T* xout = oth(l);
        for (int id = tid; id < n; id += nt) {
            int i, j, k;
            node_of<T>(lv.g, id, i, j, k);
            T ssum;
            const T acc = apply_node_T<T>(lv.g, lv.c, lv.sig, xin, i, j, k, ssum);
            T v = xin[id];
            if (node_fixed(lv.g, lv.m, id, i, j, k)) v = 0;
            else if (ssum != (T)0) v = v + lv.omega * (lv.b[id] - acc) / (-lv.c.diag4 * ssum);
            xout[id] = v;
        }
        swmask ^= (1u << l);
        __syncthreads();
    };
    // down
    for (int l = 0; l < a.nl - 1; ++l) {
        const CoarseLevel<T>& lv = sl[l];
        const int n = lv.g.nn[0] * lv.g.nn[1] * lv.g.nn[2];
        if (a.nu1 > 0) {
            T* x = cur(l);
            for (int id = tid; id < n; id += nt) {
                int i, j, k;
                node_of<T>(lv.g, id, i, j, k);
                T ssum = 0;
                for (int q = 0; q < 8; ++q)
                    ssum += lv.sig[(i + (q & 1)) + (long)lv.g.sg[0] * ((j + ((q >> 1) & 1)) +
                                                                    (long)lv.g.sg[1] * (k + ((q >> 2) & 1)))];
                x[id] = (node_fixed(lv.g, lv.m, id, i, j, k) || ssum == (T)0)
                            ? (T)0
                            : lv.omega * lv.b[id] / (-lv.c.diag4 * ssum);
            }
            __syncthreads();
            for (int s = 1; s < a.nu1; ++s) jacobi(l);
        } else {
            T* x = cur(l);
            for (int id = tid; id < n; id += nt) x[id] = 0;
            __syncthreads();
        }
        {
            const T* x = cur(l);
            for (int id = tid; id < n; id += nt) {
                int i, j, k;
                node_of<T>(lv.g, id, i, j, k);
                T ssum;
                const T acc = apply_node_T<T>(lv.g, lv.c, lv.sig, x, i, j, k, ssum);
                oth(l)[id] = node_fixed(lv.g, lv.m, id, i, j, k) ? (T)0 : lv.b[id] - acc;
            }
            __syncthreads();
        }
        {
            const CoarseLevel<T>& cv = sl[l + 1];
            const T* rf = oth(l);  // the residual just formed
            const KGeom& gf = lv.g;
            const KGeom& gc = cv.g;
            const int nc = gc.nn[0] * gc.nn[1] * gc.nn[2];
            for (int id = tid; id < nc; id += nt) {
                int I, J, K;
                node_of<T>(gc, id, I, J, K);
                T acc = 0;
                if (!node_fixed(gc, cv.m, id, I, J, K)) {
                    for (int oz = -1; oz <= 1; ++oz) {
                        int fk = 2 * K + oz;
                        if (gf.per[2]) fk = fk < 0 ? fk + gf.nn[2] : (fk >= gf.nn[2] ? fk - gf.nn[2] : fk);
                        else if (fk < 0 || fk >= gf.nn[2]) continue;
                        for (int oy = -1; oy <= 1; ++oy) {
                            int fj = 2 * J + oy;
                            if (gf.per[1]) fj = fj < 0 ? fj + gf.nn[1] : (fj >= gf.nn[1] ? fj - gf.nn[1] : fj);
                            else if (fj < 0 || fj >= gf.nn[1]) continue;
                            for (int ox = -1; ox <= 1; ++ox) {
                                int fi = 2 * I + ox;
                                if (gf.per[0]) fi = fi < 0 ? fi + gf.nn[0] : (fi >= gf.nn[0] ? fi - gf.nn[0] : fi);
                                else if (fi < 0 || fi >= gf.nn[0]) continue;
                                const T w = (ox ? (T)0.25 : (T)0.5) * (oy ? (T)0.25 : (T)0.5) *
                                            (oz ? (T)0.25 : (T)0.5);
                                acc += w * rf[fi + (long)gf.nn[0] * (fj + (long)gf.nn[1] * fk)];
                            }
                        }
                    }
                }
                cv.b[id] = acc;
            }
            __syncthreads();
        }
    }
    // bottom
    {
        const int lb = a.nl - 1;
        const NodalRows<T> op{sl[lb].g, a.cb, sl[lb].sig, sl[lb].m};
        RowPlan<NodalRows<T>, 0, false> plan(op, a.bottom.work);
        bottom_krylov(plan, sl[lb].b, cur(lb), a.bottom, swork, a.bottom.work + 27L * plan.size(), red);
        __syncthreads();
    }
    // up
    for (int l = a.nl - 2; l >= 0; --l) {
        const CoarseLevel<T>& lv = sl[l];
        const KGeom& gf = lv.g;
        const KGeom& gc = sl[l + 1].g;
        const T* xc = cur(l + 1);
        T* xf = cur(l);
        const int nf = gf.nn[0] * gf.nn[1] * gf.nn[2];
        for (int id = tid; id < nf; id += nt) {
            int i, j, k;
            node_of<T>(gf, id, i, j, k);
            if (node_fixed(gf, lv.m, id, i, j, k)) continue;
            const int f[3] = {i, j, k};
            int lo[3], hi[3];
            for (int d = 0; d < 3; ++d) {
                lo[d] = f[d] >> 1;
                hi[d] = (f[d] & 1) ? lo[d] + 1 : lo[d];
                if (gc.per[d] && hi[d] >= gc.nn[d]) hi[d] -= gc.nn[d];
            }
            T acc = 0;
            for (int q = 0; q < 8; ++q) {
                const int I = (q & 1) ? hi[0] : lo[0];
                const int J = (q & 2) ? hi[1] : lo[1];
                const int K = (q & 4) ? hi[2] : lo[2];
                acc += xc[I + (long)gc.nn[0] * (J + (long)gc.nn[1] * K)];
            }
            xf[id] += (T)0.125 * acc;
        }
        __syncthreads();
        for (int s = 0; s < a.nu2; ++s) jacobi(l);
    }
    // the top level's correction goes back to global memory
    {
        const CoarseLevel<T>& lv = sl[0];
        const int n = lv.g.nn[0] * lv.g.nn[1] * lv.g.nn[2];
        const T* xs = cur(0);
        for (int id = tid; id < n; id += nt) top_x_global[id] = xs[id];
    }
}

}  // namespace mgx
