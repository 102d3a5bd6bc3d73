// bottom_kernels.h -- the bottom solve of the nodal, EB nodal and cell-centred
// multigrid: Krylov solvers on the bottom level's stencil matrix in one
// workgroup, FP64.
//
// What bounds it: one workgroup iterates on a few hundred to a few thousand
// unknowns, so the time is a serial chain of stencil products, reductions and
// barriers; no other CU can help without device-wide barriers, which cost as
// much as the whole product.  Hence
//   * the operator is scaled symmetrically by the diagonal (S L S with S =
//     |diag|^-1/2), which evens out wall rows and small cut cells and needs fewer
//     iterations.  Its rows (27 or 7 coefficients) are assembled once per solve:
//     in registers up to 512 unknowns (1024 of 27, 2048 of 7 points for the EB and
//     cell-centred operators), streamed from L2 above.  On nodal levels of more
//     than 512 nodes columns of nodes work from the cell coefficients instead,
//     but for levels up to 4096 nodes that 512 threads do not hold in columns;
//   * each thread owns fixed unknowns, whose vector elements stay in registers
//     up to 4096 unknowns; only the multiplied vector goes through LDS, up to
//     19200 unknowns;
//   * reductions run on DPP row shifts and one barrier, several values at a
//     time: BiCGStab takes two reductions per iteration (the next rho by its
//     recurrence, the residual norm together with the next product), CG one
//     (Chronopoulos and Gear 1989).
// Measured on MI355X per solve (default options), against an unscaled solver
// with its vectors and index divisions in LDS or global memory before it:
//   nodal 1280 nodes (120 x 72 x 56 channel)          592 -> 150 us
//   nodal 2275 nodes (256 x 16 x 24 channel)         2370 -> 527 us
//   nodal 10440 nodes (224 x 232 x 88 channel)       5280 -> 3570 us
//   EB nodal 425 nodes (256 x 64 x 64 channel)       1130 -> 70 us
//   MAC 480 cells (160 x 24 x 16 channel at 2 levels) 1320 -> 200 us
#pragma once

#include <hip/hip_runtime.h>

#include "mgx_common.h"
#include "nodal_kernels.h"

namespace mgx {

// The bottom_solver choices of MLMG (MGX_BOTTOM_*): BiCGStab (van der Vorst
// 1992), CG (Hestenes and Stiefel 1952), BiCGStab and then CG from zero when
// the first one fails ("bicgcg"), the reverse ("cgbicg"), or smoothing sweeps
// only ("smoother").  A Krylov solve that does not reach rtol is followed by
// kBottomSmooths smoothing sweeps, from zero when it broke down (a zero
// inner product).  The operators are negative (semi-)definite and symmetric.
constexpr int kBottomSmooths = 8;

struct BottomArgs {
    double* work;    // BottomPlan::work doubles
    int kind;        // MGX_BOTTOM_*
    int maxiter;
    double rtol;
    double omega;    // weighted-Jacobi factor of the smoothing sweeps (nodal rows)
    int singular;
    int* iters_acc;  // may be null
};

// ---- wave and workgroup reductions ----
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_get(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int LANE>
__device__ __forceinline__ double lane_get(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, LANE);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), LANE);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// sums (MAX: maxima of non-negative values) by row shifts: lanes without a
// source take 0, which leaves both unchanged
template <bool MAX>
__device__ __forceinline__ double red_op(double a, double b) { return MAX ? fmax(a, b) : a + b; }

// over each row of 16 lanes, the result in lane 15 of the row
template <bool MAX>
__device__ __forceinline__ double row_reduce(double v) {
    v = red_op<MAX>(v, dpp_get<0x111, 0xf>(v));  // row_shr:1
    v = red_op<MAX>(v, dpp_get<0x112, 0xf>(v));  // row_shr:2
    v = red_op<MAX>(v, dpp_get<0x114, 0xf>(v));  // row_shr:4
    v = red_op<MAX>(v, dpp_get<0x118, 0xf>(v));  // row_shr:8
    return v;
}

template <bool MAX>
__device__ __forceinline__ double wave_reduce(double v) {
    v = row_reduce<MAX>(v);
    v = red_op<MAX>(v, dpp_get<0x142, 0xa>(v));  // row_bcast:15 into rows 1 and 3
    v = red_op<MAX>(v, dpp_get<0x143, 0xc>(v));  // row_bcast:31 into rows 2 and 3
    return lane_get<63>(v);
}

// NV values over the workgroup (bit i of MAXMASK: value i is a maximum), the
// same in every thread.  One barrier: the buffers alternate, so a wave that
// runs ahead writes the other one.
constexpr int kBottomRed = 5;
struct BottomRed {
    double v[2][kBottomRed][16];
};

template <int NV, unsigned MAXMASK>
__device__ __forceinline__ void block_reduce(double (&v)[NV], BottomRed& red, int& phase) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        v[i] = (MAXMASK >> i) & 1u ? wave_reduce<true>(v[i]) : wave_reduce<false>(v[i]);
    if (nw > 1) {
        if (lane == 0)
#pragma unroll
            for (int i = 0; i < NV; ++i) red.v[phase][i][wv] = v[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const double t = (lane & 15) < nw ? red.v[phase][i][lane & 15] : 0.0;
            v[i] = lane_get<15>((MAXMASK >> i) & 1u ? row_reduce<true>(t) : row_reduce<false>(t));
        }
        phase ^= 1;
    } else {
        __syncthreads();
    }
}

// ---- rows of the three operators ----
// row(): the coefficients of (L x) at the point, C[slot], and whether the
// point is an unknown.  Slots: 27 points x fastest, or centre and the six
// neighbours (-x, +x, -y, +y, -z, +z).  kRedBlack: the smoothing sweeps update
// one colour after the other, else weighted Jacobi.
template <class TS>
struct NodalRows {
    static constexpr int NS = 27;
    static constexpr bool kRedBlack = false, kNodal = true;
    KGeom g;
    Coef<double> c;
    const TS* sig;
    const unsigned char* m;  // overset mask, may be null
    __host__ __device__ int dim(int d) const { return g.nn[d]; }
    __device__ int per(int d) const { return g.per[d]; }
    __device__ bool row(int id, int i, int j, int k, double (&C)[NS]) const {
        double S[2][2][2];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    S[p][r][q] = (double)sig[(i + q) + (long)g.sg[0] * ((j + r) + (long)g.sg[1] * (k + p))];
        double sum = 0.0;
#pragma unroll
        for (int s = 0; s < 27; ++s) {
            const int o[3] = {s % 3, (s / 3) % 3, s / 9};
            double t = 0.0;
            // the cells shared by the two nodes
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int cq[3] = {q & 1, (q >> 1) & 1, q >> 2};
                bool in = true;
#pragma unroll
                for (int d = 0; d < 3; ++d) in = in && (o[d] == 1 || o[d] == 2 * cq[d]);
                if (in) t += S[cq[2]][cq[1]][cq[0]];
            }
            const int nz = (o[0] == 1) + (o[1] == 1) + (o[2] == 1);  // zero offsets
            double w = 0.0;
            if (nz == 0) w = c.corner;
            else if (nz == 1) w = c.edge[o[0] == 1 ? 0 : (o[1] == 1 ? 1 : 2)];
            else if (nz == 2) w = c.face[o[0] != 1 ? 0 : (o[1] != 1 ? 1 : 2)];
            C[s] = w * t;
            if (nz == 3) sum = t;
        }
        C[13] = -c.diag4 * sum;
        return !node_fixed(g, m, id, i, j, k);
    }
};

// ---- the scaled operator A = -S L S, S = |diag|^-1/2, over the workgroup ----
// A plan maps unknowns to threads (q < NPT or count(); each(f) calls f(q, id) for
// those that are unknowns of the level) and multiplies.  setup() returns the
// diagonal per unknown (0: not an unknown), scale() receives S through xs,
// apply() reads the vector in xs.  kDirect: the vectors of all threads together
// are laid out by id, so that apply() reads them where they are.

// Coefficient rows: in registers (CREG), or slot-major in global memory.  NPT
// 0: any number of unknowns, nothing per unknown in registers; DIRECT: their
// multiplied vector is not copied (it would not fit LDS).
template <class Rows, int NPT_, bool CREG, bool DIRECT = false>
struct RowPlan {
    static constexpr bool kDirect = DIRECT;
    static constexpr int NPT = NPT_, NS = Rows::NS;
    static constexpr bool kRedBlack = Rows::kRedBlack;
    static constexpr bool kScaled = true;  // apply() multiplies by A, not -L
    struct Nbr {  // neighbour indices: sums of one x, one y and one z offset
        int x[3], y[3], z[3];
    };
    const Rows& op;
    double* cg;  // slot s of unknown id at cg[s n + id]
    int tid, nt, d0, d1, d2, n;
    double cr[CREG ? NPT : 1][CREG ? NS : 1];
    Nbr nb[NPT ? NPT : 1];

    __device__ RowPlan(const Rows& o, double* work)
        : op(o), cg(work), tid(threadIdx.x), nt(blockDim.x), d0(o.dim(0)), d1(o.dim(1)), d2(o.dim(2)),
          n(o.dim(0) * o.dim(1) * o.dim(2)) {}
    __device__ int size() const { return n; }
    __device__ long stride() const { return n; }
    __device__ int count() const { return (n - tid + nt - 1) / nt; }
    __device__ int id(int q) const { return tid + q * nt; }
    __device__ bool live(int q) const { return NPT == 0 || id(q) < n; }
    template <class F>
    __device__ void each(F f) const {
#pragma unroll
        for (int q = 0; q < (NPT ? NPT : count()); ++q)
            if (live(q)) f(q, id(q));
    }
    __device__ void point(int id, int& i, int& j, int& k) const {
        i = id % d0;
        const int t = id / d0;
        j = t % d1;
        k = t / d1;
    }
    __device__ Nbr nbr_of(int id) const {
        int i, j, k;
        point(id, i, j, k);
        Nbr o;
        o.x[1] = i;
        o.x[0] = i > 0 ? i - 1 : (op.per(0) ? d0 - 1 : 0);
        o.x[2] = i + 1 < d0 ? i + 1 : (op.per(0) ? 0 : i);
        o.y[1] = d0 * j;
        o.y[0] = d0 * (j > 0 ? j - 1 : (op.per(1) ? d1 - 1 : 0));
        o.y[2] = d0 * (j + 1 < d1 ? j + 1 : (op.per(1) ? 0 : j));
        o.z[1] = d0 * d1 * k;
        o.z[0] = d0 * d1 * (k > 0 ? k - 1 : (op.per(2) ? d2 - 1 : 0));
        o.z[2] = d0 * d1 * (k + 1 < d2 ? k + 1 : (op.per(2) ? 0 : k));
        return o;
    }
    __device__ static int nbr_at(const Nbr& o, int s) {
        if constexpr (NS == 27) return o.x[s % 3] + o.y[(s / 3) % 3] + o.z[s / 9];
        else
            return o.x[s == 1 ? 0 : (s == 2 ? 2 : 1)] + o.y[s == 3 ? 0 : (s == 4 ? 2 : 1)] +
                   o.z[s == 5 ? 0 : (s == 6 ? 2 : 1)];
    }
    __device__ double one_row(int id, double (&c)[NS]) const {
        int i, j, k;
        point(id, i, j, k);
        const bool free = op.row(id, i, j, k, c);
        const double dg = -c[NS == 27 ? 13 : 0];
        return free && dg > 0.0 ? dg : 0.0;
    }
    // put(q, diagonal)
    template <class F>
    __device__ void setup(F put) {
        if constexpr (CREG) {
#pragma unroll
            for (int q = 0; q < NPT; ++q) {
                nb[q] = nbr_of(live(q) ? id(q) : 0);
                double dg = 0.0;
#pragma unroll
                for (int s = 0; s < NS; ++s) cr[q][s] = 0.0;
                if (live(q)) dg = one_row(id(q), cr[q]);
                put(q, dg);
            }
        } else {
            // one row at a time (unrolled, the rows of a thread would spill);
            // the diagonal slot carries the diagonal to the second loop
#pragma unroll 1
            for (int e = tid; e < n; e += nt) {
                double c[NS];
                const double dg = one_row(e, c);
#pragma unroll
                for (int s = 0; s < NS; ++s) cg[(long)s * n + e] = c[s];
                if (dg == 0.0) cg[(long)(NS == 27 ? 13 : 0) * n + e] = 0.0;
            }
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : count()); ++q) {
                if constexpr (NPT > 0) nb[q] = nbr_of(live(q) ? id(q) : 0);
                put(q, live(q) ? -cg[(long)(NS == 27 ? 13 : 0) * n + id(q)] : 0.0);
            }
        }
    }
    // rows times -s of both points (xs: s)
    __device__ void scale(const double* xs) {
        if constexpr (CREG) {
#pragma unroll
            for (int q = 0; q < NPT; ++q) {
                const double si = live(q) ? xs[id(q)] : 0.0;
#pragma unroll
                for (int s = 0; s < NS; ++s) cr[q][s] *= -si * xs[nbr_at(nb[q], s)];
            }
        } else {
#pragma unroll 1
            for (int e = tid; e < n; e += nt) {
                const Nbr o = nbr_of(e);
                const double si = xs[e];
#pragma unroll
                for (int s = 0; s < NS; ++s) cg[(long)s * n + e] *= -si * xs[nbr_at(o, s)];
            }
        }
    }
    // put(q, (A x)_q)
    template <class F>
    __device__ void apply(const double* xs, F put) {
        const double* c = cg + tid;
        // opaque per call: the loads must not be hoisted out of the iteration
        // (they would not fit the registers and come back from scratch)
        if constexpr (!CREG) asm volatile("" : "+v"(c));
#pragma unroll
        for (int q = 0; q < (NPT ? NPT : count()); ++q) {
            double acc = 0.0;
            if (live(q)) {
                Nbr o = NPT > 0 ? nb[NPT ? q : 0] : nbr_of(id(q));
                // (nor the sums of the neighbour offsets)
                if constexpr (NPT > 1) asm volatile("" : "+v"(o.x[0]), "+v"(o.x[1]), "+v"(o.x[2]));
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const double w = CREG ? cr[CREG ? q : 0][CREG ? s : 0] : c[(long)s * n + q * nt];
                    acc += w * xs[nbr_at(o, s)];
                }
            }
            put(q, acc);
        }
    }
};

// (L x) of a node from its planes of values (below, at, above) and cell
// coefficients (below, above); weights in (a, b, march) order
__device__ __forceinline__ double col_node(const double (&x0)[3][3], const double (&x1)[3][3],
                                           const double (&x2)[3][3], const double (&s0)[2][2],
                                           const double (&s1)[2][2], const Coef<double>& c) {
    double ac = 0, a2 = 0, a1 = 0, a0 = 0, f0 = 0, f1 = 0;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            ac += s0[b][a] * x0[2 * b][2 * a] + s1[b][a] * x2[2 * b][2 * a];
            a2 += (s0[b][a] + s1[b][a]) * x1[2 * b][2 * a];
        }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const double l1 = s0[0][a] + s0[1][a], h1 = s1[0][a] + s1[1][a];
        const double l0 = s0[a][0] + s0[a][1], h0 = s1[a][0] + s1[a][1];
        a1 += l1 * x0[1][2 * a] + h1 * x2[1][2 * a];
        a0 += l0 * x0[2 * a][1] + h0 * x2[2 * a][1];
        f0 += (l1 + h1) * x1[1][2 * a];
        f1 += (l0 + h0) * x1[2 * a][1];
    }
    const double t0 = s0[0][0] + s0[0][1] + s0[1][0] + s0[1][1];
    const double t1 = s1[0][0] + s1[0][1] + s1[1][0] + s1[1][1];
    return c.corner * ac + c.edge[2] * a2 + c.edge[1] * a1 + c.edge[0] * a0 +
                     c.face[0] * f0 + c.face[1] * f1 + c.face[2] * (t0 * x0[1][1] + t1 * x2[1][1]) -
                     c.diag4 * (t0 + t1) * x1[1][1];
}

// The nodal operator without stored rows: a thread owns NPT consecutive nodes
// along one axis, so a plane of 3 x 3 values read from LDS serves three of its
// products: 9 (NPT + 2) LDS reads instead of 27 NPT, and 4 (NPT + 1) of the
// cell coefficients, which are copied to LDS once.
template <class TS, int NPT_>
struct ColPlan {
    static constexpr int NPT = NPT_;
    static constexpr bool kRedBlack = false, kScaled = false, kDirect = false;
    const NodalRows<TS>& op;
    int na, nbk, nm, nseg;      // nodes along the two cross axes and the march axis
    int sa, sb, sm;             // id strides
    int ca, cb, m0;             // this thread's column and first node
    bool on;
    int oa[3], ob[3];           // neighbour offsets across
    int om[NPT + 2];            // offsets of the planes m0 - 1 .. m0 + NPT
    Coef<double> c;             // weights in (a, b, march) order
    const TS* ls;               // sigma in LDS, this thread's first cell column
    int gs[3];                  // its strides (a, b, march)
    int gm;                     // last plane from m0

    // lsig: LDS for the ghosted cell coefficients
    __device__ ColPlan(const NodalRows<TS>& o, int axis, TS* lsig) : op(o) {
        const int ns = o.g.sg[0] * o.g.sg[1] * o.g.sg[2];
        for (int e = threadIdx.x; e < ns; e += blockDim.x) lsig[e] = o.sig[e];
        __syncthreads();
        const int a = axis == 0 ? 1 : 0, b = axis == 2 ? 1 : 2;
        const int st[3] = {1, o.dim(0), o.dim(0) * o.dim(1)};
        na = o.dim(a);
        nbk = o.dim(b);
        nm = o.dim(axis);
        sa = st[a];
        sb = st[b];
        sm = st[axis];
        nseg = (nm + NPT - 1) / NPT;
        const int t = threadIdx.x, col = na * nbk;
        on = t < col * nseg;
        const int cc = on ? t % col : 0;
        ca = cc % na;
        cb = cc / na;
        m0 = on ? NPT * (t / col) : 0;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            oa[r] = sa * wrapc(ca - 1 + r, na, o.per(a));
            ob[r] = sb * wrapc(cb - 1 + r, nbk, o.per(b));
        }
#pragma unroll
        for (int p = 0; p < NPT + 2; ++p) om[p] = sm * wrapc(min(m0 - 1 + p, nm), nm, o.per(axis));
        c = o.c;
        c.edge[0] = o.c.edge[a];
        c.edge[1] = o.c.edge[b];
        c.edge[2] = o.c.edge[axis];
        c.face[0] = o.c.face[a];
        c.face[1] = o.c.face[b];
        c.face[2] = o.c.face[axis];
        const int g3[3] = {1, o.g.sg[0], o.g.sg[0] * o.g.sg[1]};
        gs[0] = g3[a];
        gs[1] = g3[b];
        gs[2] = g3[axis];
        gm = o.g.sg[axis] - 1 - m0;
        ls = lsig + gs[0] * ca + gs[1] * cb + gs[2] * m0;
    }
    // the four cells of plane l around the column
    __device__ void cells(double (&s)[2][2], int l) const {
        int m = gs[2] * min(l, gm);
        asm volatile("" : "+v"(m));
        const TS* p = ls + m;
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q >> 1][q & 1] = (double)p[gs[0] * (q & 1) + gs[1] * (q >> 1)];
    }
    __device__ int size() const { return na * nbk * nm; }
    __device__ long stride() const { return 0; }
    __device__ int count() const { return NPT; }
    __device__ bool live(int q) const { return on && m0 + q < nm; }
    __device__ int id(int q) const { return sa * ca + sb * cb + sm * min(m0 + q, nm - 1); }
    template <class F>
    __device__ void each(F f) const {
#pragma unroll
        for (int q = 0; q < NPT; ++q)
            if (live(q)) f(q, id(q));
    }
    template <class F>
    __device__ void setup(F put) {
#pragma unroll
        for (int q = 0; q < NPT; ++q) {
            double s0[2][2], s1[2][2], t = 0.0;
            cells(s0, q);
            cells(s1, q + 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) t += s0[r >> 1][r & 1] + s1[r >> 1][r & 1];
            const int e = id(q), i = e % op.dim(0), w = e / op.dim(0);
            const bool free = live(q) && t > 0.0 &&
                              !node_fixed(op.g, op.m, e, i, w % op.dim(1), w / op.dim(1));
            put(q, free ? c.diag4 * t : 0.0);
        }
    }
    __device__ void scale(const double*) {}
    // put(q, (-L x)_q); the caller multiplies by S on both sides
    template <class F>
    __device__ void apply(const double* xs, F put) {
        double X[3][3][3];  // planes below, at and above the node
        auto plane = [&](double (&x)[3][3], int p) {
            // opaque: the addresses of all planes, hoisted out of the iteration,
            // would take over a hundred registers
            int m = om[p];
            asm volatile("" : "+v"(m));
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int q = 0; q < 3; ++q) x[r][q] = xs[oa[q] + ob[r] + m];
        };
        double G[2][2][2];  // cell planes below and above the node
        plane(X[0], 0);
        plane(X[1], 1);
        cells(G[0], 0);
#pragma unroll
        for (int q = 0; q < NPT; ++q) {
            const auto &x0 = X[q % 3], &x1 = X[(q + 1) % 3];
            auto& x2 = X[(q + 2) % 3];
            plane(x2, q + 2);
            cells(G[(q + 1) & 1], q + 1);
            const auto &s0 = G[q & 1], &s1 = G[(q + 1) & 1];
            const double v = col_node(x0, x1, x2, s0, s1, c);
            put(q, -v);
            // (the loads of later planes, hoisted, would not fit the registers)
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// The same for levels whose vectors do not fit the registers: a thread owns
// segments of `len` nodes of columns along `axis` (items, column fastest), its
// vectors lie in global memory in the order it visits them.
template <class TS>
struct WidePlan {
    static constexpr int NPT = 0;
    static constexpr bool kRedBlack = false, kScaled = false, kDirect = false;
    const NodalRows<TS>& op;
    int axis, len, a, b, na, ncol, nm, sa, sb, sm, items;
    Coef<double> c;
    __device__ WidePlan(const NodalRows<TS>& o, int axis_, int len_)
        : op(o), axis(axis_), len(len_), a(axis_ == 0 ? 1 : 0), b(axis_ == 2 ? 1 : 2), c(o.c) {
        const int st[3] = {1, o.dim(0), o.dim(0) * o.dim(1)};
        na = o.dim(a);
        ncol = na * o.dim(b);
        nm = o.dim(axis);
        sa = st[a];
        sb = st[b];
        sm = st[axis];
        items = ncol * ((nm + len - 1) / len);
        c.edge[0] = o.c.edge[a];
        c.edge[1] = o.c.edge[b];
        c.edge[2] = o.c.edge[axis];
        c.face[0] = o.c.face[a];
        c.face[1] = o.c.face[b];
        c.face[2] = o.c.face[axis];
    }
    __device__ int size() const { return ncol * nm; }
    // this thread's items
    __device__ int mine() const {
        return (int)threadIdx.x < items ? (items - (int)threadIdx.x + (int)blockDim.x - 1) / (int)blockDim.x : 0;
    }
    __device__ int count() const { return mine() * len; }
    // doubles a vector takes (every thread's share padded to the longest)
    __device__ long stride() const { return (long)((items + blockDim.x - 1) / blockDim.x) * len * blockDim.x; }
    // f(w, ca, cb, m0, m1): item w, its column and its nodes m0 .. m1 - 1
    template <class F>
    __device__ void each_item(F f) const {
        const int cnt = mine();
        for (int w = 0; w < cnt; ++w) {
            const int it = threadIdx.x + w * blockDim.x, sg = it / ncol, cc = it - sg * ncol, cb = cc / na;
            f(w, cc - cb * na, cb, sg * len, min(sg * len + len, nm));
        }
    }
    template <class F>
    __device__ void each(F f) const {
        each_item([&](int w, int ca, int cb, int m0, int m1) {
            for (int m = m0; m < m1; ++m) f(w * len + m - m0, sa * ca + sb * cb + sm * m);
        });
    }
    __device__ void cells(double (&s)[2][2], int ca, int cb, int l) const {
        const int g3[3] = {1, op.g.sg[0], op.g.sg[0] * op.g.sg[1]};
        const TS* p = op.sig + (long)g3[a] * ca + (long)g3[b] * cb + (long)g3[axis] * l;
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q >> 1][q & 1] = (double)p[g3[a] * (q & 1) + g3[b] * (q >> 1)];
    }
    template <class F>
    __device__ void setup(F put) {
        each_item([&](int w, int ca, int cb, int m0, int m1) {
            double s0[2][2], s1[2][2];
            cells(s0, ca, cb, m0);
            for (int m = m0; m < m1; ++m) {
                cells(s1, ca, cb, m + 1);
                double t = 0.0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    t += s0[r >> 1][r & 1] + s1[r >> 1][r & 1];
                    s0[r >> 1][r & 1] = s1[r >> 1][r & 1];
                }
                const int e = sa * ca + sb * cb + sm * m, i = e % op.dim(0), v = e / op.dim(0);
                const bool free = t > 0.0 && !node_fixed(op.g, op.m, e, i, v % op.dim(1), v / op.dim(1));
                put(w * len + m - m0, free ? c.diag4 * t : 0.0);
            }
            for (int m = m1; m < m0 + len; ++m) put(w * len + m - m0, 0.0);
        });
    }
    __device__ void scale(const double*) {}
    template <class F>
    __device__ void apply(const double* xs, F put) {
        each_item([&](int w, int ca, int cb, int m0, int m1) {
            int o[3][3];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    o[r][q] = sa * wrapc(ca - 1 + q, na, op.per(a)) + sb * wrapc(cb - 1 + r, ncol / na, op.per(b));
            double X[3][3][3], G[2][2][2];
            auto plane = [&](double (&x)[3][3], int m) {
                const int e = sm * wrapc(m, nm, op.per(axis));
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int q = 0; q < 3; ++q) x[r][q] = xs[o[r][q] + e];
            };
            plane(X[0], m0 - 1);
            plane(X[1], m0);
            cells(G[0], ca, cb, m0);
            for (int m = m0; m < m1; ++m) {
                plane(X[2], m + 1);
                cells(G[1], ca, cb, m + 1);
                put(w * len + m - m0, -col_node(X[0], X[1], X[2], G[0], G[1], c));
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        X[0][r][q] = X[1][r][q];
                        X[1][r][q] = X[2][r][q];
                    }
#pragma unroll
                for (int q = 0; q < 4; ++q) G[0][q >> 1][q & 1] = G[1][q >> 1][q & 1];
            }
            for (int m = m1; m < m0 + len; ++m) put(w * len + m - m0, 0.0);
        });
    }
};

// ---- the solve ----
// Vector elements of this thread's unknowns: registers (NPT > 0) or global memory.
template <int NPT>
struct OwnVec {
    double v[NPT];
    __device__ void at(double*, int, int) {}
    __device__ double& operator[](int q) { return v[q]; }
};
template <>
struct OwnVec<0> {
    double* p;
    int nt;
    __device__ void at(double* base, int tid, int nt_) { p = base + tid; nt = nt_; }
    __device__ double& operator[](int q) { return p[(long)q * nt]; }
};

// xs: size() doubles (LDS or global memory) for the multiplied vector (not
// kDirect); vw: 7 stride() doubles for the vectors (NPT 0 only)
template <class Plan, class T>
__device__ __forceinline__ void bottom_krylov(Plan& pl, const T* b_in, T* x_out, const BottomArgs& a,
                                              double* xs, double* vw, BottomRed& red) {
    constexpr int NPT = Plan::NPT;
    const int tid = threadIdx.x, nt = blockDim.x;
    const long n = pl.stride();
    const int cnt = NPT ? NPT : pl.count();  // this thread's unknowns
    int phase = 0;
    OwnVec<NPT> B, R, P, V, W, Y, S;  // rhs, residual, direction, products, solution, |diag|^-1/2
    B.at(vw, tid, nt);
    R.at(vw + n, tid, nt);
    P.at(vw + 2 * n, tid, nt);
    V.at(vw + 3 * n, tid, nt);
    W.at(vw + 4 * n, tid, nt);
    Y.at(vw + 5 * n, tid, nt);
    S.at(vw + 6 * n, tid, nt);
    // dst = A src; src through xs.  The next write of xs comes after a
    // reduction or barrier that every read precedes.
    auto product = [&](OwnVec<NPT>& src, OwnVec<NPT>& dst) {
        const double* x = xs;
        if constexpr (Plan::kDirect) x = src.p - tid;
        else pl.each([&](int q, int id) { xs[id] = Plan::kScaled ? src[q] : S[q] * src[q]; });
        __syncthreads();
        pl.apply(x, [&](int q, double v) { dst[q] = Plan::kScaled ? v : S[q] * v; });
    };
    // 1: the residual of an unknown exceeds stop.  Tested on the
    // scaled one, |S r| > stop S, which needs no division (0 > 0 fails where S is 0)
    double stop = 0.0;
    auto over = [&](int q) { return nabs(R[q]) > stop * S[q] ? 1.0 : 0.0; };

    pl.setup([&](int q, double dg) {
        S[q] = dg > 0.0 ? 1.0 / sqrt(dg) : 0.0;
        B[q] = 0.0;
    });
    if constexpr (Plan::kScaled) {
        const double* x = xs;
        if constexpr (Plan::kDirect) x = S.p - tid;
        else pl.each([&](int q, int id) { xs[id] = S[q]; });
        __syncthreads();
        pl.scale(x);
    }
    double st0[2] = {0.0, 0.0};
    pl.each([&](int q, int id) {
        if (S[q] > 0.0) {
            B[q] = (double)b_in[id];
            st0[0] += B[q];
            st0[1] += 1.0;
        }
    });
    block_reduce<2, 0>(st0, red, phase);
    const double nfree = st0[1];
    const double bmean = (a.singular && nfree > 0.0) ? st0[0] / nfree : 0.0;
    double rn0[1] = {0.0};
#pragma unroll
    for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
        Y[q] = 0.0;
        if (S[q] > 0.0) {
            const double bv = B[q] - bmean;
            rn0[0] = fmax(rn0[0], nabs(bv));
            B[q] = -bv * S[q];
        }
    }
    block_reduce<1, 1>(rn0, red, phase);
    const double rnorm0 = rn0[0];
    stop = a.rtol * rnorm0;

    auto passes = [&]() {
        double u[1] = {0.0};
#pragma unroll
        for (int q = 0; q < (NPT ? NPT : cnt); ++q) u[0] = fmax(u[0], over(q));
        block_reduce<1, 1>(u, red, phase);
        return u[0] == 0.0;
    };
    // 0: converged, 1: broke down, 2: iteration limit; both from zero
    auto bicgstab = [&](int& iters) -> int {
        double g[1] = {0.0};
#pragma unroll
        for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
            R[q] = B[q];
            Y[q] = P[q] = V[q] = 0.0;
            g[0] += B[q] * B[q];
        }
        block_reduce<1, 0>(g, red, phase);
        double rho = g[0], rho_old = 1.0, alpha = 1.0, omega = 1.0;
        for (int it = 1; it <= a.maxiter; ++it) {
            // the residual that the previous iteration left is tested with the next
            // product; when rho underflows to 0 first, here
            if (rho == 0.0) return it > 1 && passes() ? 0 : 1;
            const double beta = it == 1 ? 0.0 : (rho / rho_old) * (alpha / omega);
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) P[q] = R[q] + beta * (P[q] - omega * V[q]);
            product(P, V);
            // (and the test of the residual the previous iteration left)
            double u[2] = {0.0, 0.0};
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                u[0] += B[q] * V[q];
                u[1] = fmax(u[1], over(q));
            }
            block_reduce<2, 2>(u, red, phase);
            if (it > 1 && u[1] == 0.0) return 0;
            iters = it;
            if (u[0] == 0.0) return 1;
            alpha = rho / u[0];
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                Y[q] += alpha * P[q];
                R[q] -= alpha * V[q];
            }
            product(R, W);
            double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                w[0] += W[q] * W[q];
                w[1] += W[q] * R[q];
                w[2] += B[q] * R[q];
                w[3] += B[q] * W[q];
                w[4] = fmax(w[4], over(q));
            }
            block_reduce<5, 16>(w, red, phase);
            if (w[4] == 0.0) return 0;
            if (w[0] == 0.0) return 1;
            omega = w[1] / w[0];
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                Y[q] += omega * R[q];
                R[q] -= omega * W[q];
            }
            if (omega == 0.0) return 1;
            rho_old = rho;
            rho = w[2] - omega * w[3];
        }
        return passes() ? 0 : 2;
    };
    auto cg = [&](int& iters) -> int {
#pragma unroll
        for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
            R[q] = B[q];
            Y[q] = P[q] = V[q] = 0.0;
        }
        double g_old = 1.0, alpha = 1.0;
        for (int it = 1;; ++it) {
            product(R, W);
            double u[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                u[0] += R[q] * R[q];
                u[1] += R[q] * W[q];
                u[2] = fmax(u[2], over(q));
            }
            block_reduce<3, 4>(u, red, phase);
            if (u[0] == 0.0 || (it > 1 && u[2] == 0.0)) return 0;
            if (it > a.maxiter) return 2;
            iters = it;
            const double beta = it == 1 ? 0.0 : u[0] / g_old;
            const double den = it == 1 ? u[1] : u[1] - beta * u[0] / alpha;
            if (den == 0.0) return 1;
            alpha = u[0] / den;
            g_old = u[0];
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
                P[q] = R[q] + beta * P[q];
                V[q] = W[q] + beta * V[q];
                Y[q] += alpha * P[q];
                R[q] -= alpha * V[q];
            }
        }
    };
    int it = 0;
    if (rnorm0 > 0.0) {
        int st = 2, smooths = 0;
        if (a.kind == MGX_BOTTOM_SMOOTHER) {
            smooths = kBottomSmooths;
        } else {
            const bool cg_first = a.kind == MGX_BOTTOM_CG || a.kind == MGX_BOTTOM_CGBICG;
            const bool both = a.kind == MGX_BOTTOM_BICGCG || a.kind == MGX_BOTTOM_CGBICG;
            for (int turn = 0; turn < (both ? 2 : 1) && st != 0; ++turn) {
                int k = 0;
                st = (cg_first == (turn == 0)) ? cg(k) : bicgstab(k);
                it += k;
            }
            if (st != 0) smooths = kBottomSmooths;
        }
        if (st == 1)
#pragma unroll
            for (int q = 0; q < (NPT ? NPT : cnt); ++q) Y[q] = 0.0;
        for (int sw = 0; sw < smooths; ++sw)
            for (int color = 0; color < (Plan::kRedBlack ? 2 : 1); ++color) {
                __syncthreads();
                product(Y, W);
                if constexpr (Plan::kDirect) __syncthreads();  // every read of Y before its update
                pl.each([&](int q, int id) {
                    if constexpr (Plan::kRedBlack) {
                        int i, j, k;
                        pl.point(id, i, j, k);
                        if (((i + j + k) & 1) == color) Y[q] += B[q] - W[q];
                    } else {
                        Y[q] += a.omega * (B[q] - W[q]);
                    }
                });
            }
        if (a.kind == MGX_BOTTOM_SMOOTHER) it = smooths;
    }
    double xsum[1] = {0.0};
#pragma unroll
    for (int q = 0; q < (NPT ? NPT : cnt); ++q) {
        Y[q] *= S[q];
        xsum[0] += Y[q];
    }
    __syncthreads();
    block_reduce<1, 0>(xsum, red, phase);
    const double xmean = (a.singular && nfree > 0.0) ? xsum[0] / nfree : 0.0;
    pl.each([&](int q, int id) { x_out[id] = S[q] > 0.0 ? (T)(Y[q] - xmean) : (T)0; });
    if (tid == 0 && a.iters_acc) atomicAdd(a.iters_acc, it);
}

// XLDS: the multiplied vector fits the workgroup's LDS
template <class Rows, class T, int NPT, bool CREG, int NT, bool XLDS>
static __global__ void __launch_bounds__(NT) bottom_kernel(Rows op, const T* b_in, T* x_out,
                                                           BottomArgs a) {
    extern __shared__ __align__(16) double bottom_xs[];
    __shared__ BottomRed red;
    RowPlan<Rows, NPT, CREG, !XLDS> plan(op, a.work);
    bottom_krylov(plan, b_in, x_out, a, bottom_xs, a.work + (long)Rows::NS * plan.size(), red);
}

// nodal levels of more than 512 nodes: 512 threads, columns along `axis`
template <class TS, class T, int NPT>
static __global__ void __launch_bounds__(512) bottom_cols_kernel(NodalRows<TS> op, int axis, const T* b_in,
                                                                 T* x_out, BottomArgs a) {
    extern __shared__ __align__(16) double bottom_xs[];
    __shared__ BottomRed red;
    ColPlan<TS, NPT> plan(op, axis, reinterpret_cast<TS*>(bottom_xs + op.g.nn[0] * op.g.nn[1] * op.g.nn[2]));
    bottom_krylov(plan, b_in, x_out, a, bottom_xs, nullptr, red);
}

// nodal levels that those do not hold; XLDS: the multiplied vector fits LDS
// (compile-time, for LDS instructions instead of generic ones: 20% of the time)
template <class TS, class T, bool XLDS>
static __global__ void __launch_bounds__(1024) bottom_wide_kernel(NodalRows<TS> op, int axis, int len,
                                                                  const T* b_in, T* x_out, BottomArgs a) {
    extern __shared__ __align__(16) double bottom_xs[];
    __shared__ BottomRed red;
    WidePlan<TS> plan(op, axis, len);
    double* xs = bottom_xs;
    if constexpr (!XLDS) xs = a.work + 7 * plan.stride();
    bottom_krylov(plan, b_in, x_out, a, xs, a.work, red);
}

constexpr size_t kBottomLds = 150 * 1024;

// The variant of a level and what it needs, by the number of unknowns and from
// what a CU's register file holds (512 threads get 256 VGPRs each, 1024 threads
// 128): vectors 14 VGPRs, 27-point rows 54 and 7-point rows 14 VGPRs per unknown.
// Rows read from global memory took the 1280-node nodal solve 740 us, columns
// 150; with spilled rows 8 nodes per column thread took 1900 us at 2275 nodes,
// without 527.
struct BottomPlan {
    enum Kind { REG1, REG2, REG4, COLS4, COLS8, WIDE, ROWS2, ROWS4, ROWS } kind;
    long n = 0;
    int axis = 2, len = 0;   // COLS and WIDE
    unsigned threads = 1024;
    size_t lds = 0;          // bytes; 0 for WIDE and ROWS: the multiplied vector in global memory
    size_t work = 0;         // doubles of BottomArgs::work
};

template <class Rows>
inline BottomPlan bottom_plan(const Rows& op) {
    const auto up64 = [](long v) { return (unsigned)((v + 63) / 64 * 64); };
    const long d[3] = {op.dim(0), op.dim(1), op.dim(2)}, n = d[0] * d[1] * d[2];
    BottomPlan p;
    p.n = n;
    p.lds = (size_t)n * sizeof(double);
    const auto pick = [&](BottomPlan::Kind kind, int per, size_t work) {
        p.kind = kind;
        if (per) p.threads = up64((n + per - 1) / per);
        p.work = work;
        return p;
    };
    if (n <= 512) return pick(BottomPlan::REG1, 1, 0);
    if constexpr (Rows::kNodal) {
        // columns of 4 or 8 nodes in registers, when 512 threads hold the level
        // along some axis (the first that does)
        const size_t lds = p.lds + (size_t)op.g.sg[0] * op.g.sg[1] * op.g.sg[2] * sizeof(*op.sig);
        for (int npt : {4, 8})
            for (int axis = 2; axis >= 0 && lds <= kBottomLds; --axis) {
                const long threads = n / d[axis] * ((d[axis] + npt - 1) / npt);
                if (threads > 512) continue;
                p.axis = axis;
                p.lds = lds;
                p.threads = up64(threads);
                return pick(npt == 4 ? BottomPlan::COLS4 : BottomPlan::COLS8, 0, 0);
            }
        // (13 x 26 x 10 nodes, 20 BiCGStab iterations: 1.41 ms, segments 1.54)
        if (n <= 4096) return pick(BottomPlan::ROWS4, 4, (size_t)Rows::NS * n);
        // segments of columns along y or z (x: the threads of a wave would not read
        // neighbouring nodes, up to 2.6 times slower) for 1024 threads: fewest
        // planes in all, twice, and on the busiest thread, with two more planes
        // per segment than nodes.  20 BiCGStab iterations, whole columns / halves
        // / thirds: 46^3 nodes 42.9 / 39.3 / 40.2 ms, 26^3 5.03 / 5.06 / 5.15,
        // 32 x 10 x 102 along z 15.6 / 11.8 / 11.6 (rows in global memory took
        // twice that on the levels beyond LDS: 46^3 93.6, 32 x 10 x 102 31.6)
        double best = 0.0;
        for (int axis = 2; axis >= 1; --axis)
            for (long k = 1; k <= 16 && k <= d[axis]; ++k) {
                const long len = (d[axis] + k - 1) / k, items = n / d[axis] * ((d[axis] + len - 1) / len);
                const long rounds = (items + 1023) / 1024;
                const double cost = (2.0 * items / 1024.0 + rounds) * (len + 2);
                if (best > 0.0 && cost >= best) continue;
                best = cost;
                p.axis = axis;
                p.len = (int)len;
                p.work = (size_t)rounds * len * 1024 * 7;
            }
        if (p.lds > kBottomLds) p.lds = 0;
        return pick(BottomPlan::WIDE, 0, p.work + (p.lds ? 0 : n));
    } else {
        const bool cell = Rows::NS == 7;
        if (n <= 1024) return pick(BottomPlan::REG2, 2, 0);
        if (n <= 2048 && cell) return pick(BottomPlan::REG4, 4, 0);
        if (n <= 2048) return pick(BottomPlan::ROWS2, 2, (size_t)Rows::NS * n);
        if (n <= 4096) return pick(BottomPlan::ROWS4, 4, (size_t)Rows::NS * n);
        if (p.lds > kBottomLds) p.lds = 0;
        return pick(BottomPlan::ROWS, 0, (size_t)(Rows::NS + 7) * n);
    }
}

// large dynamic LDS is announced once, outside any stream capture
template <class Rows, class T>
void bottom_prepare() {
    static const bool once = [] {
        const auto lds = [](const void* f) {
            (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kBottomLds);
        };
        if constexpr (Rows::kNodal) {
            lds((const void*)bottom_cols_kernel<T, T, 4>);
            lds((const void*)bottom_cols_kernel<T, T, 8>);
            lds((const void*)bottom_wide_kernel<T, T, true>);
        } else {
            lds((const void*)bottom_kernel<Rows, T, 0, false, 1024, true>);
        }
        return true;
    }();
    (void)once;
}

template <class Rows, class T>
void bottom_launch(const Rows& op, const T* b_in, T* x_out, const BottomArgs& a, hipStream_t s) {
    const BottomPlan p = bottom_plan(op);
    if (p.kind == BottomPlan::REG1) {
        bottom_kernel<Rows, T, 1, true, 512, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        return;
    }
    if constexpr (Rows::kNodal) {
        if (p.kind == BottomPlan::COLS4)
            bottom_cols_kernel<T, T, 4><<<1, p.threads, p.lds, s>>>(op, p.axis, b_in, x_out, a);
        else if (p.kind == BottomPlan::COLS8)
            bottom_cols_kernel<T, T, 8><<<1, p.threads, p.lds, s>>>(op, p.axis, b_in, x_out, a);
        else if (p.kind == BottomPlan::ROWS4)
            bottom_kernel<Rows, T, 4, false, 1024, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else if (p.lds > 0)
            bottom_wide_kernel<T, T, true><<<1, p.threads, p.lds, s>>>(op, p.axis, p.len, b_in, x_out, a);
        else
            bottom_wide_kernel<T, T, false><<<1, p.threads, 0, s>>>(op, p.axis, p.len, b_in, x_out, a);
    } else {
        if (p.kind == BottomPlan::REG2)
            bottom_kernel<Rows, T, 2, true, 512, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else if (p.kind == BottomPlan::REG4)
            bottom_kernel<Rows, T, Rows::NS == 7 ? 4 : 1, true, 512, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else if (p.kind == BottomPlan::ROWS2)
            bottom_kernel<Rows, T, 2, false, 1024, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else if (p.kind == BottomPlan::ROWS4)
            bottom_kernel<Rows, T, 4, false, 1024, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else if (p.lds > 0)
            bottom_kernel<Rows, T, 0, false, 1024, true><<<1, p.threads, p.lds, s>>>(op, b_in, x_out, a);
        else
            bottom_kernel<Rows, T, 0, false, 1024, false><<<1, p.threads, 0, s>>>(op, b_in, x_out, a);
    }
}

// instantiated in bottom_nodal.hip and bottom_cell.hip
#define MGX_BOTTOM_INSTANCE(EXT, ROWS, T)                                                            \
    EXT template void bottom_prepare<ROWS, T>();                                                     \
    EXT template void bottom_launch<ROWS, T>(const ROWS&, const T*, T*, const BottomArgs&, hipStream_t)
MGX_BOTTOM_INSTANCE(extern, NodalRows<float>, float);
MGX_BOTTOM_INSTANCE(extern, NodalRows<double>, double);

}  // namespace mgx
