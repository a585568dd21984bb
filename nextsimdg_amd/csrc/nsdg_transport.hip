// DG upwind transport on gfx950.
//
// One thread per element gathers everything that changes its coefficients:
// its cell term, the upwind fluxes of its four edges (each interior edge flux is
// evaluated by both neighbours from identical operands, so the pair stays exactly
// conservative without atomics), its Dirichlet outflow terms, the inverse mass
// matrix and the Runge-Kutta stage combination (after the last stage of a step the
// limiters too), in one pass over HBM. Periodic
// segments, when present, are applied by a per-entry kernel between the flux pass
// and a finishing pass. Fields are SoA (component-major) on the device.
// Reference: dynamics/src/DGTransport.cpp:158-566, ParametricMap.cpp:13-87,
// dgLimit.hpp:16-84, Interpolations.cpp:74-122.
#include "nsdg_device.hpp"
#include "nsdg_transport.hpp"

#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>

namespace nsdg {

enum StageMode { ST_PLUS = 1, ST_RK2B = 3, ST_RK3B = 4, ST_RK3C = 5 };

struct TrArgs {
    MeshView m;
    int ne, nXe, nYe;
    const double* x;    // operator input (neighbours read it)
    const double* velx;
    const double* vely;
    const double* nvX;
    const double* nvY;
    const double* ops;
    double dt;
    int mode;
    const double* base; // the field the step starts from (RK2 and RK3 stages)
    double* out;
    double* raw;        // un-finished increment (periodic path)
    double* tally;      // per-element Dirichlet outflow accumulator (mass budget), or null
    double tallyW;      // weight of this stage's outflow in the step (1/R folded in on the sphere)
    Limits lim;         // limiters applied to the stage's result
};

// ---------------------------------------------------------------- operator set-up
// Transport operators from the mesh geometry, SoA [k][ne] (one element on a uniform mesh):
// the bilinear map x(xi, eta) = x0 + X1 xi + X2 eta + X3 xi eta (and y), and the upper
// triangle of the inverse (metric) DG mass matrix (/ R on the sphere; AdvectionCellTermX/Y
// and the inverse mass, ParametricMap.cpp:13-87: on the sphere the cell terms stay the
// Cartesian ones in (longitude, latitude)). The cell terms factor through the map:
//   sum_q (cellX_i vx + cellY_i vy) phi = sum_q psi_xi,i (y_eta vx - x_eta vy) w phi
//                                            + psi_eta,i (x_xi vy - y_xi vx) w phi,
// so 6 + D (D + 1) / 2 values (27 for D = 6, 42 for D = 8) replace 2 D Q + D^2 (144, 208).
template <int DG> struct TrGeo {
    static constexpr int X1 = 0, X2 = 1, X3 = 2, Y1 = 3, Y2 = 4, Y3 = 5, MI = 6, K = 6 + DG * (DG + 1) / 2;
    __host__ __device__ static constexpr int mi(int i, int j)
    {
        return i <= j ? MI + i * DG - i * (i - 1) / 2 + (j - i) : mi(j, i);
    }
};
template <int DG> __global__ void k_transport_geom(MeshView m, int ne, double* ops)
{
    using L = TrGeo<DG>;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne)
        return;
    auto put = [&](int k, double v) { ops[static_cast<size_t>(k) * ne + e] = v; };
    double c[4][2]; // LL, LR, UL, UR
    elementCoords(m, e, c);
    put(L::X1, c[1][0] - c[0][0]);
    put(L::X2, c[2][0] - c[0][0]);
    put(L::X3, (c[0][0] - c[1][0]) - (c[2][0] - c[3][0]));
    put(L::Y1, c[1][1] - c[0][1]);
    put(L::Y2, c[2][1] - c[0][1]);
    put(L::Y3, (c[0][1] - c[1][1]) - (c[2][1] - c[3][1]));
    double M[DG][DG], Mi[DG][DG];
    metricMassMatrix<DG>(m, c, M);
    invert<DG>(M, Mi);
    for (int i = 0; i < DG; ++i)
        for (int j = i; j < DG; ++j)
            put(L::mi(i, j), m.spherical ? Mi[i][j] / kEarthRadius : Mi[i][j]);
}

// ---------------------------------------------------------------- normal velocities
// reinitnormalvelocity (DGTransport.cpp:158-252), one thread per edge: the average of
// the two adjacent ocean cells' traces along the scaled normal, times 2^k where k
// counts the Dirichlet lists naming the edge.
template <int DG> __global__ void k_normal_velocity(MeshView m, const double* vx, const double* vy, int ne,
    double* nvX, double* nvY, int nXe, int nYe)
{
    constexpr int E = edgedofs(DG);
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int nx = m.nx, ny = m.ny;
    if (t >= nXe + nYe)
        return;
    double acc[E];
#pragma unroll
    for (int k = 0; k < E; ++k)
        acc[k] = 0.0;
    double cx[DG], cy[DG], tx[E], ty[E];
    if (t < nXe) { // X-edge ie = ix + nx*iy (bottom edge of row iy)
        const int ix = t % nx, iy = t / nx;
        const int n0 = iy * (nx + 1) + ix;
        const double t0 = edgeDx(m, m.vxy[2 * (n0 + 1)] - m.vxy[2 * n0]);
        const double t1 = m.vxy[2 * (n0 + 1) + 1] - m.vxy[2 * n0 + 1];
        // both cells' coefficients are loaded before their ocean flags are tested
        double dx[DG], dy[DG];
        const bool hb = iy > 0, ht = iy < ny;
        if (hb)
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                cx[i] = vx[static_cast<size_t>(i) * ne + (t - nx)];
                cy[i] = vy[static_cast<size_t>(i) * ne + (t - nx)];
            }
        if (ht)
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                dx[i] = vx[static_cast<size_t>(i) * ne + t];
                dy[i] = vy[static_cast<size_t>(i) * ne + t];
            }
        if (hb && m.ocean[t - nx]) {
            trace<DG, 2>(cx, tx);
            trace<DG, 2>(cy, ty);
#pragma unroll
            for (int k = 0; k < E; ++k)
                acc[k] += 0.5 * (-t1 * tx[k] + t0 * ty[k]);
        }
        if (ht && m.ocean[t]) {
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                cx[i] = dx[i];
                cy[i] = dy[i];
            }
            trace<DG, 0>(cx, tx);
            trace<DG, 0>(cy, ty);
#pragma unroll
            for (int k = 0; k < E; ++k)
                acc[k] += 0.5 * (-t1 * tx[k] + t0 * ty[k]);
        }
        const double f = m.factX[t];
#pragma unroll
        for (int k = 0; k < E; ++k)
            nvX[static_cast<size_t>(k) * nXe + t] = acc[k] * f;
    } else { // Y-edge ie = ix + (nx+1)*iy (left edge of column ix)
        const int ie = t - nXe;
        const int ix = ie % (nx + 1), iy = ie / (nx + 1);
        const int n0 = iy * (nx + 1) + ix;
        const double t0 = edgeDx(m, m.vxy[2 * (n0 + nx + 1)] - m.vxy[2 * n0]);
        const double t1 = m.vxy[2 * (n0 + nx + 1) + 1] - m.vxy[2 * n0 + 1];
        const int cl = ix - 1 + nx * iy, cr = ix + nx * iy;
        double dx[DG], dy[DG];
        const bool hl = ix > 0, hr = ix < nx;
        if (hl)
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                cx[i] = vx[static_cast<size_t>(i) * ne + cl];
                cy[i] = vy[static_cast<size_t>(i) * ne + cl];
            }
        if (hr)
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                dx[i] = vx[static_cast<size_t>(i) * ne + cr];
                dy[i] = vy[static_cast<size_t>(i) * ne + cr];
            }
        if (hl && m.ocean[cl]) {
            trace<DG, 1>(cx, tx);
            trace<DG, 1>(cy, ty);
#pragma unroll
            for (int k = 0; k < E; ++k)
                acc[k] += 0.5 * (t1 * tx[k] - t0 * ty[k]);
        }
        if (hr && m.ocean[cr]) {
#pragma unroll
            for (int i = 0; i < DG; ++i) {
                cx[i] = dx[i];
                cy[i] = dy[i];
            }
            trace<DG, 3>(cx, tx);
            trace<DG, 3>(cy, ty);
#pragma unroll
            for (int k = 0; k < E; ++k)
                acc[k] += 0.5 * (t1 * tx[k] - t0 * ty[k]);
        }
        const double f = m.factY[ie];
#pragma unroll
        for (int k = 0; k < E; ++k)
            nvY[static_cast<size_t>(k) * nYe + ie] = acc[k] * f;
    }
}

// ---------------------------------------------------------------- flux helpers
template <int DG> __device__ __forceinline__ void loadCell(const double* f, int ne, int e, double* c)
{
#pragma unroll
    for (int i = 0; i < DG; ++i)
        c[i] = f[static_cast<size_t>(i) * ne + e];
}
// Edge coefficients (1, T, T^2 - 1/12) evaluated at the edge's Gauss points.
template <int E, int G> __device__ __forceinline__ void edgeEval(const double* ev, double* out)
{
    legendreValues<G>(ev[0], E > 1 ? ev[E > 1 ? 1 : 0] : 0.0, E > 2 ? ev[E > 2 ? 2 : 0] : 0.0, out);
}
template <int E> __device__ __forceinline__ void loadEdge(const double* nv, int n, int ie, double* v)
{
#pragma unroll
    for (int k = 0; k < E; ++k)
        v[k] = nv[static_cast<size_t>(k) * n + ie];
}
// Moments of edge values against (1, T, T^2 - 1/12) under the Gauss rule.
template <int E, int G> __device__ __forceinline__ void edgeMoments(const double* f, double* m)
{
    const double g = gauss_point(G, G - 1) - 0.5;
    if constexpr (G == 1) {
        m[0] = f[0];
    } else if constexpr (G == 2) {
        m[0] = 0.5 * (f[0] + f[1]);
        m[1] = (0.5 * g) * (f[1] - f[0]);
    } else {
        const double a = f[0] + f[2];
        m[0] = (5.0 / 18.0) * a + (8.0 / 18.0) * f[1];
        m[1] = (5.0 / 18.0 * g) * (f[2] - f[0]);
        m[2] = (1.0 / 54.0) * a - (1.0 / 27.0) * f[1];
    }
}
// up += sgn * dt * sum_q tmp[q] w_q PSI(side, q): the transpose of the trace, from the edge
// moments.
template <int DG, int SIDE>
__device__ __forceinline__ void edgeAccumulate(double* up, double sgn, double dt, const double* tmp)
{
    constexpr int E = edgedofs(DG), G = gp1d(DG);
    constexpr double s = (SIDE == 0 || SIDE == 3) ? -0.5 : 0.5;
    constexpr bool X = SIDE == 1 || SIDE == 3; // x~ = s along the edge, else y~ = s
    double m[E];
    edgeMoments<E, G>(tmp, m);
    const double f = sgn * dt;
#pragma unroll
    for (int k = 0; k < E; ++k)
        m[k] *= f;
    up[0] += m[0];
    if constexpr (DG > 1) {
        up[X ? 1 : 2] += s * m[0];
        up[X ? 2 : 1] += m[1];
    }
    if constexpr (DG > 3) {
        up[X ? 3 : 4] += (1.0 / 6.0) * m[0];
        up[X ? 4 : 3] += m[2];
        up[5] += s * m[1];
    }
    if constexpr (DG > 6) {
        up[X ? 6 : 7] += (1.0 / 6.0) * m[1];
        up[X ? 7 : 6] += s * m[2];
    }
}
// Upwind flux through an interior edge between c1 (left/bottom, side S1 of c1) and
// c2 (right/top): tmp = max(v,0) phi1 + min(v,0) phi2 (DGTransport.cpp:390-433).
template <int DG, int S1, int S2>
__device__ __forceinline__ void upwind(const double* p1, const double* p2, const double* nv, double* tmp)
{
    constexpr int E = edgedofs(DG), G = gp1d(DG);
    double t1[E], t2[E], g1[G], g2[G], vg[G];
    trace<DG, S1>(p1, t1);
    trace<DG, S2>(p2, t2);
    edgeEval<E, G>(nv, vg);
    edgeEval<E, G>(t1, g1);
    edgeEval<E, G>(t2, g2);
#pragma unroll
    for (int q = 0; q < G; ++q)
        tmp[q] = fmax(vg[q], 0.0) * g1[q] + fmin(vg[q], 0.0) * g2[q];
}
// Dirichlet outflow-only boundary term (DGTransport.cpp:306-351), applied count times.
// Returns the outflow: count times the flux tested with the constant basis function, the
// amount coefficient 0 loses before the inverse mass.
template <int DG, int SIDE>
__device__ __forceinline__ double boundaryTerm(double* up, const double* ph, const double* nv, double dt, int count)
{
    constexpr int E = edgedofs(DG), G = gp1d(DG);
    double tr[E], pg[G], vg[G], tmp[G];
    trace<DG, SIDE>(ph, tr);
    edgeEval<E, G>(tr, pg);
    edgeEval<E, G>(nv, vg);
    constexpr double sgn = (SIDE == 0 || SIDE == 3) ? -1.0 : 1.0;
#pragma unroll
    for (int q = 0; q < G; ++q)
        tmp[q] = pg[q] * fmax(sgn * vg[q], 0.0);
    for (int r = 0; r < count; ++r)
        edgeAccumulate<DG, SIDE>(up, -1.0, dt, tmp);
    double m[E];
    edgeMoments<E, G>(tmp, m);
    return count * (dt * m[0]);
}
// All Dirichlet terms of element e; with a.tally set, the stage-weighted outflow is added
// to the element's budget accumulator (elements without Dirichlet sides add nothing).
template <int DG> __device__ __forceinline__ void dirichletTerms(const TrArgs& a, int e, const double* ph, double* up)
{
    constexpr int E = edgedofs(DG);
    const uint32_t fl = a.m.eflags[e];
    if (!fl)
        return;
    const int nx = a.m.nx, ix = e % nx, iy = e / nx;
    double nv[E], out = 0;
    if (fl & 0xffu) {
        loadEdge<E>(a.nvX, a.nXe, nx * iy + ix, nv);
        out += boundaryTerm<DG, 0>(up, ph, nv, a.dt, fl & 0xffu);
    }
    if (fl & 0xff00u) {
        loadEdge<E>(a.nvY, a.nYe, (nx + 1) * iy + ix + 1, nv);
        out += boundaryTerm<DG, 1>(up, ph, nv, a.dt, (fl >> 8) & 0xffu);
    }
    if (fl & 0xff0000u) {
        loadEdge<E>(a.nvX, a.nXe, nx * (iy + 1) + ix, nv);
        out += boundaryTerm<DG, 2>(up, ph, nv, a.dt, (fl >> 16) & 0xffu);
    }
    if (fl & 0xff000000u) {
        loadEdge<E>(a.nvY, a.nYe, (nx + 1) * iy + ix, nv);
        out += boundaryTerm<DG, 3>(up, ph, nv, a.dt, fl >> 24);
    }
    if (a.tally)
        a.tally[e] += a.tallyW * out;
}
// LimitMax then LimitMin (dgLimit.hpp:16-84) of one cell.
template <int DG> __device__ __forceinline__ void limitCell(const Limits& l, double* c)
{
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const bool isMax = pass == 0;
        if (isMax ? !l.doMax : !l.doMin)
            continue;
        const double b = isMax ? l.maxv : l.minv;
        c[0] = isMax ? fmin(b, c[0]) : fmax(b, c[0]);
        if constexpr (DG == 3) {
            const double l0 = 2.0 * fmax(fabs(c[1] + c[2]), fabs(c[1] - c[2]));
            if (l0 != 0.0) {
                const bool ex = isMax ? (c[0] + l0 - b > 0) : (c[0] - l0 - b < 0);
                if (ex) {
                    const double s = isMax ? (b - c[0]) / l0 : (c[0] - b) / l0;
                    c[1] *= s;
                    c[2] *= s;
                }
            }
        } else if constexpr (DG == 6) {
            double ext = isMax ? -INFINITY : INFINITY;
            dgAtGauss<6, 3>(c, [&](int, double v) { ext = isMax ? fmax(ext, v) : fmin(ext, v); });
            const double l0 = ext - c[0];
            if (isMax ? (ext > b) : (ext < b)) {
                const double s = isMax ? (b - c[0]) / l0 : (c[0] - b) / l0;
#pragma unroll
                for (int k = 1; k < 6; ++k)
                    c[k] *= s;
            }
        }
    }
}
// The inverse mass of element e (its upper triangle row by row; an affine element's is
// diagonal).
template <int DG, bool UNI> struct InverseMass {
    static constexpr int K = UNI ? 1 : DG * (DG + 1) / 2;
    double m[K];
    __device__ __forceinline__ void load(const double* ops, size_t ne, int e)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            m[k] = UNI ? ops[TrGeo<DG>::MI] : ops[(TrGeo<DG>::MI + k) * ne + e];
    }
    __device__ __forceinline__ void apply(const double* up, double* k) const
    {
        if constexpr (UNI) {
#pragma unroll
            for (int i = 0; i < DG; ++i)
                k[i] = (m[0] * invMassRef(i)) * up[i];
        } else {
#pragma unroll
            for (int i = 0; i < DG; ++i)
                k[i] = 0.0;
            int n = 0;
#pragma unroll
            for (int i = 0; i < DG; ++i)
#pragma unroll
                for (int j = i; j < DG; ++j, ++n) {
                    k[i] += m[n] * up[j];
                    if (j != i)
                        k[j] += m[n] * up[i];
                }
        }
    }
};
// The Runge-Kutta stage combination (DGTransport.cpp:509-552) from the cell's operator input
// ph, its increment k and the step's base field, then the limiters.
template <int DG> __device__ __forceinline__ void finishCell(const TrArgs& a, int e, const double* ph, const double* k,
    const double* base)
{
    double r[DG];
#pragma unroll
    for (int i = 0; i < DG; ++i) {
        switch (a.mode) {
        case ST_PLUS: r[i] = ph[i] + k[i]; break;
        case ST_RK2B: r[i] = 0.5 * (base[i] + (ph[i] + k[i])); break; // phi + (k1 + k2) / 2, ph = phi + k1
        case ST_RK3B: r[i] = (k[i] + ph[i]) * 0.25 + 0.75 * base[i]; break;
        default: r[i] = base[i] * (1.0 / 3.0) + 2.0 / 3.0 * (k[i] + ph[i]); break;
        }
    }
    limitCell<DG>(a.lim, r);
#pragma unroll
    for (int i = 0; i < DG; ++i)
        a.out[static_cast<size_t>(i) * a.ne + e] = r[i];
}

// ---------------------------------------------------------------- DGTransportOperator
// FINISH: apply Dirichlet, inverse mass and the stage here (no periodic segments);
// otherwise leave the raw increment for the periodic and finishing passes.
// One element per thread; the runs of kBlock elements go to the XCDs in contiguous chunks
// (xcdTile), so the rows above and below a run, which its edge fluxes read, were loaded
// into the same XCD's L2 by the neighbouring runs.
// Bound by the latency of its loads and by its traffic. Every load is issued at the start, in
// the order of its use and whatever the ocean flags say (a clamped neighbour where there is
// none), instead of behind the flag of each neighbour; values and moments at the Gauss
// points go through the factors of the basis; an affine element's inverse mass is diagonal.
// Per stage: 500 x 333 non-affine, D = 6, 24.8 -> 15.8 us with the limiters in the last stage
// (4.8 us as a kernel of their own); 512 x 512 uniform 22.0 -> 15.5 us, D = 8 25.8 -> 18.8;
// 2048 x 2048 336 -> 260 us.
template <int DG, bool UNI, bool FINISH> __global__ __launch_bounds__(kBlock) void k_transport_op(TrArgs a)
{
    constexpr int G = gp1d(DG), Q = G * G, E = edgedofs(DG);
    const int run = xcdTile(blockIdx.x, (a.ne + kBlock - 1) / kBlock);
    if (run < 0)
        return;
    const int e = run * kBlock + threadIdx.x;
    if (e >= a.ne)
        return;
    const int nx = a.m.nx, ny = a.m.ny, ix = e % nx, iy = e / nx;
    const size_t ne = a.ne;
    // left, right, bottom, top: the neighbour and the edge
    const int nbr[4] = { ix > 0 ? e - 1 : e, ix < nx - 1 ? e + 1 : e, iy > 0 ? e - nx : e, iy < ny - 1 ? e + nx : e };
    const int edge[4] = { iy * (nx + 1) + ix, iy * (nx + 1) + ix + 1, ix + nx * iy, ix + nx * (iy + 1) };
    const bool oc = a.m.ocean[e] != 0;
    bool has[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
        has[s] = a.m.ocean[nbr[s]] != 0;
    double ph[DG], up[DG], vx[DG], vy[DG], nb[4][DG], nv[4][E], base[DG], map[6];
    loadCell<DG>(a.x, a.ne, e, ph);
    if constexpr (DG > 1) {
        loadCell<DG>(a.velx, a.ne, e, vx);
        loadCell<DG>(a.vely, a.ne, e, vy);
#pragma unroll
        for (int k = 0; k < 6; ++k)
            map[k] = UNI ? a.ops[k] : a.ops[k * ne + e];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        loadCell<DG>(a.x, a.ne, nbr[s], nb[s]);
        loadEdge<E>(s < 2 ? a.nvY : a.nvX, s < 2 ? a.nYe : a.nXe, edge[s], nv[s]);
    }
    // the 36 values of D = 8 would not fit in registers as early
    constexpr bool kEarly = UNI || DG < 8;
    InverseMass<DG, UNI> im;
    if constexpr (FINISH) {
        if (kEarly)
            im.load(a.ops, ne, e);
        if (a.base)
            loadCell<DG>(a.base, a.ne, e, base);
    }
    has[0] = has[0] && oc && ix > 0;
    has[1] = has[1] && oc && ix < nx - 1;
    has[2] = has[2] && oc && iy > 0;
    has[3] = has[3] && oc && iy < ny - 1;
#pragma unroll
    for (int i = 0; i < DG; ++i)
        up[i] = 0.0;
    if constexpr (DG > 1) {
        if (oc) {
            // cell_term (DGTransport.cpp:278-303): the fluxes phi (y_eta vx - x_eta vy) w and
            // phi (x_xi vy - y_xi vx) w against psi_xi and psi_eta
            double vxg[Q], vyg[Q], F[Q], H[Q];
            dgAtGauss<DG, G>(vx, [&](int q, double v) { vxg[q] = v; });
            dgAtGauss<DG, G>(vy, [&](int q, double v) { vyg[q] = v; });
            dgAtGauss<DG, G>(ph, [&](int q, double v) {
                const double xi = gauss_point(G, q % G), eta = gauss_point(G, q / G);
                const double w = (gauss_weight(G, q % G) * gauss_weight(G, q / G)) * v * a.dt;
                const double xxi = UNI ? map[0] : map[0] + map[2] * eta, xeta = UNI ? map[1] : map[1] + map[2] * xi;
                const double yxi = UNI ? map[3] : map[3] + map[5] * eta, yeta = UNI ? map[4] : map[4] + map[5] * xi;
                F[q] = (yeta * vxg[q] - xeta * vyg[q]) * w;
                H[q] = (xxi * vyg[q] - yxi * vxg[q]) * w;
            });
            if constexpr (G == 3) {
                const double g = gauss_point(3, 2) - 0.5;
                double s[3], d[3], p[3], t[3];
#pragma unroll
                for (int y = 0; y < 3; ++y) {
                    s[y] = F[3 * y] + F[3 * y + 1] + F[3 * y + 2];
                    d[y] = F[3 * y + 2] - F[3 * y];     // X moment / g
                    p[y] = H[y] + H[y + 3] + H[y + 6];  // by column
                    t[y] = H[y + 6] - H[y];             // Y moment / g
                }
                up[1] = s[0] + s[1] + s[2];
                up[2] = p[0] + p[1] + p[2];
                up[3] = (2.0 * g) * (d[0] + d[1] + d[2]);
                up[4] = (2.0 * g) * (t[0] + t[1] + t[2]);
                up[5] = g * ((s[2] - s[0]) + (p[2] - p[0]));
                if constexpr (DG == 8) {
                    up[6] = (2.0 * g * g) * (d[2] - d[0]) + ((1.0 / 15.0) * (p[0] + p[2]) - (1.0 / 12.0) * p[1]);
                    up[7] = (2.0 * g * g) * (t[2] - t[0]) + ((1.0 / 15.0) * (s[0] + s[2]) - (1.0 / 12.0) * s[1]);
                }
            } else {
                up[1] = (F[0] + F[1]) + (F[2] + F[3]);
                up[2] = (H[0] + H[1]) + (H[2] + H[3]);
            }
        }
    }
    // edge fluxes: this cell is c2 of its left and bottom edges, c1 of the others
    double tmp[G];
    const auto masked = [&](bool h) {
#pragma unroll
        for (int q = 0; q < G; ++q)
            tmp[q] = h ? tmp[q] : 0.0;
    };
    upwind<DG, 1, 3>(nb[0], ph, nv[0], tmp);
    masked(has[0]);
    edgeAccumulate<DG, 3>(up, 1.0, a.dt, tmp);
    upwind<DG, 1, 3>(ph, nb[1], nv[1], tmp);
    masked(has[1]);
    edgeAccumulate<DG, 1>(up, -1.0, a.dt, tmp);
    upwind<DG, 2, 0>(nb[2], ph, nv[2], tmp);
    masked(has[2]);
    edgeAccumulate<DG, 0>(up, 1.0, a.dt, tmp);
    upwind<DG, 2, 0>(ph, nb[3], nv[3], tmp);
    masked(has[3]);
    edgeAccumulate<DG, 2>(up, -1.0, a.dt, tmp);
    if constexpr (FINISH) {
        dirichletTerms<DG>(a, e, ph, up);
        double k[DG];
        if (!kEarly)
            im.load(a.ops, ne, e);
        im.apply(up, k);
        finishCell<DG>(a, e, ph, k, base);
    } else {
#pragma unroll
        for (int i = 0; i < DG; ++i)
            a.raw[i * ne + e] = up[i];
    }
}

// Periodic pairs of one segment (DGTransport.cpp:465-481): one thread per entry.
template <int DG> __global__ void k_transport_periodic(TrArgs a, const int32_t* entries, int n)
{
    constexpr int E = edgedofs(DG), G = gp1d(DG);
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n)
        return;
    const int type = entries[4 * k], c1 = entries[4 * k + 1], c2 = entries[4 * k + 2], ie = entries[4 * k + 3];
    if (!a.m.ocean[c1] || !a.m.ocean[c2])
        return;
    double p1[DG], p2[DG], nv[E], tmp[G], u1[DG], u2[DG];
    loadCell<DG>(a.x, a.ne, c1, p1);
    loadCell<DG>(a.x, a.ne, c2, p2);
    loadCell<DG>(a.raw, a.ne, c1, u1);
    loadCell<DG>(a.raw, a.ne, c2, u2);
    if (type == 0) {
        loadEdge<E>(a.nvX, a.nXe, ie, nv);
        upwind<DG, 2, 0>(p1, p2, nv, tmp);
        edgeAccumulate<DG, 2>(u1, -1.0, a.dt, tmp);
        edgeAccumulate<DG, 0>(u2, 1.0, a.dt, tmp);
    } else {
        loadEdge<E>(a.nvY, a.nYe, ie, nv);
        upwind<DG, 1, 3>(p1, p2, nv, tmp);
        edgeAccumulate<DG, 1>(u1, -1.0, a.dt, tmp);
        edgeAccumulate<DG, 3>(u2, 1.0, a.dt, tmp);
    }
#pragma unroll
    for (int i = 0; i < DG; ++i) {
        a.raw[static_cast<size_t>(i) * a.ne + c1] = u1[i];
        a.raw[static_cast<size_t>(i) * a.ne + c2] = u2[i];
    }
}

template <int DG, bool UNI> __global__ __launch_bounds__(kBlock) void k_transport_finish(TrArgs a)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= a.ne)
        return;
    double ph[DG], up[DG], base[DG], k[DG];
    loadCell<DG>(a.x, a.ne, e, ph);
    loadCell<DG>(a.raw, a.ne, e, up);
    if (a.base)
        loadCell<DG>(a.base, a.ne, e, base);
    InverseMass<DG, UNI> im;
    im.load(a.ops, a.ne, e);
    dirichletTerms<DG>(a, e, ph, up);
    im.apply(up, k);
    finishCell<DG>(a, e, ph, k, base);
}

// ---------------------------------------------------------------- limiters
// The limiters on one SoA field by themselves. With tally set, the change
// of the element's Tools::MeanValue contribution is added to tally[e] (mass budget).
template <int DG>
__global__ __launch_bounds__(kBlock) void k_limit(MeshView m, double* f, int ne, Limits lim, double* tally)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne)
        return;
    double c[DG], c0[DG];
    loadCell<DG>(f, ne, e, c);
#pragma unroll
    for (int i = 0; i < DG; ++i)
        c0[i] = c[i];
    limitCell<DG>(lim, c);
    // a cell the limits leave bit for bit as it was is not written back (most cells)
    bool moved = false;
#pragma unroll
    for (int i = 0; i < DG; ++i)
        moved = moved || __double_as_longlong(c[i]) != __double_as_longlong(c0[i]);
    if (!moved)
        return;
#pragma unroll
    for (int i = 0; i < DG; ++i)
        f[static_cast<size_t>(i) * ne + e] = c[i];
    if (tally) {
        bool changed = false;
#pragma unroll
        for (int i = 0; i < DG; ++i)
            changed = changed || c[i] != c0[i];
        if (changed)
            tally[e] += elementMean<DG>(m, e, c) - elementMean<DG>(m, e, c0);
    }
}

// ---------------------------------------------------------------- CG -> DG
// Composite per-element projection op[i*N + j] = (M^-1 PSI diag(J w c) PHI^T)[i][j], c the
// metric weight (cos(latitude) on the sphere, Interpolations.cpp:99-108).
template <int CG, int DG> __global__ void k_cg2dg_ops(MeshView m, int nOps, double* ops)
{
    constexpr int G = gp1d(DG), Q = G * G, N = cgdofs(CG);
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nOps)
        return;
    double c[4][2], J[Q], cl[Q], M[DG][DG], Mi[DG][DG];
    elementCoords(m, e, c);
    jacobian<G>(c, J);
    metricWeight<G>(m, c, cl);
    metricMassMatrix<DG>(m, c, M);
    invert<DG>(M, Mi);
    for (int i = 0; i < DG; ++i)
        for (int j = 0; j < N; ++j) {
            double s = 0;
            for (int t = 0; t < DG; ++t) {
                double r = 0;
                for (int q = 0; q < Q; ++q)
                    r += Psi<DG, G>::v[t][q] * (J[q] * W<G>::v[0][q] * cl[q]) * Phi<CG, G>::v[j][q];
                s += Mi[i][t] * r;
            }
            ops[static_cast<size_t>(i * N + j) * nOps + e] = s;
        }
}
template <int CG, int DG, bool UNI>
__global__ __launch_bounds__(kBlock) void k_cg2dg(int nx, int ne, const double* ops, size_t stride, const double* s1,
    double* d1, const double* s2, double* d2)
{
    constexpr int N = cgdofs(CG);
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne)
        return;
    const Ops<UNI> op { ops, stride };
    const int ix = e % nx, iy = e / nx, row = CG * nx + 1;
    const int cgi = CG * row * iy + CG * ix;
    double l1[N], l2[N];
#pragma unroll
    for (int r = 0; r <= CG; ++r)
#pragma unroll
        for (int cc = 0; cc <= CG; ++cc) {
            l1[cc + (CG + 1) * r] = s1[cgi + cc + r * row];
            if (s2)
                l2[cc + (CG + 1) * r] = s2[cgi + cc + r * row];
        }
#pragma unroll
    for (int i = 0; i < DG; ++i) {
        double a = 0, b = 0;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double w = op(i * N + j, e);
            a += w * l1[j];
            if (s2)
                b += w * l2[j];
        }
        d1[static_cast<size_t>(i) * ne + e] = a;
        if (s2)
            d2[static_cast<size_t>(i) * ne + e] = b;
    }
}

// ---------------------------------------------------------------- layout helpers
__global__ void k_aos_to_soa(const double* in, size_t n, int nc, double* out)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * nc)
        return;
    const size_t e = t / nc, c = t % nc;
    out[c * n + e] = in[t];
}
__global__ void k_soa_to_aos(const double* in, size_t n, int nc, double* out)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * nc)
        return;
    const size_t e = t / nc, c = t % nc;
    out[t] = in[c * n + e];
}
__global__ void k_fill(double* p, size_t n, double v)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n)
        p[t] = v;
}

// The contents of one pinned slot (n values), stored into host memory by the kernel itself;
// 16-byte accesses where the source allows them (a field's components start at any value).
template <class T> __global__ __launch_bounds__(kBlock) void k_to_slot(T* dst, const T* src, size_t n)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (t < n)
        dst[t] = src[t];
}
HostIO::~HostIO() { release(); }
void HostIO::release()
{
    for (auto& e : done) {
        if (e)
            (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (pinned)
        (void)hipHostFree(pinned);
    pinned = nullptr;
    threads = 0;
}
void HostIO::reserve(int n)
{
    if (n <= threads)
        return;
    release();
    NSDG_HIP(hipHostMalloc(reinterpret_cast<void**>(&pinned), 2 * n * kSlot * sizeof(double), hipHostMallocCoherent));
    for (int i = 0; i < 2 * n; ++i)
        NSDG_HIP(hipEventCreateWithFlags(&done[i], hipEventDisableTiming));
    threads = n;
}
// One thread's share of a copy, slot by slot through its two pinned slots.
void HostIO::part(double* host, const double* dev, size_t values, int t, hipStream_t s)
{
    const size_t n = (values + kSlot - 1) / kSlot;
    const auto size = [&](size_t i) { return std::min(kSlot, values - i * kSlot); };
    const auto slot = [&](size_t i) { return pinned + (2 * t + (i & 1)) * kSlot; };
    const auto issue = [&](size_t i) {
        const double* const from = dev + i * kSlot;
        const size_t m = size(i);
        if ((reinterpret_cast<uintptr_t>(from) & 15u) == 0 && m % 2 == 0)
            k_to_slot<<<blocksFor(m / 2), kBlock, 0, s>>>(
                reinterpret_cast<double2*>(slot(i)), reinterpret_cast<const double2*>(from), m / 2);
        else
            k_to_slot<<<blocksFor(m), kBlock, 0, s>>>(slot(i), from, m);
        checkLaunch("to_slot");
        NSDG_HIP(hipEventRecord(done[2 * t + (i & 1)], s));
    };
    for (size_t i = 0; i < std::min<size_t>(2, n); ++i)
        issue(i);
    for (size_t i = 0; i < n; ++i) {
        NSDG_HIP(hipEventSynchronize(done[2 * t + (i & 1)]));
        std::memcpy(host + i * kSlot, slot(i), size(i) * sizeof(double));
        if (i + 2 < n)
            issue(i + 2);
    }
}
void HostIO::toHost(double* host, const double* dev, size_t values, hipStream_t s)
{
    const size_t bytes = values * sizeof(double);
    // page-locked or device memory of the caller's: the copy engine writes it itself
    hipPointerAttribute_t at {};
    const bool known = bytes >= kMinSplit && hipPointerGetAttributes(&at, host) == hipSuccess
        && at.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError(); // asking about ordinary memory is no error
    if (bytes < kMinSplit || known) {
        if (bytes)
            NSDG_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
        NSDG_HIP(hipStreamSynchronize(s));
        return;
    }
    const int n = static_cast<int>(std::clamp<size_t>(bytes / kShare, 2, kThreads));
    reserve(n);
    const size_t share = ((values + n - 1) / n + 511) & ~size_t(511); // whole pages of an aligned field
    int device = 0;
    NSDG_HIP(hipGetDevice(&device));
    std::exception_ptr failed[kThreads];
    const auto run = [&](int t) noexcept {
        try {
            const size_t lo = std::min(values, t * share), hi = std::min(values, lo + share);
            NSDG_HIP(hipSetDevice(device));
            if (hi > lo)
                part(host + lo, dev + lo, hi - lo, t, s);
        } catch (...) {
            failed[t] = std::current_exception();
        }
    };
    std::thread pool[kThreads];
    for (int t = 1; t < n; ++t) {
        try {
            pool[t] = std::thread(run, t);
        } catch (...) { // no more threads to be had: this one takes the share
            run(t);
        }
    }
    run(0);
    for (int t = 1; t < n; ++t)
        if (pool[t].joinable())
            pool[t].join();
    for (int t = 0; t < n; ++t)
        if (failed[t]) {
            (void)hipStreamSynchronize(s); // no copy may still be filling a slot
            std::rethrow_exception(failed[t]);
        }
}
void uploadSoA(HostIO& io, const double* host, size_t n, int nc, double* dst, hipStream_t s)
{
    if (nc == 1) {
        NSDG_HIP(hipMemcpyAsync(dst, host, n * sizeof(double), hipMemcpyHostToDevice, s));
        return;
    }
    if (io.scratch.n < n * nc)
        io.scratch.alloc(n * nc);
    io.scratch.upload(host, n * nc, s);
    k_aos_to_soa<<<blocksFor(n * nc), kBlock, 0, s>>>(io.scratch.p, n, nc, dst);
    checkLaunch("aos_to_soa");
}
void downloadSoA(HostIO& io, const double* src, size_t n, int nc, double* host, hipStream_t s)
{
    if (nc == 1) {
        io.toHost(host, src, n, s);
        return;
    }
    if (io.scratch.n < n * nc)
        io.scratch.alloc(n * nc);
    k_soa_to_aos<<<blocksFor(n * nc), kBlock, 0, s>>>(src, n, nc, io.scratch.p);
    checkLaunch("soa_to_aos");
    io.toHost(host, io.scratch.p, n * nc, s);
}
void deviceFill(double* p, size_t n, double v, hipStream_t s)
{
    if (!n)
        return;
    k_fill<<<blocksFor(n), kBlock, 0, s>>>(p, n, v);
    checkLaunch("fill");
}
// Device-to-device copy as a plain kernel of 16-byte accesses (the runtime's blit kernel
// moves these field-sized copies at about half the rate).
__global__ void k_copy(double* dst, const double* src, size_t n)
{
    const size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (2 * t + 1 < n)
        reinterpret_cast<double2*>(dst)[t] = reinterpret_cast<const double2*>(src)[t];
    else if (2 * t < n)
        dst[2 * t] = src[2 * t];
}
void deviceCopy(double* dst, const double* src, size_t n, hipStream_t s)
{
    if (!n)
        return;
    if (((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15u) != 0) {
        NSDG_HIP(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        return;
    }
    k_copy<<<blocksFor((n + 1) / 2), kBlock, 0, s>>>(dst, src, n);
    checkLaunch("copy");
}

void CG2DGOps::build(int cg_, int dg_, const DeviceMesh& mesh, hipStream_t s)
{
    const int nOps = mesh.uniform ? 1 : static_cast<int>(mesh.ne);
    cg = 0; // until the operators are there
    ops.alloc(static_cast<size_t>(dg_) * cgdofs(cg_) * nOps);
    const MeshView mv = view(mesh);
    auto go = [&](auto kern) {
        kern<<<blocksFor(nOps), kBlock, 0, s>>>(mv, nOps, ops.p);
        checkLaunch("cg2dg_ops");
    };
    if (cg_ == 1 && dg_ == 1) go(k_cg2dg_ops<1, 1>);
    else if (cg_ == 1 && dg_ == 3) go(k_cg2dg_ops<1, 3>);
    else if (cg_ == 1 && dg_ == 6) go(k_cg2dg_ops<1, 6>);
    else if (cg_ == 2 && dg_ == 1) go(k_cg2dg_ops<2, 1>);
    else if (cg_ == 2 && dg_ == 3) go(k_cg2dg_ops<2, 3>);
    else if (cg_ == 2 && dg_ == 6) go(k_cg2dg_ops<2, 6>);
    else if (cg_ == 2 && dg_ == 8) go(k_cg2dg_ops<2, 8>);
    else throw Error(NSDG_ERR_UNSUPPORTED, "unsupported (cg, dg) for CG2DG");
    cg = cg_;
    dg = dg_;
}

void CG2DGOps::apply(const DeviceMesh& mesh, const double* src, double* dst, const double* src2, double* dst2,
    hipStream_t s, Profiler& p) const
{
    Timed t(p, s, "cg2dg");
    const int ne = static_cast<int>(mesh.ne);
    const size_t stride = mesh.uniform ? 1 : mesh.ne;
    auto go = [&](auto kern) {
        kern<<<blocksFor(ne), kBlock, 0, s>>>(mesh.nx, ne, ops.p, stride, src, dst, src2, dst2);
        checkLaunch("cg2dg");
    };
#define NSDG_CG2DG_CASE(C, D)                        \
    if (cg == C && dg == D) {                        \
        if (mesh.uniform)                            \
            go(k_cg2dg<C, D, true>);                 \
        else                                         \
            go(k_cg2dg<C, D, false>);                \
        return;                                      \
    }
    NSDG_CG2DG_CASE(1, 1)
    NSDG_CG2DG_CASE(1, 3)
    NSDG_CG2DG_CASE(1, 6)
    NSDG_CG2DG_CASE(2, 1)
    NSDG_CG2DG_CASE(2, 3)
    NSDG_CG2DG_CASE(2, 6)
    NSDG_CG2DG_CASE(2, 8)
#undef NSDG_CG2DG_CASE
    throw Error(NSDG_ERR_UNSUPPORTED, "unsupported (cg, dg) for CG2DG");
}

// ---------------------------------------------------------------- transport object
template <int DG> struct TransportImpl final : TransportBase {
    static constexpr int G = gp1d(DG), Q = G * G, E = edgedofs(DG);
    DeviceMesh& mesh;
    hipStream_t s;
    Profiler& prof;
    int scheme = 2;
    int nXe, nYe;
    DBuf<double> ops, vx, vy, nvX, nvY, tmpA, tmpB, raw, cgU, cgV;
    HostIO io;
    CG2DGOps cg2dg[3];

    TransportImpl(DeviceMesh& m, hipStream_t st, Profiler& p)
        : mesh(m)
        , s(st)
        , prof(p)
    {
        const size_t ne = mesh.ne;
        nXe = mesh.nx * (mesh.ny + 1);
        nYe = (mesh.nx + 1) * mesh.ny;
        const size_t nOps = mesh.uniform ? 1 : ne;
        ops.alloc(static_cast<size_t>(TrGeo<DG>::K) * nOps);
        k_transport_geom<DG><<<blocksFor(nOps), kBlock, 0, s>>>(view(mesh), static_cast<int>(nOps), ops.p);
        checkLaunch("transport_ops");
        for (auto* b : { &vx, &vy, &tmpA, &tmpB, &raw })
            b->alloc(ne * DG);
        nvX.alloc(static_cast<size_t>(E) * nXe);
        nvY.alloc(static_cast<size_t>(E) * nYe);
        deviceFill(vx.p, ne * DG, 0.0, s);
        deviceFill(vy.p, ne * DG, 0.0, s);
        deviceFill(nvX.p, nvX.n, 0.0, s);
        deviceFill(nvY.p, nvY.n, 0.0, s);
    }
    int dg() const override { return DG; }
    void setScheme(int rk) override
    {
        require(rk >= 1 && rk <= 3, "time stepping scheme must be rk1, rk2 or rk3");
        scheme = rk;
    }
    double* velx() override { return vx.p; }
    double* vely() override { return vy.p; }
    void setVelocityHost(const double* hx, const double* hy) override
    {
        uploadSoA(io, hx, mesh.ne, DG, vx.p, s);
        uploadSoA(io, hy, mesh.ne, DG, vy.p, s);
        NSDG_HIP(hipStreamSynchronize(s));
    }
    void prepareAdvectionHost(int cg, const double* u, const double* v) override
    {
        require(cg == 1 || cg == 2, "cg degree must be 1 or 2");
        if (cg2dg[cg].cg != cg)
            cg2dg[cg].build(cg, DG, mesh, s);
        const size_t ncg = static_cast<size_t>(cg * mesh.nx + 1) * (cg * mesh.ny + 1);
        for (auto* b : { &cgU, &cgV }) // kept for the next velocity
            if (b->n < ncg)
                b->alloc(ncg);
        cgU.upload(u, ncg, s);
        cgV.upload(v, ncg, s);
        cg2dg[cg].apply(mesh, cgU.p, vx.p, cgV.p, vy.p, s, prof);
        reinitNormalVelocity();
        NSDG_HIP(hipStreamSynchronize(s));
    }
    void reinitNormalVelocity() override
    {
        Timed t(prof, s, "normal_velocity");
        k_normal_velocity<DG><<<blocksFor(nXe + nYe), kBlock, 0, s>>>(
            view(mesh), vx.p, vy.p, static_cast<int>(mesh.ne), nvX.p, nvY.p, nXe, nYe);
        checkLaunch("normal_velocity");
    }
    TrArgs args(double dt, const double* x) const
    {
        TrArgs a {};
        a.m = view(mesh);
        a.ne = static_cast<int>(mesh.ne);
        a.nXe = nXe;
        a.nYe = nYe;
        a.x = x;
        a.velx = vx.p;
        a.vely = vy.p;
        a.nvX = nvX.p;
        a.nvY = nvY.p;
        a.ops = ops.p;
        a.dt = dt;
        return a;
    }
    // One DGTransportOperator application fused with its stage combination.
    void stage(TrArgs a)
    {
        const unsigned nb = xcdGrid(static_cast<int>(blocksFor(mesh.ne)));
        if (!mesh.hasPeriodic) {
            Timed t(prof, s, "transport_op");
            if (mesh.uniform)
                k_transport_op<DG, true, true><<<nb, kBlock, 0, s>>>(a);
            else
                k_transport_op<DG, false, true><<<nb, kBlock, 0, s>>>(a);
            checkLaunch("transport_op");
            return;
        }
        a.raw = raw.p;
        {
            Timed t(prof, s, "transport_op");
            if (mesh.uniform)
                k_transport_op<DG, true, false><<<nb, kBlock, 0, s>>>(a);
            else
                k_transport_op<DG, false, false><<<nb, kBlock, 0, s>>>(a);
            checkLaunch("transport_op");
        }
        for (const auto& seg : mesh.segments) {
            k_transport_periodic<DG><<<blocksFor(seg.second), kBlock, 0, s>>>(
                a, mesh.periodic.p + 4 * seg.first, static_cast<int>(seg.second));
            checkLaunch("transport_periodic");
        }
        if (mesh.uniform)
            k_transport_finish<DG, true><<<blocksFor(mesh.ne), kBlock, 0, s>>>(a);
        else
            k_transport_finish<DG, false><<<blocksFor(mesh.ne), kBlock, 0, s>>>(a);
        checkLaunch("transport_finish");
    }
    // step_rk1 / step_rk2 / step_rk3 (DGTransport.cpp:514-552) on a device field. With
    // tally set, each element's Dirichlet outflow over the step (in MeanValue units) is
    // added to tally[e]: the stage outflows weighted as the stages enter the new field. The
    // limiters lim are applied to the new field in its last stage.
    void step(double dt, double* phi, double* tally, const Limits& lim) override
    {
        const size_t n = mesh.ne * DG;
        // on the sphere the inverse mass carries 1/R (ParametricMap.cpp:68-87)
        const double unit = mesh.spherical ? 1.0 / kEarthRadius : 1.0;
        auto withTally = [&](TrArgs a, double w) {
            a.tally = tally;
            a.tallyW = w * unit;
            return a;
        };
        if (scheme == 1) {
            TrArgs a = withTally(args(dt, phi), 1.0);
            a.mode = ST_PLUS;
            a.out = tmpA.p;
            a.lim = lim;
            stage(a);
            deviceCopy(phi, tmpA.p, n, s);
        } else if (scheme == 2) { // phi + (k1 + k2) / 2
            TrArgs a = withTally(args(dt, phi), 0.5);
            a.mode = ST_PLUS;
            a.out = tmpA.p;
            stage(a);
            TrArgs b = withTally(args(dt, tmpA.p), 0.5);
            b.mode = ST_RK2B;
            b.base = phi;
            b.out = phi;
            b.lim = lim;
            stage(b);
        } else { // phi + (k1 + k2) / 6 + 2 k3 / 3
            TrArgs a = withTally(args(dt, phi), 1.0 / 6.0);
            a.mode = ST_PLUS;
            a.out = tmpA.p;
            stage(a);
            TrArgs b = withTally(args(dt, tmpA.p), 1.0 / 6.0);
            b.mode = ST_RK3B;
            b.base = phi;
            b.out = tmpB.p;
            stage(b);
            TrArgs c = withTally(args(dt, tmpB.p), 2.0 / 3.0);
            c.mode = ST_RK3C;
            c.base = phi;
            c.out = phi;
            c.lim = lim;
            stage(c);
        }
    }
    void limit(double* phi, const Limits& lim, double* tally) override
    {
        Timed t(prof, s, "limit");
        k_limit<DG><<<blocksFor(mesh.ne), kBlock, 0, s>>>(view(mesh), phi, static_cast<int>(mesh.ne), lim, tally);
        checkLaunch("limit");
    }
};

std::unique_ptr<TransportBase> makeTransport(int dg, DeviceMesh& mesh, hipStream_t s, Profiler& p)
{
    switch (dg) {
    case 1: return std::make_unique<TransportImpl<1>>(mesh, s, p);
    case 3: return std::make_unique<TransportImpl<3>>(mesh, s, p);
    case 6: return std::make_unique<TransportImpl<6>>(mesh, s, p);
    case 8: return std::make_unique<TransportImpl<8>>(mesh, s, p);
    default: throw Error(NSDG_ERR_UNSUPPORTED, "DG transport degree must be 1, 3, 6 or 8");
    }
}

TransportHandle::~TransportHandle()
{
    t.reset();
    if (stream)
        (void)hipStreamDestroy(stream);
}

} // namespace nsdg
