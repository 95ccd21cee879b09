// stag_kernels.hip -- the staggered compressible scheme (src_compressible_stag) on gfx950.
//
// Momentum and velocity live on faces (cumom[d], vel[d], nodal in d); density, energy and the
// species densities in cells.  One stage of RK3stepStag (timeStepStag.cpp:13-1245) is
//   transport (ref_kernels.hip, stage 0 only) -> k_stag_stress (cells grown by 1: diagonal stresses
//   and cell-centred momentum fluxes; the three edge types: off-diagonal stresses and edge momentum
//   fluxes; one launch) -> k_stag_faces (mass, energy, species and the viscous-work, heat and Dufour
//   components of faceflux; the three directions in one launch) -> k_stag_update (cells and the
//   three face momenta) -> k_stag_c2p -> ghost fill of state, momenta, velocities and prim,
// one thread per cell, edge or face.  The noise of a stage (A + w B of the step's two sets) is
// evaluated in place from a counter-based Philox keyed by the wrapped global index, so duplicate
// periodic faces and edges draw one value (OverrideSync's result) and nothing is stored.  Every
// expression keeps the reference's operation order: the results equal the oracle's
// (oracle/oracle_stag.c) bit for bit.  Scope: 3-D, periodic in every direction; with chemistry
// the update adds the reaction source (timeStepStag.cpp:389-396).
#include "stag.hpp"
#include "stage_bodies.hpp"

namespace fhdx {

constexpr int SB = 256;

// Noise fields (low byte of the counter's third word): face component c of direction d at
// 176 + 16 d + (c - 4), edge types xy, xz, yz at 224 + e, cell fields at 232 + d.
constexpr uint32_t STAG_FACE_FIELD = 176u;
constexpr uint32_t STAG_EDGE_FIELD = 224u;
constexpr uint32_t STAG_CELL_FIELD = 232u;

__device__ inline int wrapn(int i, int n) { return ((i % n) + n) % n; }

__device__ inline uint32_t wrapped_lin(const DevParams& P, int i, int j, int k)
{
    return (uint32_t)(((long)wrapn(k, P.n[2]) * P.n[1] + wrapn(j, P.n[1])) * P.n[0] + wrapn(i, P.n[0]));
}

// The edge flux array of momentum component m transported along t (m != t), in the reference's
// order edgeflux_x[0..1], edgeflux_y[0..1], edgeflux_z[0..1]: x_v, x_w, y_u, y_w, z_u, z_v.
__host__ __device__ constexpr int edge_flux_index(int m, int t)
{
    return m == 0 ? (t == 1 ? 2 : 4) : m == 1 ? (t == 0 ? 0 : 5) : (t == 0 ? 1 : 3);
}
// Edge type of the plane of two distinct axes: xy 0, xz 1, yz 2.
__host__ __device__ constexpr int edge_type(int a, int b)
{
    return (a + b == 1) ? 0 : (a + b == 2) ? 1 : 2;
}

__device__ inline void cell_of(long t, int fx, int fy, int& i, int& j, int& k)
{
    i = (int)(t % fx);
    long r = t / fx;
    j = (int)(r % fy);
    k = (int)(r / fy);
}

// ---- cells grown by 1: fluxStag.cpp:163-206, 872-924, 799-803, 1444-1449, 1838-1856 --------

__device__ __forceinline__ void stag_cell(const DevParams& P, const StagArrays& A, const NoiseKey& K, double w, double dt,
                                          long t)
{
    const int gx = P.n[0] + 2, gy = P.n[1] + 2, gz = P.n[2] + 2;
    if (t >= (long)gx * gy * gz) return;
    int i, j, k;
    cell_of(t, gx, gy, i, j, k);
    i -= 1;
    j -= 1;
    k -= 1;
    const double volinv = 1. / (P.dx[0] * P.dx[1] * P.dx[2]);
    const double dtinv = 1. / dt;
    const bool visc3 = (P.visc_type == 3 || P.visc_type == -3);
    constexpr Rcp three{3., 1. / 3.};
    const Fld prim = fld_of(A.prim, A.prim), etaf = fld_of(A.eta, A.prim), zetaf = fld_of(A.zeta, A.prim);
    const Fld td = fld_of(A.td, A.td);
    const unsigned c0 = off_of(A.prim, i, j, k), o1 = off_of(A.td, i, j, k);
    Fld vel[3], mom[3];
    unsigned fo[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        vel[d] = fld_of(A.vel[d], A.vel[d]);
        mom[d] = fld_of(A.mom[d], A.vel[d]);
        fo[d] = off_of(A.vel[d], i, j, k);
    }
    const double eta = etaf(c0, 0), zeta = zetaf(c0, 0);
    const double T = prim(c0, 4);
    double ts[3] = {0., 0., 0.};
    if (P.stoch_on) {
        const double etaT = eta * T;
        const double zetaT = zeta * T;
        const double fac1 = root(2.0 * P.k_B * etaT * volinv * dtinv);
        double fac2 = (-1.0 / 3.0) * fac1;
        if (visc3) fac2 = root(P.k_B * zetaT * volinv * dtinv / three) - fac1 / three;
        const uint32_t lin = wrapped_lin(P, i, j, k);
        const double sq2 = sqrt(2.0);
        double z[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double a, b;
            noise_ab(K, STAG_CELL_FIELD + (uint32_t)c, lin, a, b);
            z[c] = 1.0 * (sq2 * a) + w * (sq2 * b);
        }
        const double traceZ = z[0] + z[1] + z[2];
#pragma unroll
        for (int c = 0; c < 3; ++c) ts[c] = (fac1 * z[c]) + (fac2 * traceZ);
    }
    const double vl[3] = {vel[0](fo[0], 0), vel[1](fo[1], 0), vel[2](fo[2], 0)};
    const double vh[3] = {vel[0](fo[0], 0, 1, 0, 0), vel[1](fo[1], 0, 0, 1, 0), vel[2](fo[2], 0, 0, 0, 1)};
    const double g[3] = {(vh[0] - vl[0]) / P.h(0), (vh[1] - vl[1]) / P.h(1), (vh[2] - vl[2]) / P.h(2)};
    const double div = g[0] + g[1] + g[2];
    const double p = prim(c0, 5);
    double tau[3], cf[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        tau[c] = visc3 ? 2 * eta * g[c] + (zeta - 2 * eta / three) * div : 2 * eta * g[c] + (0.0 - 2 * eta / three) * div;
        cf[c] = ts[c];
        cf[c] -= tau[c];
        if (P.advection_type >= 0) {
            const double m0 = mom[c](fo[c], 0), m1 = mom[c](fo[c], 0, c == 0, c == 1, c == 2);
            cf[c] += 0.25 * (m0 + m1) * (vl[c] + vh[c]) + p;
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        td(o1, c) = ts[c];
        td(o1, 3 + c) = tau[c];
        fld_of(A.cf[c], A.td)(o1, 0) = cf[c];
    }
}

// ---- edges: fluxStag.cpp:209-295, 927-1022, 784-797, 1429-1441, 1767-1835 ----------------

template <int E>
__device__ __forceinline__ void stag_edge(const DevParams& P, const StagArrays& A, const NoiseKey& K, double w,
                                 double dt, int i, int j, int k)
{
    constexpr int a = (E == 2) ? 1 : 0, b = (E == 0) ? 1 : 2;
    constexpr int ea0 = a == 0, ea1 = a == 1, ea2 = a == 2;
    constexpr int eb0 = b == 0, eb1 = b == 1, eb2 = b == 2;
    const Fld prim = fld_of(A.prim, A.prim), eta = fld_of(A.eta, A.prim);
    const unsigned c0 = off_of(A.prim, i, j, k), oa = off_of(A.vel[a], i, j, k), ob = off_of(A.vel[b], i, j, k);
    // the four cells around the edge
    const double e0 = eta(c0, 0, -ea0 - eb0, -ea1 - eb1, -ea2 - eb2), e1 = eta(c0, 0, -ea0, -ea1, -ea2),
                 e2 = eta(c0, 0, -eb0, -eb1, -eb2), e3 = eta(c0, 0);
    double ts = 0.;
    if (P.stoch_on) {
        const double volinv = 1. / (P.dx[0] * P.dx[1] * P.dx[2]);
        const double dtinv = 1. / dt;
        double s = e0 * prim(c0, 4, -ea0 - eb0, -ea1 - eb1, -ea2 - eb2);
        s = s + e1 * prim(c0, 4, -ea0, -ea1, -ea2);
        s = s + e2 * prim(c0, 4, -eb0, -eb1, -eb2);
        s = s + e3 * prim(c0, 4);
        const double etaT = 0.25 * s;
        const double fac = root(2.0 * P.k_B * etaT * volinv * dtinv);
        double za, zb;
        noise_ab(K, STAG_EDGE_FIELD + (uint32_t)E, wrapped_lin(P, i, j, k), za, zb);
        ts = fac * (1.0 * za + w * zb);
    }
    const Fld va = fld_of(A.vel[a], A.vel[a]), vb = fld_of(A.vel[b], A.vel[b]);
    const double va1 = va(oa, 0), va0 = va(oa, 0, -eb0, -eb1, -eb2);
    const double vb1 = vb(ob, 0), vb0 = vb(ob, 0, -ea0, -ea1, -ea2);
    const double da_b = (va1 - va0) / P.h(b);
    const double db_a = (vb1 - vb0) / P.h(a);
    double es = e0;
    es = es + e1;
    es = es + e2;
    es = es + e3;
    const double eta_interp = 0.25 * es;
    const double tau = eta_interp * (da_b + db_a);
    double fa = ts, fb = ts;  // momentum a along b, momentum b along a
    fa -= tau;
    fb -= tau;
    if (P.advection_type >= 0) {
        const Fld ma = fld_of(A.mom[a], A.vel[a]), mb = fld_of(A.mom[b], A.vel[b]);
        const double adv_a = 0.25 * (ma(oa, 0, -eb0, -eb1, -eb2) + ma(oa, 0)) * (vb0 + vb1);
        const double adv_b = 0.25 * (mb(ob, 0, -ea0, -ea1, -ea2) + mb(ob, 0)) * (va0 + va1);
        fa += adv_a;
        fb += adv_b;
    }
    const Fld to = fld_of(A.to[E], A.to[E]);
    const unsigned eo = off_of(A.to[E], i, j, k);
    to(eo, 0) = ts;
    to(eo, 1) = tau;
    fld_of(A.ef[edge_flux_index(a, b)], A.to[E])(eo, 0) = fa;
    fld_of(A.ef[edge_flux_index(b, a)], A.to[E])(eo, 0) = fb;
}

template <int E>
__device__ __forceinline__ void stag_edge_at(const DevParams& P, const StagArrays& A, const NoiseKey& K, double w,
                                             double dt, long t)
{
    // the edge box: nodal along the type's two axes
    const int ex = P.n[0] + (E != 2), ey = P.n[1] + (E != 1), ez = P.n[2] + (E != 0);
    if (t >= (long)ex * ey * ez) return;
    int i, j, k;
    cell_of(t, ex, ey, i, j, k);
    stag_edge<E>(P, A, K, w, dt, i, j, k);
}

// Cells and edges do not read each other: one launch, blockIdx.y the part.  The parts follow each
// other: taken chunk by chunk in turn (as k_stag_faces takes its directions) they shared cache lines
// but wrote 21 streams at once, 459 us against 383 at argon 160^3 (464 before, in index products).
__global__ void __launch_bounds__(SB) k_stag_stress(DevParams P, StagArrays A, NoiseKey K, double w, double dt)
{
    const long t = (long)blockIdx.x * SB + threadIdx.x;
    switch (blockIdx.y) {
        case 0: stag_cell(P, A, K, w, dt, t); break;
        case 1: stag_edge_at<0>(P, A, K, w, dt, t); break;
        case 2: stag_edge_at<1>(P, A, K, w, dt, t); break;
        default: stag_edge_at<2>(P, A, K, w, dt, t); break;
    }
}

// ---- faces of direction D: fluxStag.cpp:298-780, 1026-1426, 1507-1764 --------------------

template <int NS, int D>
__device__ __forceinline__ void stag_face(const DevParams& P, const StagArrays& A, const NoiseKey& K, double w, double dt,
                                          int keep, long tid)
{
    constexpr int nv = NS + 5;
    constexpr int ed0 = D == 0, ed1 = D == 1, ed2 = D == 2;
    constexpr int t1 = (D == 0) ? 1 : 0, t2 = (D == 2) ? 1 : 2;
    const int fx = P.n[0] + ed0, fy = P.n[1] + ed1, fz = P.n[2] + ed2;
    if (tid >= (long)fx * fy * fz) return;
    int i, j, k;
    cell_of(tid, fx, fy, i, j, k);
    // The weighted noise of the face (heat, then the species) by itself, as in the collocated face_flux:
    // 853 -> 833 us a launch at 160^3 argon, 112 -> 101 at 64^3 with four species.
    double zn[NS + 1];
    if (P.stoch_on) {
        const uint32_t lin = wrapped_lin(P, i, j, k);
#pragma unroll
        for (int l = 0; l < NS + 1; ++l) {
            double za, zb;
            noise_ab(K, STAG_FACE_FIELD + 16u * D + (uint32_t)l, lin, za, zb);
            zn[l] = 1.0 * za + w * zb;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const Fld prim = fld_of(A.prim, A.prim), cu = fld_of(A.cu, A.prim), chi = fld_of(A.chi, A.prim),
              Dm = fld_of(A.D, A.prim), kappa = fld_of(A.kappa, A.prim), td = fld_of(A.td, A.td);
    // this cell and the one below the face; the face in its velocity's layout
    const unsigned c0 = off_of(A.prim, i, j, k), cm = off_of(A.prim, i - ed0, j - ed1, k - ed2);
    const unsigned o1 = off_of(A.td, i, j, k), fo = off_of(A.vel[D], i, j, k);
    const Rcp dxd = P.h(D);
    const double volinv = 1. / (P.dx[0] * P.dx[1] * P.dx[2]);
    const double dtinv = 1. / dt;
    const double Tu = prim(c0, 4), Tl = prim(cm, 4);
    const double kapU = kappa(c0, 0), kapL = kappa(cm, 0);
    const double vel_f = fld_of(A.vel[D], A.vel[D])(fo, 0);
    // the viscous work of the two transverse velocities with the edge stresses: stochastic (comp 0)
    // and deterministic (comp 1)
    double shear[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        constexpr int tt[2] = {t1, t2};
        const int t = tt[q], et0 = t == 0, et1 = t == 1, et2 = t == 2;
        const Fld vt = fld_of(A.vel[t], A.vel[t]);
        const Arr& ea = A.to[edge_type(D, t)];
        const Fld ts = fld_of(ea, ea);
        const unsigned vo = off_of(A.vel[t], i, j, k), eo = off_of(ea, i, j, k);
        const double vp = vt(vo, 0, et0, et1, et2) + vt(vo, 0, et0 - ed0, et1 - ed1, et2 - ed2);
        const double v0 = vt(vo, 0) + vt(vo, 0, -ed0, -ed1, -ed2);
#pragma unroll
        for (int c = 0; c < 2; ++c) shear[c][q] = 0.25 * (vp * ts(eo, c, et0, et1, et2) + v0 * ts(eo, c));
    }
    double f[nv + 4];
#pragma unroll
    for (int c = 0; c < nv + 4; ++c) f[c] = 0.;
    double hk[NS];

    // stochastic part
    if (P.stoch_on) {
        double wn[NS + 1];
        const double kp = kapU * Tu * Tu + kapL * Tl * Tl;
        const double meanT = 0.5 * (Tu + Tl);
        const double fw0 = root(P.k_B * kp * volinv * dtinv);
        wn[0] = fw0 * zn[0];
        f[nv] = wn[0];
        f[nv + 1] = 0.5 * vel_f * (td(o1, D, -ed0, -ed1, -ed2) + td(o1, D));
        double vsh = 0.0;
        vsh += shear[0][0];
        vsh += shear[0][1];
        f[nv + 2] = vsh;
        if (P.algorithm_type == 2) {
            double yy[NS], yyp[NS], DijY[NS * NS], sqD[NS * NS];
#pragma unroll
            for (int n = 1; n < 1 + NS; ++n) wn[n] = 0.;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                yy[s] = clamp01(prim(cm, 6 + s));
                yyp[s] = clamp01(prim(c0, 6 + s));
            }
            double sumy = 0., sumyp = 0.;
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                sumy += yy[n];
                sumyp += yyp[n];
            }
            const Rcp ry = rcp_of(sumy), ryp = rcp_of(sumyp);
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                yy[n] = yy[n] / ry;
                yyp[n] = yyp[n] / ryp;
            }
            double MWmix = 0.;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                MWmix = MWmix + 0.5 * (yy[s] + yyp[s]) / P.M(s);
#pragma unroll
                for (int l = 0; l < NS; ++l)
                    DijY[s * NS + l] = 0.5 * (Dm(cm, l * NS + s) * yy[l] + Dm(c0, l * NS + s) * yyp[l] +
                                              (Dm(cm, s * NS + l) * yy[s] + Dm(c0, s * NS + l) * yyp[s]));
            }
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (fabs(yy[s]) + fabs(yyp[s]) <= 1.e-12)
#pragma unroll
                    for (int n = 0; n < NS; ++n) {
                        DijY[s * NS + n] = 0.;
                        DijY[n * NS + s] = 0.;
                    }
            MWmix = quot(1., MWmix);
            cholesky<NS>(DijY, sqD);
            const double wsp = root(quot(P.k_B * MWmix * volinv, P.Runiv * dt));
#pragma unroll
            for (int s = 0; s < NS; ++s) {
#pragma unroll
                for (int l = 0; l <= s; ++l) {
                    const double fw = wsp * sqD[s * NS + l];
                    wn[1 + s] = wn[1 + s] + fw * zn[1 + l];
                }
                f[5 + s] = wn[1 + s];
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) hk[s] = P.e0[s] + P.hcp[s] * meanT;
            double soret = 0.;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                soret += (hk[s] + P.Runiv * meanT / P.M(s) * 0.5 * (chi(cm, s) + chi(c0, s))) *
                         wn[1 + s];
            f[nv + 3] = soret;
        }
    }

    // diffusive part
    {
        const double kp = 0.5 * (kapL + kapU);
        const double meanT = 0.5 * (Tl + Tu);
        const double pl = prim(cm, 5), pu = prim(c0, 5);
        const double meanP = 0.5 * (pl + pu);
        f[nv + 1] -= 0.5 * vel_f * (td(o1, 3 + D, -ed0, -ed1, -ed2) + td(o1, 3 + D));
        double vsh = 0.0;
        vsh -= shear[1][0];
        vsh -= shear[1][1];
        f[nv] -= kp * (Tu - Tl) / dxd;
        f[nv + 2] += vsh;
        if (P.algorithm_type == 2) {
            const Rcp rT = rcp_of(meanT), rP = rcp_of(meanP);
            double dk[NS], soret[NS], Fk[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const double Xl = prim(cm, 6 + NS + s), Xu = prim(c0, 6 + NS + s);
                const double Yl = prim(cm, 6 + s), Yu = prim(c0, 6 + s);
                const double term1 = (Xu - Xl) / dxd;
                const double meanXk = 0.5 * (Xl + Xu);
                const double meanYk = 0.5 * (Yl + Yu);
                const double term2 = (meanXk - meanYk) * (pu - pl) / dxd / rP;
                dk[s] = term1 + term2;
                const double ChiX = 0.5 * (chi(cm, s) * Xl + chi(c0, s) * Xu);
                soret[s] = ChiX * (Tu - Tl) / dxd / rT;
            }
#pragma unroll
            for (int kk = 0; kk < NS; ++kk) {
                Fk[kk] = 0.;
#pragma unroll
                for (int l = 0; l < NS; ++l) {
                    const double Fks = 0.5 * (Dm(cm, l * NS + kk) + Dm(c0, l * NS + kk)) * (dk[l] + soret[l]);
                    Fk[kk] -= Fks;
                }
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) hk[s] = P.e0[s] + P.hcp[s] * meanT;
            double Q5 = 0.;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                // z faces add chi(i,j,k) twice (fluxStag.cpp:1398)
                const double chil = (D == 2) ? chi(c0, s) : chi(cm, s);
                Q5 += (hk[s] + 0.5 * P.Runiv * meanT * (chil + chi(c0, s)) / P.M(s)) * Fk[s];
            }
            f[nv + 3] += Q5;
#pragma unroll
            for (int s = 0; s < NS; ++s) f[5 + s] += Fk[s];
        }
    }

    // hyperbolic part
    if (P.advection_type >= 0) {
        const double mom = fld_of(A.mom[D], A.vel[D])(fo, 0);
        f[0] += mom;
        const double meanT = 0.5 * (Tl + Tu);
        const double meanRho = 0.5 * (prim(cm, 0) + prim(c0, 0));
        const double meanP = 0.5 * (prim(cm, 5) + prim(c0, 5));
#pragma unroll
        for (int s = 0; s < NS; ++s) hk[s] = P.e0[s] + P.hcp[s] * meanT;
        if (P.advection_type == 1) {
            const Rcp rho = rcp_of(meanRho);
            const double meanE = 0.5 * (cu(cm, 4) + cu(c0, 4)) / rho;
            f[4] += mom * (meanE + (meanP / rho));
        } else if (P.advection_type == 2) {
            f[4] += 0.5 * (cu(cm, 4) + cu(c0, 4)) * vel_f + 0.5 * (prim(cm, 5) + prim(c0, 5)) * vel_f;
        }
        if (P.algorithm_type == 2) {
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                const double Yk = 0.5 * (prim(cm, 6 + n) + prim(c0, 6 + n));
                if (P.advection_type == 0 || P.advection_type == 1)
                    f[5 + n] += Yk * mom;
                else if (P.advection_type == 2)
                    f[5 + n] += 0.5 * (cu(cm, 5 + n) + cu(c0, 5 + n)) * vel_f;
                if (P.advection_type == 0) f[4] += mom * Yk * hk[n];
            }
        }
        if (P.advection_type == 0) {
            const int li = i - ed0, lj = j - ed1, lk = k - ed2;
            const Arr& mx = A.mom[0];
            const Arr& my = A.mom[1];
            const Arr& mz = A.mom[2];
            double keP = 0., keM = 0., s;
            s = mx(i + 1, j, k) + mx(i, j, k);
            keP += s * s;
            s = my(i, j + 1, k) + my(i, j, k);
            keP += s * s;
            s = mz(i, j, k + 1) + mz(i, j, k);
            keP += s * s;
            keP *= (0.125 / cu(c0, 0) / cu(c0, 0));
            s = mx(li + 1, lj, lk) + mx(li, lj, lk);
            keM += s * s;
            s = my(li, lj + 1, lk) + my(li, lj, lk);
            keM += s * s;
            s = mz(li, lj, lk + 1) + mz(li, lj, lk);
            keM += s * s;
            // z faces divide by the density of cell (i, j-1, k) (fluxStag.cpp:1754)
            const double rm = (D == 2) ? cu(c0, 0, 0, -1, 0) : cu(cm, 0);
            keM *= (0.125 / rm / rm);
            f[4] += mom * 0.5 * (keP + keM);
        }
    }
    f[4] += f[nv] + f[nv + 1] + f[nv + 2] + f[nv + 3];
    const Fld ff = fld_of(A.ff[D], A.ff[D]);
    const unsigned ffo = off_of(A.ff[D], i, j, k);
#pragma unroll
    for (int c = 0; c < nv + 4; ++c)
        if (keep || c == 0 || (c >= 4 && c < nv)) ff(ffo, c) = f[c];
}

// The three directions in one launch, as in the collocated k_flux: consecutive work items are the
// directions of one chunk of faces.  keep 0: the components that the stage update does not read (the
// zero momentum ones and the four parts of the energy flux) are not stored; the last stage of a
// step, and calculateFluxStag, store all.  Argon 160^3: 1096 us a stage in three launches with index
// products of each array's strides, 940 us with the directions one after another, 818 us so.
//
// The arguments are one struct, read anew in each direction's branch (see k_flux): 140 to 271 scalar
// registers spilled to vector lanes, 2 to 16 so, and six species fit two waves a SIMD.  A step of 48^3, us:
// seven species 984 and 838 (908 with a launch a direction), eight 1300 and 1083 (1315), two 237 and 222; argon
// 160^3 5477 and 5385.
struct StagFaceKernel {
    DevParams P;
    StagArrays A;
    NoiseKey K;
    double w, dt;
    int keep;
};

__device__ __forceinline__ const StagFaceKernel& stag_face_args()
{
    typedef const StagFaceKernel __attribute__((address_space(4))) * Ptr;
    Ptr p = (Ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm("" : "+s"(p));
    return *(const StagFaceKernel*)p;
}

template <int NS, int D>
__device__ __forceinline__ void stag_face_item(long t)
{
    const StagFaceKernel& F = stag_face_args();
    stag_face<NS, D>(F.P, F.A, F.K, F.w, F.dt, F.keep, t);
}

template <int NS>
__global__ void __launch_bounds__(SB) k_stag_faces(StagFaceKernel F)
{
    const unsigned item = xcd_block(blockIdx.x, gridDim.x), chunk = item / 3, d = item - 3 * chunk;
    const long t = (long)chunk * SB + threadIdx.x;
    if (d == 0) stag_face_item<NS, 0>(t);
    else if (d == 1) stag_face_item<NS, 1>(t);
    else stag_face_item<NS, 2>(t);
}

// ---- stage update: timeStepStag.cpp:470-538, 771-857, 1106-1199 --------------------------

template <int D>
__device__ __forceinline__ void stag_update_face(const DevParams& P, const StagUpdate& U, int st, double dt, long tid)
{
    constexpr int ed0 = D == 0, ed1 = D == 1, ed2 = D == 2;
    const double* grav = P.grav;
    const int fx = P.n[0] + ed0, fy = P.n[1] + ed1, fz = P.n[2] + ed2;
    if (tid >= (long)fx * fy * fz) return;
    int i, j, k;
    cell_of(tid, fx, fy, i, j, k);
    double c[3];  // flux differences along x, y, z
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        if (t == D) {
            const Fld cf = fld_of(U.cf[D], U.cf[D]);
            const unsigned o = off_of(U.cf[D], i, j, k);
            c[t] = cf(o, 0) - cf(o, 0, -ed0, -ed1, -ed2);
        } else {
            const Arr& ea = U.ef[edge_flux_index(D, t)];
            const Fld e = fld_of(ea, ea);
            const unsigned o = off_of(ea, i, j, k);
            c[t] = e(o, 0, t == 0, t == 1, t == 2) - e(o, 0);
        }
    }
    const Fld us = fld_of(U.us, U.us);
    const unsigned c0 = off_of(U.us, i, j, k), mo = off_of(U.m0[D], i, j, k);
    const double rs = us(c0, 0, -ed0, -ed1, -ed2) + us(c0, 0);
    const double m0 = fld_of(U.m0[D], U.m0[D])(mo, 0), ms = fld_of(U.ms[D], U.m0[D])(mo, 0);
    double v;
    if (st == 0)
        v = m0 - dt * c[0] / P.h(0) - dt * c[1] / P.h(1) - dt * c[2] / P.h(2) + 0.5 * dt * grav[D] * rs;
    else if (st == 1)
        v = 0.25 * 3.0 * m0 + 0.25 * ms - 0.25 * dt * c[0] / P.h(0) - 0.25 * dt * c[1] / P.h(1) -
            0.25 * dt * c[2] / P.h(2) + 0.5 * 0.25 * dt * grav[D] * rs;
    else
        v = (2. / 3.) * (0.5 * m0 + ms) - (2. / 3.) * dt * c[0] / P.h(0) - (2. / 3.) * dt * c[1] / P.h(1) -
            (2. / 3.) * dt * c[2] / P.h(2) + 0.5 * (2. / 3.) * dt * grav[D] * rs;
    fld_of(U.outm[D], U.m0[D])(mo, 0) = v;
}

template <int NS, bool CHEM>
__global__ void __launch_bounds__(SB) k_stag_update(DevParams P, StagUpdate U, int st, double dt)
{
    constexpr int nv = NS + 5;
    const int part = blockIdx.y;  // 0 cells, 1..3 faces of direction part-1
    const long tid = (long)blockIdx.x * SB + threadIdx.x;
    const double* grav = P.grav;
    if (part == 0) {
        const int n0 = P.n[0], n1 = P.n[1], n2 = P.n[2];
        if (tid >= (long)n0 * n1 * n2) return;
        int i, j, k;
        cell_of(tid, n0, n1, i, j, k);
        double src[nv];
#pragma unroll
        for (int n = 0; n < nv; ++n) src[n] = 0.0;
        if constexpr (CHEM) {  // compute_compressible_chemistry_source_CLE from the stage's prim
            const double dV = P.dx[0] * P.dx[1] * P.dx[2];
            double X[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) X[s] = U.prim(i, j, k, 6 + NS + s);
            const uint32_t lin = (uint32_t)(((long)k * n1 + j) * n0 + i);
            chem_source_cell<NS>(P, U.prim(i, j, k, 4), U.prim(i, j, k, 5), X,
                                 [&](int m) { return chem_noise(U.K, m, lin, U.w); }, dt, dV, &src[5]);
            if (U.ranchem.p)
                for (int m = 0; m < P.chem.nreaction; ++m) U.ranchem(i, j, k, m) = chem_noise(U.K, m, lin, U.w);
            if (U.source.p)
#pragma unroll
                for (int n = 5; n < nv; ++n) U.source(i, j, k, n) = src[n];
        }
        // Components 1-3 (cell-centred momentum) are skipped: the reference computes them here
        // and conservedToPrimitiveStag overwrites them (and FillBoundary their ghosts) before
        // anything reads them, so the result does not depend on them.
        const Fld us = fld_of(U.us, U.out), u0 = fld_of(U.u0, U.out), out = fld_of(U.out, U.out);
        const unsigned c0 = off_of(U.out, i, j, k);
        Fld ff[3], ms[3];
        unsigned fo[3], mo[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            ff[d] = fld_of(U.ff[d], U.ff[d]);
            ms[d] = fld_of(U.ms[d], U.ms[d]);
            fo[d] = off_of(U.ff[d], i, j, k);
            mo[d] = off_of(U.ms[d], i, j, k);
        }
        const double gs = grav[0] * (ms[0](mo[0], 0, 1, 0, 0) + ms[0](mo[0], 0)) +
                          grav[1] * (ms[1](mo[1], 0, 0, 1, 0) + ms[1](mo[1], 0)) +
                          grav[2] * (ms[2](mo[2], 0, 0, 0, 1) + ms[2](mo[2], 0));
        double o[nv];
#pragma unroll
        for (int n = 0; n < nv; ++n) {
            if (n >= 1 && n <= 3) continue;
            const double div = (ff[0](fo[0], n, 1, 0, 0) - ff[0](fo[0], n)) / P.h(0) +
                               (ff[1](fo[1], n, 0, 1, 0) - ff[1](fo[1], n)) / P.h(1) +
                               (ff[2](fo[2], n, 0, 0, 1) - ff[2](fo[2], n)) / P.h(2);
            double v;
            if (st == 0)
                v = u0(c0, n) - dt * div + dt * src[n];
            else if (st == 1)
                v = 0.25 * (3.0 * u0(c0, n) + us(c0, n) - dt * div + dt * src[n]);
            else
                v = (2. / 3.) * (0.5 * u0(c0, n) + us(c0, n) - dt * div + dt * src[n]);
            o[n] = v;
        }
        if (st == 0)
            o[4] += 0.5 * dt * gs;
        else if (st == 1)
            o[4] += 0.5 * 0.25 * dt * gs;
        else
            o[4] += 0.5 * (2. / 3.) * dt * gs;
#pragma unroll
        for (int n = 0; n < nv; ++n)
            if (n < 1 || n > 3) out(c0, n) = o[n];
        return;
    }
    if (part == 1) stag_update_face<0>(P, U, st, dt, tid);
    else if (part == 2) stag_update_face<1>(P, U, st, dt, tid);
    else stag_update_face<2>(P, U, st, dt, tid);
}

// ---- conservedToPrimitiveStag (conservedPrimitiveConversionsStag.cpp:58-140) ---------------

// TR: 0 conversion only; 1 also the transport coefficients of the parameters' type (1 or 3) and
// 2 of transport_type 2, from the prim values just computed (the same inputs k_transport reads).
// The neighbours' densities are read at their wrapped cells, so no ghost cell needs to be current.
template <int D>
__device__ __forceinline__ void stag_velocity(const DevParams& P, const Arr& va, const Arr& cons, const Arr& ma, long tid)
{
    constexpr int e0 = D == 0, e1 = D == 1, e2 = D == 2;
    const int fx = P.n[0] + e0, fy = P.n[1] + e1, fz = P.n[2] + e2;
    if (tid >= (long)fx * fy * fz) return;
    int i, j, k;
    cell_of(tid, fx, fy, i, j, k);
    const int c = D == 0 ? i : D == 1 ? j : k, n = P.n[D];
    const int up = c == n ? -n : 0, lo = c == 0 ? n - 1 : -1;  // this face's two cells, along D
    const Fld rho = fld_of(cons, cons);
    const unsigned ou = off_of(cons, i + e0 * up, j + e1 * up, k + e2 * up);
    const unsigned ol = off_of(cons, i + e0 * lo, j + e1 * lo, k + e2 * lo), mo = off_of(va, i, j, k);
    fld_of(va, va)(mo, 0) = quot(2 * fld_of(ma, va)(mo, 0), rho(ou, 0) + rho(ol, 0));
}

template <int NS, int TR>
__global__ void __launch_bounds__(SB) k_stag_c2p(DevParams P, Arr prima, Arr vx, Arr vy, Arr vz, Arr consa, Arr mxa,
                                                 Arr mya, Arr mza, StagTransport tc)
{
    // part 0 cells, 1..3 face velocities of direction part-1 (chunk by chunk in turn: 410 us for 207)
    const long tid = (long)blockIdx.x * SB + threadIdx.x;
    switch (blockIdx.y) {
        case 1: stag_velocity<0>(P, vx, consa, mxa, tid); return;
        case 2: stag_velocity<1>(P, vy, consa, mya, tid); return;
        case 3: stag_velocity<2>(P, vz, consa, mza, tid); return;
        default: break;
    }
    const int n0 = P.n[0], n1 = P.n[1], n2 = P.n[2];
    if (tid >= (long)n0 * n1 * n2) return;
    int i, j, k;
    cell_of(tid, n0, n1, i, j, k);
    const Fld prim = fld_of(prima, prima), cons = fld_of(consa, prima);
    const Fld mx = fld_of(mxa, mxa), my = fld_of(mya, mya), mz = fld_of(mza, mza);
    const unsigned c0 = off_of(prima, i, j, k);
    const unsigned ox = off_of(mxa, i, j, k), oy = off_of(mya, i, j, k), oz = off_of(mza, i, j, k);
    auto density = [&](int di, int dj, int dk) {
        const int a = i + di, b = j + dj, c = k + dk;
        return cons(off_of(prima, a < 0 ? n0 - 1 : a == n0 ? 0 : a, b < 0 ? n1 - 1 : b == n1 ? 0 : b,
                           c < 0 ? n2 - 1 : c == n2 ? 0 : c), 0);
    };
    const double rho = cons(c0, 0);
    const double mxl = mx(ox, 0), mxh = mx(ox, 0, 1, 0, 0), myl = my(oy, 0), myh = my(oy, 0, 0, 1, 0),
                 mzl = mz(oz, 0), mzh = mz(oz, 0, 0, 0, 1);
    // the face velocities of this cell, as the face pass computes them
    const double vxl = quot(2 * mxl, rho + density(-1, 0, 0)), vxh = quot(2 * mxh, density(1, 0, 0) + rho);
    const double vyl = quot(2 * myl, rho + density(0, -1, 0)), vyh = quot(2 * myh, density(0, 1, 0) + rho);
    const double vzl = quot(2 * mzl, rho + density(0, 0, -1)), vzh = quot(2 * mzh, density(0, 0, 1) + rho);
    const Rcp rrho = rcp_of(rho);
    double en = cons(c0, 4), part[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) part[n] = cons(c0, 5 + n);
    const double sx = mxh + mxl, sy = myh + myl, sz = mzh + mzl;
    double kin = 0.;
    kin += sx * sx;
    kin += sy * sy;
    kin += sz * sz;
    kin *= (0.125 / rrho);
    const double intenergy = (en - kin) / rrho;
    double Yk[NS], Yf[NS];
    double sumYk = 0.;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        Yk[n] = part[n] / rrho;
        Yf[n] = clamp01(Yk[n]);
        sumYk += Yf[n];
    }
    const Rcp sum = rcp_of(sumYk);
#pragma unroll
    for (int n = 0; n < NS; ++n) Yf[n] = Yf[n] / sum;
    const double T = eos_temperature<NS>(P, intenergy, Yf);
    double molmix = 0.;
#pragma unroll
    for (int n = 0; n < NS; ++n) molmix += Yk[n] / P.M(n);
    molmix = quot(1., molmix);
    const double pres = eos_pressure<NS>(P, Yk, rho, T);
    prim(c0, 0) = rho;
    prim(c0, 1) = 0.5 * (vxl + vxh);
    prim(c0, 2) = 0.5 * (vyl + vyh);
    prim(c0, 3) = 0.5 * (vzl + vzh);
    prim(c0, 4) = T;
    prim(c0, 5) = pres;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        prim(c0, 6 + n) = Yk[n];
        prim(c0, 6 + NS + n) = Yk[n] * molmix / P.M(n);
    }
    cons(c0, 1) = 0.5 * (mxl + mxh);
    cons(c0, 2) = 0.5 * (myl + myh);
    cons(c0, 3) = 0.5 * (mzl + mzh);
    if constexpr (TR != 0) {  // calculateTransportCoeffs of this cell (transCoeffs.cpp:37-88)
        Transport tr;
        double chiv[NS], Dv[NS * NS];
        if constexpr (TR == 2) {
            const int fl = transport_cell_vw<NS>(P, rho, T, pres, Yk, tr, chiv, Dv);
            if (fl) atomicOr(tc.err, fl);
        } else {
            if (transport_cell<NS>(P, rho, T, pres, Yk, tr, chiv, Dv)) atomicOr(tc.err, 1);
        }
        const Fld chi = fld_of(tc.chi, prima), Dm = fld_of(tc.D, prima);
        fld_of(tc.eta, prima)(c0, 0) = tr.eta;
        fld_of(tc.zeta, prima)(c0, 0) = tr.zeta;
        fld_of(tc.kappa, prima)(c0, 0) = tr.kappa;
#pragma unroll
        for (int n = 0; n < NS; ++n) chi(c0, n) = chiv[n];
#pragma unroll
        for (int n = 0; n < NS * NS; ++n) Dm(c0, n) = Dv[n];
    }
}

// ---- periodic ghost fill of cell and face FABs ----------------------------------------------

// blockIdx.y selects a few components of an array: with a whole array to a thread, its loads and stores
// were one chain, as long as the widest array is (64 components of D at eight species).  The threads enumerate only the ghost points: the two z slabs,
// then the two y slabs between them, then the two x slabs; each takes the periodic image.
__global__ void __launch_bounds__(SB) k_stag_fill(DevParams P, FillList L)
{
    const FillItem& it = L.item[blockIdx.y];
    const int g = L.g;
    int V[3], G[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        V[d] = P.n[d] + (d == it.kind - 1);
        G[d] = V[d] + 2 * g;
    }
    const long nz_slab = 2L * g * G[1] * G[0], ny_slab = 2L * V[2] * g * G[0], nx_slab = 2L * V[2] * V[1] * g;
    long t = (long)blockIdx.x * SB + threadIdx.x;
    int i, j, k;
    if (t < nz_slab) {
        const long per = (long)g * G[1] * G[0];
        const int side = t >= per;
        const long r = t - side * per;
        i = (int)(r % G[0]) - g;
        j = (int)((r / G[0]) % G[1]) - g;
        const int kk = (int)(r / ((long)G[0] * G[1]));
        k = side ? V[2] + kk : kk - g;
    } else if ((t -= nz_slab) < ny_slab) {
        const long per = (long)V[2] * g * G[0];
        const int side = t >= per;
        const long r = t - side * per;
        i = (int)(r % G[0]) - g;
        const int jj = (int)((r / G[0]) % g);
        k = (int)(r / ((long)G[0] * g));
        j = side ? V[1] + jj : jj - g;
    } else if ((t -= ny_slab) < nx_slab) {
        const long per = (long)V[2] * V[1] * g;
        const int side = t >= per;
        const long r = t - side * per;
        const int ii = (int)(r % g);
        j = (int)((r / g) % V[1]);
        k = (int)(r / ((long)g * V[1]));
        i = side ? V[0] + ii : ii - g;
    } else {
        return;
    }
    int v[3] = {i, j, k};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        while (v[d] < 0) v[d] += P.n[d];
        while (v[d] > V[d] - 1) v[d] -= P.n[d];
    }
    // up to kFillComps components: every load before the first store
    double x[kFillComps];
    const Arr& shape = L.shape[it.kind];
    const Fld f{it.p, shape.sn, shape.sy, shape.sz};
    const unsigned to = off_of(shape, i, j, k), from = off_of(shape, v[0], v[1], v[2]);
#pragma unroll
    for (int c = 0; c < kFillComps; ++c)
        if (c < it.nc) x[c] = f(from, c);
#pragma unroll
    for (int c = 0; c < kFillComps; ++c)
        if (c < it.nc) f(to, c) = x[c];
}

// ---- host launchers -----------------------------------------------------------------------

#define STAG_NS_DISPATCH(NSV, CALL)                     \
    switch (NSV) {                                      \
        case 2: { constexpr int NS = 2; CALL; } break;  \
        case 3: { constexpr int NS = 3; CALL; } break;  \
        case 4: { constexpr int NS = 4; CALL; } break;  \
        case 5: { constexpr int NS = 5; CALL; } break;  \
        case 6: { constexpr int NS = 6; CALL; } break;  \
        case 7: { constexpr int NS = 7; CALL; } break;  \
        case 8: { constexpr int NS = 8; CALL; } break;  \
        default: return FHDX_ERR_UNSUPPORTED;           \
    }

static long ghost_points(const DevParams& P, int nodal, int g)
{
    long V = 1, G = 1;
    for (int d = 0; d < 3; ++d) {
        const long v = P.n[d] + (d == nodal);
        V *= v;
        G *= v + 2 * g;
    }
    return G - V;
}

int stag_fill(const DevParams& P, const FillList& L, hipStream_t s)
{
    long mx = 0;
    for (int q = 0; q < L.count; ++q) mx = std::max(mx, ghost_points(P, L.item[q].kind - 1, L.g));
    k_stag_fill<<<dim3(grid_for(mx, SB), L.count), SB, 0, s>>>(P, L);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int stag_flux(const DevParams& P, const StagArrays& A, const NoiseKey& K, double w, double dt, bool keep, hipStream_t s)
{
    // cells grown by 1: the largest of the four parts
    const long ngrown1 = (long)(P.n[0] + 2) * (P.n[1] + 2) * (P.n[2] + 2);
    k_stag_stress<<<dim3(grid_for(ngrown1, SB), 4), SB, 0, s>>>(P, A, K, w, dt);
    long nf = 0;
    for (int d = 0; d < 3; ++d) nf = std::max(nf, (long)(P.n[0] + (d == 0)) * (P.n[1] + (d == 1)) * (P.n[2] + (d == 2)));
    STAG_NS_DISPATCH(P.ns, (k_stag_faces<NS><<<3 * grid_for(nf, SB), SB, 0, s>>>(
                                  StagFaceKernel{P, A, K, w, dt, keep ? 1 : 0})));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int stag_update(const DevParams& P, const StagUpdate& U, int st, double dt, hipStream_t s)
{
    long mx = (long)P.n[0] * P.n[1] * P.n[2];
    for (int d = 0; d < 3; ++d) mx = std::max(mx, (long)(P.n[0] + (d == 0)) * (P.n[1] + (d == 1)) * (P.n[2] + (d == 2)));
    // without chemistry the species source is a literal zero and needs no registers: 138 VGPRs and 46 (argon 160^3: 368 -> 295 us)
    if (U.chem) {
        STAG_NS_DISPATCH(P.ns, (k_stag_update<NS, true><<<dim3(grid_for(mx, SB), 4), SB, 0, s>>>(P, U, st, dt)));
    } else {
        STAG_NS_DISPATCH(P.ns, (k_stag_update<NS, false><<<dim3(grid_for(mx, SB), 4), SB, 0, s>>>(P, U, st, dt)));
    }
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int stag_c2p(const DevParams& P, Arr prim, const Arr vel[3], Arr cons, const Arr mom[3], const StagTransport* tr,
             hipStream_t s)
{
    long mx = (long)P.n[0] * P.n[1] * P.n[2];
    for (int d = 0; d < 3; ++d) mx = std::max(mx, (long)(P.n[0] + (d == 0)) * (P.n[1] + (d == 1)) * (P.n[2] + (d == 2)));
    const dim3 grid(grid_for(mx, SB), 4);
    const StagTransport tc = tr ? *tr : StagTransport{};
    if (!tr) {
        STAG_NS_DISPATCH(P.ns, (k_stag_c2p<NS, 0><<<grid, SB, 0, s>>>(P, prim, vel[0], vel[1], vel[2], cons, mom[0],
                                                                       mom[1], mom[2], tc)));
    } else if (P.transport_type == 2) {
        STAG_NS_DISPATCH(P.ns, (k_stag_c2p<NS, 2><<<grid, SB, 0, s>>>(P, prim, vel[0], vel[1], vel[2], cons, mom[0],
                                                                       mom[1], mom[2], tc)));
    } else {
        STAG_NS_DISPATCH(P.ns, (k_stag_c2p<NS, 1><<<grid, SB, 0, s>>>(P, prim, vel[0], vel[1], vel[2], cons, mom[0],
                                                                       mom[1], mom[2], tc)));
    }
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

}  // namespace fhdx
