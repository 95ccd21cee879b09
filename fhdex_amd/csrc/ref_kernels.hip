// ref_kernels.hip -- the reference-shaped kernels of calculateFlux / RK3step on gfx950.
//
// A stage is transport, corner nodes, faces (every flux family of a face and its noise in one pass, the
// three directions in one launch), the stage combination with the conversion to primitive variables,
// and every ghost cell in one launch; each thread owns one cell, face or node.  These back the drop-in
// entry points that fill the reference's own intermediate
// arrays (fhdx_calculate_flux, fhdx_rk3_step_ref).  Arithmetic follows the reference
// operation by operation (see physics.hpp for why that is required).
#include "kernels.hpp"
#include "stage_bodies.hpp"

namespace fhdx {

constexpr int BLK = 256;

// Edge-viscosity summation order per face direction and edge (pp, mp, pm, mm): offsets of the
// eta cell then of the T cell relative to the face index, flux.cpp:117-135 (x), 481-499 (y),
// 847-865 (z, including the eta(k-2)*T(k) terms of 857-858).
__device__ constexpr signed char c_mu_order[3][4][8][6] = {
    {{{0,0,0,0,0,0},{-1,0,0,-1,0,0},{0,1,0,0,1,0},{-1,1,0,-1,1,0},{0,0,1,0,0,1},{-1,0,1,-1,0,1},{0,1,1,0,1,1},{-1,1,1,-1,1,1}},
     {{0,-1,0,0,-1,0},{-1,-1,0,-1,-1,0},{0,0,0,0,0,0},{-1,0,0,-1,0,0},{0,-1,1,0,-1,1},{-1,-1,1,-1,-1,1},{0,0,1,0,0,1},{-1,0,1,-1,0,1}},
     {{0,0,-1,0,0,-1},{-1,0,-1,-1,0,-1},{0,1,-1,0,1,-1},{-1,1,-1,-1,1,-1},{0,0,0,0,0,0},{-1,0,0,-1,0,0},{0,1,0,0,1,0},{-1,1,0,-1,1,0}},
     {{0,-1,-1,0,-1,-1},{-1,-1,-1,-1,-1,-1},{0,0,-1,0,0,-1},{-1,0,-1,-1,0,-1},{0,-1,0,0,-1,0},{-1,-1,0,-1,-1,0},{0,0,0,0,0,0},{-1,0,0,-1,0,0}}},
    {{{1,-1,0,1,-1,0},{0,-1,0,0,-1,0},{1,0,0,1,0,0},{0,0,0,0,0,0},{1,-1,1,1,-1,1},{0,-1,1,0,-1,1},{1,0,1,1,0,1},{0,0,1,0,0,1}},
     {{-1,0,0,-1,0,0},{0,0,0,0,0,0},{-1,-1,0,-1,-1,0},{0,-1,0,0,-1,0},{-1,0,1,-1,0,1},{0,0,1,0,0,1},{-1,-1,1,-1,-1,1},{0,-1,1,0,-1,1}},
     {{1,-1,-1,1,-1,-1},{0,-1,-1,0,-1,-1},{1,0,-1,1,0,-1},{0,0,-1,0,0,-1},{1,-1,0,1,-1,0},{0,-1,0,0,-1,0},{1,0,0,1,0,0},{0,0,0,0,0,0}},
     {{-1,0,-1,-1,0,-1},{0,0,-1,0,0,-1},{-1,-1,-1,-1,-1,-1},{0,-1,-1,0,-1,-1},{-1,0,0,-1,0,0},{0,0,0,0,0,0},{-1,-1,0,-1,-1,0},{0,-1,0,0,-1,0}}},
    {{{1,0,-1,1,0,-1},{0,0,-1,0,0,-1},{1,1,-1,1,1,-1},{0,1,-1,0,1,-1},{1,0,0,1,0,0},{0,0,0,0,0,0},{1,1,0,1,1,0},{0,1,0,0,1,0}},
     {{-1,1,-1,-1,1,-1},{0,1,-1,0,1,-1},{-1,0,-1,-1,0,-1},{0,0,-1,0,0,-1},{-1,1,0,-1,1,0},{0,1,0,0,1,0},{-1,0,0,-1,0,0},{0,0,0,0,0,0}},
     {{1,0,0,1,0,0},{0,0,-2,0,0,0},{1,-1,0,1,-1,0},{0,-1,-2,0,-1,0},{1,0,-1,1,0,-1},{0,0,-1,0,0,-1},{1,-1,-1,1,-1,-1},{0,-1,-1,0,-1,-1}},
     {{-1,-1,0,-1,-1,0},{0,-1,0,0,-1,0},{-1,0,0,-1,0,0},{0,0,0,0,0,0},{-1,-1,-1,-1,-1,-1},{0,-1,-1,0,-1,-1},{-1,0,-1,-1,0,-1},{0,0,-1,0,0,-1}}}};

// Node (rancorn) offsets of the pp, mp, pm, mm edges (flux.cpp:277-280, 644-647, 1011-1014).
__device__ constexpr signed char c_rc_node[3][4][3] = {{{0, 1, 1}, {0, 0, 1}, {0, 1, 0}, {0, 0, 0}},
                                               {{1, 0, 1}, {0, 0, 1}, {1, 0, 0}, {0, 0, 0}},
                                               {{1, 1, 0}, {0, 1, 0}, {1, 0, 0}, {0, 0, 0}}};

// Wall faces: the four edge-viscosity cells in the ghost layer (normal offset -1 at a lo face,
// 0 at a hi face), transverse offsets per face direction and edge in the reference's order
// (flux.cpp:137-156 x, 501-520 y, 867-886 z).
__device__ constexpr signed char c_mu_wall[3][4][4][3] = {
    {{{0, 0, 0}, {0, 1, 0}, {0, 0, 1}, {0, 1, 1}}, {{0, -1, 0}, {0, 0, 0}, {0, -1, 1}, {0, 0, 1}},
     {{0, 0, -1}, {0, 1, -1}, {0, 0, 0}, {0, 1, 0}}, {{0, -1, -1}, {0, 0, -1}, {0, -1, 0}, {0, 0, 0}}},
    {{{1, 0, 0}, {0, 0, 0}, {1, 0, 1}, {0, 0, 1}}, {{-1, 0, 0}, {0, 0, 0}, {-1, 0, 1}, {0, 0, 1}},
     {{1, 0, -1}, {0, 0, -1}, {1, 0, 0}, {0, 0, 0}}, {{-1, 0, -1}, {0, 0, -1}, {-1, 0, 0}, {0, 0, 0}}},
    {{{1, 0, 0}, {0, 0, 0}, {1, 1, 0}, {0, 1, 0}}, {{-1, 1, 0}, {0, 1, 0}, {-1, 0, 0}, {0, 0, 0}},
     {{1, 0, 0}, {0, 0, 0}, {1, -1, 0}, {0, -1, 0}}, {{-1, -1, 0}, {0, -1, 0}, {-1, 0, 0}, {0, 0, 0}}}};

// Where a face of direction D stands relative to the walls: lo/hi are set on a bc_mass 1/2
// face at index 0 / n_D (the is_*_dirichlet_mass branches of flux.cpp); (wi, wj, wk) is the
// wall-side cell (the ghost at a lo face, the boundary cell at a hi face).
struct WallFace {
    bool lo, hi;
    int wi, wj, wk;
    __device__ bool any() const { return lo || hi; }
};

template <int D>
__device__ inline WallFace wall_face(const DevParams& P, int i, int j, int k)
{
    WallFace w;
    const int c = (D == 0) ? i : (D == 1) ? j : k;
    w.lo = P.any_wall && c == 0 && P.wall[2 * D];
    w.hi = P.any_wall && c == P.n[D] && P.wall[2 * D + 1];
    w.wi = i - (w.lo && D == 0);
    w.wj = j - (w.lo && D == 1);
    w.wk = k - (w.lo && D == 2);
    return w;
}

__device__ inline void face_index(long t, int fx, int fy, int& i, int& j, int& k)
{
    i = (int)(t % fx);
    long r = t / fx;
    j = (int)(r % fy);
    k = (int)(r / fy);
}

// Thread t of a launch over the launch box's cells grown by (ex, ey, ez) on the hi side (faces
// of direction d: 1 along d; nodes: 1 along every axis), as global indices (i, j, k); false
// past the end.  Wall and periodic tests keep using the domain size P.n.
__device__ inline bool box_index(const DevParams& P, long t, int ex, int ey, int ez, int& i, int& j, int& k)
{
    const int fx = P.bn[0] + ex, fy = P.bn[1] + ey, fz = P.bn[2] + ez;
    if (t >= (long)fx * fy * fz) return false;
    face_index(t, fx, fy, i, j, k);
    i += P.bo[0];
    j += P.bo[1];
    k += P.bo[2];
    return true;
}

__device__ __forceinline__ long xcd_thread() { return (long)xcd_block(blockIdx.x, gridDim.x) * BLK + threadIdx.x; }

// ---- cell kernels -------------------------------------------------------------------------

template <int NS>
__global__ void __launch_bounds__(BLK) k_c2p(DevParams P, Arr prim, Arr cons)
{
    const long t = xcd_thread();
    int i, j, k;
    if (!box_index(P, t, 0, 0, 0, i, j, k)) return;
    double c[NS + 5], pr[2 * NS + 6];
#pragma unroll
    for (int n = 0; n < NS + 5; ++n) c[n] = cons(i, j, k, n);
    cons_to_prim_cell<NS>(P, c, pr);
#pragma unroll
    for (int n = 0; n < 2 * NS + 6; ++n) prim(i, j, k, n) = pr[n];
}

template <int NS, bool VW>
__global__ void __launch_bounds__(BLK) k_transport(DevParams P, Arr prima, Arr etaa, Arr zetaa,
                                                   Arr kappaa, Arr chia, Arr Da, int* err)
{
    const int g = P.ngc;
    const int gx = P.bn[0] + 2 * g, gy = P.bn[1] + 2 * g, gz = P.bn[2] + 2 * g;
    const long t = xcd_thread();
    if (t >= (long)gx * gy * gz) return;
    int i, j, k;
    face_index(t, gx, gy, i, j, k);
    i += P.bo[0] - g;
    j += P.bo[1] - g;
    k += P.bo[2] - g;
    const Fld prim = fld_of(prima, prima), eta = fld_of(etaa, prima), zeta = fld_of(zetaa, prima),
              kappa = fld_of(kappaa, prima), chi = fld_of(chia, prima), Dm = fld_of(Da, prima);
    const unsigned cb = off_of(prima, i, j, k);
    double Y[NS], chiv[NS], Dv[NS * NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) Y[n] = prim(cb, 6 + n);
    Transport tr;
    if constexpr (VW) {  // transport_type 2
        const int fl = transport_cell_vw<NS>(P, prim(cb, 0), prim(cb, 4), prim(cb, 5), Y, tr, chiv, Dv);
        if (fl) atomicOr(err, fl);
    } else {
        bool bad = transport_cell<NS>(P, prim(cb, 0), prim(cb, 4), prim(cb, 5), Y, tr,
                                      chiv, Dv);
        if (bad) atomicOr(err, 1);
    }
    eta(cb, 0) = tr.eta;
    zeta(cb, 0) = tr.zeta;
    kappa(cb, 0) = tr.kappa;
#pragma unroll
    for (int n = 0; n < NS; ++n) chi(cb, n) = chiv[n];
#pragma unroll
    for (int n = 0; n < NS * NS; ++n) Dm(cb, n) = Dv[n];
}

// Periodic ghost fill of a cell FAB: ghost (i,j,k) <- valid (i mod n, ...) along periodic
// directions; a ghost cell outside a wall has no periodic image and is left to setBC.
__global__ void __launch_bounds__(BLK) k_fill_boundary(DevParams P, Arr a, int nc)
{
    const int g = P.ngc, n0 = P.n[0], n1 = P.n[1], n2 = P.n[2];
    const int gx = n0 + 2 * g, gy = n1 + 2 * g, gz = n2 + 2 * g;
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    if (t >= (long)gx * gy * gz) return;
    int i, j, k;
    face_index(t, gx, gy, i, j, k);
    i -= g;
    j -= g;
    k -= g;
    if ((!P.periodic[0] && (i < 0 || i >= n0)) || (!P.periodic[1] && (j < 0 || j >= n1)) ||
        (!P.periodic[2] && (k < 0 || k >= n2)))
        return;
    // the image of a ghost cell, any number of periods away (boxes thinner than ngc included)
    int iv = (i % n0 + n0) % n0, jv = (j % n1 + n1) % n1, kv = (k % n2 + n2) % n2;
    if (iv == i && jv == j && kv == k) return;
    for (int n = 0; n < nc; ++n) a(i, j, k, n) = a(iv, jv, kv, n);
}

// One face of setBC (boundary.cpp:180-1036): every cell of the grown box outside face
// (D, side) takes its value from the mirror cell (-c-1 at lo, 2n-c-1 at hi) and the wall data:
// mass fractions mirrored (bc_mass 1) or fixed (2); T and p mirrored (adiabatic) or T = t_wall
// with p mirrored (isothermal); velocity: slip (normal 0, tangential mirrored) or no slip (0);
// then rho from GetDensity and the conserved state from it.
// One launch per direction covers the ghost slabs of both faces (2*ngc layers across D, the
// grown box along the other two): the lo and hi passes write disjoint cells and read only
// mirror cells inside the box, so running them together equals running them in turn.
template <int NS>
__global__ void __launch_bounds__(BLK) k_set_bc(DevParams P, Arr prim, Arr cons, int D)
{
    const int g = P.ngc, n = P.n[D];
    int ext[3] = {P.bn[0] + 2 * g, P.bn[1] + 2 * g, P.bn[2] + 2 * g};
    ext[D] = 2 * g;
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    if (t >= (long)ext[0] * ext[1] * ext[2]) return;
    int c[3];
    face_index(t, ext[0], ext[1], c[0], c[1], c[2]);
    for (int d = 0; d < 3; ++d)
        if (d != D) c[d] += P.bo[d] - g;
    const int side = c[D] >= g;  // layers 0..g-1: lo ghosts -g..-1; g..2g-1: hi ghosts n..n+g-1
    // a box that does not reach this side of the domain has no wall ghosts there
    if (side ? P.bo[D] + P.bn[D] != n : P.bo[D] != 0) return;
    c[D] = side ? n + (c[D] - g) : c[D] - g;
    int m[3] = {c[0], c[1], c[2]};
    m[D] = side ? 2 * (n - 1) - c[D] + 1 : -c[D] - 1;
    const int f = 2 * D + side;
    const int bm = P.bcm[f], bt = P.bct[f], bv = P.bcv[f];
#define PR(a, q) prim(a[0], a[1], a[2], q)
#define CO(a, q) cons(a[0], a[1], a[2], q)
    if (bm == 1 && P.algorithm_type == 2)
#pragma unroll
        for (int q = 6; q < 6 + 2 * NS; ++q) PR(c, q) = PR(m, q);
    if (bm == 2 && P.algorithm_type == 2)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            PR(c, 6 + s) = P.Yw[f][s];
            PR(c, 6 + NS + s) = P.Xw[f][s];
        }
    if (bm == 3 && P.algorithm_type == 2) {
        // x reservoir (boundary.cpp:221-238, 260-288): the reservoir gas at rest; no thermal or velocity
        // branch follows (the x chain is else-if)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            PR(c, 6 + s) = P.Yw[f][s];
            PR(c, 6 + NS + s) = P.Xw[f][s];
        }
        const double rho = P.rhow[f];
        PR(c, 0) = rho;
        CO(c, 0) = rho;
        PR(c, 4) = P.tw[f];
        PR(c, 5) = P.pw[f];
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            CO(c, q) = 0.0;
            PR(c, q) = 0.0;
        }
        double Yr[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) Yr[s] = P.Yw[f][s];
        const double ie = eos_energy<NS>(P, Yr, P.tw[f]);
#pragma unroll
        for (int s = 0; s < NS; ++s) CO(c, 5 + s) = rho * Yr[s];
        CO(c, 4) = rho * ie + 0.5 * rho * (0.0 * 0.0 + 0.0 * 0.0 + 0.0 * 0.0);
        return;
    }
    if (bt == 1) {
        PR(c, 4) = PR(m, 4);
        PR(c, 5) = PR(m, 5);
    } else if (bt == 2) {
        PR(c, 4) = P.tw[f];
        PR(c, 5) = PR(m, 5);
    }
    if (bv != 1 && bv != 2) return;
    double v[4];
    if (bv == 1) {
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const bool normal = (q == 1 + D);
            CO(c, q) = normal ? 0.0 : CO(m, q);
            v[q] = normal ? 0.0 : PR(m, q);
            PR(c, q) = v[q];
        }
    } else {
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            v[q] = 0.0;
            PR(c, q) = 0.0;
        }
    }
    double Y[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) Y[s] = PR(c, 6 + s);
    const double T = PR(c, 4), pt = PR(c, 5);
    double molmix = 0.;
#pragma unroll
    for (int s = 0; s < NS; ++s) molmix += Y[s] / P.molmass[s];
    molmix = 1. / molmix;
    const double rho = pt / (P.Runiv / molmix) / T;  // GetDensity, compressible_functions.H:1481-1495
    const double ie = eos_energy<NS>(P, Y, T);
    PR(c, 0) = rho;
    CO(c, 0) = rho;
    if (P.algorithm_type == 2)
#pragma unroll
        for (int s = 0; s < NS; ++s) CO(c, 5 + s) = rho * Y[s];
    if (bv == 2)
#pragma unroll
        for (int q = 1; q < 4; ++q) CO(c, q) = rho * v[q];
    CO(c, 4) = rho * ie + 0.5 * rho * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]);
#undef PR
#undef CO
}

// One face of setBC in registers: pr, co hold the mirror cell's values and become the ghost cell's.
// For algorithm_type 2, where every component is written (walls are refused otherwise).
template <int NS>
__device__ __forceinline__ void wall_ghost(const DevParams& P, int f, double* pr, double* co)
{
    const int D = f >> 1, bm = P.bcm[f], bt = P.bct[f], bv = P.bcv[f];
    if (bm == 2 || bm == 3)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            pr[6 + s] = P.Yw[f][s];
            pr[6 + NS + s] = P.Xw[f][s];
        }
    double Y[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) Y[s] = pr[6 + s];
    if (bm == 3) {  // x reservoir (boundary.cpp:221-238, 260-288)
        const double rho = P.rhow[f];
        pr[0] = co[0] = rho;
        pr[4] = P.tw[f];
        pr[5] = P.pw[f];
#pragma unroll
        for (int q = 1; q < 4; ++q) co[q] = pr[q] = 0.0;
        const double ie = eos_energy<NS>(P, Y, P.tw[f]);
#pragma unroll
        for (int s = 0; s < NS; ++s) co[5 + s] = rho * Y[s];
        co[4] = rho * ie + 0.5 * rho * (0.0 * 0.0 + 0.0 * 0.0 + 0.0 * 0.0);
        return;
    }
    if (bt == 2) pr[4] = P.tw[f];
#pragma unroll
    for (int q = 1; q < 4; ++q)
        if (bv == 2 || q == 1 + D) co[q] = pr[q] = 0.0;
    const double T = pr[4], pt = pr[5];
    double molmix = 0.;
#pragma unroll
    for (int s = 0; s < NS; ++s) molmix += Y[s] / P.M(s);
    molmix = quot(1., molmix);
    const double rho = quot(quot(pt, quot(P.Runiv, molmix)), T);  // GetDensity, compressible_functions.H:1481-1495
    const double ie = eos_energy<NS>(P, Y, T);
    pr[0] = co[0] = rho;
#pragma unroll
    for (int s = 0; s < NS; ++s) co[5 + s] = rho * Y[s];
    if (bv == 2)
#pragma unroll
        for (int q = 1; q < 4; ++q) co[q] = rho * pr[q];
    co[4] = rho * ie + 0.5 * rho * (pr[1] * pr[1] + pr[2] * pr[2] + pr[3] * pr[3]);
}

// FillBoundary and setBC of a stage's state and prim in one launch, one thread per ghost cell.  Each is
// a function of one valid cell: its periodic image, mirrored in the walls, through the wall rules of
// the directions it lies outside of, x before y before z (a pass of setBC reads what the one before
// wrote).  So nothing is read that another thread writes, and the launch replaces one fill of the
// grown box and up to three dependent setBC launches a stage: temp_grad (80x10x10, walls all round) 26 -> 6.4 us,
// argon 128^3 54 -> 27 us.
template <int NS>
__global__ void __launch_bounds__(BLK) k_ghosts(DevParams P, Arr prima, Arr consa)
{
    int c[3];
    if (!ghost_cell(P.ngc, P.n[0], P.n[1], P.n[2], (long)blockIdx.x * BLK + threadIdx.x, c[0], c[1], c[2])) return;
    int m[3], face[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int n = P.n[d];
        const bool lo = c[d] < 0, hi = c[d] >= n;
        face[d] = -1;
        m[d] = c[d];
        if (P.periodic[d]) {
            m[d] = (c[d] % n + n) % n;  // any number of periods away
        } else if (lo || hi) {
            m[d] = lo ? -c[d] - 1 : 2 * (n - 1) - c[d] + 1;
            face[d] = 2 * d + (hi ? 1 : 0);
        }
    }
    const Fld prim = fld_of(prima, prima), cons = fld_of(consa, prima);
    const unsigned from = off_of(prima, m[0], m[1], m[2]), to = off_of(prima, c[0], c[1], c[2]);
    double pr[2 * NS + 6], co[NS + 5];
#pragma unroll
    for (int q = 0; q < 2 * NS + 6; ++q) pr[q] = prim(from, q);
#pragma unroll
    for (int q = 0; q < NS + 5; ++q) co[q] = cons(from, q);
    for (int d = 0; d < 3; ++d)
        if (face[d] >= 0) wall_ghost<NS>(P, face[d], pr, co);
#pragma unroll
    for (int q = 0; q < 2 * NS + 6; ++q) prim(to, q) = pr[q];
#pragma unroll
    for (int q = 0; q < NS + 5; ++q) cons(to, q) = co[q];
}

__global__ void __launch_bounds__(BLK) k_fill(double* p, long n, double v)
{
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    if (t < n) p[t] = v;
}

// ---- stochastic face flux (flux.cpp:71-1145) -----------------------------------------------
// At a wall face (bc_mass 1/2) the face-local averages read the wall-side cell for both sides:
// 2*eta*T, 2*kappa*T^2, T, 2*w*u and the species terms of flux.cpp:88-97, 137-202, 318-327,
// 343-427 are then reproduced bit for bit (every rewrite is an exact doubling or halving).
// The edge viscosities take the four ghost-layer cells, and edges touching a tangential wall
// are scaled by sqrt(2) (slip) or 0 (no slip) (:250-280).  StochFlux (boundary.cpp:1392-1970)
// then scales the face's stochastic fluxes, applied here to the values this thread wrote.

// A face's views and byte offsets: cell (i,j,k) and the one below it, the lower and upper cells of
// the face averages (both the wall-side cell at a wall), and node (i,j,k).
struct FaceView {
    Fld cons, prim, eta, zeta, kappa, chi, Dm, visccorn, rancorn;
    Fld corn[3][3];
    unsigned c0, cm, lo, up, nd;
};

// The edge terms of the face, fac sqrt(mu) rancorn summed over its four edges.
template <int D, bool WALL>
__device__ __forceinline__ double edge_sum(const DevParams& P, const FaceView& V, bool wall, int i, int j, int k)
{
    const Fld &prim = V.prim, &eta = V.eta, &zeta = V.zeta;
    const unsigned up = V.up;
    constexpr Rcp three{3., 1. / 3.};
    // tangential-wall factors of the four edges (pp, mp, pm, mm) over transverse axes (A, B)
    constexpr int TA = (D == 0) ? 1 : 0, TB = (D == 2) ? 1 : 2;
    double fac[4] = {1., 1., 1., 1.};
    if (WALL) {
        const int idx[3] = {i, j, k};
        double flo[2] = {1., 1.}, fhi[2] = {1., 1.};
        const int ax[2] = {TA, TB};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int a = ax[q];
            const int vl = P.bcv[2 * a], vh = P.bcv[2 * a + 1];
            if ((vl == 1 || vl == 2) && idx[a] == 0) flo[q] = (vl == 1) ? sqrt(2.0) : 0.;
            if ((vh == 1 || vh == 2) && idx[a] == P.n[a] - 1) fhi[q] = (vh == 1) ? sqrt(2.0) : 0.;
        }
        fac[0] = fhi[0] * fhi[1];
        fac[1] = flo[0] * fhi[1];
        fac[2] = fhi[0] * flo[1];
        fac[3] = flo[0] * flo[1];
    }

    double sum = 0.;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        double mu;
        if (wall) {
            double s4 = 0., z4 = 0.;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const signed char* o = c_mu_wall[D][c][q];
                const double T = prim(up, 4, o[0], o[1], o[2]);
                const double e = eta(up, 0, o[0], o[1], o[2]) * T;
                s4 = (q == 0) ? e : s4 + e;
                if (P.visc_type == 3 || P.visc_type == -3) {
                    const double zz = zeta(up, 0, o[0], o[1], o[2]) * T;
                    z4 = (q == 0) ? zz : z4 + zz;
                }
            }
            mu = 0.5 * s4 / three;
            if (P.visc_type == 3 || P.visc_type == -3) mu += (D == 0) ? 0.5 * z4 : 0.5 * z4 / three;
        } else {
            double s8 = 0.;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const signed char* o = c_mu_order[D][c][q];
                double term = eta(V.c0, 0, o[0], o[1], o[2]) * prim(V.c0, 4, o[3], o[4], o[5]);
                s8 = (q == 0) ? term : s8 + term;
            }
            mu = 0.25 * s8 / three;
            if (P.visc_type == 3 || P.visc_type == -3) {
                double z = 0.;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const signed char* o = c_mu_order[D][c][q];
                    double term = zeta(V.c0, 0, o[0], o[1], o[2]) * prim(V.c0, 4, o[3], o[4], o[5]);
                    z = (q == 0) ? term : z + term;
                }
                mu += 0.25 * z;
            }
        }
        const signed char* nd = c_rc_node[D][c];
        double term = fac[c] * root(mu) * V.rancorn(V.nd, 0, nd[0], nd[1], nd[2]);
        sum = (c == 0) ? term : sum + term;
    }
    return sum;
}

// Seven and eight species with walls: the edges, whose two forms are a divergent branch, before the noise and
// all else that is held in registers through them.  With them here at eight (256 VGPRs, 242 AGPRs) the
// compiler put copies of two noise values at the head of the block behind the branch, before the execution
// mask is whole again, and the lanes that had gone the other way lost them.  Fewer species have no such copies.
// 48^3 with walls, us a step here / first: four species 384/406, five 649/673, six 741/751, seven 1044/924.
template <int NS, bool WALL>
constexpr bool kEdgesFirst = WALL && NS > 6;

template <int NS, int D, bool WALL>
__device__ __forceinline__ void stoch_part(const DevParams& P, const FaceView& V, bool wall, double edges,
                                           const double* ran, double* o, double volinv, double dtinv, double dt,
                                           int i, int j, int k)
{
    const Fld &prim = V.prim, &eta = V.eta, &kappa = V.kappa, &chi = V.chi, &Dm = V.Dm;
    const unsigned lo = V.lo, up = V.up;
    const int nv = NS + 5;

    double Tu = prim(up, 4), Tl = prim(lo, 4);
    double mup = eta(up, 0) * Tu + eta(lo, 0) * Tl;
    double kp = kappa(up, 0) * Tu * Tu + kappa(lo, 0) * Tl * Tl;
    double meanT = 0.5 * (Tu + Tl);
    double w[NS + 5];
    double fw1 = root(P.k_B * mup * volinv * dtinv);
    double fw4 = root(P.k_B * kp * volinv * dtinv);
    w[1] = fw1 * ran[1];
    w[2] = fw1 * ran[2];
    w[3] = fw1 * ran[3];
    w[4] = fw4 * ran[4];
    double nweight = root(P.k_B * volinv * dtinv);

    if (!kEdgesFirst<NS, WALL>) edges = edge_sum<D, WALL>(P, V, wall, i, j, k);
    w[1 + D] = w[1 + D] + 0.25 * nweight * edges;

    // this face's flux after the stochastic pass: the reference adds to a zeroed array
    // (flux.cpp:24-26), so each term is 0.0 + term
#pragma unroll
    for (int n = 1; n < 4; ++n) o[n] = 0.0 + w[n];
    o[nv] = 0.0 + w[4];

    constexpr int t1 = (D == 0) ? 2 : 1, t2 = (D == 2) ? 2 : 3;
    double phidiag = w[1 + D] * (prim(lo, 1 + D) + prim(up, 1 + D));
    double phishear = w[t1] * (prim(lo, t1) + prim(up, t1)) +
                      w[t2] * (prim(lo, t2) + prim(up, t2));
    phidiag = -0.5 * phidiag;
    phishear = -0.5 * phishear;
    o[nv + 1] = 0.0 - phidiag;
    o[nv + 2] = 0.0 - phishear;

    if (P.algorithm_type == 2) {
        double yy[NS], yyp[NS], DijY[NS * NS], sqD[NS * NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            w[5 + s] = 0.;
            yy[s] = clamp01(prim(lo, 6 + s));
            yyp[s] = clamp01(prim(up, 6 + s));
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
                DijY[s * NS + l] = 0.5 * (Dm(lo, l * NS + s) * yy[l] + Dm(up, l * NS + s) * yyp[l] +
                                          (Dm(lo, s * NS + l) * yy[s] + Dm(up, s * NS + l) * yyp[s]));
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
        double wsp = root(quot(P.k_B * MWmix * volinv, P.Runiv * dt));
#pragma unroll
        for (int s = 0; s < NS; ++s) {
#pragma unroll
            for (int l = 0; l <= s; ++l) w[5 + s] = w[5 + s] + (wsp * sqD[s * NS + l]) * ran[5 + l];
            o[5 + s] = w[5 + s];
        }
        double soret = 0.;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double hk = P.e0[s] + P.hcp[s] * meanT;
            double ss = (hk + P.Runiv * meanT / P.M(s) * 0.5 * (chi(lo, s) + chi(up, s))) *
                        w[5 + s];
            soret = soret + ss;
        }
        o[nv + 3] = o[nv + 3] + soret;
    }

    if (WALL) {  // StochFlux on the wall planes of direction D
        const int c = (D == 0) ? i : (D == 1) ? j : k;
        const int f = (c == 0) ? 2 * D : (c == P.n[D]) ? 2 * D + 1 : -1;
        if (f >= 0) {
            const int bm = P.bcm[f], bt = P.bct[f], bv = P.bcv[f];
            if (bm == 1 || bm == 2) {
                const double factor = (bm == 1) ? 0. : sqrt(2.);
                if (P.algorithm_type == 2)
#pragma unroll
                    for (int s = 0; s < NS; ++s) o[5 + s] *= factor;
                o[nv + 3] *= factor;
            }
            if (bt == 1 || bt == 2) {
                double factor = (bt == 1) ? 0. : sqrt(2.);
                if (D == 0 && bm == 3) factor = 1.0;
                o[nv] *= factor;
            }
            if (bv == 1 || bv == 2) {
                const double factor = (bv == 1) ? 0. : sqrt(2.);
                const double sqrtTwo = sqrt(2.);
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    if (n == D) {
                        o[1 + n] *= sqrtTwo;
                        o[nv + 1] *= sqrtTwo;
                        o[nv + 2] *= factor;
                    } else {
                        o[1 + n] *= factor;
                    }
                }
            }
        }
    }
}

// ---- diffusive face flux (flux.cpp:1193-1623) ----------------------------------------------
// At a wall face the gradients span half a cell and the coefficients, means and the Soret
// chi*X read the wall-side cell (flux.cpp:1218-1290 and the y/z images; the z-face chi quirks
// of :1561, :1604 are not in those branches).  BCWallSpeciesFlux (boundary.cpp:1212-1390) then
// zeroes species, density and Dufour fluxes on bc_mass 1 faces; the corner pass in between
// touches none of those components, so it is applied here.

template <int NS, int D, bool WALL>
__device__ __forceinline__ void diff_part(const DevParams& P, const FaceView& V, const WallFace& W, double* o)
{
    const Fld &prim = V.prim, &eta = V.eta, &kappa = V.kappa, &chi = V.chi, &Dm = V.Dm;
    // gradients between c0 and cm; coefficients and means of lo and up (the wall-side cell twice)
    const unsigned c0 = V.c0, cm = V.cm, lo = V.lo, up = V.up;
    const bool wall = WALL && W.any();
    const int nv = NS + 5;
    const double half = 0.5;
    const Rcp h{wall ? 0.5 * P.dx[D] : P.dx[D], wall ? 2.0 * P.rdx[D] : P.rdx[D]};

    double mup = half * (eta(up, 0) + eta(lo, 0));
    double kp = half * (kappa(up, 0) + kappa(lo, 0));
    double tau1 = mup * (prim(c0, 1) - prim(cm, 1)) / h;
    double tau2 = mup * (prim(c0, 2) - prim(cm, 2)) / h;
    double tau3 = mup * (prim(c0, 3) - prim(cm, 3)) / h;
    double divp = 0.;
    double s1 = prim(lo, 1) + prim(up, 1);
    double s2 = prim(lo, 2) + prim(up, 2);
    double s3 = prim(lo, 3) + prim(up, 3);
    double phiflx;
    if (D == 0) phiflx = tau1 * s1 + divp * s1 + tau2 * s2 + tau3 * s3;
    else if (D == 1) phiflx = tau1 * s1 + tau2 * s2 + divp * s2 + tau3 * s3;
    else phiflx = tau1 * s1 + tau2 * s2 + tau3 * s3 + divp * s3;
    double Qflux = kp * (prim(c0, 4) - prim(cm, 4)) / h;
    o[1] = o[1] - (D == 0 ? tau1 + divp : tau1);
    o[2] = o[2] - (D == 1 ? tau2 + divp : tau2);
    o[3] = o[3] - (D == 2 ? tau3 + divp : tau3);
    o[nv] = o[nv] - Qflux;
    o[nv + 1] = o[nv + 1] - (half * phiflx);

    double meanT = 0.5 * (prim(lo, 4) + prim(up, 4));
    double meanP = 0.5 * (prim(lo, 5) + prim(up, 5));
    if (P.algorithm_type == 2) {
        const Rcp rT = rcp_of(meanT), rP = rcp_of(meanP);
        double dk[NS], soret[NS], Fk[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double XU = prim(c0, 6 + NS + s), XL = prim(cm, 6 + NS + s);
            double term1 = (XU - XL) / h;
            double mX = 0.5 * (prim(lo, 6 + NS + s) + prim(up, 6 + NS + s));
            double mY = 0.5 * (prim(lo, 6 + s) + prim(up, 6 + s));
            double term2 = (mX - mY) * (prim(c0, 5) - prim(cm, 5)) / h / rP;
            dk[s] = term1 + term2;
            double ChiX;
            if (D == 2 && !wall)  // flux.cpp:1561 reads chi at k and k+1
                ChiX = 0.5 * (chi(c0, s) * XL + chi(c0, s, 0, 0, 1) * XU);
            else
                ChiX = 0.5 * (chi(lo, s) * prim(lo, 6 + NS + s) +
                              chi(up, s) * prim(up, 6 + NS + s));
            soret[s] = ChiX * (prim(c0, 4) - prim(cm, 4)) / h / rT;
        }
#pragma unroll
        for (int kk = 0; kk < NS; ++kk) {
            double f = 0.;
#pragma unroll
            for (int ll = 0; ll < NS; ++ll) {
                double Fks = half * (Dm(lo, ll * NS + kk) + Dm(up, ll * NS + kk)) * (dk[ll] + soret[ll]);
                f = f - Fks;
            }
            Fk[kk] = f;
        }
        double Q5 = 0.;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double hk = P.e0[s] + P.hcp[s] * meanT;
            double csum = (D == 2 && !wall) ? chi(c0, s) + chi(c0, s)  // flux.cpp:1604
                                            : chi(lo, s) + chi(up, s);
            double Q5s = (hk + 0.5 * P.Runiv * meanT * csum / P.M(s)) * Fk[s];
            Q5 = Q5 + Q5s;
        }
        o[nv + 3] = o[nv + 3] + Q5;
#pragma unroll
        for (int s = 0; s < NS; ++s) o[5 + s] = o[5 + s] + Fk[s];
    }
    if (wall && P.bcm[2 * D + (W.hi ? 1 : 0)] == 1) {  // BCWallSpeciesFlux
#pragma unroll
        for (int s = 0; s < NS; ++s) o[5 + s] = 0.;
        o[0] = 0.;
        o[nv + 3] = 0.;
    }
}

// The A/B noise of component comp of face (i,j,k) of direction D, and of node (i,j,k): N(0,1) times
// the component's scale, keyed by the wrapped index.
template <int D>
__device__ __forceinline__ void face_noise(const DevParams& P, const NoiseKey& K, int comp, int i, int j, int k,
                                           double& A, double& B)
{
    const int iw = (D == 0 && i == P.n[0]) ? 0 : i;
    const int jw = (D == 1 && j == P.n[1]) ? 0 : j;
    const int kw = (D == 2 && k == P.n[2]) ? 0 : k;
    uint32_t lin = (uint32_t)(((long)kw * P.n[1] + jw) * P.n[0] + iw);
    // in a wall direction face n is a face of its own, drawn from its own field
    const int c = (D == 0) ? i : (D == 1) ? j : k;
    const uint32_t wall_hi = (c == P.n[D] && !P.periodic[D]) ? 128u : 0u;
    const double scale = (comp <= 3) ? P.var_mom : (comp == 4) ? P.var_ener : P.var_mass;
    double za, zb;
    noise_ab(K, (uint32_t)(16 * D + comp) + wall_hi, lin, za, zb);
    A = za * scale;
    B = zb * scale;
}

__device__ __forceinline__ void node_noise(const DevParams& P, const NoiseKey& K, double scale, int i, int j, int k,
                                           double& A, double& B)
{
    const int iw = (i == P.n[0]) ? 0 : i, jw = (j == P.n[1]) ? 0 : j, kw = (k == P.n[2]) ? 0 : k;
    uint32_t lin = (uint32_t)(((long)kw * P.n[1] + jw) * P.n[0] + iw);
    // nodes on the hi plane of a wall direction are distinct: field NODE_FIELD + mask
    const uint32_t mask = ((i == P.n[0] && !P.periodic[0]) ? 1u : 0u) |
                          ((j == P.n[1] && !P.periodic[1]) ? 2u : 0u) |
                          ((k == P.n[2] && !P.periodic[2]) ? 4u : 0u);
    double za, zb;
    noise_ab(K, NODE_FIELD + mask, lin, za, zb);
    A = za * scale;
    B = zb * scale;
}

// ---- corner viscous terms at nodes (flux.cpp:1627-1713) ------------------------------------

__global__ void __launch_bounds__(BLK) k_corner_node(DevParams P, Arr prima, Arr etaa, Arr zetaa,
                                                     Arr cux, Arr cvx, Arr cwx, Arr cuy, Arr cvy,
                                                     Arr cwy, Arr cuz, Arr cvz, Arr cwz, Arr vcorn, Arr rancorn,
                                                     FaceNoise nz)
{
    const long t = xcd_thread();
    int i, j, k;
    if (!box_index(P, t, 1, 1, 1, i, j, k)) return;
    const Fld prim = fld_of(prima, prima), eta = fld_of(etaa, prima), zeta = fld_of(zetaa, prima);
    const unsigned cb = off_of(prima, i, j, k), nd0 = off_of(rancorn, i, j, k);
    const long nd8 = (long)(nd0 >> 3);
    double muxp = 0.125 * (eta(cb, 0, 0, -1, -1) + eta(cb, 0, -1, -1, -1) + eta(cb, 0, 0, 0, -1) +
                           eta(cb, 0, -1, 0, -1) + eta(cb, 0, 0, -1, 0) + eta(cb, 0, -1, -1, 0) + eta(cb, 0, 0, 0, 0) +
                           eta(cb, 0, -1, 0, 0));
    double zetaxp = 0.;
    if (P.visc_type == 3 || P.visc_type == -3)
        zetaxp = 0.125 * (zeta(cb, 0, 0, -1, -1) + zeta(cb, 0, -1, -1, -1) + zeta(cb, 0, 0, 0, -1) +
                          zeta(cb, 0, -1, 0, -1) + zeta(cb, 0, 0, -1, 0) + zeta(cb, 0, -1, -1, 0) + zeta(cb, 0, 0, 0, 0) +
                          zeta(cb, 0, -1, 0, 0));
    Rcp DXa[3] = {P.h(0), P.h(1), P.h(2)};
    constexpr Rcp twelve{12., 1. / 12.};
    if (P.any_wall) {
        // wall nodes (flux.cpp:1647-1682): half spacing across each wall met, viscosities from
        // the four ghost-layer cells of the last wall met (the checks run lo x .. hi z)
        const int nd[3] = {i, j, k};
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const int d = f >> 1, side = f & 1;
            if (!P.wall[f] || nd[d] != (side ? P.n[d] : 0)) continue;
            DXa[d] = Rcp{0.5 * P.dx[d], 2.0 * P.rdx[d]};
            const int a = (d == 0) ? 1 : 0, b = (d == 2) ? 1 : 2;
            double e4 = 0., z4 = 0.;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int c[3];
                c[d] = side ? nd[d] : nd[d] - 1;
                c[a] = nd[a] - 1 + (q >> 1);
                c[b] = nd[b] - 1 + (q & 1);
                const unsigned cw = off_of(prima, c[0], c[1], c[2]);
                e4 = (q == 0) ? eta(cw, 0) : e4 + eta(cw, 0);
                z4 = (q == 0) ? zeta(cw, 0) : z4 + zeta(cw, 0);
            }
            muxp = 0.25 * e4;
            zetaxp = (P.visc_type == 3 || P.visc_type == -3) ? 0.25 * z4 : 0.;
        }
    }
    const Rcp DX0 = DXa[0], DX1 = DXa[1], DX2 = DXa[2];
    // all values first, then the stores: a store in between would make the cells load again
    double gx[3], gy[3], gz[3], vc;
#pragma unroll
    for (int n = 1; n < 4; ++n) {
        gx[n - 1] = 0.25 * muxp *
                             (prim(cb, n, 0, -1, -1) - prim(cb, n, -1, -1, -1) + prim(cb, n, 0, 0, -1) -
                              prim(cb, n, -1, 0, -1) + prim(cb, n, 0, -1, 0) - prim(cb, n, -1, -1, 0) +
                              prim(cb, n, 0, 0, 0) - prim(cb, n, -1, 0, 0)) /
                             DX0;
        gy[n - 1] = 0.25 * muxp *
                             (prim(cb, n, -1, 0, -1) - prim(cb, n, -1, -1, -1) + prim(cb, n, 0, 0, -1) -
                              prim(cb, n, 0, -1, -1) + prim(cb, n, -1, 0, 0) - prim(cb, n, -1, -1, 0) +
                              prim(cb, n, 0, 0, 0) - prim(cb, n, 0, -1, 0)) /
                             DX1;
        gz[n - 1] = 0.25 * muxp *
                             (prim(cb, n, -1, -1, 0) - prim(cb, n, -1, -1, -1) + prim(cb, n, 0, -1, 0) -
                              prim(cb, n, 0, -1, -1) + prim(cb, n, -1, 0, 0) - prim(cb, n, -1, 0, -1) +
                              prim(cb, n, 0, 0, 0) - prim(cb, n, 0, 0, -1)) /
                             DX2;
    }
    vc =
        (muxp / twelve + zetaxp / 4.) *
        ((prim(cb, 1, 0, -1, -1) - prim(cb, 1, -1, -1, -1)) / DX0 +
         (prim(cb, 1, 0, 0, -1) - prim(cb, 1, -1, 0, -1)) / DX0 +
         (prim(cb, 1, 0, -1, 0) - prim(cb, 1, -1, -1, 0)) / DX0 + (prim(cb, 1, 0, 0, 0) - prim(cb, 1, -1, 0, 0)) / DX0 +
         (prim(cb, 2, -1, 0, -1) - prim(cb, 2, -1, -1, -1)) / DX1 +
         (prim(cb, 2, 0, 0, -1) - prim(cb, 2, 0, -1, -1)) / DX1 +
         (prim(cb, 2, -1, 0, 0) - prim(cb, 2, -1, -1, 0)) / DX1 + (prim(cb, 2, 0, 0, 0) - prim(cb, 2, 0, -1, 0)) / DX1 +
         (prim(cb, 3, -1, -1, 0) - prim(cb, 3, -1, -1, -1)) / DX2 +
         (prim(cb, 3, 0, -1, 0) - prim(cb, 3, 0, -1, -1)) / DX2 +
         (prim(cb, 3, -1, 0, 0) - prim(cb, 3, -1, 0, -1)) / DX2 + (prim(cb, 3, 0, 0, 0) - prim(cb, 3, 0, 0, -1)) / DX2);
    const Arr ax[3] = {cux, cvx, cwx}, ay[3] = {cuy, cvy, cwy}, az[3] = {cuz, cvz, cwz};
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        ax[n].p[nd8] = gx[n];
        ay[n].p[nd8] = gy[n];
        az[n].p[nd8] = gz[n];
    }
    vcorn.p[nd8] = vc;
    // the node's weighted noise
    if (nz.mode == kNoiseSets) {
        rancorn(i, j, k) = 1.0 * nz.rA(i, j, k) + nz.w * nz.rB(i, j, k);
    } else if (nz.mode == kNoisePhilox) {
        double A, B;
        node_noise(P, nz.K, P.var_mom, i, j, k, A, B);
        rancorn(i, j, k) = 1.0 * A + nz.w * B;
    }
}

// ---- corner-to-face terms (flux.cpp:1770-1980) -------------------------------------------
// Sums over the 4 nodes of a face: visccorn in (hi,hi),(lo,hi),(hi,lo),(lo,lo) transverse
// order on every face; the corner arrays in that order on x/y faces and in
// (hi,hi),(hi,lo),(lo,hi),(lo,lo) order on z faces.

// Transverse offsets of face direction D: the first transverse axis moves (AI, AJ, 0), the
// second (0, BJ, BK): x faces (y, z), y faces (x, z), z faces (x, y).
template <int D>
struct Transverse {
    static constexpr int AI = (D != 0), AJ = (D == 0), BJ = (D == 2), BK = (D != 2);
};

// Left-to-right sum of `a` over the 4 nodes of face (i,j,k), starting from `s0` unless
// `first`; zorder selects (hi,hi),(hi,lo),(lo,hi),(lo,lo) instead of (hi,hi),(lo,hi),(hi,lo),(lo,lo).
template <int D>
__device__ inline double node4(const Fld& a, unsigned nd, bool zorder, double s0 = 0., bool first = true)
{
    using T = Transverse<D>;
    const int oa[4] = {1, zorder ? 1 : 0, zorder ? 0 : 1, 0};
    const int ob[4] = {1, zorder ? 0 : 1, zorder ? 1 : 0, 0};
    double s = s0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        double v = a(nd, 0, oa[q] * T::AI, oa[q] * T::AJ + ob[q] * T::BJ, ob[q] * T::BK);
        s = (first && q == 0) ? v : s + v;
    }
    return s;
}

template <int NS, int D>
__device__ __forceinline__ void corner_part(const FaceView& V, double* o)
{
    const Fld& prim = V.prim;
    // corn[a][b]: derivative direction a, velocity component b (cornx/corny/cornz of flux.cpp)
    // x face: div pair (vy, wz), tangential (uy, uz); y: (ux, wz), (vx, vz); z: (vy, ux), (wx, wy)
    const Fld &c1 = D == 1 ? V.corn[0][0] : V.corn[1][1], &c2 = D == 2 ? V.corn[0][0] : V.corn[2][2];
    const Fld &ta1 = D == 0 ? V.corn[1][0] : V.corn[0][D], &ta2 = D == 2 ? V.corn[1][2] : V.corn[2][D];
    // velocity cells of the heating term: the two neighbours, or the wall-side cell twice
    // (flux.cpp:1791-1822: 0.5*x*u_wall equals 0.25*x*(u_wall + u_wall) exactly)
    const unsigned lo = V.lo, up = V.up;
    const int nv = NS + 5;
    const bool zo = (D == 2);
    double vc4 = node4<D>(V.visccorn, V.nd, false);
    double div8 = node4<D>(c1, V.nd, zo);
    div8 = node4<D>(c2, V.nd, zo, div8, false);
    double s1 = node4<D>(ta1, V.nd, zo);
    double s2 = node4<D>(ta2, V.nd, zo);
    constexpr int cn = 1 + D;
    constexpr int tc1 = (D == 0) ? 2 : 1, tc2 = (D == 2) ? 2 : 3;
    o[cn] = o[cn] - 0.25 * vc4;
    o[cn] = o[cn] + .25 * div8;
    o[tc1] = o[tc1] - .25 * s1;
    o[tc2] = o[tc2] - .25 * s2;
    double phiflx = 0.25 * (vc4 - div8) * (prim(lo, cn) + prim(up, cn));
    phiflx = phiflx + .25 * s1 * (prim(lo, tc1) + prim(up, tc1));
    phiflx = phiflx + .25 * s2 * (prim(lo, tc2) + prim(up, tc2));
    o[nv + 1] = o[nv + 1] - 0.5 * phiflx;
}

// ---- hyperbolic face flux (flux.cpp:2016-2372) ---------------------------------------------

template <int NS, int D, bool WALL>
__device__ __forceinline__ void hyp_part(const DevParams& P, const FaceView& V, const WallFace& W, double* o, int i,
                                         int j, int k)
{
    const Fld &cons = V.cons, &prim = V.prim;
    const unsigned c0 = V.c0;
    constexpr int ex = (D == 0), ey = (D == 1), ez = (D == 2);
    const int nv = NS + 5;
    const double wgt2 = 1. / 12.;
    const double wgt1 = 0.5 + wgt2;
    double cv[NS + 5], pv[NS + 6], Yk[NS];
    // walls: the wall face takes the wall-side cell (flux.cpp:2028-2037); with conserved
    // interpolation the next face in uses the one-sided weights of :1994-1997 (:2190-2206)
    const bool wall = WALL && W.any();
    const int c = (D == 0) ? i : (D == 1) ? j : k;
    const bool near_lo = WALL && c == 1 && P.wall[2 * D];
    const bool near_hi = WALL && c == P.n[D] - 1 && P.wall[2 * D + 1];
    if (P.advection_type == 1) {
#pragma unroll
        for (int l = 0; l < NS + 6; ++l)
            pv[l] = wall ? prim(V.up, l)
                            : wgt1 * (prim(c0, l) + prim(c0, l, -ex, -ey, -ez)) -
                                  wgt2 * (prim(c0, l, -2 * ex, -2 * ey, -2 * ez) + prim(c0, l, ex, ey, ez));
        double rho = pv[0];
        cv[0] = rho;
#pragma unroll
        for (int n = 0; n < NS; ++n) Yk[n] = pv[6 + n];
        double ie = eos_energy<NS>(P, Yk, pv[4]);
        double vsqr = pv[1] * pv[1] + pv[2] * pv[2] + pv[3] * pv[3];
        cv[4] = rho * ie + 0.5 * rho * vsqr;
#pragma unroll
        for (int n = 0; n < NS; ++n) cv[5 + n] = cv[0] * pv[6 + n];
    } else {
        const double wgta = -0.2, wgtb = 0.75, wgtc = 0.5, wgtd = -0.05;
#pragma unroll
        for (int l = 0; l < NS + 5; ++l) {
            const double cm2 = cons(c0, l, -2 * ex, -2 * ey, -2 * ez), cm1 = cons(c0, l, -ex, -ey, -ez);
            const double cc = cons(c0, l), cp1 = cons(c0, l, ex, ey, ez);
            if (WALL && W.lo) cv[l] = cm1;
            else if (WALL && W.hi) cv[l] = cc;
            else if (near_lo) cv[l] = wgta * cm2 + wgtb * cm1 + wgtc * cc + wgtd * cp1;
            else if (near_hi) cv[l] = wgta * cp1 + wgtb * cc + wgtc * cm1 + wgtd * cm2;
            else cv[l] = wgt1 * (cc + cm1) - wgt2 * (cm2 + cp1);
        }
        const Rcp rho = rcp_of(cv[0]);
#pragma unroll
        for (int l = 1; l < 4; ++l) pv[l] = cv[l] / rho;
#pragma unroll
        for (int n = 0; n < NS; ++n) Yk[n] = cv[5 + n] / rho;
        double vsqr = pv[1] * pv[1] + pv[2] * pv[2] + pv[3] * pv[3];
        double ie = cv[4] / rho - 0.5 * vsqr;
        pv[4] = eos_temperature<NS>(P, ie, Yk);
        pv[5] = eos_pressure<NS>(P, Yk, cv[0], pv[4]);
    }
    const double un = pv[1 + D];
    o[0] += cv[0] * un;
    if (D == 0) {
        o[1] += cv[0] * (pv[1] * pv[1]) + pv[5];
        o[2] += cv[0] * pv[1] * pv[2];
        o[3] += cv[0] * pv[1] * pv[3];
    } else if (D == 1) {
        o[1] += cv[0] * pv[1] * pv[2];
        o[2] += cv[0] * pv[2] * pv[2] + pv[5];
        o[3] += cv[0] * pv[3] * pv[2];
    } else {
        o[1] += cv[0] * pv[1] * pv[3];
        o[2] += cv[0] * pv[2] * pv[3];
        o[3] += cv[0] * pv[3] * pv[3] + pv[5];
    }
    o[4] += un * cv[4] + pv[5] * un;
    o[4] += o[nv] + o[nv + 1] + o[nv + 2] + o[nv + 3];
    if (P.algorithm_type == 2) {
        if (P.advection_type == 1) {
#pragma unroll
            for (int n = 0; n < NS; ++n) o[5 + n] += cv[0] * pv[6 + n] * un;
        } else {
#pragma unroll
            for (int n = 0; n < NS; ++n) o[5 + n] += cv[5 + n] * un;
        }
    }
}

// ---- stage combination (timeStep.cpp:158-201, 266-306, 370-413) ----------------------------

// src: the source MultiFab (null: zero, main_driver.cpp:241-242).  The conservedToPrimitive that
// follows reads this cell's new state only, so prim is formed here from registers.
template <int NS>
__global__ void __launch_bounds__(BLK) k_stage(DevParams P, Arr outa, Arr u0a, Arr usa, Arr fxa, Arr fya,
                                               Arr fza, Arr srca, Arr prima, double dt, int mode)
{
    const long t = xcd_thread();
    int i, j, k;
    if (!box_index(P, t, 0, 0, 0, i, j, k)) return;
    const Fld out = fld_of(outa, prima), u0 = fld_of(u0a, prima), us = fld_of(usa, prima), prim = fld_of(prima, prima),
              srcf = fld_of(srca, prima), fx = fld_of(fxa, fxa), fy = fld_of(fya, fya), fz = fld_of(fza, fza);
    const unsigned cb = off_of(prima, i, j, k), ox = off_of(fxa, i, j, k), oy = off_of(fya, i, j, k),
                   oz = off_of(fza, i, j, k);
    double o[NS + 5];
#pragma unroll
    for (int n = 0; n < NS + 5; ++n) {
        const double src = srcf.p ? srcf(cb, n) : 0.0;
        double div = (fx(ox, n, 1, 0, 0) - fx(ox, n)) / P.h(0) +
                     (fy(oy, n, 0, 1, 0) - fy(oy, n)) / P.h(1) +
                     (fz(oz, n, 0, 0, 1) - fz(oz, n)) / P.h(2);
        if (mode == 0) o[n] = us(cb, n) - dt * div + dt * src;
        else if (mode == 1) o[n] = 0.25 * (3.0 * u0(cb, n) + us(cb, n) - dt * div + dt * src);
        else o[n] = (2. / 3.) * (0.5 * u0(cb, n) + us(cb, n) - dt * div + dt * src);
    }
    const double* g = P.grav;
    double r0 = us(cb, 0), r1 = us(cb, 1), r2 = us(cb, 2), r3 = us(cb, 3);
    if (mode == 0) {
#pragma unroll
        for (int n = 0; n < 3; ++n) o[n + 1] += dt * r0 * g[n];
        o[4] += dt * (g[0] * r1 + g[1] * r2 + g[2] * r3);
    } else if (mode == 1) {
#pragma unroll
        for (int n = 0; n < 3; ++n) o[n + 1] += 0.25 * dt * r0 * g[n];
        o[4] += 0.25 * dt * (g[0] * r1 + g[1] * r2 + g[2] * r3);
    } else {
#pragma unroll
        for (int n = 0; n < 3; ++n) o[n + 1] += 2. / 3. * dt * r0 * g[n];
        o[4] += 2. / 3. * dt * (g[0] * r1 + g[1] * r2 + g[2] * r3);
    }
#pragma unroll
    for (int n = 0; n < NS + 5; ++n) out(cb, n) = o[n];
    double pr[2 * NS + 6];
    cons_to_prim_cell<NS>(P, o, pr);
#pragma unroll
    for (int n = 0; n < 2 * NS + 6; ++n) prim(cb, n) = pr[n];
}

// ---- chemistry source (chemistry_functions.cpp:128-193) ------------------------------------

template <int NS>
__global__ void __launch_bounds__(BLK) k_chem_source(DevParams P, Arr prim, Arr source, Arr ranchem, double dt,
                                                     double dV)
{
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    int i, j, k;
    if (!box_index(P, t, 0, 0, 0, i, j, k)) return;
    double X[NS], src[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) X[n] = prim(i, j, k, 6 + NS + n);
    chem_source_cell<NS>(P, prim(i, j, k, 4), prim(i, j, k, 5), X, [&](int m) { return ranchem(i, j, k, m); }, dt,
                         dV, src);
#pragma unroll
    for (int n = 0; n < NS; ++n) source(i, j, k, 5 + n) = src[n];
}

// Reaction noise sets A, B (MultiFabFillRandom(ranchem_A/B, m, 1.0), timeStep.cpp:93-97).
__global__ void __launch_bounds__(BLK) k_chem_noise(DevParams P, NoiseKey K, Arr A, Arr B)
{
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    int i, j, k;
    if (!box_index(P, t, 0, 0, 0, i, j, k)) return;
    const uint32_t lin = (uint32_t)(((long)k * P.n[1] + j) * P.n[0] + i);
    for (int m = 0; m < P.chem.nreaction; ++m) {
        double za, zb;
        noise_ab(K, CHEM_FIELD + (uint32_t)m, lin, za, zb);
        A(i, j, k, m) = za;
        B(i, j, k, m) = zb;
    }
}

// ---- noise --------------------------------------------------------------------------------

// dst = 1*A + w*B (MultiFab::LinComb), components below c0 zeroed.
__global__ void __launch_bounds__(BLK) k_lincomb(double* dst, const double* a, const double* b, long npts,
                                                 int nc, int c0, double w)
{
    long t = (long)blockIdx.x * BLK + threadIdx.x;
    if (t >= npts) return;
    for (int n = 0; n < nc; ++n) {
        long q = t + (long)n * npts;
        dst[q] = (n < c0) ? 0.0 : 1.0 * a[q] + w * b[q];
    }
}

// Fills every component of direction D's face noise for sets A and B: component 0 (density)
// is zero (timeStep.cpp:74-76 skips it), components 1..nvars-1 are N(0,1) * their scale.
template <int D>
__device__ __forceinline__ void noise_face_body(const DevParams& P, const NoiseKey& K, Arr A, Arr B, long t)
{
    int i, j, k;
    if (!box_index(P, t, D == 0, D == 1, D == 2, i, j, k)) return;
    A(i, j, k, 0) = 0.0;
    B(i, j, k, 0) = 0.0;
    for (int comp = 1; comp < P.nvars; ++comp) {
        double a, b;
        face_noise<D>(P, K, comp, i, j, k, a, b);
        A(i, j, k, comp) = a;
        B(i, j, k, comp) = b;
    }
}

__device__ __forceinline__ void noise_node_body(const DevParams& P, const NoiseKey& K, Arr A, Arr B, double scale,
                                                long t)
{
    int i, j, k;
    if (!box_index(P, t, 1, 1, 1, i, j, k)) return;
    double a, b;
    node_noise(P, K, scale, i, j, k, a, b);
    A(i, j, k) = a;
    B(i, j, k) = b;
}

// One launch for a step's whole noise set (blockIdx.y: face direction 0..2, 3 = nodes); every
// value is drawn by the same body and key as in a launch of its own.
__global__ void __launch_bounds__(BLK) k_noise_all(DevParams P, NoiseKey K, Arr A0, Arr B0, Arr A1, Arr B1,
                                                   Arr A2, Arr B2, Arr rA, Arr rB)
{
    const long t = (long)blockIdx.x * BLK + threadIdx.x;
    switch (blockIdx.y) {
        case 0: noise_face_body<0>(P, K, A0, B0, t); break;
        case 1: noise_face_body<1>(P, K, A1, B1, t); break;
        case 2: noise_face_body<2>(P, K, A2, B2, t); break;
        default: noise_node_body(P, K, rA, rB, P.var_mom, t); break;
    }
}

// ---- calculateFlux's face passes in one launch -----------------------------------------------
//
// The stochastic, diffusive, corner and hyperbolic terms of a face only add to that face's flux, so one
// thread forms all of them in registers, in the reference's order, and the flux is written once
// and never read back (four passes read and wrote its nvars + 4 components through memory, and read
// the same cells four times).  The noise of a step that draws its own is evaluated in place, with
// the bits fhdx_fill_noise gives, instead of being written once and read in each of the three stages.
// Until the last stage of a whole step nobody sees the weighted noise and the four energy
// components, and they are not stored (F.keep).  Consecutive work items are the three
// directions of one chunk of faces, so they find each other's cells in L2.
// Argon 128^3: the four passes took 1614 us a stage and the noise 269 us a step; this takes 677 us.
// RT_3d deck (64x32x32, four species): 85 us a stage before, 54 us now.

template <int NS, int D, bool WALL>
__device__ __forceinline__ void flux_body(const DevParams& P, const FluxArgs& F, double volinv, double dtinv, long t)
{
    int i, j, k;
    if (!box_index(P, t, D == 0, D == 1, D == 2, i, j, k)) return;
    const WallFace W = WALL ? wall_face<D>(P, i, j, k) : WallFace{false, false, 0, 0, 0};
    const Arr& cell = F.prim;
    FaceView V;
    V.cons = fld_of(F.cons, cell);
    V.prim = fld_of(F.prim, cell);
    V.eta = fld_of(F.eta, cell);
    V.zeta = fld_of(F.zeta, cell);
    V.kappa = fld_of(F.kappa, cell);
    V.chi = fld_of(F.chi, cell);
    V.Dm = fld_of(F.D, cell);
    V.visccorn = fld_of(F.visccorn, F.rancorn);
    V.rancorn = fld_of(F.rancorn, F.rancorn);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) V.corn[a][b] = fld_of(F.corn[a][b], F.rancorn);
    V.c0 = off_of(cell, i, j, k);
    V.cm = off_of(cell, i - (D == 0), j - (D == 1), k - (D == 2));
    V.lo = V.cm;
    V.up = V.c0;
    if (WALL && W.any()) V.lo = V.up = off_of(cell, W.wi, W.wj, W.wk);
    V.nd = off_of(F.rancorn, i, j, k);
    double edges = 0.;
    if (kEdgesFirst<NS, WALL> && P.stoch_on) edges = edge_sum<D, WALL>(P, V, W.any(), i, j, k);
    double ran[NS + 5], o[NS + 9];
    ran[0] = 0.0;
    const unsigned fo = off_of(F.flux[D], i, j, k);
    const Fld flux = fld_of(F.flux[D], F.flux[D]), rn = fld_of(F.ran[D], F.flux[D]);
    if (F.noise.mode == kNoisePhilox) {
#pragma unroll
        for (int c = 1; c < NS + 5; ++c) {
            double A, B;
            face_noise<D>(P, F.noise.K, c, i, j, k, A, B);
            ran[c] = 1.0 * A + F.noise.w * B;
        }
    } else if (F.noise.mode == kNoiseSets) {
        const Fld A = fld_of(F.noise.A[D], F.flux[D]), B = fld_of(F.noise.B[D], F.flux[D]);
#pragma unroll
        for (int c = 1; c < NS + 5; ++c) ran[c] = 1.0 * A(fo, c) + F.noise.w * B(fo, c);
    } else {
#pragma unroll
        for (int c = 1; c < NS + 5; ++c) ran[c] = rn(fo, c);
    }
    if (F.noise.mode != kNoiseWeighted && F.keep)
#pragma unroll
        for (int c = 0; c < NS + 5; ++c) rn(fo, c) = ran[c];
#pragma unroll
    for (int c = 0; c < NS + 9; ++c) o[c] = 0.0;
    if (P.stoch_on) stoch_part<NS, D, WALL>(P, V, WALL && W.any(), edges, ran, o, volinv, dtinv, F.dt, i, j, k);
    diff_part<NS, D, WALL>(P, V, W, o);
    corner_part<NS, D>(V, o);
    if (P.advection_type == 1 || P.advection_type == 2) hyp_part<NS, D, WALL>(P, V, W, o, i, j, k);
#pragma unroll
    for (int c = 0; c < NS + 5; ++c) flux(fo, c) = o[c];
    if (F.keep)
#pragma unroll
        for (int c = NS + 5; c < NS + 9; ++c) flux(fo, c) = o[c];
}

// The arguments are one struct, read anew in each direction's branch, as k_faces does.  Taken as they
// come, the compiler loads those of all three branches at once (147 to 269 scalar registers spilled to vector
// lanes, 6 to 88 so), and at five and more species with walls it copied the parameters, 1960 bytes a lane, to
// scratch: 48^3 with walls, five species 994 us a step, 649 so (796 in four passes); eight 1888 and 1258 (1810).
struct FluxKernel {
    DevParams P;
    FluxArgs F;
    double volinv, dtinv;
};

__device__ __forceinline__ const FluxKernel& flux_args()
{
    typedef const FluxKernel __attribute__((address_space(4))) * Ptr;
    Ptr p = (Ptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm("" : "+s"(p));
    return *(const FluxKernel*)p;
}

template <int NS, int D, bool WALL>
__device__ __forceinline__ void flux_item(long t)
{
    const FluxKernel& A = flux_args();
    flux_body<NS, D, WALL>(A.P, A.F, A.volinv, A.dtinv, t);
}

template <int NS, bool WALL>
__global__ void __launch_bounds__(BLK) k_flux(FluxKernel A)
{
    const unsigned item = xcd_block(blockIdx.x, gridDim.x), chunk = item / 3, d = item - 3 * chunk;
    const long t = (long)chunk * BLK + threadIdx.x;
    if (d == 0) flux_item<NS, 0, WALL>(t);
    else if (d == 1) flux_item<NS, 1, WALL>(t);
    else flux_item<NS, 2, WALL>(t);
}

// ---- host launchers ---------------------------------------------------------------------

#define NS_DISPATCH(NSV, CALL)                          \
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

// counts over the launch box (cells, faces of direction d, nodes, cells grown by ngc)
static long ncell(const DevParams& P) { return (long)P.bn[0] * P.bn[1] * P.bn[2]; }
static long nface(const DevParams& P, int d)
{
    return (long)(P.bn[0] + (d == 0)) * (P.bn[1] + (d == 1)) * (P.bn[2] + (d == 2));
}
static long nnode(const DevParams& P) { return (long)(P.bn[0] + 1) * (P.bn[1] + 1) * (P.bn[2] + 1); }
static long ngrown(const DevParams& P)
{
    const int g = P.ngc;
    return (long)(P.bn[0] + 2 * g) * (P.bn[1] + 2 * g) * (P.bn[2] + 2 * g);
}

int ref_c2p(const DevParams& P, Arr prim, Arr cons, hipStream_t s)
{
    NS_DISPATCH(P.ns, (k_c2p<NS><<<grid_for(ncell(P), BLK), BLK, 0, s>>>(P, prim, cons)));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_transport(const DevParams& P, Arr prim, Arr eta, Arr zeta, Arr kappa, Arr chi, Arr Dm,
                  int* err, hipStream_t s)
{
    if (P.transport_type == 2) {
        NS_DISPATCH(P.ns, (k_transport<NS, true><<<grid_for(ngrown(P), BLK), BLK, 0, s>>>(
                              P, prim, eta, zeta, kappa, chi, Dm, err)));
    } else {
        NS_DISPATCH(P.ns, (k_transport<NS, false><<<grid_for(ngrown(P), BLK), BLK, 0, s>>>(
                              P, prim, eta, zeta, kappa, chi, Dm, err)));
    }
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_fill_boundary(const DevParams& P, Arr a, int nc, hipStream_t s)
{
    k_fill_boundary<<<grid_for(ngrown(P), BLK), BLK, 0, s>>>(P, a, nc);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_set_bc(const DevParams& P, Arr prim, Arr cons, hipStream_t s)
{
    if (!P.any_wall) return FHDX_OK;
    const int g = P.ngc;
    for (int d = 0; d < 3; ++d) {
        if (P.periodic[d]) continue;
        long slab = 2L * g;
        for (int e = 0; e < 3; ++e)
            if (e != d) slab *= P.bn[e] + 2 * g;
        NS_DISPATCH(P.ns, (k_set_bc<NS><<<grid_for(slab, BLK), BLK, 0, s>>>(P, prim, cons, d)));
    }
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_ghosts(const DevParams& P, Arr prim, Arr cons, hipStream_t s)
{
    NS_DISPATCH(P.ns, (k_ghosts<NS><<<grid_for(ngrown(P) - ncell(P), BLK), BLK, 0, s>>>(P, prim, cons)));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int fill_value(double* p, long n, double v, hipStream_t s)
{
    if (n <= 0) return FHDX_OK;
    k_fill<<<grid_for(n, BLK), BLK, 0, s>>>(p, n, v);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

template <int NS>
static void flux_passes(const DevParams& P, const FluxArgs& a, hipStream_t s)
{
    const double volinv = 1. / (P.dx[0] * P.dx[1] * P.dx[2]);
    const double dtinv = 1. / a.dt;
    const Arr(&c)[3][3] = a.corn;
    k_corner_node<<<grid_for(nnode(P), BLK), BLK, 0, s>>>(P, a.prim, a.eta, a.zeta, c[0][0], c[0][1], c[0][2],
                                                          c[1][0], c[1][1], c[1][2], c[2][0], c[2][1], c[2][2],
                                                          a.visccorn, a.rancorn, a.noise);
    long mf = nface(P, 0);
    for (int d = 1; d < 3; ++d) mf = nface(P, d) > mf ? nface(P, d) : mf;
    const unsigned grid = 3 * grid_for(mf, BLK);  // every body checks its own direction's face count
    if (P.any_wall) k_flux<NS, true><<<grid, BLK, 0, s>>>(FluxKernel{P, a, volinv, dtinv});
    else k_flux<NS, false><<<grid, BLK, 0, s>>>(FluxKernel{P, a, volinv, dtinv});
}

int ref_calculate_flux(const DevParams& P, const FluxArgs& a, int flux_ncomp[3], hipStream_t s)
{
    const int nc = P.nvars + 4;
    for (int d = 0; d < 3; ++d) {
        // flux_in.setVal(0) (flux.cpp:24-26): the face pass writes all nvars + 4 components itself;
        // any further ones are zeroed
        if (flux_ncomp[d] == nc) continue;
        int r = fill_value(a.flux[d].p + a.flux[d].sn * nc, a.flux[d].sn * (flux_ncomp[d] - nc), 0.0, s);
        if (r) return r;
    }
    NS_DISPATCH(P.ns, flux_passes<NS>(P, a, s));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_stage(const DevParams& P, Arr out, Arr u0, Arr us, const Arr flux[3], Arr source, Arr prim, double dt,
              int mode, hipStream_t s)
{
    NS_DISPATCH(P.ns, (k_stage<NS><<<grid_for(ncell(P), BLK), BLK, 0, s>>>(P, out, u0, us, flux[0], flux[1],
                                                                             flux[2], source, prim, dt, mode)));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_chem_source(const DevParams& P, Arr prim, Arr source, Arr ranchem, double dt, hipStream_t s)
{
    const double dV = P.dx[0] * P.dx[1] * P.dx[2];
    NS_DISPATCH(P.ns, (k_chem_source<NS><<<grid_for(ncell(P), BLK), BLK, 0, s>>>(P, prim, source, ranchem, dt,
                                                                                   dV)));
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_fill_chem_noise(const DevParams& P, const NoiseKey& K, Arr A, Arr B, hipStream_t s)
{
    k_chem_noise<<<grid_for(ncell(P), BLK), BLK, 0, s>>>(P, K, A, B);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_lincomb(double* dst, const double* a, const double* b, long npts, int nc, int c0, double w,
                hipStream_t s)
{
    k_lincomb<<<grid_for(npts, BLK), BLK, 0, s>>>(dst, a, b, npts, nc, c0, w);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

int ref_fill_noise(const DevParams& P, const NoiseKey& K, const Arr A[3], const Arr B[3], Arr rA, Arr rB,
                   hipStream_t s)
{
    long mx = nnode(P);                       // the node box is the largest; each body checks its own
    for (int d = 0; d < 3; ++d) mx = nface(P, d) > mx ? nface(P, d) : mx;
    k_noise_all<<<dim3(grid_for(mx, BLK), 4), BLK, 0, s>>>(P, K, A[0], B[0], A[1], B[1], A[2], B[2], rA, rB);
    FHDX_HIP_TRY(hipGetLastError());
    return FHDX_OK;
}

}  // namespace fhdx
