// kernels.hpp -- host launchers of the device kernels (ref_kernels.hip, fused_kernels.hip).
#pragma once

#include "common.hpp"

namespace fhdx {

// The noise of a calculateFlux call: ran[] and rancorn hold it weighted already (calculateFlux's
// own arguments), or it is A + w B of a stage, from the caller's sets or drawn in place from key K.  In
// the last two cases the kernels store the weighted noise into rancorn (the faces read it there)
// and, with keep, ran[], as the reference's MultiFab::LinComb leaves them (timeStep.cpp:99-107).
constexpr int kNoiseWeighted = 0, kNoiseSets = 1, kNoisePhilox = 2;

struct FaceNoise {
    int mode = kNoiseWeighted;
    Arr A[3], B[3], rA, rB;
    NoiseKey K{};
    double w = 0.;
};

// Views of every array calculateFlux touches (flux.cpp:4-16).
struct FluxArgs {
    Arr cons, prim, eta, zeta, kappa, chi, D;
    Arr flux[3], ran[3];
    Arr corn[3][3];  // [derivative direction][velocity component]: cornx/corny/cornz
    Arr visccorn, rancorn;
    double dt;
    FaceNoise noise;
    bool keep = true;  // also store ran[] and the flux components past nvars, which no later pass reads
};

int ref_c2p(const DevParams& P, Arr prim, Arr cons, hipStream_t s);
int ref_transport(const DevParams& P, Arr prim, Arr eta, Arr zeta, Arr kappa, Arr chi, Arr Dm, int* err,
                  hipStream_t s);
int ref_fill_boundary(const DevParams& P, Arr a, int nc, hipStream_t s);
// setBC: the ghost cells outside walls, faces lo x .. hi z in turn (no-op when periodic).
int ref_set_bc(const DevParams& P, Arr prim, Arr cons, hipStream_t s);
// Every ghost cell of a whole-domain state and its prim: FillBoundary of both, then setBC.
int ref_ghosts(const DevParams& P, Arr prim, Arr cons, hipStream_t s);
int fill_value(double* p, long n, double v, hipStream_t s);
// flux_ncomp: the components of each flux FAB (>= nvars + 4)
int ref_calculate_flux(const DevParams& P, const FluxArgs& a, int flux_ncomp[3], hipStream_t s);
// The stage combination and conservedToPrimitive of its result on the valid cells; source: the source
// MultiFab (p == nullptr: zero).
int ref_stage(const DevParams& P, Arr out, Arr u0, Arr us, const Arr flux[3], Arr source, Arr prim, double dt,
              int mode, hipStream_t s);
// compute_compressible_chemistry_source_CLE over the valid cells; reaction noise sets A, B.
int ref_chem_source(const DevParams& P, Arr prim, Arr source, Arr ranchem, double dt, hipStream_t s);
int ref_fill_chem_noise(const DevParams& P, const NoiseKey& K, Arr A, Arr B, hipStream_t s);
int ref_lincomb(double* dst, const double* a, const double* b, long npts, int nc, int c0, double w,
                hipStream_t s);
int ref_fill_noise(const DevParams& P, const NoiseKey& K, const Arr A[3], const Arr B[3], Arr rA, Arr rB,
                   hipStream_t s);

// evaluateStats passes (stats.hip).  yz: n0*19 doubles, part: nparts*n0*19, misc: 20 (device).
struct StatsArgs {
    Arr cu, cm, cv, prim, pm, pv, sc, ms;
    double *yz, *part, *misc;
    int nparts, steps, cross_cell;
};
int stats_launch(const DevParams& P, const StatsArgs& a, hipStream_t s);

}  // namespace fhdx
