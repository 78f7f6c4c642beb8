// Internal launch interface between the C ABI (capi.cpp) and the kernel
// translation units. Every launcher checks its shapes against what the
// kernel's grid assumes before launching and returns the HIP status.
#pragma once

#include <hip/hip_runtime.h>

#include "device/layout.hpp"
#include "device/form_f64.hpp"
#include "device/form_f32c.hpp"
#include "device/ghost_dt.hpp"
#include "device/stage_core.hpp"
#include "device/stage3d.hpp"
#include "device/tracer.hpp"
#include "device/lte_eos.hpp"
#include "device/lte_table.hpp"

namespace mh {

struct Schemes {
    Reconstruction recon;
    SlopeLimiter limiter;
    RiemannSolver solver;
    TimeStepScheme stepper;
};

constexpr int kSimds = 1024;  // of the chip: 256 CUs of four

// Number of marches that `rows` rows (or planes) are split into when `units`
// wavefronts run side by side for each. A wavefront costs its rows plus a
// prologue of `prologue` rows' worth, so fewer and longer marches do less
// work, but the chip has 1024 SIMDs to keep busy, equally. Candidates put k
// wavefronts on every SIMD (as many marches as fit k * 1024 wavefronts, one
// row each at least). Their time: the wavefronts of the fullest SIMD, in
// rounds of as many as reside there (2 in FP64, 4 in FP32C), times a
// wavefront's rows, times what a row takes with so many neighbours
// (wavefronts that share a SIMD hide each other's latency: a lone FP32C row
// takes 1.9 times its share of a full SIMD), plus a quarter of a wavefront
// for the last round's uneven end.
// (Those are the WENO5-Z + HLLC marches' counts. Schemes that need fewer
// registers hold more, the FP32C general instances three; over FOG to WENO5-Z,
// every solver, both forms, 2-D and 3-D from 62^3 and 70x50 up, none is slower
// than with the fixed minimum, but for 1 to 2 % of 186^3 in FP32C.)
// Measured, WENO5-Z + HLLC, with every split from k = 1/2 to 16 on 256^2 to 4096^2 and 64^3
// to 256^3: the pick is within 3 % of the best split, and against a fixed
// minimum of 8 rows the WENO5-Z stage at 256^2 went from 42 to 18 us (FP64)
// and 28 to 14 us (FP32C), at 512^2 from 44 to 32 and 31 to 21 us, at 1024^2
// from 99 to 78 and 49 to 40 us; 2048^2 and up are unchanged to 1 %.
inline int split_marches(int64_t units, int rows, double prologue, bool fp64) {
    const int resident = fp64 ? 2 : 4;
    const double share64[] = {0.0, 1.18, 2.08}, share32[] = {0.0, 1.9, 2.4, 3.15, 4.0};  // of 1, 2, .. wavefronts
    const double* share = fp64 ? share64 : share32;
    int best = 1;
    double least = 0.0;
    for (int k = 1; k <= 16; ++k) {
        const int64_t fit = (int64_t)k * kSimds / units;
        const int n = (int)(fit < 1 ? 1 : fit < rows ? fit : rows);
        const int64_t per_simd = (n * units + kSimds - 1) / kSimds;
        const double rounds = (double)(per_simd / resident) * share[resident] + share[per_simd % resident];
        const double t = (rounds + 0.25) * ((double)rows / n + prologue);
        if (k == 1 || t < least) {
            least = t;
            best = n;
        }
    }
    return best;
}

// 2-D fused stage over the interior, one wavefront per (strip, span).
hipError_t launch_stage2d_f64(const Schemes& s, const StageGrid& g, const FormF64::Ptrs& p, hipStream_t st);
hipError_t launch_stage2d_f32c(const Schemes& s, const StageGrid& g, const FormF32c::Ptrs& p, hipStream_t st);
// 3-D stage: the z sweep into `dz` (NV values per cell, [var][k][j][i]),
// then the x-y march of every interior plane (g.zc, g.nz set).
hipError_t launch_stage3d_f64(const Schemes& s, const StageGrid& g, const FormF64::Ptrs& p, double* dz,
                              hipStream_t st);
hipError_t launch_stage3d_f32c(const Schemes& s, const StageGrid& g, const FormF32c::Ptrs& p, float* dz,
                               hipStream_t st);
// 1-D stage over one row of xc cells (ng ghosts each side); virt: ghosts read
// from their sources, faces: ghost_faces of the ends.
hipError_t launch_stage1d_f64(const Schemes& s, int kind, int reduce_dt, int xc, int ng, const FormF64::Ptrs& p,
                              hipStream_t st, int virt = 0, int32_t faces = 0);
hipError_t launch_stage1d_f32c(const Schemes& s, int kind, int reduce_dt, int xc, int ng, const FormF32c::Ptrs& p,
                               hipStream_t st, int virt = 0, int32_t faces = 0);

// Tracer planes of a 2-D stage (p.frx / p.fry hold the stage's density fluxes).
hipError_t launch_tracer_f64(const Schemes& s, const TracerGrid& g, const FormF64::Ptrs& p, hipStream_t st);
hipError_t launch_tracer_f32c(const Schemes& s, const TracerGrid& g, const FormF32c::Ptrs& p, hipStream_t st);
hipError_t launch_tracer_ghost_f64(const GhostGrid& g, int ntr, FormF64::Planes in, FormF64::Planes out,
                                   hipStream_t st);
hipError_t launch_tracer_ghost_f32c(const GhostGrid& g, int ntr, FormF32c::Planes in, FormF32c::Planes out,
                                    hipStream_t st);

hipError_t launch_ghost_f64(int nd, const GhostGrid& g, FormF64::Planes in, FormF64::Planes out,
                            unsigned long long* amax, hipStream_t st);
hipError_t launch_ghost_f32c(int nd, const GhostGrid& g, FormF32c::Planes in, FormF32c::Planes out,
                             unsigned long long* amax, hipStream_t st);
// 3-D ghost fill of one buffer (x, y, z passes), folding the ghost cells
// into the CFL max when g.reduce_dt is set.
hipError_t launch_ghost3d_f64(const Ghost3Grid& g, FormF64::Planes q, unsigned long long* amax, hipStream_t st);
hipError_t launch_ghost3d_f32c(const Ghost3Grid& g, FormF32c::Planes q, unsigned long long* amax, hipStream_t st);
hipError_t launch_cfl_f64(int nd, FormF64::Planes q, int ncells, double gamma, unsigned long long* amax,
                          hipStream_t st);
hipError_t launch_cfl_f32c(int nd, FormF32c::Planes q, int ncells, double gamma, unsigned long long* amax,
                           hipStream_t st);

// Analytic LTE EOS fields (ionisation fraction, temperature) of every cell.
hipError_t launch_lte_eos_f64(int nd, FormF64::Planes q, int ncells, const LteParams& p, double* y, double* T,
                              int* flipped, hipStream_t st);
hipError_t launch_lte_eos_f32c(int nd, FormF32c::Planes q, int ncells, const LteParams& p, double* y, double* T,
                               int* flipped, hipStream_t st);

// Tabulated LTE EOS update_eos over every cell of `in` into `out` (same
// buffer, or a copy of all nvar planes with E updated).
hipError_t launch_tab_eos_f64(int nd, FormF64::Planes in, FormF64::Planes out, int ncells, int nvar,
                              const TabParams& t, const double* ytab, const double* ltab, double* y_space,
                              double* T_space, int* neg, hipStream_t st);
hipError_t launch_tab_eos_f32c(int nd, FormF32c::Planes in, FormF32c::Planes out, int ncells, int nvar,
                               const TabParams& t, const double* ytab, const double* ltab, double* y_space,
                               double* T_space, int* neg, hipStream_t st);

hipError_t launch_clock_finalize(Clock* c, int advance, hipStream_t st);
hipError_t launch_clock_set_dt(Clock* c, double dt, hipStream_t st);
hipError_t launch_clock_reset_max(Clock* c, hipStream_t st);
// The clock's fields from the host (and its CFL slots cleared, with reset);
// those and the step size they and the slots give, also into pinned host
// memory; the clock into pinned host memory.
hipError_t launch_clock_start(Clock* c, const Clock& fields, int reset, hipStream_t st);
hipError_t launch_clock_dt(Clock* c, const Clock& fields, double* host_dt, hipStream_t st);
hipError_t launch_clock_read(const Clock* c, Clock* host, hipStream_t st);

// Conversions between the FP64 layout and the compensated hi/lo planes.
hipError_t launch_split_f64_to_f32c(const double* src, FormF32c::Planes dst, int n, hipStream_t st);
hipError_t launch_join_f32c_to_f64(FormF32c::Planes src, double* dst, int n, hipStream_t st);

// Functor probes for the unit tests: run the device functors on n inputs.
hipError_t launch_probe_reconstruct(int recon, int limiter, int prec, int n, const double* stencils, double* wl,
                                    double* wr, hipStream_t st);
hipError_t launch_probe_riemann(int solver, int axis, int nd, int prec, double gamma, int n, const double* wl,
                                const double* wr, double* flux, hipStream_t st);
hipError_t launch_probe_math(int op, int n, const double* a, const double* b, double* out, hipStream_t st);

}  // namespace mh
