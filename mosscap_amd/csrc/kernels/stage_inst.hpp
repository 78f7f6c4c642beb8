// Kernel entry points and scheme dispatch for the fused stages, instantiated
// once per state form (stage_f64.hip, stage_f32c.hip).
#pragma once

#include "../launch.hpp"
#include "../device/tracer.hpp"

// Occupancy targets of the fused stage (waves per SIMD the register allocator
// must allow); each form's translation unit sets its own values, which may
// depend on the instance's scheme (R, RS).
#ifndef MH_STAGE_WAVES_PER_EU
#define MH_STAGE_WAVES_PER_EU 1
#endif
// ... of the instance with the gravity source and tracer stores (and, where
// MH_STAGE_WAVES_LONE is set, of its WENO5-Z + HLLC scheme in launches of no
// more wavefronts than SIMDs)
#ifndef MH_STAGE_WAVES_EXTRAS
#define MH_STAGE_WAVES_EXTRAS MH_STAGE_WAVES_PER_EU
#endif
// ... and of the plain instance with the positivity floors
#ifndef MH_STAGE_WAVES_FLOORS
#define MH_STAGE_WAVES_FLOORS MH_STAGE_WAVES_PER_EU
#endif

namespace mh {

template <Reconstruction R, RiemannSolver RS>
constexpr int stage_waves(int inst) {
    return inst == kStageExtras ? MH_STAGE_WAVES_EXTRAS
                                : inst == kStageFloors ? MH_STAGE_WAVES_FLOORS : MH_STAGE_WAVES_PER_EU;
}

template <class Form, Reconstruction R, SlopeLimiter SL, RiemannSolver RS, int Inst, bool Copies,
          int Waves = stage_waves<R, RS>(Inst)>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(Waves)))
void stage2d_kernel(StageGrid g, typename Form::Ptrs p) {
    stage2d_march<Form, R, SL, RS, 2, Inst, Copies>(g, p);
}

struct Stage1dGrid {
    int32_t xc, ng, nx, kind, reduce_dt;
    int32_t virt, faces;  // ghosts read from their sources (StageGrid::virt, ghost_faces of the ends)
};

template <class Form, Reconstruction R, SlopeLimiter SL, RiemannSolver RS>
__global__ __launch_bounds__(64) void stage1d_kernel(Stage1dGrid g, typename Form::Ptrs p) {
    using T = typename Form::real;
    constexpr int ORD = stencil_order(R);
    __shared__ T lds[3 * (kWave + 2 * ORD)];
    const int i0 = g.ng + (int)blockIdx.x * kStripOut;
    const T dt = (T)p.dt[0];
    const T dtdx = dt / (T)p.dx;
    double amax = 0.0;
    unsigned int hits = 0;
    stage1d_segment<Form, R, SL, RS>(p, g.kind, g.reduce_dt, 0, g.xc, g.ng, g.nx, i0, dtdx, dt, lds, amax, hits,
                                     Form::kVirtualGhosts ? g.virt : 0, g.faces);
    if (g.reduce_dt) {
        const uint64_t m = wave_max_u64(__builtin_bit_cast(uint64_t, amax));
        if (threadIdx.x == 0) atomicMax(p.amax_bits, (unsigned long long)m);
    }
    if (p.floor_hits != nullptr) {
        const unsigned int total = wave_sum_u32(hits);
        if (threadIdx.x == 0 && total != 0u) atomicAdd(p.floor_hits, total);
    }
}

template <class Form>
using Stage2dFn = void (*)(StageGrid, typename Form::Ptrs);
template <class Form>
using Stage1dFn = void (*)(Stage1dGrid, typename Form::Ptrs);

template <class Form, Reconstruction R, SlopeLimiter SL>
struct SolverPick {
    template <int Inst, bool Copies>
    static Stage2dFn<Form> two(RiemannSolver rs) {
        switch (rs) {
            case RiemannSolver::Rusanov: return stage2d_kernel<Form, R, SL, RiemannSolver::Rusanov, Inst, Copies>;
            case RiemannSolver::Hll: return stage2d_kernel<Form, R, SL, RiemannSolver::Hll, Inst, Copies>;
            default: return stage2d_kernel<Form, R, SL, RiemannSolver::Hllc, Inst, Copies>;
        }
    }
#ifdef MH_STAGE_WAVES_LONE
    // the general WENO5-Z + HLLC instance for wavefronts that have a SIMD each
    template <bool Copies>
    static Stage2dFn<Form> lone() {
        return stage2d_kernel<Form, R, SL, RiemannSolver::Hllc, kStageExtras, Copies, MH_STAGE_WAVES_LONE>;
    }
#endif
    static Stage1dFn<Form> one(RiemannSolver rs) {
        switch (rs) {
            case RiemannSolver::Rusanov: return stage1d_kernel<Form, R, SL, RiemannSolver::Rusanov>;
            case RiemannSolver::Hll: return stage1d_kernel<Form, R, SL, RiemannSolver::Hll>;
            default: return stage1d_kernel<Form, R, SL, RiemannSolver::Hllc>;
        }
    }
};

// (reconstruction, limiter) -> instance; FOG and WENO5-Z ignore the limiter
// (is_limiter_agnostic, Reconstruct.hpp:34-45).
template <class Form, class Pick>
auto pick_scheme(const Schemes& s, Pick pick) {
    using SL = SlopeLimiter;
    using RC = Reconstruction;
    switch (s.recon) {
        case RC::Fog: return pick.template operator()<RC::Fog, SL::MonotonizedCentral>();
        case RC::Weno5Z: return pick.template operator()<RC::Weno5Z, SL::MonotonizedCentral>();
        case RC::Muscl:
            if (s.limiter == SL::VanLeer) return pick.template operator()<RC::Muscl, SL::VanLeer>();
            if (s.limiter == SL::Minmod) return pick.template operator()<RC::Muscl, SL::Minmod>();
            return pick.template operator()<RC::Muscl, SL::MonotonizedCentral>();
        default:
            if (s.limiter == SL::VanLeer) return pick.template operator()<RC::Ppm, SL::VanLeer>();
            if (s.limiter == SL::Minmod) return pick.template operator()<RC::Ppm, SL::Minmod>();
            return pick.template operator()<RC::Ppm, SL::MonotonizedCentral>();
    }
}

template <class Form>
hipError_t launch_stage2d_impl(const Schemes& s, const StageGrid& g, const typename Form::Ptrs& p, hipStream_t st) {
    if (g.nx < 1 || g.ny < 1 || g.ng < min_ghost_cells(s.recon) || g.xc != g.nx + 2 * g.ng ||
        g.yc != g.ny + 2 * g.ng || g.nspans < 1 || g.nspans > g.ny || g.strips != (g.nx + kStripOut - 1) / kStripOut) {
        return hipErrorInvalidValue;
    }
    // the plain instance (buffer-resource addressing, no source, tracer
    // stores or floors), with the floors compiled in when they are on (forms
    // that have them), and the general instance for a gravity source or
    // tracer flux stores or when the state's byte offsets do not fit the
    // buffer offsets' 31 bits
    const bool big = (int64_t)4 * g.xc * g.yc * Form::kElem >= ((int64_t)1 << 31);
    const bool extras = p.gravity != 0 || p.frx != nullptr || p.fry != nullptr || big;
    const bool floors = Form::floors_on(p);
    const bool copies = copy_stage_ghosts(g);
    auto pick = [&]<Reconstruction R, SlopeLimiter SL>() -> Stage2dFn<Form> {
        using P = SolverPick<Form, R, SL>;
#ifdef MH_STAGE_WAVES_LONE
        if constexpr (R == Reconstruction::Weno5Z) {
            // no more wavefronts than SIMDs: none shares one
            const bool lone = (int64_t)g.strips * g.nspans <= kSimds;
            if (extras && lone && s.solver == RiemannSolver::Hllc) return copies ? P::template lone<true>() : P::template lone<false>();
        }
#endif
        if (extras) return copies ? P::template two<kStageExtras, true>(s.solver) : P::template two<kStageExtras, false>(s.solver);
        if constexpr (Form::kHasFloors) {
            if (floors) return copies ? P::template two<kStageFloors, true>(s.solver) : P::template two<kStageFloors, false>(s.solver);
        }
        return copies ? P::template two<kStagePlain, true>(s.solver) : P::template two<kStagePlain, false>(s.solver);
    };
    Stage2dFn<Form> fn = pick_scheme<Form>(s, pick);
    hipLaunchKernelGGL(fn, dim3((unsigned)(g.strips * g.nspans)), dim3(kWave), 0, st, g, p);
    return hipGetLastError();
}

template <class Form>
hipError_t launch_stage1d_impl(const Schemes& s, int kind, int reduce_dt, int xc, int ng,
                               const typename Form::Ptrs& p, hipStream_t st, int virt, int32_t faces) {
    const int nx = xc - 2 * ng;
    if (nx < 1 || ng < min_ghost_cells(s.recon)) return hipErrorInvalidValue;
    auto pick = [&]<Reconstruction R, SlopeLimiter SL>() { return SolverPick<Form, R, SL>::one(s.solver); };
    Stage1dFn<Form> fn = pick_scheme<Form>(s, pick);
    const Stage1dGrid g{xc, ng, nx, kind, reduce_dt, virt, faces};
    const int segs = (nx + kStripOut - 1) / kStripOut;
    hipLaunchKernelGGL(fn, dim3((unsigned)segs), dim3(kWave), 0, st, g, p);
    return hipGetLastError();
}

#ifdef MH_STAGE3D_INSTANCES
template <class Form, Reconstruction R, SlopeLimiter SL, RiemannSolver RS, bool Extras, bool Copies>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(stage_waves<R, RS>(Extras ? kStageExtras : kStagePlain))))
void stage3d_kernel(StageGrid g, typename Form::Ptrs p) {
    stage2d_march<Form, R, SL, RS, 3, Extras ? kStageExtras : kStagePlain, Copies>(g, p);
}

template <class Form, Reconstruction R, SlopeLimiter SL, RiemannSolver RS, bool Copies>
__global__ __launch_bounds__(128) void zsweep_kernel(ZSweepGrid g, typename Form::Ptrs p, typename Form::real* dz) {
    zsweep_column<Form, R, SL, RS, Copies>(g, p, dz);
}

template <class Form>
hipError_t launch_stage3d_impl(const Schemes& s, const StageGrid& g, const typename Form::Ptrs& p,
                               typename Form::real* dz, hipStream_t st) {
    if (g.nx < 1 || g.ny < 1 || g.nz < 1 || g.ng < min_ghost_cells(s.recon) || g.xc != g.nx + 2 * g.ng ||
        g.yc != g.ny + 2 * g.ng || g.zc != g.nz + 2 * g.ng || g.nspans < 1 || g.nspans > g.ny || !dz) {
        return hipErrorInvalidValue;
    }
    const MarchColumns cols = march_columns(g.nx, g.nz, 3, s.recon, sizeof(typename Form::real) == 8);
    if (g.strips != cols.strips || g.flat != cols.flat) return hipErrorInvalidValue;
    using ZFn = void (*)(ZSweepGrid, typename Form::Ptrs, typename Form::real*);
    const bool copies = copy_stage_ghosts(g);
    auto zsolver = [&]<Reconstruction R, SlopeLimiter SL, bool Copies>() -> ZFn {
        switch (s.solver) {
            case RiemannSolver::Rusanov: return zsweep_kernel<Form, R, SL, RiemannSolver::Rusanov, Copies>;
            case RiemannSolver::Hll: return zsweep_kernel<Form, R, SL, RiemannSolver::Hll, Copies>;
            default: return zsweep_kernel<Form, R, SL, RiemannSolver::Hllc, Copies>;
        }
    };
    auto zpick = [&]<Reconstruction R, SlopeLimiter SL>() -> ZFn {
        return copies ? zsolver.template operator()<R, SL, true>() : zsolver.template operator()<R, SL, false>();
    };
    // plain instance (buffer addressing, no source or floors) unless gravity
    // or the floors are on or a byte offset could pass 2^31
    const bool big = (int64_t)5 * g.xc * g.yc * g.zc * Form::kElem >= ((int64_t)1 << 31);
    const bool extras = p.gravity != 0 || Form::floors_on(p) || big;
    auto msolver = [&]<Reconstruction R, SlopeLimiter SL, bool Copies>() -> Stage2dFn<Form> {
        switch (s.solver) {
            case RiemannSolver::Rusanov:
                return extras ? stage3d_kernel<Form, R, SL, RiemannSolver::Rusanov, true, Copies>
                              : stage3d_kernel<Form, R, SL, RiemannSolver::Rusanov, false, Copies>;
            case RiemannSolver::Hll:
                return extras ? stage3d_kernel<Form, R, SL, RiemannSolver::Hll, true, Copies>
                              : stage3d_kernel<Form, R, SL, RiemannSolver::Hll, false, Copies>;
            default:
                return extras ? stage3d_kernel<Form, R, SL, RiemannSolver::Hllc, true, Copies>
                              : stage3d_kernel<Form, R, SL, RiemannSolver::Hllc, false, Copies>;
        }
    };
    auto mpick = [&]<Reconstruction R, SlopeLimiter SL>() -> Stage2dFn<Form> {
        return copies ? msolver.template operator()<R, SL, true>() : msolver.template operator()<R, SL, false>();
    };
    // z sweep: each thread walks a chunk of the planes, columns of the interior
    // across the grid's x; a chunk's prologue (its window of planes, the first
    // reconstruction) is worth 1.5 planes. With chunks of up to 32 planes
    // instead, the 128^3 FP64 stage took 408 us (now 351) and 64^3 140 (100).
    const int blocks = (g.nx * g.ny + 127) / 128;
    const int chunks = split_marches(2 * (int64_t)blocks, g.nz, 1.5, sizeof(typename Form::real) == 8);
    ZSweepGrid zg{g.xc, g.yc, g.zc, g.ng, g.nx, g.ny, g.nz, (g.nz + chunks - 1) / chunks};
    zg.virt = g.virt;
    zg.zf = g.zf;
    hipLaunchKernelGGL(pick_scheme<Form>(s, zpick), dim3((unsigned)blocks, (unsigned)chunks), dim3(128), 0, st, zg, p,
                       dz);
    typename Form::Ptrs pm = p;
    pm.dz3 = dz;
    hipLaunchKernelGGL(pick_scheme<Form>(s, mpick), dim3((unsigned)(g.strips * g.nspans)), dim3(kWave), 0, st,
                       g, pm);
    return hipGetLastError();
}
#endif

// Tracer planes of one 2-D stage, after the hydro stage stored the density
// fluxes. A span's prologue (its window of rows, two reconstructions) is worth
// two rows.
template <class Form>
hipError_t launch_tracer_impl(const Schemes& s, TracerGrid g, const typename Form::Ptrs& p, hipStream_t st) {
    if (g.ntr < 1 || g.nx < 1 || g.ny < 1 || g.ng < min_ghost_cells(s.recon) || g.xc != g.nx + 2 * g.ng ||
        g.yc != g.ny + 2 * g.ng || !p.frx || !p.fry)
        return hipErrorInvalidValue;
    const int outs = kWave - 2 * (stencil_order(s.recon) + 1);
    g.strips = (g.nx + outs - 1) / outs;
    g.nspans = split_marches((int64_t)g.strips * g.ntr, g.ny, 2.0, sizeof(typename Form::real) == 8);
    using Fn = void (*)(TracerGrid, typename Form::Ptrs);
    auto pick = [&]<Reconstruction R, SlopeLimiter SL>() -> Fn { return tracer_stage_kernel<Form, R, SL>; };
    Fn fn = pick_scheme<Form>(s, pick);
    hipLaunchKernelGGL(fn, dim3((unsigned)(g.strips * g.nspans * g.ntr)), dim3(kWave), 0, st, g, p);
    return hipGetLastError();
}

}  // namespace mh
