// Passive tracer fields (simulation.n_extra_fields) of a 2-D stage.
//
// The reference carries each tracer as a conserved density Q_t; its primitive
// is the mass fraction W_t = Q_t * (1/rho) (Hydro.cpp:27-33), reconstructed
// like the hydro variables (Hydro.cpp:55-102), and its face flux is the
// density flux times the upwind face value: F_t = F_rho * RR(left) when
// F_rho >= 0, else F_rho * RL(right) (Hydro.cpp:155-162). The divergence and
// the stage combination are those of the hydro variables with a zero source
// (TimeStepping.cpp stage lambdas, `var >= n_hydro`).
//
// Here the fused hydro stage stores F_rho of every x and y face it computes;
// the tracer march then reads the stage input's tracer and density planes and
// those fluxes. Tracers never feed back into the hydro variables or the time
// step.
//
// March: one wavefront per tracer, strip of columns and span of rows, lanes
// along x, rows downwards, as the hydro stage: each cell's W_t is formed and
// reconstructed once per axis. (A thread per cell reconstructed its two
// neighbours along each axis as well, six reconstructions of which two are
// its own, and read W_t from a pass of its own before it: 640x480, two
// tracers, FP64 WENO5-Z 23.8 us a stage, 15.6 now.) A row's chain of two
// reconstructions bounds it there, with two wavefronts per SIMD; from 80 to 170
// spans (split_marches takes 85) the time is the same to 2 %, 60 take 18.4 us
// and 240 take 16.5. The outer ORD + 1 lanes on each side carry the columns that the
// strip's outermost faces need, so that no lane has a halo to load beside its
// own column.
#pragma once

#include "functors.hpp"
#include "ghost_dt.hpp"
#include "wave.hpp"

namespace mh {

struct TracerGrid {
    int32_t xc, yc, ng, nx, ny;
    int32_t ntr;   // tracer count; planes 4 .. 3+ntr of the state
    int32_t kind;  // StageKind
    int32_t strips, nspans;  // wavefronts side by side and spans of rows (the launcher's)
    int32_t virt, xf, yf;  // ghosts read from their sources (StageGrid::virt), where they are not filled
};

// output columns per wavefront of the tracer march
template <Reconstruction R>
constexpr int kTracerOut = kWave - 2 * (stencil_order(R) + 1);

template <class Form, Reconstruction R, SlopeLimiter SL>
__global__ __launch_bounds__(64) void tracer_stage_kernel(TracerGrid g, typename Form::Ptrs p) {
    using T = typename Form::real;
    using Raw = typename Form::raw;
    constexpr int ORD = stencil_order(R);
    // window of the lane's column, rows j+1-ORD .. j+1+ORD and row j (stage2d_march)
    constexpr int WIN = 2 * ORD + 1 + (ORD == 0 ? 1 : 0);
    constexpr int WY = WIN - 1 - ORD;
    constexpr int WX = WY - 1;
    __shared__ T xrow[kWave + 2 * ORD];

    const int lane = threadIdx.x;
    const int b = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int strip = b % g.strips, rest = b / g.strips;
    const int span = rest % g.nspans, tracer = rest / g.nspans;
    const int j0 = g.ng + (int)(((int64_t)span * g.ny) / g.nspans);
    const int j1 = g.ng + (int)(((int64_t)(span + 1) * g.ny) / g.nspans);
    const int xc = g.xc, plane = g.xc * g.yc;
    const int c = g.ng + strip * kTracerOut<R> - (ORD + 1) + lane;
    const int c_in = min(c, xc - 1);
    const int c_ld = g.virt ? face_source(c_in, g.nx, g.ng, g.xf) : c_in;
    const bool out_lane = lane >= ORD + 1 && lane < kWave - (ORD + 1) && c < g.ng + g.nx;
    const int tr = (4 + tracer) * plane;
    const T dt = (T)p.dt[0];
    const T dtdx = dt / (T)p.dx;
    const T src = T(0) * dt;

    T win[WIN] = {};
    Raw q, rho;
    auto fetch = [&](int r) {
        const int row = (g.virt ? face_source(r, g.ny, g.ng, g.yf) : r) * xc;
        rho = Form::get(p.qs, row + c_ld);
        q = Form::get(p.qs, tr + row + c_ld);
    };
    // W_t = Q_t * (1/rho), FP64 reciprocal as in global_cons_to_prim_impl
    // (neither a density nor a tracer changes its sign beyond a wall)
    auto commit = [&] {
#pragma unroll
        for (int k = 0; k + 1 < WIN; ++k) win[k] = win[k + 1];
        win[WIN - 1] = (T)(Form::value(q) * div_ieee(1.0, Form::value(rho)));
    };
    auto recon_y = [&](T& l, T& r) {
        auto s = [&](int o) -> T { return win[WY + o]; };
        reconstruct_stencil<R, SL, T>(s, l, r);
    };
    T yl, yr, yRp, Gp;
#pragma unroll
    for (int k = 0; k < 2 * ORD + 1; ++k) {  // rows j0-1-ORD .. j0-1+ORD
        fetch(j0 - 1 - ORD + k);
        commit();
    }
    recon_y(yl, yRp);  // cell j0-1
    fetch(j0 + ORD);
    commit();
    recon_y(yl, yr);  // cell j0
    {
        const T f = p.fry[j0 * xc + c_in];
        Gp = f >= T(0) ? f * yRp : f * yl;
    }
    yRp = yr;
    fetch(j0 + 1 + ORD);
    for (int j = j0; j < j1; ++j) {
        // this row's operands, then (the row that the window takes having
        // arrived) the row after it: in flight while the row is swept
        const T fx = p.frx[j * xc + c_in], fy = p.fry[(j + 1) * xc + c_in];
        const int idx = tr + j * xc + c_in;
        const Raw qs = Form::get(p.qs, idx);
        const Raw qn = Form::needs_qn(g.kind) ? Form::get(p.qn, idx) : qs;
        commit();
        if (j + 1 < j1) fetch(j + 2 + ORD);

        recon_y(yl, yr);  // cell j+1, face j+1
        const T G = fy >= T(0) ? fy * yRp : fy * yl;
        const T dy = Gp - G;
        Gp = G;
        yRp = yr;

        wave_lds_sync();
        xrow[lane + ORD] = win[WX];
        wave_lds_sync();
        T xl, xr;
        auto s = [&](int o) -> T { return xrow[lane + ORD + o]; };
        reconstruct_stencil<R, SL, T>(s, xl, xr);
        const T xrm = lane_from_left(xr);  // (every lane takes part, whatever its flux's sign)
        const T F = fx >= T(0) ? fx * xrm : fx * xl;
        const T Fp = lane_from_right(F);
        if (out_lane) {
            T q_update = T(0);
            q_update += F - Fp;
            q_update += dy;
            q_update *= dtdx;
            Form::put(p.out, idx, Form::combine(g.kind, qs, qn, q_update, src));
        }
    }
}

// Ghost fill of the tracer planes: the hydro fill's index maps (x pass, then
// y pass reading the x-filled rows) with no modification, since wall,
// symmetric and diode faces only change the normal momentum and the energy.
template <class Form>
__global__ __launch_bounds__(256) void tracer_ghost_kernel(GhostGrid g, int ntr, typename Form::Planes in,
                                                           typename Form::Planes out) {
    const int xc = g.xc, yc = g.yc, ng = g.ng;
    const int plane = xc * yc;
    const int nxband = 2 * ng * yc, nyband = 2 * ng * xc;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    // (source buffer is `in`, source cell); x pass value at (j, i), i an x-ghost column
    auto xsource = [&](int j, int i, bool& from_in) -> int {
        const bool start = i < ng;
        const BoundaryType b = (BoundaryType)(start ? g.bc[0] : g.bc[1]);
        if (b == BoundaryType::UserFn) {
            from_in = true;
            return j * xc + i;
        }
        const bool yghost = j < ng || j >= yc - ng;
        from_in = yghost;
        return j * xc + ghost_source(i, xc, ng, b);
    };
    int dst = -1, srcc = 0;
    bool from_in = false;
    if (tid < nxband) {
        const int pp = tid % (2 * ng);
        const int j = tid / (2 * ng);
        const int i = pp < ng ? pp : (xc - 1) - (pp - ng);
        bool skip = false;
        if (j < ng || j >= yc - ng) skip = (BoundaryType)(j < ng ? g.bc[2] : g.bc[3]) != BoundaryType::UserFn;
        if (!skip) {
            dst = j * xc + i;
            srcc = xsource(j, i, from_in);
        }
    } else if (tid < nxband + nyband) {
        const int tt = tid - nxband;
        const int pp = tt / xc;
        const int i = tt % xc;
        const int j = pp < ng ? pp : (yc - 1) - (pp - ng);
        const BoundaryType b = (BoundaryType)(j < ng ? g.bc[2] : g.bc[3]);
        dst = j * xc + i;
        if (b == BoundaryType::UserFn) {
            from_in = true;
            srcc = dst;
        } else {
            const int js = ghost_source(j, yc, ng, b);
            if (i < ng || i >= xc - ng) {
                srcc = xsource(js, i, from_in);
            } else {
                from_in = false;
                srcc = js * xc + i;
            }
        }
    }
    if (dst < 0) return;
    for (int k = 0; k < ntr; ++k) {
        const int off = (4 + k) * plane;
        Form::put(out, off + dst, Form::get(from_in ? in : out, off + srcc));
    }
}

}  // namespace mh
