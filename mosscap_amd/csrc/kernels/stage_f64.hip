// Fused stage kernels of the FP64 drop-in path. Built with -ffp-contract=off:
// no multiply-add contraction, so results match the reference CPU build bitwise.
#ifndef MH_STAGE_WAVES_F64
#define MH_STAGE_WAVES_F64 1
#endif
// PPM + Rusanov fits three: left alone, its van Leer instance with mirrored ghosts
// takes 171 VGPRs and two (2048^2 between walls: step 644 us, 599 so).
#define MH_STAGE_WAVES_PER_EU (R == Reconstruction::Ppm && RS == RiemannSolver::Rusanov ? 3 : MH_STAGE_WAVES_F64)
// The general WENO5-Z + HLLC instance takes 259 VGPRs (266 with mirrored
// ghosts) when left alone, 3 to 10 more than let two wavefronts share a SIMD;
// held to 256 it spills 1 (9) of them. A step with gravity then takes 893 us
// instead of 1208 on 2048^2 periodic (953 instead of 1225 between walls) and
// 253 instead of 314 on 1024^2. Launches of no more wavefronts than SIMDs
// keep the one without spills: 640x480 with two tracers, stage 41.3 us against
// 42.6. The other schemes fit 256 as they are.
#define MH_STAGE_WAVES_EXTRAS 2
#define MH_STAGE_WAVES_LONE 1
// The raw Q^(s) of the stencil rows stays in registers for the combine (no
// second load of row j) with WENO5-Z; the other schemes keep 3 waves per
// SIMD without it (PPM + HLL: 154 VGPRs, 180 with it).
#ifndef MH_STAGE_QS_RING_F64
#define MH_STAGE_QS_RING_F64 2
#endif
#define MH_STAGE_QS_RING MH_STAGE_QS_RING_F64
#include "stage_inst.hpp"

namespace mh {

hipError_t launch_stage2d_f64(const Schemes& s, const StageGrid& g, const FormF64::Ptrs& p, hipStream_t st) {
    return launch_stage2d_impl<FormF64>(s, g, p, st);
}

hipError_t launch_stage1d_f64(const Schemes& s, int kind, int reduce_dt, int xc, int ng, const FormF64::Ptrs& p,
                              hipStream_t st, int virt, int32_t faces) {
    return launch_stage1d_impl<FormF64>(s, kind, reduce_dt, xc, ng, p, st, virt, faces);
}

hipError_t launch_tracer_f64(const Schemes& s, const TracerGrid& g, const FormF64::Ptrs& p,
                              hipStream_t st) {
    return launch_tracer_impl<FormF64>(s, g, p, st);
}

}  // namespace mh
