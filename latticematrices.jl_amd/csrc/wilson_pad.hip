// wilson_pad.hip -- mul! on the reference's own storage: psi and C are
// LatticeMatrix.A arrays (complex128 or complex64, column-major
// [3,4,L1+2nw,...,L4+2nw]).  psi's halo is not read: neighbours wrap in-kernel
// with the spinor phases (the halo fill of set_halo!,
// src/LatticeMatrices_core.jl:707-723, applied on the fly); only C's core
// sites are written.  Links and the clover cache are the operator's own
// (core-indexed).
#include "wilson_hops.h"

namespace lmx {

int launch_wilson_padded(lmx_context* ctx, const double2* U, const double2* clover, double kappa, double csw,
                         double2* C, const double2* psi, int nw, int nrhs, int flags) {
    return launch_hops_pad<1>(ctx, LinkF64{U, (int)ctx->V}, F64Clover{clover}, clover != nullptr, kappa, csw, C, psi, nw,
                              nrhs, flags);
}

int launch_wilson_padded_f32(lmx_context* ctx, const float2* U, const float2* clover, double kappa, double csw,
                             float2* C, const float2* psi, int nw, int nrhs, int flags) {
    const LinkF32 l{U, (int)ctx->V};
    const F32Clover F{clover};
    // two components per load and store where both arrays are 16-byte aligned
    // (a site is 96 bytes, so every site then is)
    if (((uintptr_t)C | (uintptr_t)psi) % 16 == 0)
        return launch_hops_pad<2>(ctx, l, F, clover != nullptr, kappa, csw, C, psi, nw, nrhs, flags);
    return launch_hops_pad<1>(ctx, l, F, clover != nullptr, kappa, csw, C, psi, nw, nrhs, flags);
}

}  // namespace lmx
