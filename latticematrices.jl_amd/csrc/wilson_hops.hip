// wilson_hops.hip -- the eight-wavefront stencil's FP64 and FP32 launches.
#include "wilson_hops.h"

namespace lmx {

bool hops_f64(const lmx_context* ctx, bool clover) {
    const Geom& g = ctx->g;
    const long V3 = g.stride[3];
    if (V3 % 256 != 0 || g.general) return true;  // no t-streaming there
    // k_stream's grid: 256-site blocks by chunks of TL t-slices, the largest TL with at least 256 workgroups
    long tl = 16, wgs = 0;
    for (; tl >= 1; tl /= 2) {
        if (g.L[3] % tl) continue;
        wgs = V3 / 256 * (g.L[3] / tl);
        if (wgs >= 256) break;
    }
    const double fill = (double)wgs / (256.0 * ((wgs + 255) / 256));
    // measured, us (this kernel / k_stream).  Wilson: 16^3 x 32 27 / 31, 24^3 x 48
    // 150 / 199, 40^3 x 80 1210 / 1308, 48^3 x 96 2650 / 2925; k_stream wins
    // only where its workgroups fill the 256 CUs exactly once and walk far
    // (32^3 x 16 123 / 115, 32^4 250 / 232; two rounds, 32^3 x 64: 482 / 505).
    // Clover, where each wavefront pair reads the planes again: 16^3 x 32
    // 36 / 39, 24^3 x 48 221 / 269 (k_stream's grid fills 63% there), but 32^4
    // 369 / 322, 32^3 x 64 715 / 640, 40^3 x 80 1740 / 1693, 48^3 x 96 3900 / 3870.
    if (clover) return tl < 4 || fill < 0.8;
    return tl < 8 || wgs > 256 || fill < 0.8;
}

int launch_hops_f64(lmx_context* ctx, double2* out, const double2* in, const double2* U, const double2* clover,
                    const double2* p, double kappa, double csw, int nrhs, int flags, const Epilogue& e) {
    const int V = (int)ctx->V;
    const double ccoef = (-kappa) * csw;
    const SpF64Out o{out, V};
    const SpF64In i{in, V}, aux{p, V};
    const LinkF64 l{U, V};
    const F64Clover F{clover};
    const EpiArgs epi{e.partials, 0, e.st, e.gate};
    if (e.kind == 1)
        return launch_hops<SpF64In, LinkF64, SpF64Out, F64Clover, EPI_PAP>(ctx, o, i, l, F, aux, kappa, ccoef, nrhs,
                                                                          flags, clover != nullptr, epi);
    return launch_hops<SpF64In, LinkF64, SpF64Out, F64Clover, EPI_NONE>(ctx, o, i, l, F, i, kappa, ccoef, nrhs, flags,
                                                                       clover != nullptr, epi);
}

}  // namespace lmx
