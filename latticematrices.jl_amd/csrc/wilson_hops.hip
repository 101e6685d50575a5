// wilson_hops.hip -- the eight-wavefront stencil's FP64 and FP32 launches.
#include "wilson_hops.h"

namespace lmx {

// k_stream's launch for this many RHS groups: t-slices per workgroup (0: it
// does not stream there) and how much of the chip its rounds of `round`
// workgroups fill.
struct StreamUse {
    int tl;
    long wgs;
    double fill;
};
static StreamUse stream_use(const lmx_context* ctx, int ngroups, int round) {
    const Shape sh = pick_shape(ctx, ngroups, round, 0);
    if (!sh.stream) return {0, 0, 0.0};
    const long wgs = ctx->V / 256 / sh.TL * ngroups;
    return {sh.TL, wgs, (double)wgs / (double)((wgs + round - 1) / round * round)};
}
// The caller has named a streaming shape (LMX_STREAM_TL, LMX_STREAM_ZS).
static bool shape_forced(const lmx_context* ctx) { return ctx->tune_tl > 0 || ctx->tune_zs > 0; }

// Right-hand sides per workgroup: all that share the links where the blocks
// alone fill the chip (24^3 x 48, 12 FP64 fields: 1280 us against 1500 one by
// one), one where they do not (8^3 x 16: 17 against 24).
static int rhs_per_block(const lmx_context* ctx, int nrhs) {
    return slab_order(ctx->g, false).blocks >= 512 ? std::min(nrhs, 12) : 1;
}

// Measured, us, this kernel / the other.
bool hops_f64(const lmx_context* ctx, int nrhs, bool clover) {
    // several clover fields: the planes are read for each (16^4 x 4 59 / 50,
    // 24^3 x 48 x 4 690 / 699, but 8^3 x 16 x 4 9 / 12)
    if (clover && nrhs > 1) return ctx->V * nrhs <= 100000;
    const StreamUse st = stream_use(ctx, clover ? nrhs : (nrhs + 1) / 2, 256);
    if (st.tl == 0 || ctx->g.general) return true;  // k_site: 18x20x22x30 42 / 80, four fields 173 / 252
    if (shape_forced(ctx)) return false;
    // Clover: 16^3 x 32 36 / 39, 24^3 x 48 213 / 268 (k_stream fills 63%), but
    // 32^4 365 / 321, 40^3 x 80 1740 / 1693, 48^3 x 96 3850 / 3867.
    if (clover) return st.tl < 4 || st.fill < 0.8;
    // One field: 16^3 x 32 26 / 31, 24^3 x 48 146 / 198, 40^3 x 80 1185 / 1310,
    // 48^3 x 96 2610 / 2920; k_stream wins where its workgroups fill the 256
    // CUs exactly once and walk far (32^3 x 16 122 / 115, 32^4 253 / 230).
    // Several, two of them to its work item: 16^3 x 32 x 4 80 / 93, 24^3 x 48 x 4
    // 471 / 598, but 32^4 x 4 798 / 684, 40^3 x 80 x 2 2270 / 1940.
    return st.tl < 8 || st.fill < 0.8 || (nrhs == 1 && st.wgs > 256);
}

bool hops_f32(const lmx_context* ctx, int nrhs, bool clover) {
    // clover, the planes read twice and more: 8^3 x 16 6 / 11, but 24^3 x 48 146 / 129
    if (clover) return ctx->V * nrhs <= 50000;
    // several fields share the links (24^3 x 48 x 4 266 / 341, 32^4 x 12 1246 / 1546);
    // one: 24^3 x 48 63 / 79, 40^3 x 80 682 / 718, and as above 32^4 151 / 145
    const Geom& g = ctx->g;
    if (nrhs > 1 || g.general || !(g.phase_one[0] && g.phase_one[1] && g.phase_one[2])) return true;
    const StreamUse st = stream_use(ctx, 1, 512);
    return st.tl < 8 || st.fill < 0.8 || st.wgs > 512;
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
        return launch_hops<SpF64In, LinkF64, SpF64Out, F64Clover, EPI_PAP>(ctx, o, i, l, F, aux, kappa, ccoef, nrhs, 1,
                                                                          flags, clover != nullptr, epi);
    return launch_hops<SpF64In, LinkF64, SpF64Out, F64Clover, EPI_NONE>(ctx, o, i, l, F, i, kappa, ccoef, nrhs, rhs_per_block(ctx, nrhs), flags,
                                                                       clover != nullptr, epi);
}

int launch_hops_f32(lmx_context* ctx, const LoArgs& a) {
    const int V = (int)ctx->V;
    const EpiArgs epi{nullptr, 0, const_cast<CGState*>(a.st), a.gate};
    const SpF32In in = SpF32In::at(a.in, nullptr, V, 0);
    return launch_hops<SpF32In, LinkF32, SpF32Out, F32Clover, EPI_NONE>(
        ctx, SpF32Out::at(a.out, nullptr, V, 0), in, LinkF32{(const float2*)a.links, V},
        F32Clover{(const float2*)a.clover}, in, a.kappa, (-a.kappa) * a.csw, a.nrhs, rhs_per_block(ctx, a.nrhs), a.flags, a.clover != nullptr, epi);
}

}  // namespace lmx
