// wilson_hops.hip -- the eight-wavefront stencil's FP64 and FP32 launches, and
// the LDS-staged stencil's on plain FP32 fields.
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
// Right-hand sides per workgroup: all that share the links where the blocks
// alone fill the chip (24^3 x 48, 12 FP64 fields: 1280 us against 1500 one by
// one), one where they do not (8^3 x 16: 17 against 24).
static int rhs_per_block(const lmx_context* ctx, int nrhs) {
    return slab_order(ctx->g, false, 12 * sizeof(double2)).blocks >= 512 ? std::min(nrhs, 12) : 1;
}

// Slices this large (64^3, 64x64x48) leave no slab in an XCD's L2 from one
// slice to the next without cutting it small; k_stream keeps its neighbours in
// t in registers.
constexpr long kLargeSlice = 150000;

// Measured, us, this kernel / the other.
bool hops_f64(const lmx_context* ctx, int nrhs, bool clover) {
    const StreamUse st = stream_use(ctx, clover ? nrhs : (nrhs + 1) / 2, 256);
    // against k_site: 18x20x22x30 42 / 80, four fields 173 / 252; clover 65 / 93, 227 / 242
    if (st.tl == 0 || ctx->g.general) return true;
    if (shape_forced(ctx)) return false;
    const long V3 = ctx->g.stride[3];
    const bool large = V3 >= kLargeSlice;
    // k_stream wins where its workgroups fill the 256 CUs an exact number of
    // times and walk far, the sooner the larger the slices.  Clover, one field
    // per work item: 32^4 335 / 324, x 4 1055 / 981, 16^4 x 4 53 / 50, 32^3 x 4 x 2
    // 61 / 56, 64^3 x 4 377 / 361, x 2 640 / 586, but 16^3 x 32 35 / 39, 24^3 x 48
    // 192 / 270, 40^3 x 80 1560 / 1697, 48^3 x 96 3501 / 3866.
    if (clover) return st.fill < 0.99 || st.tl < (nrhs >= 4 || large || (nrhs >= 2 && V3 >= 32768) ? 4 : 8);
    // One field: 32^3 x 16 122 / 115, 32^4 253 / 230 and 16^3 x 128 (one round of
    // workgroups, 256), but two rounds or more 32^3 x 64 491 / 503, 64x32^3 510 /
    // 523, 32^3 x 96 737 / 744, 96x32^3 808 / 840, on the largest slices 64^3 x 8
    // 585 / 564, x 12 856 / 844, 64x64x32x8 287 / 275 (128x64x32x8 600 / 642: rows
    // longer than a quarter of its blocks); 16^3 x 32 26 / 31, 24^3 x 48 146 / 198,
    // 40^3 x 80 1185 / 1310, 48^3 x 96 2610 / 2920.
    if (nrhs == 1) {
        const bool stream_large = V3 >= (st.tl == ctx->g.L[3] ? 131072 : kLargeSlice) && ctx->g.L[0] <= 64 &&
                                  st.tl >= 4 && st.fill >= 0.99;
        return !stream_large && (st.tl < 8 || st.fill < 0.8 || st.wgs > 256);
    }
    // Two, in turn here, in one work item there: 32^4 381 / 374, 32^3 x 48 725 / 666,
    // 48x32^3 754 / 696, 24^3 x 32 187 / 179, 40^3 x 8 242 / 214, 64^3 x 4 556 / 435,
    // but 16^3 x 96 170 / 178, 32x32x16x16 at one round of workgroups, 24^3 x 48
    // (0.63 full) 250 / 297.
    if (nrhs == 2 && st.fill >= 0.75 && st.tl >= (st.wgs > 256 ? 4 : 8) && V3 >= 13000) return false;
    // More: 32^4 x 4 798 / 684, 32^3 x 12 x 4 294 / 276, 64^3 x 4 x 6 1378 / 1297, but
    // 32^3 x 12 x 6 and x 12 are 8 and 9% faster here, 16^3 x 32 x 4 80 / 93, 24^3 x
    // 48 x 4 456 / 598.
    if (st.tl == 4 && st.wgs > 256 && st.fill >= 0.9 && V3 >= 32768 && (nrhs <= 4 || large)) return false;
    return st.tl < 8 || st.fill < 0.8;
}

// The LDS-staged kernel (streaming lattices) where it has work enough.
bool lds_f32(const lmx_context* ctx, int nrhs, bool clover) {
    if (!lds_ok(ctx)) return false;
    const int64_t n = ctx->V * nrhs;
    // clover, LDS-staged / eight wavefronts: 24^3 x 48 110 / 111, x 12 820 / 1031,
    // 32^4 163 / 195, x 4 456 / 599, 16^3 x 32 x 4 58 / 61, but 32x16x24x36 68 / 60,
    // 16^4 x 4 34 / 33
    if (clover) return n >= 500000;
    // 32^4 116 / 150, x 12 1063 / 1158, 24^3 x 48 x 2 136 / 151, x 4 252 / 256, but
    // 24^3 x 48 69 / 63, 32x16x24x36 x 2 82 / 79; on a small lattice many fields
    // share the links there: 16^3 x 32 x 12 113 / 108, 24^3 x 48 x 12 700 / 675
    return n >= 1000000 && (nrhs <= 4 || ctx->V >= 1000000);
}

// Else the eight wavefronts, but for clover fields where they do not share the
// links and the lattice does not stream: k_site at 20^3 x 40 x 4 159 against
// 171, but 27x29x31x35 x 12 1546 against 1460.
bool hops_f32(const lmx_context* ctx, int nrhs, bool clover) {
    return nrhs == 1 || !clover || lds_ok(ctx) || ctx->V * nrhs <= 550000 || ctx->V >= 500000;
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

// D or D^dagger of FP32 fields, up to twelve in a launch.
int launch_lds_f32(lmx_context* ctx, const LoArgs& a) {
    const int V = (int)ctx->V;
    const Geom& gg = ctx->g;
    const bool rows = gg.L[0] <= 256 && 256 % gg.L[0] == 0 && gg.L[1] % (256 / gg.L[0]) == 0;
    const bool dag = (a.flags & LMX_DAGGER) != 0, donly = (a.flags & LMX_DONLY) != 0, clover = a.clover != nullptr;
    const LinkF32 U{(const float2*)a.links, V};
    const F32Clover F{(const float2*)a.clover};
    const double ccoef = (-a.kappa) * a.csw;
    for (int r0 = 0; r0 < a.nrhs; r0 += 12) {
        const int n = std::min(12, a.nrhs - r0);
        const Shape sh = pick_shape(ctx, n, 512, lds_slices(ctx, n), 1);
        const int nb = (int)(ctx->V / 256 / sh.TL) * n;
        const SpF32Out o = SpF32Out::at(a.out, nullptr, V, r0);
        const SpF32In i = SpF32In::at(a.in, nullptr, V, r0);
        const EpiArgs epi{nullptr, 0, const_cast<CGState*>(a.st), a.gate};
#define LMX_LDS_ONE(FPM, MODE, ROWS)                                                                                      \
    hipLaunchKernelGGL((k_lds<SpF32In, LinkF32, SpF32Out, F32Clover, SpF32In, NoEx, FPM, MODE, EPI_NONE, ROWS>), dim3(nb), \
                       dim3(256), 0, ctx->stream, o, i, U, F, i, NoEx{}, gg, a.kappa, ccoef, n, sh.TL, sh.ZS, epi)
#define LMX_LDS_GO(FPM, MODE)               \
    do {                                    \
        if (rows)                           \
            LMX_LDS_ONE(FPM, MODE, true);   \
        else                                \
            LMX_LDS_ONE(FPM, MODE, false);  \
    } while (0)
        if (donly && dag)
            LMX_LDS_GO(1, MODE_DONLY);
        else if (donly)
            LMX_LDS_GO(-1, MODE_DONLY);
        else if (dag && clover)
            LMX_LDS_GO(1, MODE_CLOVER);
        else if (dag)
            LMX_LDS_GO(1, MODE_WILSON);
        else if (clover)
            LMX_LDS_GO(-1, MODE_CLOVER);
        else
            LMX_LDS_GO(-1, MODE_WILSON);
#undef LMX_LDS_GO
#undef LMX_LDS_ONE
        LMX_HIP(hipGetLastError());
    }
    return LMX_OK;
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
