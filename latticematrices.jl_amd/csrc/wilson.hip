// wilson.hip -- FP64 Wilson(-clover) apply (bit-exact with the reference's
// kernels) and the dispatch of the low-precision variants built in
// wilson_lo.hip.  The stencil itself is in wilson_kernels.h.
#include "wilson_kernels.h"

namespace lmx {

#define LMX_EXTERN(In, Out, Lk, Cl, NR) extern template int launch_lo_nr<In, Out, Lk, Cl, NR>(lmx_context*, const LoArgs&, Lk, Cl, bool);
LMX_LO_ALL(LMX_EXTERN)
#undef LMX_EXTERN
extern template int launch_lo_loop<SpF32In, SpF32Out, F16Clover>(lmx_context*, const LoArgs&, LinkF16, F16Clover, bool);
extern template int launch_lo_loop<SpH16In, SpH16Out, F16Clover>(lmx_context*, const LoArgs&, LinkF16, F16Clover, bool);
#define LMX_EXTERN_LDS(In, Out, Lk, Cl, NR) extern template int launch_lo_lds<In, Out, Lk, Cl>(lmx_context*, const LoArgs&, Lk, Cl, bool);
LMX_LO_COMBOS(LMX_EXTERN_LDS, 1)
#undef LMX_EXTERN_LDS

int launch_wilson_f64(lmx_context* ctx, const double2* U, const double2* clover, double kappa, double csw,
                      double2* out, const double2* in, int nrhs, int flags, const Epilogue& e) {
    if (ctx->V == 0 || nrhs == 0) return LMX_OK;
    if (ctx->nc != 3) {  // the reference's generic-NC kernels (wilson_nc.hip)
        LMX_CHECK(e.kind == 0, LMX_ERR_UNSUPPORTED, "fused epilogues are built for NC = 3");
        return launch_wilson_nc(ctx, U, clover, kappa, csw, out, in, nrhs, flags, -1, e.st, e.gate);
    }
    const double ccoef = (-kappa) * csw;  // coefficient = -kappa * cSW (:572)
    const int V = (int)ctx->V;
    SpF64Out o{out, V};
    SpF64In i{in, V};
    LinkF64 l{U, V};
    F64Clover F{clover};
    EpiArgs epi{e.partials, 0, e.st, e.gate};
    const NoEx none{};
    // the eight-wavefront kernel where it is the faster one; a gated launch,
    // which mostly only finds its gate off, keeps the smaller grids
    const bool hops = e.gate == nullptr && hops_f64(ctx, nrhs, clover != nullptr);
    if (hops) {
        LMX_TRY(launch_hops_f64(ctx, out, in, U, clover, e.aux, kappa, csw, nrhs, flags, e));
        return e.kind == 1 ? launch_finalize(ctx, nblocks(ctx->V), FIN_PAP, false, e.st, nullptr, true) : LMX_OK;
    }
    if (e.kind == 1) {
        LMX_CHECK(nrhs == 1, LMX_ERR_UNSUPPORTED, "fused p.Ap needs a single right-hand side");
        SpF64In aux{e.aux, V};
        LMX_TRY((dispatch<SpF64In, LinkF64, SpF64Out, F64Clover, SpF64In, NoEx, 1, EPI_PAP, true, true>(
            ctx, o, i, l, F, aux, none, kappa, ccoef, 1, 1, flags, clover != nullptr, epi, 256)));
        return launch_finalize(ctx, nblocks(ctx->V), FIN_PAP, false, e.st, nullptr);
    }
    // several Wilson RHS: two per work item share each link load (the same
    // per-RHS arithmetic, so bit-identical to one per work item); the clover
    // variant would spill at two, so it keeps one
    if (nrhs >= 2 && clover == nullptr)
        return dispatch<SpF64In, LinkF64, SpF64Out, F64Clover, SpF64In, NoEx, 2, EPI_NONE, true, true>(
            ctx, o, i, l, F, i, none, kappa, ccoef, (nrhs + 1) / 2, nrhs, flags, false, epi, 256);
    return dispatch<SpF64In, LinkF64, SpF64Out, F64Clover, SpF64In, NoEx, 1, EPI_NONE, true, true>(
        ctx, o, i, l, F, i, none, kappa, ccoef, nrhs, nrhs, flags, clover != nullptr, epi, 256);
}

template <class SO>
static int wilson_f64_true(lmx_context* ctx, const double2* U, const double2* clover, double kappa, double csw,
                           const double2* in, const double2* b, SO rout, const int* done, const int* fold,
                           int dstride, int force, double* partials, long pstride, int nrhs, const int* gate) {
    const double ccoef = (-kappa) * csw;
    const int V = (int)ctx->V;
    SpF64Out o{nullptr, V};  // D^dagger in itself is not stored
    SpF64In i{in, V};
    LinkF64 l{U, V};
    F64Clover F{clover};
    EpiArgs epi{partials, pstride, nullptr, gate};
    TrueEx<SO> ex{SpF64In{b, V}, rout, done, fold, dstride, force};
    if (nrhs >= 2 && clover == nullptr)  // as launch_wilson_f64: two Wilson RHS per work item
        return dispatch<SpF64In, LinkF64, SpF64Out, F64Clover, SpF64In, TrueEx<SO>, 2, EPI_TRUE, true, true>(
            ctx, o, i, l, F, i, ex, kappa, ccoef, (nrhs + 1) / 2, nrhs, LMX_DAGGER, false, epi, 256);
    return dispatch<SpF64In, LinkF64, SpF64Out, F64Clover, SpF64In, TrueEx<SO>, 1, EPI_TRUE, true, true>(
        ctx, o, i, l, F, i, ex, kappa, ccoef, nrhs, nrhs, LMX_DAGGER, clover != nullptr, epi, 256);
}

int launch_wilson_f64_true(lmx_context* ctx, const double2* U, const double2* clover, double kappa, double csw,
                           const double2* in, const double2* b, void* r, float* r_norm, int spinor_prec,
                           const int* done, const int* fold, int dstride, int force, double* partials, long pstride,
                           int nrhs, const int* gate) {
    if (ctx->V == 0 || nrhs == 0) return LMX_OK;
    LMX_CHECK(ctx->nc == 3, LMX_ERR_UNSUPPORTED, "the fused true residual is built for NC = 3");
    const int V = (int)ctx->V;
    if (spinor_prec == LMX_H16)
        return wilson_f64_true(ctx, U, clover, kappa, csw, in, b, SpH16Out::at(r, r_norm, V, 0), done, fold, dstride,
                               force, partials, pstride, nrhs, gate);
    return wilson_f64_true(ctx, U, clover, kappa, csw, in, b, SpF32Out::at(r, r_norm, V, 0), done, fold, dstride,
                           force, partials, pstride, nrhs, gate);
}

// ---------------------------------------------------------------------------
// Low-precision variants for the mixed / multi-RHS solver: spinors FP32 or
// 16-bit (fixed point with a per-site FP32 scale), links FP32 or FP16, FP32
// arithmetic.
// ---------------------------------------------------------------------------
template <class In, class Out, class Lk, class Cl>
static int launch_lo_sp(lmx_context* ctx, const LoArgs& a, Lk U, Cl F, bool clover) {
    if constexpr (std::is_same<Lk, LinkF16>::value) {
        if ((a.rhs_block & kRhsLoop) && rhsloop_ok(ctx)) return launch_lo_loop<In, Out, Cl>(ctx, a, U, F, clover);
    }
    if ((a.rhs_block & kLdsStage) && lds_ok(ctx)) return launch_lo_lds<In, Out, Lk, Cl>(ctx, a, U, F, clover);
    switch (a.rhs_block & 15) {
    case 0:
    case 1:
        return launch_lo_nr<In, Out, Lk, Cl, 1>(ctx, a, U, F, clover);
    case 2:
        return launch_lo_nr<In, Out, Lk, Cl, 2>(ctx, a, U, F, clover);
    case 4:
        return launch_lo_nr<In, Out, Lk, Cl, 4>(ctx, a, U, F, clover);
    default:
        set_error("unsupported rhs register block %d (built: 1, 2, 4)", a.rhs_block & 15);
        return LMX_ERR_UNSUPPORTED;
    }
}

int launch_wilson_lo(lmx_context* ctx, const LoArgs& a) {
    if (ctx->V == 0 || a.nrhs == 0) return LMX_OK;
    const bool cl = a.clover != nullptr;
    const int V = (int)ctx->V;
    if (a.link_prec == LMX_F32 && a.spinor_prec == LMX_F32 && a.epi == EPI_NONE) {
        if (lds_f32(ctx, a.nrhs, cl)) return launch_lds_f32(ctx, a);
        if (hops_f32(ctx, a.nrhs, cl)) return launch_hops_f32(ctx, a);
    }
    if (a.link_prec == LMX_F32 && a.spinor_prec == LMX_F32)
        return launch_lo_sp<SpF32In, SpF32Out>(ctx, a, LinkF32{(const float2*)a.links, V},
                                               F32Clover{(const float2*)a.clover}, cl);
    if (a.link_prec == LMX_F16 && a.spinor_prec == LMX_F32)
        return launch_lo_sp<SpF32In, SpF32Out>(ctx, a, LinkF16{(const int4*)a.links, V},
                                               F16Clover{(const __half2*)a.clover}, cl);
    if (a.link_prec == LMX_F16 && a.spinor_prec == LMX_H16)
        return launch_lo_sp<SpH16In, SpH16Out>(ctx, a, LinkF16{(const int4*)a.links, V},
                                               F16Clover{(const __half2*)a.clover}, cl);
    set_error("unsupported precision pair (spinor %d, links %d)", a.spinor_prec, a.link_prec);
    return LMX_ERR_UNSUPPORTED;
}

}  // namespace lmx
