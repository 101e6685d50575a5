// wilson_hops.h -- the Wilson(-clover) stencil with the eight hops of a site
// on eight wavefronts (FP64 and FP32 fields).
//
// A workgroup of 512 work items owns 64 consecutive sites: lane i of every
// wavefront is site i, wavefront 2 mu the forward and 2 mu + 1 the backward
// hop of direction mu.  Each wavefront loads one neighbour spinor and one
// link, forms its half-spinor U P psi and leaves it in LDS; after one barrier
// wavefronts 0-5 each sum two of the site's twelve components over the eight
// hops, in the reference's order, and write them (results bit-identical to
// k_site's and k_stream's).  The clover planes' words are loaded once by all
// eight, an eighth each, and wait in LDS (read by each wavefront that needs
// them instead: 48^3 x 96 3850 us against 3500).  Several right-hand sides take their turns in the
// workgroup with the links kept in registers, the next one's spinors in
// flight while the last one's components are summed.
//
// Why: with the hops one after the other in one work item (k_site, k_stream)
// a site waits for nine loads in turn, at 230-256 VGPRs and one or two
// wavefronts per SIMD in FP64.  Here it waits for one, at four wavefronts per
// SIMD (a workgroup is two on each; 88 VGPRs in FP64, 120 with complex phases,
// 128 with the clover term, where D^dagger with p.Ap spills 12 of them and the
// complex-phase variants 8 and 13), at the price of 1.5 KB of LDS traffic per
// site and of the neighbours in t read again.  To keep those in L2 the blocks
// are ordered slab by slab (slab_order): an eighth of the 3-D volume, one XCD's
// share, for t = 0, 1, ... (lattice order instead: 174 against 148 us at 24^3 x
// 48, 3400 against 2650 us at 48^3 x 96; tiles in y and z, nontemporal loads of
// links and a walk over t within the workgroup were no faster).  Bound by the
// L2 misses that remain: 24^3 x 48 0.78 GB moved at 5.2 TB/s, 1.22x the fields
// themselves, with the clover term 1.09 GB at 5.3 TB/s (1.18x), 48^3 x 96 with
// it 23.8 GB at 6.7 TB/s (1.61x); the vector pipes issue a fifth of the time.
//
#pragma once

#include "wilson_kernels.h"

namespace lmx {

constexpr int kHopSites = kSlabSites;

// U P psi of one hop (the reference's half-spin order), the boundary phase
// applied where the neighbour wraps.
template <int MU, int PM, bool FWD, bool GP, typename R>
__device__ __forceinline__ void hop_product(cx<R> (&psi)[12], const cx<R> (&u)[9], bool w, const Geom& g,
                                            cx<R> (&o)[6]) {
    cx<R> h[6];
    if (GP) {
        if (w && !g.phase_one[MU]) {
            if (FWD)
                phase_spinor(psi, g.ph_re[MU], g.ph_im[MU]);
            else
                phase_spinor(psi, g.iph_re[MU], g.iph_im[MU]);
        }
    }
    half_project<PM, MU>(psi, h);
    if (!GP) neg_select(h, w && g.phase_neg[MU]);
    if (FWD)
        matvec_fwd(u, h, o);
    else
        matvec_bwd(u, h, o);
}

// Add one hop's half-spinor (h1, h2) of a colour to spins (0, 1) or (2, 3) of
// that colour's accumulator: the pair's share of reconstruct_add.
template <int PM, int MU, bool HIGH, typename R>
__device__ __forceinline__ void reconstruct_pair(cx<R>& a, cx<R>& b, cx<R> h1, cx<R> h2) {
    if (!HIGH) {
        a = cadd(a, h1);
        b = cadd(b, h2);
    } else if (MU == 0) {
        a = cadd(a, pmi<PM>(h2));
        b = cadd(b, pmi<PM>(h1));
    } else if (MU == 1) {
        a = cadd(a, pmr<PM>(h2));
        b = csub(b, pmr<PM>(h1));
    } else if (MU == 2) {
        a = cadd(a, pmi<PM>(h1));
        b = csub(b, pmi<PM>(h2));
    } else {
        a = csub(a, pmr<PM>(h1));
        b = csub(b, pmr<PM>(h2));
    }
}

// A complex number in LDS as one aligned word, so that a lane moves it whole.
template <typename R>
struct alignas(2 * sizeof(R)) LdsCx {
    R re, im;
    __device__ __forceinline__ LdsCx& operator=(cx<R> z) {
        using V2 = R __attribute__((ext_vector_type(2)));
        *reinterpret_cast<V2*>(this) = V2{z.re, z.im};
        return *this;
    }
    __device__ __forceinline__ operator cx<R>() const {
        using V2 = R __attribute__((ext_vector_type(2)));
        const V2 v = *reinterpret_cast<const V2*>(this);
        return mk<R>(v.x, v.y);
    }
};
// U P psi of each hop: [hop][2 colour + half-spin][site]; the clover planes
// take their place once they are summed.
template <typename R>
union HopBuf {
    LdsCx<R> hop[8][6][kHopSites];
    LdsCx<R> F[27][kHopSites];
    __device__ HopBuf() {}
};
// Wavefront W's share of the 27 clover words of the workgroup's sites: into
// registers before the hops are summed, into LDS after.
template <int W>
struct CloverShare {
    static constexpr int kFirst = W < 3 ? 4 * W : 3 * W + 3, kNum = W < 3 ? 4 : 3;
};
template <int W, typename R, class Cl>
__device__ __forceinline__ void ld_clover_share(const Cl& F, int V, int s, cx<R> (&f)[CloverShare<W>::kNum]) {
    ld_comps(F.p + (size_t)CloverShare<W>::kFirst * V, V, s, f);
}
template <int W, typename R>
__device__ __forceinline__ void put_clover_share(LdsCx<R> (&F)[27][kHopSites], int lane,
                                                 const cx<R> (&f)[CloverShare<W>::kNum]) {
#pragma unroll
    for (int k = 0; k < CloverShare<W>::kNum; ++k) F[CloverShare<W>::kFirst + k][lane] = f[k];
}
// Several fields alternate between two buffers, so that one barrier a field
// is enough: the products of a field overwrite what was summed two fields ago
// (one buffer and two barriers: four FP64 fields at 24^3 x 48 490 us against
// 456, twelve FP32 ones at 32^4 1249 against 1165).
template <typename R, int MODE, bool LOOP>
struct HopLds {
    HopBuf<R> b[LOOP ? 2 : 1];
    LdsCx<R> psi[MODE == MODE_CLOVER ? 12 : 1][kHopSites];  // the site's own spinor, for the clover term
};
// two components of the site's own spinor
template <typename R, typename T>
__device__ __forceinline__ void ld_own(const T* spin, int V, int ka, int kb, int s, cx<R> (&z)[2]) {
    using V2 = R __attribute__((ext_vector_type(2)));
    const V2 a = ld_sbase<V2>(spin + (size_t)ka * V, s), b = ld_sbase<V2>(spin + (size_t)kb * V, s);
    z[0] = mk<R>(a.x, a.y);
    z[1] = mk<R>(b.x, b.y);
}

template <int FPM, bool HIGH, typename R>
__device__ __forceinline__ void sum_hops(const LdsCx<R> (&hop)[8][6][kHopSites], int c, int lane, cx<R>& a, cx<R>& b) {
    a = mk<R>(R(0), R(0));
    b = a;
#define LMX_HOP_ADD(H, PM, MU) \
    reconstruct_pair<PM, MU, HIGH, R>(a, b, hop[H][2 * c][lane], hop[H][2 * c + 1][lane])
    LMX_HOP_ADD(0, FPM, 0);
    LMX_HOP_ADD(1, -FPM, 0);
    LMX_HOP_ADD(2, FPM, 1);
    LMX_HOP_ADD(3, -FPM, 1);
    LMX_HOP_ADD(4, FPM, 2);
    LMX_HOP_ADD(5, -FPM, 2);
    LMX_HOP_ADD(6, FPM, 3);
    LMX_HOP_ADD(7, -FPM, 3);
#undef LMX_HOP_ADD
}

// The clover term of colour C's spins (0, 1) or (2, 3): that pair's share of
// clover_add, in its order, from the site's own spinor in LDS.
template <int C, bool HIGH, int P, typename R>
__device__ __forceinline__ void clover_pair(const LdsCx<R> (&F)[27][kHopSites], const LdsCx<R> (&psi)[12][P], int lane,
                                            R coefficient, cx<R>& ra, cx<R>& rb) {
    cx<R> v1 = mk<R>(R(0), R(0)), v2 = v1;
    R d[6];
    cx<R> u[6][2];
#pragma unroll
    for (int pl = 0; pl < 6; ++pl) {
        const int q = 3 * pl + C;
        const cx<R> v = F[q / 2][lane];
        d[pl] = (q & 1) ? v.im : v.re;
        // the row's two off-diagonal entries, by their column: 0 and 1 of the other two
        constexpr int j0 = C == 0 ? 0 : (C == 1 ? 0 : 1), j1 = C == 0 ? 1 : 2;
        u[pl][0] = F[9 + 3 * pl + j0][lane];
        u[pl][1] = F[9 + 3 * pl + j1][lane];
    }
#pragma unroll
    for (int ic = 0; ic < 3; ++ic) {
        cx<R> f[6];
#pragma unroll
        for (int pl = 0; pl < 6; ++pl) {
            if (ic == C)
                f[pl] = mk<R>(R(0), d[pl]);
            else if (C < ic)
                f[pl] = u[pl][C == 0 ? ic - 1 : 1];
            else
                f[pl] = cneg(cconj(u[pl][C == 1 ? 0 : ic]));
        }
        const cx<R> f12 = f[0], f13 = f[1], f14 = f[2], f23 = f[3], f24 = f[4], f34 = f[5];
        if (!HIGH) {
            const cx<R> s1 = cadd(f12, f34), s3 = cadd(f14, f23);
            const cx<R> dp = mk<R>(-s1.im, s1.re), odp = mk<R>(-s3.im, s3.re);
            const cx<R> p1 = psi[ic][lane], p2 = psi[3 + ic][lane];
            v1 = cadd(v1, cadd(cmul(dp, p1), cmul(cadd(cadd(cneg(f13), odp), f24), p2)));
            v2 = cadd(v2, cadd(cmul(cneg(dp), p2), cmul(csub(cadd(f13, odp), f24), p1)));
        } else {
            const cx<R> s2 = csub(f12, f34), s4 = csub(f23, f14);
            const cx<R> dm = mk<R>(-s2.im, s2.re), odm = mk<R>(-s4.im, s4.re);
            const cx<R> p3 = psi[6 + ic][lane], p4 = psi[9 + ic][lane];
            v1 = cadd(v1, cadd(cmul(dm, p3), cmul(csub(cadd(cneg(f13), odm), f24), p4)));
            v2 = cadd(v2, cadd(cmul(cneg(dm), p4), cmul(cadd(cadd(f13, odm), f24), p3)));
        }
    }
    ra = cadd(ra, rmul(coefficient, v1));
    rb = cadd(rb, rmul(coefficient, v2));
}

template <class In, class Lk, class Out, class Cl>
struct HopArgs {
    Out out;
    In in;
    Lk U;
    Cl F;
    In aux;  // p of EPI_PAP
    typename In::R kappa, ccoef;
    int r0, r1;  // the workgroup's right-hand sides
    double* partials;
};

// Wavefront W's part of the workgroup (hop W; the sum of two components for W < 6).
template <int W, int FPM, int MODE, int EPI, bool GP, bool LOOP, class In, class Lk, class Out, class Cl>
__device__ __forceinline__ void hop_wave(const HopArgs<In, Lk, Out, Cl>& a, HopLds<typename In::R, MODE, LOOP>& sh,
                                         double (*pap)[kHopSites], const Geom& g, int s0, int lane, int end) {
    using R = typename In::R;
    constexpr int MU = W >> 1;
    constexpr bool FWD = (W & 1) == 0;
    constexpr int PM = FWD ? FPM : -FPM;
    // the summed components: colour c, spins (0, 1) or (2, 3)
    constexpr int c = W >> 1;
    constexpr bool kHigh = (W & 1) != 0;
    constexpr int ka = (kHigh ? 6 : 0) + c, kb = ka + 3;
    int s = s0 + lane;
    const bool live = s < end;
    if (!live) s = end - 1;  // a ragged last block: recompute, do not store
    int x[4];
    site_coords(s, g, x);
    bool w;
    const int t = FWD ? nbr_fwd(s, x, MU, g, w) : nbr_bwd(s, x, MU, g, w);
    cx<R> psi[12], u[9], own[2];
    const auto* spin = a.in.p + (size_t)a.r0 * 12 * g.V;
    ld_comps(a.U.p + (size_t)MU * 9 * g.V, g.V, FWD ? s : t, u);
    ld_comps(spin, g.V, t, psi);
    if constexpr (W < 6 && MODE != MODE_DONLY) ld_own(spin, g.V, ka, kb, s, own);
    const int r1 = LOOP ? a.r1 : a.r0 + 1;
    for (int r = a.r0; r < r1; ++r) {
        cx<R> o[6], mine[2];
        HopBuf<R>& buf = sh.b[LOOP ? (r - a.r0) & 1 : 0];
        hop_product<MU, PM, FWD, GP>(psi, u, w, g, o);
#pragma unroll
        for (int k = 0; k < 6; ++k) buf.hop[W][k][lane] = o[k];
        if constexpr (W < 6 && MODE != MODE_DONLY) {
            mine[0] = own[0];
            mine[1] = own[1];
            if constexpr (MODE == MODE_CLOVER) {
                sh.psi[ka][lane] = mine[0];
                sh.psi[kb][lane] = mine[1];
            }
        }
        if (LOOP && r + 1 < r1) {  // the next field's, in flight while this one is summed
            spin += (size_t)12 * g.V;
            ld_comps(spin, g.V, t, psi);
            if constexpr (W < 6 && MODE != MODE_DONLY) ld_own(spin, g.V, ka, kb, s, own);
        }
        cx<R> f[MODE == MODE_CLOVER ? CloverShare<W>::kNum : 1];
        if constexpr (MODE == MODE_CLOVER) ld_clover_share<W>(a.F, g.V, s, f);
        __syncthreads();
        cx<R> ra, rb;
        if constexpr (W < 6) sum_hops<FPM, kHigh>(buf.hop, c, lane, ra, rb);
        if constexpr (MODE == MODE_CLOVER) {
            __syncthreads();
            put_clover_share<W>(buf.F, lane, f);
            __syncthreads();
        }
        if constexpr (W < 6) {
            if (MODE == MODE_DONLY) {
                const R half = R(1) / R(2);
                ra = cadd(mk<R>(R(0), R(0)), rmul(half, ra));
                rb = cadd(mk<R>(R(0), R(0)), rmul(half, rb));
            } else {
                ra = cadd(mine[0], rmul(-a.kappa, ra));
                rb = cadd(mine[1], rmul(-a.kappa, rb));
                if constexpr (MODE == MODE_CLOVER)
                    clover_pair<c, kHigh>(buf.F, sh.psi, lane, a.ccoef, ra, rb);
            }
            if (live) {
                a.out.st1(r, ka, s, ra);
                a.out.st1(r, kb, s, rb);
            }
            if constexpr (EPI == EPI_PAP) {
                // the terms of Re sum conj(p) Ap, summed per site in kernel_dot_D order by wavefront 7
                const cx<R> pa = a.aux.ld1(r, ka, s), pb = a.aux.ld1(r, kb, s);
                pap[ka][lane] = live ? cmul(cconj(pa), ra).re : 0.0;
                pap[kb][lane] = live ? cmul(cconj(pb), rb).re : 0.0;
            }
        }
        if (EPI == EPI_PAP) __syncthreads();
        if constexpr (EPI == EPI_PAP && W == 7) {
            double v = 0.0;
#pragma unroll
            for (int k = 0; k < 12; ++k) v = v + pap[k][lane];
            v = wave_halve(v);
            if (lane == 0) a.partials[s0 / kHopSites] = v;
        }
    }
}

// Wavefronts per SIMD to compile for: one field, four in FP64 (its registers;
// LDS would admit six without the clover term) and six in FP32; several, where
// the next field's operands stay in registers across the sum, two and four
// (FP64 at four: spills, 24^3 x 48 x 4 597 us against 456).
template <typename R>
constexpr int hop_waves(bool loop) {
    return sizeof(R) == 8 ? (loop ? 2 : 4) : (loop ? 4 : 6);
}

// Block lb is RHS group lb % ngroups (per fields each) of site block lb / ngroups.
template <class In, class Lk, class Out, class Cl, int FPM, int MODE, int EPI, bool GP, bool LOOP>
__global__ void __launch_bounds__(512, hop_waves<typename In::R>(LOOP))
    k_hops(Out out, In in, Lk U, Cl F, In aux, Geom g, double kappa_d, double ccoef_d, int ngroups, int per, int nrhs,
           int slab, EpiArgs epi) {
    using R = typename In::R;
    if (epi.st != nullptr && epi.st->done) return;
    if (epi.gate != nullptr && *epi.gate == 0) return;
    static_assert(!LOOP || (MODE != MODE_CLOVER && EPI == EPI_NONE), "one barrier a field");
    __shared__ HopLds<R, MODE, LOOP> sh;
    __shared__ double pap[EPI == EPI_PAP ? 12 : 1][kHopSites];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int r0 = lb % ngroups * per;
    int s0, end;
    slab_block(lb / ngroups, slab, g, s0, end);
    const HopArgs<In, Lk, Out, Cl> a{out, in, U, F, aux, R(kappa_d), R(ccoef_d), r0, min(r0 + per, nrhs), epi.partials};
    switch (wave) {
#define LMX_HOP_WAVE(W)                                                                       \
    case W:                                                                                   \
        hop_wave<W, FPM, MODE, EPI, GP, LOOP, In, Lk, Out, Cl>(a, sh, pap, g, s0, lane, end); \
        break
        LMX_HOP_WAVE(0);
        LMX_HOP_WAVE(1);
        LMX_HOP_WAVE(2);
        LMX_HOP_WAVE(3);
        LMX_HOP_WAVE(4);
        LMX_HOP_WAVE(5);
        LMX_HOP_WAVE(6);
        LMX_HOP_WAVE(7);
#undef LMX_HOP_WAVE
    }
}

// Launch over nrhs fields, up to per_hint of them in a workgroup; flags LMX_DAGGER / LMX_DONLY.  EPI_PAP (on
// D^dagger, one field): partials gets one sum per 64 consecutive sites.
template <class In, class Lk, class Out, class Cl, int EPI>
int launch_hops(lmx_context* ctx, Out out, In in, Lk U, Cl F, In aux, double kappa, double ccoef, int nrhs, int per_hint,
                int flags, bool clover, const EpiArgs& epi) {
    const bool dag = (flags & LMX_DAGGER) != 0, donly = (flags & LMX_DONLY) != 0;
    const Geom& g = ctx->g;
    // the sums of EPI_PAP need whole blocks
    const SlabOrder so = slab_order(g, EPI == EPI_PAP, 24 * sizeof(typename In::R));
    // clover fields one by one: a loop over them would hold the planes' entries too
    const int per = clover || EPI != EPI_NONE ? 1 : std::min(std::max(per_hint, 1), nrhs);
    const int ngroups = (nrhs + per - 1) / per;
    const long nb = so.blocks * ngroups;
    LMX_CHECK(nb < (1L << 31), LMX_ERR_ARG, "too many right-hand sides (%d)", nrhs);
#define LMX_HOPS(FPM, MODE, GP)                                                                                     \
    do {                                                                                                            \
        if constexpr (EPI == EPI_NONE && MODE != MODE_CLOVER) {                                                     \
            if (per > 1) {                                                                                          \
                hipLaunchKernelGGL((k_hops<In, Lk, Out, Cl, FPM, MODE, EPI, GP, true>), dim3((unsigned)nb), dim3(512), 0, \
                                   ctx->stream, out, in, U, F, aux, g, kappa, ccoef, ngroups, per, nrhs, so.slab, epi); \
                break;                                                                                              \
            }                                                                                                       \
        }                                                                                                           \
        hipLaunchKernelGGL((k_hops<In, Lk, Out, Cl, FPM, MODE, EPI, GP, false>), dim3((unsigned)nb), dim3(512), 0,  \
                           ctx->stream, out, in, U, F, aux, g, kappa, ccoef, ngroups, per, nrhs, so.slab, epi);     \
    } while (0)
#define LMX_HOPS_GP(FPM, MODE)            \
    do {                                  \
        if (g.general)                    \
            LMX_HOPS(FPM, MODE, true);    \
        else                              \
            LMX_HOPS(FPM, MODE, false);   \
    } while (0)
#define LMX_HOPS_MODE(FPM)                          \
    do {                                            \
        if (clover)                                 \
            LMX_HOPS_GP(FPM, MODE_CLOVER);          \
        else                                        \
            LMX_HOPS_GP(FPM, MODE_WILSON);          \
    } while (0)
    if constexpr (EPI == EPI_PAP) {
        LMX_CHECK(dag && !donly && nrhs == 1, LMX_ERR_UNSUPPORTED, "fused p.Ap is built for one field on D^dagger");
        LMX_HOPS_MODE(1);
    } else if (donly) {
        if (dag)
            LMX_HOPS_GP(1, MODE_DONLY);
        else
            LMX_HOPS_GP(-1, MODE_DONLY);
    } else if (dag) {
        LMX_HOPS_MODE(1);
    } else {
        LMX_HOPS_MODE(-1);
    }
#undef LMX_HOPS_MODE
#undef LMX_HOPS_GP
#undef LMX_HOPS
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

// ---------------------------------------------------------------------------
// The same stencil on the reference's own storage (LatticeMatrix.A: component
// spin*3 + colour of padded site p at p*12 + k; halo not read, only core sites
// written).  A wavefront loads its 64 neighbours' spinors as they lie, 16 (8)
// consecutive bytes per lane across a row of sites, and turns them to one site
// per lane in its own 6 (3) KB of LDS, 32 sites at a time, projecting colour by
// colour as it reads; the results leave the same way.  One site per lane
// straight from memory touches a line per lane and load, twelve times over, and
// takes the hops in turn: 24^3 x 48 276 us against 168 here, in ComplexF32
// 126 against 89, 32^4 392 against 288.  Bound by L2 misses, as above.
// ---------------------------------------------------------------------------
struct PadGeom {
    int PS[4];  // padded strides (1, P1, P1 P2, P1 P2 P3)
    int nw;
    long Vp;    // padded volume
};
constexpr int kPadPitch = kHopSites + 1;  // a site's twelve components lie in different banks

template <typename R>
struct PadLds {
    HopBuf<R> b;
    LdsCx<R> psi[12][kPadPitch];  // the site's own spinor, then the results
    int site[kHopSites];          // padded index of the workgroup's sites
};

// N consecutive components of a site as one word (16 bytes; 8 for a FP32 array
// that is not 16-byte aligned)
template <typename E, int N>
struct alignas(N * sizeof(E)) PadWord {
    E e[N];
};

template <typename E, class Lk, class Cl>
struct PadArgs {
    E* out;
    const E* in;
    Lk U;
    Cl F;
    double kappa, ccoef;
};

template <int W, int FPM, int MODE, bool GP, int N, typename R, typename E, class Lk, class Cl>
__device__ __forceinline__ void pad_wave(const PadArgs<E, Lk, Cl>& a, PadLds<R>& sh, const Geom& g, const PadGeom& pg,
                                         int s0, int lane, int end) {
    constexpr int MU = W >> 1;
    constexpr bool FWD = (W & 1) == 0;
    constexpr int PM = FWD ? FPM : -FPM;
    constexpr int c = W >> 1;
    constexpr bool kHigh = (W & 1) != 0;
    constexpr int ka = (kHigh ? 6 : 0) + c, kb = ka + 3;
    int s = s0 + lane;
    if (s >= end) s = end - 1;
    int x[4];
    site_coords(s, g, x);
    bool w;
    const int t = FWD ? nbr_fwd(s, x, MU, g, w) : nbr_bwd(s, x, MU, g, w);
    const int sp = (x[0] + pg.nw) + pg.PS[1] * (x[1] + pg.nw) + pg.PS[2] * (x[2] + pg.nw) + pg.PS[3] * (x[3] + pg.nw);
    const int step = FWD ? (w ? -(g.L[MU] - 1) : 1) : (w ? g.L[MU] - 1 : -1);
    const int tp = sp + step * pg.PS[MU];
    // word 64 j + lane of the 64 spinors end to end, M words a site
    using Word = PadWord<E, N>;
    constexpr int M = 12 / N;
    Word land[M];
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const int e = 64 * j + lane, i = e / M;
        land[j] = reinterpret_cast<const Word*>(a.in)[(long)__shfl(tp, i, 64) * M + (e - M * i)];
    }
    cx<R> u[9];
    ld_comps(a.U.p + (size_t)MU * 9 * g.V, g.V, FWD ? s : t, u);
    if constexpr (W == 0) sh.site[lane] = sp;
    LdsCx<R>* mine = &sh.b.hop[W][0][0];
    cx<R> h[6];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int j = 0; j < M / 2; ++j)
#pragma unroll
            for (int n = 0; n < N; ++n) {
                const E v = land[M / 2 * half + j].e[n];
                mine[N * (64 * j + lane) + n] = mk<R>(v.x, v.y);
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if ((lane >> 5) == half) {
            const LdsCx<R>* q = mine + 12 * (lane & 31);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                cx<R> p[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    p[d] = q[3 * d + k];
                    if (GP && w && !g.phase_one[MU])
                        p[d] = cmul(p[d], FWD ? mk<R>(R(g.ph_re[MU]), R(g.ph_im[MU]))
                                              : mk<R>(R(g.iph_re[MU]), R(g.iph_im[MU])));
                }
                half_project1<PM, MU>(p[0], p[1], p[2], p[3], h[2 * k], h[2 * k + 1]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (!GP) neg_select(h, w && g.phase_neg[MU]);
    cx<R> o[6];
    if (FWD)
        matvec_fwd(u, h, o);
    else
        matvec_bwd(u, h, o);
#pragma unroll
    for (int k = 0; k < 6; ++k) sh.b.hop[W][k][lane] = o[k];
    cx<R> f[MODE == MODE_CLOVER ? CloverShare<W>::kNum : 1];
    if constexpr (MODE == MODE_CLOVER) ld_clover_share<W>(a.F, g.V, s, f);
    __syncthreads();
    cx<R> ra, rb;
    if constexpr (W < 6) sum_hops<FPM, kHigh>(sh.b.hop, c, lane, ra, rb);
    if constexpr (MODE == MODE_CLOVER) {
        __syncthreads();
        put_clover_share<W>(sh.b.F, lane, f);
        __syncthreads();
    }
    if constexpr (W < 6) {
        const R kappa = R(a.kappa);
        if (MODE == MODE_DONLY) {
            const R half = R(1) / R(2);
            ra = cadd(mk<R>(R(0), R(0)), rmul(half, ra));
            rb = cadd(mk<R>(R(0), R(0)), rmul(half, rb));
        } else {
            ra = cadd(cx<R>(sh.psi[ka][lane]), rmul(-kappa, ra));
            rb = cadd(cx<R>(sh.psi[kb][lane]), rmul(-kappa, rb));
            if constexpr (MODE == MODE_CLOVER)
                clover_pair<c, kHigh>(sh.b.F, sh.psi, lane, R(a.ccoef), ra, rb);
        }
    }
    __syncthreads();  // the own spinors have been read: results take their place
    if constexpr (W < 6) {
        sh.psi[ka][lane] = ra;
        sh.psi[kb][lane] = rb;
    }
}

template <int FPM, int MODE, bool GP, int N, typename E, class Lk, class Cl>
__global__ void __launch_bounds__(512, sizeof(E) == 16 ? 4 : 6)
    k_hops_pad(E* __restrict__ C, const E* __restrict__ psi, Lk U, Cl F, Geom g, PadGeom pg, double kappa,
               double ccoef, int nrhs, int slab) {
    using R = typename std::conditional<std::is_same<E, float2>::value, float, double>::type;
    __shared__ PadLds<R> sh;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const long field = (long)(lb % nrhs) * pg.Vp * 12;
    int s0, end;
    slab_block(lb / nrhs, slab, g, s0, end);
    const PadArgs<E, Lk, Cl> a{C + field, psi + field, U, F, kappa, ccoef};
    const int n = min(kHopSites, end - s0);
    using Word = PadWord<E, N>;
    constexpr int M = 12 / N;
    if (MODE != MODE_DONLY) {  // the sites' own spinors, word after word
        for (int e = threadIdx.x; e < M * n; e += 512) {
            const int i = e / M, k = N * (e - M * i);
            int x[4];
            site_coords(s0 + i, g, x);
            const long sp = (x[0] + pg.nw) + (long)pg.PS[1] * (x[1] + pg.nw) + (long)pg.PS[2] * (x[2] + pg.nw) +
                            (long)pg.PS[3] * (x[3] + pg.nw);
            const Word v = reinterpret_cast<const Word*>(a.in)[sp * M + k / N];
#pragma unroll
            for (int c = 0; c < N; ++c) sh.psi[k + c][i] = mk<R>(v.e[c].x, v.e[c].y);
        }
    }
    switch (wave) {
#define LMX_PAD_WAVE(W)                                                                    \
    case W:                                                                                \
        pad_wave<W, FPM, MODE, GP, N, R, E, Lk, Cl>(a, sh, g, pg, s0, lane, end);          \
        break
        LMX_PAD_WAVE(0);
        LMX_PAD_WAVE(1);
        LMX_PAD_WAVE(2);
        LMX_PAD_WAVE(3);
        LMX_PAD_WAVE(4);
        LMX_PAD_WAVE(5);
        LMX_PAD_WAVE(6);
        LMX_PAD_WAVE(7);
#undef LMX_PAD_WAVE
    }
    __syncthreads();
    for (int e = threadIdx.x; e < M * n; e += 512) {
        const int i = e / M, k = N * (e - M * i);
        Word v;
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const cx<R> z = sh.psi[k + c][i];
            v.e[c].x = z.re;
            v.e[c].y = z.im;
        }
        reinterpret_cast<Word*>(a.out)[(long)sh.site[i] * M + k / N] = v;
    }
}

template <int N, typename E, class Lk, class Cl>
int launch_hops_pad(lmx_context* ctx, Lk l, Cl F, bool clover, double kappa, double csw, E* C, const E* psi, int nw,
                    int nrhs, int flags) {
    if (ctx->V == 0 || nrhs == 0) return LMX_OK;
    const Geom& g = ctx->g;
    PadGeom pg;
    pg.nw = nw;
    long st = 1;
    for (int d = 0; d < 4; ++d) {
        pg.PS[d] = (int)st;
        st *= g.L[d] + 2 * nw;
    }
    pg.Vp = st;
    LMX_CHECK(st < (1L << 31), LMX_ERR_ARG, "padded volume too large");
    const double ccoef = (-kappa) * csw;
    const SlabOrder so = slab_order(g, false, 12 * sizeof(E));
    const long nb = so.blocks * nrhs;
    LMX_CHECK(nb < (1L << 31), LMX_ERR_ARG, "too many right-hand sides (%d)", nrhs);
    const bool dag = (flags & LMX_DAGGER) != 0, donly = (flags & LMX_DONLY) != 0;
#define LMX_PAD(FPM, MODE)                                                                                       \
    do {                                                                                                         \
        if (g.general)                                                                                           \
            hipLaunchKernelGGL((k_hops_pad<FPM, MODE, true, N, E, Lk, Cl>), dim3((unsigned)nb), dim3(512), 0,       \
                               ctx->stream, C, psi, l, F, g, pg, kappa, ccoef, nrhs, so.slab);                   \
        else                                                                                                     \
            hipLaunchKernelGGL((k_hops_pad<FPM, MODE, false, N, E, Lk, Cl>), dim3((unsigned)nb), dim3(512), 0,      \
                               ctx->stream, C, psi, l, F, g, pg, kappa, ccoef, nrhs, so.slab);                   \
    } while (0)
    if (donly) {
        if (dag)
            LMX_PAD(1, MODE_DONLY);
        else
            LMX_PAD(-1, MODE_DONLY);
    } else if (clover) {
        if (dag)
            LMX_PAD(1, MODE_CLOVER);
        else
            LMX_PAD(-1, MODE_CLOVER);
    } else {
        if (dag)
            LMX_PAD(1, MODE_WILSON);
        else
            LMX_PAD(-1, MODE_WILSON);
    }
#undef LMX_PAD
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

}  // namespace lmx
