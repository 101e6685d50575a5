// force.hip -- hand-written adjoint of the Wilson hopping term (the fermion
// force) and the traceless anti-Hermitian projection.
//
// Link cotangent, per site x and direction mu (row r, column c):
//   dU_mu(x)[r,c] += coefficient * ( sum_k P-(dres(x))_r,k conj(P-(psi(x+mu))_c,k)
//                                  + sum_k P+(psi(x))_r,k  conj(P+(dres(x+mu))_c,k) )
// with P-/P+ the half-spin projections of (1 -+ gamma_mu): the Enzyme reverse
// rule kernel _kernel_wilson_link_pullback! (ext/AD/WilsonDiracOperator.jl:62-91)
// and _wilson_halfspin_link_pullback_direction3!/_row3!
// (src/Operators/WilsonDiracOperator.jl:354-410), in its operation order.
// Values at x+mu carry the spinor boundary phase, as the reference's
// set_halo! of both fields does.
#include "lmx_internal.h"

namespace lmx {

template <int MU>
__device__ __forceinline__ void pullback_mu(double2* __restrict__ dU, const double2* __restrict__ dres,
                                            const double2* __restrict__ psi, const Geom& g, int s, double coefficient) {
    int x[4];
    site_coords(s, g, x);
    bool w;
    const int sp = nbr_fwd(s, x, MU, g, w);
    const bool ph = w && !g.phase_one[MU];
    cx<double> plus_psi[6], minus_dres[6], dplus[6], mpsi[6];
    cx<double> z[12];
    ld_comps(psi, g.V, sp, z);
    if (ph) phase_spinor(z, g.ph_re[MU], g.ph_im[MU]);
    half_project<-1, MU>(z, plus_psi);
    ld_comps(dres, g.V, sp, z);
    if (ph) phase_spinor(z, g.ph_re[MU], g.ph_im[MU]);
    half_project<1, MU>(z, minus_dres);
    ld_comps(dres, g.V, s, z);
    half_project<-1, MU>(z, dplus);
    ld_comps(psi, g.V, s, z);
    half_project<1, MU>(z, mpsi);
#pragma unroll
    for (int row = 0; row < 3; ++row) {
#pragma unroll
        for (int col = 0; col < 3; ++col) {
            cx<double> v = cmul(dplus[2 * row], cconj(plus_psi[2 * col]));
            v = cadd(v, cmul(dplus[2 * row + 1], cconj(plus_psi[2 * col + 1])));
            v = cadd(v, cmul(mpsi[2 * row], cconj(minus_dres[2 * col])));
            v = cadd(v, cmul(mpsi[2 * row + 1], cconj(minus_dres[2 * col + 1])));
            const size_t i = (size_t)(MU * 9 + row * 3 + col) * g.V + s;
            double2 o = dU[i];
            cx<double> nv = cadd(mk<double>(o.x, o.y), rmul(coefficient, v));
            dU[i] = make_double2(nv.re, nv.im);
        }
    }
}

// A wavefront of a workgroup takes one direction of the workgroup's 64 sites,
// blocks in the stencil's slab order: 126 registers and four wavefronts per
// SIMD, where one work item for all four directions held two own spinors
// besides two neighbours' (240, two).  Bound by its 384 B read and 1152 B read
// and written per site: 16^3 x 32 49 us (4.1 TB/s) against 55.
__global__ void __launch_bounds__(256, 3) k_pullback(double2* __restrict__ dU, const double2* __restrict__ dres,
                                                     const double2* __restrict__ psi, Geom g, double coefficient,
                                                     int slab) {
    int s0, end;
    slab_block(xcd_block(blockIdx.x, gridDim.x), slab, g, s0, end);
    const int s = s0 + (threadIdx.x & 63);
    if (s >= end) return;
    switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
    case 0:
        pullback_mu<0>(dU, dres, psi, g, s, coefficient);
        break;
    case 1:
        pullback_mu<1>(dU, dres, psi, g, s, coefficient);
        break;
    case 2:
        pullback_mu<2>(dU, dres, psi, g, s, coefficient);
        break;
    default:
        pullback_mu<3>(dU, dres, psi, g, s, coefficient);
    }
}

// F = TA(U G^dagger): M[i][j] = muladdmulti over k of U[i][k] conj(G[j][k]),
// then kernel_traceless_antihermitian! NC=3 (src/TA/TA.jl:68-116).
__global__ void __launch_bounds__(256) k_ta_project(double2* __restrict__ F, const double2* __restrict__ U,
                                                    const double2* __restrict__ G, int V) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= V) return;
    for (int mu = 0; mu < 4; ++mu) {
        cx<double> u[9], gg[9], m[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            double2 a = U[(long)(mu * 9 + k) * V + s], b = G[(long)(mu * 9 + k) * V + s];
            u[k] = mk<double>(a.x, a.y);
            gg[k] = mk<double>(b.x, b.y);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                m[3 * i + j] = muladdmulti(u[3 * i], cconj(gg[3 * j]), u[3 * i + 1], cconj(gg[3 * j + 1]),
                                           u[3 * i + 2], cconj(gg[3 * j + 2]));
        const double fac13 = 1.0 / 3.0;
        const double tri = fac13 * ((m[0].im + m[4].im) + m[8].im);
        cx<double> o[9];
        o[0] = mk<double>(0.0, m[0].im - tri);
        o[4] = mk<double>(0.0, m[4].im - tri);
        o[8] = mk<double>(0.0, m[8].im - tri);
        cx<double> x12 = csub(m[1], cconj(m[3]));
        cx<double> x13 = csub(m[2], cconj(m[6]));
        cx<double> x23 = csub(m[5], cconj(m[7]));
        o[1] = rmul(0.5, x12);
        o[2] = rmul(0.5, x13);
        o[5] = rmul(0.5, x23);
        o[3] = rmul(0.5, cneg(cconj(x12)));
        o[6] = rmul(0.5, cneg(cconj(x13)));
        o[7] = rmul(0.5, cneg(cconj(x23)));
#pragma unroll
        for (int k = 0; k < 9; ++k) F[(long)(mu * 9 + k) * V + s] = make_double2(o[k].re, o[k].im);
    }
}

int launch_pullback_f64(lmx_context* ctx, double2* dU, const double2* dres, const double2* psi, double coefficient) {
    if (ctx->V == 0) return LMX_OK;
    const SlabOrder so = slab_order(ctx->g, false, 12 * sizeof(double2));
    hipLaunchKernelGGL(k_pullback, dim3((unsigned)so.blocks), dim3(256), 0, ctx->stream, dU, dres, psi, ctx->g,
                       coefficient, so.slab);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

int launch_ta_project(lmx_context* ctx, double2* F, const double2* U, const double2* G) {
    if (ctx->V == 0) return LMX_OK;
    hipLaunchKernelGGL(k_ta_project, dim3(nblocks(ctx->V)), dim3(256), 0, ctx->stream, F, U, G, (int)ctx->V);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

// ---------------------------------------------------------------------------
// Wilson-clover link pullback (wilson_clover_link_pullback!,
// src/Operators/WilsonCloverPullback.jl:349-389): the hopping part above plus
//   1. the field-strength cotangent per plane
//      dF[c][ic] += coefficient * sum_out dres[c,out] conj(sum_in g[out,in] psi[ic,in])
//      with g = gamma_mu gamma_nu (_kernel_clover_field_cotangent_plane!, :102-119);
//   2. its chain rule through F = (Q - Q^dagger)/8 and the four leaves of Q
//      onto the links (_kernel_clover_links_pullback!, :236-280): for each link
//      and each occurrence K in a leaf, with dQ = (dF - dF^dagger)/8 at the
//      leaf's anchor, left^dagger dQ right^dagger, or right dQ^dagger left for
//      an adjointed factor.
// Matrix products are plain complex arithmetic summed left to right; the
// operation order follows the reference's loops (planes 12..34, leaves,
// occurrences 1..4).
// ---------------------------------------------------------------------------

__device__ __forceinline__ void mat_mul_plain(const cx<double> A[9], const cx<double> B[9], cx<double> out[9]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            out[3 * i + j] =
                cadd(cadd(cmul(A[3 * i], B[j]), cmul(A[3 * i + 1], B[3 + j])), cmul(A[3 * i + 2], B[6 + j]));
}
__device__ __forceinline__ void add9(cx<double> (&a)[9], const cx<double> (&b)[9]) {
#pragma unroll
    for (int k = 0; k < 9; ++k) a[k] = cadd(a[k], b[k]);
}
__device__ __forceinline__ void mat_dag(const cx<double> A[9], cx<double> out[9]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) out[3 * i + j] = cconj(A[3 * j + i]);
}

// Row o of gamma_mu gamma_nu in the chiral basis (src/Operators/Operators.jl:44-67)
// has one entry, a power of i: its column and that power.
struct GammaEntry {
    int col, pow;
};
constexpr GammaEntry gamma_entry(int mu, int row) {
    constexpr int col[4][4] = {{3, 2, 1, 0}, {3, 2, 1, 0}, {2, 3, 0, 1}, {2, 3, 0, 1}};
    constexpr int pw[4][4] = {{3, 3, 1, 1}, {2, 0, 0, 2}, {3, 1, 1, 3}, {2, 2, 2, 2}};
    return {col[mu][row], pw[mu][row]};
}
constexpr GammaEntry gamma_product_entry(int mu, int nu, int row) {
    const GammaEntry a = gamma_entry(mu, row), b = gamma_entry(nu, a.col);
    return {b.col, (a.pow + b.pow) & 3};
}
template <int POW>
__device__ __forceinline__ cx<double> i_pow(cx<double> z) {
    return POW == 0 ? z : POW == 1 ? mk<double>(-z.im, z.re) : POW == 2 ? cneg(z) : mk<double>(z.im, -z.re);
}

// dF[c][ic] of plane (MU, NU): coefficient * sum_out dres[c,out] conj(sum_in g[out,in] psi[ic,in])
template <int MU, int NU, int O>
__device__ __forceinline__ void cotangent_add(const cx<double> d[12], const cx<double> p[12], cx<double> f[9]) {
    constexpr GammaEntry e = gamma_product_entry(MU, NU, O);
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int ic = 0; ic < 3; ++ic)
            f[3 * c + ic] = cadd(f[3 * c + ic], cmul(d[O * 3 + c], cconj(i_pow<e.pow>(p[e.col * 3 + ic]))));
}
template <int PL, int MU, int NU>
__device__ __forceinline__ void cotangent_plane(double2* __restrict__ dQ, cx<double> (&d)[12], const cx<double> p[12],
                                                int s, int V, double coefficient) {
    // the planes three by three: the products of all interleaved spill
    if (PL == 3) {
#pragma unroll
        for (int k = 0; k < 12; ++k) asm volatile("" : "+v"(d[k].re), "+v"(d[k].im)::"memory");
    }
    cx<double> f[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k] = mk<double>(0.0, 0.0);
    cotangent_add<MU, NU, 0>(d, p, f);
    cotangent_add<MU, NU, 1>(d, p, f);
    cotangent_add<MU, NU, 2>(d, p, f);
    cotangent_add<MU, NU, 3>(d, p, f);
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k] = rmul(coefficient, f[k]);
    double2* q = dQ + (size_t)PL * 5 * V;
    // (re - re is zero, or the NaN of an infinite real part, which the imaginary part carries on)
    const auto diag = [](cx<double> z) { return 0.125 * (z.im + z.im) + (z.re - z.re); };
    const double d0 = diag(f[0]), d1 = diag(f[4]), d2 = diag(f[8]);
    const cx<double> u0 = rmul(0.125, csub(f[1], cconj(f[3]))), u1 = rmul(0.125, csub(f[2], cconj(f[6]))),
                     u2 = rmul(0.125, csub(f[5], cconj(f[7])));
    q[s] = make_double2(d0, d1);
    q[(size_t)V + s] = make_double2(d2, 0.0);
    q[(size_t)2 * V + s] = make_double2(u0.re, u0.im);
    q[(size_t)3 * V + s] = make_double2(u1.re, u1.im);
    q[(size_t)4 * V + s] = make_double2(u2.re, u2.im);
}

// dQ = (dF - dF^dagger) / 8 of the six planes.  It is anti-Hermitian exactly
// (the differences negate and the sums commute), so five words per plane hold
// it: the three imaginary diagonals and the upper entries.  That is all the
// links' chain rule reads; the products with gamma_mu gamma_nu are one term
// each.  Bound by its 384 B read and 480 B written per site: 16^3 x 32 in
// 21 us, against 17 + 59 us for a zero fill and full planes read and written.
__global__ void __launch_bounds__(256) k_clover_cotangent(double2* __restrict__ dQ, const double2* __restrict__ dres,
                                                          const double2* __restrict__ psi, int V, double coefficient) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= V) return;
    cx<double> d[12], p[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        double2 a = dres[(long)k * V + s], b = psi[(long)k * V + s];
        d[k] = mk<double>(a.x, a.y);
        p[k] = mk<double>(b.x, b.y);
    }
    cotangent_plane<0, 0, 1>(dQ, d, p, s, V, coefficient);
    cotangent_plane<1, 0, 2>(dQ, d, p, s, V, coefficient);
    cotangent_plane<2, 0, 3>(dQ, d, p, s, V, coefficient);
    cotangent_plane<3, 1, 2>(dQ, d, p, s, V, coefficient);
    cotangent_plane<4, 1, 3>(dQ, d, p, s, V, coefficient);
    cotangent_plane<5, 2, 3>(dQ, d, p, s, V, coefficient);
}

__device__ __forceinline__ void ld_link(const double2* U, int V, int mu, int s, bool dag, cx<double> (&u)[9]) {
    cx<double> v[9];
    ld_comps(U + (size_t)mu * 9 * V, V, s, v);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) u[3 * i + j] = dag ? cconj(v[3 * j + i]) : v[3 * i + j];
}
// dQ of plane pl at s, or its adjoint (exactly -dQ)
template <bool DAG>
__device__ __forceinline__ void ld_dq(const double2* dQ, int V, int pl, int s, cx<double> q[9]) {
    const double2* a = dQ + (size_t)pl * 5 * V;
    const double2 d01 = ldv(a, s), d2 = ldv(a + (size_t)V, s), u0 = ldv(a + (size_t)2 * V, s),
                  u1 = ldv(a + (size_t)3 * V, s), u2 = ldv(a + (size_t)4 * V, s);
    q[0] = mk<double>(0.0, d01.x);
    q[4] = mk<double>(0.0, d01.y);
    q[8] = mk<double>(0.0, d2.x);
    q[1] = mk<double>(u0.x, u0.y);
    q[2] = mk<double>(u1.x, u1.y);
    q[5] = mk<double>(u2.x, u2.y);
    q[3] = cneg(cconj(q[1]));
    q[6] = cneg(cconj(q[2]));
    q[7] = cneg(cconj(q[5]));
    if (DAG) {
#pragma unroll
        for (int k = 0; k < 9; ++k) q[k] = cneg(q[k]);
    }
}
// keep a matrix in registers here: the loads that follow are not hoisted above it
__device__ __forceinline__ void pin9(cx<double> (&a)[9]) {
#pragma unroll
    for (int k = 0; k < 9; ++k) asm volatile("" : "+v"(a[k].re), "+v"(a[k].im)::"memory");
}

// The terms of one plaquette loop through a link L at y: L A B C (DAG false)
// or L^dagger A B C, the leaves of the plane being the loop begun at its four
// corners.  Begun at L the cotangent enters before L (site s0), at C before C
// (s3), at B before B (s2), at A before A (s1); with X Y the factors to its
// left and right in the leaf, the term is X^dagger dQ Y^dagger, or
// Y dQ^dagger X.  Links are loaded where they are used, so that few matrices
// are live at once.
template <bool DAG, bool DA, bool DB, bool DC>
struct Plaquette {
    const double2 *U, *dQ;
    int V, pl, mA, sA, mB, sB, mC, sC, s0, s1, s2, s3;

    // (the pointer is made opaque, or a link that another term needs again would be kept, spilled, instead)
    __device__ __forceinline__ void lnk(int mu, int s, bool dag, cx<double> (&u)[9]) const {
        const double2* p = U;
        asm volatile("" : "+s"(p));
        ld_link(p, V, mu, s, dag, u);
    }
    __device__ __forceinline__ void link_b(cx<double> (&B)[9]) const { lnk(mB, sB, DB, B); }
    // z = X^dagger dQ of site s (DAG false), or Y dQ^dagger
    __device__ __forceinline__ void dq_left(const cx<double> (&X)[9], int s, cx<double> (&z)[9]) const {
        cx<double> q[9], t[9];
        ld_dq<DAG>(dQ, V, pl, s, q);
        mat_dag(X, t);
        mat_mul_plain(t, q, z);
        pin9(z);
    }
    __device__ __forceinline__ void dq_right(const cx<double> (&Y)[9], int s, cx<double> (&z)[9]) const {
        cx<double> q[9];
        ld_dq<DAG>(dQ, V, pl, s, q);
        mat_mul_plain(Y, q, z);
        pin9(z);
    }
    // (B C)^dagger dQ A^dagger or A dQ^dagger (B C); A and B are given back
    template <class F>
    __device__ __forceinline__ void begun_at_b(cx<double> (&A)[9], cx<double> (&B)[9], F&& emit) const {
        cx<double> X[9], z[9];
        {
            cx<double> C[9];
            lnk(mB, sB, DB, B);
            lnk(mC, sC, DC, C);
            mat_mul_plain(B, C, X);
        }
        pin9(X);
        lnk(mA, sA, DA, A);
        if (!DAG) {
            dq_left(X, s2, z);
            cx<double> t[9];
            mat_dag(A, t);
            mul_emit(z, t, emit);
        } else {
            dq_right(A, s2, z);
            mul_emit(z, X, emit);
        }
    }
    // C^dagger dQ (A B)^dagger or (A B) dQ^dagger C; C is given back
    template <class F>
    __device__ __forceinline__ void begun_at_c(const cx<double> (&AB)[9], cx<double> (&C)[9], F&& emit) const {
        cx<double> z[9];
        lnk(mC, sC, DC, C);
        if (!DAG) {
            dq_left(C, s3, z);
            cx<double> t[9];
            mat_dag(AB, t);
            mul_emit(z, t, emit);
        } else {
            dq_right(AB, s3, z);
            mul_emit(z, C, emit);
        }
    }
    // X = A B C: dQ X^dagger or X dQ^dagger
    template <class F>
    __device__ __forceinline__ void begun_at_l(const cx<double> (&X)[9], F&& emit) const {
        cx<double> q[9], t[9];
        ld_dq<DAG>(dQ, V, pl, s0, q);
        if (!DAG) {
            mat_dag(X, t);
            mul_emit(q, t, emit);
        } else {
            mul_emit(X, q, emit);
        }
    }
    // X^dagger dQ or dQ^dagger X
    template <class F>
    __device__ __forceinline__ void begun_at_a(const cx<double> (&X)[9], F&& emit) const {
        cx<double> q[9], t[9];
        ld_dq<DAG>(dQ, V, pl, s1, q);
        if (!DAG) {
            mat_dag(X, t);
            mul_emit(t, q, emit);
        } else {
            mul_emit(q, X, emit);
        }
    }
    // emit(k, entry k of a b)
    template <class F>
    static __device__ __forceinline__ void mul_emit(const cx<double> (&a)[9], const cx<double> (&b)[9], F&& emit) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                emit(3 * i + j,
                     cadd(cadd(cmul(a[3 * i], b[j]), cmul(a[3 * i + 1], b[3 + j])), cmul(a[3 * i + 2], b[6 + j])));
    }
};
// Neighbour of a site (with its coordinates) one step along +-mu.
__device__ __forceinline__ int step_site(const Geom& g, int s, const int x[4], int mu, bool fwd) {
    bool w;
    return fwd ? nbr_fwd(s, x, mu, g, w) : nbr_bwd(s, x, mu, g, w);
}

// Chain rule of the six planes onto the links: wavefront a of a workgroup
// takes U_a of 64 sites, with the three planes that hold direction a and in
// each the plaquette on either side.  The four leaves that share a plaquette
// share its partial products (three products and six with dQ where the leaves
// one by one take twelve).  Bound by the unfused FP64 products (the operation
// order is the reference's): 216 3x3 products or 43k operations per site,
// 148 us at 16^3 x 32 at the nominal rate with every lane busy, 190 us at the
// 4.8 cycles an instruction that two wavefronts per SIMD reach.  A wavefront
// alone issues an FP64 instruction every six cycles, so the terms come in an
// order that keeps few matrices at once, two wait in LDS and one link is read
// twice: 256 registers and two wavefronts per SIMD, 284 us against 324 with
// everything in 460 registers at one.  (More links read again and less parked
// loses it: 320 us at 1.4 times the loads.)  Blocks in the stencil's slab order.
__global__ void __launch_bounds__(256, 2) k_clover_links_pullback(double2* dU,
                                                                  const double2* U,
                                                                  const double2* dQ, Geom g, int slab) {
    // matrices that wait while others need the registers (each work item its own)
    __shared__ double2 park[2][9][256];
    int y0, end;
    slab_block(xcd_block(blockIdx.x, gridDim.x), slab, g, y0, end);
    const int y = y0 + (threadIdx.x & 63);
    const int a = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (y >= end) return;
    const int V = g.V;
    int x[4];
    site_coords(y, g, x);
    const int ya = step_site(g, y, x, a, true);
    int xa[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
    for (int d = 0; d < 4; ++d)
        if (d == a) xa[d] = x[d] + 1 == g.L[d] ? 0 : x[d] + 1;
#pragma unroll 1
    for (int b = 0; b < 4; ++b) {
        if (b == a) continue;
        const int lo = a < b ? a : b, hi = a < b ? b : a;
        const int pl = lo == 0 ? hi - 1 : lo + hi;  // (01,02,03,12,13,23)
        const int yb = step_site(g, y, x, b, true), ymb = step_site(g, y, x, b, false);
        const int yab = step_site(g, ya, xa, b, true), yamb = step_site(g, ya, xa, b, false);
        // h_p: the two terms of leaf p; h0 becomes ((h0 + h1) + h2) + h3
        cx<double> h0[9], h1[9], A[9], B[9], AB[9], C[9], X[9];
        const auto set = [](cx<double> (&h)[9]) { return [&h](int k, cx<double> v) { h[k] = v; }; };
        const auto add = [](cx<double> (&h)[9]) { return [&h](int k, cx<double> v) { h[k] = cadd(h[k], v); }; };
        const auto put = [&](int j) {
            return [j](int k, cx<double> v) { park[j][k][threadIdx.x] = make_double2(v.re, v.im); };
        };
        // the parked term completes leaf j's two terms
        const auto fetch_add = [&](int j, cx<double> (&h)[9]) {
            return [&h, j](int k, cx<double> v) {
                const double2 o = park[j][k][threadIdx.x];
                h[k] = cadd(mk<double>(o.x, o.y), v);
            };
        };
        if (a < b) {
            // U_a is the plane's first direction: L U_b(y+a) U_a(y+b)^+ U_b(y)^+ and
            // L^+ U_b(y-b)^+ U_a(y-b) U_b(y-b+a)
            const Plaquette<false, false, true, true> p{U, dQ, V, pl, b, ya, a, yb, b, y, y, ya, yab, yb};
            const Plaquette<true, true, false, false> m{U, dQ, V, pl, b, ymb, a, ymb, b, yamb, ya, y, ymb, yamb};
            p.begun_at_b(A, B, put(0));  // leaf 2
            mat_mul_plain(A, B, AB);
            pin9(AB);
            p.begun_at_c(AB, C, put(1));  // leaf 3
            mat_mul_plain(AB, C, X);
            pin9(X);
            p.begun_at_l(X, set(h0));
            pin9(h0);
            p.begun_at_a(X, set(h1));
            pin9(h1);
            m.begun_at_b(A, B, add(h0));
            pin9(h0);
            m.link_b(B);
            mat_mul_plain(A, B, AB);
            pin9(AB);
            m.begun_at_c(AB, C, add(h1));
            add9(h0, h1);
            pin9(h0);
            mat_mul_plain(AB, C, X);
            pin9(X);
            m.begun_at_l(X, fetch_add(0, h1));
            add9(h0, h1);
            pin9(h0);
            m.begun_at_a(X, fetch_add(1, h1));
            add9(h0, h1);
        } else {
            // the second: L U_b(y-b+a)^+ U_a(y-b)^+ U_b(y-b) and L^+ U_b(y) U_a(y+b) U_b(y+a)^+
            const Plaquette<false, true, true, false> p{U, dQ, V, pl, b, yamb, a, ymb, b, ymb, y, ya, yamb, ymb};
            const Plaquette<true, false, false, true> m{U, dQ, V, pl, b, y, a, yb, b, ya, ya, y, yb, yab};
            p.begun_at_b(A, B, put(0));  // leaf 3
            mat_mul_plain(A, B, AB);
            pin9(AB);
            p.begun_at_c(AB, C, set(h0));
            pin9(h0);
            mat_mul_plain(AB, C, X);
            pin9(X);
            p.begun_at_a(X, put(1));  // leaf 2
            p.begun_at_l(X, set(h1));
            pin9(h1);
            m.begun_at_b(A, B, add(h1));
            pin9(h1);
            m.link_b(B);
            mat_mul_plain(A, B, AB);
            pin9(AB);
            cx<double> h2[9];
            m.begun_at_c(AB, C, fetch_add(1, h2));
            pin9(h2);
            mat_mul_plain(AB, C, X);
            pin9(X);
            m.begun_at_a(X, add(h0));
            add9(h0, h1);
            add9(h0, h2);
            pin9(h0);
            m.begun_at_l(X, fetch_add(0, h1));
            add9(h0, h1);
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            double2* o = dU + (size_t)(a * 9 + k) * V + y;
            *o = make_double2(o->x + h0[k].re, o->y + h0[k].im);
        }
    }
}

int launch_clover_pullback(lmx_context* ctx, double2* dU, const double2* U, double2* dQ, const double2* dres,
                           const double2* psi, double coefficient) {
    if (ctx->V == 0) return LMX_OK;
    hipLaunchKernelGGL(k_clover_cotangent, dim3(nblocks(ctx->V)), dim3(256), 0, ctx->stream, dQ, dres, psi,
                       (int)ctx->V, coefficient);
    const SlabOrder so = slab_order(ctx->g, false, 12 * sizeof(double2));
    hipLaunchKernelGGL(k_clover_links_pullback, dim3((unsigned)so.blocks), dim3(256), 0, ctx->stream, dU, U,
                       (const double2*)dQ, ctx->g, so.slab);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

}  // namespace lmx
