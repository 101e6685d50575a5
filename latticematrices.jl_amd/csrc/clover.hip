// clover.hip -- clover field strength cache and precision conversions.
//
// F_mu,nu = (Q - Q^dagger)/8 with Q the four-leaf clover, planes
// (12,13,14,23,24,34): kernel_clover_field_strength_halo! NC=3 and
// _clover_store_antihermitian3! (src/Operators/WilsonDiracCloverOperator.jl:164-226).
// The cache holds only the 9 independent reals of each anti-Hermitian plane
// (27 complex slots per site, 432 B FP64 instead of 864 B for full matrices);
// the full matrices are recovered exactly (diagonal real parts are exactly 0,
// lower entries are -conj of upper ones, as the reference stores them).
#include "lmx_internal.h"

namespace lmx {

// A = A*B row by row with muladdmulti (_clover_mul_matrix3, :137-149)
__device__ __forceinline__ void mul3(cx<double> (&A)[9], const cx<double> (&B)[9]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const cx<double> a0 = A[3 * i], a1 = A[3 * i + 1], a2 = A[3 * i + 2];
#pragma unroll
        for (int j = 0; j < 3; ++j) A[3 * i + j] = muladdmulti(a0, B[j], a1, B[3 + j], a2, B[6 + j]);
    }
}
__device__ __forceinline__ void dag3(cx<double> (&u)[9]) {
    cx<double> t[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) t[3 * i + j] = cconj(u[3 * j + i]);
#pragma unroll
    for (int k = 0; k < 9; ++k) u[k] = t[k];
}

// keep a product in registers here: the loads that follow are not hoisted above it
__device__ __forceinline__ void pin9(cx<double> (&a)[9]) {
#pragma unroll
    for (int k = 0; k < 9; ++k) asm volatile("" : "+v"(a[k].re), "+v"(a[k].im)::"memory");
}

// U_mu(s) or its adjoint, mu the same in the whole wavefront
template <bool DAG>
__device__ __forceinline__ void ld_factor(const double2* __restrict__ U, int V, int mu, int s, cx<double> (&u)[9]) {
    ld_comps(U + (size_t)mu * 9 * V, V, s, u);
    if (DAG) dag3(u);
}

// a <- ((a*B)*C)*d with B, C loaded (each U or U^dagger), d given
template <bool DB, bool DC>
__device__ __forceinline__ void leaf(const double2* __restrict__ U, int V, cx<double> (&a)[9], int mb, int sb, int mc,
                                     int sc, const cx<double> (&d)[9]) {
    cx<double> b[9];
    ld_factor<DB>(U, V, mb, sb, b);
    mul3(a, b);
    pin9(a);
    ld_factor<DC>(U, V, mc, sc, b);
    mul3(a, b);
    mul3(a, d);
    pin9(a);
}

// A wavefront of a workgroup takes one plane of the workgroup's 64 sites: the
// six share their links in L1, a leaf's last link is the next leaf's first,
// and blocks follow slab_block's order.  Bound by latency: the 78 link loads of
// a site (11.2 KB through L1) come in eight rounds, each behind the product
// before it, and wavefronts wait 39% of their cycles (the 72 products are 131
// us at 24^3 x 48 with every lane busy; 56 loads, shared links through LDS,
// were slower).  400-430 us there and 76 us at 16^3 x 32, against 868 and 155
// us for one work item per site that kept all planes' results in scratch, in
// lattice order over all XCDs.  Without pin9
// the loads are hoisted and spilled (690 us), at 4 wavefronts per SIMD it
// spills (1180), at 2 it waits (430); at 3 one of the 168 registers spills.
__global__ void __launch_bounds__(384, 3) k_clover_build(const double2* __restrict__ U, double2* __restrict__ F, Geom g,
                                                         int slab) {
    int s0, end;
    slab_block(xcd_block(blockIdx.x, gridDim.x), slab, g, s0, end);
    const int s = s0 + (threadIdx.x & 63);
    if (s >= end) return;
    const int pl = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int V = g.V;
    const int mu = pl < 3 ? 0 : (pl < 5 ? 1 : 2), nu = pl < 3 ? pl + 1 : (pl < 5 ? pl - 1 : 3);
    int x[4];
    site_coords(s, g, x);
    const int xm = mu == 0 ? x[0] : (mu == 1 ? x[1] : x[2]), xn = nu == 1 ? x[1] : (nu == 2 ? x[2] : x[3]);
    // offsets of one step along each direction of the plane (they commute)
    const int fm = xm == g.L[mu] - 1 ? -(g.L[mu] - 1) * g.stride[mu] : g.stride[mu];
    const int bm = xm == 0 ? (g.L[mu] - 1) * g.stride[mu] : -g.stride[mu];
    const int fn = xn == g.L[nu] - 1 ? -(g.L[nu] - 1) * g.stride[nu] : g.stride[nu];
    const int bn = xn == 0 ? (g.L[nu] - 1) * g.stride[nu] : -g.stride[nu];
    // each leaf's last factor is the next one's first, adjointed
    cx<double> q[9], a[9], d[9];
    ld_factor<false>(U, V, mu, s, q);
    ld_factor<true>(U, V, nu, s, d);
    leaf<false, true>(U, V, q, nu, s + fm, mu, s + fn, d);
    dag3(d);
#pragma unroll
    for (int k = 0; k < 9; ++k) a[k] = d[k];
    ld_factor<false>(U, V, mu, s + bm, d);
    leaf<true, true>(U, V, a, mu, s + fn + bm, nu, s + bm, d);
#pragma unroll
    for (int k = 0; k < 9; ++k) q[k] = cadd(q[k], a[k]);
    dag3(d);
#pragma unroll
    for (int k = 0; k < 9; ++k) a[k] = d[k];
    ld_factor<false>(U, V, nu, s + bn, d);
    leaf<true, false>(U, V, a, nu, s + bm + bn, mu, s + bm + bn, d);
#pragma unroll
    for (int k = 0; k < 9; ++k) q[k] = cadd(q[k], a[k]);
    dag3(d);
#pragma unroll
    for (int k = 0; k < 9; ++k) a[k] = d[k];
    ld_factor<true>(U, V, mu, s, d);
    leaf<false, false>(U, V, a, mu, s + bn, nu, s + bn + fm, d);
#pragma unroll
    for (int k = 0; k < 9; ++k) q[k] = cadd(q[k], a[k]);
    const double f = 1.0 / 8.0;
    // diagonal i is half of slot (3 pl + i) / 2
    double* diag = reinterpret_cast<double*>(F);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int e = 3 * pl + i;
        diag[2 * ((size_t)(e >> 1) * V + s) + (e & 1)] = rmul(f, csub(q[4 * i], cconj(q[4 * i]))).im;
    }
    const cx<double> u0 = rmul(f, csub(q[1], cconj(q[3]))), u1 = rmul(f, csub(q[2], cconj(q[6]))),
                     u2 = rmul(f, csub(q[5], cconj(q[7])));
    F[(size_t)(9 + 3 * pl) * V + s] = make_double2(u0.re, u0.im);
    F[(size_t)(10 + 3 * pl) * V + s] = make_double2(u1.re, u1.im);
    F[(size_t)(11 + 3 * pl) * V + s] = make_double2(u2.re, u2.im);
}

// compact cache -> full planes [6][V][3][3] complex
__global__ void __launch_bounds__(256) k_clover_export(const double2* __restrict__ F, double2* __restrict__ out, int V) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= V) return;
    for (int pl = 0; pl < 6; ++pl) {
        double d[3];
        for (int i = 0; i < 3; ++i) {
            const int q = 3 * pl + i;
            double2 v = F[(long)(q / 2) * V + s];
            d[i] = (q % 2) ? v.y : v.x;
        }
        double2 u01 = F[(long)(9 + 3 * pl + 0) * V + s];
        double2 u02 = F[(long)(9 + 3 * pl + 1) * V + s];
        double2 u12 = F[(long)(9 + 3 * pl + 2) * V + s];
        double2* o = out + ((long)pl * V + s) * 9;
        o[0] = make_double2(0.0, d[0]);
        o[1] = u01;
        o[2] = u02;
        o[3] = make_double2(-u01.x, u01.y);
        o[4] = make_double2(0.0, d[1]);
        o[5] = u12;
        o[6] = make_double2(-u02.x, u02.y);
        o[7] = make_double2(-u12.x, u12.y);
        o[8] = make_double2(0.0, d[2]);
    }
}

__global__ void __launch_bounds__(256) k_convert(const double2* __restrict__ in, float2* __restrict__ o32,
                                                 __half2* __restrict__ o16, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double2 v = in[i];
    float2 f = make_float2((float)v.x, (float)v.y);
    if (o32) o32[i] = f;
    if (o16) o16[i] = __float22half2_rn(f);
}

int launch_clover_build_f64(lmx_context* ctx, const double2* U, double2* clover) {
    if (ctx->V == 0) return LMX_OK;
    const SlabOrder so = slab_order(ctx->g, false, 12 * sizeof(double2));
    hipLaunchKernelGGL(k_clover_build, dim3((unsigned)so.blocks), dim3(384), 0, ctx->stream, U, clover, ctx->g, so.slab);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

int launch_clover_export(lmx_context* ctx, const double2* clover, double2* F_out) {
    if (ctx->V == 0) return LMX_OK;
    hipLaunchKernelGGL(k_clover_export, dim3(nblocks(ctx->V)), dim3(256), 0, ctx->stream, clover, F_out, (int)ctx->V);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

static int convert(lmx_context* ctx, const double2* in, float2* o32, __half2* o16, int64_t n) {
    if (n == 0) return LMX_OK;
    hipLaunchKernelGGL(k_convert, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, in, o32, o16, n);
    LMX_HIP(hipGetLastError());
    return LMX_OK;
}

// FP16 links packed per direction: entries 0-3 and 4-7 as two 16-byte words
// (int4 [4][2][V]), entry 8 as one 4-byte word (half2 [4][V]) after them.
__global__ void __launch_bounds__(256) k_pack_links16(const double2* __restrict__ U, int4* __restrict__ P, int V) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    const int mu = blockIdx.y;
    if (s >= V) return;
    int w[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        double2 v = U[((size_t)mu * 9 + k) * V + s];
        __half2 h = __float22half2_rn(make_float2((float)v.x, (float)v.y));
        w[k] = *reinterpret_cast<int*>(&h);
    }
    P[((size_t)2 * mu) * V + s] = make_int4(w[0], w[1], w[2], w[3]);
    P[((size_t)2 * mu + 1) * V + s] = make_int4(w[4], w[5], w[6], w[7]);
    reinterpret_cast<int*>(P + (size_t)8 * V)[(size_t)mu * V + s] = w[8];
}

int launch_convert_links(lmx_context* ctx, const double2* U, float2* U32, __half2* U16) {
    LMX_TRY(convert(ctx, U, U32, nullptr, 36 * ctx->V));
    if (U16 && ctx->V > 0) {
        hipLaunchKernelGGL(k_pack_links16, dim3(nblocks(ctx->V), 4), dim3(256), 0, ctx->stream, U, (int4*)U16,
                           (int)ctx->V);
        LMX_HIP(hipGetLastError());
    }
    return LMX_OK;
}

int launch_convert_clover(lmx_context* ctx, const double2* F, float2* F32, __half2* F16) {
    return convert(ctx, F, F32, F16, 27 * ctx->V);
}

}  // namespace lmx
