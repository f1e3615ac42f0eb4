// gfx950 kernels of the FR P=3 compressible Navier-Stokes RK3 step.
//
// Per RK stage (drunkseal/opendynamo: solver.rs:610-738, rhs.cu, rk.cu):
//   viscous kernel    BR1-corrected gradient from the element's states and its
//                     neighbours' face traces, gradient face extrapolation,
//                     viscous normal flux at the element's 6 faces -> fv
//                     (replaces the gradient half of compute_rhs_volume_kernel
//                     and the viscous half of the face kernels), and, since it
//                     holds the gradient, the volume part that needs it: the
//                     divergence of the viscous fluxes (fast f32 build) or the
//                     whole volume RHS (strict build) -> fv, after the face part
//   update kernel     volume RHS (Euler mode: formed here; fast f32 build: the
//                     divergence of the Euler fluxes here, plus the stored
//                     viscous one), interface fluxes at all own faces
//                     (SLAU2 / AUSM+ / Rusanov, slip wall), FR correction,
//                     SSP-RK3 blend, face traces of the new state (replaces the
//                     rest of the volume kernel, the x/y/wall/z face kernels,
//                     the j arrays and rk_stage*_kernel)
// Forms of both: tiles of two elements (od_visc_kernel, od_update_kernel), blocks
// of 2x2x2 (fast: od_*_block_kernel; strict: od_visc_lines_block_kernel,
// od_update_face_block_kernel), both in one launch for a box with an odd
// dimension (od_*_core_shell_kernel), four consecutive elements (strict:
// od_visc_line_kernel), and batches of boxes (od_batch_*).
// A face flux is evaluated from the same operands in the same order wherever it
// is formed, once for both elements inside a block, else by both elements that
// share the face, so both sides see identical bits and no face array, atomic or
// second pass is needed.
//
// Point-wise phases: lane = solution point pt = i + 4j + 16k of the element; by
// lines: lane = line of four points (the viscous kernels on blocks and on four
// elements).  Line contractions of point-wise phases stage through LDS.  The
// arithmetic of every quantity in the strict build (association order,
// no contraction: built with -ffp-contract=off) is that of the reference
// kernel that computes it; comments cite the reference line.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "od_internal.hpp"

// OD_FAST = 1 builds the fast-math variant of the same kernels (selected by
// the [solver] fast_math key for f32 compute): divisions become reciprocal
// multiplies, square roots the hardware approximation, normal-vector zero
// terms are dropped, and the translation unit is compiled with contraction.
#ifndef OD_FAST
#define OD_FAST 0
#endif

namespace od {
#if OD_FAST
namespace fastmath {
#endif

// FR operators in constant memory, set once per device by upload_ops (the
// same P = 3 values for every solver): kept out of the kernel arguments so
// they do not occupy scalar registers for the whole kernel.
__constant__ Ops<float> g_ops_f32;
__constant__ Ops<double> g_ops_f64;

namespace {

template <class C>
__device__ __forceinline__ const Ops<C>& dev_ops() {
    if constexpr (sizeof(C) == 4)
        return g_ops_f32;
    else
        return g_ops_f64;
}

// a / b and sqrt(x): IEEE (correctly rounded) in the strict build; in the
// fast build for f32, v_rcp_f32 / v_sqrt_f32 (1 ulp).
template <class C>
__device__ __forceinline__ C dv(C a, C b) {
#if OD_FAST
    if constexpr (sizeof(C) == 4) return a * __builtin_amdgcn_rcpf(b);
#endif
    return a / b;
}
template <class C>
__device__ __forceinline__ C sq(C x) {
#if OD_FAST
    if constexpr (sizeof(C) == 4) return __builtin_amdgcn_sqrtf(x);
#endif
    return sqrt(x);
}

// A denominator that several quotients share.  In the strict build its
// reciprocal is formed once, in f64 (v_rcp_f64 to 24 bits, then the cubic
// iteration y (1 + e + e^2), e = 1 - b y), and each quotient is the correctly
// rounded a / b in three or four more instructions:
//   f32  q = a y in f64, its last three bits cleared, rounded to f32.  A quotient
//        of two 24-bit numbers in [2^e, 2^(e+1)) that is not itself the middle
//        between two f32 numbers lies 2^(e-48) or more from it.  Where the
//        quotient is subnormal it can be the middle, which has few bits; a y a
//        hair beside it would then round the wrong way.  So y is 2^-51 of itself
//        too large (the 1 in e is 1 + 2^-51): with y and q each rounded to within
//        2^-53 of themselves q exceeds the quotient by 1 to 3 2^-52 of it, less
//        than the 2^(e-49) that clearing takes off, and is a middle again exactly
//        where the quotient is one.
//   f64  q = a y, then one correction with the residual a - b q, exact in an
//        FMA (Markstein, IBM J. Res. Dev. 34, 1990: the last steps of the
//        compiler's own a / b; his theorem asks for y rounded correctly, which
//        one b in 700,000 misses: 10^7 quotients by 37,000 such b, those nearest
//        the middle between two numbers, all came out right).  v_div_fixup gives
//        zeros, infinities and NaN their IEEE results; |a| between 0 and 2^-969
//        may be off by one unit in the last place, and b below 2^-1022 or above
//        2^1021, whose reciprocal is not a normal number, is not covered.
// A division takes 46 (f32) and 65 (f64) cycles of a SIMD, a quotient 14 (f32,
// without the clearing, one instruction more: 48^3 visc 1267 -> 1320 instructions a
// wave, 235 -> 245 us) and 20, a reciprocal 37; a point has about 90 quotients by some ten
// denominators, which were nearly half of the strict kernels' instructions.
template <class C>
struct Recip {
    C b;
    double y;
};
template <class C>
constexpr double kRecipOne = sizeof(C) == 8 ? 1.0 : 1.0 + 0x1p-51;
template <class C>
__device__ __forceinline__ Recip<C> recip(C b) {
#if OD_FAST
    return {b, 0.0};  // quot takes v_rcp_f32 as dv does
#else
    const double d = (double)b, y0 = __builtin_amdgcn_rcp(d);
    const double e = __builtin_fma(-d, y0, kRecipOne<C>);
    const double y = __builtin_fma(__builtin_fma(e, e, e), y0, y0);
    if constexpr (sizeof(C) == 8) return {b, y};
    return {b, e == e ? y : y0};  // b zero or infinite: y0 is infinite or zero, and e NaN
#endif
}
template <class C>
__device__ __forceinline__ C quot(C a, Recip<C> r) {
#if OD_FAST
    return a * __builtin_amdgcn_rcpf(r.b);
#else
    if constexpr (sizeof(C) == 8) {
        const double q = a * r.y;
        return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-r.b, q, a), r.y, q), r.b, a);
    }
    return (C)__longlong_as_double(__double_as_longlong((double)a * r.y) & ~7LL);
#endif
}

// Fast build: the arithmetic of the point and interface fluxes may fuse a
// multiply into an add only within one source expression (as the C standard
// allows), not across statements.  Fusion across statements is decided per
// kernel from the shape of the whole computation (for a*b + c*d, which
// product to fuse depends on how many other expressions use each), so the
// same flux could round differently in the two-element-tile and the block
// kernels; within an expression the choice is fixed by the source.
#if OD_FAST
#define OD_CONTRACT_IN_EXPRESSIONS _Pragma("clang fp contract(on)")
#else
#define OD_CONTRACT_IN_EXPRESSIONS
#endif

template <class T>
__device__ __forceinline__ T sel3(T a0, T a1, T a2, int d) {
    return d == 0 ? a0 : (d == 1 ? a1 : a2);
}

// The RK stage blend kA u^n + kB u + kC r (stage 1: kA u^n + kC r; rk.cu:12-25).
// The fast build writes the fusion out, fma(kC, r, fma(kB, u, kA u^n)),
// so that every kernel form rounds it alike; the strict build rounds each
// product and sum, left to right.
template <class T>
__device__ __forceinline__ T fma_t(T a, T b, T c) {
    if constexpr (sizeof(T) == 4)
        return __builtin_fmaf(a, b, c);
    else
        return __builtin_fma(a, b, c);
}
template <class T>
__device__ __forceinline__ T rk_blend1(T kA, T kC, T un, T r) {
#if OD_FAST
    return fma_t(kC, r, kA * un);
#else
    return kA * un + kC * r;
#endif
}
template <class T>
__device__ __forceinline__ T rk_blend(T kA, T kB, T kC, T un, T u, T r) {
#if OD_FAST
    return fma_t(kC, r, fma_t(kB, u, kA * un));
#else
    return kA * un + kB * u + kC * r;
#endif
}

// ---------------------------------------------------------------------------
// Point physics in the compute type C (device_functions.cuh:1-257).
// Direction d = 0/1/2 is an argument; all three reference variants
// (compute_euler_flux_{x,y,z}, compute_viscous_flux_{x,y,z}) are the same
// expression tree with the direction's operands, which is what the selects
// pick, so the result is bitwise that of the matching variant.
// ---------------------------------------------------------------------------
template <class C>
__device__ __forceinline__ C gamma_m1() { return ((C)1.4) - ((C)1.0); }

template <class C>
__device__ __forceinline__ C pressure(Recip<C> ir, C ru, C rv, C rw, C e) {  // :1-5
    OD_CONTRACT_IN_EXPRESSIONS
#if OD_FAST
    if constexpr (sizeof(C) == 4) {  // fast build: the fusions written out
        const C h = ((C)0.5) * __builtin_fmaf(rw, rw, __builtin_fmaf(rv, rv, ru * ru));
        const C p = gamma_m1<C>() * __builtin_fmaf(-h, __builtin_amdgcn_rcpf(ir.b), e);
        return fmax(((C)1e-7), p);
    }
#endif
    C ke = quot(((C)0.5) * (ru * ru + rv * rv + rw * rw), ir);
    C p = gamma_m1<C>() * (e - ke);
    return fmax(((C)1e-7), p);
}

template <class C>
__device__ __forceinline__ void euler_flux(int d, const C* s, C* f) {  // :7-21
    OD_CONTRACT_IN_EXPRESSIONS
    C e = s[4];
    const Recip<C> ir = recip(s[0]);
    C p = pressure(ir, s[1], s[2], s[3], e);
    C md = sel3(s[1], s[2], s[3], d);
    C ud = quot(md, ir);
    f[0] = md;
#pragma unroll
    for (int c = 0; c < 3; ++c) f[1 + c] = (c == d) ? s[1 + c] * ud + p : s[1 + c] * ud;
    f[4] = ud * (e + p);
}

// :23-102.  g[3*var + dir]; G[a][b] = d(u_a)/d(x_b).
// The direction-independent part of the three directional viscous fluxes of
// a point: velocity, stress tensor and the heat flux along each direction.
// Every entry is the expression the directional flux evaluates, so the
// fluxes assembled from it are bitwise those of compute_viscous_flux_{x,y,z};
// the volume pass forms it once for its three directions.
template <class C>
struct ViscPoint {
    C u[3];
    C t00, t11, t22, t01, t02, t12;
    C q[3];
};
template <class C>
__device__ __forceinline__ C heat_flux(int d, const C* s, const C* g, C mu, Recip<C> ir, Recip<C> irr, C ke, C p) {
    C gd = sel3(g[0], g[1], g[2], d);
    C gu = sel3(g[3], g[4], g[5], d);
    C gv = sel3(g[6], g[7], g[8], d);
    C gw = sel3(g[9], g[10], g[11], d);
    C ge = sel3(g[12], g[13], g[14], d);
    C dke = quot(s[1] * gu + s[2] * gv + s[3] * gw, ir) - quot(ke * gd, ir);
    C dp = gamma_m1<C>() * (ge - dke);
    C coeff = dv(mu * ((C)1.4), ((C)0.72) * gamma_m1<C>());
    return -coeff * (quot(dp, ir) - quot(p * gd, irr));
}
// dirs: bit d set = the heat flux along d is needed.
template <class C>
__device__ __forceinline__ ViscPoint<C> viscous_point(const C* s, const C* g, C mu, int dirs) {
    ViscPoint<C> vp;
    C rho = s[0];
    const Recip<C> ir = recip(rho), irr = recip(rho * rho);
    vp.u[0] = quot(s[1], ir);
    vp.u[1] = quot(s[2], ir);
    vp.u[2] = quot(s[3], ir);
    C G[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) G[a][b] = quot(g[3 * (a + 1) + b] - vp.u[a] * g[b], ir);
    C div = G[0][0] + G[1][1] + G[2][2];
    const C two = (C)2.0, tt = ((C)2.0) / ((C)3.0);
    vp.t00 = mu * (two * G[0][0] - tt * div);
    vp.t11 = mu * (two * G[1][1] - tt * div);
    vp.t22 = mu * (two * G[2][2] - tt * div);
    vp.t01 = mu * (G[0][1] + G[1][0]);
    vp.t02 = mu * (G[0][2] + G[2][0]);
    vp.t12 = mu * (G[1][2] + G[2][1]);
    C ke = quot(((C)0.5) * (s[1] * s[1] + s[2] * s[2] + s[3] * s[3]), ir);
    C p = gamma_m1<C>() * (s[4] - ke);
#pragma unroll
    for (int d = 0; d < 3; ++d) vp.q[d] = (dirs >> d) & 1 ? heat_flux(d, s, g, mu, ir, irr, ke, p) : (C)0;
    return vp;
}
template <class C>
__device__ __forceinline__ void viscous_flux_dir(int d, const ViscPoint<C>& vp, C* f) {
    C r0 = sel3(vp.t00, vp.t01, vp.t02, d), r1 = sel3(vp.t01, vp.t11, vp.t12, d), r2 = sel3(vp.t02, vp.t12, vp.t22, d);
    f[0] = (C)0.0;
    f[1] = r0;
    f[2] = r1;
    f[3] = r2;
    f[4] = vp.u[0] * r0 + vp.u[1] * r1 + vp.u[2] * r2 - vp.q[d];
}
template <class C>
__device__ __forceinline__ void viscous_flux(int d, const C* s, const C* g, C mu, C* f) {
    viscous_flux_dir(d, viscous_point(s, g, mu, 1 << d), f);
}

#if OD_FAST
// The fast build's viscous fluxes, every fusion written out, so that the tile
// and the block kernels form the same bits.  The heat flux takes the gradient
// of the internal energy e = E / rho - |u|^2 / 2 (its p / rho is (gamma - 1) e):
//   grad e = (grad E - (E / rho) grad rho) / rho - sum_a u_a grad u_a,
// from the velocity gradients that the stresses need anyway, where the
// reference's form (heat_flux above, the strict build's) goes through the
// gradients of the kinetic energy and the pressure: 10 instructions fewer a
// face point and 27 a solution point.
struct FastVisc {
    float r, u[3], er;  // 1 / rho, velocity, E / rho
    float G[3][3];      // du_a / dx_b
    float h[3];         // grad e
    float mu;
};
// s: state, g: its gradient [var][3].  e: the element, for its eddy viscosity.
template <class Args>
__device__ __forceinline__ FastVisc fast_visc(const Args& a, const float* s, const float* g, int64_t e) {
#pragma clang fp contract(off)
    FastVisc f;
    f.r = __builtin_amdgcn_rcpf(s[0]);
#pragma unroll
    for (int c = 0; c < 3; ++c) f.u[c] = s[1 + c] * f.r;
    f.er = s[4] * f.r;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int b = 0; b < 3; ++b) f.G[c][b] = __builtin_fmaf(-f.u[c], g[b], g[3 * (c + 1) + b]) * f.r;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const float x = __builtin_fmaf(-f.er, g[b], g[12 + b]) * f.r;
        f.h[b] = __builtin_fmaf(-f.u[2], f.G[2][b], __builtin_fmaf(-f.u[1], f.G[1][b], __builtin_fmaf(-f.u[0], f.G[0][b], x)));
    }
    f.mu = a.mu;
    if (a.sutherland) {  // theta = gamma p / rho, p as in pressure()
        const float k = __builtin_fmaf(f.u[2], f.u[2], __builtin_fmaf(f.u[1], f.u[1], f.u[0] * f.u[0]));
        const float th = fmaxf((1.4f * gamma_m1<float>()) * __builtin_fmaf(-0.5f, k, f.er), 1.4e-7f * f.r);
        f.mu = (a.mu_ref * (a.t_ref + a.s_suth)) * (th * __builtin_amdgcn_sqrtf(th)) *
               __builtin_amdgcn_rcpf(__builtin_fmaf(a.t_ref, th, a.s_suth));
    }
    if (a.mu_t) f.mu = f.mu + a.mu_t[e];
    return f;
}
// Components 1..4 of the viscous flux along d.
__device__ __forceinline__ void fast_visc_flux(int d, const FastVisc& f, float* out) {
#pragma clang fp contract(off)
    const float div = (f.G[0][0] + f.G[1][1]) + f.G[2][2];
    float t[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
        t[c] = f.mu * (c == d ? __builtin_fmaf(-2.0f / 3.0f, div, 2.0f * f.G[c][c]) : f.G[c][d] + f.G[d][c]);
    out[0] = t[0];
    out[1] = t[1];
    out[2] = t[2];
    const float q = (f.mu * (1.4f / 0.72f)) * sel3(f.h[0], f.h[1], f.h[2], d);
    out[3] = __builtin_fmaf(f.u[0], t[0], __builtin_fmaf(f.u[1], t[1], __builtin_fmaf(f.u[2], t[2], q)));
}
#endif

template <class C>
__device__ __forceinline__ C sound_speed(C p, Recip<C> ir) {
    OD_CONTRACT_IN_EXPRESSIONS
    const C rho = ir.b;
#if OD_FAST
    if constexpr (sizeof(C) == 4) {
        // 1 / max(1e-7, rho) as a select: the reciprocal of rho is the one
        // the fluxes form anyway (one transcendental fewer per state)
        const C inv = rho >= (C)1e-7 ? __builtin_amdgcn_rcpf(rho) : __builtin_amdgcn_rcpf((C)1e-7);
        return __builtin_amdgcn_sqrtf(fmax(((C)0.0), (((C)1.4) * p) * inv));
    }
#endif
    // by max(1e-7, rho): rho's reciprocal, or that of the constant
    const Recip<C> im = rho >= (C)1e-7 ? ir : Recip<C>{(C)1e-7, kRecipOne<C> / (double)(C)1e-7};
    return sq(fmax(((C)0.0), quot(((C)1.4) * p, im)));
}

// Normal velocity u . n and momentum flux component m v_n + p n_c for the
// face normal n = e_D.  The strict build keeps the reference's arithmetic
// with the zero components (u*1 + v*0 + w*0, p*0), which is what fixes the
// sign of zero results; the fast build drops the zero terms.
template <int D, class C>
__device__ __forceinline__ C nvel(C u, C v, C w) {
    OD_CONTRACT_IN_EXPRESSIONS
#if OD_FAST
    return D == 0 ? u : (D == 1 ? v : w);
#else
    const C n0 = D == 0 ? (C)1.0 : (C)0.0, n1 = D == 1 ? (C)1.0 : (C)0.0, n2 = D == 2 ? (C)1.0 : (C)0.0;
    return u * n0 + v * n1 + w * n2;
#endif
}
template <int D, class C>
__device__ __forceinline__ C mflux(int c, C a, C b, C p) {
    OD_CONTRACT_IN_EXPRESSIONS
#if OD_FAST
    return c == D ? a * b + p : a * b;
#else
    return a * b + p * (c == D ? (C)1.0 : (C)0.0);
#endif
}

template <int D, class C>
__device__ __forceinline__ void rusanov(const C* l, const C* r, C* f) {  // :104-128
    OD_CONTRACT_IN_EXPRESSIONS
    const Recip<C> il = recip(l[0]), ir = recip(r[0]);
    C ul = quot(l[1], il), vl = quot(l[2], il), wl = quot(l[3], il);
    C ur = quot(r[1], ir), vr = quot(r[2], ir), wr = quot(r[3], ir);
    C pl = pressure(il, l[1], l[2], l[3], l[4]);
    C pr = pressure(ir, r[1], r[2], r[3], r[4]);
    C vnl = nvel<D>(ul, vl, wl);
    C vnr = nvel<D>(ur, vr, wr);
    C cl = sound_speed(pl, il), cr = sound_speed(pr, ir);
    C lam = fmax(fabs(vnl) + cl, fabs(vnr) + cr);
    C fl[5], fr[5];
    fl[0] = l[0] * vnl;
    fr[0] = r[0] * vnr;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        fl[1 + c] = mflux<D>(c, l[1 + c], vnl, pl);
        fr[1 + c] = mflux<D>(c, r[1 + c], vnr, pr);
    }
    fl[4] = vnl * (l[4] + pl);
    fr[4] = vnr * (r[4] + pr);
#pragma unroll
    for (int v = 0; v < 5; ++v) f[v] = ((C)0.5) * (fl[v] + fr[v] - lam * (r[v] - l[v]));
}

template <int D, class C>
__device__ __forceinline__ void ausm_plus(const C* l, const C* r, C* f) {  // :130-188
    OD_CONTRACT_IN_EXPRESSIONS
    const Recip<C> il = recip(l[0]), ir = recip(r[0]);
    C ul = quot(l[1], il), vl = quot(l[2], il), wl = quot(l[3], il);
    C ur = quot(r[1], ir), vr = quot(r[2], ir), wr = quot(r[3], ir);
    C pl = pressure(il, l[1], l[2], l[3], l[4]);
    C pr = pressure(ir, r[1], r[2], r[3], r[4]);
    C vnl = nvel<D>(ul, vl, wl);
    C vnr = nvel<D>(ur, vr, wr);
    C hl = quot(l[4] + pl, il), hr = quot(r[4] + pr, ir);
    C cl = sound_speed(pl, il), cr = sound_speed(pr, ir);
    C cm = fmax(cl, cr);
    const Recip<C> icm = recip(cm);
    C ml = quot(vnl, icm), mr = quot(vnr, icm);
    const C one = (C)1.0, q = (C)0.25, alpha = (C)0.1875, beta = (C)0.125, zero = (C)0.0;
    C mp, mm, pp, pm;
    if (fabs(ml) >= one) {
        mp = ((C)0.5) * (ml + fabs(ml));
        pp = (ml > zero) ? one : zero;
    } else {
        mp = q * (ml + one) * (ml + one) + beta * (ml * ml - one) * (ml * ml - one);
        pp = q * (ml + one) * (ml + one) * (((C)2.0) - ml) + alpha * ml * (ml * ml - one) * (ml * ml - one);
    }
    if (fabs(mr) >= one) {
        mm = ((C)0.5) * (mr - fabs(mr));
        pm = (mr < zero) ? one : zero;
    } else {
        mm = -q * (mr - one) * (mr - one) - beta * (mr * mr - one) * (mr * mr - one);
        pm = q * (mr - one) * (mr - one) * (((C)2.0) + mr) - alpha * mr * (mr * mr - one) * (mr * mr - one);
    }
    C mach = mp + mm;
    C p = pp * pl + pm * pr;
    bool pos = mach > zero;
    C mf = mach * cm * (pos ? l[0] : r[0]);
    C vs[3] = {pos ? ul : ur, pos ? vl : vr, pos ? wl : wr};
    C hs = pos ? hl : hr;
    f[0] = mf;
#pragma unroll
    for (int c = 0; c < 3; ++c) f[1 + c] = mflux<D>(c, mf, vs[c], p);
    f[4] = mf * hs;
}

template <int D, class C>
__device__ __forceinline__ void slau2(const C* l, const C* r, C* f) {  // :190-257
    OD_CONTRACT_IN_EXPRESSIONS
    const Recip<C> il = recip(l[0]), ir = recip(r[0]);
    C ul = quot(l[1], il), vl = quot(l[2], il), wl = quot(l[3], il);
    C ur = quot(r[1], ir), vr = quot(r[2], ir), wr = quot(r[3], ir);
    C pl = pressure(il, l[1], l[2], l[3], l[4]);
    C pr = pressure(ir, r[1], r[2], r[3], r[4]);
    C vnl = nvel<D>(ul, vl, wl);
    C vnr = nvel<D>(ur, vr, wr);
    C hl = quot(l[4] + pl, il), hr = quot(r[4] + pr, ir);
    C sql = ul * ul + vl * vl + wl * wl;
    C sqr = ur * ur + vr * vr + wr * wr;
    C cl = sound_speed(pl, il), cr = sound_speed(pr, ir);
    const C half = (C)0.5, one = (C)1.0, zero = (C)0.0;
    C cf = half * (cl + cr);
    const Recip<C> icf = recip(cf);
    C ml = quot(vnl, icf), mr = quot(vnr, icf);
    C mt = fmin(one, quot(one, icf) * sq(half * (sql + sqr)));
    C chi = one - mt;
    chi = chi * chi;
    C g = -fmax(fmin(ml, zero), -one) * fmin(fmax(mr, zero), one);
    C vavg = dv(l[0] * fabs(vnl) + r[0] * fabs(vnr), l[0] + r[0]);
    C val = (one - g) * vavg + g * fabs(vnl);
    C var = (one - g) * vavg + g * fabs(vnr);
    C mf = half * (l[0] * (vnl + val) + r[0] * (vnr - var) - quot(chi, icf) * (pr - pl));
    C bl = (fabs(ml) < one) ? ((C)0.25) * (((C)2.0) - ml) * (ml + one) * (ml + one)
                            : ((ml >= zero) ? one : zero);
    C br = (fabs(mr) < one) ? ((C)0.25) * (((C)2.0) + mr) * (mr - one) * (mr - one)
                            : ((mr >= zero) ? zero : one);
    C pf = half * (pl + pr) + half * (bl - br) * (pl - pr);
    pf += sq(half * (sql + sqr)) * (bl + br - one) * cf * half * (l[0] + r[0]);
    bool pos = mf > zero;
    C vs[3] = {pos ? ul : ur, pos ? vl : vr, pos ? wl : wr};
    C hs = pos ? hl : hr;
    f[0] = mf;
#pragma unroll
    for (int c = 0; c < 3; ++c) f[1 + c] = mflux<D>(c, mf, vs[c], pf);
    f[4] = mf * hs;
}

template <int D, class C>
__device__ __forceinline__ void interface_flux(int scheme, const C* l, const C* r, C* f) {
    if (scheme == 0)
        slau2<D>(l, r, f);
    else if (scheme == 1)
        ausm_plus<D>(l, r, f);
    else
        rusanov<D>(l, r, f);
}

// Sutherland law, theta = gamma p / rho (no reference counterpart; the
// reference parses the keys but uses a constant mu, constants.cuh:42).
template <class C>
__device__ __forceinline__ C sutherland(const C* s, C mu_ref, C t_ref, C s_suth) {
    const Recip<C> ir = recip(s[0]);
    C theta = quot(((C)1.4) * pressure(ir, s[1], s[2], s[3], s[4]), ir);
    return dv((mu_ref * (theta * sq(theta))) * (t_ref + s_suth), t_ref * theta + s_suth);
}

// ---------------------------------------------------------------------------
// Work-group layout: two elements per 128-thread work-group, wave w owns
// element 2*blockIdx.x + w for the point-wise phases (lane = solution point
// pt = i + 4j + 16k).  Face-point phases work on both elements at once,
// direction by direction: a direction has 2 elements x 2 faces x 16 points
// = 64 tasks, one full wave pass with direction-specialised code.  Wave 0
// takes x and z, wave 1 takes y (3 full passes per 2 elements; a wave that
// finishes early waits at the barrier and frees its SIMD for other waves).
// ---------------------------------------------------------------------------
constexpr int kEpb = 2;

struct Elem {
    int32_t xl, xr, yl, yr, zl, zr;  // neighbours across each face; -1 = slip wall (box-local, < 2^31)
};

// Element (ex, ey, ez) and its face neighbours; coordinates come from the
// launch grid, so no integer division is needed.
__device__ __forceinline__ Elem make_elem(int ex, int ey, int ez, int nx, int ny, int nz, int wall) {
    Elem r;
    const int sy = nx, sz = nx * ny;
    const int e = ex + sy * ey + sz * ez;
    r.xl = e + (ex == 0 ? nx - 1 : -1);
    r.xr = e + (ex == nx - 1 ? 1 - nx : 1);
    const int yl = e + (ey == 0 ? (ny - 1) * sy : -sy);
    const int yr = e + (ey == ny - 1 ? -(ny - 1) * sy : sy);
    r.yl = (wall && ey == 0) ? -1 : yl;
    r.yr = (wall && ey == ny - 1) ? -1 : yr;
    r.zl = e + (ez == 0 ? (nz - 1) * sz : -sz);
    r.zr = e + (ez == nz - 1 ? -(nz - 1) * sz : sz);
    return r;
}

// Points of the line through face point fp of a face normal to d:
// x: fp = j+4k, y: fp = i+4k, z: fp = i+4j.
__device__ __forceinline__ void face_line(int d, int fp, int& base, int& stride) {
    base = d == 0 ? 4 * fp : (d == 1 ? (fp & 3) + 16 * (fp >> 2) : fp);
    stride = d == 0 ? 1 : (d == 1 ? 4 : 16);
}

// Trace orders of the reference: 0 = pairwise (t0+t1)+(t2+t3) (shuffle
// butterfly, rhs.cu:68-85, 595-599, 665-674), 1 = sequential from 0
// (rhs.cu:89-101, 171-176, 716-727), 2 = sequential from the first product
// (rhs.cu:131-138, 540-543).
template <class C>
__device__ __forceinline__ C trace4(const C* q, int base, int stride, C c0, C c1, C c2, C c3, int order) {
#if OD_FAST
    // Fast build: explicit fused forms, so that a trace comes out bitwise the
    // same in every kernel that forms it (the trace kernel and the update
    // kernel write the traces the next stage reads) whatever the compiler
    // would contract in each context.
    if constexpr (sizeof(C) == 4) {
        const C q0 = q[base], q1 = q[base + stride], q2 = q[base + 2 * stride], q3 = q[base + 3 * stride];
        if (order == 0) return __builtin_fmaf(q1, c1, q0 * c0) + __builtin_fmaf(q3, c3, q2 * c2);
        return __builtin_fmaf(q3, c3, __builtin_fmaf(q2, c2, __builtin_fmaf(q1, c1, q0 * c0)));
    }
#endif
    C t0 = q[base] * c0, t1 = q[base + stride] * c1, t2 = q[base + 2 * stride] * c2, t3 = q[base + 3 * stride] * c3;
    if (order == 0) return (t0 + t1) + (t2 + t3);
    if (order == 1) {
        C s0 = (C)0;
        s0 += t0;
        s0 += t1;
        s0 += t2;
        s0 += t3;
        return s0;
    }
    return t0 + t1 + t2 + t3;
}

// Bank-conflict-free position of point p = i + 4j + 16k in a 64-value LDS
// row (the visc kernel's gradient tile is stored in this order): a face pass
// reads, per half-wave, the 16 face lines of one element at one line
// position (fixed i, j or k), which in the plain layout hit 8 of the 32
// banks twice for x and y faces.  Bits of the position: i0^j0, i0^k1,
// i1, j1, k0, i0 -- a bijection under which each of those 16-point sets, and
// the 32 points a half-wave writes, fall in 16 or 32 distinct banks.
__device__ __forceinline__ int swz64(int p) {
    const int i0 = p & 1, j0 = (p >> 2) & 1, k1 = (p >> 5) & 1;
    return (i0 ^ j0) | ((i0 ^ k1) << 1) | (p & 2) << 1 | (p & 8) | (p & 16) | (i0 << 5);
}
// trace4 over a swizzled row: line points base + m * stride.
template <class C>
__device__ __forceinline__ C trace4_swz(const C* q, int base, int stride, C c0, C c1, C c2, C c3, int order) {
    const C r[4] = {q[swz64(base)], q[swz64(base + stride)], q[swz64(base + 2 * stride)], q[swz64(base + 3 * stride)]};
    return trace4(r, 0, 1, c0, c1, c2, c3, order);
}

// The fast build forms every trace in the pairwise (fused) form and keeps a
// single x trace per face (faces 0/1) for BR1 and the Riemann flux alike;
// the strict build keeps the reference's orders below, with two x traces
// (0/1 pairwise for BR1, 6/7 sequential for the interface flux).  Both
// sides of a face see the same two traces either way, so the interface
// flux stays single-valued (conservative).
constexpr bool kOneX = OD_FAST;
// The visc kernel, which holds the corrected gradient anyway, also forms what
// the volume RHS needs of it and stores that after the element's face viscous
// fluxes (fv + kFvFaces), so that the update kernel forms no gradient of its
// own.  Fast f32 build (kSplitVisc): the divergence of the viscous fluxes; the
// update kernel takes that of the Euler fluxes.  Strict build: the reference's
// single divergence of F_e - F_v (rhs.cu:229-266) keeps its rounding only if it
// is formed in one place, so the visc kernel forms the whole volume RHS.  The
// second set of jumps and gradients it saves the update kernel was a third of
// the strict step's instructions, for one value per variable and point written
// and read: 48^3 f32, 40 steps 76.2 -> 73.1 ms; 24x26x22 f64, 50 steps 29.8 -> 26.3.
template <class CT>
constexpr bool kSplitVisc = OD_FAST && std::is_same<CT, float>::value;
constexpr int kFvStride = fv_stride(OD_FAST);
// The x line through point (i, j, k) is the four consecutive lanes of the
// point's quad, so the fast f32 build contracts it from registers with DPP
// quad broadcasts instead of an LDS round trip: the same products summed in
// the same order, so the results are those of the LDS form bit for bit.
// Sum of Dd[m] * (f of lane m of the quad), first a product, then fused in the
// order of m.  The broadcasts are the multiplies' own DPP operands; left to
// itself the compiler moves three of the four to a register first.  (s_nop: DPP
// may read a register two instructions after it was written at the earliest.)
__device__ __forceinline__ float quad_line(const float* Dd, float f) {
    float s;
    asm("s_nop 1\n\t"
        "v_mul_f32_dpp %0, %1, %2 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %3 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %4 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %5 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf"
        : "=&v"(s)
        : "v"(f), "v"(Dd[0]), "v"(Dd[1]), "v"(Dd[2]), "v"(Dd[3]));
    return s;
}
// Fast f32 build: the interface correction takes the viscous fluxes of the
// two sides as their half-difference (F_vL - F_vR) / 2, which the block visc
// kernel stores once per interior face instead of the two fluxes; the strict
// build keeps the reference's F* = F_riemann - (F_vL + F_vR) / 2.
template <class CT>
constexpr bool kHalfDiff = OD_FAST && std::is_same<CT, float>::value;
// Order of the BR1 traces (rhs.cu:385-455): x, y pairwise; z sequential from 0.
__device__ __forceinline__ constexpr int br1_order(int d) { return (d == 2 && !kOneX) ? 1 : 0; }
// Order of the Riemann inputs and gradient slices (rhs.cu:126-180, 540-543,
// 663-674, 716-727): x sequential from the first product, y pairwise, z from 0.
__device__ __forceinline__ constexpr int face_order(int d) { return kOneX ? 0 : (d == 0 ? 2 : (d == 1 ? 0 : 1)); }
// Order of the state and gradient traces the viscous face fluxes take: the
// reference's face order; the fast build takes the state traces of BR1 and, for
// the gradient's, which are formed and used inside one kernel, the fused
// sequential form (one instruction fewer per trace than the pairwise one).
__device__ __forceinline__ constexpr int fv_order(int d) { return kOneX ? 1 : face_order(d); }
// Faces of the trace layout the build writes, and the direction and order of face f.
constexpr int kOwnFaces = kOneX ? 6 : 8;
__device__ __forceinline__ int trace_face_dir(int f) { return f < 6 ? f >> 1 : 0; }
__device__ __forceinline__ int trace_face_order(int f) { return kOneX ? 0 : (f < 4 ? 0 : (f < 6 ? 1 : 2)); }

template <class C>
struct Coef4 {
    C c0, c1, c2, c3;
};

// The FR operators in LDS, laid out so that a lane reads the row or the side
// it needs directly: selecting among 4 wave-uniform scalars costs 3
// v_cndmask and 2 v_mov per coefficient and lane (one scalar operand per
// VALU instruction).
#if OD_FAST
// Per direction, with the Jacobian in them (BoxOps): an instruction less for
// every sum along a line, and for every lane's correction slopes.
struct alignas(16) BoxTable {
    float D[3][4][4];  // D[d][i][m] = J_d l_m'(x_i)
    float g[3][4][2];  // J_d {g_left'(x_i), g_right'(x_i)}
};
template <class C>
struct alignas(16) CoefTable : BoxTable {
    C e[2][4];  // {l_m(-1)}, {l_m(+1)}
};
template <class C>
using Rows = BoxTable;
// A tile's own copy, and the coefficients of its lines' derivatives.
struct TileTable : BoxTable {
    BoxOps::EvenOdd line[3][2];
};
#else
template <class C>
struct alignas(16) CoefTable {
    C D[4][4];  // D[i][m] = l_m'(x_i)
    C g[4][2];  // {g_left'(x_i), g_right'(x_i)}
    C e[2][4];  // {l_m(-1)}, {l_m(+1)}
};
template <class C>
using Rows = CoefTable<C>;
struct TileTable {};
#endif
template <class C>
__device__ __forceinline__ CoefTable<C>& coef_lds() {
    __shared__ CoefTable<C> t;
    return t;
}
// The first threads of the work-group copy the table from memory: the
// load is issued first thing (coef_load), the LDS store comes just before the
// body's first barrier (coef_store), which orders it before every read, so
// the load's latency hides behind the body's own loads.
template <class C>
constexpr int kCoefs = sizeof(CoefTable<C>) / sizeof(C);
template <class UT, class C>
__device__ __forceinline__ C coef_load(const StageArgs<UT, C>& a, int tid) {
#if OD_FAST
    static_assert(sizeof(BoxOps::table) == sizeof(CoefTable<C>) && kCoefs<C> <= 128, "table layout");
    return tid < kCoefs<C> ? a.ops->table[tid] : (C)0;
#else
    static_assert(sizeof(Ops<C>) == 32 * sizeof(C) && kCoefs<C> == 32, "table layout");
    // Ops order: D[16], eL[4], eR[4], gL[4], gR[4]; the index stays inside
    // Ops for every thread, whether or not the load is speculated
    const int t = tid & 31;
    const int src = t < 16 ? t : (t < 24 ? 24 + ((t - 16) & 1) * 4 + ((t - 16) >> 1) : t - 8);
    return tid < 32 ? reinterpret_cast<const C*>(&dev_ops<C>())[src] : (C)0;
#endif
}
template <class C>
__device__ __forceinline__ void coef_store(int tid, C v) {
    if (tid < kCoefs<C>) reinterpret_cast<C*>(&coef_lds<C>())[tid] = v;
}
#if OD_FAST
// The same for a tile's own copy, by its 128 threads: the visc kernel's with the
// coefficients of the lines' derivatives (TileTable), the update kernel's, which
// takes none, without (BoxTable).
template <class Table>
constexpr int kTableValues = (sizeof(BoxTable) + (std::is_same<Table, TileTable>::value ? sizeof(BoxOps::line) : 0)) / sizeof(float);
template <class Table, class UT>
__device__ __forceinline__ float tile_table_load(const StageArgs<UT, float>& a, int tid) {
    constexpr int kRows = kTableValues<BoxTable>, kAll = kTableValues<Table>;
    static_assert(kAll <= 128 && sizeof(Table) >= kAll * sizeof(float), "one value a thread");
    const float* src = tid < kRows ? a.ops->table + tid : &a.ops->line[0][0].ps + (tid - kRows);
    return tid < kAll ? *src : 0.f;
}
template <class Table>
__device__ __forceinline__ void tile_table_store(Table& t, int tid, float v) {
    if (tid < kTableValues<Table>) reinterpret_cast<float*>(&t)[tid] = v;
}
#endif
template <class C>
__device__ __forceinline__ Coef4<C> side_coef(bool right) {
    const C* r = coef_lds<C>().e[right];
    return {r[0], r[1], r[2], r[3]};
}

// Task of a direction-D face pass: lane -> (local element, side, face point).
struct FaceTask {
    int le, side, fp, f;
};
template <int D>
__device__ __forceinline__ FaceTask face_task(int lane) {
    FaceTask t;
    t.le = lane >> 5;
    t.side = (lane >> 4) & 1;
    t.fp = lane & 15;
    t.f = 2 * D + t.side;
    return t;
}

// The work-group's two elements, held in named scalars (no private arrays).
struct Tile {
    int32_t e0, e1;
    bool v0, v1;
    int32_t walls;  // bit 2 le + side: face yL/yR of element le is a slip wall
    Elem el0, el1;
};

// Whether the side `side` face of direction D of element le is a wall (only
// y faces can be); needs no neighbour index.
template <int D>
__device__ __forceinline__ bool tile_wall(const Tile& t, int le, int side) {
    return D == 1 && ((t.walls >> (2 * le + side)) & 1);
}

// Tile (t0, t1, t2) of a box: two elements adjacent along `orient`
// (0 x, 1 y, 2 z); the tile coordinate along `orient` counts pairs.
template <class UT, class CT>
__device__ __forceinline__ Tile make_tile_at(const StageArgs<UT, CT>& a, int orient, int t0, int t1, int t2) {
    Tile t;
    int ex = t0, ey = t1, ez = t2;
    int step;
    bool v1;
    if (orient == 0) {
        ex = kEpb * t0;
        v1 = ex + 1 < a.nx;
        step = 1;
    } else if (orient == 1) {
        ey = kEpb * t1;
        v1 = ey + 1 < a.ny;
        step = a.nx;
    } else {
        ez = kEpb * t2;
        v1 = ez + 1 < a.nz;
        step = a.nx * a.ny;
    }
    t.e0 = ex + a.nx * (ey + a.ny * ez);
    t.e1 = t.e0 + step;
    t.v0 = true;
    t.v1 = v1;
    t.el0 = make_elem(ex, ey, ez, a.nx, a.ny, a.nz, a.wall);
    const int d = v1 ? 1 : 0;
    t.el1 = make_elem(ex + (orient == 0 ? d : 0), ey + (orient == 1 ? d : 0), ez + (orient == 2 ? d : 0), a.nx, a.ny,
                      a.nz, a.wall);
    t.walls = (t.el0.yl < 0 ? 1 : 0) | (t.el0.yr < 0 ? 2 : 0) | (t.el1.yl < 0 ? 4 : 0) | (t.el1.yr < 0 ? 8 : 0);
    return t;
}

// Single-box launch grid: blockIdx = (pair of x elements, ey, ez).
template <class UT, class CT>
__device__ __forceinline__ Tile make_tile(const StageArgs<UT, CT>& a) {
    return make_tile_at(a, 0, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z);
}
// The same tiles in reverse order (the update kernels: they start where the
// visc kernel ended, on the data it touched last).
template <class UT, class CT>
__device__ __forceinline__ Tile make_tile_reversed(const StageArgs<UT, CT>& a) {
    return make_tile_at(a, 0, (int)(gridDim.x - 1 - blockIdx.x), (int)(gridDim.y - 1 - blockIdx.y),
                        (int)(gridDim.z - 1 - blockIdx.z));
}

__device__ __forceinline__ bool tile_valid(const Tile& t, int le) { return le ? t.v1 : t.v0; }
__device__ __forceinline__ int64_t tile_eidx(const Tile& t, int le) { return (int64_t)(le ? t.e1 : t.e0); }
// Neighbour across the side `side` face of direction D of local element le.
template <int D>
__device__ __forceinline__ int64_t tile_nb(const Tile& t, int le, int side) {
    const Elem& a = t.el0;
    const Elem& b = t.el1;
    int l0 = D == 0 ? a.xl : (D == 1 ? a.yl : a.zl), r0 = D == 0 ? a.xr : (D == 1 ? a.yr : a.zr);
    int l1 = D == 0 ? b.xl : (D == 1 ? b.yl : b.zl), r1 = D == 0 ? b.xr : (D == 1 ? b.yr : b.zr);
    int n0 = side ? r0 : l0, n1 = side ? r1 : l1;
    return (int64_t)(le ? n1 : n0);
}

// Neighbour across face f (0..5) of local element le, -1 = wall; selects on
// named fields only.
// Neighbour across face f (lane-varying) of tile element le (lane-varying):
// selects among the twelve wave-uniform indices, taken by value so that the
// selects stay in registers (a nested conditional on the struct fields
// compiles to divergent branches, a select of field references to a
// scratch-memory load).
__device__ __forceinline__ int64_t tile_nb_rt(const Tile& t, int le, int f) {
    const int xl = le ? t.el1.xl + 0 : t.el0.xl + 0, xr = le ? t.el1.xr + 0 : t.el0.xr + 0;
    const int yl = le ? t.el1.yl + 0 : t.el0.yl + 0, yr = le ? t.el1.yr + 0 : t.el0.yr + 0;
    const int zl = le ? t.el1.zl + 0 : t.el0.zl + 0, zr = le ? t.el1.zr + 0 : t.el0.zr + 0;
    const int x = (f & 1) ? xr : xl, y = (f & 1) ? yr : yl, z = (f & 1) ? zr : zl;
    return (int64_t)(f < 2 ? x : (f < 4 ? y : z));
}

// ---------------------------------------------------------------------------
// Neighbour-trace prefetch (f32 compute).  At kernel start each work-group
// copies the neighbour traces it will read straight from global memory into
// LDS with gfx950's global_load_lds_dwordx4 (no registers, one exposed
// latency), as 240 16-byte chunks: the facing traces of faces 0..5 of both
// elements, [2][6][5][16] -- in the BR1 order for the visc kernel, in that of
// the Riemann inputs for the update kernel (RIEMANN; in the strict build the x
// faces' other trace).
// The face viscous fluxes fv are read from global memory in the face pass
// instead: staging them too (another 1536 floats) limited the update kernel
// to 4.5 waves per SIMD by LDS; without them it runs 6 (a step measured
// ~6 % faster in both builds).
constexpr int kPfChunks = 240;
constexpr int kPfFloats = 4 * kPfChunks;

// Source of chunk `id`; false for chunks of a missing second element (odd
// nx), which are not copied.
template <bool RIEMANN, class UT, class CT>
__device__ __forceinline__ bool prefetch_chunk(const StageArgs<UT, CT>& a, const Tile& tl, int id, const CT*& src) {
    const int le = id / 120, f = (id % 120) / 20, c = id % 20;
    if (!tile_valid(tl, le)) return false;
    const int64_t own = tile_eidx(tl, le), nb = tile_nb_rt(tl, le, f);
    const int slot = (RIEMANN && !kOneX && f < 2) ? 7 - f : f ^ 1;
    src = a.tr_in + (nb >= 0 ? nb : own) * kTraceStride + slot * 80 + c * 4;
    return true;
}

// Issue the chunks; waves split the 64-chunk instructions.
// The caller waits (s_waitcnt 0, then a barrier for the other wave's copies)
// before reading the buffer.
template <bool RIEMANN, class UT, class CT>
__device__ __forceinline__ void prefetch_issue(const StageArgs<UT, CT>& a, const Tile& tl, float* pf, int wave,
                                               int lane) {
    constexpr int n_inst = (kPfChunks + 63) / 64;
    wave = __builtin_amdgcn_readfirstlane(wave);  // wave-uniform: a scalar loop
    const int first = wave == 0 ? 0 : (n_inst + 1) / 2;
    const int last = wave == 0 ? (n_inst + 1) / 2 : n_inst;
    for (int q = first; q < last; ++q) {
        const int id = q * 64 + lane;
        const CT* src = nullptr;
        if (id < kPfChunks && prefetch_chunk<RIEMANN>(a, tl, id, src)) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)(pf + q * 256), 16, 0, 0);
        }
    }
}

#if OD_FAST
// Corrected derivative along a line, d u / d xi + j_L g_L' + j_R g_R' with the
// jumps j = (u_nb - u_own) / 2, in even and odd parts (fast f32 build).  The
// points and operators mirror about the element's centre, D[3-i][m] =
// -D[i][3-m] and g_R'[i] = -g_L'[3-i], and a constant has no derivative, so with
//   t = (u0 + u3) - (u1 + u2),  d0 = u0 - u3,  d1 = u1 - u2,
//   p = w_L - w_R,  q = w_L + w_R,  w = u_nb - u_own = 2 j,
// the derivative at points i and 3 - i (i = 0, 1) is odd +- even:
//   even = ps t + pb q,  odd = qa d0 + qb d1 + qp p.
// 21 operations and the jumps' 2 for the line's four points with the Jacobian in
// the coefficients (BoxOps); row by row they were 28 and 4.  Differences are
// formed first, so less cancels than in the rows' sums.  One form for every
// kernel, explicitly fused: the same bits.  With the Jacobians in the other
// tables and the DPP operands of quad_line the block visc kernel issues a tenth
// less: 48^3 132 -> 126 us, 64^3 292 -> 275 us a launch.
using EvenOdd = BoxOps::EvenOdd;
__device__ __forceinline__ float line_even(const EvenOdd& c, float t, float q) {
    return __builtin_fmaf(c.pb, q, c.ps * t);
}
__device__ __forceinline__ float line_odd(const EvenOdd& c, float d0, float d1, float p) {
    return __builtin_fmaf(c.qp, p, __builtin_fmaf(c.qb, d1, c.qa * d0));
}
// The coefficients along D of point pair i (wave-uniform: scalar loads).
__device__ __forceinline__ EvenOdd even_odd(const BoxOps* ops, int D, int i) {
    const auto* c = (const __attribute__((address_space(4))) float*)&ops->line[D][i];
    return {c[0], c[1], c[2], c[3], c[4]};
}
// Those of a lane at point i of its line, the even part's sign with them.
__device__ __forceinline__ EvenOdd lane_even_odd(const EvenOdd* line, int i) {
    const EvenOdd& c = line[i == 1 || i == 2];
    return {i < 2 ? c.ps : -c.ps, i < 2 ? c.pb : -c.pb, c.qa, c.qb, c.qp};
}
// The derivative at a lane's point from the line u[0], u[stride], ...
__device__ __forceinline__ float lane_derivative(const EvenOdd& c, const float* u, int stride, float wl, float wr) {
    const float u0 = u[0], u1 = u[stride], u2 = u[2 * stride], u3 = u[3 * stride];
    return line_odd(c, u0 - u3, u1 - u2, wl - wr) + line_even(c, (u0 + u3) - (u1 + u2), wl + wr);
}
#endif

// BR1 jump 1/2 (u_nb + u_own) - u_own (fast build: twice that, u_nb - u_own)
// at every face point of direction D (accumulate_jump, rhs.cu:105-108; wall ghost rhs.cu:111-114), once per face
// point instead of once per lane of the normal line.
template <int D, bool PF, class UT, class CT>
__device__ __forceinline__ void br1_jumps(const StageArgs<UT, CT>& a, const CT (*sU)[5][64], CT (*sJmp)[6][5][16],
                                          const Tile& tl, const CT* pf, int lane) {
    const FaceTask t = face_task<D>(lane);
    if (!tile_valid(tl, t.le)) return;
    int base, stride;
    face_line(D, t.fp, base, stride);
    const Coef4<CT> c = side_coef<CT>(t.side);
    // with the prefetch the neighbour index is not needed here, only whether
    // the face is a wall (keeps 12 indices out of the registers)
    const int64_t nb = PF ? 0 : tile_nb<D>(tl, t.le, t.side);
    const bool wall = PF ? tile_wall<D>(tl, t.le, t.side) : nb < 0;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT own = trace4(sU[t.le][v], base, stride, c.c0, c.c1, c.c2, c.c3, br1_order(D));
        const CT sign = (v > 0 && v < 4) ? ((CT)-1.0) : ((CT)1.0);
        CT far;
        if constexpr (PF)
            far = pf[(t.le * 6 + t.f) * 80 + v * 16 + t.fp];
        else
            far = !wall ? a.tr_in[nb * kTraceStride + (t.f ^ 1) * 80 + v * 16 + t.fp] : (CT)0;
        CT nbv = !wall ? far : own * sign;
        sJmp[t.le][t.f][v][t.fp] = OD_FAST ? nbv - own : ((CT)0.5) * (nbv + own) - own;
    }
}

// BR1-corrected gradient at the lane's point (rhs.cu:366-465) from the
// element's LDS tile and the face jumps; Q round trip included.
// J0..J5: the jump blocks [5][16] of faces xL, xR, yL, yR, zL, zR.
template <class UT, class CT>
__device__ __forceinline__ void lane_gradient_faces(const StageArgs<UT, CT>& a, const CT (*sU)[64], const CT* J0,
                                                    const CT* J1, const CT* J2, const CT* J3, const CT* J4,
                                                    const CT* J5, const TileTable& t, int i, int j, int k, CT* g) {
    const int xb = 4 * j + 16 * k, yb = i + 16 * k, zb = i + 4 * j;
    const int fpx = j + 4 * k, fpy = i + 4 * k, fpz = i + 4 * j;
#if OD_FAST
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const EvenOdd c = lane_even_odd(t.line[d], d == 0 ? i : (d == 1 ? j : k));
        const int base = d == 0 ? xb : (d == 1 ? yb : zb), stride = d == 0 ? 1 : (d == 1 ? 4 : 16);
        const int fp = d == 0 ? fpx : (d == 1 ? fpy : fpz);
        const CT *JL = d == 0 ? J0 : (d == 1 ? J2 : J4), *JR = d == 0 ? J1 : (d == 1 ? J3 : J5);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            g[3 * v + d] = lane_derivative(c, &sU[v][base], stride, JL[v * 16 + fp], JR[v * 16 + fp]);
            asm volatile("" : "+v"(g[3 * v + d])::"memory");  // one by one, as below
        }
    }
#else
    const CoefTable<CT>& o = coef_lds<CT>();
    const CT* Di = o.D[i];
    const CT* Dj = o.D[j];
    const CT* Dk = o.D[k];
    const CT gLi = o.g[i][0], gRi = o.g[i][1];
    const CT gLj = o.g[j][0], gRj = o.g[j][1];
    const CT gLk = o.g[k][0], gRk = o.g[k][1];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT dz = 0, dxi = 0, deta = 0;
#pragma unroll
        for (int m = 0; m < 4; ++m) dz += Dk[m] * sU[v][zb + 16 * m];
#pragma unroll
        for (int m = 0; m < 4; ++m) dxi += Di[m] * sU[v][xb + m];
#pragma unroll
        for (int m = 0; m < 4; ++m) deta += Dj[m] * sU[v][yb + 4 * m];
        CT gx = dxi * a.jx, gy = deta * a.jy, gz = dz * a.jz;
        gx += J0[v * 16 + fpx] * gLi * a.jx;
        gx += J1[v * 16 + fpx] * gRi * a.jx;
        gy += J2[v * 16 + fpy] * gLj * a.jy;
        gy += J3[v * 16 + fpy] * gRj * a.jy;
        gz += J4[v * 16 + fpz] * gLk * a.jz;
        gz += J5[v * 16 + fpz] * gRk * a.jz;
        if (a.round_q) {  // Q_REAL round trip (rhs.cu:457-461), narrows only when CT is double
            gx = (CT)(float)gx;
            gy = (CT)(float)gy;
            gz = (CT)(float)gz;
        }
        // Finish variable v before the next variable's LDS reads: left to
        // itself the compiler issues all 90 reads first and computes at the
        // first use, which needs ~140 VGPRs (and spills at 4 waves/SIMD).
        asm volatile("" : "+v"(gx), "+v"(gy), "+v"(gz)::"memory");
        g[3 * v + 0] = gx;
        g[3 * v + 1] = gy;
        g[3 * v + 2] = gz;
    }
#endif
}

template <class UT, class CT>
__device__ __forceinline__ void lane_gradient(const StageArgs<UT, CT>& a, const CT (*sU)[64], const CT (*sJmp)[5][16],
                                              const TileTable& t, int i, int j, int k, CT* g) {
    lane_gradient_faces(a, sU, &sJmp[0][0][0], &sJmp[1][0][0], &sJmp[2][0][0], &sJmp[3][0][0], &sJmp[4][0][0],
                        &sJmp[5][0][0], t, i, j, k, g);
}

template <bool PF, class UT, class CT>
__device__ __forceinline__ void run_br1_jumps(const StageArgs<UT, CT>& a, const CT (*sU)[5][64],
                                              CT (*sJmp)[6][5][16], const Tile& tl, const CT* pf, int wave,
                                              int lane) {
    if (wave == 0) {
        br1_jumps<0, PF>(a, sU, sJmp, tl, pf, lane);
        br1_jumps<2, PF>(a, sU, sJmp, tl, pf, lane);
    } else {
        br1_jumps<1, PF>(a, sU, sJmp, tl, pf, lane);
    }
}

// The four viscous flux components 1..4 of one point, stored together
// (fv is point-major, component fastest) so that each lane moves them with
// one 16-byte (f32) access instead of four 4-byte ones.
template <class C>
struct alignas(4 * sizeof(C)) FvQuad {
    C c[4];
};

// Viscous normal flux at the element faces of direction D (the
// dispatch_viscous_flux calls of compute_face_j / compute_face_j_wall,
// rhs.cu:284-285, 318) from the Riemann-order state trace and the gradient
// slice; only the 11 gradient components the direction reads are traced.
// One face point: element e (state tile sUe, gradient tile sGe), face side
// `side` of direction D, face point fp.
template <int D, class UT, class CT>
__device__ __forceinline__ FvQuad<CT> fv_value(const StageArgs<UT, CT>& a, const CT (*sUe)[64],
                                               const CT (*sGe)[64], int64_t e, int side, int fp) {
    int base, stride;
    face_line(D, fp, base, stride);
    const Coef4<CT> c = side_coef<CT>(side);
    CT st[5], gt[15], fvv[5];
#pragma unroll
    for (int v = 0; v < 5; ++v)
        st[v] = trace4(sUe[v], base, stride, c.c0, c.c1, c.c2, c.c3, kOneX ? br1_order(D) : fv_order(D));
#pragma unroll
    for (int q = 0; q < 15; ++q) gt[q] = trace4_swz(sGe[q], base, stride, c.c0, c.c1, c.c2, c.c3, fv_order(D));
#if OD_FAST
    fast_visc_flux(D, fast_visc(a, st, gt, e), fvv + 1);
#else
    CT mu = a.sutherland ? sutherland(st, a.mu_ref, a.t_ref, a.s_suth) : a.mu;
    if (a.mu_t) mu = mu + a.mu_t[e];
    viscous_flux(D, st, gt, mu, fvv);
#endif
    return FvQuad<CT>{{fvv[1], fvv[2], fvv[3], fvv[4]}};
}

template <int D, class UT, class CT>
__device__ __forceinline__ void fv_point(const StageArgs<UT, CT>& a, const CT (*sUe)[64], const CT (*sGe)[64],
                                         int64_t e, int side, int fp) {
    *reinterpret_cast<FvQuad<CT>*>(a.fv + e * kFvStride + (2 * D + side) * 64 + fp * 4) =
        fv_value<D>(a, sUe, sGe, e, side, fp);
}

template <int D, class UT, class CT>
__device__ __forceinline__ void fv_pass(const StageArgs<UT, CT>& a, const CT (*sU)[5][64], const CT (*sG)[15][64],
                                        const Tile& tl, int lane) {
    const FaceTask t = face_task<D>(lane);
    if (!tile_valid(tl, t.le)) return;
    fv_point<D>(a, sU[t.le], sG[t.le], tile_eidx(tl, t.le), t.side, t.fp);
}

// Own-side face correction j from the interface flux fr of a face point
// (compute_face_j / compute_face_j_wall, rhs.cu:273-339): own is the
// element's trace, fvo / fvn the own and the neighbour's viscous normal flux
// (component 0 zero), right = the face is the element's right face.
template <int D, bool VISC, class CT>
__device__ __forceinline__ void face_correction(const CT* fr, const CT* own, const CT* fvo, const CT* fvn, bool wall,
                                                bool right, CT* jv) {
    OD_CONTRACT_IN_EXPRESSIONS
    CT fe[5];
    euler_flux(D, own, fe);
    CT wall_p = (CT)0;
    if (D == 1) wall_p = fe[2] - dv(own[2] * own[2], own[0]);  // rhs.cu:323-326
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const CT wf = (D == 1 && v == 2) ? wall_p : (CT)0.0;
        if (VISC) {
            const CT fl = right ? fvo[v] : fvn[v];
            const CT frr = right ? fvn[v] : fvo[v];
            CT jn;
            if constexpr (kHalfDiff<CT>) {
                // F* - (F_e - F_v,own) = (F_riemann - F_e) +- (F_vL - F_vR) / 2
                const CT hd = ((CT)0.5) * (fl - frr);
                jn = (fr[v] - fe[v]) + (right ? hd : -hd);
            } else {
                CT fc = fr[v] - ((CT)0.5) * (fl + frr);
                jn = fc - (fe[v] - fvo[v]);
            }
            CT jw = (wf - fvo[v]) - (fe[v] - fvo[v]);
            jv[v] = wall ? jw : jn;
        } else {
            jv[v] = wall ? (wf - fe[v]) : (fr[v] - fe[v]);
        }
    }
}

// The same correction at an interior face whose viscous half-difference
// hd = (F_vL - F_vR) / 2 (component 0 zero) is stored (fast f32 build).
template <int D, class CT>
__device__ __forceinline__ void face_correction_hd(const CT* fr, const CT* own, const CT* hd, bool right, CT* jv) {
    OD_CONTRACT_IN_EXPRESSIONS
    CT fe[5];
    euler_flux(D, own, fe);
#pragma unroll
    for (int v = 0; v < 5; ++v) jv[v] = (fr[v] - fe[v]) + (right ? hd[v] : -hd[v]);
}

// Interface flux at the element faces of direction D -> own-side correction
// j into LDS (compute_face_j / compute_face_j_wall, rhs.cu:273-339).
template <int D, bool VISC, bool PF, class UT, class CT>
__device__ __forceinline__ void flux_pass(const StageArgs<UT, CT>& a, const CT (*sU)[5][64], CT (*sJ)[6][5][16],
                                          const Tile& tl, const CT* pf, int lane) {
    const FaceTask t = face_task<D>(lane);
    if (!tile_valid(tl, t.le)) return;
    int base, stride;
    face_line(D, t.fp, base, stride);
    const Coef4<CT> c = side_coef<CT>(t.side);
    const bool right = t.side;
    CT own[5], oth[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) own[v] = trace4(sU[t.le][v], base, stride, c.c0, c.c1, c.c2, c.c3, face_order(D));
    const int64_t nb = (PF && !VISC) ? 0 : tile_nb<D>(tl, t.le, t.side);
    const bool wall = PF ? tile_wall<D>(tl, t.le, t.side) : nb < 0;
    // the neighbour's facing trace in the same order (x: 7/6 strict, 1/0 fast;
    // y: 3/2; z: 5/4)
    const int rf = (D == 0 && !kOneX) ? (right ? 6 : 7) : (t.f ^ 1);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT far;
        if constexpr (PF)
            far = pf[(t.le * 6 + t.f) * 80 + v * 16 + t.fp];
        else
            far = wall ? own[v] : a.tr_in[nb * kTraceStride + rf * 80 + v * 16 + t.fp];
        oth[v] = wall ? own[v] : far;
    }
    CT fvo[5] = {(CT)0, (CT)0, (CT)0, (CT)0, (CT)0}, fvn[5] = {(CT)0, (CT)0, (CT)0, (CT)0, (CT)0};
    if (VISC) {
        const FvQuad<CT> o =
            *reinterpret_cast<const FvQuad<CT>*>(a.fv + tile_eidx(tl, t.le) * kFvStride + t.f * 64 + t.fp * 4);
        FvQuad<CT> n = o;
        if (!wall) n = *reinterpret_cast<const FvQuad<CT>*>(a.fv + nb * kFvStride + (t.f ^ 1) * 64 + t.fp * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fvo[1 + q] = o.c[q];
            fvn[1 + q] = n.c[q];
        }
    }
    CT L[5], R[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        L[v] = right ? own[v] : oth[v];
        R[v] = right ? oth[v] : own[v];
    }
    CT fr[5], jv[5];
    interface_flux<D>(a.flux, L, R, fr);
    face_correction<D, VISC>(fr, own, fvo, fvn, wall, right, jv);
#pragma unroll
    for (int v = 0; v < 5; ++v) sJ[t.le][t.f][v][t.fp] = jv[v];
}

// Index of this wave in its work-group, as a wave-uniform (scalar) value: the
// compiler cannot tell that threadIdx.x >> 6 is the same in every lane, and
// per-wave conditions derived from it (the wave's element is valid, the
// wave's face directions) would otherwise branch on the execution mask.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Orders this wave's earlier LDS writes before its later LDS reads (of
// other lanes' data): a wave's LDS operations execute in order, so this only
// has to keep the compiler from moving them.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Streaming (non-temporal) accesses of the update kernels: the new state and
// its traces are read next by the visc kernel, which is bound by instruction
// issue rather than by memory, and the previous stage's state is not read
// again in this stage.  Marked as streaming they do not displace, in the
// memory-side cache, the viscous fluxes, state and traces that the visc
// kernel has just touched and the update kernel is about to read.
template <class T>
__device__ __forceinline__ T stream_load(const T* p) { return __builtin_nontemporal_load(p); }
template <class T>
__device__ __forceinline__ void stream_store(T v, T* p) { __builtin_nontemporal_store(v, p); }

// c * dt of the stage, from device memory where it is given there.  The update
// kernels read it before the FR correction, whose arithmetic covers the load:
// at the kernel's start it held up the first loads of the state, 0.1 us a
// launch, and after the first barrier it took registers for the whole kernel.
template <class UT, class CT>
__device__ __forceinline__ StageDt<UT, CT> stage_dt(const StageArgs<UT, CT>& a) {
    return a.dt ? *a.dt : StageDt<UT, CT>{a.cc, a.uc};
}

// Face traces of one element (its state tile sUe in LDS) -> dst, the
// element's kTraceStride block of tr_out.  The element's own wave writes
// them: 16 lanes per face, 4 faces per pass.  Without BR1 (Euler) the strict
// build skips the pairwise x traces, which only BR1 reads.  STREAM: streaming
// stores (the update kernels).
template <class CT, bool STREAM = false>
__device__ __forceinline__ void write_traces_own(const CT (*sUe)[64], CT* dst, int lane, bool need_pairwise_x) {
    const int fp = lane & 15;
#pragma unroll
    for (int pass = 0; pass < (kOwnFaces + 3) / 4; ++pass) {
        const int f = 4 * pass + (lane >> 4);
        if (f >= kOwnFaces || (!kOneX && !need_pairwise_x && f < 2)) continue;
        int base, stride;
        face_line(trace_face_dir(f), fp, base, stride);
        const Coef4<CT> c = side_coef<CT>(f & 1);
        const int order = trace_face_order(f);
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const CT tv = trace4(sUe[v], base, stride, c.c0, c.c1, c.c2, c.c3, order);
            if constexpr (STREAM)
                stream_store(tv, &dst[f * 80 + v * 16 + fp]);
            else
                dst[f * 80 + v * 16 + fp] = tv;
        }
    }
}

// State tile of element e into LDS, sUe[v][pt] = u[v][e][pt].  With an f32
// state and f32 compute each wave copies its element with LDS-DMA
// (global_load_lds_dword: no registers; the data lands with the
// neighbour-trace prefetch and is covered by the same wait); otherwise
// through registers with the cast to the compute type.
// Cache-policy operand of an LDS-DMA load: 0, or the non-temporal (streaming)
// bit of gfx950's cache policy, for data read once.
constexpr int kDmaDefault = 0;
constexpr int kDmaStream = 2;

template <class UT, class CT, int POLICY = kDmaDefault>
__device__ __forceinline__ void load_state_tile(const UT* u, int64_t NP, int64_t e, CT (*sUe)[64], int pt) {
    if constexpr (std::is_same<UT, float>::value && std::is_same<CT, float>::value) {
#pragma unroll
        for (int v = 0; v < 5; ++v)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(u + v * NP + e * 64 + pt),
                                             (__attribute__((address_space(3))) void*)&sUe[v][0], 4, 0, POLICY);
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) sUe[v][pt] = (CT)u[v * NP + e * 64 + pt];
    }
}

#if OD_FAST
// Divergence of the volume viscous fluxes at the lane's point (the F_v half
// of accumulate_volume_rhs_shfl / _z, rhs.cu:229-266) from its state st and
// corrected gradient g, x then y then z, components 1..4 (F_v of the mass
// equation is zero) -> the element's fv block after its face part.  S: this
// wave's 256-float LDS staging area.
template <class UT>
__device__ __forceinline__ void visc_divergence(const StageArgs<UT, float>& a, int64_t e, const float* st,
                                                const float* g, const BoxTable& o, float* S, int i, int j, int k, int pt) {
    const FastVisc f = fast_visc(a, st, g, e);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        float fvv[4];
        fast_visc_flux(d, f, fvv);
        if (d == 0) {
            const float* Dx = o.D[0][i];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] = quad_line(Dx, fvv[q]);
            continue;
        }
        if (d > 1) wave_sync();  // the previous direction's reads are done
#pragma unroll
        for (int q = 0; q < 4; ++q) S[q * 64 + pt] = fvv[q];
        wave_sync();
        const int idx = d == 1 ? j : k;
        const int base = d == 1 ? i + 16 * k : i + 4 * j;
        const int stride = d == 1 ? 4 : 16;
        const float* Dd = o.D[d][idx];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[q] = __builtin_fmaf(Dd[m], S[q * 64 + base + m * stride], acc[q]);
    }
    FvQuad<float>* dst = reinterpret_cast<FvQuad<float>*>(a.fv + e * kFvStride + kFvFaces + pt * 4);
    *dst = FvQuad<float>{{acc[0], acc[1], acc[2], acc[3]}};
}
#endif

// Volume RHS at the lane's point, state st (rhs.cu:229-266, 490-510): minus the
// divergence of F_e (VISC: of F_e - F_v, from the corrected gradient g), x then
// y then z, plus the body force, with the RHS_REAL round trip (rhs.cu:509,
// rk.cu:52).  S: this wave's [5][64] LDS staging area.  Strict build, and the
// fast build's Euler fluxes (vdiv: the divergence of the viscous ones).
template <bool VISC, class UT, class CT>
__device__ __forceinline__ void volume_rhs(const StageArgs<UT, CT>& a, const CT* st, const CT* g, CT mu,
                                           const CT* vdiv, const Rows<CT>& o, CT (*S)[64], int i, int j, int k,
                                           int pt, CT* out) {
    CT rs[5] = {(CT)0, (CT)0, (CT)0, (CT)0, (CT)0};
    ViscPoint<CT> vp;
    if constexpr (VISC) vp = viscous_point(st, g, mu, 7);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        CT F[5];
        euler_flux(d, st, F);
        if constexpr (VISC) {
            CT fvv[5];
            viscous_flux_dir(d, vp, fvv);
#pragma unroll
            for (int v = 0; v < 5; ++v) F[v] = F[v] - fvv[v];
        }
#if OD_FAST
        if (d == 0) {
            const float* Dx = o.D[0][i];
#pragma unroll
            for (int v = 0; v < 5; ++v) rs[v] = quad_line(Dx, F[v]);
            continue;
        }
#endif
        if (d > (OD_FAST ? 1 : 0)) wave_sync();  // the previous direction's reads are done
#pragma unroll
        for (int v = 0; v < 5; ++v) S[v][pt] = F[v];
        wave_sync();
        const int idx = d == 0 ? i : (d == 1 ? j : k);
        const int base = d == 0 ? 4 * j + 16 * k : (d == 1 ? i + 16 * k : i + 4 * j);
        const int stride = d == 0 ? 1 : (d == 1 ? 4 : 16);
#if OD_FAST
        const float* Dd = o.D[d][idx];
#pragma unroll
        for (int v = 0; v < 5; ++v)
#pragma unroll
            for (int m = 0; m < 4; ++m) rs[v] = __builtin_fmaf(Dd[m], S[v][base + m * stride], rs[v]);
#else
        const CT jac = d == 0 ? a.jx : (d == 1 ? a.jy : a.jz);
        const CT* Dd = o.D[idx];
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            CT dd = 0;
#pragma unroll
            for (int m = 0; m < 4; ++m) dd += Dd[m] * S[v][base + m * stride];
            rs[v] += dd * jac;
        }
#endif
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT val = -rs[v];
        if (vdiv && v > 0) val += vdiv[v - 1];  // + div F_v from the visc kernel
        if (v == 1) val += a.bf;
        out[v] = a.round_rhs ? (CT)(float)val : val;
    }
}

// ---------------------------------------------------------------------------
// Kernels.
// ---------------------------------------------------------------------------
// LDS of one tile (two elements).  The prefetch buffer comes first so that
// its 16-byte LDS-DMA rows start on a 16-byte boundary.
// With the prefetch (f32 compute) the gradient tile sG reuses the prefetched
// traces and the BR1 jumps (960 floats each, contiguous): element 0's
// gradients take the prefetch buffer, element 1's the jumps, written only
// after both waves have finished reading them (a barrier).  Between the
// jumps and the gradient tile the volume fluxes' lines of element w are staged
// (vol_stage) in its half of the prefetch buffer, whose traces are consumed by
// then, or without a prefetch in the element's own jumps, which only wave w
// reads and has read by then.
template <class CT>
struct ViscLds {
    static constexpr bool kPF = std::is_same<CT, float>::value;
    float pf[kPF ? kPfFloats : 4];
    CT sJmp[kEpb][6][5][16];
    CT sU[kEpb][5][64];
    CT sG_own[kPF ? 0 : kEpb][15][64];  // zero-length when aliased
#if OD_FAST
    TileTable tab;  // of the tile's box: a batch's work-group may have tiles of two boxes
    __device__ const BoxTable& rows() { return tab; }
    __device__ const TileTable& tile_table() { return tab; }
#else
    __device__ TileTable tile_table() { return {}; }
    __device__ const CoefTable<CT>& rows() { return coef_lds<CT>(); }
#endif
    __device__ CT (*sG())[15][64] {
        static_assert(!kPF || (kPfFloats == 15 * 64 && sizeof(sJmp) == kPfFloats * sizeof(float)), "sG aliasing layout");
        if constexpr (kPF) return reinterpret_cast<CT(*)[15][64]>(pf);
        else return sG_own;
    }
    __device__ CT* vol_stage(int w) {  // 5 * 64 values
        if constexpr (kPF) return reinterpret_cast<CT*>(pf) + w * 320;
        else return &sJmp[w][0][0][0];
    }
};

// With the prefetch (f32 compute) the face-correction array sJ shares the
// prefetched neighbour traces (they have sJ's exact layout and each face
// point's lane reads its entries there before it writes them).  sF: staging of
// the volume fluxes' lines, where this kernel forms them (kVol): the Euler mode
// and the fast build.
template <class CT, bool VISC>
struct UpdateLds {
    static constexpr bool kPF = std::is_same<CT, float>::value;
    static constexpr bool kVol = !VISC || kSplitVisc<CT>;
    float pf[kPF ? kPfFloats : 4];
    CT sU[kEpb][5][64];
    CT sJ_own[kPF ? 0 : kEpb][6][5][16];  // zero-length when aliased
    CT sF[kVol ? kEpb : 0][5][64];
#if OD_FAST
    BoxTable tab;  // of the tile's box: a batch's work-group may have tiles of two boxes
    __device__ const BoxTable& rows() { return tab; }
#else
    __device__ const CoefTable<CT>& rows() { return coef_lds<CT>(); }
#endif
    __device__ CT (*sJ())[6][5][16] {
        if constexpr (kPF) return reinterpret_cast<CT(*)[6][5][16]>(pf);
        else return sJ_own;
    }
};

// Face traces of the state -> tr_out (wave w loads element w of the tile).
template <class UT, class CT>
__device__ __forceinline__ void trace_body(const StageArgs<UT, CT>& a, const Tile& tl, CT (*sU)[5][64], int wave,
                                           int pt) {
    const CT cf = coef_load(a, (int)threadIdx.x);
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    if (tile_valid(tl, wave)) {
#pragma unroll
        for (int v = 0; v < 5; ++v) sU[wave][v][pt] = (CT)a.uin[v * NP + tile_eidx(tl, wave) * 64 + pt];
    }
    coef_store<CT>((int)threadIdx.x, cf);
    __syncthreads();
    if (tile_valid(tl, wave)) write_traces_own(sU[wave], a.tr_out + tile_eidx(tl, wave) * kTraceStride, pt, true);
}

// Corrected gradients of the tile's elements and the viscous fluxes at
// their own faces -> fv.
template <class UT, class CT>
__device__ __forceinline__ void visc_body(const StageArgs<UT, CT>& a, const Tile& tl, ViscLds<CT>& L, int wave,
                                          int pt) {
    constexpr bool PF = std::is_same<CT, float>::value;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    const CT cf = coef_load(a, (int)threadIdx.x);
#if OD_FAST
    const float row = tile_table_load<TileTable>(a, wave * 64 + pt);
#endif
    if constexpr (PF) prefetch_issue<false>(a, tl, L.pf, wave, pt);
    if (tile_valid(tl, wave)) load_state_tile(a.uin, NP, tile_eidx(tl, wave), L.sU[wave], pt);
    coef_store<CT>((int)threadIdx.x, cf);
#if OD_FAST
    tile_table_store(L.tab, wave * 64 + pt, row);
#endif
    if constexpr (PF) __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS copies have landed
    __syncthreads();
    run_br1_jumps<PF>(a, L.sU, L.sJmp, tl, reinterpret_cast<const CT*>(L.pf), wave, pt);
    __syncthreads();
    CT g[15];
    if (tile_valid(tl, wave)) lane_gradient(a, L.sU[wave], L.sJmp[wave], L.tile_table(), i, j, k, g);
    if (tile_valid(tl, wave)) {
        const int64_t e = tile_eidx(tl, wave);
        CT st[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) st[v] = L.sU[wave][v][pt];
        wave_sync();  // without a prefetch the staging area is the jumps just read
#if OD_FAST
        visc_divergence(a, e, st, g, L.rows(), L.vol_stage(wave), i, j, k, pt);
#else
        CT r[5];
        CT mu = a.sutherland ? sutherland(st, a.mu_ref, a.t_ref, a.s_suth) : a.mu;
        if (a.mu_t) mu = mu + a.mu_t[e];
        volume_rhs<true>(a, st, g, mu, (const CT*)nullptr, L.rows(), (CT(*)[64])L.vol_stage(wave), i, j, k, pt, r);
#pragma unroll
        for (int v = 0; v < 5; ++v) a.fv[e * kFvStride + kFvFaces + v * 64 + pt] = r[v];
#endif
    }
    if constexpr (PF) __syncthreads();  // sG overwrites the jumps the other wave may still read
    if (tile_valid(tl, wave)) {
#pragma unroll
        for (int q = 0; q < 15; ++q) L.sG()[wave][q][swz64(pt)] = g[q];
    }
    __syncthreads();
    if (wave == 0) {
        fv_pass<0>(a, L.sU, L.sG(), tl, pt);
        fv_pass<2>(a, L.sU, L.sG(), tl, pt);
    } else {
        fv_pass<1>(a, L.sU, L.sG(), tl, pt);
    }
}

// Stage update of a point: u^n, the stage's state and its RHS -> the new state
// (rk.cu:12-25, 63-82).
template <class UT, class CT>
__device__ __forceinline__ void rk_stage(const StageArgs<UT, CT>& a, const StageDt<UT, CT>& cdt, const UT* uprv,
                                         const UT* ucr, const CT* rts, UT* unew) {
    if constexpr (std::is_same<UT, CT>::value) {
        // one type: the compute-type and the state-type blends differ only
        // in their coefficients, chosen once; uniform branch on the stage
        const CT kA = a.accum_state ? a.ua : a.ca;
        const CT kB = a.accum_state ? a.ub : a.cb;
        const CT kC = a.accum_state ? cdt.uc : cdt.cc;
        if (a.stage1) {
#pragma unroll
            for (int v = 0; v < 5; ++v) unew[v] = rk_blend1(kA, kC, uprv[v], rts[v]);
        } else {
#pragma unroll
            for (int v = 0; v < 5; ++v) unew[v] = rk_blend(kA, kB, kC, uprv[v], ucr[v], rts[v]);
        }
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const CT rt = rts[v];
            if (!a.accum_state) {
                CT up = (CT)uprv[v], uc = (CT)ucr[v];
                CT val = a.stage1 ? (a.ca * up + cdt.cc * rt) : (a.ca * up + a.cb * uc + cdt.cc * rt);
                unew[v] = (UT)val;
            } else {
                UT rr = (UT)rt;
                unew[v] =
                    a.stage1 ? (UT)(a.ua * uprv[v] + cdt.uc * rr) : (UT)(a.ua * uprv[v] + a.ub * ucr[v] + cdt.uc * rr);
            }
        }
    }
}

// Full stage for the tile: volume RHS, interface fluxes, FR correction, RK
// blend, and the face traces of the new state.  WIDE, for small boxes, whose
// kernels last as long as one work-group: more waves than elements; the first
// two own an element in the point-wise phases, and the faces of each direction
// are another wave's, beside the volume RHS where this kernel forms it, so that
// no wave does two things in a row that could be done at once.  HOLD: a state of
// another type than the fluxes' stays in registers (see kHoldTiles; in the strict
// build it would cost them a wave per SIMD).
template <class CT, bool VISC>
constexpr int kWideWaves = UpdateLds<CT, VISC>::kVol ? 5 : 3;
template <class UT, class CT, bool VISC, bool WIDE = false, bool HOLD = false>
__device__ __forceinline__ void update_body(const StageArgs<UT, CT>& a, const Tile& tl, UpdateLds<CT, VISC>& L,
                                            int wave, int pt) {
    constexpr bool PF = std::is_same<CT, float>::value;
    const CT* pfc = reinterpret_cast<const CT*>(L.pf);
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const bool owner = !WIDE || wave < kEpb;
    const bool mine = owner && tile_valid(tl, wave);
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    const int64_t gbase = tile_eidx(tl, wave) * 64 + pt;
    const CT cf = coef_load(a, (int)threadIdx.x);
#if OD_FAST
    const float row = tile_table_load<BoxTable>(a, wave * 64 + pt);
#endif
    if constexpr (PF) {
        if (owner) prefetch_issue<true>(a, tl, L.pf, wave, pt);
    }

    constexpr bool SAME = std::is_same<UT, CT>::value;  // sU holds the state exactly
    static_assert(!(SAME && HOLD), "sU holds it");
    UT held[HOLD ? 5 : 1];
    if constexpr (SAME && PF) {  // f32 state and compute: LDS-DMA
        if (mine) {
            load_state_tile(a.uin, NP, tile_eidx(tl, wave), L.sU[wave], pt);
        } else if (owner) {
#pragma unroll
            for (int v = 0; v < 5; ++v) L.sU[wave][v][pt] = (CT)1;
        }
    } else if (owner) {
#pragma unroll
        for (int v = 0; v < 5; ++v) {
            const UT x = mine ? a.uin[v * NP + gbase] : (UT)1;
            if constexpr (HOLD) held[v] = x;
            L.sU[wave][v][pt] = (CT)x;
        }
    }
    coef_store<CT>((int)threadIdx.x, cf);
#if OD_FAST
    tile_table_store(L.tab, wave * 64 + pt, row);
#endif
    if constexpr (PF) __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS copies have landed
    __syncthreads();

    // Volume RHS: formed here in the Euler mode and the fast build (which adds
    // the visc kernel's viscous divergence) and kept in LDS during the face
    // passes; else the visc kernel's, read after them.
    constexpr bool VOL = UpdateLds<CT, VISC>::kVol;
    if constexpr (VOL) if (owner) {
        CT vdiv[4] = {(CT)0, (CT)0, (CT)0, (CT)0}, r[5];
        if constexpr (VISC) {
            if (mine) {
                const FvQuad<CT> src =
                    *reinterpret_cast<const FvQuad<CT>*>(a.fv + tile_eidx(tl, wave) * kFvStride + kFvFaces + pt * 4);
#pragma unroll
                for (int q = 0; q < 4; ++q) vdiv[q] = src.c[q];
            }
        }
        CT st[5];
#pragma unroll
        for (int v = 0; v < 5; ++v) st[v] = L.sU[wave][v][pt];
        volume_rhs<false>(a, st, (const CT*)nullptr, (CT)0, VISC ? vdiv : (const CT*)nullptr, L.rows(), L.sF[wave], i, j,
                          k, pt, r);
        wave_sync();
#pragma unroll
        for (int v = 0; v < 5; ++v) L.sF[wave][v][pt] = r[v];
    }

    // Interface fluxes at all own faces, direction by direction.
    if constexpr (WIDE) {
        const int d = wave - (VOL ? kEpb : 0);
        if (d == 0)
            flux_pass<0, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
        else if (d == 1)
            flux_pass<1, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
        else if (d == 2)
            flux_pass<2, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
    } else if (wave == 0) {
        flux_pass<0, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
        flux_pass<2, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
    } else {
        flux_pass<1, VISC, PF>(a, L.sU, L.sJ(), tl, pfc, pt);
    }
    __syncthreads();
    if (!owner) return;

    // FR correction and stage update (rk.cu:12-25, 63-82).
    const StageDt<UT, CT> cdt = stage_dt(a);
    const Rows<CT>& o = L.rows();
#if OD_FAST
    const CT gLi = o.g[0][i][0], gRi = o.g[0][i][1];
    const CT gLj = o.g[1][j][0], gRj = o.g[1][j][1];
    const CT gLk = o.g[2][k][0], gRk = o.g[2][k][1];
#else
    const CT gLi = o.g[i][0], gRi = o.g[i][1];
    const CT gLj = o.g[j][0], gRj = o.g[j][1];
    const CT gLk = o.g[k][0], gRk = o.g[k][1];
#endif
    const int fpx = j + 4 * k, fpy = i + 4 * k, fpz = i + 4 * j;
    UT uprv[5], ucr[5];
    CT r[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        // the state in its own type: from LDS, held, or again from L2
        if constexpr (SAME)
            ucr[v] = (UT)L.sU[wave][v][pt];
        else if constexpr (HOLD)
            ucr[v] = held[v];
        else
            ucr[v] = mine ? a.uin[v * NP + gbase] : (UT)1;
        if constexpr (VOL)
            r[v] = L.sF[wave][v][pt];
        else
            r[v] = mine ? stream_load(&a.fv[tile_eidx(tl, wave) * kFvStride + kFvFaces + v * 64 + pt]) : (CT)0;
    }
    if (a.stage1) {  // u^n is the state this stage read (uprev == uin): no second load
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = ucr[v];
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = mine ? stream_load(&a.uprev[v * NP + gbase]) : (UT)1;
    }
    CT rts[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const CT(*J)[5][16] = L.sJ()[wave];
#if OD_FAST
        CT cx = -(J[0][v][fpx] * gLi + J[1][v][fpx] * gRi);
        CT cy = -(J[2][v][fpy] * gLj + J[3][v][fpy] * gRj);
        CT cz = -(J[4][v][fpz] * gLk + J[5][v][fpz] * gRk);
#else
        CT cx = -(J[0][v][fpx] * gLi * a.jx) - (J[1][v][fpx] * gRi * a.jx);
        CT cy = -(J[2][v][fpy] * gLj * a.jy) - (J[3][v][fpy] * gRj * a.jy);
        CT cz = -(J[4][v][fpz] * gLk * a.jz) - (J[5][v][fpz] * gRk * a.jz);
#endif
        rts[v] = r[v] + (cx + cy + cz);
    }
    if (a.mode == 1) {  // the stage's RHS into dbg, state unchanged
#pragma unroll
        for (int v = 0; v < 5; ++v)
            if (mine) a.dbg[v * NP + gbase] = rts[v];
        return;
    }
    UT unew[5];
    rk_stage(a, cdt, uprv, ucr, rts, unew);
#pragma unroll
    for (int v = 0; v < 5; ++v)
        if (mine) stream_store(unew[v], &a.uout[v * NP + gbase]);

    // Face traces of the new state for the next stage, each wave those of its
    // own element: from the RK phase on only wave w reads sU[w], so no
    // work-group barrier is needed.
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sU[wave][v][pt] = (CT)unew[v];
    wave_sync();
    if (mine) write_traces_own<CT, true>(L.sU[wave], a.tr_out + tile_eidx(tl, wave) * kTraceStride, pt, VISC);
}

template <class UT, class CT>
__global__ __launch_bounds__(128) void od_trace_kernel(StageArgs<UT, CT> a) {
    __shared__ CT sU[kEpb][5][64];
    trace_body(a, make_tile(a), sU, wave_index(), threadIdx.x & 63);
}

#if OD_FAST
template <class UT, class CT>
__global__ __launch_bounds__(128) void od_visc_kernel(StageArgs<UT, CT> a) {
    __shared__ ViscLds<CT> L;
    visc_body(a, make_tile(a), L, wave_index(), threadIdx.x & 63);
}
#endif

// Occupancy target of the update kernels.  The fast all-f32 single-box kernel
// and the batch kernel's single-unit form are held to 64 VGPRs (8 waves per
// SIMD; they need 51 to 59 with no spills; their LDS, 9.6 KB per work-group of
// 128 threads, allows 8).  The strict build (70 VGPRs, 7 waves), f64 states and
// the persistent batch kernel keep their natural allocation (the 4-wave cap does
// not bind); f64 compute needs 115 to 122 VGPRs (4 waves).
template <class CT>
constexpr int kMinWaves = sizeof(CT) == 4 ? 4 : 1;
template <class UT, class CT>
constexpr int kMinWavesUpdate = (OD_FAST && sizeof(UT) == 4 && sizeof(CT) == 4) ? 8 : kMinWaves<CT>;

template <class UT, class CT, bool VISC, bool WIDE, bool HOLD>
__global__ __launch_bounds__((64 * (WIDE ? kWideWaves<CT, VISC> : kEpb))) __attribute__((amdgpu_waves_per_eu(kMinWavesUpdate<UT, CT>))) void od_update_kernel(
    StageArgs<UT, CT> a) {
    __shared__ UpdateLds<CT, VISC> L;
    update_body<UT, CT, VISC, WIDE, HOLD>(a, make_tile_reversed(a), L, wave_index(), threadIdx.x & 63);
}

// LDS area of one element in the kernels that work by lines: [5][64] or
// [15][64] in swz64 order; areas lie 4 values further apart than their size.
constexpr int kAreaStride = 15 * 64 + 4;
// swz64 position of the line point m of direction D relative (XOR) to m = 0.
template <int D>
__device__ constexpr int line_xor(int m) {
    const int lo = m & 1, hi = m >> 1;
    return D == 0 ? ((lo ? 1 | 2 | 32 : 0) | hi << 2) : (D == 1 ? (lo | hi << 3) : (hi << 1 | lo << 4));
}

// Blocks of 2x2x2 elements: local element lx + 2 ly + 4 lz.
constexpr int kBlk = 8;

struct Block {
    int32_t ex0, ey0, ez0;  // coordinates of local element 0 (even)
    int32_t e0;             // its element index
};

// REVERSE: the work-group -> block map runs backwards (the last block of the
// mesh first).  The visc kernel walks the mesh forwards and the update kernel
// backwards, so each kernel starts where the previous one ended, on the data
// that kernel touched last (its neighbour traces, viscous fluxes, state),
// which is the most likely to still be in the memory-side cache.
template <bool REVERSE, class UT, class CT>
__device__ __forceinline__ Block make_block(const StageArgs<UT, CT>& a) {
    Block b;
    const int bx = REVERSE ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
    const int by = REVERSE ? (int)(gridDim.y - 1 - blockIdx.y) : (int)blockIdx.y;
    const int bz = REVERSE ? (int)(gridDim.z - 1 - blockIdx.z) : (int)blockIdx.z;
    b.ex0 = 2 * bx;
    b.ey0 = 2 * by;
    b.ez0 = 2 * bz;
    b.e0 = b.ex0 + a.nx * (b.ey0 + a.ny * b.ez0);
    return b;
}

// Bit d of a local element index: its coordinate along d in the block, and
// the side (0 left, 1 right) of its external face normal to d.
__device__ __forceinline__ int blk_bit(int le, int d) { return (le >> d) & 1; }

template <class UT, class CT>
__device__ __forceinline__ int blk_elem(const StageArgs<UT, CT>& a, const Block& b, int le) {
    return b.e0 + (le & 1) + a.nx * (((le >> 1) & 1) + a.ny * (le >> 2));
}

// Neighbour across the external face normal to d of local element le (as
// make_elem forms it); -1 = slip wall.  Branch-free: the offsets of the
// block's left (bit d = 0) and right (bit d = 1) external neighbours are
// block-uniform, each lane selects by its element's bit.
template <class UT, class CT>
__device__ __forceinline__ int blk_ext_nb(const StageArgs<UT, CT>& a, const Block& b, int le, int d) {
    const int e = blk_elem(a, b, le);
    const int s = blk_bit(le, d);
    const int n = d == 0 ? a.nx : (d == 1 ? a.ny : a.nz);
    const int c0 = d == 0 ? b.ex0 : (d == 1 ? b.ey0 : b.ez0);  // the block's left coordinate along d
    const int stride = d == 0 ? 1 : (d == 1 ? a.nx : a.nx * a.ny);
    const int off_l = (c0 == 0 ? n - 1 : -1) * stride;
    const int off_r = (c0 + 1 == n - 1 ? 1 - n : 1) * stride;
    const bool wall_l = d == 1 && a.wall && c0 == 0;
    const bool wall_r = d == 1 && a.wall && c0 + 1 == n - 1;
    return (s ? wall_r : wall_l) ? -1 : e + (s ? off_r : off_l);
}

// Left element of pair p (0..3) along direction D of a block; the right one is
// 2^D further.
template <int D>
__device__ __forceinline__ int blk_pair(int p) {
    return D == 0 ? 2 * p : (D == 1 ? ((p & 1) | ((p >> 1) << 2)) : p);
}

// The line waves are waves 0..5 or 2..7 of a work-group in turn, so that the
// SIMDs of a CU get equally many of them.  Work-groups go round the XCDs, so
// it is every eighth that turns.
__device__ __forceinline__ int line_role(int group) { return (wave_index() + ((group >> 3) & 1) * 6) & 7; }

// The value of the lane's partner, lane ^ 1.
__device__ __forceinline__ float lane_partner(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, false));  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ double lane_partner(double x) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xF, 0xF, false),
                            __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xF, 0xF, false));
}

#if !OD_FAST
// ---------------------------------------------------------------------------
// Strict build, one box: the visc kernel by lines.  A 256-thread work-group has
// four consecutive elements; in the line phases wave d < 3 takes direction d,
// lane = (element, line of four points), and forms from one read of the line's
// states both end traces, both BR1 jumps and the corrected derivative at its
// four points, then from one read of the line's gradients the viscous fluxes at
// both ends.  The neighbours' traces come straight from memory, the operators
// are wave-uniform.  The volume RHS is point-wise, a wave per element.  Every
// value is the expression of visc_body, in the reference's order.
// Bounds: instruction issue.  Against the point-wise form (visc_body, which the
// batches' tiles use), whose lanes read each state 12 and each gradient 6 to 8
// times from LDS: 24x26x22 f64 102 -> 61 us, 48^3 f32 279 -> 231 us, 24x20x28
// f64 state with f32 fluxes 40 -> 33 us a launch.
// LDS: one area per element, the states, then the gradients over them.
// ---------------------------------------------------------------------------
constexpr int kQuad = 4;

template <class CT>
struct StrictLine {
    int e;            // element, -1: none
    int fp, side;     // face point; blocks: the element's coordinate along D
    CT u[5][4];
    CT tl[5], tr[5];  // end traces in the order of the viscous fluxes
    CT nl[5], nr[5];  // the neighbours' facing traces (blocks: nl, across the external face)
    bool wl, wr;      // slip walls (blocks: wl, at the external face)
    int pos[4];
};

// A block's line wave: half of the pairs of elements along D, lane = (pair,
// line, side).  The neighbour across the internal face is the next lane.
template <int D, class UT, class CT>
__device__ __forceinline__ void strict_block_begin(const StageArgs<UT, CT>& a, const Block& b, int half, int lane,
                                                   StrictLine<CT>& w) {
    w.side = lane & 1;
    w.fp = (lane >> 1) & 15;
    const int le = blk_pair<D>(2 * half + (lane >> 5)) + (w.side << D);
    w.e = blk_elem(a, b, le);
    const int nb = blk_ext_nb(a, b, le, D);
    w.wl = D == 1 && nb < 0;
    const CT* t = a.tr_in + (int64_t)(w.wl ? w.e : nb) * kTraceStride + (2 * D + 1 - w.side) * 80 + w.fp;
#pragma unroll
    for (int v = 0; v < 5; ++v) w.nl[v] = t[v * 16];
    int base, stride;
    face_line(D, w.fp, base, stride);
    const int s0 = swz64(base);
#pragma unroll
    for (int m = 0; m < 4; ++m) w.pos[m] = le * kAreaStride + (s0 ^ line_xor<D>(m));
}

// Element e0's coordinates and the neighbours across both faces of direction D
// of the lane's element e0 + le (those past the mesh's last one repeat it).
template <int D, class UT, class CT>
__device__ __forceinline__ void strict_line_begin(const StageArgs<UT, CT>& a, int e0, int E, int lane,
                                                  StrictLine<CT>& w) {
    const int le = lane >> 4;
    w.e = e0 + le < E ? e0 + le : -1;
    w.fp = lane & 15;
    int ez = e0 / (a.nx * a.ny), ey = (e0 - ez * a.nx * a.ny) / a.nx, ex = e0 - a.nx * (ey + a.ny * ez);
    int l[kQuad], r[kQuad];
#pragma unroll
    for (int q = 0; q < kQuad; ++q) {
        const Elem n = make_elem(ex, ey, ez, a.nx, a.ny, a.nz, a.wall);
        l[q] = D == 0 ? n.xl : (D == 1 ? n.yl : n.zl);
        r[q] = D == 0 ? n.xr : (D == 1 ? n.yr : n.zr);
        if (e0 + q + 1 < E) {
            ++ex;
            if (ex == a.nx) {
                ex = 0;
                ++ey;
                if (ey == a.ny) {
                    ey = 0;
                    ++ez;
                }
            }
        }
    }
    const bool b0 = le & 1, b1 = le & 2;
    const int nl = b1 ? (b0 ? l[3] : l[2]) : (b0 ? l[1] : l[0]);
    const int nr = b1 ? (b0 ? r[3] : r[2]) : (b0 ? r[1] : r[0]);
    w.wl = D == 1 && nl < 0;
    w.wr = D == 1 && nr < 0;
    const CT* tl = a.tr_in + (int64_t)(w.wl ? 0 : nl) * kTraceStride + (2 * D + 1) * 80 + w.fp;
    const CT* tr = a.tr_in + (int64_t)(w.wr ? 0 : nr) * kTraceStride + (2 * D) * 80 + w.fp;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        w.nl[v] = tl[v * 16];
        w.nr[v] = tr[v * 16];
    }
    int base, stride;
    face_line(D, w.fp, base, stride);
    const int s0 = swz64(base);
#pragma unroll
    for (int m = 0; m < 4; ++m) w.pos[m] = le * kAreaStride + (s0 ^ line_xor<D>(m));
}

// Jumps (br1_jumps) and corrected derivative along D (lane_gradient_faces) ->
// the gradient's rows 3 v + D.
template <int D, bool BLOCK, class UT, class CT>
__device__ __forceinline__ void strict_line_gradient(const StageArgs<UT, CT>& a, CT* area, StrictLine<CT>& w) {
    const Ops<CT>& o = dev_ops<CT>();
    const CT jac = D == 0 ? a.jx : (D == 1 ? a.jy : a.jz);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const CT* u = w.u[v];
        const CT tl = trace4(u, 0, 1, o.eL[0], o.eL[1], o.eL[2], o.eL[3], br1_order(D));
        const CT tr = trace4(u, 0, 1, o.eR[0], o.eR[1], o.eR[2], o.eR[3], br1_order(D));
        const CT sign = (v > 0 && v < 4) ? ((CT)-1.0) : ((CT)1.0);
        CT nl, nr;
        if constexpr (BLOCK) {
            const CT in = lane_partner(w.side ? tl : tr);
            const CT ext = w.wl ? (w.side ? tr : tl) * sign : w.nl[v];
            nl = w.side ? in : ext;
            nr = w.side ? ext : in;
        } else {
            nl = w.wl ? tl * sign : w.nl[v];
            nr = w.wr ? tr * sign : w.nr[v];
        }
        const CT jl = ((CT)0.5) * (nl + tl) - tl, jr = ((CT)0.5) * (nr + tr) - tr;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            CT d = 0;
#pragma unroll
            for (int m = 0; m < 4; ++m) d += o.D[4 * i + m] * u[m];
            CT g = d * jac;
            g += jl * o.gL[i] * jac;
            g += jr * o.gR[i] * jac;
            if (a.round_q) g = (CT)(float)g;  // Q_REAL round trip (rhs.cu:457-461)
            area[w.pos[i] + (3 * v + D) * 64] = g;
        }
        w.tl[v] = D == 0 ? trace4(u, 0, 1, o.eL[0], o.eL[1], o.eL[2], o.eL[3], fv_order(D)) : tl;
        w.tr[v] = D == 0 ? trace4(u, 0, 1, o.eR[0], o.eR[1], o.eR[2], o.eR[3], fv_order(D)) : tr;
        asm volatile("" : "+v"(w.tl[v]), "+v"(w.tr[v])::"memory");  // variable by variable (see lane_gradient_faces)
    }
}

// Viscous flux at one end of the line (fv_value) from its state trace and
// gradient trace -> the element's slot of face 2 D + side.
template <int D, class UT, class CT>
__device__ __forceinline__ void strict_end_flux(const StageArgs<UT, CT>& a, int64_t e, bool valid, const CT* st,
                                                const CT* gt, int side, int fp) {
    CT f[5];
    CT mu = a.sutherland ? sutherland(st, a.mu_ref, a.t_ref, a.s_suth) : a.mu;
    if (a.mu_t) mu = mu + a.mu_t[e];
    viscous_flux(D, st, gt, mu, f);
    if (valid)
        *reinterpret_cast<FvQuad<CT>*>(a.fv + e * kFvStride + (2 * D + side) * 64 + fp * 4) =
            FvQuad<CT>{{f[1], f[2], f[3], f[4]}};
}
template <int D, class UT, class CT>
__device__ __forceinline__ void strict_line_flux(const StageArgs<UT, CT>& a, const CT* area, const StrictLine<CT>& w) {
    const Ops<CT>& o = dev_ops<CT>();
    CT gl[15], gr[15];
#pragma unroll
    for (int q = 0; q < 15; ++q) {
        // what the flux along D reads: the density's gradient, the momenta's
        // along D, across D of momentum D and on the diagonal, the energy's along D
        const int v = q / 3, c = q % 3;
        const bool used = v == 0 || c == D || (v < 4 && (v - 1 == D || v - 1 == c));
        if (!used) {
            gl[q] = gr[q] = (CT)0;
            continue;
        }
        CT x[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = area[w.pos[m] + q * 64];
        gl[q] = trace4(x, 0, 1, o.eL[0], o.eL[1], o.eL[2], o.eL[3], fv_order(D));
        gr[q] = trace4(x, 0, 1, o.eR[0], o.eR[1], o.eR[2], o.eR[3], fv_order(D));
        asm volatile("" : "+v"(gl[q]), "+v"(gr[q])::"memory");
    }
    const bool valid = w.e >= 0;
    const int64_t e = valid ? w.e : 0;
    strict_end_flux<D>(a, e, valid, w.tl, gl, 0, w.fp);
    asm volatile("" ::: "memory");  // one end, then the other
    strict_end_flux<D>(a, e, valid, w.tr, gr, 1, w.fp);
}

// BLOCK: the elements of block b, else the N consecutive ones from e0.
// D, half: this wave's direction (3: none) and half of the pairs along it.
template <bool BLOCK, class UT, class CT>
__device__ __forceinline__ void strict_visc_body(const StageArgs<UT, CT>& a, const Block& b, int e0, CT* area, int D,
                                                 int half) {
    const int wave = wave_index(), pt = threadIdx.x & 63;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int E = a.nx * a.ny * a.nz;
    const int64_t NP = (int64_t)E * 64;
    const bool valid = BLOCK || e0 + wave < E;
    const int64_t e = BLOCK ? blk_elem(a, b, wave) : (valid ? e0 + wave : E - 1);
    const CT cf = coef_load(a, (int)threadIdx.x);
    UT s0[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) s0[v] = a.uin[v * NP + e * 64 + pt];
    StrictLine<CT> w;
    if constexpr (BLOCK) {
        if (D == 0)
            strict_block_begin<0>(a, b, half, pt, w);
        else if (D == 1)
            strict_block_begin<1>(a, b, half, pt, w);
        else if (D == 2)
            strict_block_begin<2>(a, b, half, pt, w);
    } else {
        if (D == 0)
            strict_line_begin<0>(a, e0, E, pt, w);
        else if (D == 1)
            strict_line_begin<1>(a, e0, E, pt, w);
        else if (D == 2)
            strict_line_begin<2>(a, e0, E, pt, w);
    }
    {
        CT* A = area + wave * kAreaStride + swz64(pt);
#pragma unroll
        for (int v = 0; v < 5; ++v) A[v * 64] = (CT)s0[v];
    }
    coef_store<CT>((int)threadIdx.x, cf);
    __syncthreads();
    if (D < 3) {
#pragma unroll
        for (int v = 0; v < 5; ++v)
#pragma unroll
            for (int m = 0; m < 4; ++m) w.u[v][m] = area[w.pos[m] + v * 64];
    }
    __syncthreads();  // the gradients overwrite the states
    if (D == 0)
        strict_line_gradient<0, BLOCK>(a, area, w);
    else if (D == 1)
        strict_line_gradient<1, BLOCK>(a, area, w);
    else if (D == 2)
        strict_line_gradient<2, BLOCK>(a, area, w);
    __syncthreads();
    if (D == 0)
        strict_line_flux<0>(a, area, w);
    else if (D == 1)
        strict_line_flux<1>(a, area, w);
    else if (D == 2)
        strict_line_flux<2>(a, area, w);
    CT g[15], st[5], r[5];
    {
        const CT* A = area + wave * kAreaStride + swz64(pt);
#pragma unroll
        for (int q = 0; q < 15; ++q) g[q] = A[q * 64];
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) st[v] = (CT)a.uin[v * NP + e * 64 + pt];  // again (from L2), not held all along
    __syncthreads();  // the volume fluxes' lines are staged over the gradients
    CT mu = a.sutherland ? sutherland(st, a.mu_ref, a.t_ref, a.s_suth) : a.mu;
    if (a.mu_t) mu = mu + a.mu_t[e];
    volume_rhs<true>(a, st, g, mu, (const CT*)nullptr, coef_lds<CT>(), (CT(*)[64])(area + wave * kAreaStride), i, j, k, pt, r);
    if (valid) {
#pragma unroll
        for (int v = 0; v < 5; ++v) a.fv[e * kFvStride + kFvFaces + v * 64 + pt] = r[v];
    }
}

template <class UT, class CT>
__global__ __launch_bounds__(64 * kQuad) void od_visc_line_kernel(StageArgs<UT, CT> a) {
    __shared__ CT area[kQuad * kAreaStride];
    // wave -> direction (3: none), turning from work-group to work-group of an
    // XCD so that the SIMDs get equally many line waves
    const int D = (wave_index() + ((int)blockIdx.x >> 3)) & 3;
    strict_visc_body<false>(a, Block{}, kQuad * (int)blockIdx.x, area, D, 0);
}

// Waves per SIMD asked of the strict block kernels: three work-groups to a CU
// with f32 compute (78 and 70 VGPRs; held to 64 they spill), two with f64 (124
// and 128).
template <class CT>
constexpr int kMinWavesBlock = sizeof(CT) == 4 ? 6 : 4;

// The same by blocks, for boxes whose update runs on blocks: the traces across
// internal faces come from the next lane, so the update kernel need not write
// them.  As fast as by fours (24x26x22 f64 61 us both; 48^3 f32 237 against
// 234 us, VALU bound).
template <class UT, class CT>
__global__ __launch_bounds__(64 * kBlk) __attribute__((amdgpu_waves_per_eu(kMinWavesBlock<CT>))) void od_visc_lines_block_kernel(StageArgs<UT, CT> a) {
    __shared__ CT area[kBlk * kAreaStride];
    const int group = (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
    const int role = line_role(group), half = role / 3;
    strict_visc_body<true>(a, make_block<false>(a), 0, area, role < 6 ? role - 3 * half : 3, half);
}

// ---------------------------------------------------------------------------
// Strict build, one box: the update kernel on 2x2x2 blocks (wave w owns local
// element w in the point-wise phases).  Bounds: f32 memory, f64 the chain of
// the interface fluxes at 16 waves per CU.  Of an element's six faces three face
// another element of the block: their traces come from the block's LDS states,
// their flux is evaluated once for both elements (9 wave passes for 8 elements
// instead of 12), both elements' viscous fluxes are read once, and their traces
// of the new state are not written: 2309 values moved per element instead of
// 3061.  Per launch against the two-element tiles: 48^3 f32 211 -> 172 us,
// 24x26x22 f64 57.8 -> 49 us, 24x20x28 f64 state with f32 fluxes 40.9 -> 34 us.
// Every value is the expression of update_body.
// LDS: states in swz64 order; lanes go (pair, side, face point), so a half-wave
// reads the two elements of a pair, 4, 8 or 16 banks apart as in BlockViscLds.
// ---------------------------------------------------------------------------
constexpr int kStateStride = 5 * 64 + 4;  // as kAreaStride
template <class CT>
struct FaceBlockLds {
    CT sJe[kBlk][3][5][16];  // corrections j at the external faces
    CT sJi[kBlk][3][5][16];  // and at the internal ones
    CT sU[kBlk * kStateStride];
};

// Whether a face lane reads the viscous fluxes only after the interface flux:
// in f64, and beside an f64 state, they cost registers over it (24x26x22 f64:
// 14 to 70 spilled, 58 us, none and 49 us); all in f32 they fit and their
// latency is covered (48^3 172 against 181 us).
template <class UT, class CT>
constexpr bool kLateFv = sizeof(UT) == 8 || sizeof(CT) == 8;
template <class CT>
__device__ __forceinline__ const FvQuad<CT>& fv_quad(const CT* fv, int64_t e, int f, int fp) {
    return *reinterpret_cast<const FvQuad<CT>*>(fv + e * kFvStride + f * 64 + fp * 4);
}
// Element of an external face lane: lane = (pair, side, face point).
template <int D>
__device__ __forceinline__ int ext_elem(int half, int lane) {
    return blk_pair<D>(2 * half + (lane >> 5)) + (((lane >> 4) & 1) << D);
}
// The neighbour's trace at an external face (its own at a slip wall, unused).
template <int D, class UT, class CT>
__device__ __forceinline__ void ext_face_load(const StageArgs<UT, CT>& a, const Block& b, int half, int lane, CT* far) {
    const int le = ext_elem<D>(half, lane), side = (lane >> 4) & 1, fp = lane & 15;
    const int nb = blk_ext_nb(a, b, le, D);
    const int64_t src = nb < 0 ? blk_elem(a, b, le) : nb;
    const int rf = D == 0 ? 7 - side : 2 * D + 1 - side;
#pragma unroll
    for (int v = 0; v < 5; ++v) far[v] = stream_load(&a.tr_in[src * kTraceStride + rf * 80 + v * 16 + fp]);
}
// Trace of local element le at the left or right end of the line of face point fp.
template <int D, class CT>
__device__ __forceinline__ void block_trace(const CT* sU, int le, int fp, bool right, CT* t) {
    int base, stride;
    face_line(D, fp, base, stride);
    const int q = swz64(base);
    const CT* row = sU + le * kStateStride;
    const Coef4<CT> c = side_coef<CT>(right);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT x[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = row[v * 64 + (q ^ line_xor<D>(m))];
        t[v] = trace4(x, 0, 1, c.c0, c.c1, c.c2, c.c3, face_order(D));
    }
}
// External faces of direction D of half a block: flux_pass, a face point per lane.
template <int D, class UT, class CT>
__device__ __forceinline__ void ext_face(const StageArgs<UT, CT>& a, const Block& b, FaceBlockLds<CT>& L, int half,
                                         int lane, const CT* far) {
    const int le = ext_elem<D>(half, lane), side = (lane >> 4) & 1, fp = lane & 15;
    const bool right = side;
    const int e = blk_elem(a, b, le), nb = blk_ext_nb(a, b, le, D);
    const bool wall = D == 1 && nb < 0;
    FvQuad<CT> fo, fn;
    const auto load_fv = [&] {
        fo = fv_quad(a.fv, e, 2 * D + side, fp);
        fn = fv_quad(a.fv, wall ? e : nb, 2 * D + 1 - side, fp);
    };
    if constexpr (!kLateFv<UT, CT>) load_fv();
    CT own[5], Lq[5], Rq[5], fvo[5], fvn[5], fr[5], jv[5];
    block_trace<D>(L.sU, le, fp, right, own);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const CT oth = wall ? own[v] : far[v];
        Lq[v] = right ? own[v] : oth;
        Rq[v] = right ? oth : own[v];
    }
    interface_flux<D>(a.flux, Lq, Rq, fr);
    if constexpr (kLateFv<UT, CT>) {
        asm volatile("" : "+v"(fr[0]), "+v"(fr[1]), "+v"(fr[2]), "+v"(fr[3]), "+v"(fr[4])::"memory");
        load_fv();
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        fvo[v] = v ? fo.c[v - 1] : (CT)0;
        fvn[v] = v ? fn.c[v - 1] : (CT)0;
    }
    face_correction<D, true>(fr, own, fvo, fvn, wall, right, jv);
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sJe[le][D][v][fp] = jv[v];
}
// Internal faces of direction D: lane = (pair, face point), one flux, each
// side's correction as flux_pass forms it.
template <int D, class UT, class CT>
__device__ __forceinline__ void int_face(const StageArgs<UT, CT>& a, const Block& b, FaceBlockLds<CT>& L, int lane) {
    const int lL = blk_pair<D>(lane >> 4), lR = lL + (1 << D), fp = lane & 15;
    FvQuad<CT> fl, fn;
    const auto load_fv = [&] {
        fl = fv_quad(a.fv, blk_elem(a, b, lL), 2 * D + 1, fp);
        fn = fv_quad(a.fv, blk_elem(a, b, lR), 2 * D, fp);
    };
    if constexpr (!kLateFv<UT, CT>) load_fv();
    CT tl[5], tr[5], fvl[5], fvr[5], fr[5], jv[5];
    block_trace<D>(L.sU, lL, fp, true, tl);
    block_trace<D>(L.sU, lR, fp, false, tr);
    interface_flux<D>(a.flux, tl, tr, fr);
    if constexpr (kLateFv<UT, CT>) {
        asm volatile("" : "+v"(fr[0]), "+v"(fr[1]), "+v"(fr[2]), "+v"(fr[3]), "+v"(fr[4])::"memory");
        load_fv();
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        fvl[v] = v ? fl.c[v - 1] : (CT)0;
        fvr[v] = v ? fn.c[v - 1] : (CT)0;
    }
    face_correction<D, true>(fr, tl, fvl, fvr, false, true, jv);
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sJi[lL][D][v][fp] = jv[v];
    face_correction<D, true>(fr, tr, fvr, fvl, false, false, jv);
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sJi[lR][D][v][fp] = jv[v];
}

template <class UT, class CT>
__device__ __forceinline__ void face_block_body(const StageArgs<UT, CT>& a, const Block& b, FaceBlockLds<CT>& L,
                                                int role) {
    constexpr bool SAME = std::is_same<UT, CT>::value;
    const int wave = wave_index(), pt = threadIdx.x & 63;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    const int64_t e = blk_elem(a, b, wave);
    const int64_t gbase = e * 64 + pt;
    const CT cf = coef_load(a, (int)threadIdx.x);
    UT s0[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) s0[v] = a.uin[v * NP + gbase];
    CT far[5];
    switch (role) {
        case 0: ext_face_load<0>(a, b, 0, pt, far); break;
        case 1: ext_face_load<0>(a, b, 1, pt, far); break;
        case 2: ext_face_load<1>(a, b, 0, pt, far); break;
        case 3: ext_face_load<1>(a, b, 1, pt, far); break;
        case 4: ext_face_load<2>(a, b, 0, pt, far); break;
        case 5: ext_face_load<2>(a, b, 1, pt, far); break;
        default: break;
    }
    CT* own = L.sU + wave * kStateStride + swz64(pt);
#pragma unroll
    for (int v = 0; v < 5; ++v) own[v * 64] = (CT)s0[v];
    coef_store<CT>((int)threadIdx.x, cf);
    __syncthreads();
    // 6 external passes (4 elements x 16 points) and 3 internal ones (4 pairs x
    // 16 points), 9 over 8 waves
    switch (role) {
        case 0:
            ext_face<0>(a, b, L, 0, pt, far);
            int_face<2>(a, b, L, pt);
            break;
        case 1: ext_face<0>(a, b, L, 1, pt, far); break;
        case 2: ext_face<1>(a, b, L, 0, pt, far); break;
        case 3: ext_face<1>(a, b, L, 1, pt, far); break;
        case 4: ext_face<2>(a, b, L, 0, pt, far); break;
        case 5: ext_face<2>(a, b, L, 1, pt, far); break;
        case 6: int_face<0>(a, b, L, pt); break;
        default: int_face<1>(a, b, L, pt); break;
    }
    // the volume RHS and u^n (stage 1: the state), before the barrier's wait
    UT uprv[5], ucr[5];
    CT r[5], rts[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        ucr[v] = SAME ? (UT)own[v * 64] : a.uin[v * NP + gbase];
        r[v] = stream_load(&a.fv[e * kFvStride + kFvFaces + v * 64 + pt]);
    }
    if (a.stage1) {
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = ucr[v];
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = stream_load(&a.uprev[v * NP + gbase]);
    }
    const StageDt<UT, CT> cdt = stage_dt(a);
    __syncthreads();

    const CoefTable<CT>& o = coef_lds<CT>();
    const CT gLi = o.g[i][0], gRi = o.g[i][1];
    const CT gLj = o.g[j][0], gRj = o.g[j][1];
    const CT gLk = o.g[k][0], gRk = o.g[k][1];
    const int fpx = j + 4 * k, fpy = i + 4 * k, fpz = i + 4 * j;
    const CT* Je = &L.sJe[wave][0][0][0];
    const CT* Ji = &L.sJi[wave][0][0][0];
    const int lx = wave & 1, ly = (wave >> 1) & 1, lz = wave >> 2;
    const CT *Jx0 = lx ? Ji : Je, *Jx1 = lx ? Je : Ji;
    const CT *Jy0 = (ly ? Ji : Je) + 80, *Jy1 = (ly ? Je : Ji) + 80;
    const CT *Jz0 = (lz ? Ji : Je) + 160, *Jz1 = (lz ? Je : Ji) + 160;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        CT cx = -(Jx0[v * 16 + fpx] * gLi * a.jx) - (Jx1[v * 16 + fpx] * gRi * a.jx);
        CT cy = -(Jy0[v * 16 + fpy] * gLj * a.jy) - (Jy1[v * 16 + fpy] * gRj * a.jy);
        CT cz = -(Jz0[v * 16 + fpz] * gLk * a.jz) - (Jz1[v * 16 + fpz] * gRk * a.jz);
        rts[v] = r[v] + (cx + cy + cz);
    }
    if (a.mode == 1) {  // the stage's RHS into dbg, state unchanged
#pragma unroll
        for (int v = 0; v < 5; ++v) a.dbg[v * NP + gbase] = rts[v];
        return;
    }
    UT unew[5];
    rk_stage(a, cdt, uprv, ucr, rts, unew);
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        stream_store(unew[v], &a.uout[v * NP + gbase]);
        own[v * 64] = (CT)unew[v];
    }
    wave_sync();

    // Traces of the new state on the element's external faces (x in both
    // orders), 16 lanes each; only they are read (the internal ones come from
    // the blocks' LDS tiles).
    const int g = pt >> 4, fp = pt & 15, d = g == 3 ? 0 : g;
    const int tf = 2 * g + blk_bit(wave, d);
    int base, stride;
    face_line(d, fp, base, stride);
    const int q = swz64(base);
    const int x1 = d == 0 ? line_xor<0>(1) : (d == 1 ? line_xor<1>(1) : line_xor<2>(1));
    const int x2 = d == 0 ? line_xor<0>(2) : (d == 1 ? line_xor<1>(2) : line_xor<2>(2));
    const Coef4<CT> c = side_coef<CT>(tf & 1);
    const int order = trace_face_order(tf);
    CT* dst = a.tr_out + e * kTraceStride + tf * 80 + fp;
    const CT* row = L.sU + wave * kStateStride;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const CT x[4] = {row[v * 64 + q], row[v * 64 + (q ^ x1)], row[v * 64 + (q ^ x2)], row[v * 64 + (q ^ x1 ^ x2)]};
        stream_store(trace4(x, 0, 1, c.c0, c.c1, c.c2, c.c3, order), &dst[v * 16]);
    }
}

template <class UT, class CT>
__global__ __launch_bounds__(64 * kBlk) __attribute__((amdgpu_waves_per_eu(kMinWavesBlock<CT>))) void od_update_face_block_kernel(StageArgs<UT, CT> a) {
    __shared__ FaceBlockLds<CT> L;
    const int group = (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
    face_block_body(a, make_block<true>(a), L, (wave_index() + (group >> 3)) & 7);
}
#endif

#if OD_FAST
// ---------------------------------------------------------------------------
// Fast f32 build: the update kernel on blocks of 2x2x2 elements (512 threads; wave w owns local element w = lx + 2 ly +
// 4 lz in the point-wise phases).  Three of an element's six faces face
// another element of the block.  Their neighbour traces come from the
// block's LDS state tiles instead of HBM, and the interface flux of such an
// internal face is evaluated once for both of its elements.  Every value is
// formed from the same operands in the same order as in update_body, so each
// element gets the same bits as in the two-element-tile kernels (which take the
// last layers of boxes with an odd dimension, and boxes 1 element wide).
// ---------------------------------------------------------------------------
// Source of 16-byte chunk `chunk` (0..59) of the external-face traces of
// local element le, as the LDS prefetch lays them out ([d][5][16]): the
// neighbour's facing trace (its own at a slip wall, where it is not used).
// le is wave-uniform, so the three neighbours are scalar work and each lane
// only selects its direction's.
template <class UT, class CT>
__device__ __forceinline__ const UT* blk_ext_trace_src(const StageArgs<UT, CT>& a, const Block& b, int le,
                                                       int chunk) {
    const int nb0 = blk_ext_nb(a, b, le, 0), nb1 = blk_ext_nb(a, b, le, 1), nb2 = blk_ext_nb(a, b, le, 2);
    const int d = chunk >= 40 ? 2 : (chunk >= 20 ? 1 : 0), c = chunk - 20 * d;
    const int nb = d == 0 ? nb0 : (d == 1 ? nb1 : nb2);
    const int src_e = nb >= 0 ? nb : blk_elem(a, b, le);
    const int f = 2 * d + blk_bit(le, d);
    return a.tr_in + (int64_t)src_e * kTraceStride + (f ^ 1) * 80 + c * 4;
}

// Traces of the element's three external faces (face 2d + bit d of le, one
// face point per lane, lanes 48..63 idle), as write_traces_own forms them.
__device__ __forceinline__ void blk_write_ext_traces(const float (*sUe)[64], float* dst, int le, int lane) {
    const int d = lane >> 4, fp = lane & 15;
    if (d > 2) return;
    const int f = 2 * d + blk_bit(le, d);
    int base, stride;
    face_line(d, fp, base, stride);
    const Coef4<float> c = side_coef<float>(f & 1);
#pragma unroll
    for (int v = 0; v < 5; ++v)
        stream_store(trace4(sUe[v], base, stride, c.c0, c.c1, c.c2, c.c3, trace_face_order(f)),
                     &dst[f * 80 + v * 16 + fp]);
}

// State tiles of a block's elements, one every 5 * 64 + 16 floats: the pad
// puts consecutive elements' tiles 16 banks apart, so the two elements whose
// face points one half-wave reads in a face pass do not share banks.
struct BlockTiles {
    float t[kBlk][5 * 64 + 16];
    __device__ float (*operator[](int le))[64] { return reinterpret_cast<float(*)[64]>(t[le]); }
};

// LDS of a block.  sJe[le][d]: the external face of direction d of element
// le -- first the neighbour's facing trace (LDS-DMA, chunk id = 4 x its
// float offset), then the element's correction j there; sJi[le][d]: j at
// the internal face of direction d.
struct BlockUpdateLds {
    alignas(16) float sJe[kBlk][3][5][16];
    float sJi[kBlk][3][5][16];
    BlockTiles sU;
    float sF[kBlk][5][64];  // volume-flux line staging, then the volume RHS
};

// External faces of direction D of the four elements 4h .. 4h+3: one face
// point per lane.  The arithmetic is flux_pass's.
template <int D, bool VISC>
__device__ __forceinline__ void blk_ext_pass(const StageArgs<float, float>& a, const Block& b, BlockUpdateLds& L,
                                             int h, int lane) {
    const int le = 4 * h + (lane >> 4), fp = lane & 15;
    const int side = blk_bit(le, D);
    const bool right = side;
    int base, stride;
    face_line(D, fp, base, stride);
    const Coef4<float> c = side_coef<float>(side);
    float own[5], oth[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) own[v] = trace4(L.sU[le][v], base, stride, c.c0, c.c1, c.c2, c.c3, face_order(D));
    const int nb = blk_ext_nb(a, b, le, D);
    const bool wall = D == 1 && nb < 0;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const float far = L.sJe[le][D][v][fp];
        oth[v] = wall ? own[v] : far;
    }
    float fvo[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, fvn[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    if (VISC) {
        const int f = 2 * D + side;
        const FvQuad<float> o =
            *reinterpret_cast<const FvQuad<float>*>(a.fv + (int64_t)blk_elem(a, b, le) * kFvStride + f * 64 + fp * 4);
        FvQuad<float> n = o;
        if (!wall) n = *reinterpret_cast<const FvQuad<float>*>(a.fv + (int64_t)nb * kFvStride + (f ^ 1) * 64 + fp * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fvo[1 + q] = o.c[q];
            fvn[1 + q] = n.c[q];
        }
    }
    float Lq[5], Rq[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        Lq[v] = right ? own[v] : oth[v];
        Rq[v] = right ? oth[v] : own[v];
    }
    float fr[5], jv[5];
    interface_flux<D>(a.flux, Lq, Rq, fr);
    face_correction<D, VISC>(fr, own, fvo, fvn, wall, right, jv);
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sJe[le][D][v][fp] = jv[v];
}

// Internal faces of direction D: pair p = lane / 16 (left element lL, right
// element lL + 2^D), one face point per lane; one interface flux for both
// sides, each side's correction as flux_pass forms it.
template <int D, bool VISC>
__device__ __forceinline__ void blk_int_pass(const StageArgs<float, float>& a, const Block& b, BlockUpdateLds& L,
                                             int lane) {
    const int p = lane >> 4, fp = lane & 15;
    const int lL = blk_pair<D>(p);
    const int lR = lL + (1 << D);
    int base, stride;
    face_line(D, fp, base, stride);
    const Coef4<float> cr = side_coef<float>(true), cl = side_coef<float>(false);
    float tl[5], tr[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) tl[v] = trace4(L.sU[lL][v], base, stride, cr.c0, cr.c1, cr.c2, cr.c3, face_order(D));
#pragma unroll
    for (int v = 0; v < 5; ++v) tr[v] = trace4(L.sU[lR][v], base, stride, cl.c0, cl.c1, cl.c2, cl.c3, face_order(D));
    float fr[5], jl[5], jr[5];
    interface_flux<D>(a.flux, tl, tr, fr);
    if constexpr (VISC) {
        // the half-difference the block visc kernel stored in the left
        // element's slot of the face; component 0 as the tile kernels form it
        const FvQuad<float> q = *reinterpret_cast<const FvQuad<float>*>(
            a.fv + (int64_t)blk_elem(a, b, lL) * kFvStride + (2 * D + 1) * 64 + fp * 4);
        const float hd[5] = {0.5f * (0.f - 0.f), q.c[0], q.c[1], q.c[2], q.c[3]};
        face_correction_hd<D>(fr, tl, hd, true, jl);
        face_correction_hd<D>(fr, tr, hd, false, jr);
    } else {
        const float zero[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        face_correction<D, VISC>(fr, tl, zero, zero, false, true, jl);
        face_correction<D, VISC>(fr, tr, zero, zero, false, false, jr);
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        L.sJi[lL][D][v][fp] = jl[v];
        L.sJi[lR][D][v][fp] = jr[v];
    }
}

// The new state's traces are written on the external faces only (the block visc
// kernel forms the internal ones from its LDS state tiles).
template <bool VISC>
__device__ __forceinline__ void update_block_body(const StageArgs<float, float>& a, const Block& b,
                                                  BlockUpdateLds& L) {
    const int wave = wave_index(), pt = threadIdx.x & 63;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    const int64_t e = blk_elem(a, b, wave);
    const int64_t gbase = e * 64 + pt;
    const float cf = coef_load(a, (int)threadIdx.x);
    // the element's three external neighbour traces (60 16-byte LDS-DMA
    // chunks) and its state, both read for the last time in this stage:
    // streaming, like the update kernel's stores
    if (pt < 60) {
        const float* src = blk_ext_trace_src(a, b, wave, pt);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)&L.sJe[wave][0][0][0], 16, 0,
                                         kDmaStream);
    }
    load_state_tile<float, float, kDmaStream>(a.uin, NP, e, L.sU[wave], pt);
    coef_store<float>((int)threadIdx.x, cf);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's LDS copies have landed
    __syncthreads();

    const CoefTable<float>& o = coef_lds<float>();
    // Volume RHS of the wave's element (update_body's fast f32 path).
    float st[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) st[v] = L.sU[wave][v][pt];
    float vdiv[4] = {0.f, 0.f, 0.f, 0.f};
    if (VISC) {
        const FvQuad<float> src = *reinterpret_cast<const FvQuad<float>*>(a.fv + e * kFvStride + kFvFaces + pt * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) vdiv[q] = src.c[q];
    }
    float rs[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        float F[5];
        euler_flux(d, st, F);
        if (d == 0) {
            const float* Dx = o.D[0][i];
#pragma unroll
            for (int v = 0; v < 5; ++v) rs[v] = quad_line(Dx, F[v]);
            continue;
        }
        if (d > 1) wave_sync();  // the y lines have been read
#pragma unroll
        for (int v = 0; v < 5; ++v) L.sF[wave][v][pt] = F[v];
        wave_sync();
        const int idx = d == 1 ? j : k;
        const int base = d == 1 ? i + 16 * k : i + 4 * j;
        const int stride = d == 1 ? 4 : 16;
        const float* Dd = o.D[d][idx];
#pragma unroll
        for (int v = 0; v < 5; ++v)
#pragma unroll
            for (int m = 0; m < 4; ++m) rs[v] = __builtin_fmaf(Dd[m], L.sF[wave][v][base + m * stride], rs[v]);
    }
    wave_sync();
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        float val = -rs[v];
        if (VISC && v > 0) val += vdiv[v - 1];
        if (v == 1) val += a.bf;
        L.sF[wave][v][pt] = val;
    }

    // Interface fluxes: 6 external passes (4 elements x 16 points each) and
    // 3 internal ones (4 pairs x 16 points), 9 wave passes over 8 waves.
    switch (wave) {
        case 0: blk_ext_pass<0, VISC>(a, b, L, 0, pt); blk_int_pass<2, VISC>(a, b, L, pt); break;
        case 1: blk_ext_pass<0, VISC>(a, b, L, 1, pt); break;
        case 2: blk_ext_pass<1, VISC>(a, b, L, 0, pt); break;
        case 3: blk_ext_pass<1, VISC>(a, b, L, 1, pt); break;
        case 4: blk_ext_pass<2, VISC>(a, b, L, 0, pt); break;
        case 5: blk_ext_pass<2, VISC>(a, b, L, 1, pt); break;
        case 6: blk_int_pass<0, VISC>(a, b, L, pt); break;
        default: blk_int_pass<1, VISC>(a, b, L, pt); break;
    }
    __syncthreads();

    // FR correction and stage update of the wave's element (rk.cu:12-25,
    // 63-82; update_body's fast f32 path).
    const StageDt<float, float> cdt = stage_dt(a);
    const float gLi = o.g[0][i][0], gRi = o.g[0][i][1];
    const float gLj = o.g[1][j][0], gRj = o.g[1][j][1];
    const float gLk = o.g[2][k][0], gRk = o.g[2][k][1];
    const int fpx = j + 4 * k, fpy = i + 4 * k, fpz = i + 4 * j;
    const int lx = wave & 1, ly = (wave >> 1) & 1, lz = wave >> 2;
    const float* Jext = &L.sJe[wave][0][0][0];
    const float* Jint = &L.sJi[wave][0][0][0];
    const float* Jx0 = (lx == 0 ? Jext : Jint);
    const float* Jx1 = (lx == 1 ? Jext : Jint);
    const float* Jy0 = (ly == 0 ? Jext : Jint) + 80;
    const float* Jy1 = (ly == 1 ? Jext : Jint) + 80;
    const float* Jz0 = (lz == 0 ? Jext : Jint) + 160;
    const float* Jz1 = (lz == 1 ? Jext : Jint) + 160;
    float uprv[5], ucr[5], r[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        ucr[v] = L.sU[wave][v][pt];
        r[v] = L.sF[wave][v][pt];
    }
    if (a.stage1) {
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = ucr[v];
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) uprv[v] = stream_load(&a.uprev[v * NP + gbase]);
    }
    float rt[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        float cx = -(Jx0[v * 16 + fpx] * gLi + Jx1[v * 16 + fpx] * gRi);
        float cy = -(Jy0[v * 16 + fpy] * gLj + Jy1[v * 16 + fpy] * gRj);
        float cz = -(Jz0[v * 16 + fpz] * gLk + Jz1[v * 16 + fpz] * gRk);
        rt[v] = r[v] + (cx + cy + cz);
    }
    if (a.mode == 1) {  // the stage's RHS into dbg, state unchanged
#pragma unroll
        for (int v = 0; v < 5; ++v) a.dbg[v * NP + gbase] = rt[v];
        return;
    }
    // the blend in the compute or the state type: both float here, so the
    // two differ only in their coefficients, chosen once (scalar selects)
    const float kA = a.accum_state ? a.ua : a.ca;
    const float kB = a.accum_state ? a.ub : a.cb;
    const float kC = a.accum_state ? cdt.uc : cdt.cc;
    float unew[5];
    if (a.stage1) {  // uniform branch: each form computes only its own blend
#pragma unroll
        for (int v = 0; v < 5; ++v) unew[v] = rk_blend1(kA, kC, uprv[v], rt[v]);
    } else {
#pragma unroll
        for (int v = 0; v < 5; ++v) unew[v] = rk_blend(kA, kB, kC, uprv[v], ucr[v], rt[v]);
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) stream_store(unew[v], &a.uout[v * NP + gbase]);

    // Face traces of the new state.
#pragma unroll
    for (int v = 0; v < 5; ++v) L.sU[wave][v][pt] = unew[v];
    wave_sync();
    blk_write_ext_traces(L.sU[wave], a.tr_out + e * kTraceStride, wave, pt);
}

// ---------------------------------------------------------------------------
// The visc kernel on the same 2x2x2 blocks, by lines.  A lane of a line wave
// owns one line of four points along direction D of one element (8 elements x
// 16 lines x 3 directions = 6 full waves; lane = [pair of elements][line][side]
// with side = the element's coordinate along D): it reads the line's states
// once, forms both end traces, both BR1 jumps and the corrected derivative at
// its four points, and later, from the gradients of the line, the viscous
// fluxes at both ends.  The neighbour across the block's internal face is the
// neighbouring lane (DPP); the external trace comes straight from memory.  The
// operators are wave-uniform here (scalar registers).  Point-wise work (volume
// fluxes and their divergence) stays a wave per element.
//
// The point-wise form of all this (a lane per solution point for the gradient,
// a lane per face point for jumps and fluxes) read each state 12 times and each
// gradient 6 to 8 times from LDS and formed the state's face traces twice: its
// VALU instructions (753 per element's wave) took 78 % of the kernel's time and
// its LDS reads about as much, at 6 waves to a SIMD.  By lines it is 8 waves
// (64 VGPRs, 31 KB per work-group) and at 48^3 132 us a launch instead of 195
// (0.51 GB moved, 82 us at the update kernel's 6.2 TB/s; 126 us with the even
// and odd parts, see line_even).
// Every value is the same expression as in visc_body.
//
// LDS: one area per element, first its state [5][64], then, once every line has
// been read, its gradient [15][64], both in swz64 order, under which the 16
// lines of an element fall in distinct banks; areas lie 4 floats further apart
// than their size, so that the partner along x, y, z is 4, 8, 16 banks away,
// the bit that swz64 keeps fixed over a face of that direction.
// ---------------------------------------------------------------------------
template <bool WIDE>
struct BlockViscLds {
    alignas(16) float area[kBlk * kAreaStride];
    float own_stage[WIDE ? kBlk : 0][4 * 64];  // staging of the volume fluxes' lines: over the gradients, or its own
    __device__ float* of(int le) { return area + le * kAreaStride; }
    __device__ float* stage(int le) { return WIDE ? own_stage[le] : of(le); }
};

// End trace sum_m q[m] l_m(+-1) in the BR1 order (the right end's coefficients
// are the left one's backwards).
__device__ __forceinline__ float line_trace(const float* q, const float* c) {
    return __builtin_fmaf(q[1], c[1], q[0] * c[0]) + __builtin_fmaf(q[3], c[3], q[2] * c[2]);
}

// One line wave's state through the kernel's phases.
struct LineWave {
    int le, side, fp;       // element, its coordinate along D, face point of the line
    float u[5][4];          // the line's states
    float tl[5], tr[5];     // their traces at the left and right end
    float ext[5];           // the neighbour's trace across the external face
    int pos[4];             // positions of the four points in the element's area
};

template <int D>
__device__ __forceinline__ void line_begin(const StageArgs<float, float>& a, const Block& b, int half, int lane,
                                           LineWave& w) {
    w.side = lane & 1;
    w.fp = (lane >> 1) & 15;
    const int p = 2 * half + (lane >> 5);  // pair of elements along D
    w.le = blk_pair<D>(p) + (w.side << D);
    const int nb = blk_ext_nb(a, b, w.le, D);
    const int src = nb >= 0 ? nb : blk_elem(a, b, w.le);  // at a slip wall its own, unused
    const float* t = a.tr_in + (int64_t)src * kTraceStride + (2 * D + 1 - w.side) * 80 + w.fp;
#pragma unroll
    for (int v = 0; v < 5; ++v) w.ext[v] = t[v * 16];
    int base, stride;
    face_line(D, w.fp, base, stride);
    const int s0 = swz64(base);
#pragma unroll
    for (int m = 0; m < 4; ++m) w.pos[m] = w.le * kAreaStride + (s0 ^ line_xor<D>(m));
}

// Jumps and corrected derivative along D (br1_jumps, lane_gradient_faces) ->
// the gradient's rows 3 v + D.
template <int D>
__device__ __forceinline__ void line_gradient(const StageArgs<float, float>& a, const Block& b, float* area,
                                              LineWave& w) {
    const Ops<float>& o = dev_ops<float>();
    const bool wall = D == 1 && blk_ext_nb(a, b, w.le, D) < 0;
    const EvenOdd c[2] = {even_odd(a.ops, D, 0), even_odd(a.ops, D, 1)};
#pragma unroll
    for (int v = 0; v < 5; ++v) {
        const float* u = w.u[v];
        const float tl = line_trace(u, o.eL), tr = line_trace(u, o.eR);
        const float in = lane_partner(w.side ? tl : tr);
        const float own = w.side ? tr : tl;
        const float ext = wall ? ((v > 0 && v < 4) ? -own : own) : w.ext[v];
        const float wl = (w.side ? in : ext) - tl, wr = (w.side ? ext : in) - tr;
        const float t = (u[0] + u[3]) - (u[1] + u[2]), d0 = u[0] - u[3], d1 = u[1] - u[2];
        const float p = wl - wr, q = wl + wr;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float ev = line_even(c[i], t, q), od = line_odd(c[i], d0, d1, p);
            area[w.pos[i] + (3 * v + D) * 64] = od + ev;
            area[w.pos[3 - i] + (3 * v + D) * 64] = od - ev;
        }
        w.tl[v] = tl;
        w.tr[v] = tr;
        asm volatile("" : "+v"(w.tl[v]), "+v"(w.tr[v])::"memory");  // variable by variable (see lane_gradient_faces)
    }
}

// Viscous fluxes at both ends of the line (fv_value).  The external end's goes
// to the element's slot of that face; of the pair's internal face the left
// element stores the half-difference (F_vL - F_vR) / 2, all the update kernel
// reads there.
template <int D>
__device__ __forceinline__ void line_flux(const StageArgs<float, float>& a, const Block& b, const float* area,
                                          const LineWave& w) {
    const Ops<float>& o = dev_ops<float>();
    float gl[15], gr[15];
#pragma unroll
    for (int q = 0; q < 15; ++q) {
        // what the flux along D reads: the density's gradient, the momenta's
        // along D, across D of momentum D and on the diagonal, the energy's along D
        const int v = q / 3, c = q % 3;
        const bool used = v == 0 || c == D || (v < 4 && (v - 1 == D || v - 1 == c));
        if (!used) {
            gl[q] = gr[q] = 0.f;
            continue;
        }
        float x[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) x[m] = area[w.pos[m] + q * 64];
        gl[q] = __builtin_fmaf(x[3], o.eL[3], __builtin_fmaf(x[2], o.eL[2], __builtin_fmaf(x[1], o.eL[1], x[0] * o.eL[0])));
        gr[q] = __builtin_fmaf(x[3], o.eR[3], __builtin_fmaf(x[2], o.eR[2], __builtin_fmaf(x[1], o.eR[1], x[0] * o.eR[0])));
        asm volatile("" : "+v"(gl[q]), "+v"(gr[q])::"memory");
    }
    const int64_t e = blk_elem(a, b, w.le);
    float fl[4], fr[4];
    fast_visc_flux(D, fast_visc(a, w.tl, gl, e), fl);
    asm volatile("" : "+v"(fl[0]), "+v"(fl[1]), "+v"(fl[2]), "+v"(fl[3])::"memory");  // one end, then the other
    fast_visc_flux(D, fast_visc(a, w.tr, gr, e), fr);
    FvQuad<float> ext, h;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        ext.c[c] = w.side ? fr[c] : fl[c];
        const float other = lane_partner(w.side ? fl[c] : fr[c]);
        h.c[c] = 0.5f * (fr[c] - other);  // left element
    }
    FvQuad<float>* dst = reinterpret_cast<FvQuad<float>*>(a.fv + e * kFvStride + 2 * D * 64 + w.fp * 4);
    dst[w.side ? 16 : 0] = ext;
    if (!w.side) dst[16] = h;
}

// role: 0..5 the line waves (direction role % 3, half of the pairs role / 3),
// 6 and 7 none.
template <bool WIDE = false>
__device__ __forceinline__ void visc_block_body(const StageArgs<float, float>& a, const Block& b,
                                                BlockViscLds<WIDE>& L, int role) {
    const int wave = wave_index(), pt = threadIdx.x & 63;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int64_t NP = (int64_t)a.nx * a.ny * a.nz * 64;
    const bool owner = !WIDE || wave < kBlk;
    const int64_t e = blk_elem(a, b, wave & (kBlk - 1));
    const int half = role / 3, D = role < 6 ? role - 3 * half : 3;
    const float cf = coef_load(a, (int)threadIdx.x);
    float s0[5];
    if (owner) {
#pragma unroll
        for (int v = 0; v < 5; ++v) s0[v] = a.uin[v * NP + e * 64 + pt];
    }
    LineWave w;
    if (D == 0)
        line_begin<0>(a, b, half, pt, w);
    else if (D == 1)
        line_begin<1>(a, b, half, pt, w);
    else if (D == 2)
        line_begin<2>(a, b, half, pt, w);
    if (owner) {
        float* A = L.of(wave) + swz64(pt);
#pragma unroll
        for (int v = 0; v < 5; ++v) A[v * 64] = s0[v];
    }
    coef_store<float>((int)threadIdx.x, cf);
    __syncthreads();
    if (D < 3) {
#pragma unroll
        for (int v = 0; v < 5; ++v)
#pragma unroll
            for (int m = 0; m < 4; ++m) w.u[v][m] = L.area[w.pos[m] + v * 64];
    }
    __syncthreads();  // the gradients overwrite the states
    if (D == 0)
        line_gradient<0>(a, b, L.area, w);
    else if (D == 1)
        line_gradient<1>(a, b, L.area, w);
    else if (D == 2)
        line_gradient<2>(a, b, L.area, w);
    __syncthreads();
    if (D == 0)
        line_flux<0>(a, b, L.area, w);
    else if (D == 1)
        line_flux<1>(a, b, L.area, w);
    else if (D == 2)
        line_flux<2>(a, b, L.area, w);
    if (!owner) return;
    float g[15];
    {
        const float* A = L.of(wave) + swz64(pt);
#pragma unroll
        for (int q = 0; q < 15; ++q) g[q] = A[q * 64];
    }
    float st[5];  // the point's state again (from L2), not held through the line phases
#pragma unroll
    for (int v = 0; v < 5; ++v) st[v] = a.uin[v * NP + e * 64 + pt];
    if constexpr (!WIDE) __syncthreads();  // the volume fluxes' lines are staged over the gradients
    visc_divergence(a, e, st, g, coef_lds<float>(), L.stage(wave), i, j, k, pt);
}

// One box: the update kernel walks the blocks backwards, the visc kernel
// forwards (make_block).
template <bool VISC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(8))) void od_update_block_kernel(
    StageArgs<float, float> a) {
    __shared__ BlockUpdateLds L;
    update_block_body<VISC>(a, make_block<true>(a), L);
}
// WIDE, for small boxes, whose kernels last as long as one work-group: the six
// line waves are waves of their own beside the eight of the elements, so that
// the fluxes at the lines' ends and the divergence at the points, which both need
// the gradients, run at once.
constexpr int kWideBlockWaves = kBlk + 6;
template <bool WIDE>
__global__ __launch_bounds__((64 * (WIDE ? kWideBlockWaves : kBlk))) __attribute__((amdgpu_waves_per_eu(WIDE ? 7 : 8))) void od_visc_block_kernel(
    StageArgs<float, float> a) {
    __shared__ BlockViscLds<WIDE> L;
    const int group = (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
    const int role = WIDE ? (wave_index() < kBlk ? 6 : wave_index() - kBlk) : line_role(group);
    visc_block_body<WIDE>(a, make_block<false>(a), L, role);
}
#endif

// ---------------------------------------------------------------------------
// Ensembles: the tiles of every box of a batch in one launch per phase.  A
// work unit is `PAIRS` consecutive tiles (one 128-thread tile each); work-
// groups walk the units in a fixed order, so every unit is done exactly once
// and the result of each element does not depend on the schedule.
// ---------------------------------------------------------------------------

// Unit handled by this work-group at iteration `it`, or -1 when it is done.
// order 0: round robin over all units.  order 1: work-groups are dispatched
// round robin over the 8 XCDs, so XCD x = blockIdx.x % 8 takes the x-th
// contiguous eighth of the units (its neighbours' traces stay in its L2).
__device__ __forceinline__ int sched_unit(int order, int n_units, int it) {
    if (order == 0) {
        const int u = (int)blockIdx.x + it * (int)gridDim.x;
        return u < n_units ? u : -1;
    }
    const int m = (int)gridDim.x >> 3, x = (int)blockIdx.x & 7, s = (int)blockIdx.x >> 3;
    const int chunk = (n_units + 7) >> 3;
    const int r0 = x * chunk, r1 = min(n_units, r0 + chunk);
    const int u = r0 + s + it * m;
    return u < r1 ? u : -1;
}

// Wave-uniform copies (SGPRs) of values loaded from the box table: the
// loads sit after stores of earlier units, so the compiler cannot use
// scalar loads by itself.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uni(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
__device__ __forceinline__ int64_t uni(int64_t x) {
    const uint64_t u = (uint64_t)x;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double uni(double x) { return __longlong_as_double(uni((int64_t)__double_as_longlong(x))); }
__device__ __forceinline__ Elem uni(const Elem& e) {
    return Elem{uni(e.xl), uni(e.xr), uni(e.yl), uni(e.yr), uni(e.zl), uni(e.zr)};
}

// Stage arguments of one box of a batch: the batch's arguments with the
// box's dimensions, Jacobians, stage coefficients and buffer offsets.
template <class UT, class CT>
__device__ __forceinline__ void batch_box_args(const StageArgs<UT, CT>& a, const BoxDev<UT, CT>* boxes, int box, int stage,
                                               StageArgs<UT, CT>& ab) {
    const BoxDev<UT, CT>& bx = boxes[box];
    ab = a;
    ab.ops = a.ops + box;
    ab.nx = uni(bx.nx);
    ab.ny = uni(bx.ny);
    ab.nz = uni(bx.nz);
    ab.jx = uni(bx.jx);
    ab.jy = uni(bx.jy);
    ab.jz = uni(bx.jz);
    ab.cc = uni(bx.cc[stage]);
    ab.uc = uni(bx.uc[stage]);
    const int64_t e_off = uni(bx.e_off);
    const int64_t so = e_off * 320;  // box state [5][E_box][64] starts at 5 * 64 * e_off
    ab.uin = a.uin + so;
    ab.uprev = a.uprev + so;
    ab.uout = a.uout + so;
    ab.dbg = a.dbg ? a.dbg + so : a.dbg;
    ab.tr_in = a.tr_in + e_off * kTraceStride;
    ab.tr_out = a.tr_out + e_off * kTraceStride;
    ab.fv = a.fv ? a.fv + e_off * kFvStride : a.fv;
    ab.mu_t = a.mu_t ? a.mu_t + e_off : a.mu_t;
}

// Tile lt of the shell of a box whose core runs on 2x2x2 blocks: the
// elements with x = nx - 1 (odd nx), then y = ny - 1 (odd ny), then z = nz - 1
// (odd nz), each element in the first of these slabs it lies in.  The x slab
// pairs its elements along y, the others along x.  A tile's elements and
// neighbours come from make_tile_at as for any tile, so each face is formed
// as in a box run on tiles alone.
template <class UT, class CT>
__device__ __forceinline__ Tile shell_tile(const StageArgs<UT, CT>& a, int lt) {
    const int hx = a.nx >> 1, hy = (a.ny + 1) >> 1;
    const int nA = (a.nx & 1) ? hy * a.nz : 0;
    const int nB = (a.ny & 1) ? hx * a.nz : 0;
    if (lt < nA) return make_tile_at(a, 1, a.nx - 1, lt % hy, lt / hy);
    lt -= nA;
    if (lt < nB) return make_tile_at(a, 0, lt % hx, a.ny - 1, lt / hx);
    lt -= nB;
    return make_tile_at(a, 0, lt % hx, lt / hx, a.nz - 1);
}

// Stage arguments and tile of batch tile t (t >= n_tiles: an empty tile).
template <class UT, class CT>
__device__ __forceinline__ void batch_tile(const StageArgs<UT, CT>& a, const BatchArgs<UT, CT>& b, int t,
                                           StageArgs<UT, CT>& ab, Tile& tl) {
    const bool ok = t < b.n_tiles;
    const int tt = ok ? t : 0;
    int lo = 0, hi = b.n_boxes - 1;
    if (b.n_boxes <= kInlineBoxes) {  // kernel-argument copy: scalar loads, no memory latency chain
        while (lo < hi) {  // last box whose first tile is <= tt
            const int mid = (lo + hi + 1) >> 1;
            if (b.tile_off[mid] <= tt)
                lo = mid;
            else
                hi = mid - 1;
        }
    } else {
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (uni(b.boxes[mid].tile_off) <= tt)
                lo = mid;
            else
                hi = mid - 1;
        }
    }
    const BoxDev<UT, CT>& bx = b.boxes[lo];
    batch_box_args(a, b.boxes, uni(lo), b.stage, ab);
    const int tile_off = uni(bx.tile_off);
    const int lt = tt - tile_off;
    if (uni(bx.shell)) {
        tl = shell_tile(ab, lt);
    } else {
        const int d0 = b.orient == 0 ? (ab.nx + kEpb - 1) / kEpb : ab.nx;
        const int d1 = b.orient == 1 ? (ab.ny + kEpb - 1) / kEpb : ab.ny;
        const int t0 = uni(lt % d0), r = uni(lt / d0);
        tl = make_tile_at(ab, b.orient, t0, uni(r % d1), uni(r / d1));
    }
    tl.e0 = uni(tl.e0);
    tl.e1 = uni(tl.e1);
    tl.el0 = uni(tl.el0);
    tl.el1 = uni(tl.el1);
    tl.walls = uni(tl.walls);
    tl.v0 = ok;
    tl.v1 = ok && tl.v1;
}

#if OD_FAST
// Block lb of a box's core, x fastest.
__device__ __forceinline__ Block core_block(const StageArgs<float, float>& a, int lb) {
    Block b;
    const int gx = a.nx >> 1, gy = a.ny >> 1;
    b.ex0 = 2 * (lb % gx);
    b.ey0 = 2 * ((lb / gx) % gy);
    b.ez0 = 2 * (lb / (gx * gy));
    b.e0 = b.ex0 + a.nx * (b.ey0 + a.ny * b.ez0);
    return b;
}
// Ensembles on 2x2x2-element blocks: the core of every box (the box less the
// last layer along each odd dimension; the whole box when all are even) runs
// the block kernels, one launch per phase for all boxes, and the shell the
// tile kernels (shell_tile).  The blocks' neighbour map (blk_ext_nb) needs
// no change: a core block's right neighbour is the next element unless the
// block ends the box, and its left one across x = 0 (y = 0, z = 0) is the
// last element of the box, a shell element when that dimension is odd.
// Batch block t -> its box (the last whose first block is
// <= t; a box without blocks shares the next box's first block, so it is
// never the last such box) -> the box's stage arguments and the block within
// the box, x fastest.  The update kernel walks the blocks backwards, as the
// single-box one does.
template <bool REVERSE>
__device__ __forceinline__ void batch_block(const StageArgs<float, float>& a, const BlockBatch& bb,
                                            StageArgs<float, float>& ab, Block& b) {
    const int t = REVERSE ? bb.n_blocks - 1 - (int)blockIdx.x : (int)blockIdx.x;
    int lo = 0, hi = bb.n_boxes - 1, off;
    if (bb.n_boxes <= kInlineBoxes) {  // kernel-argument copy: scalar loads, no memory latency chain
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (bb.blk_off[mid] <= t)
                lo = mid;
            else
                hi = mid - 1;
        }
        off = bb.blk_off[lo];
    } else {
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (uni(bb.boxes[mid].blk_off) <= t)
                lo = mid;
            else
                hi = mid - 1;
        }
        off = uni(bb.boxes[lo].blk_off);
    }
    batch_box_args(a, bb.boxes, lo, bb.stage, ab);
    b = core_block(ab, t - off);
}

template <bool VISC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(8))) void od_batch_update_block_kernel(
    StageArgs<float, float> a, BlockBatch bb) {
    StageArgs<float, float> ab;
    Block b;
    batch_block<true>(a, bb, ab, b);
    __shared__ BlockUpdateLds L;
    update_block_body<VISC>(ab, b, L);
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(8))) void od_batch_visc_block_kernel(StageArgs<float, float> a, BlockBatch bb) {
    StageArgs<float, float> ab;
    Block b;
    batch_block<false>(a, bb, ab, b);
    __shared__ BlockViscLds<false> L;
    visc_block_body<false>(ab, b, L, line_role((int)blockIdx.x));
}

// One box with an odd dimension: its core on blocks and its shell on tiles in
// one launch.  A 512-thread work-group takes a block of the core, or as many
// tiles of the shell as fit its threads and a block's LDS: three in the visc
// kernel (10.6 KB each), four in the update kernel (9.2 KB).  The shell, a small
// part of the box, whose tiles take longest from start to end, comes first in
// both, so that the blocks cover it (after the blocks it ended the launch alone:
// 33x25x37 visc 41.5 against 39.2 us, update 43.8 against 43.4 us); a launch of
// its own would cost its latency twice a stage.  The update kernel walks the
// blocks backwards, as in the even boxes.  33x25x37 (AUSM+, 100 steps): 37.4 ms
// with every element on tiles, 29.0 so.
struct CoreShell {
    int32_t n_blocks, n_tiles;  // blocks of the core, tiles of the shell
};
constexpr int kShellTiles[2] = {3, 4};  // tiles of a shell work-group: visc, update kernel
// Tile of this 128-thread part of shell work-group `group`; none left for it:
// an empty one, which touches no LDS of its own.
template <int TILES>
__device__ __forceinline__ Tile core_shell_tile(const StageArgs<float, float>& a, const CoreShell& cs, int group) {
    const int part = uni((int)(threadIdx.x >> 7));
    const int lt = TILES * group + part;
    const bool ok = part < TILES && lt < cs.n_tiles;
    Tile tl = shell_tile(a, ok ? lt : 0);
    tl.v0 = ok;
    tl.v1 = ok && tl.v1;
    return tl;
}

template <bool VISC>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(8))) void od_update_core_shell_kernel(
    StageArgs<float, float> a, CoreShell cs) {
    __shared__ union {
        BlockUpdateLds block;
        UpdateLds<float, VISC> tile[kShellTiles[1]];
    } L;
    const int w = (int)(gridDim.x - 1 - blockIdx.x);
    if (w < cs.n_blocks)
        update_block_body<VISC>(a, core_block(a, w), L.block);
    else
        update_body<float, float, VISC>(a, core_shell_tile<kShellTiles[1]>(a, cs, w - cs.n_blocks),
                                        L.tile[threadIdx.x >> 7],
                                        wave_index() & 1, threadIdx.x & 63);
}
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(8))) void od_visc_core_shell_kernel(StageArgs<float, float> a, CoreShell cs) {
    __shared__ union {
        BlockViscLds<false> block;
        ViscLds<float> tile[kShellTiles[0]];
    } L;
    const int shell = (int)gridDim.x - cs.n_blocks, w = (int)blockIdx.x - shell;
    if (w < 0) {
        int pt = threadIdx.x & 63;
        asm volatile("" : "+v"(pt));  // its own: what both forms derive from it is not hoisted and held (6 spills)
        visc_body(a, core_shell_tile<kShellTiles[0]>(a, cs, w + shell),
                  L.tile[min((int)(threadIdx.x >> 7), kShellTiles[0] - 1)], wave_index() & 1, pt);
        return;
    }
    visc_block_body<false>(a, core_block(a, w), L.block, line_role(w));
}
#endif

// LOOP = false: one unit per work-group (grid >= units, order 0); the
// persistent loop is a separate instantiation, so that its loop-carried
// state does not raise the register count of the single-unit kernel.
template <class UT, class CT, int PAIRS, bool LOOP>
__global__ __launch_bounds__(128 * PAIRS) void od_batch_visc_kernel(StageArgs<UT, CT> a, BatchArgs<UT, CT> b) {
    __shared__ ViscLds<CT> L[PAIRS];
    const int pair = PAIRS == 1 ? 0 : (int)(threadIdx.x >> 7);
    const int wave = wave_index() & 1, pt = threadIdx.x & 63;
    if constexpr (!LOOP) {
        StageArgs<UT, CT> ab;
        Tile tl;
        batch_tile(a, b, (int)blockIdx.x * PAIRS + pair, ab, tl);
        visc_body(ab, tl, L[pair], wave, pt);
        return;
    }
    for (int it = 0;; ++it) {
        const int unit = sched_unit(b.order, b.n_units, it);
        if (unit < 0) break;
        // A fresh copy of the lane index each unit keeps the compiler from
        // hoisting lane-dependent values out of the loop (they would stay
        // live in registers across the whole kernel).
        int wv = wave, pv = pt;
        asm volatile("" : "+v"(wv), "+v"(pv));
        StageArgs<UT, CT> ab;
        Tile tl;
        batch_tile(a, b, unit * PAIRS + pair, ab, tl);
        visc_body(ab, tl, L[pair], wv, pv);
        __syncthreads();  // LDS is reused by the next unit
    }
}

template <class UT, class CT, bool VISC, int PAIRS, bool LOOP>
__global__ __launch_bounds__(128 * PAIRS) __attribute__((amdgpu_waves_per_eu(LOOP ? kMinWaves<CT> : kMinWavesUpdate<UT, CT>))) void od_batch_update_kernel(
    StageArgs<UT, CT> a, BatchArgs<UT, CT> b) {
    __shared__ UpdateLds<CT, VISC> L[PAIRS];
    const int pair = PAIRS == 1 ? 0 : (int)(threadIdx.x >> 7);
    const int wave = wave_index() & 1, pt = threadIdx.x & 63;
    if constexpr (!LOOP) {  // units in reverse order, as the single-box update kernels
        StageArgs<UT, CT> ab;
        Tile tl;
        batch_tile(a, b, ((int)gridDim.x - 1 - (int)blockIdx.x) * PAIRS + pair, ab, tl);
        update_body<UT, CT, VISC>(ab, tl, L[pair], wave, pt);
        return;
    }
    for (int it = 0;; ++it) {
        const int unit = sched_unit(b.order, b.n_units, it);
        if (unit < 0) break;
        // A fresh copy of the lane index each unit keeps the compiler from
        // hoisting lane-dependent values out of the loop (they would stay
        // live in registers across the whole kernel).
        int wv = wave, pv = pt;
        asm volatile("" : "+v"(wv), "+v"(pv));
        StageArgs<UT, CT> ab;
        Tile tl;
        batch_tile(a, b, unit * PAIRS + pair, ab, tl);
        update_body<UT, CT, VISC>(ab, tl, L[pair], wv, pv);
        __syncthreads();  // LDS is reused by the next unit
    }
}

#if !OD_FAST
// Sum over d of (|u_d| + c) / dx_d at a point: the signal speed of the CFL condition.
__device__ __forceinline__ double cfl_signal(double r, double ru, double rv, double rw, double e, double dx, double dy,
                                             double dz) {
    const double ke = 0.5 * (ru * ru + rv * rv + rw * rw) / r;
    const double pp = fmax(1e-7, 0.4 * (e - ke));
    const double cs = sqrt(1.4 * pp / r);
    return (fabs(ru / r) + cs) / dx + (fabs(rv / r) + cs) / dy + (fabs(rw / r) + cs) / dz;
}
#endif

// Conservation sums: per-element GL-weighted sums (sequential over points),
// then one block reduces them in a fixed order -> deterministic.
struct W3 {
    double w[64];
};

template <class UT>
__global__ __launch_bounds__(256) void od_sums_partial_kernel(const UT* u, double* partial, int64_t E, W3 w3) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const int64_t NP = E * 64;
    for (int v = 0; v < 5; ++v) {
        double s = 0.0;
        for (int pt = 0; pt < 64; ++pt) s += w3.w[pt] * (double)u[v * NP + e * 64 + pt];
        partial[v * E + e] = s;
    }
}

__global__ __launch_bounds__(256) void od_sums_final_kernel(const double* partial, double* out, int64_t E, double jac) {
    __shared__ double red[256];
    const int t = threadIdx.x;
    for (int v = 0; v < 5; ++v) {
        double s = 0.0;
        for (int64_t e = t; e < E; e += 256) s += partial[v * E + e];
        red[t] = s;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (t < w) red[t] = red[t] + red[t + w];
            __syncthreads();
        }
        if (t == 0) out[v] = red[0] * jac;
        __syncthreads();
    }
}

#if !OD_FAST
template <class UT, class CT>
struct DtTable {
    StageDt<UT, CT> s[3];
};
template <class UT, class CT>
__global__ void od_set_dt_kernel(StageDt<UT, CT>* table, DtTable<UT, CT> v, double* dt_value, double dt) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        for (int s = 0; s < 3; ++s) table[s] = v.s[s];
        *dt_value = dt;
    }
}

// The largest signal speed of the CFL condition, in f64 from the state's values
// (the operations that the host used on its copy of the state, so that the dt is
// the same to the last bit: a maximum does not depend on its order).
// Reads the state once.
template <class UT>
__global__ __launch_bounds__(256) void od_cfl_kernel(const UT* __restrict__ u, double* __restrict__ partial, int64_t E,
                                                     double dx, double dy, double dz) {
    __shared__ double red[4];
    const int64_t NP = E * 64;
    double lam = 0.0;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < NP; q += (int64_t)gridDim.x * 256)
        lam = fmax(lam, cfl_signal((double)u[q], (double)u[NP + q], (double)u[2 * NP + q], (double)u[3 * NP + q],
                                   (double)u[4 * NP + q], dx, dy, dz));
    for (int m = 32; m >= 1; m >>= 1) lam = fmax(lam, __shfl_xor(lam, m, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = lam;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}
#endif

inline int check_launch() { return hipGetLastError() == hipSuccess ? 0 : 1; }

template <class UT, class CT>
dim3 grid_of(const StageArgs<UT, CT>& a) {
    return dim3((unsigned)((a.nx + kEpb - 1) / kEpb), (unsigned)a.ny, (unsigned)a.nz);
}

}  // namespace

template <class UT, class CT>
int launch_trace(const StageArgs<UT, CT>& a, int64_t n_elem, void* stream) {
    hipLaunchKernelGGL((od_trace_kernel<UT, CT>), grid_of(a), dim3(64 * kEpb), 0, (hipStream_t)stream, a);
    return check_launch();
}

template <class UT, class CT>
dim3 block_grid(const StageArgs<UT, CT>& a) {
    return dim3((unsigned)(a.nx / 2), (unsigned)(a.ny / 2), (unsigned)(a.nz / 2));
}

#if !OD_FAST
template <class UT, class CT>
int launch_strict_block(const StageArgs<UT, CT>& a, int kind, void* stream) {
    if (a.nx % 2 || a.ny % 2 || a.nz % 2) return 1;  // blocks of 2x2x2 elements tile the box exactly
    if (kind == 0)
        hipLaunchKernelGGL((od_visc_lines_block_kernel<UT, CT>), block_grid(a), dim3(64 * kBlk), 0, (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL((od_update_face_block_kernel<UT, CT>), block_grid(a), dim3(64 * kBlk), 0, (hipStream_t)stream, a);
    return check_launch();
}
#endif

template <class UT, class CT>
int launch_visc(const StageArgs<UT, CT>& a, int64_t n_elem, void* stream) {
#if OD_FAST
    hipLaunchKernelGGL((od_visc_kernel<UT, CT>), grid_of(a), dim3(64 * kEpb), 0, (hipStream_t)stream, a);
#else
    hipLaunchKernelGGL((od_visc_line_kernel<UT, CT>), dim3((unsigned)((n_elem + kQuad - 1) / kQuad)),
                       dim3(64 * kQuad), 0, (hipStream_t)stream, a);
#endif
    return check_launch();
}

// Largest number of tiles that the wide update kernel takes: its work-groups must
// all be resident at once, or it loses to the narrow one's finer grain (256 CUs;
// two work-groups of five waves with f64 compute, more of three).  us a step,
// narrow and wide: Euler f64 8^3 (256 tiles) 23.5 18.1, 10^3 (500) 30.0 23.5,
// 12x11x11 (726) 33.0 34.0, 16^3 58 87; Euler f32 8^3 19.9 15.9; f64 8^3 52.5
// 47.8, 13x12x12 (1008) 77.8 74.4, 15^3 (1800) 103 109; f32 8^3 40.7 38.9, 17^3
// (2601) 82.4 85.8; fast 1x16x16 (128) 33.6 31.2, 1x39x39 (760) 52.5 52.8.
template <class CT, bool VISC>
constexpr int64_t kWideTiles = 256 * (UpdateLds<CT, VISC>::kVol ? 2 : 4);

// Tiles above which the fast kernel with an f64 state holds that state in registers
// from its first load instead of loading it again for the blend.  Held it takes 70
// to 72 VGPRs, 7 waves per SIMD; loaded again 64, 8 waves, at which 4096 tiles are
// resident at once: up to there the second load is the smaller cost, above it the
// state's traffic counts.  us a step, loaded again and held: Euler 20^3 (4000 tiles)
// 61 69, 20x20x21 (4200) 73.7 71.8, 40^3 408 377; viscous 2x48x48 (2304) 84 88, 21^3
// (4851) 145 140, 40^3 784 747.
constexpr int64_t kHoldTiles = 4096;

template <class UT, class CT, bool VISC>
int launch_update(const StageArgs<UT, CT>& a, int64_t n_elem, void* stream) {
    const dim3 g = grid_of(a);
    const int64_t tiles = (int64_t)g.x * g.y * g.z;
    if (tiles <= kWideTiles<CT, VISC>) {
        hipLaunchKernelGGL((od_update_kernel<UT, CT, VISC, true, false>), g, dim3(64 * kWideWaves<CT, VISC>), 0,
                           (hipStream_t)stream, a);
        return check_launch();
    }
    if constexpr (OD_FAST && !std::is_same<UT, CT>::value) {
        if (tiles > kHoldTiles) {
            hipLaunchKernelGGL((od_update_kernel<UT, CT, VISC, false, true>), g, dim3(64 * kEpb), 0,
                               (hipStream_t)stream, a);
            return check_launch();
        }
    }
    hipLaunchKernelGGL((od_update_kernel<UT, CT, VISC, false, false>), g, dim3(64 * kEpb), 0, (hipStream_t)stream, a);
    return check_launch();
}

#if OD_FAST
template <bool VISC>
int launch_update_block(const StageArgs<float, float>& a, void* stream) {
    if (a.nx % 2 || a.ny % 2 || a.nz % 2) return 1;  // blocks of 2x2x2 elements tile the box exactly
    hipLaunchKernelGGL((od_update_block_kernel<VISC>), block_grid(a), dim3(64 * kBlk), 0, (hipStream_t)stream, a);
    return check_launch();
}
template int launch_update_block<true>(const StageArgs<float, float>&, void*);
template int launch_update_block<false>(const StageArgs<float, float>&, void*);

// Largest number of blocks that the wide visc kernel takes: one work-group to
// each of the 256 CUs.  us a launch, narrow and wide: 4^3 7.9 7.4, 8^3 (64 blocks)
// 8.4 7.7, 12^3 (216) 9.9 9.3, 14^3 (343) 11.9 12.9, 16^3 (512) 13.6 14.4.  (The
// update kernel gains 0.1 us of 8 from the like, which is not worth a second form.)
constexpr int64_t kWideBlocks = 256;
int launch_visc_block(const StageArgs<float, float>& a, void* stream) {
    if (a.nx % 2 || a.ny % 2 || a.nz % 2) return 1;
    const dim3 g = block_grid(a);
    if ((int64_t)g.x * g.y * g.z <= kWideBlocks)
        hipLaunchKernelGGL(od_visc_block_kernel<true>, g, dim3(64 * kWideBlockWaves), 0, (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL(od_visc_block_kernel<false>, g, dim3(64 * kBlk), 0, (hipStream_t)stream, a);
    return check_launch();
}
namespace {
// Blocks and shell tiles of a box at least 2 elements wide in each direction.
CoreShell core_shell(const StageArgs<float, float>& a) {
    CoreShell cs;
    cs.n_blocks = (a.nx / 2) * (a.ny / 2) * (a.nz / 2);
    cs.n_tiles = (int32_t)shell_tiles(a.nx, a.ny, a.nz);
    return cs;
}
dim3 core_shell_grid(const CoreShell& cs, int kind) {
    return dim3((unsigned)(cs.n_blocks + (cs.n_tiles + kShellTiles[kind] - 1) / kShellTiles[kind]));
}
}  // namespace

template <bool VISC>
int launch_update_core_shell(const StageArgs<float, float>& a, void* stream) {
    if (a.nx < 2 || a.ny < 2 || a.nz < 2) return 1;
    const CoreShell cs = core_shell(a);
    hipLaunchKernelGGL((od_update_core_shell_kernel<VISC>), core_shell_grid(cs, 1), dim3(64 * kBlk), 0,
                       (hipStream_t)stream, a, cs);
    return check_launch();
}
template int launch_update_core_shell<true>(const StageArgs<float, float>&, void*);
template int launch_update_core_shell<false>(const StageArgs<float, float>&, void*);

int launch_visc_core_shell(const StageArgs<float, float>& a, void* stream) {
    if (a.nx < 2 || a.ny < 2 || a.nz < 2) return 1;
    const CoreShell cs = core_shell(a);
    hipLaunchKernelGGL(od_visc_core_shell_kernel, core_shell_grid(cs, 0), dim3(64 * kBlk), 0, (hipStream_t)stream, a, cs);
    return check_launch();
}
template <bool VISC>
int launch_batch_update_block(const StageArgs<float, float>& a, const BlockBatch& bb, void* stream) {
    if (bb.n_blocks <= 0) return 0;
    hipLaunchKernelGGL((od_batch_update_block_kernel<VISC>), dim3((unsigned)bb.n_blocks), dim3(64 * kBlk), 0,
                       (hipStream_t)stream, a, bb);
    return check_launch();
}
int launch_batch_visc_block(const StageArgs<float, float>& a, const BlockBatch& bb, void* stream) {
    if (bb.n_blocks <= 0) return 0;
    hipLaunchKernelGGL(od_batch_visc_block_kernel, dim3((unsigned)bb.n_blocks), dim3(64 * kBlk), 0,
                       (hipStream_t)stream, a, bb);
    return check_launch();
}
template int launch_batch_update_block<true>(const StageArgs<float, float>&, const BlockBatch&, void*);
template int launch_batch_update_block<false>(const StageArgs<float, float>&, const BlockBatch&, void*);
#endif

template <class UT, class CT>
int launch_batch_visc(const StageArgs<UT, CT>& a, const BatchArgs<UT, CT>& b, int pairs, int groups, void* stream) {
    const bool single = groups >= b.n_units && b.order == 0;  // one unit per work-group
    const hipStream_t st = (hipStream_t)stream;
    if (pairs == 2) {
        if (single)
            hipLaunchKernelGGL((od_batch_visc_kernel<UT, CT, 2, false>), dim3(groups), dim3(256), 0, st, a, b);
        else
            hipLaunchKernelGGL((od_batch_visc_kernel<UT, CT, 2, true>), dim3(groups), dim3(256), 0, st, a, b);
    } else {
        if (single)
            hipLaunchKernelGGL((od_batch_visc_kernel<UT, CT, 1, false>), dim3(groups), dim3(128), 0, st, a, b);
        else
            hipLaunchKernelGGL((od_batch_visc_kernel<UT, CT, 1, true>), dim3(groups), dim3(128), 0, st, a, b);
    }
    return check_launch();
}

template <class UT, class CT, bool VISC>
int launch_batch_update(const StageArgs<UT, CT>& a, const BatchArgs<UT, CT>& b, int pairs, int groups, void* stream) {
    const bool single = groups >= b.n_units && b.order == 0;  // one unit per work-group
    const hipStream_t st = (hipStream_t)stream;
    if (pairs == 2) {
        if (single)
            hipLaunchKernelGGL((od_batch_update_kernel<UT, CT, VISC, 2, false>), dim3(groups), dim3(256), 0, st, a, b);
        else
            hipLaunchKernelGGL((od_batch_update_kernel<UT, CT, VISC, 2, true>), dim3(groups), dim3(256), 0, st, a, b);
    } else {
        if (single)
            hipLaunchKernelGGL((od_batch_update_kernel<UT, CT, VISC, 1, false>), dim3(groups), dim3(128), 0, st, a, b);
        else
            hipLaunchKernelGGL((od_batch_update_kernel<UT, CT, VISC, 1, true>), dim3(groups), dim3(128), 0, st, a, b);
    }
    return check_launch();
}

template <class UT, class CT>
int batch_occupancy(int kind, int pairs, bool visc, int* groups_per_cu) {
    int n = 0;
    hipError_t e;
    // the persistent (loop) kernels: the grid this sizes is a persistent one
    if (kind == 0)
        e = pairs == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, od_batch_visc_kernel<UT, CT, 2, true>, 256, 0)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, od_batch_visc_kernel<UT, CT, 1, true>, 128, 0);
    else if (visc)
        e = pairs == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                             &n, od_batch_update_kernel<UT, CT, true, 2, true>, 256, 0)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                             &n, od_batch_update_kernel<UT, CT, true, 1, true>, 128, 0);
    else
        e = pairs == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                             &n, od_batch_update_kernel<UT, CT, false, 2, true>, 256, 0)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                             &n, od_batch_update_kernel<UT, CT, false, 1, true>, 128, 0);
    *groups_per_cu = n;
    return e == hipSuccess ? 0 : 1;
}

template <class UT>
int launch_sums(const UT* u, double* partial, double* out, int64_t n_elem, const double w3[64], double jac,
                void* stream) {
    W3 w;
    for (int q = 0; q < 64; ++q) w.w[q] = w3[q];
    unsigned blocks = (unsigned)((n_elem + 255) / 256);
    hipLaunchKernelGGL((od_sums_partial_kernel<UT>), dim3(blocks), dim3(256), 0, (hipStream_t)stream, u, partial,
                       n_elem, w);
    if (check_launch()) return 1;
    hipLaunchKernelGGL(od_sums_final_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, partial, out, n_elem, jac);
    return check_launch();
}

#if !OD_FAST
template <class UT, class CT>
int launch_set_dt(StageDt<UT, CT>* table, const StageDt<UT, CT> v[3], double* dt_value, double dt, void* stream) {
    DtTable<UT, CT> t;
    for (int s = 0; s < 3; ++s) t.s[s] = v[s];
    hipLaunchKernelGGL((od_set_dt_kernel<UT, CT>), dim3(1), dim3(64), 0, (hipStream_t)stream, table, t, dt_value, dt);
    return check_launch();
}
template <class UT>
int launch_cfl(const UT* u, double* partial, int64_t n_elem, double dx, double dy, double dz, void* stream) {
    hipLaunchKernelGGL((od_cfl_kernel<UT>), dim3((unsigned)cfl_groups(n_elem)), dim3(256), 0, (hipStream_t)stream, u,
                       partial, n_elem, dx, dy, dz);
    return check_launch();
}

#endif

#define OD_INST(UT, CT)                                                                                      \
    template int launch_trace<UT, CT>(const StageArgs<UT, CT>&, int64_t, void*);                             \
    template int launch_visc<UT, CT>(const StageArgs<UT, CT>&, int64_t, void*);                              \
    template int launch_update<UT, CT, true>(const StageArgs<UT, CT>&, int64_t, void*);                      \
    template int launch_update<UT, CT, false>(const StageArgs<UT, CT>&, int64_t, void*);                     \
    template int launch_batch_visc<UT, CT>(const StageArgs<UT, CT>&, const BatchArgs<UT, CT>&, int, int, void*); \
    template int launch_batch_update<UT, CT, true>(const StageArgs<UT, CT>&, const BatchArgs<UT, CT>&, int, int, \
                                                   void*);                                                   \
    template int launch_batch_update<UT, CT, false>(const StageArgs<UT, CT>&, const BatchArgs<UT, CT>&, int, int, \
                                                    void*);                                                  \
    template int batch_occupancy<UT, CT>(int, int, bool, int*);
OD_INST(float, float)
OD_INST(double, float)
#if !OD_FAST
OD_INST(double, double)
OD_INST(float, double)
#endif
#undef OD_INST
#if !OD_FAST
template int launch_strict_block<float, float>(const StageArgs<float, float>&, int, void*);
template int launch_strict_block<double, float>(const StageArgs<double, float>&, int, void*);
template int launch_strict_block<double, double>(const StageArgs<double, double>&, int, void*);
template int launch_strict_block<float, double>(const StageArgs<float, double>&, int, void*);
template int launch_set_dt<float, float>(StageDt<float, float>*, const StageDt<float, float>*, double*, double, void*);
template int launch_set_dt<double, float>(StageDt<double, float>*, const StageDt<double, float>*, double*, double, void*);
template int launch_set_dt<double, double>(StageDt<double, double>*, const StageDt<double, double>*, double*, double, void*);
template int launch_set_dt<float, double>(StageDt<float, double>*, const StageDt<float, double>*, double*, double, void*);
template int launch_cfl<float>(const float*, double*, int64_t, double, double, double, void*);
template int launch_cfl<double>(const double*, double*, int64_t, double, double, double, void*);
template int launch_sums<float>(const float*, double*, double*, int64_t, const double*, double, void*);
template int launch_sums<double>(const double*, double*, double*, int64_t, const double*, double, void*);
#endif

int upload_ops(const Ops<float>& f32, const Ops<double>& f64) {
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_ops_f32), &f32, sizeof(f32)) != hipSuccess) return 1;
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_ops_f64), &f64, sizeof(f64)) != hipSuccess) return 1;
    return 0;
}

#if OD_FAST
}  // namespace fastmath
#endif
}  // namespace od
