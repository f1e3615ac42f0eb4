// Host-side pieces shared by the single-box (od_api.hip) and the ensemble
// (od_batch.hip) front ends: error reporting, the FR operators, stage
// arguments, CFL step and type conversion.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>

#include "../../include/opendynamo.h"
#include "od_internal.hpp"

namespace od::host {

// Sets the thread-local message read by od_last_error and returns s.
od_status fail(od_status s, const std::string& msg);
const char* last_error();

#define HIP_TRY(expr)                                                                    \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess)                                                            \
            return ::od::host::fail(OD_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

// FR P = 3 operators in f64 (fr_math.rs:3-142) and GL weights.
struct HostOps {
    double x[4], D[16], eL[4], eR[4], gL[4], gR[4], w[4];
};
HostOps fr_operators();

template <class C>
od::Ops<C> cast_ops(const HostOps& h) {
    od::Ops<C> o;
    for (int q = 0; q < 16; ++q) o.D[q] = (C)h.D[q];
    for (int q = 0; q < 4; ++q) {
        o.eL[q] = (C)h.eL[q];
        o.eR[q] = (C)h.eR[q];
        o.gL[q] = (C)h.gL[q];
        o.gR[q] = (C)h.gR[q];
    }
    return o;
}

// Whether a context's kernels are the fast build's: f32 compute with fast_math.
inline bool fast_kernels(const od_params& p) { return p.fast_math && p.compute_real == OD_F32; }

// Whether the kernels on 2x2x2-element blocks take a box's core: fast f32, at
// least 2 elements wide in each direction.
inline bool block_core(const od_params& p, int nx, int ny, int nz) {
    return p.fast_math && p.u_real == OD_F32 && p.compute_real == OD_F32 && nx >= 2 && ny >= 2 && nz >= 2;
}
// The kernels of a box that is a context of its own: boxes with a block core on
// blocks, with the last layer along each odd dimension on two-element tiles in
// the same launch; all others, and small boxes with an odd dimension, on tiles.
// Those are over with their longest work-group, which a block and a tile of the
// shell in one launch make longer than a tile is, above all beside the update
// kernel's wide form (512 tiles).  us a step, tiles against core and shell:
//   viscous  3^3 (18 tiles) 30.3 39.0, 9^3 (405) 38.5 43.9, 3x16x16 (512) 38.9
//            44.3, 8x17x8 (544) 46.0 44.4, 16x5x16 (640) 44.3 45.9, 11^3 (726)
//            47.4 47.6, 12x13x12 (936) 52.2 50.2, 13^3 (1183) 55.2 56.8, 15^3
//            (1800) 69 62
//   Euler    3^3 13.1 18.8, 9^3 15.9 20.2, 11^3 20.3 21.1, 13^3 22.9 24.7, 30x3x30
//            (1350) 24.9 25.2, 33x3x33 (1683) 27.2 26.3, 15^3 26.9 26.3, 16x16x17
//            (2176) 31.2 32.4, 17^3 (2601) 35.2 33.4
enum class BoxForm { tiles, blocks, core_shell };
inline BoxForm box_form(const od_params& p, int nx, int ny, int nz) {
    if (!block_core(p, nx, ny, nz)) return BoxForm::tiles;
    if (nx % 2 == 0 && ny % 2 == 0 && nz % 2 == 0) return BoxForm::blocks;
    const int64_t tiles = (int64_t)((nx + 1) / 2) * ny * nz;
    return tiles <= (p.viscous ? 512 : 1500) ? BoxForm::tiles : BoxForm::core_shell;
}
// Whether a strict viscous box runs on 2x2x2-element blocks when it is a context
// of its own (a batch's boxes all run on tiles): even dimensions, and two and a
// half blocks for each of the 256 CUs.  Below that the smaller work-groups of
// the other kernels fill the chip better and finish sooner: us a step, blocks
// against them, f32 / f64 / f64 state with f32 fluxes: 8^3 44 40 / 59 50 / 47 43,
// 12^3 54 51 / 73 74 / 56 56, 16^3 71 71 / 102 107 / 80 78, 20^3 107 117 /
// 178 196 / 124 139.
constexpr int64_t kStrictBlocks = 640;
inline bool strict_blocks(const od_params& p) {
    return !fast_kernels(p) && p.viscous && p.nx % 2 == 0 && p.ny % 2 == 0 && p.nz % 2 == 0 &&
           (int64_t)p.nx * p.ny * p.nz >= 8 * kStrictBlocks;
}
// Launch of kind 0 visc, 1 update of a box with a block core: blocks, or core and shell.
int launch_block_form(const od::StageArgs<float, float>& a, bool viscous, int kind, hipStream_t stream);

inline bool real_ok(int r) { return r == OD_F32 || r == OD_F64; }

template <class Dst, class Src>
void convert(Dst* d, const Src* s, size_t n) {
    for (size_t q = 0; q < n; ++q) d[q] = (Dst)s[q];
}

// SSP-RK3 Shu-Osher coefficients u = a u^n + b u^(k) + c dt L (solver.rs:275-316).
struct Coeffs {
    double a, b, cm;
    bool stage1;
};
constexpr Coeffs kStage[3] = {{1.0, 0.0, 1.0, true}, {0.75, 0.25, 0.25, false}, {1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0, false}};

// Per-box scalars, formed exactly as the reference forms them.
template <class CT>
CT jacobian(double l, int n) {  // jac = 2 / (L / n) in the compute type (rhs.cu:366-369; rk.cu:93-95)
    return ((CT)2.0) / (((CT)l) / ((CT)n));
}
inline od::BoxOps box_ops(const HostOps& h, double lx, int nx, double ly, int ny, double lz, int nz) {
    od::BoxOps o{};
    const double jac[3] = {jacobian<float>(lx, nx), jacobian<float>(ly, ny), jacobian<float>(lz, nz)};
    for (int d = 0; d < 3; ++d) {
        for (int q = 0; q < 16; ++q) o.table[16 * d + q] = (float)(jac[d] * h.D[q]);
        for (int q = 0; q < 4; ++q) {
            o.table[48 + 8 * d + 2 * q] = (float)(jac[d] * h.gL[q]);
            o.table[48 + 8 * d + 2 * q + 1] = (float)(jac[d] * h.gR[q]);
        }
        for (int i = 0; i < 2; ++i) {
            const double* D = h.D + 4 * i;
            o.line[d][i] = {(float)(jac[d] * 0.25 * ((D[0] + D[3]) - (D[1] + D[2]))),
                            (float)(jac[d] * 0.25 * (h.gL[i] + h.gR[i])), (float)(jac[d] * 0.5 * (D[0] - D[3])),
                            (float)(jac[d] * 0.5 * (D[1] - D[2])), (float)(jac[d] * 0.25 * (h.gL[i] - h.gR[i]))};
        }
    }
    for (int q = 0; q < 4; ++q) {
        o.table[72 + q] = (float)h.eL[q];
        o.table[76 + q] = (float)h.eR[q];
    }
    return o;
}
template <class T>
T stage_dt_coef(int stage, double dt) {  // c * dt in type T from the f32 dt (solver.rs:256)
    return (T)kStage[stage].cm * (T)dt;
}

// Kernel arguments of one stage for a box whose state buffers are u[0], u[1]
// and whose traces / fv / debug arrays start at the given pointers.
// Buffer roles: stage 1 u0 -> u1, stage 2 u1 -> u1, stage 3 u1 -> u0; traces
// tr[s] -> tr[s+1 mod 3].
template <class UT, class CT>
od::StageArgs<UT, CT> make_stage_args(const od_params& p, int nx, int ny, int nz, double lx, double ly, double lz,
                                      void* const u[2], void* const tr[3], void* fv, void* dbg, int stage,
                                      double dt) {
    od::StageArgs<UT, CT> a{};
    UT* u0 = (UT*)u[0];
    UT* u1 = (UT*)u[1];
    a.uin = stage == 0 ? u0 : u1;
    a.uprev = u0;
    a.uout = stage == 2 ? u0 : u1;
    a.tr_in = (const CT*)tr[stage];
    a.tr_out = (CT*)tr[(stage + 1) % 3];
    a.fv = (CT*)fv;
    a.dbg = (CT*)dbg;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.wall = p.y_wall ? 1 : 0;
    a.flux = p.flux_scheme;
    a.sutherland = p.viscosity_model == 1 ? 1 : 0;
    a.round_q = (sizeof(CT) == 8 && p.q_real == OD_F32) ? 1 : 0;
    a.round_rhs = (sizeof(CT) == 8 && p.rhs_real == OD_F32) ? 1 : 0;
    a.accum_state = p.rk_accum ? 1 : 0;
    a.stage1 = kStage[stage].stage1 ? 1 : 0;
    a.mode = 0;
    a.jx = jacobian<CT>(lx, nx);
    a.jy = jacobian<CT>(ly, ny);
    a.jz = jacobian<CT>(lz, nz);
    a.mu = (CT)p.mu_ref;
    a.mu_ref = (CT)p.mu_ref;
    a.t_ref = (CT)p.t_ref;
    a.s_suth = (CT)p.s_suth;
    a.bf = (CT)p.body_force_x;
    const Coeffs& k = kStage[stage];
    a.ca = (CT)k.a;
    a.cb = (CT)k.b;
    a.cc = stage_dt_coef<CT>(stage, dt);
    a.ua = (UT)k.a;
    a.ub = (UT)k.b;
    a.uc = stage_dt_coef<UT>(stage, dt);
    return a;
}

// dt = cfl / ((2P+1) max_points sum_d (|u_d| + c) / dx_d), rounded to f32: the
// launch for a state [5][64 E] on the device, which leaves the maxima of
// od::cfl_groups(E) groups in partial, and the dt from those, on the host.
od_status enqueue_cfl(const void* u, int u_real, int64_t E, double dx, double dy, double dz, double* partial,
                      hipStream_t stream);
double cfl_dt(const double* partial, int groups, double cfl);

}  // namespace od::host
