// Learned closure (no reference counterpart): element features, the MLP
// (BF16 weights and activations on MFMA, FP32 accumulation; hand-written
// forward and backward), Adam, and the eddy-viscosity refresh of a solver
// context with its training-range and kinetic-energy-budget fallbacks.
//
// MFMA used: v_mfma_f32_16x16x16_bf16, D[16x16] = A[16x16] B[16x16] + C with,
// for lane l (r = l % 16, g = l / 16):
//   A: row r, k = 4g .. 4g+3        B: column r, k = 4g .. 4g+3
//   D: rows 4g .. 4g+3, column r
// A tile is 16 elements; a layer Z = H W^T (H [16][K], W [64][K]) is 4
// column blocks x K/16 k-steps.  The transposes between the D layout
// (elements along the 4 registers) and the A layout (elements along lanes)
// go through LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "od_ctx.hpp"
#include "od_order.hpp"

using namespace od::host;

namespace {

constexpr int NF = OD_MLP_FEATURES;    // 12 input features
constexpr int KP = 16;                 // padded input width
constexpr int NH = OD_MLP_HIDDEN;      // 64 hidden units
constexpr int FS = OD_FEATURE_STRIDE;  // floats per element from the feature kernel
constexpr int oW1 = 0, oB1 = oW1 + NH * NF, oW2 = oB1 + NH, oB2 = oW2 + NH * NH, oW3 = oB2 + NH,
              oB3 = oW3 + NH * NH, oW4 = oB3 + NH, oB4 = oW4 + NH, NPARAM = oB4 + 1;
static_assert(NPARAM == OD_MLP_PARAMS, "parameter layout");
constexpr int LDH = NH + 8;  // LDS row stride (bf16) of a 16 x 64 activation tile

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// f32 -> bf16, round to nearest even (finite inputs).
__host__ __device__ inline unsigned short f2bf(float x) {
    uint32_t u;
    std::memcpy(&u, &x, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ inline float bf2f(unsigned short b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// tanh-form GELU; d: its derivative
__device__ inline float gelu(float x, float* d = nullptr) {
    const float a = 0.7978845608028654f, b = 0.044715f;
    const float t = tanhf(a * (x + b * x * x * x));
    if (d) *d = 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * a * (1.0f + 3.0f * b * x * x);
    return 0.5f * x * (1.0f + t);
}
__device__ inline float softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }
__device__ inline float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

// Lane exchanges without LDS.
template <int CTRL>
__device__ inline float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
// Sum over the wave in every lane: the butterfly over lane ^ 32, 16, 8, 4, 2, 1, as
// half and row swaps and DPP operands (after the step over 8 a row's lanes 8 apart
// hold the same value, so a rotation by 4 is the exchange with lane ^ 4).  With
// the 18 sums of an element's features off the LDS permutes their kernel takes 9.2
// instead of 10.7 us for 4096 elements.
__device__ inline float wave_sum(float v) {
    auto h = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = __int_as_float(h[0]) + __int_as_float(h[1]);
    h = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    v = __int_as_float(h[0]) + __int_as_float(h[1]);
    v += dpp<0x128>(v);  // row_ror:8
    v += dpp<0x124>(v);  // row_ror:4
    v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
    return v;
}
// sum over the 16 lanes that share l / 16
__device__ inline float group16_sum(float v) {
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}
// sum over the 4 lane groups (same l % 16)
__device__ inline float across_groups(float v) {
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}

// ---------------------------------------------------------------------------
// Feature kernel: one wave per element, lane = solution point.
// ---------------------------------------------------------------------------
struct FeatConsts {
    float D[16];    // D[i][m] = l_m'(x_i)
    float L[16];    // L[a][i] = (2a+1)/2 w_i P_a(x_i): nodal -> Legendre modal
    float w[4];     // GL weights
    float nrm[4];   // 2 / (2a+1)
    float jx, jy, jz;      // 2 / h_d
    float vol8;            // element volume / 8 (dV = vol8 dxi deta dzeta)
    float delta;           // (h_x h_y h_z)^(1/3) / 4
    float mu_mol;
};

template <class UT>
__global__ __launch_bounds__(256) void od_features_kernel(const UT* __restrict__ u, int64_t E, FeatConsts fc,
                                                          float* __restrict__ out) {
    __shared__ float sv[4][3][64];
    __shared__ float sm[4][3][64];
    const int wave = threadIdx.x >> 6, pt = threadIdx.x & 63;
    const int i = pt & 3, j = (pt >> 2) & 3, k = pt >> 4;
    const int64_t e = (int64_t)blockIdx.x * 4 + wave;
    const bool ok = e < E;
    const int64_t NP = E * 64;
    float rho = 1.0f, mx = 0.0f, my = 0.0f, mz = 0.0f, en = 2.5f;
    if (ok) {
        const int64_t q = e * 64 + pt;
        rho = (float)u[q];
        mx = (float)u[NP + q];
        my = (float)u[2 * NP + q];
        mz = (float)u[3 * NP + q];
        en = (float)u[4 * NP + q];
    }
    const float ux = mx / rho, uy = my / rho, uz = mz / rho;
    const float u2 = ux * ux + uy * uy + uz * uz;
    const float ke = 0.5f * rho * u2;
    const float p = 0.4f * (en - ke);
    const float c = sqrtf(fmaxf(1.4f * p / rho, 0.0f));
    sv[wave][0][pt] = ux;
    sv[wave][1][pt] = uy;
    sv[wave][2][pt] = uz;
    __syncthreads();
    // velocity gradient A[a][d] = du_a / dx_d
    float A[3][3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int idx = d == 0 ? i : (d == 1 ? j : k);
        const int base = d == 0 ? 4 * j + 16 * k : (d == 1 ? i + 16 * k : i + 4 * j);
        const int stride = d == 0 ? 1 : (d == 1 ? 4 : 16);
        const float jac = d == 0 ? fc.jx : (d == 1 ? fc.jy : fc.jz);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float s = 0.0f;
#pragma unroll
            for (int m = 0; m < 4; ++m) s += fc.D[idx * 4 + m] * sv[wave][a][base + m * stride];
            A[a][d] = s * jac;
        }
    }
    // Legendre modal coefficients of the velocity: x, then y, then z
    float t[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float s = 0.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m) s += fc.L[i * 4 + m] * sv[wave][a][m + 4 * j + 16 * k];
        t[a] = s;
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) sm[wave][a][pt] = t[a];
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float s = 0.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m) s += fc.L[j * 4 + m] * sm[wave][a][i + 4 * m + 16 * k];
        t[a] = s;
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 3; ++a) sv[wave][a][pt] = t[a];
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float s = 0.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m) s += fc.L[k * 4 + m] * sv[wave][a][i + 4 * j + 16 * m];
        t[a] = s;
    }
    const float emode = (t[0] * t[0] + t[1] * t[1] + t[2] * t[2]) * fc.nrm[i] * fc.nrm[j] * fc.nrm[k];
    const int top = max(i, max(j, k));

    // invariants at the point
    const float div = A[0][0] + A[1][1] + A[2][2];
    float ss = 0.0f, oo = 0.0f, tr3 = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const float sab = 0.5f * (A[a][b] + A[b][a]) - (a == b ? div / 3.0f : 0.0f);
            const float oab = 0.5f * (A[a][b] - A[b][a]);
            ss += sab * sab;
            oo += oab * oab;
#pragma unroll
            for (int q = 0; q < 3; ++q) tr3 += A[a][b] * A[b][q] * A[q][a];
        }
    const float smag = sqrtf(2.0f * ss), omag = sqrtf(2.0f * oo);
    float sfull = 0.0f;  // S_ij S_ij of the full strain for Q
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const float sab = 0.5f * (A[a][b] + A[b][a]);
            sfull += sab * sab;
        }
    const float Q = 0.5f * (oo - sfull);
    const float R = -tr3 / 3.0f;

    const float w = fc.w[i] * fc.w[j] * fc.w[k];
    const float inv8 = 0.125f;  // 1 / sum of the weights
    const float s_rho = wave_sum(w * rho), s_p = wave_sum(w * p), s_c = wave_sum(w * c);
    const float s_S = wave_sum(w * smag), s_O = wave_sum(w * omag), s_Q = wave_sum(w * Q), s_R = wave_sum(w * R);
    const float s_div = wave_sum(w * div);
    const float s_ux = wave_sum(w * ux), s_uy = wave_sum(w * uy), s_uz = wave_sum(w * uz);
    const float s_ke = wave_sum(w * ke), s_SS = wave_sum(w * 2.0f * ss);
    // second moments about the element means (two passes, no cancellation)
    const float dr = rho - s_rho * inv8, dp = p - s_p * inv8;
    const float dux = ux - s_ux * inv8, duy = uy - s_uy * inv8, duz = uz - s_uz * inv8;
    const float v_rho = wave_sum(w * dr * dr), v_p = wave_sum(w * dp * dp);
    const float v_u = wave_sum(w * (dux * dux + duy * duy + duz * duz));
    const float e1 = wave_sum(top == 1 ? emode : 0.0f), e2 = wave_sum(top == 2 ? emode : 0.0f),
                e3 = wave_sum(top == 3 ? emode : 0.0f);
    if (!ok) return;
    const float rb = s_rho * inv8, pb = s_p * inv8, cb = s_c * inv8, dl = fc.delta;
    const float S = fmaxf(s_S * inv8, 1e-6f * cb / dl);
    const float etot = e1 + e2 + e3 + 1e-30f;
    float f[FS];
    f[0] = logf(rb * dl * dl * S / fc.mu_mol);
    f[1] = s_O * inv8 / S;
    f[2] = s_Q * inv8 / (S * S);
    f[3] = s_R * inv8 / (S * S * S);
    f[4] = s_div * inv8 / S;
    f[5] = e1 / etot;
    f[6] = e2 / etot;
    f[7] = e3 / etot;
    f[8] = sqrtf(v_rho * inv8) / rb;
    f[9] = sqrtf(v_p * inv8) / pb;
    f[10] = dl * S / cb;
    f[11] = sqrtf(v_u * inv8) / (dl * S);
    f[12] = rb;
    f[13] = dl * dl * S;
    f[14] = s_ke * fc.vol8;
    f[15] = s_SS * fc.vol8;
    float val = 0.0f;
#pragma unroll
    for (int q = 0; q < FS; ++q) val = pt == q ? f[q] : val;
    if (pt < FS) out[e * FS + pt] = val;
}

// ---------------------------------------------------------------------------
// MLP device weights: bf16 copies of W1 (padded to [64][16]), W2, W3 and their
// transposes, w4, and f32 biases, refreshed from the f32 master vector after
// each update.
// ---------------------------------------------------------------------------
struct DevNet {
    unsigned short* w1;   // [64][16]
    unsigned short* w2;   // [64][64]
    unsigned short* w3;   // [64][64]
    unsigned short* w2t;  // w2t[in][out] = W2[out][in]
    unsigned short* w3t;
    unsigned short* w4;   // [64]
    const float* params;  // f32 master (biases read from it)
};
constexpr int kNetShorts = NH * KP + 4 * NH * NH + NH;

struct Scaling {
    float shift[NF], scale[NF], lo[NF], hi[NF];
    float out_scale;  // C = out_scale * softplus(z)
};

// bf16 copies of parameter p of the master vector (the pads of w1 stay zero).
__device__ inline void store_weight(const DevNet& net, int p, float x) {
    const unsigned short b = f2bf(x);
    if (p < oB1) {
        net.w1[p / NF * KP + p % NF] = b;
    } else if (p >= oW2 && p < oB2) {
        const int q = p - oW2;
        net.w2[q] = b;
        net.w2t[q % NH * NH + q / NH] = b;
    } else if (p >= oW3 && p < oB3) {
        const int q = p - oW3;
        net.w3[q] = b;
        net.w3t[q % NH * NH + q / NH] = b;
    } else if (p >= oW4 && p < oB4) {
        net.w4[p - oW4] = b;
    }
}

__global__ void od_mlp_cast_kernel(DevNet net) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < NH * KP && t % KP >= NF) net.w1[t] = 0;
    if (t < NPARAM) store_weight(net, t, net.params[t]);
}

// ---------------------------------------------------------------------------
// A tile of 16 elements is the work of a 256-thread group: wave nb owns the 16
// columns 16 nb .. 16 nb + 15 of every layer.  Its weight rows (and, for the
// backward pass, its rows of the transposes) are the same for every tile, so
// they stay in registers (8-byte loads of the bf16 copies, 10 or 18 per lane);
// LDS holds the activations only, and the group's four waves share the GELUs,
// which are most of a tile's instructions.  With one tile to a wave and the
// weights in LDS (55 KB a group) there was one wave to a SIMD: the gradient
// took 112 us (batches of 65536 and 32768 samples in turn), here 60 us, and the
// inference of 4096 elements 25 us, here 6 us.  Every value is the same sum in
// the same order in both forms.
// ---------------------------------------------------------------------------
struct ColNet {
    bf16x4 w1[1], w2[4], w3[4];  // rows 16 nb + r, k = 16 kb + 4 g ..
    float b1, b2, b3, b4;
    float w4[4];                 // w4[16 q + r], every column block
};
__device__ inline bf16x4 get4(const unsigned short* p) { return *reinterpret_cast<const bf16x4*>(p); }

__device__ inline ColNet load_cols(const DevNet& net, int nb, int lane) {
    ColNet c;
    const int n = nb * 16 + (lane & 15), kq = (lane >> 4) * 4;
    c.w1[0] = get4(net.w1 + n * KP + kq);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        c.w2[kb] = get4(net.w2 + n * NH + kb * 16 + kq);
        c.w3[kb] = get4(net.w3 + n * NH + kb * 16 + kq);
        c.w4[kb] = bf2f(net.w4[kb * 16 + (lane & 15)]);
    }
    c.b1 = net.params[oB1 + n];
    c.b2 = net.params[oB2 + n];
    c.b3 = net.params[oB3 + n];
    c.b4 = net.params[oB4];
    return c;
}

// The wave's 16 columns of Z[16][64] = H[16][16 KB] W^T + b: z[q] = Z[4g + q][16 nb + r].
template <int KB>
__device__ inline f32x4 dense_col(const unsigned short* H, int ldh, const bf16x4* w, float b, int lane) {
    f32x4 z = f32x4{b, b, b, b};
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) z = mfma(get4(H + (lane & 15) * ldh + kb * 16 + (lane >> 4) * 4), w[kb], z);
    return z;
}

constexpr int LDT = 20;  // LDS row stride (bf16) of a transposed tile [column][16 elements]

// h = GELU(z) in bf16 -> the wave's columns of Hout[16][LDH]; the transposed
// tile HT [64][LDT] too, where the backward pass reads it.  d: GELU'(z), from
// the same tanh.
__device__ inline bf16x4 act_col(const f32x4 z, unsigned short* Hout, unsigned short* HT, int nb, int lane,
                                 f32x4* d = nullptr) {
    const int r = lane & 15, g = lane >> 4;
    bf16x4 h;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float dq;
        h[q] = (short)f2bf(gelu(z[q], d ? &dq : nullptr));
        if (d) (*d)[q] = dq;
        Hout[(4 * g + q) * LDH + nb * 16 + r] = (unsigned short)h[q];
    }
    if (HT) *reinterpret_cast<bf16x4*>(HT + (nb * 16 + r) * LDT + 4 * g) = h;
    return h;
}

// Output layer before softplus: z4[q] for element 4g + q (every lane of the group of 16).
__device__ inline void out_layer(const unsigned short* H3, const ColNet& c, int lane, float z4[4]) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float s = 0.0f;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) s += bf2f(H3[(4 * g + q) * LDH + nb * 16 + r]) * c.w4[nb];
        z4[q] = group16_sum(s) + c.b4;
    }
}
__device__ inline float pick4(const float v[4], int q) {
    return q == 0 ? v[0] : (q == 1 ? v[1] : (q == 2 ? v[2] : v[3]));
}

struct TileLds {
    alignas(16) unsigned short h0[16 * KP];
    alignas(16) unsigned short h1[16 * LDH];
    alignas(16) unsigned short h2[16 * LDH];
    alignas(16) unsigned short h3[16 * LDH];
};

// The tile's hidden layers from the standardised inputs in S.h0 (a barrier
// first), every wave its columns; returns z4 of every element.
__device__ inline void forward_tile(TileLds& S, const ColNet& c, int nb, int lane, float z4[4]) {
    __syncthreads();
    act_col(dense_col<1>(S.h0, KP, c.w1, c.b1, lane), S.h1, nullptr, nb, lane);
    __syncthreads();
    act_col(dense_col<4>(S.h1, LDH, c.w2, c.b2, lane), S.h2, nullptr, nb, lane);
    __syncthreads();
    act_col(dense_col<4>(S.h2, LDH, c.w3, c.b3, lane), S.h3, nullptr, nb, lane);
    __syncthreads();
    out_layer(S.h3, c, lane, z4);
}

// ---- inference: mu_t per element of a solver context -----------------------
template <class CT>
__global__ __launch_bounds__(256) void od_mlp_infer_kernel(DevNet net, Scaling sc, const float* __restrict__ feat,
                                                           int64_t E, CT* __restrict__ mu_t,
                                                           float* __restrict__ eps, float* __restrict__ out_of_range) {
    __shared__ TileLds S;
    __shared__ float aux[16][4];  // features 12..15 of the tile's elements
    __shared__ int inside[16];
    const int nb = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const ColNet c = load_cols(net, nb, lane);
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const float shift = col < NF ? sc.shift[col] : 0.0f, scale = col < NF ? sc.scale[col] : 0.0f;
    const float lo = col < NF ? sc.lo[col] : 0.0f, hi = col < NF ? sc.hi[col] : 0.0f;
    const int64_t tiles = (E + 15) / 16;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t e0 = tile * 16;
        static_assert(FS == 16 && KP == 16, "one thread per feature");
        const float f = e0 + row < E ? feat[(e0 + row) * FS + col] : 0.0f;
        const bool ok = col >= NF || (f >= lo && f <= hi);
        const unsigned long long all = __ballot(ok);
        if (tile != blockIdx.x) __syncthreads();  // the previous tile's reads of LDS are done
        S.h0[row * KP + col] = f2bf(col < NF ? (e0 + row < E ? (f - shift) * scale : 0.0f) : 0.0f);
        if (col >= NF) aux[row][col - NF] = f;
        if (col == 0) inside[row] = ((all >> (lane & 48)) & 0xffffull) == 0xffffull;
        float z4[4];
        forward_tile(S, c, nb, lane, z4);
        const int q = lane & 15, r = 4 * (lane >> 4) + q;  // wave 0: lanes q < 4 take element r
        if (nb == 0 && q < 4 && e0 + r < E) {
            const bool in = inside[r];
            const float m = in ? aux[r][0] * aux[r][1] * (sc.out_scale * softplus(pick4(z4, q))) : 0.0f;
            mu_t[e0 + r] = (CT)m;
            eps[e0 + r] = m * aux[r][3];
            out_of_range[e0 + r] = in ? 0.0f : 1.0f;
        }
    }
}

// ---- forward on host-given features (testing / evaluation) ----------------
__global__ __launch_bounds__(256) void od_mlp_forward_kernel(DevNet net, Scaling sc, const float* __restrict__ x,
                                                             int64_t n, float* __restrict__ y) {
    __shared__ TileLds S;
    const int nb = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const ColNet c = load_cols(net, nb, lane);
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const float shift = col < NF ? sc.shift[col] : 0.0f, scale = col < NF ? sc.scale[col] : 0.0f;
    const int64_t tiles = (n + 15) / 16;
    for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t e0 = tile * 16;
        const float v = e0 + row < n && col < NF ? (x[(e0 + row) * NF + col] - shift) * scale : 0.0f;
        if (tile != blockIdx.x) __syncthreads();  // the previous tile's reads of LDS are done
        S.h0[row * KP + col] = f2bf(v);
        float z4[4];
        forward_tile(S, c, nb, lane, z4);
        const int q = lane & 15, r = 4 * (lane >> 4) + q;
        if (nb == 0 && q < 4 && e0 + r < n) y[e0 + r] = sc.out_scale * softplus(pick4(z4, q));
    }
}

// ---- backward ----------------------------------------------------------------
struct GradLds {
    alignas(16) unsigned short h0[16 * KP];
    alignas(16) unsigned short h1[16 * LDH];
    alignas(16) unsigned short h2[16 * LDH];
    alignas(16) unsigned short h3[16 * LDH];
    alignas(16) unsigned short h0t[KP * LDT];  // transposed inputs and activations
    alignas(16) unsigned short h1t[NH * LDT];
    alignas(16) unsigned short h2t[NH * LDT];
    alignas(16) unsigned short g3[16 * LDH];   // bf16 dZ of layers 3 and 2
    alignas(16) unsigned short g2[16 * LDH];
    alignas(16) unsigned short w2t[NH * LDH];  // the transposed weights
    alignas(16) unsigned short w3t[NH * LDH];
    float tgt[16];
};

// The wave's columns of dZ in bf16 (-> G[16][LDH], where the layer below needs
// all of them); bias gradient accumulated.
__device__ inline bf16x4 dz_col(const f32x4 dz, unsigned short* G, int nb, int lane, float& db) {
    const int r = lane & 15, g = lane >> 4;
    bf16x4 b;
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        b[q] = (short)f2bf(dz[q]);
        if (G) G[(4 * g + q) * LDH + nb * 16 + r] = (unsigned short)b[q];
        s += dz[q];
    }
    db += across_groups(s);
    return b;
}
// dW[16 nb ..][in] += sum_e dZ[e][out] H[e][in] over the tile's 16 elements.
// The A operand (dZ^T: row out, k element) is the lane's own dz.
template <int CB>
__device__ inline void weight_grad_col(const bf16x4 dz, const unsigned short* HT, int lane, f32x4 acc[CB]) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
        acc[cb] = mfma(dz, get4(HT + (cb * 16 + (lane & 15)) * LDT + (lane >> 4) * 4), acc[cb]);
}

// The wave's columns of dH[16][64] = dZ[16][64] W, from the transpose of W in LDS.
__device__ inline f32x4 back_col(const unsigned short* G, const unsigned short* WT, int nb, int lane) {
    const int r = lane & 15, kq = (lane >> 4) * 4;
    f32x4 d = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
        d = mfma(get4(G + r * LDH + kb * 16 + kq), get4(WT + (nb * 16 + r) * LDH + kb * 16 + kq), d);
    return d;
}

constexpr int kPartialRow = (NPARAM + 1 + 31) / 32 * 32;  // floats; rows start on 128 bytes

// Partial gradients of work-group gw over its contiguous range of 16-element
// tiles of the (gathered) batch -> partial[gw][NPARAM + 1] (last entry: sum of
// the squared errors).  Loss = mean over the batch of (C - t)^2.  At most 1024
// groups (four to a CU: all resident), each with the next tile's inputs on the
// way while it works on this one's.  At the 128 VGPRs that four waves per SIMD
// leave it, 60 registers are spilled (236 bytes a lane).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void od_mlp_grad_kernel(
    DevNet net, Scaling sc, const float* __restrict__ x, const float* __restrict__ tgt, const int* __restrict__ idx,
    int64_t n, int tiles_per_group, float* __restrict__ partial) {
    __shared__ GradLds S;
    const int nb = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
    const float shift = col < NF ? sc.shift[col] : 0.0f, scale = col < NF ? sc.scale[col] : 0.0f;
    const int64_t first = (int64_t)blockIdx.x * tiles_per_group * 16;
    // column col < 12: a raw feature, column 12: the target of the tile's row
    auto fetch = [&](int64_t e) -> float {
        if (e >= n || col > NF) return 0.0f;
        const int64_t src = idx ? (int64_t)idx[e] : e;
        return col < NF ? x[src * NF + col] : tgt[src];
    };
    float in = fetch(first + row);
    const ColNet c = load_cols(net, nb, lane);
    for (int q = threadIdx.x; q < NH * NH / 4; q += 256) {
        *reinterpret_cast<bf16x4*>(S.w2t + q / 16 * LDH + q % 16 * 4) = get4(net.w2t + 4 * q);
        *reinterpret_cast<bf16x4*>(S.w3t + q / 16 * LDH + q % 16 * 4) = get4(net.w3t + 4 * q);
    }
    const float inv_n = 1.0f / (float)n;
    const float w4 = pick4(c.w4, nb);
    f32x4 aW1[1] = {f32x4{0, 0, 0, 0}}, aW2[4], aW3[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) aW2[b] = aW3[b] = f32x4{0, 0, 0, 0};
    float db1 = 0.0f, db2 = 0.0f, db3 = 0.0f, dw4 = 0.0f, db4 = 0.0f, sse = 0.0f;
    for (int tt = 0; tt < tiles_per_group; ++tt) {
        const int64_t e0 = first + (int64_t)tt * 16;
        if (e0 >= n) break;
        __syncthreads();  // the previous tile's reads of LDS are done
        const unsigned short hb = f2bf(e0 + row < n && col < NF ? (in - shift) * scale : 0.0f);
        S.h0[row * KP + col] = hb;
        S.h0t[col * LDT + row] = hb;
        if (col == NF) S.tgt[row] = in;
        if (tt + 1 < tiles_per_group) in = fetch(e0 + 16 + row);
        __syncthreads();
        f32x4 d1, d2, d3;
        act_col(dense_col<1>(S.h0, KP, c.w1, c.b1, lane), S.h1, S.h1t, nb, lane, &d1);
        __syncthreads();
        act_col(dense_col<4>(S.h1, LDH, c.w2, c.b2, lane), S.h2, S.h2t, nb, lane, &d2);
        __syncthreads();
        const bf16x4 h3 = act_col(dense_col<4>(S.h2, LDH, c.w3, c.b3, lane), S.h3, nullptr, nb, lane, &d3);
        __syncthreads();
        float z4[4];
        out_layer(S.h3, c, lane, z4);
        // dL/dz4: lane r & 3 = q of a group forms element 4g + q's, the others take it from there
        float dz4[4];
        {
            const int q = r & 3;
            const float z = pick4(z4, q);
            float d = 0.0f, err = 0.0f;
            if (e0 + 4 * g + q < n) {
                err = sc.out_scale * softplus(z) - S.tgt[4 * g + q];
                d = 2.0f * err * inv_n * sc.out_scale * sigmoid(z);
            }
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                dz4[p] = __shfl(d, (lane & 48) | p, 64);
                const float ep = __shfl(err, (lane & 48) | p, 64);
                if (r == 0) sse += ep * ep;
            }
        }
        // output layer gradients
        {
            float s = 0.0f, sb = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                s += dz4[q] * bf2f((unsigned short)h3[q]);
                sb += dz4[q];
            }
            dw4 += across_groups(s);
            db4 += across_groups(r == 0 ? sb : 0.0f);
        }
        // layer 3
        f32x4 dz;
#pragma unroll
        for (int q = 0; q < 4; ++q) dz[q] = dz4[q] * w4 * d3[q];
        weight_grad_col<4>(dz_col(dz, S.g3, nb, lane, db3), S.h2t, lane, aW3);
        __syncthreads();
        f32x4 dh = back_col(S.g3, S.w3t, nb, lane);
        // layer 2
#pragma unroll
        for (int q = 0; q < 4; ++q) dz[q] = dh[q] * d2[q];
        weight_grad_col<4>(dz_col(dz, S.g2, nb, lane, db2), S.h1t, lane, aW2);
        __syncthreads();
        dh = back_col(S.g2, S.w2t, nb, lane);
        // layer 1
#pragma unroll
        for (int q = 0; q < 4; ++q) dz[q] = dh[q] * d1[q];
        weight_grad_col<1>(dz_col(dz, nullptr, nb, lane, db1), S.h0t, lane, aW1);
    }
    float* out = partial + (int64_t)blockIdx.x * kPartialRow;
    // weight matrices: acc[cb][q] = dW[out = 16 nb + 4g + q][in = 16 cb + r]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int o = 16 * nb + 4 * g + q;
        if (r < NF) out[oW1 + o * NF + r] = aW1[0][q];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            out[oW2 + o * NH + 16 * cb + r] = aW2[cb][q];
            out[oW3 + o * NH + 16 * cb + r] = aW3[cb][q];
        }
    }
    if (g == 0) {
        out[oB1 + nb * 16 + r] = db1;
        out[oB2 + nb * 16 + r] = db2;
        out[oB3 + nb * 16 + r] = db3;
        out[oW4 + nb * 16 + r] = dw4;
    }
    const float tot = wave_sum(sse);
    if (nb == 0 && lane == 0) {
        out[oB4] = db4;
        out[NPARAM] = tot;
    }
}

struct Adam {
    float *p, *m, *v;
    float lr, b1t, b2t;
    float* sse;  // the batch's sum of squared errors goes here as well
};

// grad[p] = sum over the partial rows, in row order (deterministic), for the 32
// parameters of this work-group; with STEP the Adam update of those parameters
// and their bf16 copies too.  The rows come through LDS 128 at a time, all 256
// threads loading the next 128 while 32 lanes add up these: the additions stay
// in one chain per parameter, but no load waits in it: 15 us with the Adam step
// for 1024 rows, where one thread per parameter reading its column took 242 us
// (and the step and the bf16 copies 11 us more).
template <bool STEP>
__global__ __launch_bounds__(256) void od_mlp_reduce_kernel(const float* __restrict__ partial, int rows,
                                                            float* __restrict__ grad, Adam ad, DevNet net) {
    constexpr int R = 128, C = 32, PER = R * C / 256;
    __shared__ float buf[2][R][C];
    const int c = threadIdx.x % C, r0 = threadIdx.x / C;
    const int p = blockIdx.x * C + c;  // < kPartialRow: inside the row
    float v[PER];
    auto load = [&](int at) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int row = at + r0 + q * (256 / C);
            v[q] = row < rows ? partial[(int64_t)row * kPartialRow + p] : 0.0f;
        }
    };
    load(0);
    float s = 0.0f;
    for (int at = 0, k = 0; at < rows; at += R, k ^= 1) {
#pragma unroll
        for (int q = 0; q < PER; ++q) buf[k][r0 + q * (256 / C)][c] = v[q];
        __syncthreads();
        if (at + R < rows) load(at + R);
        if (threadIdx.x < C) {
            const int m = min(R, rows - at);
            if (m == R) {
#pragma unroll 16
                for (int q = 0; q < R; ++q) s += buf[k][q][c];
            } else {
                for (int q = 0; q < m; ++q) s += buf[k][q][c];
            }
        }
    }
    if (threadIdx.x >= C || p > NPARAM) return;
    grad[p] = s;
    if constexpr (STEP) {
        if (p == NPARAM) {
            *ad.sse = s;
            return;
        }
        const float mm = 0.9f * ad.m[p] + 0.1f * s;
        const float vv = 0.999f * ad.v[p] + 0.001f * s * s;
        ad.m[p] = mm;
        ad.v[p] = vv;
        const float mh = mm / (1.0f - ad.b1t), vh = vv / (1.0f - ad.b2t);
        const float x = ad.p[p] - ad.lr * mh / (sqrtf(vh) + 1e-8f);
        ad.p[p] = x;
        store_weight(net, p, x);
    }
}

// The kinetic-energy budget of a closure interval, on the device: its state is
// kept there so that a step with a network never waits for the device.
enum { kKePrev, kEpsPrev, kActive, kStats, kBudget = kStats + 6 };

// Sums (one block of 256, fixed order) of the elements' kinetic energy, model
// dissipation and out-of-range flags, then the check of the interval that just
// ended; when it fails, mu_t is zero for the next one.  dt: the step size;
// interval = update_interval.
// The model over-dissipates when, over an interval in which the kinetic energy
// decayed, the energy it removed exceeds kappa times the whole observed decay.
// An interval in which the energy grew is not held against the model (it only
// removes energy).
template <class CT>
__global__ __launch_bounds__(256) void od_budget_kernel(const float* __restrict__ feat, const float* __restrict__ eps,
                                                        const float* __restrict__ oor, int64_t n,
                                                        const double* __restrict__ dt, double interval, double kappa,
                                                        double* __restrict__ st, CT* __restrict__ mu_t) {
    __shared__ double ra[256], rb[256], rc[256];
    __shared__ int off;
    double sa = 0.0, sb = 0.0, sc = 0.0;
#pragma unroll 4
    for (int64_t q = threadIdx.x; q < n; q += 256) {
        sa += (double)feat[q * FS + 14];
        sb += (double)eps[q];
        sc += (double)oor[q];
    }
    ra[threadIdx.x] = sa;
    rb[threadIdx.x] = sb;
    rc[threadIdx.x] = sc;
    __syncthreads();
    for (int h = 128; h >= 1; h >>= 1) {
        if ((int)threadIdx.x < h) {
            ra[threadIdx.x] += ra[threadIdx.x + h];
            rb[threadIdx.x] += rb[threadIdx.x + h];
            rc[threadIdx.x] += rc[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double ke = ra[0], eps_now = rb[0];
        bool active = true;
        if (kappa > 0.0 && st[kKePrev] >= 0.0 && st[kActive] != 0.0) {
            const double dke = st[kKePrev] - ke;                    // observed decay
            const double work = st[kEpsPrev] * (*dt * interval);    // energy the model removed
            if (dke > 0.0 && work > kappa * dke) active = false;
        }
        off = !active;
        st[kKePrev] = ke;
        st[kEpsPrev] = active ? eps_now : 0.0;
        st[kActive] = active ? 1.0 : 0.0;
        st[kStats + 0] += 1.0;
        if (!active) st[kStats + 1] += 1.0;
        st[kStats + 2] += rc[0];
        st[kStats + 3] = ke;
        st[kStats + 4] = eps_now;
        st[kStats + 5] = active ? 1.0 : 0.0;
    }
    __syncthreads();
    if (off)
        for (int64_t q = threadIdx.x; q < n; q += 256) mu_t[q] = (CT)0;
}

template <class CT>
__global__ void od_fill_kernel(CT* p, int64_t n) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = (CT)0;
}

int check() { return hipGetLastError() == hipSuccess ? 0 : 1; }

}  // namespace

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
struct od_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    float* params = nullptr;  // f32 master
    float* adam_m = nullptr;
    float* adam_v = nullptr;
    float* grad = nullptr;    // NPARAM + 1
    unsigned short* wb = nullptr;  // bf16 copies: w1 | w2 | w3 | w2t | w3t | w4
    Scaling sc{};
    std::mutex uses_mu;
    std::vector<std::shared_ptr<od::UseEvent>> uses;  // of the solvers the network was attached to
    float* partial = nullptr;  // partial gradient rows of the largest batch so far (at most 1024)
    size_t partial_rows = 0;
    uint64_t adam_t = 0;
};

namespace {

DevNet dev_net(const od_mlp* m) {
    DevNet n;
    n.w1 = m->wb;
    n.w2 = m->wb + NH * KP;
    n.w3 = n.w2 + NH * NH;
    n.w2t = n.w3 + NH * NH;
    n.w3t = n.w2t + NH * NH;
    n.w4 = n.w3t + NH * NH;
    n.params = m->params;
    return n;
}

int cast_weights(od_mlp* m) {
    hipLaunchKernelGGL(od_mlp_cast_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, m->stream, dev_net(m));
    return check();
}

struct DevBuf {  // scoped device allocation
    void* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
};

// One epoch of a training run in flight (od_mlp_train).
struct EpochSlot {
    int *idx = nullptr, *host_idx = nullptr;      // sample order
    float *sse = nullptr, *host_sse = nullptr;    // sum of squared errors per batch
    hipEvent_t done = nullptr;
    uint32_t epoch = 0;
    bool busy = false;
};

// What a training run holds on the device (samples, targets, and the order and
// losses of the epochs in flight) and on the host (order and losses), one
// allocation each: with one for every array, two of everything and all host
// memory pinned, a call of one epoch of 64 samples took 210 us, now 57, five
// epochs of 1000 samples 650, now 490.  Without room for a second epoch in flight,
// or without pinned memory, a run goes on with one and with pageable memory.
struct TrainScratch {
    float *x = nullptr, *t = nullptr;
    EpochSlot slot[2];
    int slots = 0;
    TrainScratch() = default;
    TrainScratch(const TrainScratch&) = delete;
    TrainScratch& operator=(const TrainScratch&) = delete;
    ~TrainScratch() { release(); }
    od_status allocate(size_t n, size_t n_batches, int want) {
        const size_t per_slot = n + n_batches;  // values of 4 bytes
        for (slots = want; slots > 0; --slots) {
            if (hipMalloc((void**)&x, (n * (NF + 1) + slots * per_slot) * 4) == hipSuccess && host_block(slots * per_slot * 4))
                break;
            (void)hipGetLastError();
            release();
        }
        if (!slots) return fail(OD_ERR_HIP, "od_mlp_train: allocation failed");
        t = x + n * NF;
        for (int q = 0; q < slots; ++q) {
            slot[q].idx = (int*)(t + n) + q * per_slot;
            slot[q].sse = (float*)(slot[q].idx + n);
            slot[q].host_idx = (int*)host + q * per_slot;
            slot[q].host_sse = (float*)(slot[q].host_idx + n);
            HIP_TRY(hipEventCreateWithFlags(&slot[q].done, hipEventDisableTiming));
        }
        return OD_OK;
    }

   private:
    void* host = nullptr;
    bool pinned = false;
    bool host_block(size_t bytes) {
        // one epoch at a time: no copy runs beside the host's work
        pinned = slots > 1 && hipHostMalloc(&host, bytes, hipHostMallocDefault) == hipSuccess;
        if (!pinned) {
            (void)hipGetLastError();
            host = slots > 1 ? nullptr : std::malloc(bytes);
        }
        return host != nullptr;
    }
    void release() {
        if (x) (void)hipFree(x);  // waits for the device
        if (host && pinned) (void)hipHostFree(host);
        if (host && !pinned) std::free(host);
        for (EpochSlot& q : slot)
            if (q.done) (void)hipEventDestroy(q.done);
        x = t = nullptr;
        host = nullptr;
        pinned = false;
    }
};

// Gradient of the mean squared error over n gathered samples; grad and the
// sum of squared errors in m->grad (device).  With `adam` the parameters take
// their step in the same launch as the sum over the groups.
od_status run_grad(od_mlp* m, const float* dx, const float* dt, const int* didx, int64_t n, const Adam* adam) {
    const int64_t tiles = (n + 15) / 16;
    const int tpg = (int)std::max<int64_t>(1, (tiles + 1023) / 1024);
    const int64_t groups = (tiles + tpg - 1) / tpg;
    if ((size_t)groups > m->partial_rows) {
        HIP_TRY(hipStreamSynchronize(m->stream));  // no batch still reads the smaller array
        if (m->partial) (void)hipFree(m->partial);
        m->partial = nullptr;
        m->partial_rows = 0;
        HIP_TRY(hipMalloc((void**)&m->partial, (size_t)groups * kPartialRow * sizeof(float)));
        m->partial_rows = (size_t)groups;
    }
    hipLaunchKernelGGL(od_mlp_grad_kernel, dim3((unsigned)groups), dim3(256), 0, m->stream, dev_net(m), m->sc, dx, dt,
                       didx, n, tpg, m->partial);
    if (check()) return fail(OD_ERR_HIP, "od_mlp_grad_kernel launch failed");
    if (adam)
        hipLaunchKernelGGL(od_mlp_reduce_kernel<true>, dim3(kPartialRow / 32), dim3(256), 0, m->stream, m->partial,
                           (int)groups, m->grad, *adam, dev_net(m));
    else
        hipLaunchKernelGGL(od_mlp_reduce_kernel<false>, dim3(kPartialRow / 32), dim3(256), 0, m->stream, m->partial,
                           (int)groups, m->grad, Adam{}, dev_net(m));
    if (check()) return fail(OD_ERR_HIP, "od_mlp_reduce_kernel launch failed");
    return OD_OK;
}

// Host f64 FR operators for the feature kernel.
FeatConsts feat_consts(const od_ctx* c) {
    FeatConsts f{};
    const HostOps& o = c->ops;
    for (int q = 0; q < 16; ++q) f.D[q] = (float)o.D[q];
    for (int a = 0; a < 4; ++a) {
        for (int i = 0; i < 4; ++i) {
            // Legendre P_a at x_i
            const double x = o.x[i];
            double p0 = 1.0, p1 = x, pa = a == 0 ? 1.0 : x;
            for (int kk = 2; kk <= a; ++kk) {
                const double p2 = ((2.0 * kk - 1.0) * x * p1 - (kk - 1.0) * p0) / kk;
                p0 = p1;
                p1 = p2;
                pa = p2;
            }
            f.L[a * 4 + i] = (float)((2.0 * a + 1.0) / 2.0 * o.w[i] * pa);
        }
        f.w[a] = (float)o.w[a];
        f.nrm[a] = (float)(2.0 / (2.0 * a + 1.0));
    }
    const double hx = c->p.lx / c->p.nx, hy = c->p.ly / c->p.ny, hz = c->p.lz / c->p.nz;
    f.jx = (float)(2.0 / hx);
    f.jy = (float)(2.0 / hy);
    f.jz = (float)(2.0 / hz);
    f.vol8 = (float)(hx * hy * hz / 8.0);
    f.delta = (float)(std::cbrt(hx * hy * hz) / 4.0);
    f.mu_mol = (float)(c->p.mu_ref > 0 ? c->p.mu_ref : 1e-30);
    return f;
}

od_status ensure_closure_buffers(od_ctx* c) {
    if (!c->feat) {
        if (hipMalloc(&c->feat, (size_t)c->E * (FS + 2) * sizeof(float)) != hipSuccess)
            return fail(OD_ERR_NOMEM, "closure buffers: allocation failed");
        c->device_bytes += (size_t)c->E * (FS + 2) * sizeof(float);
    }
    if (!c->budget) {
        const double zero[kBudget] = {};
        HIP_TRY(hipMalloc((void**)&c->budget, sizeof(zero)));
        HIP_TRY(hipMemcpy(c->budget, zero, sizeof(zero), hipMemcpyHostToDevice));
    }
    return OD_OK;
}

od_status ensure_mu_t(od_ctx* c) {
    if (c->mu_t) return OD_OK;
    if (hipMalloc(&c->mu_t, (size_t)c->E * c->cbytes) != hipSuccess)
        return fail(OD_ERR_NOMEM, "eddy viscosity buffer: allocation failed");
    c->device_bytes += (size_t)c->E * c->cbytes;
    const unsigned blocks = (unsigned)((c->E + 255) / 256);
    if (c->cbytes == 4)
        hipLaunchKernelGGL(od_fill_kernel<float>, dim3(blocks), dim3(256), 0, c->stream, (float*)c->mu_t, c->E);
    else
        hipLaunchKernelGGL(od_fill_kernel<double>, dim3(blocks), dim3(256), 0, c->stream, (double*)c->mu_t, c->E);
    return check() ? fail(OD_ERR_HIP, "fill kernel launch failed") : OD_OK;
}

int launch_features(od_ctx* c) {
    const FeatConsts fc = feat_consts(c);
    const unsigned blocks = (unsigned)((c->E + 3) / 4);
    if (c->p.u_real == OD_F32)
        hipLaunchKernelGGL(od_features_kernel<float>, dim3(blocks), dim3(256), 0, c->stream, (const float*)c->u[0],
                           c->E, fc, (float*)c->feat);
    else
        hipLaunchKernelGGL(od_features_kernel<double>, dim3(blocks), dim3(256), 0, c->stream,
                           (const double*)c->u[0], c->E, fc, (float*)c->feat);
    return check();
}

}  // namespace

namespace {

// Everything a refresh is launched with that can change between two refreshes
// of one attachment, as bytes.
struct RefreshKey {
    DevNet net;
    Scaling sc;
    int32_t interval;
    double kappa;
};
static_assert(sizeof(RefreshKey) <= sizeof(od_ctx::closure_key), "room for the key");
void refresh_key(const od_ctx* c, unsigned char* bytes) {
    const DevNet net = dev_net(c->mlp);
    std::memset(bytes, 0, sizeof(RefreshKey));  // padding too
    std::memcpy(bytes + offsetof(RefreshKey, net), &net, sizeof(net));
    std::memcpy(bytes + offsetof(RefreshKey, sc), &c->mlp->sc, sizeof(Scaling));
    std::memcpy(bytes + offsetof(RefreshKey, interval), &c->closure.update_interval, sizeof(int32_t));
    std::memcpy(bytes + offsetof(RefreshKey, kappa), &c->closure.budget_kappa, sizeof(double));
}

template <class CT>
od_status enqueue_refresh(od_ctx* c) {
    if (launch_features(c)) return fail(OD_ERR_HIP, "od_features_kernel launch failed");
    const float* feat = (const float*)c->feat;
    float* eps = (float*)c->feat + (size_t)c->E * FS;
    float* oor = eps + c->E;
    const unsigned blocks = (unsigned)std::min<int64_t>(2048, (c->E + 15) / 16);  // up to 8 groups a CU
    hipLaunchKernelGGL(od_mlp_infer_kernel<CT>, dim3(blocks), dim3(256), 0, c->stream, dev_net(c->mlp), c->mlp->sc, feat,
                       c->E, (CT*)c->mu_t, eps, oor);
    if (check()) return fail(OD_ERR_HIP, "od_mlp_infer_kernel launch failed");
    hipLaunchKernelGGL(od_budget_kernel<CT>, dim3(1), dim3(256), 0, c->stream, feat, eps, oor, c->E, c->dt_value,
                       (double)c->closure.update_interval, c->closure.budget_kappa, c->budget, (CT*)c->mu_t);
    return check() ? fail(OD_ERR_HIP, "od_budget_kernel launch failed") : OD_OK;
}

// Drops the uses of solvers that are gone or attached anew (both wait for
// their streams).
void prune_uses(od_mlp* m) {
    m->uses.erase(std::remove_if(m->uses.begin(), m->uses.end(), [](const auto& u) { return u.use_count() == 1; }),
                  m->uses.end());
}

// Waits for the refreshes that still read the network's weights.
void wait_for_uses(od_mlp* m) {
    std::lock_guard<std::mutex> lk(m->uses_mu);
    for (const auto& u : m->uses) (void)hipEventSynchronize(u->ev);
    prune_uses(m);
}

}  // namespace

// Enqueues a refresh of mu_t from the current state (od_step, every
// update_interval steps while a network is attached).
od_status od_closure_refresh_internal(od_ctx* c) {
    return c->cbytes == 4 ? enqueue_refresh<float>(c) : enqueue_refresh<double>(c);
}

bool od_closure_key_changed_internal(od_ctx* c) {
    unsigned char key[sizeof(RefreshKey)];
    refresh_key(c, key);
    if (std::memcmp(key, c->closure_key, sizeof(key)) == 0) return false;
    std::memcpy(c->closure_key, key, sizeof(key));
    return true;
}

od_status od_closure_used_internal(od_ctx* c) {
    HIP_TRY(hipEventRecord(c->mlp_use->ev, c->stream));
    return OD_OK;
}

void od_closure_release_internal(od_ctx* c) {
    if (c->feat) (void)hipFree(c->feat);
    if (c->budget) (void)hipFree(c->budget);
    if (c->mu_t) (void)hipFree(c->mu_t);
    c->feat = nullptr;
    c->budget = nullptr;
    c->mu_t = nullptr;
    c->mlp_use.reset();
}

extern "C" {

od_status od_mlp_create(int device, od_mlp** out) {
    if (!out) return fail(OD_ERR_INVALID, "od_mlp_create: null argument");
    *out = nullptr;
    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return fail(OD_ERR_INVALID, "no such HIP device");
    HIP_TRY(hipSetDevice(device));
    od_mlp* m = new od_mlp();
    m->device = device;
    auto bad = [&](const char* what) {
        od_mlp_destroy(m);
        return fail(OD_ERR_NOMEM, what);
    };
    if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) return bad("stream creation failed");
    if (hipMalloc((void**)&m->params, NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc((void**)&m->adam_m, NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc((void**)&m->adam_v, NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc((void**)&m->grad, (NPARAM + 1) * sizeof(float)) != hipSuccess ||
        hipMalloc((void**)&m->wb, kNetShorts * sizeof(unsigned short)) != hipSuccess)
        return bad("device allocation failed");
    // Default: Glorot-uniform weights, zero biases (seed 0); identity scaling, open range.
    std::vector<float> p(NPARAM, 0.0f);
    std::mt19937_64 rng(0);
    auto fill = [&](int off, int fan_out, int fan_in) {
        const double a = std::sqrt(6.0 / (fan_in + fan_out));
        std::uniform_real_distribution<double> U(-a, a);
        for (int q = 0; q < fan_out * fan_in; ++q) p[off + q] = (float)U(rng);
    };
    fill(oW1, NH, NF);
    fill(oW2, NH, NH);
    fill(oW3, NH, NH);
    fill(oW4, 1, NH);
    for (int q = 0; q < NF; ++q) {
        m->sc.shift[q] = 0.0f;
        m->sc.scale[q] = 1.0f;
        m->sc.lo[q] = -INFINITY;
        m->sc.hi[q] = INFINITY;
    }
    m->sc.out_scale = 1.0f;
    od_status s = od_mlp_set_params(m, p.data(), p.size());
    if (s != OD_OK) {
        od_mlp_destroy(m);
        return s;
    }
    *out = m;
    return OD_OK;
}

void od_mlp_destroy(od_mlp* m) {
    if (!m) return;
    (void)hipSetDevice(m->device);
    wait_for_uses(m);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (void* q : {(void*)m->params, (void*)m->adam_m, (void*)m->adam_v, (void*)m->grad, (void*)m->wb,
                    (void*)m->partial})
        if (q) (void)hipFree(q);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

od_status od_mlp_set_params(od_mlp* m, const float* params, size_t n) {
    if (!m || !params) return fail(OD_ERR_INVALID, "od_mlp_set_params: null argument");
    if (n != (size_t)NPARAM) return fail(OD_ERR_INVALID, "od_mlp_set_params: expected OD_MLP_PARAMS values");
    HIP_TRY(hipSetDevice(m->device));
    wait_for_uses(m);
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(m->params, params, NPARAM * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemsetAsync(m->adam_m, 0, NPARAM * sizeof(float), m->stream));
    HIP_TRY(hipMemsetAsync(m->adam_v, 0, NPARAM * sizeof(float), m->stream));
    m->adam_t = 0;
    if (cast_weights(m)) return fail(OD_ERR_HIP, "od_mlp_cast_kernel launch failed");
    HIP_TRY(hipStreamSynchronize(m->stream));
    return OD_OK;
}

od_status od_mlp_get_params(od_mlp* m, float* params, size_t n) {
    if (!m || !params) return fail(OD_ERR_INVALID, "od_mlp_get_params: null argument");
    if (n != (size_t)NPARAM) return fail(OD_ERR_INVALID, "od_mlp_get_params: expected OD_MLP_PARAMS values");
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(hipMemcpy(params, m->params, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
    return OD_OK;
}

od_status od_mlp_set_scaling(od_mlp* m, const float shift[12], const float scale[12], const float lo[12],
                             const float hi[12]) {
    if (!m || !shift || !scale || !lo || !hi) return fail(OD_ERR_INVALID, "od_mlp_set_scaling: null argument");
    for (int q = 0; q < NF; ++q) {
        if (!(lo[q] <= hi[q])) return fail(OD_ERR_INVALID, "od_mlp_set_scaling: lo must be <= hi");
        m->sc.shift[q] = shift[q];
        m->sc.scale[q] = scale[q];
        m->sc.lo[q] = lo[q];
        m->sc.hi[q] = hi[q];
    }
    return OD_OK;
}

od_status od_mlp_set_output_scale(od_mlp* m, float s) {
    if (!m) return fail(OD_ERR_INVALID, "od_mlp_set_output_scale: null argument");
    if (!(s > 0.0f) || !std::isfinite(s)) return fail(OD_ERR_INVALID, "od_mlp_set_output_scale: scale must be positive");
    m->sc.out_scale = s;
    return OD_OK;
}

od_status od_mlp_forward(od_mlp* m, const float* x, size_t n, float* y) {
    if (!m || !x || !y) return fail(OD_ERR_INVALID, "od_mlp_forward: null argument");
    if (n == 0) return OD_OK;
    HIP_TRY(hipSetDevice(m->device));
    DevBuf dx, dy;
    HIP_TRY(hipMalloc(&dx.p, n * NF * sizeof(float)));
    HIP_TRY(hipMalloc(&dy.p, n * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(dx.p, x, n * NF * sizeof(float), hipMemcpyHostToDevice, m->stream));
    const unsigned blocks = (unsigned)std::min<size_t>(2048, (n + 15) / 16);
    hipLaunchKernelGGL(od_mlp_forward_kernel, dim3(blocks), dim3(256), 0, m->stream, dev_net(m), m->sc,
                       (const float*)dx.p, (int64_t)n, (float*)dy.p);
    if (check()) return fail(OD_ERR_HIP, "od_mlp_forward_kernel launch failed");
    HIP_TRY(hipMemcpyAsync(y, dy.p, n * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    HIP_TRY(hipStreamSynchronize(m->stream));
    return OD_OK;
}

od_status od_mlp_loss_grad(od_mlp* m, const float* x, const float* t, size_t n, double* loss, float* grad) {
    if (!m || !x || !t) return fail(OD_ERR_INVALID, "od_mlp_loss_grad: null argument");
    if (n == 0) return fail(OD_ERR_INVALID, "od_mlp_loss_grad: empty batch");
    HIP_TRY(hipSetDevice(m->device));
    DevBuf dx, dt;
    HIP_TRY(hipMalloc(&dx.p, n * NF * sizeof(float)));
    HIP_TRY(hipMalloc(&dt.p, n * sizeof(float)));
    HIP_TRY(hipMemcpyAsync(dx.p, x, n * NF * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIP_TRY(hipMemcpyAsync(dt.p, t, n * sizeof(float), hipMemcpyHostToDevice, m->stream));
    od_status s = run_grad(m, (const float*)dx.p, (const float*)dt.p, nullptr, (int64_t)n, nullptr);
    std::vector<float> g(NPARAM + 1);
    if (s == OD_OK && hipMemcpyAsync(g.data(), m->grad, (NPARAM + 1) * sizeof(float), hipMemcpyDeviceToHost,
                                     m->stream) != hipSuccess)
        s = fail(OD_ERR_HIP, "od_mlp_loss_grad: copy failed");
    (void)hipStreamSynchronize(m->stream);
    if (s != OD_OK) return s;
    if (loss) *loss = (double)g[NPARAM] / (double)n;
    if (grad) std::memcpy(grad, g.data(), NPARAM * sizeof(float));
    return OD_OK;
}

od_status od_mlp_train(od_mlp* m, const float* x, const float* t, size_t n, uint32_t epochs, uint32_t batch,
                       float lr, uint64_t seed, float* loss_per_epoch) {
    if (!m || !x || !t) return fail(OD_ERR_INVALID, "od_mlp_train: null argument");
    if (n == 0 || batch == 0) return fail(OD_ERR_INVALID, "od_mlp_train: empty data or batch");
    if (n > (size_t)0x7fffffff) return fail(OD_ERR_INVALID, "od_mlp_train: too many samples");
    HIP_TRY(hipSetDevice(m->device));
    wait_for_uses(m);
    // Two epochs are in flight: while the device works through one, the host
    // orders the next one's samples.  Each slot has its index array, the sums of
    // squared errors of its batches and an event at the end of its work.
    const size_t n_batches = (n + batch - 1) / batch;
    TrainScratch scratch;
    od_status s = scratch.allocate(n, n_batches, epochs > 1 ? 2 : 1);
    if (s != OD_OK) return s;
    const float *dx = scratch.x, *dt = scratch.t;
    HIP_TRY(hipMemcpyAsync(scratch.x, x, n * NF * sizeof(float), hipMemcpyHostToDevice, m->stream));
    HIP_TRY(hipMemcpyAsync(scratch.t, t, n * sizeof(float), hipMemcpyHostToDevice, m->stream));
    od::SampleOrder order(n, seed, epochs > 1);
    // waits for the epoch in slot q and takes its loss
    auto finish = [&](EpochSlot& q) -> od_status {
        if (!q.busy) return OD_OK;
        q.busy = false;
        HIP_TRY(hipEventSynchronize(q.done));
        double sse = 0.0;
        for (size_t k = 0; k < n_batches; ++k) sse += q.host_sse[k];
        if (loss_per_epoch) loss_per_epoch[q.epoch] = (float)(sse / (double)n);
        return OD_OK;
    };
    auto run_epoch = [&](EpochSlot& q, uint32_t ep) -> od_status {
        od_status s = finish(q);
        if (s != OD_OK) return s;
        order.next(q.host_idx);
        HIP_TRY(hipMemcpyAsync(q.idx, q.host_idx, n * sizeof(int), hipMemcpyHostToDevice, m->stream));
        for (size_t b0 = 0, k = 0; b0 < n; b0 += batch, ++k) {
            const uint64_t at = m->adam_t + 1;
            const Adam ad{m->params,
                          m->adam_m,
                          m->adam_v,
                          lr,
                          (float)std::pow(0.9, (double)at),
                          (float)std::pow(0.999, (double)at),
                          q.sse + k};
            s = run_grad(m, dx, dt, q.idx + b0, (int64_t)std::min<size_t>(batch, n - b0), &ad);
            if (s != OD_OK) return s;
            m->adam_t = at;
        }
        HIP_TRY(hipMemcpyAsync(q.host_sse, q.sse, n_batches * sizeof(float), hipMemcpyDeviceToHost, m->stream));
        HIP_TRY(hipEventRecord(q.done, m->stream));
        q.epoch = ep;
        q.busy = true;
        return OD_OK;
    };
    const uint32_t slots = (uint32_t)scratch.slots;
    for (uint32_t ep = 0; ep < epochs && s == OD_OK; ++ep) s = run_epoch(scratch.slot[ep % slots], ep);
    for (uint32_t k = 0; k < slots && s == OD_OK; ++k) s = finish(scratch.slot[(epochs + k) % slots]);
    (void)hipStreamSynchronize(m->stream);
    return s;
}

od_status od_closure_features(od_ctx* c, float* out, size_t n) {
    if (!c || !out) return fail(OD_ERR_INVALID, "od_closure_features: null argument");
    if (n != (size_t)c->E * FS) return fail(OD_ERR_INVALID, "od_closure_features: expected E * 16 values");
    if (!c->state_set) return fail(OD_ERR_STATE, "od_closure_features: state not set");
    HIP_TRY(hipSetDevice(c->device));
    od_status s = ensure_closure_buffers(c);
    if (s != OD_OK) return s;
    if (launch_features(c)) return fail(OD_ERR_HIP, "od_features_kernel launch failed");
    HIP_TRY(hipMemcpyAsync(out, c->feat, n * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return OD_OK;
}

od_status od_set_eddy_viscosity(od_ctx* c, const void* host, size_t n, od_real dtype) {
    if (!c) return fail(OD_ERR_INVALID, "od_set_eddy_viscosity: null context");
    if (c->mlp) return fail(OD_ERR_STATE, "od_set_eddy_viscosity: a network is attached");
    HIP_TRY(hipSetDevice(c->device));
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (!host) {
        c->mu_t_on = false;
        return OD_OK;
    }
    if (n != (size_t)c->E) return fail(OD_ERR_INVALID, "od_set_eddy_viscosity: expected E values");
    if (!real_ok(dtype)) return fail(OD_ERR_INVALID, "od_set_eddy_viscosity: bad dtype");
    if (!c->p.viscous) return fail(OD_ERR_STATE, "od_set_eddy_viscosity: Euler mode has no viscous fluxes");
    od_status s = ensure_mu_t(c);
    if (s != OD_OK) return s;
    std::vector<unsigned char> tmp(n * c->cbytes);
    if (c->cbytes == 4) {
        if (dtype == OD_F32)
            std::memcpy(tmp.data(), host, n * 4);
        else
            convert((float*)tmp.data(), (const double*)host, n);
    } else {
        if (dtype == OD_F64)
            std::memcpy(tmp.data(), host, n * 8);
        else
            convert((double*)tmp.data(), (const float*)host, n);
    }
    HIP_TRY(hipMemcpy(c->mu_t, tmp.data(), n * c->cbytes, hipMemcpyHostToDevice));
    c->mu_t_on = true;
    return OD_OK;
}

od_status od_get_eddy_viscosity(od_ctx* c, void* host, size_t n, od_real dtype) {
    if (!c || !host) return fail(OD_ERR_INVALID, "od_get_eddy_viscosity: null argument");
    if (n != (size_t)c->E) return fail(OD_ERR_INVALID, "od_get_eddy_viscosity: expected E values");
    if (!real_ok(dtype)) return fail(OD_ERR_INVALID, "od_get_eddy_viscosity: bad dtype");
    HIP_TRY(hipSetDevice(c->device));
    std::vector<unsigned char> tmp(n * c->cbytes, 0);
    if (c->mu_t) {
        HIP_TRY(hipStreamSynchronize(c->stream));
        HIP_TRY(hipMemcpy(tmp.data(), c->mu_t, n * c->cbytes, hipMemcpyDeviceToHost));
    }
    if ((size_t)dtype == c->cbytes)
        std::memcpy(host, tmp.data(), n * c->cbytes);
    else if (c->cbytes == 4)
        convert((double*)host, (const float*)tmp.data(), n);
    else
        convert((float*)host, (const double*)tmp.data(), n);
    return OD_OK;
}

od_status od_closure_attach(od_ctx* c, od_mlp* m, const od_closure_opts* opts) {
    if (!c) return fail(OD_ERR_INVALID, "od_closure_attach: null context");
    HIP_TRY(hipSetDevice(c->device));
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (!m) {
        c->mlp = nullptr;
        c->mu_t_on = false;
        return OD_OK;
    }
    if (!opts || opts->update_interval < 1) return fail(OD_ERR_INVALID, "od_closure_attach: update_interval >= 1");
    if (!c->p.viscous) return fail(OD_ERR_STATE, "od_closure_attach: Euler mode has no viscous fluxes");
    if (m->device != c->device) return fail(OD_ERR_INVALID, "od_closure_attach: network on another device");
    HIP_TRY(hipStreamSynchronize(m->stream));
    od_status s = ensure_closure_buffers(c);
    if (s == OD_OK) s = ensure_mu_t(c);
    if (s != OD_OK) return s;
    // a fresh budget: no previous energy, nothing removed, active
    double st[kBudget] = {};
    st[kKePrev] = -1.0;
    st[kActive] = 1.0;
    HIP_TRY(hipMemcpy(c->budget, st, sizeof(st), hipMemcpyHostToDevice));
    auto use = std::make_shared<od::UseEvent>();
    HIP_TRY(hipEventCreateWithFlags(&use->ev, hipEventDisableTiming));
    {
        std::lock_guard<std::mutex> lk(m->uses_mu);
        prune_uses(m);
        m->uses.push_back(use);
    }
    c->mlp_use = use;
    c->mlp = m;
    c->closure = *opts;
    c->steps_done = 0;
    c->mu_t_on = true;
    return OD_OK;
}

od_status od_closure_stats(od_ctx* c, double out[6]) {
    if (!c || !out) return fail(OD_ERR_INVALID, "od_closure_stats: null argument");
    for (int q = 0; q < 6; ++q) out[q] = 0.0;
    if (!c->budget) return OD_OK;
    HIP_TRY(hipSetDevice(c->device));
    HIP_TRY(hipStreamSynchronize(c->stream));
    HIP_TRY(hipMemcpy(out, c->budget + kStats, 6 * sizeof(double), hipMemcpyDeviceToHost));
    return OD_OK;
}

}  // extern "C"
