// Surrogate network of the delayed-acceptance rotor move, and its training kernels.
//
// Network: 4 inputs -> 128 -> 128 -> 128 -> 1, SiLU after each hidden layer.  Inputs are the
// atom-rotor pair geometry in the rotor's body frame (R, ux, uy, uz) normalised by the training
// set's mean and spread; the output, scaled back, is the pair energy in Kelvin.
//
// Master weights are FP32 in one flat vector `theta` (MLP_NW floats, layout MLP_OFF_*); the
// gradient has the same layout.  Training runs on the matrix cores (v_mfma_f32_32x32x8bf16_1k: BF16
// operands, FP32 accumulation), one kernel for the rows and one for the weights; the sampler reads
// a packed copy (MlpPacked: BF16 matrices in the lane order of the matrix instructions, FP32
// biases), staged in LDS by the kernels that use it.
//
// Inference layout.  One wave evaluates 32 rows as H^T = W X^T, hidden units on the MFMA's M
// axis and rows on its N axis.  D layout of the 32x32 MFMAs: element i of lane l is
// D[8*(i/4)+4*(l/32)+i%4][l%32].  Layer 1 (K = 4, padded to 8) uses the 32x32x8 MFMA
// (A: lane l holds A[l%32][4*(l/32)+j], j < 4; B: B[4*(l/32)+j][l%32]).  The 128 -> 128 layers
// use gfx950's 32x32x16 MFMA (A: A[l%32][8*(l/32)+j], j < 8; B: B[8*(l/32)+j][l%32]) with the
// contraction index permuted: k-block kb takes, on lane l, elements 8*(kb%2)..8*(kb%2)+7 of the
// previous layer's output tile kb/2, i.e. hidden units 16*kb + 8*(j/4) + 4*(l/32) + j%4.  The
// packed weights follow the same permutation, so activations stay in registers from layer to
// layer and every A operand is one 16-byte LDS read.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "pimc_device.hpp"

constexpr int MLP_IN = 4;
constexpr int MLP_H = 128;
constexpr int MLP_OFF_W1 = 0;                                // [128][4]
constexpr int MLP_OFF_B1 = MLP_OFF_W1 + MLP_H * MLP_IN;      // [128]
constexpr int MLP_OFF_W2 = MLP_OFF_B1 + MLP_H;               // [128][128] (out, in)
constexpr int MLP_OFF_B2 = MLP_OFF_W2 + MLP_H * MLP_H;
constexpr int MLP_OFF_W3 = MLP_OFF_B2 + MLP_H;               // [128][128]
constexpr int MLP_OFF_B3 = MLP_OFF_W3 + MLP_H * MLP_H;
constexpr int MLP_OFF_W4 = MLP_OFF_B3 + MLP_H;               // [128]
constexpr int MLP_OFF_B4 = MLP_OFF_W4 + MLP_H;               // [1]
constexpr int MLP_NW = MLP_OFF_B4 + 1;                       // 33793
// FLOP of one evaluation: 2*(4*128 + 128*128 + 128*128 + 128)
constexpr double MLP_FLOP = 2.0 * (MLP_IN * MLP_H + 2 * MLP_H * MLP_H + MLP_H);

struct alignas(16) MlpPacked {
    uint16_t w1[4 * 64 * 4];      // layer 1 A operands [tile][lane][4] (inputs 4..7 zero)
    uint16_t w2[4 * 8 * 64 * 8];  // layer 2 A operands [tile][k-block][lane][8], permuted k
    uint16_t w3[4 * 8 * 64 * 8];
    float b1[MLP_H], b2[MLP_H], b3[MLP_H], w4[MLP_H];
    float b4;
    float xm[MLP_IN], xinv[MLP_IN];  // normalised input = (x - xm) * xinv
    float ym, ys;                    // energy = ys * output + ym
};
static_assert(sizeof(MlpPacked) % 16 == 0, "staged with 16-byte copies");

typedef short mlp_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 mlp_bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short mlp_u16x8 __attribute__((ext_vector_type(8)));
typedef float mlp_f32x16 __attribute__((ext_vector_type(16)));

__host__ __device__ inline uint16_t f2bf(float x) {  // round to nearest even
    union { float f; uint32_t u; } c;
    c.f = x;
    uint32_t u = c.u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// SiLU z * sigmoid(z) from the hardware exponential and reciprocal (v_exp_f32, v_rcp_f32): the
// activation is the bulk of the vector work per row, and BF16 operands bound the accuracy anyway.
__device__ __forceinline__ float mlp_sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ __forceinline__ float mlp_silu(float z) { return z * mlp_sigmoid(z); }

__device__ __forceinline__ mlp_f32x16 mlp_mfma(mlp_bf16x4 a, mlp_bf16x4 b, mlp_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ mlp_f32x16 mlp_mfma16(mlp_bf16x8 a, mlp_bf16x8 b, mlp_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// unit of the output element i of lane half hi in tile mb
__device__ __forceinline__ int mlp_unit(int mb, int i, int hi) { return mb * 32 + 8 * (i >> 2) + 4 * hi + (i & 3); }

__device__ __forceinline__ mlp_bf16x4 mlp_load4(const uint16_t* p) {  // 4 BF16, 8-byte aligned
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    mlp_bf16x4 r;
    r[0] = (short)(v.x & 0xffffu);
    r[1] = (short)(v.x >> 16);
    r[2] = (short)(v.y & 0xffffu);
    r[3] = (short)(v.y >> 16);
    return r;
}

// One hidden 128 -> 128 layer on D-layout activations h (in place): bias and SiLU applied.  Operands
// are rounded by integer operations: with the pair conversion instruction a delayed-acceptance pass
// took 10 to 20 percent longer (200 passes of one top 2.05 against 1.85 s, waters 11.4 against 9.5).
// w: the layer's packed A operands (in LDS).
__device__ __forceinline__ void mlp_hidden(const uint16_t* __restrict__ w, const float* __restrict__ b,
                                           mlp_f32x16 h[4], int l) {
    const int hi = l >> 5;
    mlp_bf16x8 bin[8];
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
        mlp_u16x8 t;
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = f2bf(h[kb >> 1][8 * (kb & 1) + j]);
        bin[kb] = __builtin_bit_cast(mlp_bf16x8, t);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
        mlp_f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 8; ++kb) {
            const uint4 a = *reinterpret_cast<const uint4*>(w + (((mb * 8 + kb) * 64 + l) << 3));
            acc = mlp_mfma16(__builtin_bit_cast(mlp_bf16x8, a), bin[kb], acc);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = mlp_silu(acc[i] + b[mlp_unit(mb, i, hi)]);
        h[mb] = acc;
    }
}

// The whole wave evaluates 32 rows.  Lane l < 32 passes the normalised inputs of row l in
// f[0..3] (lanes 32..63 pass anything).  Every lane returns the raw network output of row l%32.
// W: the packed network staged in LDS.
__device__ __forceinline__ float mlp_rows32(const MlpPacked* __restrict__ W, const float f[MLP_IN]) {
    const int l = threadIdx.x & 63, hi = l >> 5;
    mlp_bf16x4 bx;
#pragma unroll
    for (int j = 0; j < 4; ++j) bx[j] = hi ? (short)0 : (short)f2bf(f[j]);
    mlp_f32x16 h[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
        mlp_f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
        acc = mlp_mfma(mlp_load4(W->w1 + ((mb * 64 + l) << 2)), bx, acc);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = mlp_silu(acc[i] + W->b1[mlp_unit(mb, i, hi)]);
        h[mb] = acc;
    }
    mlp_hidden(W->w2, W->b2, h, l);
    mlp_hidden(W->w3, W->b3, h, l);
    float part = 0.0f;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 16; ++i) part += W->w4[mlp_unit(mb, i, hi)] * h[mb][i];
    part += __shfl_xor(part, 32);
    return part + W->b4;
}

// Copies the packed network into LDS (all lanes of the block take part; caller synchronises).
__device__ __forceinline__ void mlp_stage(const MlpPacked* __restrict__ g, MlpPacked* s) {
    const uint4* src = reinterpret_cast<const uint4*>(g);
    uint4* dst = reinterpret_cast<uint4*>(s);
    for (int i = threadIdx.x; i < (int)(sizeof(MlpPacked) / 16); i += blockDim.x) dst[i] = src[i];
}

// Pair geometry in the rotor's body frame: distance and the direction cosines of the partner
// on the body axes (the axes vcord reads from the rotation matrix; z is normalised by its length).
__device__ __forceinline__ void mlp_pair_features(const double m[9], double zn, double cx, double cy, double cz,
                                                  double px, double py, double pz, float out[MLP_IN]) {
    const double rx = px - cx, ry = py - cy, rz = pz - cz;
    const double rn = sqrt(rx * rx + ry * ry + rz * rz);
    const double inv = rn > 0.0 ? 1.0 / rn : 0.0;
    out[0] = (float)rn;
    out[1] = (float)((m[0] * rx + m[1] * ry + m[2] * rz) * inv);
    out[2] = (float)((m[3] * rx + m[4] * ry + m[5] * rz) * inv);
    out[3] = (float)((m[6] * rx + m[7] * ry + m[8] * rz) * inv / zn);
}

// ------------------------------------------------------------------------------ training
// A step is two launches: k_mlp_rows takes blocks of 32 rows of the batch forward and back, and
// k_mlp_grads forms the weight gradients and takes the Adam step.  All products take BF16 operands
// and FP32 sums on 32x32x8 matrix instructions, eight values of the contraction at a time in
// ascending order: training feeds a rounding of the gradient back into every later step, so the
// order of the sums is part of the result.
//
// What bounds a step is that order: a weight gradient sums over the batch, 512 dependent matrix
// instructions for 4096 rows (20 us), on 40 tiles of 32x32.  Everything else is arranged around that
// chain: activations stay in registers and LDS from the gather to dZ1, operands are written once in
// the lane order in which the chain reads them and staged ahead of it by the block's four waves,
// and the step on the weights, with their operands for the next step, is the chain's last act.
// A launch per product and per elementwise operation, a wave per tile reading FP32 operands one by
// one, took 1.56 ms a step of 4096 rows; the two kernels now take 19 and 22 us.

// Operand order of a 32x32x8 product whose contraction runs over rows: [rows / 16][tile][lane][8],
// value 4 s + j of lane l is row 8 s + 4 (l / 32) + j of the sixteen, unit l % 32 of the tile.  The
// D layout of a tile of 32 rows holds exactly these: elements 0..7, then 8..15.
struct MlpTrain {
    const float* X;         // [n][4], [n]: the normalised rows
    const float* Y;
    const int* perm;        // batch row b is row perm[b] of them
    uint16_t* ops;          // [6][pad/16][4][64][8]: H1, H2, H3, dZ1, dZ2, dZ3
    uint16_t* opx;          // [pad/16][64][8]: inputs (units 0..3)
    uint16_t* opd;          // [pad/16][64][8]: dL/dout (unit 0)
    float* dz;              // [3][pad][128]: dZ1, dZ2, dZ3 for the bias sums
    float* dout;            // [pad]
    float *th, *m, *v;      // weights and Adam's moments
    float* g;               // if not null: takes the gradient, and th, m, v stay
    uint16_t* pw;           // [4][4 tiles][8][64][8]: W2, W3 for the way forward, W2, W3 for the way back
    double* loss;           // [blocks of 32 rows]
    int B, pad;             // rows of the batch, padded to 32
};

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// forward operand of W[o][i]: lane o % 32 + 32 (i % 8 / 4) of tile o / 32, block i / 8, value i % 4
__device__ __forceinline__ int mlp_pw_fwd(int mat, int o, int i) {
    return ((((mat * 4 + (o >> 5)) * 8 + (i >> 4)) * 64 + (o & 31) + 32 * ((i >> 2) & 1)) << 3) + 4 * ((i >> 3) & 1) + (i & 3);
}
// the same of the transposed product, whose contraction runs over o
__device__ __forceinline__ int mlp_pw_back(int mat, int o, int i) { return mlp_pw_fwd(2 + mat, i, o); }

__global__ void k_mlp_train_pack(const float* __restrict__ th, uint16_t* __restrict__ pw) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= 2 * MLP_H * MLP_H) return;
    const int mat = e / (MLP_H * MLP_H), o = e / MLP_H % MLP_H, i = e % MLP_H;
    const uint16_t w = f2bf(th[(mat ? MLP_OFF_W3 : MLP_OFF_W2) + o * MLP_H + i]);
    pw[mlp_pw_fwd(mat, o, i)] = w;
    pw[mlp_pw_back(mat, o, i)] = w;
}

__device__ __forceinline__ mlp_bf16x4 mlp_half(const uint4& q, int s) {  // value block s of an operand pair
    const uint32_t a = s ? q.z : q.x, b = s ? q.w : q.y;
    mlp_bf16x4 r;
    r[0] = (short)(a & 0xffffu);
    r[1] = (short)(a >> 16);
    r[2] = (short)(b & 0xffffu);
    r[3] = (short)(b >> 16);
    return r;
}

// Sixteen values of the D layout as operands, to global memory (a tile's lane order)
__device__ __forceinline__ void mlp_put_operands(uint16_t* __restrict__ dst, size_t stride, const uint16_t (&e)[16]) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        uint32_t d[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = (uint32_t)e[8 * q + 2 * k] | (uint32_t)e[8 * q + 2 * k + 1] << 16;
        *reinterpret_cast<uint4*>(dst + q * stride) = make_uint4(d[0], d[1], d[2], d[3]);
    }
}

// 32 rows forward and back: a block of four waves, wave w the 32 units of tile w of every layer.
// Rows are on the products' M axis, so a lane holds one unit's values of 16 rows and the outputs are
// operands of the weight gradients as they are; the next layer's operands pass through LDS.  The
// wave's share of all four weight products is asked for at the start (32 KB a block from L2).
constexpr int MLP_XS = MLP_H + 4;  // units of a row in LDS: 66 banks, so that 32 rows' reads meet no bank twice

__global__ __launch_bounds__(256) void k_mlp_rows(MlpTrain t) {
    __shared__ alignas(16) uint16_t ex[5][32 * MLP_XS];
    __shared__ float4 xs[32];
    __shared__ float ys[32], ds[32];
    __shared__ alignas(8) uint16_t w4s[MLP_H];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, hi = l >> 5, u = l & 31, unit = 32 * w + u;
    const int row0 = blockIdx.x * 32;
    const size_t opn = (size_t)t.pad * MLP_H;  // values of one operand array
    uint4 wt[4][8];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int k = 0; k < 8; ++k) wt[m][k] = *reinterpret_cast<const uint4*>(t.pw + ((((m * 4 + w) * 8 + k) * 64 + l) << 3));
    if (threadIdx.x < 32) {
        const int b = row0 + (int)threadIdx.x;
        float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float y = 0.0f;
        if (b < t.B) {
            const int s = t.perm ? t.perm[b] : b;
            x = reinterpret_cast<const float4*>(t.X)[s];
            y = t.Y[s];
        }
        xs[threadIdx.x] = x;
        ys[threadIdx.x] = y;
    }
    const float4 w1 = *reinterpret_cast<const float4*>(t.th + MLP_OFF_W1 + unit * MLP_IN);
    const float b1 = t.th[MLP_OFF_B1 + unit], b2 = t.th[MLP_OFF_B2 + unit], b3 = t.th[MLP_OFF_B3 + unit],
                b4 = t.th[MLP_OFF_B4];
    const uint16_t w4 = f2bf(t.th[MLP_OFF_W4 + unit]);
    if (hi == 0) w4s[unit] = w4;
    pimc::lds_barrier();
    auto row_of = [&](int i) { return 8 * (i >> 2) + 4 * hi + (i & 3); };
    // a tile's values to LDS for the next product and to memory as operands of the gradient
    auto put = [&](int x, const float (&h)[16], int a) {
        uint16_t e[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            e[i] = f2bf(h[i]);
            ex[x][row_of(i) * MLP_XS + unit] = e[i];
        }
        mlp_put_operands(t.ops + a * opn + ((((size_t)(row0 >> 4) * 4 + w) * 64 + l) << 3), 4 * 64 * 8, e);
    };
    auto put_dz = [&](int layer, const float (&d)[16]) {
        float* p = t.dz + layer * opn + (size_t)row0 * MLP_H + unit;
#pragma unroll
        for (int i = 0; i < 16; ++i) p[row_of(i) * MLP_H] = d[i];
    };
    auto operand = [&](int x, int kb) { return mlp_load4(&ex[x][u * MLP_XS + 8 * kb + 4 * hi]); };
    auto product = [&](int x, const uint4 (&wm)[8]) {
        mlp_f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 16; ++kb) acc = mlp_mfma(operand(x, kb), mlp_half(wm[kb >> 1], kb & 1), acc);
        return acc;
    };
    float z1[16], z2[16], z3[16], h[16];
    auto activate = [&](const mlp_f32x16& acc, float b, float (&z)[16]) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            z[i] = acc[i] + b;
            h[i] = row0 + row_of(i) < t.B ? mlp_silu(z[i]) : 0.0f;
        }
    };
    {
        mlp_bf16x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
        if (hi == 0) {
            const float4 x = xs[u];
            a[0] = (short)f2bf(x.x); a[1] = (short)f2bf(x.y); a[2] = (short)f2bf(x.z); a[3] = (short)f2bf(x.w);
            b[0] = (short)f2bf(w1.x); b[1] = (short)f2bf(w1.y); b[2] = (short)f2bf(w1.z); b[3] = (short)f2bf(w1.w);
        }
        mlp_f32x16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
        activate(mlp_mfma(a, b, acc), b1, z1);
    }
    put(0, h, 0);
    pimc::lds_barrier();
    activate(product(0, wt[0]), b2, z2);
    put(1, h, 1);
    pimc::lds_barrier();
    activate(product(1, wt[1]), b3, z3);
    put(2, h, 2);
    pimc::lds_barrier();
    // the output row by row, in every wave: column 0 of H3 w4
    mlp_f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 16; ++kb) {
        const mlp_bf16x4 none = {0, 0, 0, 0}, b = mlp_load4(&w4s[8 * kb + 4 * hi]);
        acc = mlp_mfma(operand(2, kb), u == 0 ? b : none, acc);
    }
    float dout[16], d[16];
    uint16_t eo[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float o = __shfl(acc[i], 32 * hi) + b4;
        const float e = o - ys[row_of(i)];
        const bool in = row0 + row_of(i) < t.B;
        dout[i] = in ? e / (float)t.B : 0.0f;
        eo[i] = u == 0 ? f2bf(dout[i]) : (uint16_t)0;
        if (w == 3 && u == 0) ds[row_of(i)] = in ? e : 0.0f;
    }
    // dZ3 = (dout w4) SiLU'(Z3): the product of two BF16 values is exact
    const float w4b = bf2f(w4);
    auto back = [&](float dh, float z) {
        const float s = mlp_sigmoid(z);
        dh *= s * (1.0f + z * (1.0f - s));
        return dh;
    };
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = back(bf2f(f2bf(dout[i])) * w4b, z3[i]);
    put(3, d, 5);
    put_dz(2, d);
    if (w == 0) mlp_put_operands(t.opd + (((size_t)(row0 >> 4) * 64 + l) << 3), 64 * 8, eo);
    if (w == 1) {
        uint16_t e[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) e[i] = u < MLP_IN ? f2bf(reinterpret_cast<const float*>(xs)[row_of(i) * MLP_IN + (u & 3)]) : (uint16_t)0;
        mlp_put_operands(t.opx + (((size_t)(row0 >> 4) * 64 + l) << 3), 64 * 8, e);
    }
    if (w == 2 && u == 0)
#pragma unroll
        for (int i = 0; i < 16; ++i) t.dout[row0 + row_of(i)] = dout[i];
    pimc::lds_barrier();
    if (w == 3) {  // loss: (1/2n) sum (out - y)^2
        const float e = u == l ? ds[u] : 0.0f;
        double s = 0.5 * (double)e * (double)e / (double)t.B;
        for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (l == 0) t.loss[blockIdx.x] = s;
    }
    acc = product(3, wt[3]);
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = back(acc[i], z2[i]);
    put(4, d, 4);
    put_dz(1, d);
    pimc::lds_barrier();
    acc = product(4, wt[2]);
    uint16_t e[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        d[i] = back(acc[i], z1[i]);
        e[i] = f2bf(d[i]);
    }
    mlp_put_operands(t.ops + 3 * opn + ((((size_t)(row0 >> 4) * 4 + w) * 64 + l) << 3), 4 * 64 * 8, e);
    put_dz(0, d);
}

// Adam (Kingma & Ba 2015): m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2;
// theta -= lr * (m / (1 - b1^t)) / (sqrt(v / (1 - b2^t)) + eps).
struct MlpAdam {
    float lr, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
};
__device__ __forceinline__ float mlp_adam(float th, float gi, float& m, float& v, const MlpAdam& a) {
    const float mi = 0.9f * m + 0.1f * gi;
    const float vi = 0.999f * v + 0.001f * gi * gi;
    m = mi;
    v = vi;
    th -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + 1e-8f);
    return th;
}

// Weight gradients of a batch and the step on the weights.  Blocks 0..39 take a 32x32 tile of dW3,
// dW2, dW4 and dW1 = dZ^T H each: one wave runs the chain of products over the batch from LDS while
// the other three bring in the chunks after it, the next in LDS's other half and the one after that
// in registers.  The other blocks sum biases: 16 columns of a dZ each, and dout.
constexpr int MLP_TILE_JOBS = 40, MLP_COL = 16, MLP_COL_JOBS = 3 * MLP_H / MLP_COL;
constexpr int MLP_GRAD_JOBS = MLP_TILE_JOBS + MLP_COL_JOBS + 1;
constexpr int MLP_CHUNK = 24;                           // groups of 16 rows staged at a time
constexpr int MLP_CHUNK_Q = MLP_CHUNK * 64;             // 16-byte words of one operand of a chunk
constexpr int MLP_CHUNK_T = MLP_CHUNK_Q / 192;          // of them per lane of three waves
constexpr int MLP_GRAD_LDS = 4 * MLP_CHUNK_Q * 16;      // two operands, two buffers

__global__ __launch_bounds__(256) void k_mlp_grads(MlpTrain t, MlpAdam ad) {
    extern __shared__ uint4 mlp_lds[];
    const int job = blockIdx.x, tid = threadIdx.x;
    const size_t opn = (size_t)t.pad * MLP_H;
    if (job >= MLP_TILE_JOBS) {
        // lane t's share of a column is rows t, t + 256, ..., then a tree over the 256
        float* red = reinterpret_cast<float*>(mlp_lds);
        const int cj = job - MLP_TILE_JOBS;
        const bool out = cj == MLP_COL_JOBS;
        const int layer = out ? 0 : cj / (MLP_H / MLP_COL), c0 = out ? 0 : cj % (MLP_H / MLP_COL) * MLP_COL;
        const int off = out ? MLP_OFF_B4 : (layer == 0 ? MLP_OFF_B1 : layer == 1 ? MLP_OFF_B2 : MLP_OFF_B3) + c0;
        const int nc = out ? 1 : MLP_COL;
        if (out) {
            float s = 0.0f;
            for (int r = tid; r < t.B; r += 256) s += t.dout[r];
            red[tid] = s;
        } else {
            const int q = tid & 3, rl = tid >> 2;  // four columns, rows rl + 64 k of every 256
            const float* p = t.dz + layer * opn + c0 + 4 * q;
            float4 s[4] = {};
#pragma unroll 4
            for (int r = rl; r < t.B; r += 256)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (r + 64 * k < t.B) {
                        const float4 x = *reinterpret_cast<const float4*>(p + (size_t)(r + 64 * k) * MLP_H);
                        s[k].x += x.x;
                        s[k].y += x.y;
                        s[k].z += x.z;
                        s[k].w += x.w;
                    }
#pragma unroll
            for (int k = 0; k < 4; ++k) *reinterpret_cast<float4*>(red + (rl + 64 * k) * MLP_COL + 4 * q) = s[k];
        }
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            for (int i = tid; i < o * nc; i += 256) red[i] += red[i + o * nc];
            __syncthreads();
        }
        if (tid < nc) {
            const float g = red[tid];
            const int i = off + tid;
            if (t.g) t.g[i] = g;
            else t.th[i] = mlp_adam(t.th[i], g, t.m[i], t.v[i], ad);
        }
        return;
    }
    const bool square = job < 32;  // dW3, dW2
    const int mt = square ? (job & 15) >> 2 : job & 3, nt = square ? job & 3 : 0;
    const int aop = job < 16 ? 5 : job < 32 ? 4 : job < 36 ? 2 : 3;  // dZ3, dZ2, H3, dZ1
    const uint4* A = reinterpret_cast<const uint4*>(t.ops + aop * opn) + mt * 64;
    const uint4* Bp = job < 16 ? reinterpret_cast<const uint4*>(t.ops + opn) + nt * 64          // H2
                      : job < 32 ? reinterpret_cast<const uint4*>(t.ops) + nt * 64             // H1
                      : reinterpret_cast<const uint4*>(job < 36 ? t.opd : t.opx);
    const int sb = square ? 4 * 64 : 64;  // 16-byte words between groups of rows
    const int ng = t.pad >> 4, nchunk = (ng + MLP_CHUNK - 1) / MLP_CHUNK;
    const int l = tid & 63, hi = l >> 5, u = l & 31;
    const bool chain = __builtin_amdgcn_readfirstlane(tid) < 64;
    // element (m, n) of the tile is weight off + m ld + n
    const int ld = square ? MLP_H : job < 36 ? 1 : MLP_IN, ncol = square ? 32 : ld;
    const int off = (job < 16 ? MLP_OFF_W3 : job < 32 ? MLP_OFF_W2 : job < 36 ? MLP_OFF_W4 : MLP_OFF_W1) + 32 * mt * ld + 32 * nt;
    const bool mine = chain && u < ncol;
    float th[16], am[16], av[16];
    if (mine && !t.g)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int e = off + (8 * (i >> 2) + 4 * hi + (i & 3)) * ld + u;
            th[i] = t.th[e];
            am[i] = t.m[e];
            av[i] = t.v[e];
        }
    struct Words {
        uint4 a[MLP_CHUNK_T], b[MLP_CHUNK_T];
    };
    auto fetch = [&](int c, Words& r) {
#pragma unroll
        for (int k = 0; k < MLP_CHUNK_T; ++k) {
            const int q = tid - 64 + 192 * k, grp = c * MLP_CHUNK + (q >> 6);
            r.a[k] = r.b[k] = make_uint4(0, 0, 0, 0);
            if (grp < ng) {
                r.a[k] = A[(size_t)grp * 256 + (q & 63)];
                r.b[k] = Bp[(size_t)grp * sb + (q & 63)];
            }
        }
    };
    auto stage = [&](int c, const Words& r) {
        uint4* d = mlp_lds + (c & 1) * 2 * MLP_CHUNK_Q;
#pragma unroll
        for (int k = 0; k < MLP_CHUNK_T; ++k) {
            d[tid - 64 + 192 * k] = r.a[k];
            d[MLP_CHUNK_Q + tid - 64 + 192 * k] = r.b[k];
        }
    };
    mlp_f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    auto step = [&](int c, Words& next, Words& after) {
        if (!chain) {
            if (c + 2 < nchunk) fetch(c + 2, after);
            if (c + 1 < nchunk) stage(c + 1, next);
        } else {
            const uint4* s = mlp_lds + (c & 1) * 2 * MLP_CHUNK_Q;
#pragma unroll
            for (int k = 0; k < MLP_CHUNK; ++k) {
                const uint4 a = s[64 * k + l], b = s[MLP_CHUNK_Q + 64 * k + l];
                acc = mlp_mfma(mlp_half(a, 0), mlp_half(b, 0), acc);
                acc = mlp_mfma(mlp_half(a, 1), mlp_half(b, 1), acc);
            }
        }
        pimc::lds_barrier();
    };
    Words w0, w1;
    if (!chain) {
        fetch(0, w0);
        if (nchunk > 1) fetch(1, w1);
        stage(0, w0);
    }
    pimc::lds_barrier();
    for (int c = 0; c < nchunk; c += 2) {
        step(c, w1, w0);
        if (c + 1 < nchunk) step(c + 1, w0, w1);
    }
    if (!mine) return;
    if (t.g) {
#pragma unroll
        for (int i = 0; i < 16; ++i) t.g[off + (8 * (i >> 2) + 4 * hi + (i & 3)) * ld + u] = acc[i];
        return;
    }
    uint16_t w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int e = off + (8 * (i >> 2) + 4 * hi + (i & 3)) * ld + u;
        const float n = mlp_adam(th[i], acc[i], am[i], av[i], ad);
        t.th[e] = n;
        t.m[e] = am[i];
        t.v[e] = av[i];
        w[i] = f2bf(n);
    }
    if (square) {  // the operands of the next step: this lane holds in-unit u of 16 out-units
        const int mat = job < 16 ? 1 : 0;
        mlp_put_operands(t.pw + mlp_pw_back(mat, 32 * mt + 4 * hi, 32 * nt + u), 64 * 8, w);
#pragma unroll
        for (int i = 0; i < 16; ++i) t.pw[mlp_pw_fwd(mat, 32 * mt + 8 * (i >> 2) + 4 * hi + (i & 3), 32 * nt + u)] = w[i];
    }
}

// Packs theta and the normalisation into the sampler's copy, weights in the lane order of the
// matrix instructions (see the layout note at the top of this file).
__global__ void k_mlp_pack(const float* __restrict__ th, const float* __restrict__ norm, MlpPacked* __restrict__ p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 4 * 64 * 4) {  // [mb][lane][j]: W1[mb*32 + lane%32][4*(lane/32) + j]
        const int j = i & 3, lane = (i >> 2) & 63, mb = i >> 8;
        const int o = mb * 32 + (lane & 31), k = 4 * (lane >> 5) + j;
        p->w1[i] = k < MLP_IN ? f2bf(th[MLP_OFF_W1 + o * MLP_IN + k]) : (uint16_t)0;
    }
    if (i < MLP_H * MLP_H) {  // [mb][kb][lane][j]: W[mb*32 + lane%32][16*kb + 8*(j/4) + 4*(lane/32) + j%4]
        const int j = i & 7, lane = (i >> 3) & 63, kb = (i >> 9) & 7, mb = i >> 12;
        const int o = mb * 32 + (lane & 31), u = 16 * kb + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
        p->w2[i] = f2bf(th[MLP_OFF_W2 + o * MLP_H + u]);
        p->w3[i] = f2bf(th[MLP_OFF_W3 + o * MLP_H + u]);
    }
    if (i < MLP_H) {
        p->b1[i] = th[MLP_OFF_B1 + i];
        p->b2[i] = th[MLP_OFF_B2 + i];
        p->b3[i] = th[MLP_OFF_B3 + i];
        p->w4[i] = th[MLP_OFF_W4 + i];
    }
    if (i == 0) {
        p->b4 = th[MLP_OFF_B4];
        for (int j = 0; j < MLP_IN; ++j) {
            p->xm[j] = norm[j];
            p->xinv[j] = 1.0f / norm[MLP_IN + j];
        }
        p->ym = norm[2 * MLP_IN];
        p->ys = norm[2 * MLP_IN + 1];
    }
}

// Batched inference on raw inputs (the sampler's code path): out = ys * net((x - xm)/xs) + ym.
// One wave per 32 rows; the network is staged in LDS (dynamic, sizeof(MlpPacked) bytes).
__global__ __launch_bounds__(256) void k_mlp_infer(const MlpPacked* __restrict__ Wg, const float* __restrict__ X,
                                                   int n, float* __restrict__ out) {
    extern __shared__ uint4 mlp_lds[];
    MlpPacked* W = reinterpret_cast<MlpPacked*>(mlp_lds);
    mlp_stage(Wg, W);
    __syncthreads();
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    const int row = wave * 32 + (l & 31);
    if (wave * 32 >= n) return;  // whole waves leave together
    float f[MLP_IN];
    for (int j = 0; j < MLP_IN; ++j) f[j] = row < n ? (X[(long long)row * MLP_IN + j] - W->xm[j]) * W->xinv[j] : 0.0f;
    const float o = mlp_rows32(W, f);
    if (l < 32 && row < n) out[row] = W->ys * o + W->ym;
}
