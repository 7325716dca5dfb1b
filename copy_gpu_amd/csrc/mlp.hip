// mlp.hip -- learned k-space importance proposal: a 4 -> 64 -> 64 -> 1 MLP
// (SiLU, softplus output, BF16 weights, FP32 accumulation) with hand-written
// forward, backward and Adam kernels.
//
// The reference has no learned component; the proposal replaces its analytic
// Gaussian sampler (rbmd/framework/model/RBEPSample.h:143-175) as the source of
// the RBE k-vectors, with importance weights keeping the force estimator
// unbiased (weights are computed by the force engine's sampler, kspace.hip).
//
// Parameter vector (4545 FP32 values, master copy; a BF16 copy feeds the
// forward pass): W1[64][4], b1[64], W2[64][64], b2[64], w3[64], b3.
// Input features: (|kx|, |ky|, |kz|, |k|) / k_scale.  Output h = softplus(z).
// Training loss over a batch: sum_s w_s (log h_s - y_s)^2.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/rbmd_force.h"
#include "engine.h"

namespace rbmd {

namespace {

constexpr int kH = 64;
constexpr int kNP = kH * 4 + kH + kH * kH + kH + kH + 1;  // 4545
constexpr int oW1 = 0, oB1 = 256, oW2 = 320, oB2 = 4416, oW3 = 4480, oB3 = 4544;
constexpr int kGradBlocks = 256;       // most workgroups of a gradient pass: one per CU
constexpr int kMlpWaves = 8;           // waves of a workgroup, each with its own samples
constexpr int kMlpTile = 16;           // samples of a wave at a time
constexpr int kWRow = kH + 4;          // LDS row of a weight matrix: the 16 rows of a fragment
                                       // start on different banks
constexpr int kTRow = kH + 16;         // LDS row of a transposed tile: 4 samples x 16 units of
                                       // a fragment fall on all 64 banks once

using f4 = float __attribute__((ext_vector_type(4)));

__device__ inline float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ inline uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (uint16_t)(u >> 16);
}

// silu(x) = x / (1 + e^-x) and its derivative from one reciprocal: v_rcp_f32 with a Newton
// step, and the quotient corrected by its residual, 8 instructions for the 22 of two IEEE
// divisions.  e^-x is 2^(p + r), p = -x log2 e and r the rest of that product, with x held to
// -88.5 .. 87 there so that neither it nor the denominator leaves the finite range: above 87 the
// quotient is x, and where e^-x passes 2^126 (x < -87.3) v_rcp_f32 gives 0, as it does for every
// reciprocal below the normal range, so silu and its derivative are 0, which they are to 1e-36.
__device__ inline float silu_d(float x, float* d)
{
    constexpr float kLog2e = 1.44269504f, kLog2eLo = 1.92596299e-8f, kLn2 = 0.693147181f;
    const float n = __builtin_amdgcn_fmed3f(-x, -87.0f, 88.5f);
    const float p = n * kLog2e, r = fmaf(n, kLog2eLo, fmaf(n, kLog2e, -p));
    const float q = __builtin_amdgcn_exp2f(p);
    const float e = 1.0f + fmaf(q, r * kLn2, q);
    float s = __builtin_amdgcn_rcpf(e);
    s = fmaf(fmaf(-e, s, 1.0f), s, s);
    const float a = x * s;
    *d = s * (1.0f + x * (1.0f - s));
    return fabsf(x) < 1e30f ? fmaf(fmaf(-e, a, x), s, a) : a;
}
__device__ inline float silu(float x)
{
    float d;
    return silu_d(x, &d);
}
__device__ inline float softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// The network on the matrix cores, in FP32 (v_mfma_f32_16x16x4_f32; the BF16 weights are
// exact in FP32).  A wave takes 16 samples: matrix rows are hidden units, columns samples,
// so lane (g = lane / 16, c = lane % 16) holds units 16 t + 4 g + v (t, v < 4) of sample c.
// The contraction of the next layer runs over these units in the order (t, v) with one g per
// lane group, which is the layout that the B operand wants: activations pass from layer to
// layer in registers, and the weight fragment of step t is one 16-byte LDS read.
struct alignas(16) MlpLds {
    float W2[kH * kWRow];   // [j][i]
    float W1[kH * 4], b1[kH], b2[kH], w3[kH], b3[4];
};
struct MlpGradLds {
    MlpLds w;
    float W2T[kH * kWRow];  // [i][j]
    float ta[kMlpWaves][kMlpTile * kTRow], td[kMlpWaves][kMlpTile * kTRow];
};

__device__ inline void mlp_stage(const uint16_t* __restrict__ p16, MlpLds& W, float* W2T)
{
    // W2 eight at a time (its offset and rows are multiples of 16 bytes), all loads in flight
    constexpr int kLoads = kH * kH / 8 / (64 * kMlpWaves);
    uint4 w8[kLoads];
#pragma unroll
    for (int k = 0; k < kLoads; ++k)
        w8[k] = ((const uint4*)(p16 + oW2))[threadIdx.x + k * 64 * kMlpWaves];
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
        const int e = (threadIdx.x + k * 64 * kMlpWaves) * 8, j = e / kH, i = e % kH;
        const uint32_t u[4] = {w8[k].x, w8[k].y, w8[k].z, w8[k].w};
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            const float w = __uint_as_float(h & 1 ? u[h >> 1] & 0xffff0000u : u[h >> 1] << 16);
            W.W2[j * kWRow + i + h] = w;
            if (W2T) W2T[(i + h) * kWRow + j] = w;
        }
    }
    for (int e = threadIdx.x; e < kH * 4; e += blockDim.x) W.W1[e] = bf2f(p16[oW1 + e]);
    if (threadIdx.x < kH) {
        W.b1[threadIdx.x] = bf2f(p16[oB1 + threadIdx.x]);
        W.b2[threadIdx.x] = bf2f(p16[oB2 + threadIdx.x]);
        W.w3[threadIdx.x] = bf2f(p16[oW3 + threadIdx.x]);
    }
    if (threadIdx.x == 0) W.b3[0] = bf2f(p16[oB3]);
    __syncthreads();
}

__device__ inline f4 mfma4(float a, float b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// out[rt] += M x for the 64 x 64 matrix M (rows of kWRow floats) and 16 columns x.
__device__ inline void mlp_product(const float* __restrict__ M, const f4 x[4], f4 out[4])
{
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        f4 w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = *(const f4*)&M[(16 * r + c) * kWRow + 16 * t + 4 * g];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = mfma4(w[r][v], x[t][v], out[r]);
    }
}

// Pre-activations of both layers for the wave's 16 samples (f: feature g of sample c);
// act(pre1) gives a1, and z is the network's last sum, the same in all lanes of a sample.
template <class Act1, class Act2>
__device__ inline float mlp_forward(const MlpLds& W, float f, Act1 act1, Act2 act2)
{
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    f4 a1[4], p2[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const f4 pre = mfma4(W.W1[(16 * t + c) * 4 + g], f, *(const f4*)&W.b1[16 * t + 4 * g]);
#pragma unroll
        for (int v = 0; v < 4; ++v) a1[t][v] = act1(t, v, pre[v]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) p2[t] = *(const f4*)&W.b2[16 * t + 4 * g];
    mlp_product(W.W2, a1, p2);
    float z = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const f4 w3 = *(const f4*)&W.w3[16 * t + 4 * g];
#pragma unroll
        for (int v = 0; v < 4; ++v) z = fmaf(w3[v], act2(t, v, p2[t][v]), z);
    }
    z += __shfl_xor(z, 16, 64);
    z += __shfl_xor(z, 32, 64);
    return z + W.b3[0];
}

// First of a wave's 16-sample tiles (then every grid's worth of waves): consecutive tiles go to
// different workgroups, so that the last, partial round adds one wave to a workgroup and not
// eight to some.
__device__ inline int64_t mlp_first_tile()
{
    return (int64_t)(threadIdx.x >> 6) * gridDim.x + blockIdx.x;
}

// Bound by the VALU (32 activations per lane and 16 samples, about 2,800 cycles, against 68
// matrix instructions of 32).  274,625 samples: 46 us; 218 us with one thread per sample.
__global__ __launch_bounds__(64 * kMlpWaves, 2) void k_mlp_forward(const uint16_t* __restrict__ p16,
                                                     const float* __restrict__ feat, int64_t B,
                                                     float* __restrict__ out)
{
    __shared__ MlpLds W;
    mlp_stage(p16, W, nullptr);
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int64_t nt = (B + kMlpTile - 1) / kMlpTile;
    for (int64_t tl = mlp_first_tile(); tl < nt; tl += (int64_t)gridDim.x * kMlpWaves) {
        const int64_t s = tl * kMlpTile + c;
        const float f = s < B ? feat[4 * s + g] : 0.0f;
        auto act = [](int, int, float p) { return silu(p); };
        const float z = mlp_forward(W, f, act, act);
        if (g == 0 && s < B) out[s] = softplus(z);
    }
}

// Orders a wave's LDS writes before its later reads of other lanes' values (and the reads
// before the next writes).
__device__ inline void mlp_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Loss (and with GRAD the parameter gradients) of the weighted log-MSE.  Each wave runs
// forward and backward for 16 samples at a time and keeps its sums of the gradients in
// registers; the contractions over samples (dW2 = d2 a1^T, dW1 = d1 f^T with a column of
// ones for db1) take their operands transposed through LDS.  The workgroup adds its waves in
// order: gpart[block][4545], loss to lossp[block].
//
// Per 16 samples 212 matrix instructions of 32 cycles and 32 activations per lane, two waves
// per SIMD to overlap them; eight waves share one workgroup per CU, so the staging of the
// weights and the partial gradients (18 KB a workgroup) are paid once per CU.  35,937 samples:
// 27 us (with 512 workgroups of four waves the sum of twice the partials takes 11 us instead
// of 7); 352 us with one thread per sample and a scalar loop per parameter.
template <bool GRAD>
__global__ __launch_bounds__(64 * kMlpWaves, 2) void k_mlp_loss_grad(
    const uint16_t* __restrict__ p16, const float* __restrict__ feat, const float* __restrict__ y,
    const float* __restrict__ wt, int64_t B, float* __restrict__ gpart, double* __restrict__ lossp)
{
    extern __shared__ __align__(16) float mlp_lds[];
    __shared__ double lred[kMlpWaves];
    MlpGradLds& L = *(MlpGradLds*)mlp_lds;
    MlpLds& W = L.w;
    mlp_stage(p16, W, GRAD ? L.W2T : nullptr);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    float* ta = L.ta[wv];
    float* td = L.td[wv];
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f4 gW2[4][4], gW1[4], gb2[4], gw3[4];
    float gb3 = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        gW1[r] = gb2[r] = gw3[r] = zero;
#pragma unroll
        for (int k = 0; k < 4; ++k) gW2[r][k] = zero;
    }
    double loss = 0.0;
    const int64_t nt = (B + kMlpTile - 1) / kMlpTile;
    for (int64_t tl = mlp_first_tile(); tl < nt; tl += (int64_t)gridDim.x * kMlpWaves) {
        const int64_t s = tl * kMlpTile + c;
        const bool ok = s < B;
        const float f = ok ? feat[4 * s + g] : 0.0f;
        const float ys = ok ? y[s] : 0.0f, ws = ok ? wt[s] : 0.0f;
        f4 a1[4], d1[4], a2[4], d2[4];
        const float z = mlp_forward(
            W, f,
            [&](int t, int v, float p) {
                float d;
                a1[t][v] = silu_d(p, &d);
                d1[t][v] = d;
                return a1[t][v];
            },
            [&](int t, int v, float p) {
                float d;
                a2[t][v] = silu_d(p, &d);
                d2[t][v] = d;
                return a2[t][v];
            });
        float dz = 0.0f;
        if (ok) {
            // log softplus(z) and its derivative sigmoid(z) / softplus(z); below
            // z = -15 both equal z and 1 to FP32 precision (and softplus(z)
            // would underflow further down)
            const float h = softplus(z);
            const bool tiny = z < -15.0f;
            const float t = (tiny ? z : logf(h)) - ys;
            if (g == 0) loss += (double)ws * (double)t * (double)t;
            const float dlog = tiny ? 1.0f : 1.0f / ((1.0f + expf(-z)) * h);
            dz = 2.0f * ws * t * dlog;
        }
        if (!GRAD) continue;
        gb3 += dz;
        mlp_wave_sync();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f4 w3 = *(const f4*)&W.w3[16 * t + 4 * g];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                gw3[t][v] = fmaf(dz, a2[t][v], gw3[t][v]);
                d2[t][v] = dz * w3[v] * d2[t][v];
                gb2[t][v] += d2[t][v];
            }
            *(f4*)&ta[c * kTRow + 16 * t + 4 * g] = a1[t];
            *(f4*)&td[c * kTRow + 16 * t + 4 * g] = d2[t];
        }
        f4 u[4] = {zero, zero, zero, zero};
        mlp_product(L.W2T, d2, u);
        mlp_wave_sync();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float a[4], b[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                a[r] = td[(4 * k + g) * kTRow + 16 * r + c];
                b[r] = ta[(4 * k + g) * kTRow + 16 * r + c];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) gW2[r][q] = mfma4(a[r], b[q], gW2[r][q]);
        }
        mlp_wave_sync();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int v = 0; v < 4; ++v) d1[t][v] *= u[t][v];
            *(f4*)&td[c * kTRow + 16 * t + 4 * g] = d1[t];
        }
        mlp_wave_sync();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // column c < 4: feature c of sample 4 k + g; column 4: one
            const float fc = __shfl(f, (c & 3) * 16 + 4 * k + g, 64);
            const float b = c < 4 ? fc : c == 4 ? 1.0f : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                gW1[r] = mfma4(td[(4 * k + g) * kTRow + 16 * r + c], b, gW1[r]);
        }
    }
    loss = wave_sum(loss);
    if (lane == 0) lred[wv] = loss;
    __syncthreads();
    if (threadIdx.x == 0) {
        double l = 0.0;
        for (int w = 0; w < kMlpWaves; ++w) l += lred[w];
        lossp[blockIdx.x] = l;
    }
    if (!GRAD) return;
    // the workgroup's gradients: each wave's in parameter order, then the waves in order
    float* red = mlp_lds + (size_t)wv * kNP;
    // sum of a 16-lane row in all of its lanes, by DPP moves (xor 1, xor 2, mirrors)
    auto row_sum = [](float v) {
        v += __int_as_float(dpp_i<0xB1>(__float_as_int(v)));
        v += __int_as_float(dpp_i<0x4E>(__float_as_int(v)));
        v += __int_as_float(dpp_i<0x141>(__float_as_int(v)));
        v += __int_as_float(dpp_i<0x140>(__float_as_int(v)));
        return v;
    };
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = 16 * r + 4 * g + v;
#pragma unroll
            for (int q = 0; q < 4; ++q) red[oW2 + j * kH + 16 * q + c] = gW2[r][q][v];
            if (c < 4) red[oW1 + 4 * j + c] = gW1[r][v];
            if (c == 4) red[oB1 + j] = gW1[r][v];
            const float sb = row_sum(gb2[r][v]), sw = row_sum(gw3[r][v]);
            if (c == 0) {
                red[oB2 + j] = sb;
                red[oW3 + j] = sw;
            }
        }
    gb3 = row_sum(gb3);
    if (lane == 0) red[oB3] = gb3;
    __syncthreads();
    for (int e = threadIdx.x; e < kNP; e += 64 * kMlpWaves) {
        double acc = 0.0;
        for (int w = 0; w < kMlpWaves; ++w) acc += (double)mlp_lds[(size_t)w * kNP + e];
        gpart[(size_t)blockIdx.x * kNP + e] = (float)acc;
    }
}

// Sum of the block partials in a fixed order, in FP64 (16 strided sums per parameter, then
// those in order), and with ADAM the update (Kingma & Ba 2015) of the FP32 master weights and
// their BF16 copy.  64 parameters per workgroup: 72 workgroups of 16 waves, each reading 256
// contiguous bytes of a partial.  One thread per parameter summing all of them took 74 us.
constexpr int kSumEntries = 64, kSumSlices = 16;
constexpr int kSumBlocks = (kNP + kSumEntries - 1) / kSumEntries;
struct MlpAdam {
    float *p, *m, *v;
    uint16_t* p16;
    float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(kSumEntries* kSumSlices) void k_mlp_reduce(
    const float* __restrict__ gpart, int nb, float* __restrict__ grad, MlpAdam a)
{
    __shared__ double red[kSumSlices][kSumEntries];
    const int k = threadIdx.x % kSumEntries, sl = threadIdx.x / kSumEntries;
    const int e = blockIdx.x * kSumEntries + k;
    double acc = 0.0;
    if (e < kNP)
        for (int b = sl; b < nb; b += kSumSlices) acc += (double)gpart[(size_t)b * kNP + e];
    red[sl][k] = acc;
    __syncthreads();
    if (sl || e >= kNP) return;
    acc = 0.0;
    for (int s = 0; s < kSumSlices; ++s) acc += red[s][k];
    const float ge = (float)acc;
    if (!ADAM) {
        grad[e] = ge;
        return;
    }
    const float mm = a.b1 * a.m[e] + (1.0f - a.b1) * ge;
    const float vv = a.b2 * a.v[e] + (1.0f - a.b2) * ge * ge;
    a.m[e] = mm;
    a.v[e] = vv;
    const float pe = a.p[e] - a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + a.eps);
    a.p[e] = pe;
    a.p16[e] = f2bf(pe);
}

// The loss from the blocks' (nb <= kGradBlocks), one wave in a fixed order.
__global__ __launch_bounds__(64) void k_mlp_loss(const double* __restrict__ lossp, int nb,
                                                 double* __restrict__ loss)
{
    double l = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) l += lossp[b];
    l = wave_sum(l);
    if (threadIdx.x == 0) *loss = l;
}

__global__ void k_mlp_cast(const float* __restrict__ p, uint16_t* __restrict__ p16)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < kNP) p16[e] = f2bf(p[e]);
}

constexpr size_t kGradLds = std::max(sizeof(MlpGradLds), sizeof(float) * kMlpWaves * kNP);
static_assert(kGradLds <= 160 * 1024 - 1024, "fits a CU's LDS");

// Workgroups of a pass over B samples: as many as there are tiles for, one per CU at most.
inline int mlp_blocks(int64_t B)
{
    const int64_t nt = (B + kMlpTile - 1) / kMlpTile;
    return (int)std::min<int64_t>((nt + kMlpWaves - 1) / kMlpWaves, kGradBlocks);
}

}  // namespace

}  // namespace rbmd

using namespace rbmd;

struct rbmd_mlp_s {
    float* p = nullptr;
    uint16_t* p16 = nullptr;
    float *m = nullptr, *v = nullptr, *grad = nullptr, *gpart = nullptr;
    double *lossp = nullptr, *loss = nullptr;
    int64_t step = 0;
    std::string err;
};

static int mlp_fail(rbmd_mlp_t h, hipError_t e, const char* what)
{
    h->err = std::string(what) + ": " + hipGetErrorString(e);
    return RBMD_ERR_HIP;
}

#define MLP_TRY(expr)                                  \
    do {                                               \
        hipError_t _e = (expr);                        \
        if (_e != hipSuccess) return mlp_fail(h, _e, #expr); \
    } while (0)

extern "C" {

int rbmd_mlp_nparams(void) { return kNP; }

int rbmd_mlp_create(uint64_t seed, rbmd_mlp_t* out)
{
    if (!out) return RBMD_ERR_INVALID;
    rbmd_mlp_t h = new rbmd_mlp_s();
    *out = nullptr;
    // Glorot-uniform weights from Philox, zero biases, b3 = log(e - 1) so h = 1 at start
    std::vector<float> p(kNP, 0.0f);
    const uint32_t key[2] = {(uint32_t)seed, (uint32_t)(seed >> 32)};
    auto uni = [&](uint32_t idx) {
        uint32_t c[4] = {idx, 0x4D4C5031u, 0u, 0u}, r[4];
        philox4x32_10(c, key, r);
        return (float)u53(r[0], r[1]) * 2.0f - 1.0f;
    };
    const float s1 = sqrtf(6.0f / (4 + kH)), s2 = sqrtf(6.0f / (kH + kH)), s3 = sqrtf(6.0f / (kH + 1));
    for (int e = 0; e < kH * 4; ++e) p[oW1 + e] = s1 * uni(oW1 + e);
    for (int e = 0; e < kH * kH; ++e) p[oW2 + e] = s2 * uni(oW2 + e);
    for (int e = 0; e < kH; ++e) p[oW3 + e] = s3 * uni(oW3 + e);
    p[oB3] = logf(expf(1.0f) - 1.0f);
    int rc = RBMD_OK;
    hipError_t e;
    if ((e = hipMalloc((void**)&h->p, kNP * 4)) != hipSuccess ||
        (e = hipMalloc((void**)&h->p16, kNP * 2)) != hipSuccess ||
        (e = hipMalloc((void**)&h->m, kNP * 4)) != hipSuccess ||
        (e = hipMalloc((void**)&h->v, kNP * 4)) != hipSuccess ||
        (e = hipMalloc((void**)&h->grad, kNP * 4)) != hipSuccess ||
        (e = hipMalloc((void**)&h->gpart, (size_t)kGradBlocks * kNP * 4)) != hipSuccess ||
        (e = hipMalloc((void**)&h->lossp, kGradBlocks * 8)) != hipSuccess ||
        (e = hipMalloc((void**)&h->loss, 8)) != hipSuccess ||
        (e = hipMemcpy(h->p, p.data(), kNP * 4, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemset(h->m, 0, kNP * 4)) != hipSuccess ||
        (e = hipMemset(h->v, 0, kNP * 4)) != hipSuccess) {
        rc = RBMD_ERR_HIP;
    }
    if (rc == RBMD_OK &&
        (e = hipFuncSetAttribute((const void*)k_mlp_loss_grad<true>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGradLds)) !=
            hipSuccess) {
        h->err = std::string("dynamic LDS of the gradient kernel: ") + hipGetErrorString(e);
        rc = RBMD_ERR_HIP;
    }
    if (rc == RBMD_OK) {
        k_mlp_cast<<<(kNP + 255) / 256, 256>>>(h->p, h->p16);
        if (hipDeviceSynchronize() != hipSuccess) rc = RBMD_ERR_HIP;
    }
    if (rc != RBMD_OK) {
        rbmd_mlp_destroy(h);
        return rc;
    }
    *out = h;
    return RBMD_OK;
}

void rbmd_mlp_destroy(rbmd_mlp_t h)
{
    if (!h) return;
    void* ptrs[] = {h->p, h->p16, h->m, h->v, h->grad, h->gpart, h->lossp, h->loss};
    for (void* q : ptrs)
        if (q) hipFree(q);
    delete h;
}

const char* rbmd_mlp_last_error(rbmd_mlp_t h) { return h ? h->err.c_str() : "null handle"; }

int rbmd_mlp_get_params(rbmd_mlp_t h, float* params)
{
    if (!h || !params) return RBMD_ERR_INVALID;
    MLP_TRY(hipDeviceSynchronize());
    MLP_TRY(hipMemcpy(params, h->p, kNP * 4, hipMemcpyDeviceToHost));
    return RBMD_OK;
}

int rbmd_mlp_set_params(rbmd_mlp_t h, const float* params)
{
    if (!h || !params) return RBMD_ERR_INVALID;
    MLP_TRY(hipMemcpy(h->p, params, kNP * 4, hipMemcpyHostToDevice));
    MLP_TRY(hipMemset(h->m, 0, kNP * 4));
    MLP_TRY(hipMemset(h->v, 0, kNP * 4));
    h->step = 0;
    k_mlp_cast<<<(kNP + 255) / 256, 256>>>(h->p, h->p16);
    MLP_TRY(hipGetLastError());
    return RBMD_OK;
}

int rbmd_mlp_forward(rbmd_mlp_t h, const float* feat, int64_t B, float* out, void* stream)
{
    if (!h || B < 0 || (B > 0 && (!feat || !out))) return RBMD_ERR_INVALID;
    if (B == 0) return RBMD_OK;
    // one workgroup per CU, as the registers allow: each stages the weights once
    const int64_t nt = (B + kMlpTile - 1) / kMlpTile;
    const int blocks = (int)std::min<int64_t>((nt + kMlpWaves - 1) / kMlpWaves, kGradBlocks);
    k_mlp_forward<<<blocks, 64 * kMlpWaves, 0, (hipStream_t)stream>>>(h->p16, feat, B, out);
    MLP_TRY(hipGetLastError());
    return RBMD_OK;
}

static void mlp_grad(rbmd_mlp_t h, const float* feat, const float* y, const float* w, int64_t B,
                     hipStream_t s)
{
    k_mlp_loss_grad<true><<<mlp_blocks(B), 64 * kMlpWaves, kGradLds, s>>>(h->p16, feat, y, w, B,
                                                                       h->gpart, h->lossp);
}

int rbmd_mlp_loss_grad(rbmd_mlp_t h, const float* feat, const float* y, const float* w,
                       int64_t B, double* loss, float* grad, void* stream)
{
    if (!h || B < 1 || !feat || !y || !w) return RBMD_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    mlp_grad(h, feat, y, w, B, s);
    k_mlp_reduce<false><<<kSumBlocks, kSumEntries * kSumSlices, 0, s>>>(h->gpart, mlp_blocks(B),
                                                                    h->grad, MlpAdam{});
    k_mlp_loss<<<1, 64, 0, s>>>(h->lossp, mlp_blocks(B), h->loss);
    MLP_TRY(hipGetLastError());
    MLP_TRY(hipStreamSynchronize(s));
    if (loss) MLP_TRY(hipMemcpy(loss, h->loss, 8, hipMemcpyDeviceToHost));
    if (grad) MLP_TRY(hipMemcpy(grad, h->grad, kNP * 4, hipMemcpyDeviceToHost));
    return RBMD_OK;
}

int rbmd_mlp_train(rbmd_mlp_t h, const float* feat, const float* y, const float* w, int64_t B,
                   int32_t iters, double lr, double* final_loss, void* stream)
{
    if (!h || B < 1 || iters < 0 || !feat || !y || !w || !(lr > 0)) return RBMD_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int32_t it = 0; it < iters; ++it) {
        mlp_grad(h, feat, y, w, B, s);
        h->step += 1;
        const float c1 = 1.0f - powf(b1, (float)h->step), c2 = 1.0f - powf(b2, (float)h->step);
        const MlpAdam a{h->p, h->m, h->v, h->p16, (float)lr, b1, b2, eps, c1, c2};
        k_mlp_reduce<true><<<kSumBlocks, kSumEntries * kSumSlices, 0, s>>>(
            h->gpart, mlp_blocks(B), nullptr, a);
    }
    MLP_TRY(hipGetLastError());
    if (final_loss) {
        k_mlp_loss_grad<false><<<mlp_blocks(B), 64 * kMlpWaves, sizeof(MlpLds), s>>>(
            h->p16, feat, y, w, B, nullptr, h->lossp);
        k_mlp_loss<<<1, 64, 0, s>>>(h->lossp, mlp_blocks(B), h->loss);
        MLP_TRY(hipGetLastError());
        MLP_TRY(hipStreamSynchronize(s));
        MLP_TRY(hipMemcpy(final_loss, h->loss, 8, hipMemcpyDeviceToHost));
    }
    return RBMD_OK;
}

}  // extern "C"
