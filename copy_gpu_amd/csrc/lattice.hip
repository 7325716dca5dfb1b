// lattice.hip -- structure factors on a lattice box by FP64 matrix products (lattice.h),
// and the |rho(m)|^2 spectrum that trains the learned k-space proposal.
//
// rho(k) itself: rbmd/framework/run/worklet/RunWorklet.cpp:1616-1677 and
// rbmd/framework/run/ExecutionMD.cpp:412-448 (paths relative to the reference checkout).
#include <algorithm>
#include <string>

#include "../../include/rbmd_force.h"
#include "lattice.h"

namespace rbmd {

namespace {

struct LatSumArgs {
    const double *x, *y, *z, *q;
    int64_t n;
    Box box;
    LatGeom g;
    double* part;
};

// T of one atom slice for 256 rows x (16 NC) columns.  Per stage of 32 atoms the
// workgroup tabulates the basis values that its rows and columns use (q folded into the x
// table), then each wave forms its 64 rows x 16 NC columns with v_mfma_f64_16x16x4_f64:
// the A fragment is the product of an x and a y table value, the B fragment a z value, and
// the constant column (c = 0) is the running sum of the A fragments.
//
// Tables: sines and cosines of m = 1 .. 8 per axis by sincospi, larger m by rotating eight
// further at a time (one rounding of about 2^-53 each, far below the phase's own).  The
// positions come through LDS 256 atoms at a time, as exact box fractions.
//
// Bound by FP64 issue: 8 x 4 NC matrix instructions of 64 cycles per wave and stage (67% of
// the cycles) and about three sines and cosines per thread.  100,000 ions, |m_d| <= 32 (5.4e10
// operations): 1.20 ms, 45 TFLOP/s of the 72 that a large FP64 product reaches here; with a
// sine and cosine per (m, atom) the sums took 29 ms.
constexpr int kLatBase = 8;      // m that get a sine and cosine of their own
constexpr int kLatLoad = 256;    // atoms per load of positions

template <int NC>
__global__ __launch_bounds__(256, 2) void k_lat_sums(LatSumArgs A)
{
    extern __shared__ double lat_lds[];
    const LatGeom& g = A.g;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int kl = lane >> 4, rl = lane & 15;
    const int B = g.B, C = g.C;
    const int64_t r0 = (int64_t)blockIdx.x * kLatRows;
    const int64_t rl1 = r0 + kLatRows <= g.R ? r0 + kLatRows - 1 : g.R - 1;
    const int a0 = (int)(r0 / B), b0 = (int)(r0 % B);
    const int nx = (int)(rl1 / B) - a0 + 1, ny = g.ny;
    const int c0 = (int)blockIdx.y * 16 * NC;  // columns c0 + 1 .. c0 + 16 NC
    double* Xt = lat_lds;
    double* Yt = Xt + (size_t)g.nx * kLatStride;
    double* Zt = Yt + (size_t)ny * kLatStride;
    double* base = Zt + (size_t)16 * NC * kLatStride;  // [y, z][m - 1][cos, sin][atom]
    double* frac = base + 2 * kLatBase * 2 * kLatStage;  // [x hi, x lo, y .., z .., q][atom]

    int xo[4], yo[4];
    for (int i = 0; i < 4; ++i) {
        int64_t r = r0 + wv * 64 + i * 16 + rl;
        r = r < g.R ? r : g.R - 1;
        xo[i] = ((int)(r / B) - a0) * kLatStride + kl;
        yo[i] = (int)((r - r0) % ny) * kLatStride + kl;
    }
    const int zo = rl * kLatStride + kl;
    d4 acc[4][NC];
    double ones[4];
    for (int i = 0; i < 4; ++i) {
        ones[i] = 0.0;
        for (int c = 0; c < NC; ++c) acc[i][c] = d4{0.0, 0.0, 0.0, 0.0};
    }

    const int64_t j0 = (int64_t)blockIdx.z * g.aps;
    const int64_t j1 = j0 + g.aps < A.n ? j0 + g.aps : A.n;
    const int at = t & (kLatStage - 1), grp = t / kLatStage;
    constexpr int kGrp = 256 / kLatStage;
    static_assert(kGrp == kLatBase, "a thread's multiples of one axis are one rotation apart");
    const int mx0 = (a0 + 1) >> 1, nmx = ((a0 + nx) >> 1) - mx0 + 1;
    const int items = 2 * kLatBase + nmx;
    for (int64_t j = j0; j < j1; j += kLatStage) {
        const int fo = (int)((j - j0) & (kLatLoad - 1));
        if (fo == 0) {
            const int64_t i = j + t;
            LatFrac s[3] = {{0, 0}, {0, 0}, {0, 0}};
            double q = 0.0;
            if (i < j1) {
                s[0] = lat_frac(A.x[i] - A.box.lo[0], A.box.L[0], A.box.invL[0]);
                s[1] = lat_frac(A.y[i] - A.box.lo[1], A.box.L[1], A.box.invL[1]);
                s[2] = lat_frac(A.z[i] - A.box.lo[2], A.box.L[2], A.box.invL[2]);
                q = A.q[i];
            }
            for (int d = 0; d < 3; ++d) {
                frac[(2 * d) * kLatLoad + t] = s[d].hi;
                frac[(2 * d + 1) * kLatLoad + t] = s[d].lo;
            }
            frac[6 * kLatLoad + t] = q;
        }
        __syncthreads();  // the fractions are there; the last stage's tables are read
        for (int e = grp; e < items; e += kGrp) {
            const int d = e < kLatBase ? 1 : e < 2 * kLatBase ? 2 : 0;
            const int m = d == 0 ? mx0 + e - 2 * kLatBase : (e & (kLatBase - 1)) + 1;
            const LatFrac s{frac[(2 * d) * kLatLoad + fo + at], frac[(2 * d + 1) * kLatLoad + fo + at]};
            double sn, cs;
            lat_sincos(s, m, &sn, &cs);
            if (d == 0) {
                const double q = frac[6 * kLatLoad + fo + at];
                const int ic = lat_cos(m) - a0, is = lat_sin(m) - a0;
                if (ic >= 0 && ic < nx) Xt[ic * kLatStride + at] = q * cs;
                if (m && is >= 0 && is < nx) Xt[is * kLatStride + at] = q * sn;
            } else {
                base[(2 * e) * kLatStage + at] = cs;
                base[(2 * e + 1) * kLatStage + at] = sn;
            }
        }
        __syncthreads();
        {
            // y: m = grp, grp + 8, ...
            const double C8 = base[(2 * kLatBase - 2) * kLatStage + at],
                         S8 = base[(2 * kLatBase - 1) * kLatStage + at];
            double cs = grp ? base[(2 * grp - 2) * kLatStage + at] : 1.0,
                   sn = grp ? base[(2 * grp - 1) * kLatStage + at] : 0.0;
            for (int m = grp; m <= g.M[1]; m += kGrp) {
                int ic = lat_cos(m) - b0, is = lat_sin(m) - b0;
                ic += ic < 0 ? B : 0;
                is += is < 0 ? B : 0;
                if (ic < ny) Yt[ic * kLatStride + at] = cs;
                if (m && is < ny) Yt[is * kLatStride + at] = sn;
                const double c = fma(cs, C8, -(sn * S8));
                sn = fma(sn, C8, cs * S8);
                cs = c;
            }
        }
        {
            // z: m = c0 / 2 + 1 + grp, .. + 8, ..., columns 2 m - 1 and 2 m
            const double* zb = base + 2 * kLatBase * kLatStage;
            const double C8 = zb[(2 * kLatBase - 2) * kLatStage + at],
                         S8 = zb[(2 * kLatBase - 1) * kLatStage + at];
            double cs, sn;
            if (c0 == 0) {
                cs = zb[(2 * grp) * kLatStage + at];
                sn = zb[(2 * grp + 1) * kLatStage + at];
            } else {
                lat_sincos({frac[4 * kLatLoad + fo + at], frac[5 * kLatLoad + fo + at]},
                           (c0 >> 1) + 1 + grp, &sn, &cs);
            }
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int e = grp + kGrp * i;
                const bool in = (c0 >> 1) + 1 + e <= g.M[2];
                Zt[(2 * e) * kLatStride + at] = in ? cs : 0.0;
                Zt[(2 * e + 1) * kLatStride + at] = in ? sn : 0.0;
                const double c = fma(cs, C8, -(sn * S8));
                sn = fma(sn, C8, cs * S8);
                cs = c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kLatStage; k += 4) {
            double b[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) b[c] = Zt[c * 16 * kLatStride + zo + k];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double a = Xt[xo[i] + k] * Yt[yo[i] + k];
                ones[i] += a;
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    acc[i][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[c], acc[i][c], 0, 0, 0);
            }
        }
    }

    double* out = A.part + (int64_t)blockIdx.z * g.sums();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t rb = r0 + wv * 64 + i * 16;
        double o = ones[i];
        o += __shfl_xor(o, 16, 64);
        o += __shfl_xor(o, 32, 64);
        if (blockIdx.y == 0 && lane < 16 && rb + lane < g.R) out[(rb + lane) * C] = o;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int col = c0 + 1 + c * 16 + rl;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // element v of lane l: row 4 v + l / 16, column l % 16
                const int64_t r = rb + 4 * v + kl;
                if (r < g.R && col < C) out[r * C + col] = acc[i][c][v];
            }
        }
    }
}

// Sum of the slices in slice order, in place.
__global__ __launch_bounds__(256) void k_lat_reduce(double* __restrict__ part, int64_t len,
                                                    int slices)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= len) return;
    double v = part[i];
    for (int s = 1; s < slices; ++s) v += part[(int64_t)s * len + i];
    part[i] = v;
}

// |rho(m)|^2 of the whole box (x fastest) from the sums: one thread per octant point
// writes (or adds to) its up to eight images, each once; 0 at m = 0.
__global__ __launch_bounds__(256) void k_lat_spectrum(const double* __restrict__ T, int B, int C,
                                                      int M, int add, double* __restrict__ s2)
{
    const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t h = M + 1, side = 2 * M + 1;
    if (o >= h * h * h) return;
    const int mz = (int)(o % h), my = (int)(o / h % h), mx = (int)(o / (h * h));
    const LatOct t = lat_octant(T, B, C, mx, my, mz);
    const int64_t mid = (side * side * side) / 2;  // index of m = 0; -m is mirrored in it
    for (int gy = 1; gy >= (my ? -1 : 1); gy -= 2)
        for (int gz = 1; gz >= (mz ? -1 : 1); gz -= 2) {
            double re, im;
            lat_rho(t, (double)gy, (double)gz, &re, &im);
            const int64_t d = mx + side * (gy * my + side * (int64_t)(gz * mz));
            const double v = d ? re * re + im * im : 0.0;
            s2[mid + d] = (add ? s2[mid + d] : 0.0) + v;
            if (mx) s2[mid - d] = (add ? s2[mid - d] : 0.0) + v;
        }
}

thread_local std::string g_lat_err;

}  // namespace

LatGeom lat_geometry(const int M[3], int64_t n)
{
    LatGeom g{};
    for (int d = 0; d < 3; ++d) g.M[d] = M[d];
    g.B = 2 * M[1] + 1;
    g.C = 2 * M[2] + 1;
    g.R = (int64_t)(2 * M[0] + 1) * g.B;
    const int nct = (2 * M[2] + 15) / 16;
    g.cblk = (nct + 3) / 4;
    g.nc = (nct + g.cblk - 1) / g.cblk;
    g.rblk = (int)((g.R + kLatRows - 1) / kLatRows);
    g.ny = std::min(g.B, kLatRows);
    g.nx = std::min(2 * M[0] + 1, (kLatRows - 1) / g.B + 2);
    g.lds = ((size_t)(g.nx + g.ny + 16 * g.nc) * kLatStride +
             (size_t)4 * kLatBase * kLatStage + (size_t)7 * kLatLoad) * sizeof(double);
    static_assert(kLatBase == 8 && kLatLoad == 256, "kLatMaxLds");
    // atom slices: one round of two workgroups per CU (a second, partial round would leave
    // CUs idle), while the partial sums stay bounded and a slice keeps two stages
    int64_t want = std::max<int64_t>(1, kLatTargetWg / ((int64_t)g.rblk * g.cblk));
    want = std::min(want, std::max<int64_t>(1, kLatMaxPart / g.sums()));
    want = std::min(want, std::max<int64_t>(1, n / (2 * kLatStage)));
    g.max_slices = (int)want;
    const int64_t per = (n + want - 1) / want;
    g.aps = (int)std::max<int64_t>(kLatStage, (per + kLatStage - 1) / kLatStage * kLatStage);
    g.slices = (int)std::max<int64_t>(1, (n + g.aps - 1) / g.aps);
    return g;
}

// f(kernel of the geometry's column tiles)
template <class F>
static auto lat_kernel(const LatGeom& g, F f)
{
    switch (g.nc) {
    case 1: return f(k_lat_sums<1>);
    case 2: return f(k_lat_sums<2>);
    case 3: return f(k_lat_sums<3>);
    default: return f(k_lat_sums<4>);
    }
}

hipError_t lattice_sums_prepare(const LatGeom& g)
{
    if (g.lds <= 65536) return hipSuccess;  // what any kernel may have
    return lat_kernel(g, [](auto kern) {
        return hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)kLatMaxLds);
    });
}

void launch_lattice_sums(const LatGeom& g, const Box& box, int64_t n, const double* x,
                         const double* y, const double* z, const double* q, double* part,
                         hipStream_t s)
{
    const LatSumArgs a{x, y, z, q, n, box, g, part};
    const dim3 grid(g.rblk, g.cblk, g.slices);
    lat_kernel(g, [&](auto kern) { kern<<<grid, 256, g.lds, s>>>(a); });
    if (g.slices > 1)
        k_lat_reduce<<<(unsigned)((g.sums() + 255) / 256), 256, 0, s>>>(part, g.sums(), g.slices);
}

}  // namespace rbmd

using namespace rbmd;

extern "C" {

const char* rbmd_lattice_last_error(void) { return g_lat_err.c_str(); }

static int lat_fail(int code, const std::string& msg)
{
    g_lat_err = msg;
    return code;
}

// The lattice box and atom count that both entry points take.
static int lat_check(int64_t n, int32_t Mg)
{
    if (Mg < 1 || Mg > 1024) return lat_fail(RBMD_ERR_INVALID, "Mg must be in [1, 1024]");
    if (n < 0 || n > (int64_t)INT32_MAX / 2)
        return lat_fail(RBMD_ERR_INVALID, "n must be in [0, 2^30)");
    return RBMD_OK;
}

int64_t rbmd_lattice_spectrum_workspace(int64_t n, int32_t Mg)
{
    g_lat_err.clear();
    if (lat_check(n, Mg) != RBMD_OK) return -1;
    const int M[3] = {Mg, Mg, Mg};
    const LatGeom g = lat_geometry(M, n);
    return (int64_t)g.slices * g.sums() * (int64_t)sizeof(double);
}

int rbmd_lattice_spectrum(const double* box_lo, const double* box_len, int64_t n, const double* x,
                          const double* y, const double* z, const double* q, int32_t Mg,
                          int32_t accumulate, double* s2, void* workspace, int64_t bytes,
                          void* stream)
{
    g_lat_err.clear();
    const int rc = lat_check(n, Mg);
    if (rc != RBMD_OK) return rc;
    if (!box_lo || !box_len || !s2 || !workspace || (n > 0 && (!x || !y || !z || !q)))
        return lat_fail(RBMD_ERR_INVALID, "null pointer");
    Box box;
    for (int d = 0; d < 3; ++d) {
        if (!(box_len[d] > 0)) return lat_fail(RBMD_ERR_INVALID, "box lengths must be positive");
        box.lo[d] = box_lo[d];
        box.L[d] = box_len[d];
        box.invL[d] = 1.0 / box_len[d];
    }
    const int M[3] = {Mg, Mg, Mg};
    const LatGeom g = lat_geometry(M, n);
    if (bytes < (int64_t)g.slices * g.sums() * (int64_t)sizeof(double))
        return lat_fail(RBMD_ERR_CAPACITY, "workspace smaller than rbmd_lattice_spectrum_workspace");
    hipError_t st = lattice_sums_prepare(g);
    if (st != hipSuccess)
        return lat_fail(RBMD_ERR_HIP, std::string("dynamic LDS: ") + hipGetErrorString(st));
    hipStream_t s = (hipStream_t)stream;
    launch_lattice_sums(g, box, n, x, y, z, q, (double*)workspace, s);
    const int64_t pts = (int64_t)(Mg + 1) * (Mg + 1) * (Mg + 1);
    k_lat_spectrum<<<(unsigned)((pts + 255) / 256), 256, 0, s>>>((const double*)workspace, g.B, g.C,
                                                              Mg, accumulate, s2);
    st = hipGetLastError();
    if (st != hipSuccess)
        return lat_fail(RBMD_ERR_HIP, std::string("launch: ") + hipGetErrorString(st));
    return RBMD_OK;
}

}  // extern "C"
