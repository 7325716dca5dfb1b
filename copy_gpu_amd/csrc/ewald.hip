// ewald.hip -- full Ewald in FP64 on the lattice box that holds its k-list: the structure
// factor from the lattice sums (lattice.h), and the k-space force by the transposed matrix
// products.
//
// Reference (paths relative to the reference checkout):
//   rho(k)                 rbmd/framework/run/worklet/RunWorklet.cpp:1616-1677
//   Ewald force / energy   rbmd/framework/forceFunction/ExecForceFunction.h:226-245
//
// With A_k, B_k the force coefficients, F_i = q_i grad Psi(r_i),
//   Psi(r) = sum_k A_k sin(k.r) + B_k cos(k.r) = sum_abc D[a,b][c] e_a(x) e_b(y) e_c(z)
// in the basis of the sums, so that
//   H[a,b](i) = sum_c D[a,b][c] e_c(z_i),    H'[a,b](i) = sum_c D[a,b][c] e_c'(z_i)
// are matrix products, and F_x = q sum e_a' e_b H, F_y = q sum e_a e_b' H, F_z = q sum e_a e_b H'.
#include <algorithm>
#include <vector>

#include "kspace.h"
#include "lattice.h"
#include "state.h"

namespace rbmd {

namespace {

// rho, per-k terms and coefficients of the k-list, and D, from the sums: one thread per
// octant point; idx[point][class] is the list index of (m_x, +-m_y, +-m_z) or -1.
__global__ __launch_bounds__(256) void k_ewald_final(RhoFinalArgs<double> A,
                                                     const double* __restrict__ T, EwaldLat l)
{
    const int64_t o = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int hy = l.M[1] + 1, hz = l.M[2] + 1;
    if (o >= (int64_t)(l.M[0] + 1) * hy * hz) return;
    const int mz = (int)(o % hz), my = (int)(o / hz % hy), mx = (int)(o / ((int64_t)hy * hz));
    const int B = 2 * l.M[1] + 1, C = 2 * l.M[2] + 1;
    const LatOct t = lat_octant(T, B, C, mx, my, mz);
    double D[8] = {};
    for (int cl = 0; cl < 4; ++cl) {
        const int k = l.idx[o * 4 + cl];
        if (k < 0) continue;
        const double gy = cl & 2 ? -1.0 : 1.0, gz = cl & 1 ? -1.0 : 1.0;
        double re, im;
        lat_rho(t, gy, gz, &re, &im);
        const KCoef<double> kc = rho_final_emit<double, false>(A, k, re, im);
        D[0] += kc.B;
        D[6] -= gy * kc.B;
        D[5] -= gz * kc.B;
        D[3] -= gy * gz * kc.B;
        D[4] += kc.A;
        D[2] += gy * kc.A;
        D[1] += gz * kc.A;
        D[7] -= gy * gz * kc.A;
    }
    for (int k = 0; k < 8; ++k) {
        const int sx = k >> 2, sy = (k >> 1) & 1, sz = k & 1;
        if ((sx && !mx) || (sy && !my) || (sz && !mz)) continue;
        const int a = sx ? lat_sin(mx) : lat_cos(mx), b = sy ? lat_sin(my) : lat_cos(my),
                  c = sz ? lat_sin(mz) : lat_cos(mz);
        l.D[ewald_d_pos(l, a * B + b, c)] = D[k];
    }
}

// Forces of 64 atoms (16 per wave) from a share of the row tiles.  The z basis and its
// derivative of the wave's atoms stay in registers (64 columns c at a time) and are the B
// operands of v_mfma_f64_16x16x4_f64; D comes in fragment order, 16 bytes per lane for two
// steps.  Of a tile only the steps inside the Ewald sphere are run, and the shares hold equal
// numbers of steps.  The x and y bases are in LDS: y for every m_y, x for kEwX values of m_x
// at a time.
//
// Bound by FP64 issue, two matrix instructions of 64 cycles per 4 columns and 16 rows.  6,000
// ions, 52,800 k-vectors (|m| <= 29): 95 us, and 79 us for the sums; 2,020 and 706 us with a
// sine and cosine per (k, atom).  The matrix cores are busy 58% of the cycles in both.
constexpr int kEwAtoms = 64;
constexpr int kEwStride = 80;  // doubles between table rows: two rows on disjoint banks
constexpr int kEwX = 8;        // m_x held at a time (a tile of 16 rows spans at most 5)
constexpr int kEwMaxLds = 140 * 1024;
// Fewest k-vectors that take the lattice: it has two to three launches more, and its sums and
// forces fill 256-row and 64-column tiles whatever the box.  An evaluation without and with it,
// us: 4,000 ions 29 and 58 for 46 k-vectors, 45 and 61 for 447, 70 and 67 for 1,051; 100,000
// ions 334 and 358 for 459, 537 and 381 for 1,051; 64 ions 42 and 43 for 459, 62 and 49 for 1,051.
constexpr int kEwMinK = 800;

struct EwForceArgs {
    const double *x, *y, *z;
    int n;
    Box box;
    EwaldLat l;
    int split;
    double* fpart;  // [split][3][n]
};

__device__ inline int ew_share(const EwaldLat& l, int s, int split)
{
    const int64_t want = (int64_t)l.steps * s / split;
    int lo = 0, hi = l.ntile;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (l.before[mid] < want) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(256, 3) void k_ewald_force(EwForceArgs A)
{
    extern __shared__ double ew_lds[];
    const EwaldLat& l = A.l;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, kl = lane >> 4, al = lane & 15;
    const int B = 2 * l.M[1] + 1, C = 2 * l.M[2] + 1;
    // rows of basis value a at a + 1, so the cosine and sine of m are at 2 m and 2 m + 1 (each
    // the other's derivative) and the constant at 1
    double* Yt = ew_lds;
    double* Xt = Yt + (size_t)2 * (l.M[1] + 1) * kEwStride;  // from m0 on
    const int t0 = ew_share(l, blockIdx.y, A.split),
              t1 = (int)blockIdx.y + 1 == A.split ? l.ntile : ew_share(l, blockIdx.y + 1, A.split);
    constexpr double kTwoPi = 2.0 * kPi;

    // tables: thread -> atom t % 64, every fourth m
    const int ta = blockIdx.x * kEwAtoms + (t & 63), tg = t >> 6;
    const int tc = ta < A.n ? ta : A.n - 1;
    const LatFrac fx = lat_frac(A.x[tc] - A.box.lo[0], A.box.L[0], A.box.invL[0]);
    {
        const LatFrac fy = lat_frac(A.y[tc] - A.box.lo[1], A.box.L[1], A.box.invL[1]);
        double c4, s4, cs, sn;
        lat_sincos(fy, 4, &s4, &c4);
        lat_sincos(fy, tg, &sn, &cs);
        for (int m = tg; m <= l.M[1]; m += 4) {
            Yt[(2 * m) * kEwStride + (t & 63)] = m ? cs : 0.0;
            Yt[(2 * m + 1) * kEwStride + (t & 63)] = m ? sn : 1.0;
            const double c = fma(cs, c4, -(sn * s4));
            sn = fma(sn, c4, cs * s4);
            cs = c;
        }
    }
    // this lane's atom in the products
    const int la = wv * 16 + al, ia = blockIdx.x * kEwAtoms + la;
    const int ic = ia < A.n ? ia : A.n - 1;
    const LatFrac fz = lat_frac(A.z[ic] - A.box.lo[2], A.box.L[2], A.box.invL[2]);
    double F0 = 0.0, F1 = 0.0, F2 = 0.0;
    for (int kb = 0; kb * 64 < C; ++kb) {
        // columns c = 64 kb + 4 s + kl of the basis, m = (c + 1) / 2: the lane keeps to cosines
        // or sines, and m advances by 2 from step to step
        double Z[16], Zd[16];
        {
            const int m0 = 32 * kb + (kl + 1) / 2;
            const bool sine = (kl & 1) == 0;  // c even: sine (c = 0: the constant)
            double c2, s2, cs, sn;
            lat_sincos(fz, 2, &s2, &c2);
            lat_sincos(fz, m0, &sn, &cs);
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const double k = (double)(m0 + 2 * s);
                Z[s] = sine ? (m0 + 2 * s ? sn : 1.0) : cs;
                Zd[s] = sine ? k * cs : -(k * sn);
                const double c = fma(cs, c2, -(sn * s2));
                sn = fma(sn, c2, cs * s2);
                cs = c;
            }
        }
        for (int tb = t0; tb < t1;) {
            // rows of tb .. te - 1 use m_x = m0 .. m0 + kEwX - 1
            const int m0 = (tb * 16 / B + 1) >> 1;
            const int te = min(t1, max(tb + 1, (2 * (m0 + kEwX - 1) + 1) * B / 16));
            __syncthreads();
            for (int j = tg; j < kEwX; j += 4) {
                double sn, cs;
                lat_sincos(fx, m0 + j, &sn, &cs);
                Xt[(2 * j) * kEwStride + (t & 63)] = m0 + j ? cs : 0.0;
                Xt[(2 * j + 1) * kEwStride + (t & 63)] = m0 + j ? sn : 1.0;
            }
            __syncthreads();
            for (int tl = tb; tl < te; ++tl) {
                const int np = l.pairs[kb * l.ntile + tl];
                if (np == 0) continue;
                const double2* Dp =
                    (const double2*)(l.D + ((int64_t)kb * l.ntile + tl) * 1024) + lane;
                const int4 rw = ((const int4*)l.rows)[tl * 4 + kl];
                d4 h = {0.0, 0.0, 0.0, 0.0}, hd = {0.0, 0.0, 0.0, 0.0};
                // four pairs of steps at a time, their loads in flight together
#pragma unroll
                for (int p0 = 0; p0 < 8; p0 += 4) {
                    if (p0 >= np) break;
                    double2 d[4];
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        if (p0 + p < np) d[p] = Dp[(p0 + p) * 64];
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        if (p0 + p >= np) break;
                        const int s = 2 * (p0 + p);
                        h = __builtin_amdgcn_mfma_f64_16x16x4f64(d[p].x, Z[s], h, 0, 0, 0);
                        hd = __builtin_amdgcn_mfma_f64_16x16x4f64(d[p].x, Zd[s], hd, 0, 0, 0);
                        h = __builtin_amdgcn_mfma_f64_16x16x4f64(d[p].y, Z[s + 1], h, 0, 0, 0);
                        hd = __builtin_amdgcn_mfma_f64_16x16x4f64(d[p].y, Zd[s + 1], hd, 0, 0, 0);
                    }
                }
                const int rv[4] = {rw.x, rw.y, rw.z, rw.w};
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // table rows of the x and y values of row 4 v + kl; derivatives without 2 pi / L
                    const int ix = rv[v] & 0xffff, iy = rv[v] >> 16;
                    const double* xp = Xt + la - 2 * m0 * kEwStride;
                    const double X = xp[ix * kEwStride], Xp = xp[(ix ^ 1) * kEwStride];
                    const double Y = Yt[iy * kEwStride + la], Yp = Yt[(iy ^ 1) * kEwStride + la];
                    const double Xd = (double)(ix & 1 ? ix >> 1 : -(ix >> 1)) * Xp,
                                 Yd = (double)(iy & 1 ? iy >> 1 : -(iy >> 1)) * Yp;
                    F0 = fma(Xd, Y * h[v], F0);
                    F1 = fma(Yd, X * h[v], F1);
                    F2 = fma(X * Y, hd[v], F2);
                }
            }
            tb = te;
        }
    }
    // the four row groups of an atom
    F0 += __shfl_xor(F0, 16, 64);
    F1 += __shfl_xor(F1, 16, 64);
    F2 += __shfl_xor(F2, 16, 64);
    F0 += __shfl_xor(F0, 32, 64);
    F1 += __shfl_xor(F1, 32, 64);
    F2 += __shfl_xor(F2, 32, 64);
    if (kl == 0 && ia < A.n) {
        double* o = A.fpart + (int64_t)blockIdx.y * 3 * A.n + ia;
        o[0] = kTwoPi / A.box.L[0] * F0;
        o[(int64_t)A.n] = kTwoPi / A.box.L[1] * F1;
        o[(int64_t)2 * A.n] = kTwoPi / A.box.L[2] * F2;
    }
}

// f += q times the shares in order (a random batch list's mean near force leaves first).
__global__ __launch_bounds__(256) void k_ewald_add(const double* __restrict__ fpart, int split,
                                                   const double* __restrict__ q, int n,
                                                   const double* __restrict__ rbl_mean,
                                                   double* __restrict__ fx,
                                                   double* __restrict__ fy,
                                                   double* __restrict__ fz)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double* f[3] = {fx, fy, fz};
    for (int d = 0; d < 3; ++d) {
        double v = 0.0;
#pragma unroll 8
        for (int s = 0; s < split; ++s) v += fpart[((int64_t)s * 3 + d) * n + i];
        double b = f[d][i];
        if (rbl_mean) b -= rbl_mean[d];
        f[d][i] = b + q[i] * v;
    }
}

// Shares of the row tiles: three workgroups per CU, as registers and LDS allow, in one
// dispatch round.
int ewald_split(const EwaldLat& l, int64_t n)
{
    const int64_t groups = (n + kEwAtoms - 1) / kEwAtoms;
    return (int)std::max<int64_t>(1, std::min<int64_t>(768 / std::max<int64_t>(groups, 1),
                                                       l.ntile));
}

size_t ewald_lds(const EwaldLat& l)
{
    return (size_t)(2 * (l.M[1] + 1) + 2 * kEwX) * kEwStride * sizeof(double);
}

}  // namespace

void ewald_free(Engine& e)
{
    EwaldLat& l = e.ew;
    if (l.rows) hipFree(l.rows);  // the one block
    l = EwaldLat{};
}

// m: the k-list [P][3], m_x >= 0, at most one of k and -k.
hipError_t ewald_setup(Engine& e, const std::vector<int32_t>& m)
{
    EwaldLat& l = e.ew;
    if (m.size() / 3 < kEwMinK) return hipSuccess;
    for (size_t k = 0; k < m.size(); ++k) l.M[k % 3] = std::max(l.M[k % 3], std::abs(m[k]));
    for (int d = 0; d < 3; ++d) l.M[d] = std::max(l.M[d], 1);
    // the y basis of 64 atoms has to fit the LDS: boxes beyond (|m_y| > 103) keep the sums
    // over single k-vectors
    const int lds = std::min(e.lds_max, kEwMaxLds);
    if (ewald_lds(l) > (size_t)lds || e.n_max < 1) return hipSuccess;
    const int B = 2 * l.M[1] + 1, C = 2 * l.M[2] + 1;
    const int64_t R = (int64_t)(2 * l.M[0] + 1) * B;
    const int hy = l.M[1] + 1, hz = l.M[2] + 1;
    l.ntile = (int)((R + 15) / 16);
    const int nkb = (C + 63) / 64;
    std::vector<int32_t> idx((size_t)(l.M[0] + 1) * hy * hz * 4, -1);
    std::vector<int32_t> top((size_t)(l.M[0] + 1) * hy, -1);  // largest |m_z| of (m_x, |m_y|)
    for (size_t k = 0; k < m.size() / 3; ++k) {
        const int a = m[3 * k], b = m[3 * k + 1], g = m[3 * k + 2];
        const size_t row = (size_t)a * hy + std::abs(b);
        idx[(row * hz + std::abs(g)) * 4 + (b < 0) * 2 + (g < 0)] = (int32_t)k;
        top[row] = std::max(top[row], std::abs(g));
    }
    // steps of a tile: pairs of 4 columns up to the largest c of its rows
    std::vector<int32_t> pairs((size_t)nkb * l.ntile), before(l.ntile);
    int64_t steps = 0;
    for (int t = 0; t < l.ntile; ++t) {
        int c = -1;
        for (int64_t r = (int64_t)t * 16; r < std::min<int64_t>(R, (int64_t)t * 16 + 16); ++r)
            c = std::max(c, 2 * top[(size_t)((r / B + 1) / 2) * hy + (size_t)((r % B + 1) / 2)]);
        before[t] = (int32_t)steps;
        for (int kb = 0; kb < nkb; ++kb) {
            const int np = c < 64 * kb ? 0 : std::min(8, (c - 64 * kb) / 8 + 1);
            pairs[(size_t)kb * l.ntile + t] = np;
            steps += np;
        }
    }
    l.steps = (int32_t)steps;
    int64_t fp = 0;
    for (int64_t g = 1; g <= 768 && (g - 1) * kEwAtoms < e.n_max; ++g) {
        const int64_t n = std::min<int64_t>(g * kEwAtoms, e.n_max);
        fp = std::max(fp, ewald_split(l, n) * n);
    }
    fp = std::max<int64_t>(fp, e.n_max);
    const LatGeom g = lat_geometry(l.M, e.n_max);
    // one block: the tables (uploaded together), D, the sums and the force shares
    // table rows of every tile row, in the order that lanes hold them
    std::vector<int32_t> rows((size_t)l.ntile * 16);
    for (size_t t = 0; t < rows.size() / 16; ++t)
        for (int k = 0; k < 16; ++k) {
            const int64_t r = std::min<int64_t>(R - 1, (int64_t)t * 16 + 4 * (k & 3) + (k >> 2));
            rows[t * 16 + k] = (int32_t)((r / B + 1) | (r % B + 1) << 16);
        }
    std::vector<int32_t> tab(rows);
    tab.insert(tab.end(), idx.begin(), idx.end());
    tab.insert(tab.end(), pairs.begin(), pairs.end());
    tab.insert(tab.end(), before.begin(), before.end());
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t dbytes = (size_t)nkb * l.ntile * 1024 * sizeof(double);
    const size_t od = up(tab.size() * 4), op = od + dbytes,
                 of = op + up((size_t)g.max_slices * g.sums() * 8);
    char* m0 = nullptr;
    hipError_t st;
    if (hipMalloc((void**)&m0, of + (size_t)fp * 3 * 8) != hipSuccess) {
        (void)hipGetLastError();  // no memory for it: the sums over single k-vectors need less
        return hipSuccess;
    }
    l.rows = (int32_t*)m0;
    l.idx = l.rows + rows.size();
    l.pairs = l.idx + idx.size();
    l.before = l.pairs + pairs.size();
    l.D = (double*)(m0 + od);
    l.part = (double*)(m0 + op);
    l.fpart = (double*)(m0 + of);
    if ((st = hipMemcpy(m0, tab.data(), tab.size() * 4, hipMemcpyHostToDevice)) != hipSuccess ||
        (st = hipMemset(l.D, 0, dbytes)) != hipSuccess ||
        (st = lattice_sums_prepare(g)) != hipSuccess ||
        // (the limit belongs to the kernel, not to this handle: always the bound above)
        (st = hipFuncSetAttribute((const void*)k_ewald_force,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds)) != hipSuccess)
        return st;
    l.on = true;
    return hipSuccess;
}

void launch_ewald_rho(Engine& e, const double* x, const double* y, const double* z,
                      hipStream_t s)
{
    const EwaldLat& l = e.ew;
    {
        ScopedTimer t(e, P_RHO, s);
        launch_lattice_sums(lat_geometry(l.M, e.n), e.box, e.n, x, y, z, e.q, l.part, s);
    }
    ScopedTimer t(e, P_RHO_FINAL, s);
    const int64_t pts = (int64_t)(l.M[0] + 1) * (l.M[1] + 1) * (l.M[2] + 1);
    k_ewald_final<<<(unsigned)((pts + 255) / 256), 256, 0, s>>>(
        rho_final_args<double>(e, nullptr), l.part, l);
}

void launch_ewald_force(Engine& e, const double* x, const double* y, const double* z, double* fx,
                        double* fy, double* fz, hipStream_t s)
{
    const EwaldLat& l = e.ew;
    ScopedTimer t(e, P_KFORCE, s);
    const int n = (int)e.n, split = ewald_split(l, n);
    const dim3 grid((n + kEwAtoms - 1) / kEwAtoms, split);
    k_ewald_force<<<grid, 256, ewald_lds(l), s>>>(
        EwForceArgs{x, y, z, n, e.box, l, split, l.fpart});
    k_ewald_add<<<(n + 255) / 256, 256, 0, s>>>(l.fpart, split, e.q, n,
                                                e.rbl ? e.rbl_mean : nullptr, fx, fy, fz);
}

}  // namespace rbmd
