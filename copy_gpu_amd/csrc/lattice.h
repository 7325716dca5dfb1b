// lattice.h -- structure factor on a whole lattice box |m_d| <= M_d in FP64.
//
// exp(2 pi i m.s) factors into one phase per axis, so rho(m) of every m of the box is a
// matrix product over the atoms instead of one sine and cosine per (m, atom).  In real
// arithmetic, with the per-axis basis e_0 = 1, e_(2m-1) = cos(2 pi m s), e_(2m) =
// sin(2 pi m s), the sums
//   T[a, b][c] = sum_j q_j e_a(x_j) e_b(y_j) e_c(z_j),   a <= 2 M_x, b <= 2 M_y, c <= 2 M_z
// hold rho of (m_x, +-m_y, +-m_z) as combinations of eight of them, with half the products
// of the complex form.  Rows are (a, b), columns c, and the contraction runs over atoms.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "engine.h"

namespace rbmd {

constexpr int kLatRows = 256;    // rows of one workgroup: 4 waves x 4 row tiles of 16
constexpr int kLatStage = 32;    // atoms per LDS stage
constexpr int kLatStride = 34;   // doubles between rows of a table: the 16 rows x 2 atoms of
                                 // half a fragment fall on all 64 banks once
constexpr int kLatTargetWg = 512;  // two workgroups per CU on the 256 CUs of an MI355X
constexpr int64_t kLatMaxPart = (int64_t)1 << 26;  // most doubles of the partial sums

// Position of cos / sin of m in an axis basis.
RBMD_HD inline int lat_cos(int m) { return m ? 2 * m - 1 : 0; }
RBMD_HD inline int lat_sin(int m) { return 2 * m; }  // m >= 1

struct LatGeom {
    int M[3];
    int B, C;              // basis sizes of the y and z axes
    int64_t R;             // rows (2 M_x + 1) B
    int nc, rblk, cblk;    // 16-column tiles per workgroup; row and column blocks
    int nx, ny;            // LDS table rows of the x and y axes
    int slices, aps;       // atom slices and atoms per slice
    int max_slices;        // most slices of any atom count up to this one
    size_t lds;
    RBMD_HD int64_t sums() const { return R * (int64_t)C; }
};

// LDS that a sums kernel may be launched with: 256 rows touch at most 258 rows of the x and y
// tables together.  The limit is a property of the kernel, shared by every caller, so it is set
// to this bound and never to one call's need.
constexpr size_t kLatMaxLds = ((size_t)(kLatRows + 2 + 64) * kLatStride + 4 * 8 * kLatStage +
                               7 * 256) * sizeof(double);

LatGeom lat_geometry(const int M[3], int64_t n);

// Allows the sums kernel of a geometry its LDS; once per device before launch_lattice_sums (it
// may be called again at any time).
hipError_t lattice_sums_prepare(const LatGeom& g);

// T of every slice into part [slices][R][C], then their sum in slice order into part[0].
void launch_lattice_sums(const LatGeom& g, const Box& box, int64_t n, const double* x,
                         const double* y, const double* z, const double* q, double* part,
                         hipStream_t s);

// Full Ewald of a handle on its lattice box (ewald.hip).
struct EwaldLat {
    bool on = false;
    int M[3] = {0, 0, 0};
    int ntile = 0;               // 16-row tiles of the (a, b) rows
    int32_t steps = 0;           // pairs of 4-column steps over all tiles
    // one block of device memory, from rows on
    int32_t* rows = nullptr;     // [tile][row % 4][row / 4]: a + 1, b + 1 of the row
    int32_t* idx = nullptr;      // [octant point][4] k-list index or -1
    int32_t* pairs = nullptr;    // [64-column block][tile] pairs of steps
    int32_t* before = nullptr;   // [tile] pairs of steps before the tile
    double* D = nullptr;         // force coefficients in fragment order
    double* part = nullptr;      // lattice sums
    double* fpart = nullptr;     // force shares
};

// Position of D[row][c]: per 64-column block and tile, lane (c % 4) 16 + row % 16 holds its
// value of step (c % 64) / 4, two steps side by side.
RBMD_HD inline int64_t ewald_d_pos(const EwaldLat& l, int row, int c)
{
    const int s = (c & 63) >> 2, lane = (c & 3) * 16 + (row & 15);
    return ((int64_t)(c >> 6) * l.ntile + (row >> 4)) * 1024 + (s >> 1) * 128 + lane * 2 + (s & 1);
}

#ifdef __HIPCC__
using d4 = double __attribute__((ext_vector_type(4)));

// Fraction s = t / L of a box edge as an unevaluated sum hi + lo, and the sine and cosine of
// m s turns, the phase reduced exactly up to the rounding of the reduced value.
struct LatFrac {
    double hi, lo;
};
__device__ inline LatFrac lat_frac(double t, double L, double invL)
{
    const double h = t * invL;
    return {h, fma(-h, L, t) * invL};
}
__device__ inline void lat_sincos(const LatFrac& s, int m, double* sn, double* cs)
{
    const double md = (double)m, p = md * s.hi;
    const double f = (p - rint(p)) + (fma(md, s.hi, -p) + md * s.lo);
    sincospi(2.0 * f, sn, cs);
}

// The eight sums of an octant point, axes x, y, z as bits 2, 1, 0 (1: sine).
struct LatOct {
    double t[8];
};
__device__ inline LatOct lat_octant(const double* __restrict__ T, int B, int C, int mx, int my,
                                    int mz)
{
    LatOct o;
    for (int k = 0; k < 8; ++k) {
        const int sx = k >> 2, sy = (k >> 1) & 1, sz = k & 1;
        const bool ok = (!sx || mx) && (!sy || my) && (!sz || mz);
        const int a = sx ? lat_sin(mx) : lat_cos(mx), b = sy ? lat_sin(my) : lat_cos(my),
                  c = sz ? lat_sin(mz) : lat_cos(mz);
        o.t[k] = ok ? T[((int64_t)a * B + b) * C + c] : 0.0;
    }
    return o;
}
// rho(mx, gy my, gz mz), gy and gz = +-1.
__device__ inline void lat_rho(const LatOct& o, double gy, double gz, double* re, double* im)
{
    *re = o.t[0] - gy * o.t[6] - gz * o.t[5] - gy * gz * o.t[3];
    *im = o.t[4] + gy * o.t[2] + gz * o.t[1] - gy * gz * o.t[7];
}
#endif

}  // namespace rbmd
