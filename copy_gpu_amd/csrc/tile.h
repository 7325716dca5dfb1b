// tile.h -- cell tiles shared by the Verlet-list build and the pair pass.
//
// A tile is one home cell c plus its 27-cell periodic stencil.  The stencil's
// atoms (cell-sorted, so each stencil cell is one contiguous range) are
// concatenated in stencil order st = 9(a+1) + 3(b+1) + (g+1), a,b,g in {-1,0,1};
// a candidate's position in that concatenation is its tile-local index u.
// Verlet rows store u as uint16, and the whole concatenation is staged in LDS
// once per workgroup, so the pair pass reads neighbour positions from LDS.
// Each stencil cell carries the periodic image shift s (k L, k in {-1,0,1})
// such that x_j - s is the image of x_j next to the home cell.
#pragma once
#include <type_traits>

#include "engine.h"

namespace rbmd {

constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kHomeSeg = 13;  // stencil slot of the home cell (a = b = g = 0)

struct TileHdr {
    int off[28];     // segment offsets in the concatenation, off[27] = total
    int gstart[27];  // first cell-sorted index of each segment
    int cnt[27];
    double sx[27], sy[27], sz[27];
    double4 dummy;   // position of the row sentinel `total`: beyond every cutoff, charge 0
};

#ifdef __HIPCC__
// Fill the tile header of home cell c (all threads of the block call it).
__device__ inline void tile_setup(int c, int3 dims, const Box& box,
                                  const int32_t* __restrict__ cell_start, TileHdr& h)
{
    const int t = threadIdx.x;
    if (t < 64) {
        int cnt = 0;
        if (t < 27) {
            const int cz = c / (dims.x * dims.y);
            const int cy = (c / dims.x) % dims.y;
            const int cx = c % dims.x;
            int ax = cx + t / 9 - 1, ay = cy + (t / 3) % 3 - 1, az = cz + t % 3 - 1;
            double sx = 0.0, sy = 0.0, sz = 0.0;
            if (ax < 0) { ax += dims.x; sx = box.L[0]; }
            else if (ax >= dims.x) { ax -= dims.x; sx = -box.L[0]; }
            if (ay < 0) { ay += dims.y; sy = box.L[1]; }
            else if (ay >= dims.y) { ay -= dims.y; sy = -box.L[1]; }
            if (az < 0) { az += dims.z; sz = box.L[2]; }
            else if (az >= dims.z) { az -= dims.z; sz = -box.L[2]; }
            const int cc = ax + ay * dims.x + az * dims.x * dims.y;
            const int g0 = cell_start[cc];
            cnt = cell_start[cc + 1] - g0;
            h.gstart[t] = g0;
            h.cnt[t] = cnt;
            h.sx[t] = sx;
            h.sy[t] = sy;
            h.sz[t] = sz;
        }
        // wave-level inclusive scan of the 27 segment sizes
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if (t >= o) incl += v;
        }
        if (t < 27) h.off[t] = incl - cnt;
        if (t == 26) h.off[27] = incl;
        if (t == 0)
            h.dummy = make_double4(box.lo[0] + 8.0 * box.L[0] + 64.0,
                                   box.lo[1] + 8.0 * box.L[1] + 64.0,
                                   box.lo[2] + 8.0 * box.L[2] + 64.0, 0.0);
    }
    __syncthreads();
}

// ---------------------------------------------------------------- binning
// Wrap into the box (x - L floor((x-lo)/L), no contraction: the CPU oracle
// computes the same bits) and the cell trunc((x-lo)/cell), clamped.
__device__ inline int wrap_cell(const double p[3], const Box& box, int3 dims, double3 cell,
                                double w[3])
{
#pragma clang fp contract(off)
    const int dm[3] = {dims.x, dims.y, dims.z};
    const double cs[3] = {cell.x, cell.y, cell.z};
    int c[3];
    for (int d = 0; d < 3; ++d) {
        double f = floor((p[d] - box.lo[d]) / box.L[d]);
        double fl = f * box.L[d];
        w[d] = p[d] - fl;
        int v = (int)((w[d] - box.lo[d]) / cs[d]);
        v = v < 0 ? 0 : v;
        v = v > dm[d] - 1 ? dm[d] - 1 : v;
        c[d] = v;
    }
    return c[0] + c[1] * dims.x + c[2] * dims.x * dims.y;
}

// Wave-aggregated binning for lanes that mostly share one cell (the home atoms
// of a tile): one atomic per distinct cell of the wave, ranks by ballot order.
// Atom v sits in slot s.  Every lane of the wave calls it; inactive lanes bin
// nothing.
__device__ inline void md_bin_wave(const MdBins& b, int buf, bool active, int s, int v,
                                   const double p[3], const Box& box, int3 dims, double3 cell)
{
    int c = -1;
    if (active) {
        double w[3];
        c = wrap_cell(p, box, dims, cell, w);
        b.cell[s] = c;
        b.vid[s] = v;
        b.xw[s] = w[0];
        b.yw[s] = w[1];
        b.zw[s] = w[2];
    }
    const int lane = (int)__lane_id();
    uint64_t pending = __ballot(active);
    while (pending != 0ull) {
        const int leader = __ffsll((unsigned long long)pending) - 1;
        const int cl = __shfl(c, leader, 64);
        const uint64_t grp = __ballot(c == cl) & pending;
        int base = 0;
        if (lane == leader) {
            base = atomicAdd(&b.count[buf * b.ncell + cl], __popcll(grp));
            if (b.nchunk > 0) atomicAdd(&b.chunk[buf * b.nchunk + cl / kBinChunk], __popcll(grp));
        }
        base = __shfl(base, leader, 64);
        if ((grp >> lane) & 1ull) {
            const int rank = base + (int)mbcnt64(grp);
            if (rank < b.cap) b.bucket[((size_t)buf * b.ncell + cl) * b.cap + rank] = s;
        }
        pending &= ~grp;
    }
}

// SPILL: an atom beyond its cell's bucket goes to one of the cell's lists (slot and atom are
// the same there).
template <bool SPILL = false>
__device__ inline void md_bin_atom(const MdBins& b, int buf, int s, int v, const double p[3],
                                   const Box& box, int3 dims, double3 cell)
{
    double w[3];
    const int c = wrap_cell(p, box, dims, cell, w);
    b.cell[s] = c;
    b.vid[s] = v;
    b.xw[s] = w[0];
    b.yw[s] = w[1];
    b.zw[s] = w[2];
    const int bc = buf * b.ncell + c;
    const int rank = atomicAdd(&b.count[bc], 1);
    if (rank < b.cap) b.bucket[(size_t)bc * b.cap + rank] = s;
    else if (SPILL)
        b.spill_next[v].x = atomicExch(&b.spill[(size_t)c * kSpillChains + rank % kSpillChains], v);
}

// ---------------------------------------------------------------- tile order
// Order of the tile workgroups, for load balance only (a tile's results do not
// depend on which workgroup computes it).  Used when the tiles fit about one
// dispatch round (ncell * split <= 3 ncu): then the kernel ends when its most
// loaded CU does, and the dispatcher gives workgroup t to CU t mod ncu.  The
// work of cell c is estimated as w_c = n_c x (atoms of its 27-cell stencil);
// cells are counting-sorted into kOrderBuckets classes of w, heaviest first
// (order within a class is arbitrary), and the first round takes the heaviest
// tiles in reverse order, so a CU that starts with a lighter tile receives
// heavier ones in the later rounds.  With more tiles the dispatcher balances by
// itself and the cell order (spatial, L2-friendly) is kept.  One workgroup of
// at least 256 threads runs it, ncell <= kOrderMaxCells; lds holds kOrderLds ints.
constexpr int kOrderBuckets = 256;
constexpr int kOrderMaxCells = 1024;
constexpr int kOrderLds = 2 * kOrderBuckets + 8 + 2 * kOrderMaxCells;

__device__ inline void tile_order_build(const int32_t* __restrict__ count, int ncell, int3 dims,
                                        int split, int ncu, int32_t* __restrict__ order,
                                        int32_t* lds)
{
    const int nt = (int)blockDim.x, t = (int)threadIdx.x;
    int32_t* hist = lds;
    int32_t* cur = lds + kOrderBuckets;
    int32_t* misc = lds + 2 * kOrderBuckets;  // [0] max weight, [1..4] wave sums
    int32_t* cnt = misc + 8;
    int32_t* w = cnt + kOrderMaxCells;
    for (int k = t; k < kOrderBuckets; k += nt) hist[k] = 0;
    for (int c = t; c < ncell; c += nt) cnt[c] = count[c];
    if (t == 0) misc[0] = 0;
    __syncthreads();
    int mx = 0;
    for (int c = t; c < ncell; c += nt) {
        const int cz = c / (dims.x * dims.y), cy = (c / dims.x) % dims.y, cx = c % dims.x;
        int sum = 0;
        for (int a = -1; a <= 1; ++a)
            for (int b = -1; b <= 1; ++b)
                for (int g = -1; g <= 1; ++g) {
                    const int x = (cx + a + dims.x) % dims.x, y = (cy + b + dims.y) % dims.y,
                              z = (cz + g + dims.z) % dims.z;
                    sum += cnt[x + y * dims.x + z * dims.x * dims.y];
                }
        const int wc = cnt[c] * sum;
        w[c] = wc;
        mx = wc > mx ? wc : mx;
    }
    atomicMax(&misc[0], mx);
    __syncthreads();
    const long long scale = (long long)misc[0] + 1;
    auto bucket = [&](int wc) {
        return kOrderBuckets - 1 - (int)(((long long)wc * kOrderBuckets) / scale);
    };
    for (int c = t; c < ncell; c += nt) atomicAdd(&hist[bucket(w[c])], 1);
    __syncthreads();
    // exclusive prefix over the buckets: threads [0, 256) one bucket each
    // (4 waves: wave scans, then the waves' totals)
    int v = 0, incl = 0;
    if (t < kOrderBuckets) {
        v = hist[t];
        incl = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(incl, o, 64);
            if ((t & 63) >= o) incl += u;
        }
        if ((t & 63) == 63) misc[1 + (t >> 6)] = incl;
    }
    __syncthreads();
    if (t < kOrderBuckets) {
        int off = 0;
        for (int k = 0; k < (t >> 6); ++k) off += misc[1 + k];
        cur[t] = off + incl - v;
    }
    __syncthreads();
    const int ntile = ncell * split;
    const int r0 = ncu < ntile ? ncu : ntile;
    for (int c = t; c < ncell; c += nt) {
        const int pos = atomicAdd(&cur[bucket(w[c])], 1);
        for (int p = 0; p < split; ++p) {
            const int slot = pos * split + p;
            order[slot < r0 ? r0 - 1 - slot : slot] = c * split + p;
        }
    }
}

// Whether a system's tiles get the load-balanced order (ncu passed to the
// builder) or keep the cell order (0).
inline int tile_order_ncu(int ncell, int split, int num_cu)
{
    return (ncell <= kOrderMaxCells && ncell * split <= 3 * num_cu) ? num_cu : 0;
}

// Segment holding tile-local index u (largest st with off[st] <= u; empty
// segments before it have smaller st, empty ones after it start above u).
__device__ inline int tile_seg(const TileHdr& h, int u)
{
    int lo = 0, hi = 26;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (h.off[mid] <= u)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}
// ---------------------------------------------------------------- Verlet list
// One workgroup per (home cell, part) builds the rows of its home atoms.  A
// candidate j of home atom i is kept iff (r_list^2 - d2 > 1e-4) && (d2 > 1e-4) with
// dx = (x_j - s) - x_i (s the image shift of j's stencil cell) and
// d2 = fma(dz,dz, fma(dy,dy, dx*dx)) -- the reference's operation order
// (RunWorklet.cpp:77-83) and the exact bits the CPU oracle uses.
//
// Testing every candidate of every home atom that way costs about 25 VALU
// instructions per 64 pairs, and 85% of the pairs miss.  So the squared distances are
// formed on the matrix cores in FP32, |j|^2 - 2 i.j + (|i|^2 - t) for 16 home atoms x
// 16 candidates per v_mfma_f32_16x16x4_f32 (positions relative to the home cell's
// centre): the sign bits are the hits, and those of the same values moved to the
// LJ range are its entries.  A value within rounding (list_margin) of a threshold is
// settled by the exact criterion, so the rows hold exactly the pairs that it accepts.
//
// Steps, per block of up to 4096 candidates staged in LDS (float4: position and
// |j|^2):
//   near_masks  the 8 waves share the 16-candidate chunks (wave w: chunks w T ..
//               w T + T - 1); each lane keeps one bit per chunk for its four rows of
//               every 16-row tile and stores them to LDS: 64 words per row and mask
//   row_hits    one wave per row: lane (g, column) holds the column's bits of waves 2g
//               and 2g + 1, and the wave writes one hit of every lane per trip
// A row's consecutive entries then come from different columns (u mod 16), and the
// pair pass, which gathers 16 consecutive entries at a time, reads different LDS banks.
// Tiles larger than the LDS stage are staged block by block.  Tiles beyond the 15-bit
// index range mark their rows overflowed.
//
// Bound by VALU issue: at 100,000 ions (1,229 candidates a tile, 45 rows) staging takes
// 6 us, the masks 28 us and the rows about 40 us of a rebuild's tile pass, at 0.89 vector
// instructions per CU cycle.  Against one wave per row testing every candidate in FP64: 163 ->
// 132 us (the whole pass, the pair part 47 of it), 27 -> 21 us at 2,000 ions; where the tile is
// staged in blocks (1,000 ions in a box of one cell, 27,000 candidates) 6.6 ms -> 135 us,
// with the tile split among 62 workgroups instead of four.
//
// Row layout (uint16 tile-local indices, cap slots per home atom): the LJ-range
// entries (d2 < r_in^2) first, then the others, then one sentinel slot holding
// the tile's dummy index `total` (staged far from every atom), so a reader may
// clamp its slot to the row length instead of testing it.  A row of n entries
// needs n + 1 <= cap slots; ncount = (LJ-range, other) entries, or (n, 0) with
// n >= cap for a row that did not fit.
constexpr int kInnerFlag = 0x8000;
constexpr int kMaxTile = 0x7fff;  // tile-local indices and the sentinel fit in 15 bits

__device__ inline double4 stage_ref(const TileHdr& h, const double4* __restrict__ xs_ref, int u)
{
#pragma clang fp contract(off)
    const int st = tile_seg(h, u);
    const double4 p = xs_ref[h.gstart[st] + (u - h.off[st])];
    return make_double4(p.x - h.sx[st], p.y - h.sy[st], p.z - h.sz[st], p.w);
}

constexpr int kListBlock = 4096;  // most candidates of one block (32 chunks per wave)
constexpr int kMaskRow = 256;     // bytes of a row's mask (64 uint32 words)

// Staged candidates of a build: whole 16-candidate chunks.
__host__ __device__ inline int list_len(int stage_cap) { return (stage_cap + 15) / 16 * 16; }

// Row buffers of a build, one per wave.  Rows of more than 8,192 entries leave room for seven
// beside the smallest stage and its masks (up to the 9,600 entries that handles accept); the
// last wave then writes no rows.
__host__ __device__ inline int list_bufs(int cap)
{
    return cap <= 8192 ? kTileWaves : kTileWaves - 1;
}

// Rows of one mask group (a multiple of 16): as many as fit beside the candidates in
// the LDS that the pair pass's stage takes anyway (pass_bytes), between 32 and 64.
inline size_t list_fixed_bytes(int stage_cap, int cap, bool rbl)
{
    return (size_t)(rbl ? 20 : 16) * (size_t)list_len(stage_cap) +
           (size_t)list_bufs(cap) * (size_t)cap * sizeof(uint16_t);
}
inline int list_rows(int stage_cap, int cap, size_t pass_bytes, bool rbl)
{
    const size_t c = list_fixed_bytes(stage_cap, cap, rbl);
    const size_t fit = pass_bytes > c ? (pass_bytes - c) / (2 * kMaskRow) : 0;
    return fit >= 64 ? 64 : fit < 48 ? 32 : 48;
}

// LDS bytes of the list build: the candidates (and, for a random batch list, their atom
// ids), the row buffers of cap entries and two masks of `rows` rows.
inline size_t list_lds_bytes(int stage_cap, int cap, int rows = 32, bool rbl = false)
{
    return list_fixed_bytes(stage_cap, cap, rbl) + 2 * kMaskRow * (size_t)rows;
}

struct ListLds {
    float4* cand;    // [list_len]
    char* mask;      // two masks, mask_bytes apart: hits, then their LJ-range ones
    int mask_bytes;
    uint16_t* buf;   // this wave's row buffer [cap], waves below bufs
    int bufs;
    int32_t* ids;    // random batch list: [list_len] atom ids
    __device__ ListLds(double4* lds, int stage_cap, int cap, int rows, int wv)
    {
        cand = (float4*)lds;
        mask = (char*)(cand + list_len(stage_cap));
        mask_bytes = kMaskRow * rows;
        uint16_t* b = (uint16_t*)(mask + 2 * mask_bytes);
        buf = b + (size_t)wv * cap;
        bufs = list_bufs(cap);
        ids = (int32_t*)(b + (size_t)bufs * cap);
    }
};

// Bound of the rounding of near_masks' squared distances: candidates lie within 1.5
// cells per axis of the centre (R^2 the square of that corner), and with u = 2^-24 the
// rounded positions, products and five-term sums add up to less than 27 u R^2;
// 2^-19 R^2 = 32 u R^2.
inline float list_margin(const double cell[3])
{
    double r2 = 0.0;
    for (int d = 0; d < 3; ++d) r2 += 2.25 * cell[d] * cell[d];
    return (float)(r2 * 1.9073486328125e-6);
}

// Random batch list of a build: rows keep every pair closer than r_near = r_core +
// skin (it may come inside r_core before the next build) and the shell pairs that
// rbl_select keeps, tagged with kRblSel so the pair pass weights them.
constexpr int kRblSel = 0x8000;
struct RblBuild {
    uint64_t seed;
    uint32_t epoch;    // list build number
    uint32_t pice;
    const int32_t* perm;  // sorted slot -> atom id
};

// Atom id of tile-local candidate u (random batch list builds and their fallback).
__device__ inline int32_t tile_atom_id(const TileHdr& h, const int32_t* __restrict__ perm, int u)
{
    const int st = tile_seg(h, u);
    return perm[h.gstart[st] + (u - h.off[st])];
}

// The same value, unknown to the compiler: keeps what is computed from it inside the
// phase that uses it, where hoisting it over the whole build would cost registers that the
// pair pass's occupancy does not have.
__device__ inline int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

struct ListArgs {
    const double4* xs_ref;
    double rl2, tag2;  // r_list^2; LJ range (full list) or the always-kept near band (RBL)
    float margin;      // list_margin
    double ctr[3];     // centre of the home cell
    int cap;
    uint16_t* nlist;
    int2* ncount;
    unsigned long long* stats;
    unsigned long long* host;  // pinned mirror of stats: the host reads its word 2 (rows that
                               // overflowed) before the next evaluation, without a copy each time
};

// A row of n entries did not fit.
__device__ inline void list_overflow(const ListArgs& a, int n)
{
    atomicAdd(&a.stats[2], 1ull);
    atomicMax(&a.stats[4], (unsigned long long)n);
    __hip_atomic_store(&a.host[2], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

typedef float list_f4 __attribute__((ext_vector_type(4)));

// FP32 position relative to the home cell's centre, its square in w.  One that is not a number
// stands far from everything, as the exact criterion has it: the masks take the sign bits of
// the distances, and a NaN has one too.
__device__ inline float4 list_pos(const ListArgs& A, double x, double y, double z)
{
    const float a = (float)(x - A.ctr[0]), b = (float)(y - A.ctr[1]), c = (float)(z - A.ctr[2]);
    const float w = fmaf(c, c, fmaf(b, b, a * a));
    return w < 1.0e30f ? make_float4(a, b, c, w) : make_float4(0.0f, 0.0f, 0.0f, 1.0e30f);
}

// The home rows of one near_masks call: NMT 16-row tiles, rows [0, nrow) being home
// atoms s0 + row, tile index u0 + row relative to the staged block.
struct MaskRows {
    const float4* home;  // staged positions of the rows, or null: from xs_ref
    int s0, u0, nrow;
};

// Masks of NMT x 16 rows against the nch chunks of the staged block.  Word of (row,
// wave pair, column): the pair's 2T chunks, the first in bit 2T - 1 (W: uint32 for
// T <= 16, else uint64, built in two halves).  cb: tile index of the block's first
// candidate.  Per 256 pairs 32 cycles of a SIMD's matrix core and 18 VALU instructions (two
// sign bits, the LJ-range shift and the smallest distances from the thresholds).
//
// A lane that finds one of its values within rounding of a threshold settles it at once by
// the exact criterion (about one pair in 130,000).  Building the whole row again by that
// criterion, 2,000 candidates by one wave, took longer than all the other rows of a
// workgroup: 7 us of the 23 of a build at 5,775 ions, 12 of 23 at 2,000.
template <int NMT, typename H>
__device__ inline void near_masks(const TileHdr& h, const ListArgs& a, const float4* cand,
                                  const MaskRows& R, const ListLds& L, int cb, int row0, int nch,
                                  int T, int wv, int lane_in)
{
    const int lane = opaque(lane_in), col = lane & 15, q = lane >> 4;
    const int tw = min(T, nch - wv * T);
    const float t0 = (float)(a.rl2 - 1e-4);         // d = d2 - t0
    const float tin = (float)(a.rl2 - 1e-4 - a.tag2);  // d + tin = d2 - tag2
    const float tiny = 2e-4f - t0 + a.margin;  // x below: d2 within rounding of 1e-4
    float av[NMT];
    list_f4 c[NMT];
    uint32_t hit[NMT][4], in[NMT][4];
#pragma unroll
    for (int m = 0; m < NMT; ++m) {
        const int ra = min(16 * m + col, R.nrow - 1);
        float4 f;
        if (R.home) {
            f = R.home[ra];
        } else {
            const double4 p = a.xs_ref[R.s0 + ra];
            f = list_pos(a, p.x, p.y, p.z);
        }
        const float fq = q == 0 ? f.x : q == 1 ? f.y : f.z;
        av[m] = q == 3 ? 1.0f : -2.0f * fq;
        // rows past the last: far from everything
        const float w = 16 * m + col < R.nrow ? f.w - t0 : 1.0e30f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            c[m][r] = __shfl(w, 4 * q + r, 64);
            hit[m][r] = in[m][r] = 0u;
        }
    }
    const float* b0 = (const float*)cand + 4 * (16 * wv * T + col) + q;
    float bn = tw > 0 ? b0[0] : 0.0f;
    for (int t = 0; t < tw; ++t) {
        const float bv = bn;
        bn = b0[64 * min(t + 1, tw - 1)];
        list_f4 d[NMT];
#pragma unroll
        for (int m = 0; m < NMT; ++m)
            d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[m], bv, c[m], 0, 0, 0);
        const int uc = 16 * (wv * T + t);
        if (uc + 15 >= R.u0 && uc < R.u0 + R.nrow) {
            // the rows themselves: not their own neighbours
#pragma unroll
            for (int m = 0; m < NMT; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (uc + col == R.u0 + 16 * m + 4 * q + r) d[m][r] = 1.0e30f;
        }
        float near = 3.0e38f, dmin = 3.0e38f;
#pragma unroll
        for (int m = 0; m < NMT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = d[m][r], y = x + tin;
                hit[m][r] = __builtin_amdgcn_alignbit(hit[m][r], __float_as_uint(x), 31);
                in[m][r] = __builtin_amdgcn_alignbit(in[m][r], __float_as_uint(y), 31);
                near = fminf(fminf(near, fabsf(x)), fabsf(y));
                dmin = fminf(dmin, x);
            }
        if (near < a.margin || dmin < tiny) {
#pragma clang fp contract(off)
            // bit e = 4 m + r: the values to settle, then their exact bits
            uint32_t todo = 0u, eh = 0u, ei = 0u;
#pragma unroll
            for (int e = 0; e < 4 * NMT; ++e) {
                const float x = d[e >> 2][e & 3], y = x + tin;
                if (fabsf(x) < a.margin || fabsf(y) < a.margin || x < tiny) todo |= 1u << e;
            }
            const double4 pj = stage_ref(h, a.xs_ref, cb + uc + col);
            for (uint32_t w = todo; w != 0u; w &= w - 1u) {
                const int e = __ffs((int)w) - 1;
                const double4 pi = a.xs_ref[R.s0 + 16 * (e >> 2) + 4 * q + (e & 3)];
                const double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
                const double d2 = fma(dz, dz, fma(dy, dy, dx * dx));
                if ((a.rl2 - d2) > 1e-4 && d2 > 1e-4) eh |= 1u << e;
                if (d2 < a.tag2) ei |= 1u << e;
            }
#pragma unroll
            for (int e = 0; e < 4 * NMT; ++e) {
                const uint32_t b = (todo >> e) & 1u;
                uint32_t &hb = hit[e >> 2][e & 3], &ib = in[e >> 2][e & 3];
                hb = (hb & ~b) | ((eh >> e) & 1u & b);
                ib = (ib & ~b) | ((ei >> e) & 1u & b);
            }
        }
    }
    const int sh = T - (tw > 0 ? tw : 0);
#pragma unroll
    for (int m = 0; m < NMT; ++m) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = row0 + 16 * m + 4 * q + r;
            // a word's two halves: waves 2g (high) and 2g + 1 (low)
            H* w = (H*)L.mask + (((row * 4 + (wv >> 1)) * 16 + col) * 2 + (1 - (wv & 1)));
            w[0] = tw > 0 ? (H)(hit[m][r] << sh) : (H)0;
            w[L.mask_bytes / (int)sizeof(H)] = tw > 0 ? (H)(in[m][r] << sh) : (H)0;
        }
    }
}

// Wave sum of an int, uniform.
__device__ inline int wave_sum_int(int v)
{
    v += dpp_i<0xB1>(v);
    v += dpp_i<0x4E>(v);
    v += dpp_i<0x141>(v);
    v += dpp_i<0x140>(v);
    v += dpp_i<0x142, 0xa>(v);
    v += dpp_i<0x143, 0xc>(v);
    return __builtin_amdgcn_readlane(v, 63);
}

// Number of leading zero bits of a non-zero word.
__device__ inline int lead0(uint32_t v) { return __clz((int)v); }
__device__ inline int lead0(uint64_t v) { return __clzll((long long)v); }

// One wave: the hits of row `row` (home atom s) in the staged block, whose first candidate is
// tile index cb.  SINGLE: the block is the whole tile, and the row collects in the wave's LDS
// buffer, the LJ range first; else over the blocks in its slots in global memory, the LJ range
// from the front and the others from the back.  have: entries that earlier blocks gave the row.
// The last block writes the row.
template <bool RBL, typename W, bool SINGLE>
__device__ inline int2 row_hits(const TileHdr& h, const ListArgs& a, const ListLds& L, int row,
                                int s, int cb, const int32_t* ids, int T, int lane_in, bool last,
                                int2 have, const RblBuild& rb)
{
    const int lane = opaque(lane_in);
    const int cap = a.cap, total = h.off[27];
    const int g = lane >> 4, col = lane & 15;
    uint16_t* __restrict__ rowp = a.nlist + (size_t)s * cap;
    int ci = have.x, co = have.y;
    auto put1 = [&](int k, int u) {
        if (SINGLE) L.buf[k] = (uint16_t)u;
        else rowp[k] = (uint16_t)u;
    };
    {
        constexpr int kBits = 8 * sizeof(W);
        const int wo = (row * 4 + g) * 16 + col;
        W m, mi;
        {
            // the halves T bits wide, joined; the first chunk in the top bit
            using H = typename std::conditional<sizeof(W) == 4, uint16_t, uint32_t>::type;
            const H* p = (const H*)L.mask + 2 * wo;
            const H* pi = p + L.mask_bytes / (int)sizeof(H);
            m = (((W)p[1] << T) | (W)p[0]) << (kBits - 2 * T);
            mi = (((W)pi[1] << T) | (W)pi[0]) << (kBits - 2 * T);
        }
        W mo = m & ~mi;
        mi &= m;
        const int ub = cb + 32 * g * T + col;
        const W top = (W)1 << (kBits - 1);
        // the row's counts first: a row that fits is written without tests, one that
        // does not is only counted
        int pc = sizeof(W) == 4 ? __popc((uint32_t)mi) | (__popc((uint32_t)mo) << 16)
                                : __popcll(mi) | (__popcll(mo) << 16);
        pc = wave_sum_int(pc);
        const int ni = pc & 0xffff, no = pc >> 16;
        // each trip gives put the next hit of every lane that has one
        auto expand = [&](W w, int k0, auto put) {
            while (w != 0) {
                const uint64_t act = __builtin_amdgcn_ballot_w64(true);
                const int k = (int)__builtin_amdgcn_mbcnt_hi(
                    (uint32_t)(act >> 32),
                    __builtin_amdgcn_mbcnt_lo((uint32_t)act, (uint32_t)k0));
                const int z = lead0(w);
                put(k, ub + 16 * z);
                w ^= top >> z;
                k0 += __popcll(act);
            }
        };
        if (RBL) {
            // the block's hits to the buffer, the near band first; then each draws its selection,
            // 64 at a time (a lane drawing for its own column's hits leaves most lanes idle: an
            // evaluation of 200,000 ions with a rebuild took 568 us so, 453 now).  A near-band
            // entry kept for being near counts only if selected should it lie in the shell
            // when evaluated.  co: hits of the blocks so far; rows whose hits do not fit overflow.
            if (co + ni + no < cap) {
                auto put = [&](int k, int u) { L.buf[k] = (uint16_t)u; };
                expand(mi, 0, put);
                expand(mo, ni, put);
                __syncwarp();
                const int32_t id_i = rb.perm[s];
                for (int k0 = 0; k0 < ni + no; k0 += 64) {
                    const int k = k0 + lane;
                    const bool hit = k < ni + no;
                    const int u = hit ? (int)L.buf[k] : 0;
                    bool sel = false;
                    if (hit) sel = rbl_select(rb.seed, rb.epoch, id_i, ids[u - cb], rb.pice);
                    const bool keep = hit && (k < ni || sel);
                    const uint64_t mk = __builtin_amdgcn_ballot_w64(keep);
                    if (keep) rowp[ci + (int)mbcnt64(mk)] = (uint16_t)(sel ? (u | kRblSel) : u);
                    ci += __popcll(mk);
                }
                __syncwarp();  // the buffer is reused for the wave's next row
            }
            co += ni + no;
            if (last && lane == 0) {
                if (co < cap) rowp[ci] = (uint16_t)total;
                a.ncount[s] = co < cap ? make_int2(ci, 0) : make_int2(co, 0);
                if (co >= cap) list_overflow(a, co + 1);
            }
            return make_int2(ci, co);
        }
        if (ci + co + ni + no < cap) {
            expand(mi, ci, put1);
            expand(mo, SINGLE ? ni : co, [&](int k, int u) { put1(SINGLE ? k : cap - 1 - k, u); });
        }
        ci += ni;
        co += no;
    }
    if (!last) return make_int2(ci, co);
    const int n = ci + co;
    if (n < cap) {
        __syncwarp();
        if (!SINGLE) {
            // the row from global memory into the buffer, in order
            __threadfence_block();
            for (int k = lane; k < n; k += 64)
                L.buf[k] = rowp[k < ci ? k : cap - 1 - (k - ci)];
        }
        // two entries per 32-bit word (rows start at multiples of 64 entries)
        if (lane == 0) L.buf[n] = (uint16_t)total;
        __syncwarp();
        for (int k = lane; 2 * k <= n; k += 64)
            ((uint32_t*)rowp)[k] = ((const uint32_t*)L.buf)[k];
        __syncwarp();  // the buffer is reused for the wave's next row
    }
    if (lane == 0) {
        a.ncount[s] = n < cap ? make_int2(ci, co) : make_int2(n, 0);
        if (n >= cap) list_overflow(a, n + 1);
    }
    return make_int2(ci, co);
}

// LDS of the build besides the stage: entries per row over the blocks of one tile.
struct ListRows {
    int2 cnt[64];
};

// One block of the build: masks, then rows, for the row group [0, nrow) of home atoms
// s0.. (tile index u0..).
template <bool RBL, typename W>
__device__ inline void list_block(const TileHdr& h, const ListArgs& a, const ListLds& L,
                                  ListRows& lr, const float4* cand, const float4* home,
                                  const int32_t* ids, int cb, int cn, int s0, int u0, int nrow,
                                  bool single, bool last, int wv, int lane, const RblBuild& rb)
{
    using H = typename std::conditional<sizeof(W) == 4, uint16_t, uint32_t>::type;
    const int nch = (cn + 15) / 16, T = (nch + kTileWaves - 1) / kTileWaves;
    // 32 rows at a time: more row tiles would take the tile pass past the registers
    // that its LDS stage's occupancy allows
    for (int r0 = 0; r0 < nrow; r0 += 32) {
        const MaskRows R{home ? home + r0 : nullptr, s0 + r0, u0 + r0 - cb, min(32, nrow - r0)};
        if (R.nrow > 16) near_masks<2, H>(h, a, cand, R, L, cb, r0, nch, T, wv, lane);
        else near_masks<1, H>(h, a, cand, R, L, cb, r0, nch, T, wv, lane);
    }
    __syncthreads();
    for (int row = wv < L.bufs ? wv : nrow; row < nrow; row += L.bufs) {
        if (single) {
            row_hits<RBL, W, true>(h, a, L, row, s0 + row, cb, ids, T, lane, true,
                                   make_int2(0, 0), rb);
            continue;
        }
        const int2 n = row_hits<RBL, W, false>(h, a, L, row, s0 + row, cb, ids, T, lane, last,
                                               cb > 0 ? lr.cnt[row] : make_int2(0, 0), rb);
        if (!last && lane == 0) lr.cnt[row] = n;
    }
    __syncthreads();
}

// Rows of a tile of at most 64 candidates (a thin gas): one wave per row, one candidate per
// lane, by the exact criterion.  No barriers and no LDS; the masks of a few candidates cost
// their barriers all the same.  30,000 ions in 15,625 cells, a rebuild every second step: 158 ->
// 134 us a step; a rebuild of 4,000 in 4,096 cells 64 -> 50 us.
template <bool RBL>
__device__ inline void list_few(const TileHdr& h, const ListArgs& a, int a0, int a1, int wv,
                                int lane_in, const RblBuild& rb)
{
#pragma clang fp contract(off)
    const int lane = opaque(lane_in), total = h.off[27], cap = a.cap;
    if (a0 + wv >= a1) return;
    const bool live = lane < total;
    const int u = live ? lane : 0;
    const double4 pj = stage_ref(h, a.xs_ref, u);
    const int32_t id_j = RBL ? tile_atom_id(h, rb.perm, u) : 0;
    for (int s = a0 + wv; s < a1; s += kTileWaves) {
        const double4 pi = a.xs_ref[s];
        const double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
        const double d2 = fma(dz, dz, fma(dy, dy, dx * dx));
        const bool hit = live && (a.rl2 - d2) > 1e-4 && d2 > 1e-4, in = hit && d2 < a.tag2;
        const int n = __popcll(__builtin_amdgcn_ballot_w64(hit));
        bool sel = false;
        if (RBL) sel = hit && rbl_select(rb.seed, rb.epoch, rb.perm[s], id_j, rb.pice);
        // front: LJ range, or every entry that a random batch list keeps
        const bool front = RBL ? in || sel : in, back = !RBL && hit && !in;
        const uint64_t mf = __builtin_amdgcn_ballot_w64(front), mb = __builtin_amdgcn_ballot_w64(back);
        const int nf = __popcll(mf), nb = __popcll(mb);
        if (n < cap) {
            uint16_t* __restrict__ row = a.nlist + (size_t)s * cap;
            if (front || back)
                row[front ? (int)mbcnt64(mf) : nf + (int)mbcnt64(mb)] =
                    (uint16_t)(sel ? (u | kRblSel) : u);
            if (lane == 0) row[nf + nb] = (uint16_t)total;
        }
        if (lane == 0) {
            a.ncount[s] = n < cap ? make_int2(nf, nb) : make_int2(n, 0);
            if (n >= cap) list_overflow(a, n + 1);
        }
    }
}

// Rows of the home atoms [a0, a1) of a tile (every thread of the workgroup).  staged:
// the whole tile fits the LDS stage.
template <bool RBL>
__device__ inline void list_tile(const TileHdr& h, const ListArgs& a, double4* lds, ListRows& lr,
                                 int stage_cap, int rows, bool staged, int a0, int a1, int h0,
                                 int wv, int lane, const RblBuild& rb)
{
    const int total = h.off[27];
    if (a0 >= a1) return;  // no home atoms
    if (total >= kMaxTile) {
        for (int s = a0 + (int)threadIdx.x; s < a1; s += kTileThreads) {
            a.ncount[s] = make_int2(a.cap + 1, 0);
            list_overflow(a, a.cap + 1);
        }
        return;
    }
    if (total <= 64) {
        list_few<RBL>(h, a, a0, a1, wv, lane, rb);
        return;
    }
    const ListLds L(lds, stage_cap, a.cap, rows, wv);
    // candidates [cb, cb + cn) into LDS, padded to whole chunks with points far from
    // every row
    auto stage = [&](int cb, int cn) {
        const int pad = (cn + 15) / 16 * 16;
        for (int k = opaque(threadIdx.x); k < pad; k += kTileThreads) {
            if (k < cn) {
                const double4 p = stage_ref(h, a.xs_ref, cb + k);
                L.cand[k] = list_pos(a, p.x, p.y, p.z);
                if (RBL) L.ids[k] = tile_atom_id(h, rb.perm, cb + k);
            } else {
                L.cand[k] = make_float4(0.0f, 0.0f, 0.0f, 1.0e30f);
            }
        }
    };
    const int blk = min(kListBlock, staged ? kListBlock : stage_cap / 16 * 16);
    if (staged) stage(0, total);
    const bool narrow = min(blk, total) <= 16 * 16 * kTileWaves;
    const int group = narrow ? rows : rows / 32 * 16;  // 256 or 512 bytes a row and mask
    const bool single = total <= blk;
    const int uh = h.off[kHomeSeg] - h0;
    for (int s0 = a0; s0 < a1; s0 += group) {
        const int nrow = min(group, a1 - s0);
        // the home atoms of the group, when the whole tile is staged
        const float4* home = staged ? L.cand + s0 + uh : nullptr;
        for (int cb = 0; cb < total; cb += blk) {
            const int cn = min(blk, total - cb);
            if (!staged) stage(cb, cn);
            __syncthreads();
            const float4* cand = staged ? L.cand + cb : L.cand;
            const int32_t* ids = RBL ? (staged ? L.ids + cb : L.ids) : nullptr;
            const bool last = cb + blk >= total;
            if (narrow)
                list_block<RBL, uint32_t>(h, a, L, lr, cand, home, ids, cb, cn, s0, s0 + uh, nrow,
                                          single, last, wv, lane, rb);
            else
                list_block<RBL, uint64_t>(h, a, L, lr, cand, home, ids, cb, cn, s0, s0 + uh, nrow,
                                          single, last, wv, lane, rb);
        }
    }
}

#endif

}  // namespace rbmd
