// nlist.hip -- list part of the force pass (displacement check, cell bins and sort,
// position gather; the structure factor beside them), the MD-run binning prologue and
// list statistics.
// (The Verlet rows are built inside the tile pass, pair.hip; the MD-step kernels
// are in md.h / md.hip.)
//
// Reference behaviour followed (paths relative to the reference checkout):
//   cell grid / binning / sort    rbmd/framework/locator/ContPointLocator.{h,cxx} (h:44-53, cxx:38-92)
//   27-cell stencil + periodic    rbmd/framework/locator/ExecPointLocator.h:303-319
//   list criterion                rbmd/framework/run/worklet/RunWorklet.cpp:40-96 (:83)
// The list radius adds a Verlet skin; the list is rebuilt on the device when an
// atom has moved more than half the skin since the last build.
#include "md.h"
#include "state.h"
#include "tile.h"

namespace rbmd {

namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------- force pass
// The list part of a force evaluation is three launches.  As seven of their own, with the
// two of the structure factor and a copy of the statistics, a pass took 45 us at 4,000 ions
// (28 now), most of it launch gaps.
//   CheckRho   displacement check, and the rho(k) partials, which need only the positions
//   BinGather  on a rebuild the atoms into the cell bins (those of the MD step, which every
//              MD run fills anew), else their positions into the sorted array
//   SortFinal  on a rebuild the cell sort of the bins; the rho(k) final reduction
// With more than kBinChunkMinCells cells, ChunkSum between the last two.

// Max-displacement test against the positions of the last build; clears the bin counts
// that a rebuild fills.
struct Check {
    static constexpr int kThreads = kBlock;
    struct Args {
        const double *x, *y, *z, *xr, *yr, *zr;
        int n;
        Box box;
        double thr2;
        uint32_t* flags;
        MdBins bins;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        const int i = blk * kBlock + threadIdx.x;
        const int b = (int)(a.flags[3] & 1u);
        if (i < a.bins.ncell) a.bins.count[b * a.bins.ncell + i] = 0;
        if (i < a.n) {
            double dx = min_image(a.x[i] - a.xr[i], a.box.L[0], a.box.invL[0]);
            double dy = min_image(a.y[i] - a.yr[i], a.box.L[1], a.box.invL[1]);
            double dz = min_image(a.z[i] - a.zr[i], a.box.L[2], a.box.invL[2]);
            double d2 = dx * dx + dy * dy + dz * dz;
            if (d2 > a.thr2) a.flags[0] = 1u;
            if (d2 != d2) a.flags[1] = 1u;
        }
    }
};

template <typename T>
struct CheckRho {
    static constexpr int kThreads = kBlock;
    static_assert(kBlock == kRhoBlock, "one block size for both parts");
    struct Args {
        typename RhoPartial<T>::Args rho;
        int nrho;
        Check::Args check;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        if (blk < a.nrho) RhoPartial<T>::run(a.rho, blk, a.nrho);
        else Check::run(a.check, blk - a.nrho, 0);
    }
};

__global__ void k_set_flag(uint32_t* flags) { flags[0] = 1u; }

// A rebuild bins the current positions; otherwise they go to the sorted packed array,
// unwrapped against the reference positions (x_ref + min_image(x - x_ref)), so that the
// image of every list pair stays the one seen at the build.  SPILL: SortFinal follows, which
// empties the lists of the atoms beyond their buckets.
template <bool SPILL>
struct BinGather {
    static constexpr int kThreads = kBlock;
    struct Args {
        const double *x, *y, *z, *xr, *yr, *zr, *q;
        const int32_t* inv_perm;
        int n;
        Box box;
        double4* xs;
        int3 dims;
        double3 cell;
        MdBins bins;
        const uint32_t* flags;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        const int i = blk * kBlock + threadIdx.x;
        if (i >= a.n) return;
        const double x[3] = {a.x[i], a.y[i], a.z[i]};
        if (a.flags[0] != 0u) {
            md_bin_atom<SPILL>(a.bins, (int)(a.flags[3] & 1u), i, i, x, a.box, a.dims, a.cell);
            return;
        }
        const double p = a.xr[i], b = a.yr[i], c = a.zr[i];
        const double dx = min_image(x[0] - p, a.box.L[0], a.box.invL[0]);
        const double dy = min_image(x[1] - b, a.box.L[1], a.box.invL[1]);
        const double dz = min_image(x[2] - c, a.box.L[2], a.box.invL[2]);
        a.xs[a.inv_perm[i]] = make_double4(p + dx, b + dy, c + dz, a.q[i]);
    }
};

// rho(k) final reduction (workgroups [0, nfin), one k each), the cell sort and the tile
// order (as in SortRho).
template <typename T>
struct SortFinal {
    static constexpr int kThreads = kRhoBlock;
    static_assert(RhoFinal<T>::kThreads == kThreads, "one block size for both parts");
    struct Args {
        RhoFinalArgs<T> fin;
        int nfin;
        CellSortMDArgs cs;
        int nsort;
        int parts;
        int3 dims;
        int split, ncu;
        int32_t* tile_order;
    };
    __device__ static void run(const Args& A, int blk, int)
    {
        if (blk < A.nfin) {
            RhoFinal<T>::run(A.fin, blk, A.nfin);
            return;
        }
        blk -= A.nfin;
        constexpr int kWaves = kThreads / 64;
        constexpr int kInts = kWaves * kSortWaveBuf > kOrderLds ? kWaves * kSortWaveBuf : kOrderLds;
        __shared__ int32_t lds[kInts];
        if (blk == A.nsort) {
            if (A.ncu > 0 && A.cs.flags[0] != 0u)
                tile_order_build(A.cs.bins.count + (size_t)(A.cs.flags[3] & 1u) * A.cs.ncell,
                                 A.cs.ncell, A.dims, A.split, A.ncu, A.tile_order, lds);
            return;
        }
        cellsort_md<kThreads, true>(A.cs, blk, A.parts, lds);
    }
};

// MD-step binning before the first step of a run: bins the current positions
// into buffer (epoch & 1) of the MD bins (which the caller cleared), as the tile
// pass of a previous step would have.
// It also opens the run's device state: the long-step flag (flags[4]) cleared and
// the graph's step counter set to the run's first step (no fill or copy launches).
struct MdBin {
    static constexpr int kThreads = kBlock;
    struct Args {
        const double *x, *y, *z;
        int n;
        Box box;
        int3 dims;
        double3 cell;
        MdBins bins;
        uint32_t* flags;
        unsigned long long* step;  // device step counter of graph replays
        unsigned long long step0;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        const int i = blk * kBlock + threadIdx.x;
        if (i == 0) {
            a.flags[4] = 0u;
            *a.step = a.step0;
        }
        if (i >= a.n) return;
        const double p[3] = {a.x[i], a.y[i], a.z[i]};
        // any one-to-one slot numbering serves the cell sort: atom i bins in slot i
        md_bin_atom(a.bins, (int)(a.flags[3] & 1u), i, i, p, a.box, a.dims, a.cell);
    }
};

// Zeroes n ints (a replica's MD bin counts before MdBin, one grid for the batch).
struct ClearInts {
    static constexpr int kThreads = kBlock;
    struct Args {
        int32_t* p;
        int n;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        const int i = blk * kBlock + threadIdx.x;
        if (i < a.n) a.p[i] = 0;
    }
};

// One replica's build statistics and flags into its kStatsOutWords words of the
// batch's readback block, so a batched run ends with one copy to the host.
struct StatsOut {
    static constexpr int kThreads = 64;
    struct Args {
        const unsigned long long* stats;
        const uint32_t* flags;
        unsigned long long* out;
    };
    __device__ static void run(const Args& a, int, int)
    {
        const int t = threadIdx.x;
        if (t < 8)
            a.out[t] = a.stats[t];
        else if (t < 13)
            a.out[t] = a.flags[t - 8];
    }
};

// Chunk counts of MdBin's bins: block k sums the counts of cells [256 k, 256 k + 256)
// of the buffer MdBin filled and writes chunk k (no atomics: atoms in id order land
// in every chunk, so per-atom or per-wave chunk atomics serialise on few counters).
struct ChunkSum {
    static constexpr int kThreads = kBinChunk;
    struct Args {
        MdBins bins;
        const uint32_t* flags;
    };
    __device__ static void run(const Args& a, int blk, int)
    {
        __shared__ int red[kThreads / 64];
        const int b = (int)(a.flags[3] & 1u);
        const int c = blk * kBinChunk + (int)threadIdx.x;
        int v = c < a.bins.ncell ? a.bins.count[b * a.bins.ncell + c] : 0;
        v = wave_sum(v);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            int s = 0;
            for (int w = 0; w < kThreads / 64; ++w) s += red[w];
            a.bins.chunk[b * a.bins.nchunk + blk] = s;
        }
    }
};

// ---------------------------------------------------------------- Verlet list
// (the row builder list_tile lives in tile.h)
// List statistics on demand: entries, LJ-range entries, longest row.
__global__ __launch_bounds__(256) void k_list_stats(const int2* __restrict__ ncount, int n,
                                                    unsigned long long* __restrict__ out)
{
    __shared__ unsigned long long se[256], si[256], sm[256];
    unsigned long long e = 0, in = 0, mx = 0;
    for (int s = threadIdx.x; s < n; s += 256) {
        const int2 c = ncount[s];
        e += (unsigned long long)(c.x + c.y);
        in += (unsigned long long)c.x;
        mx = mx > (unsigned long long)(c.x + c.y) ? mx : (unsigned long long)(c.x + c.y);
    }
    se[threadIdx.x] = e;
    si[threadIdx.x] = in;
    sm[threadIdx.x] = mx;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            se[threadIdx.x] += se[threadIdx.x + o];
            si[threadIdx.x] += si[threadIdx.x + o];
            sm[threadIdx.x] = sm[threadIdx.x] > sm[threadIdx.x + o] ? sm[threadIdx.x]
                                                                    : sm[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = se[0];
        out[1] = si[0];
        out[2] = sm[0];
    }
}

__global__ __launch_bounds__(kBlock) void k_copy(uint4* __restrict__ dst,
                                                 const uint4* __restrict__ src, int64_t n16)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n16;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

inline int nblk(int64_t n, int b = kBlock) { return (int)((n + b - 1) / b); }

// ---------------------------------------------------------------- argument packing
Check::Args check_args(Engine& e, const double* x, const double* y, const double* z)
{
    const double h = 0.5 * e.skin;
    return Check::Args{x, y, z, e.xr, e.yr, e.zr, (int)e.n, e.box, h * h, e.flags, md_bins(e)};
}

template <bool SPILL>
typename BinGather<SPILL>::Args bin_args(Engine& e, const double* x, const double* y,
                                         const double* z)
{
    return typename BinGather<SPILL>::Args{x, y, z, e.xr, e.yr, e.zr, e.q, e.atom_rank /* inverse perm */,
                           (int)e.n, e.box, e.xs, make_int3(e.dims[0], e.dims[1], e.dims[2]),
                           make_double3(e.cell[0], e.cell[1], e.cell[2]), md_bins(e), e.flags};
}

MdBin::Args mdbin_args(Engine& e, const double* x, const double* y, const double* z,
                       unsigned long long step0)
{
    return MdBin::Args{x,         y,           z,          (int)e.n, e.box,
                       make_int3(e.dims[0], e.dims[1], e.dims[2]),
                       make_double3(e.cell[0], e.cell[1], e.cell[2]),
                       md_bins(e), e.flags,     e.d_step,   step0};
}

}  // namespace

// ================================================================= launchers

template <typename T>
void check_rho_t(Engine& e, const double* x, const double* y, const double* z, bool rho,
                 hipStream_t s)
{
    typename CheckRho<T>::Args a;
    memset(&a.rho, 0, sizeof a.rho);
    a.nrho = 0;
    if (rho) a.rho = rho_args<T>(e, x, y, z, &a.nrho);
    a.check = check_args(e, x, y, z);
    const int64_t cover = e.n > e.ncell ? e.n : e.ncell;
    k_one<CheckRho<T>><<<a.nrho + nblk(cover), kBlock, 0, s>>>(a);
}

template <typename T>
void sort_final_t(Engine& e, const double* x, const double* y, const double* z, bool rho,
                  hipStream_t s)
{
    typename SortFinal<T>::Args a;
    memset(&a.fin, 0, sizeof a.fin);
    if (rho) a.fin = rho_final_args<T>(e, nullptr);
    a.nfin = rho ? e.P : 0;
    a.cs = cellsort_md_args(e, x, y, z);
    a.parts = sort_parts(e.n, e.ncell);
    a.nsort = sortrho_cell_blocks(e.ncell * a.parts);
    a.dims = make_int3(e.dims[0], e.dims[1], e.dims[2]);
    a.split = e.split;
    a.ncu = tile_order_ncu(e.ncell, e.split, e.num_cu);
    a.tile_order = e.tile_order;
    k_one<SortFinal<T>><<<a.nfin + a.nsort + 1, kRhoBlock, 0, s>>>(a);
}

void launch_force_lists(Engine& e, const double* x, const double* y, const double* z,
                        hipStream_t s)
{
    // FP64 full Ewald forms its sums on the lattice box instead (ewald.hip)
    const bool rho = has_kspace(e) && e.P > 0 && !e.ew.on;
    {
        ScopedTimer t(e, P_CHECK, s);
        if (e.precision == 32) check_rho_t<float>(e, x, y, z, rho, s);
        else check_rho_t<double>(e, x, y, z, rho, s);
    }
    {
        ScopedTimer t(e, P_BIN, s);
        k_one<BinGather<true>><<<nblk(e.n), kBlock, 0, s>>>(bin_args<true>(e, x, y, z));
        if (md_nchunk(e.ncell) > 0)
            k_one<ChunkSum><<<md_nchunk(e.ncell), ChunkSum::kThreads, 0, s>>>(
                ChunkSum::Args{md_bins(e), e.flags});
    }
    {
        ScopedTimer t(e, P_CELLSORT, s);
        if (e.precision == 32) sort_final_t<float>(e, x, y, z, rho, s);
        else sort_final_t<double>(e, x, y, z, rho, s);
    }
    if (e.ew.on) launch_ewald_rho(e, x, y, z, s);
    // the Verlet rows are built inside the tile pass (pair.hip)
}

void launch_force_rebuild(Engine& e, hipStream_t s) { k_set_flag<<<1, 1, 0, s>>>(e.flags); }

void launch_md_bin(Engine& e, const double* x, const double* y, const double* z,
                   unsigned long long step0, hipStream_t s)
{
    // the counts cleared by a kernel of the library (a runtime fill costs the host
    // about twice the launch time)
    const int nc = (int)(md_count_bytes(e.ncell) / sizeof(int32_t));
    k_one<ClearInts><<<nblk(nc), kBlock, 0, s>>>(ClearInts::Args{e.md_count, nc});
    k_one<MdBin><<<nblk(e.n > 0 ? e.n : 1), kBlock, 0, s>>>(mdbin_args(e, x, y, z, step0));
    if (md_nchunk(e.ncell) > 0)
        k_one<ChunkSum><<<md_nchunk(e.ncell), ChunkSum::kThreads, 0, s>>>(
            ChunkSum::Args{md_bins(e), e.flags});
}

void launch_list_stats(Engine& e, unsigned long long* out, hipStream_t s)
{
    k_list_stats<<<1, 256, 0, s>>>(e.ncount, (int)e.n, out);
}

void launch_copy(void* dst, const void* src, int64_t nbytes, hipStream_t s)
{
    const int64_t n16 = nbytes / 16;
    int blocks = (int)((n16 + kBlock - 1) / kBlock);
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    k_copy<<<blocks, kBlock, 0, s>>>((uint4*)dst, (const uint4*)src, n16);
}

// ================================================================= batched phases

hipError_t nlist_batch_prepare(Batch& b)
{
    const size_t R = b.es.size();
    std::vector<BinGather<false>::Args> bi(R);
    std::vector<MdBin::Args> mb(R);
    std::vector<ClearInts::Args> mc(R);
    std::vector<StatsOut::Args> so(R);
    std::vector<int> nmc(R);
    std::vector<ChunkSum::Args> cks(R);
    std::vector<int> nat(R), none(R, 1), nch(R);
    for (size_t r = 0; r < R; ++r) {
        Engine& e = *b.es[r];
        const RepState& st = b.st[r];
        bi[r] = bin_args<false>(e, st.x, st.y, st.z);
        mb[r] = mdbin_args(e, st.x, st.y, st.z, b.step0);
        const int ncount = (int)(md_count_bytes(e.ncell) / sizeof(int32_t));
        mc[r] = ClearInts::Args{e.md_count, ncount};
        nmc[r] = (ncount + kBlock - 1) / kBlock;
        so[r] = StatsOut::Args{e.stats, e.flags, b.d_out ? b.d_out + r * kStatsOutWords : nullptr};
        cks[r] = ChunkSum::Args{md_bins(e), e.flags};
        nat[r] = nblk(e.n > 0 ? e.n : 1);
        nch[r] = md_nchunk(e.ncell);
    }
    hipError_t err;
    if ((err = phase_upload(b.ph[BP_BIN], bi, nat, 0)) != hipSuccess) return err;
    if ((err = phase_upload(b.ph[BP_MDCLEAR], mc, nmc, 0)) != hipSuccess) return err;
    if ((err = phase_upload(b.ph[BP_MDBIN], mb, nat, 0)) != hipSuccess) return err;
    if ((err = phase_upload(b.ph[BP_CHUNKSUM], cks, nch, 0)) != hipSuccess) return err;
    if (b.d_out && (err = phase_upload(b.ph[BP_STATS_OUT], so, none, 0)) != hipSuccess)
        return err;
    return hipSuccess;
}

void nlist_batch_launch(Batch& b, int phase, hipStream_t s)
{
    switch (phase) {
    case BP_BIN: phase_launch<BinGather<false>>(b.ph[phase], s); break;
    case BP_MDCLEAR: phase_launch<ClearInts>(b.ph[phase], s); break;
    case BP_MDBIN: phase_launch<MdBin>(b.ph[phase], s); break;
    case BP_STATS_OUT: phase_launch<StatsOut>(b.ph[phase], s); break;
    case BP_CHUNKSUM: phase_launch<ChunkSum>(b.ph[phase], s); break;
    default: break;
    }
}

}  // namespace rbmd
