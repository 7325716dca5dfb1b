// kcompute.hip -- the RBE / Ewald k-space step of a given k-list without a force
// handle: structure factor rho(k) = sum_j q_j exp(i k.r_j) (per-workgroup partials,
// then a fixed-order FP64 reduction per k with the force coefficients and per-k
// energy / virial terms) and the k-space force scatter, with the kernel bodies of
// the force pass (kspace.h: RhoPartial, RhoFinal, kforce_block).
//
// Reference (paths relative to the reference checkout):
//   ExecutionMD::ComputeRBEEleForce      rbmd/framework/run/ExecutionMD.cpp:389-410
//   ComputeNewChargeStructureFactorRBE   rbmd/framework/run/ExecutionMD.cpp:412-448
//   rho(k) worklet                       rbmd/framework/run/worklet/RunWorklet.cpp:1616-1677
//   RBE force worklet                    RunWorklet.cpp:1508-1548, ExecForceFunction.h:247-269
//
// Calls of few atoms and k-vectors that ask for rho need no scratch (ks_small): one workgroup
// per k writes rho, and the force kernel forms coefficients and terms from it (1,000 atoms, 124
// k-vectors, FP64: 92 -> 44 us a call).  For others rbmd_kspace_compute allocates its scratch (partials,
// rho, per-k coefficients and terms, weights) for the call.  rbmd_kspace_compute_noalloc
// runs the same kernels on a fixed block of device memory (`scratch` below, 4 MiB per
// device) and allocates nothing, for callers that cannot call hipMalloc.

#include <mutex>

#include "kspace.h"
#include "state.h"

namespace rbmd {

double rbe_S(double alpha, const double* L);

namespace {

// Scratch of one call, carved from one block of device memory: weights [P],
// partial structure factors [nbx][P][2], rho [P][2], coefficients KCoef<T>[P],
// per-k energy / virial terms [7][P].  Offsets are multiples of 256 bytes.
struct KsLayout {
    size_t kw, kpart, rho, coef, kev, total;
};

inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }

// The force pass's rho(k) geometry for n atoms and P k-vectors (kspace.hip
// rho_geometry with the default workgroup size): about 2048 workgroups of 64 k's
// by atom tiles, so the partials hold at most 2048 x 64 x 2 doubles.
void ks_geometry(int64_t n, int P, int* apb, int* nbx, int* nkt)
{
    *nkt = (P + 63) / 64;
    int want = 2048 / *nkt;
    if (want < 1) want = 1;
    int a = (int)((n + want - 1) / want);
    a = ((a + 63) / 64) * 64;
    if (a < 64) a = 64;
    *apb = a;
    *nbx = (int)((n + a - 1) / a);
    if (*nbx < 1) *nbx = 1;
}

KsLayout ks_layout(int64_t n, int P)
{
    int apb, nbx, nkt;
    ks_geometry(n, P, &apb, &nbx, &nkt);
    KsLayout l;
    size_t o = 0;
    l.kw = o;
    o += up256((size_t)P * 8);
    l.kpart = o;
    o += up256((size_t)nbx * P * 2 * 8);
    l.rho = o;
    o += up256((size_t)P * 2 * 8);
    l.coef = o;
    o += up256((size_t)P * sizeof(KCoef<double>));
    l.kev = o;
    o += up256((size_t)P * 7 * 8);
    l.total = o;
    return l;
}

}  // namespace

namespace {

constexpr int kKsSmall = 4096;    // most atoms of the calls without scratch
constexpr int kKsSmallP = 16384;  // and most k-vectors

// rho(k) of at most kKsSmall atoms: one workgroup per k, each thread 16 atoms at most, so no
// partials go through memory.  (With more atoms the loop would be longer than the reduction
// it saves: one workgroup takes 4 us for 4,096.)
template <typename T>
__global__ __launch_bounds__(256) void k_ks_rho(const double* __restrict__ x,
                                                const double* __restrict__ y,
                                                const double* __restrict__ z,
                                                const double* __restrict__ q, int n, Box box,
                                                const int32_t* __restrict__ km,
                                                double* __restrict__ rho)
{
#pragma clang fp contract(off)
    __shared__ double red[4][2];
    const int k = blockIdx.x, t = threadIdx.x;
    const double mx = km[3 * (size_t)k], my = km[3 * (size_t)k + 1], mz = km[3 * (size_t)k + 2];
    T br = 0, bi = 0;
    // FP32: thread (tile, w) sums the 16 atoms 64 tile + w, + 4, ... as wave w of RhoPartial
    // does, so that rounding is the same for calls of any size; FP64: strided
    constexpr bool kBlocks = sizeof(T) == 4;
    static_assert(kRhoFlush == 16 && kKsSmall <= 256 * kRhoFlush, "one block per thread");
    const int step = kBlocks ? 4 : 256, i0 = kBlocks ? 64 * (t >> 2) + (t & 3) : t;
    const int i1 = kBlocks ? min(n, 64 * (t >> 2) + 64) : n;
    for (int i = i0; i < i1; i += step) {
        const double sx = (x[i] - box.lo[0]) * box.invL[0], sy = (y[i] - box.lo[1]) * box.invL[1],
                     sz = (z[i] - box.lo[2]) * box.invL[2];
        T sn, cs;
        sincos2pi<T>(fma(mz, sz, fma(my, sy, mx * sx)), &sn, &cs);
        const T qa = (T)q[i];
        br = fma_t(qa, cs, br);
        bi = fma_t(qa, sn, bi);
    }
    const double re = wave_sum_dpp((double)br), im = wave_sum_dpp((double)bi);
    if ((t & 63) == 0) {
        red[t >> 6][0] = re;
        red[t >> 6][1] = im;
    }
    __syncthreads();
    if (t < 2) rho[2 * (size_t)k + t] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

// The k-space forces (workgroups [0, nforce)) and, one workgroup each, the seven sums of
// energy and virial terms in a fixed order.  DIRECT: coefficients and terms from rho, by each
// workgroup for itself; else those that the rho(k) reduction stored.  STAGED: in LDS.
template <typename T, bool DIRECT, bool STAGED = DIRECT>
struct KsForce {
    static constexpr int kThreads = kKfThreads;
    struct Args {
        KForceArgs<T> f;
        int nforce;
        double alpha, qqr2e;
        const int32_t* m;
        const double* w;  // or null: wdef
        double wdef;
        const double* rho;
        const double* kev;
        double* ev;
    };
    __device__ static KCoef<T> coef(const Args& A, int k, double* ev)
    {
        return rho_terms<T>(A.f.box, A.alpha, A.qqr2e, A.m + 3 * (size_t)k, A.w ? A.w[k] : A.wdef,
                            A.rho[2 * (size_t)k], A.rho[2 * (size_t)k + 1], ev);
    }
    __device__ static void run(const Args& A, int blk, int)
    {
        __shared__ KForceLds<T, STAGED> L;
        if (blk < A.nforce) {
            auto pre = [](int) { return 0; };
            auto fin = [&](int i, T f0, T f1, T f2, int) {
                A.f.fx[i] = f0;
                A.f.fy[i] = f1;
                A.f.fz[i] = f2;
            };
            if constexpr (DIRECT) {
                auto of_rho = [&](int k) {
                    double ev[7];
                    return coef(A, k, ev);
                };
                kforce_block(A.f, blk, L, of_rho, pre, fin);
            } else {
                kforce_block(A.f, blk, L, pre, fin);
            }
            return;
        }
        double* red = (double*)&L;
        const int c = blk - A.nforce, t = threadIdx.x;
        double v = 0.0;
        for (int k = t; k < A.f.P; k += kThreads) {
            if constexpr (DIRECT) {
                double ev[7];
                coef(A, k, ev);
                double e = ev[0];
#pragma unroll
                for (int d = 1; d < 7; ++d) e = c == d ? ev[d] : e;
                v += e;
            } else {
                v += A.kev[(size_t)c * A.f.P + k];
            }
        }
        v = wave_sum_dpp(v);
        if ((t & 63) == 0) red[t >> 6] = v;
        __syncthreads();
        if (t == 0) {
            double s = 0.0;
            for (int w = 0; w < kThreads / 64; ++w) s += red[w];
            A.ev[c] = s;
        }
    }
};

__global__ void k_fill_w(double* __restrict__ a, int n, double v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

struct KsCall {
    double lo[3], L[3], alpha, qqr2e;
    int precision;
    int64_t n;
    const double *x, *y, *z, *q;
    int P;
    const int32_t* m;
    const double* w;
    void *fx, *fy, *fz;
    double* rho_out;
    double* ev_out;
};

// Whether a call runs without scratch memory; the same for both entry points, which give the
// same bits.  Every k reads all positions again and every force workgroup forms all
// coefficients, so the general path overtakes with P, though it has to allocate (or, in the
// second figure of each, has the fixed scratch).  Without and with scratch, us: FP32, 4,096
// atoms 117 / 97 and 127 / 70 for 4,000 k-vectors, 222 / 202 and 185 / 127 for 8,192, 790 and
// 489 for 30,000; 1,000 atoms 255 and 275 for 16,000.  FP64, 4,096 atoms 210 / 190 and 230 /
// 175 for 4,000, 573 and 561 for 12,000; 1,000 atoms 665 and 640 for 16,000.
bool ks_small(const KsCall& c)
{
    const int64_t most = (int64_t)1 << (c.precision == 32 ? 24 : 25);
    return c.rho_out && c.n <= kKsSmall && c.P <= kKsSmallP && c.n * c.P <= most;
}

// buf: scratch, or null for a call that runs without (ks_small).
template <typename T>
void ks_launch(const KsCall& c, char* buf, hipStream_t s)
{
    Box box;
    for (int d = 0; d < 3; ++d) {
        box.lo[d] = c.lo[d];
        box.L[d] = c.L[d];
        box.invL[d] = 1.0 / c.L[d];
    }
    KForceArgs<T> ka{};
    ka.x = c.x;
    ka.y = c.y;
    ka.z = c.z;
    ka.q = c.q;
    ka.n = (int)c.n;
    ka.box = box;
    ka.P = c.P;
    ka.fx = (T*)c.fx;
    ka.fy = (T*)c.fy;
    ka.fz = (T*)c.fz;
    ka.slices = kf_slices(c.n, c.P);
    const int nforce = c.n > 0 ? kf_blocks(c.n, ka.slices) : 0, nev = c.ev_out ? 7 : 0;
    const double wdef = c.w ? 0.0 : rbe_S(c.alpha, c.L) / (double)c.P;
    if (!buf) {
        k_ks_rho<T><<<c.P, 256, 0, s>>>(c.x, c.y, c.z, c.q, (int)c.n, box, c.m, c.rho_out);
        if (nforce + nev > 0)
            k_one<KsForce<T, true>><<<nforce + nev, kKfThreads, 0, s>>>(
                typename KsForce<T, true>::Args{ka, nforce, c.alpha, c.qqr2e, c.m, c.w, wdef,
                                                c.rho_out, nullptr, c.ev_out});
        return;
    }
    const KsLayout l = ks_layout(c.n, c.P);
    double* kw = (double*)(buf + l.kw);
    double* kpart = (double*)(buf + l.kpart);
    double* rho = c.rho_out ? c.rho_out : (double*)(buf + l.rho);
    KCoef<T>* coef = (KCoef<T>*)(buf + l.coef);
    double* kev = (double*)(buf + l.kev);
    const double* w = c.w;
    if (!w) {
        k_fill_w<<<(c.P + 255) / 256, 256, 0, s>>>(kw, c.P, wdef);
        w = kw;
    }
    int apb, nbx, nkt;
    ks_geometry(c.n, c.P, &apb, &nbx, &nkt);
    k_one<RhoPartial<T>><<<nbx * nkt, kRhoBlock, 0, s>>>(typename RhoPartial<T>::Args{
        c.x, c.y, c.z, c.q, (int)c.n, apb, nbx, box, c.m, c.P, kpart});
    k_one<RhoFinal<T>><<<c.P, RhoFinal<T>::kThreads, 0, s>>>(RhoFinalArgs<T>{
        kpart, nbx, c.P, c.m, w, box, c.alpha, c.qqr2e, rho, coef, kev, nullptr});
    ka.coef = coef;
    if (nforce + nev > 0)
        kf_dispatch<T>(kf_staged<T>(nforce, c.P), [&](auto sg) {
            using K = KsForce<T, false, decltype(sg)::value>;
            k_one<K><<<nforce + nev, kKfThreads, 0, s>>>(typename K::Args{
                ka, nforce, c.alpha, c.qqr2e, c.m, w, wdef, rho, kev, c.ev_out});
        });
}

thread_local std::string g_ks_err;

int ks_fail(int code, const std::string& msg)
{
    g_ks_err = msg;
    return code;
}

int ks_check(const KsCall& c)
{
    if (c.precision != 32 && c.precision != 64)
        return ks_fail(RBMD_ERR_INVALID, "precision must be 32 or 64");
    if (c.n < 0 || c.n > (int64_t)INT32_MAX / 2 || c.P < 1)
        return ks_fail(RBMD_ERR_INVALID, "n must be in [0, 2^30) and P >= 1");
    if (!(c.alpha > 0)) return ks_fail(RBMD_ERR_INVALID, "alpha must be positive");
    for (int d = 0; d < 3; ++d)
        if (!(c.L[d] > 0)) return ks_fail(RBMD_ERR_INVALID, "box lengths must be positive");
    if (!c.m) return ks_fail(RBMD_ERR_INVALID, "null k-vector array");
    if (c.n > 0 && (!c.x || !c.y || !c.z || !c.q || !c.fx || !c.fy || !c.fz))
        return ks_fail(RBMD_ERR_INVALID, "null atom or force array");
    return RBMD_OK;
}

KsCall ks_call(const rbmd_kspace_params* p, int64_t n, const double* x, const double* y,
               const double* z, const double* q, int32_t P, const int32_t* m, const double* w,
               void* fx, void* fy, void* fz, double* rho, double* ev)
{
    KsCall c{};
    for (int d = 0; d < 3; ++d) {
        c.lo[d] = p->box_lo[d];
        c.L[d] = p->box_len[d];
    }
    c.alpha = p->alpha;
    c.qqr2e = p->qqr2e;
    c.precision = p->precision;
    c.n = n;
    c.x = x;
    c.y = y;
    c.z = z;
    c.q = q;
    c.P = P;
    c.m = m;
    c.w = w;
    c.fx = fx;
    c.fy = fy;
    c.fz = fz;
    c.rho_out = rho;
    c.ev_out = ev;
    return c;
}

void ks_dispatch(const KsCall& c, char* buf, hipStream_t s)
{
    if (c.precision == 32) ks_launch<float>(c, buf, s);
    else ks_launch<double>(c, buf, s);
}

}  // namespace
}  // namespace rbmd

// Fixed scratch of rbmd_kspace_compute_noalloc, one copy per device, held until the
// process ends.  4 MiB covers every P <= 8192 at any n: the partials hold at most
// 2048 x 64 x 2 doubles (2 MiB, ks_geometry) and the per-k arrays 120 bytes per k.
// In host code `scratch` is only the symbol's host-side stand-in; kernels take the
// device address hipGetSymbolAddress returns (ks_scratch_ptr).
constexpr size_t kKsScratchBytes = (size_t)4 << 20;
constexpr int kKsScratchMaxP = 8192;
static __device__ __align__(256) unsigned char scratch[kKsScratchBytes];

namespace rbmd {
namespace {

constexpr int kKsMaxDevices = 64;
std::mutex g_ks_scratch_mu;
char* g_ks_scratch[kKsMaxDevices] = {};

// Device address of the current device's `scratch`, looked up once per device.
int ks_scratch_ptr(char** out)
{
    int dev = -1;
    hipError_t st = hipGetDevice(&dev);
    if (st != hipSuccess)
        return ks_fail(RBMD_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(st));
    if (dev < 0 || dev >= kKsMaxDevices) return ks_fail(RBMD_ERR_HIP, "device index out of range");
    std::lock_guard<std::mutex> lk(g_ks_scratch_mu);
    if (!g_ks_scratch[dev]) {
        void* p = nullptr;
        st = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (st != hipSuccess || !p)
            return ks_fail(RBMD_ERR_HIP,
                           std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(st));
        g_ks_scratch[dev] = (char*)p;
    }
    *out = g_ks_scratch[dev];
    return RBMD_OK;
}

}  // namespace
}  // namespace rbmd

using namespace rbmd;

extern "C" {

const char* rbmd_kspace_last_error(void) { return g_ks_err.c_str(); }

int rbmd_kspace_compute(const rbmd_kspace_params* p, int64_t n, const double* x, const double* y,
                        const double* z, const double* q, int32_t P, const int32_t* m,
                        const double* w, void* fx, void* fy, void* fz, double* rho, double* ev,
                        void* stream)
{
    g_ks_err.clear();
    if (!p) return ks_fail(RBMD_ERR_INVALID, "null parameters");
    const KsCall c = ks_call(p, n, x, y, z, q, P, m, w, fx, fy, fz, rho, ev);
    int rc = ks_check(c);
    if (rc != RBMD_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    char* buf = nullptr;
    hipError_t st;
    if (!ks_small(c)) {
        st = hipMalloc((void**)&buf, ks_layout(n, P).total);
        if (st != hipSuccess)
            return ks_fail(RBMD_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(st));
    }
    ks_dispatch(c, buf, s);
    st = hipGetLastError();
    hipError_t st2 = hipStreamSynchronize(s);
    if (buf) (void)hipFree(buf);
    if (st != hipSuccess) return ks_fail(RBMD_ERR_HIP, std::string("launch: ") + hipGetErrorString(st));
    if (st2 != hipSuccess)
        return ks_fail(RBMD_ERR_HIP, std::string("hipStreamSynchronize: ") + hipGetErrorString(st2));
    return RBMD_OK;
}

int rbmd_kspace_compute_noalloc(const rbmd_kspace_params* p, int64_t n, const double* x,
                                const double* y, const double* z, const double* q, int32_t P,
                                const int32_t* m, const double* w, void* fx, void* fy, void* fz,
                                double* rho, double* ev, void* stream)
{
    g_ks_err.clear();
    if (!p) return ks_fail(RBMD_ERR_INVALID, "null parameters");
    const KsCall c = ks_call(p, n, x, y, z, q, P, m, w, fx, fy, fz, rho, ev);
    int rc = ks_check(c);
    if (rc != RBMD_OK) return rc;
    if (P > kKsScratchMaxP || ks_layout(n, P).total > kKsScratchBytes)
        return ks_fail(RBMD_ERR_INVALID,
                       "rbmd_kspace_compute_noalloc: P = " + std::to_string(P) +
                           " exceeds the fixed scratch (P <= " +
                           std::to_string(kKsScratchMaxP) + ")");
    char* buf = nullptr;
    if (!ks_small(c)) {
        rc = ks_scratch_ptr(&buf);
        if (rc != RBMD_OK) return rc;
    }
    ks_dispatch(c, buf, (hipStream_t)stream);
    const hipError_t st = hipGetLastError();
    if (st != hipSuccess) return ks_fail(RBMD_ERR_HIP, std::string("launch: ") + hipGetErrorString(st));
    return RBMD_OK;
}

}  // extern "C"
