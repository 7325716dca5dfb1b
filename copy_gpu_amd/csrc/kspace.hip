// kspace.hip -- Random Batch Ewald (and full Ewald) k-space launches of the
// force pass: sampler arguments, rho(k) geometry and the per-atom k-space force
// (bodies in kspace.h; the sampler's in md.h).
//
// Reference (paths relative to the reference checkout):
//   sampler target / normaliser S   rbmd/framework/model/RBEPSample.h:38-61, 87-93, 143-175
//   rho(k)                          rbmd/framework/run/worklet/RunWorklet.cpp:1616-1677,
//                                   rbmd/framework/run/ExecutionMD.cpp:412-448
//   RBE force                       RunWorklet.cpp:1508-1548, ExecForceFunction.h:247-269
//   Ewald force / energy            ExecForceFunction.h:226-245, output/ThermoOutput.cpp:209-255
#include "kspace.h"
#include "state.h"

namespace rbmd {

void rho_geometry(const Engine& e, int* atoms_per_block, int* nbx, int* nkt)
{
    const int n = (int)e.n;
    *nkt = (e.P + 63) / 64;
    int apb;
    if (e.rho_apb > 0) {
        apb = e.rho_apb;
    } else {
        int want = 2048 / *nkt;
        if (want < 1) want = 1;
        apb = (n + want - 1) / want;
    }
    // the partials [nbx][P][2] must fit the kpart buffer
    const int64_t max_nbx = e.P > 0 ? e.kpart_cap / (2 * (int64_t)e.P) : 1;
    if (max_nbx >= 1 && (int64_t)apb * max_nbx < (int64_t)n)
        apb = (int)(((int64_t)n + max_nbx - 1) / max_nbx);
    apb = ((apb + 63) / 64) * 64;
    if (apb < 64) apb = 64;
    *atoms_per_block = apb;
    *nbx = (n + apb - 1) / apb;
    if (*nbx < 1) *nbx = 1;
}

namespace {

__global__ void k_fill(double* __restrict__ a, int n, double v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

}  // namespace

// ================================================================= launchers

SampleArgs sample_args(const Engine& e, int P, uint64_t seed, const uint64_t* step_host)
{
    SampleArgs sa;
    sa.P = P;
    sa.seed = seed;
    sa.step = step_host ? *step_host : 0ull;
    sa.step_dev = step_host ? nullptr : e.d_step;
    sa.cdf = e.kcdf;
    sa.M = make_int3(e.kM[0], e.kM[1], e.kM[2]);
    sa.w = e.S / (double)P;
    sa.gp = e.gp;
    sa.w_out = e.gp.cdf ? e.S / ((1.0 - e.gp.lambda) * (double)P) : 0.0;
    sa.km = e.km;
    sa.kw = e.kw;
    return sa;
}

void launch_kweights_default(Engine& e, hipStream_t s)
{
    k_fill<<<(e.P + 255) / 256, 256, 0, s>>>(e.kw, e.P, e.S / (double)e.P);
}

void launch_kforce(Engine& e, const double* x, const double* y, const double* z, void* fx,
                   void* fy, void* fz, hipStream_t s)
{
    if (e.ew.on) {
        launch_ewald_force(e, x, y, z, (double*)fx, (double*)fy, (double*)fz, s);
        return;
    }
    ScopedTimer t(e, P_KFORCE, s);
    auto go = [&](auto t) {
        using T = decltype(t);
        const int blocks = kforce_blocks(e);
        const auto a = kforce_args<T>(e, x, y, z, fx, fy, fz, nullptr, nullptr, nullptr, nullptr, 0.0);
        kf_dispatch<T>(kf_staged<T>(blocks, a.P), [&](auto st) {
            k_one<KForce<T, false, decltype(st)::value>><<<blocks, kKfThreads, 0, s>>>(a);
        });
    };
    if (e.precision == 32) go(0.0f);
    else go(0.0);
}

}  // namespace rbmd
