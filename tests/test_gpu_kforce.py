"""The k-space force with its coefficients in LDS (FP32 launches of at most one workgroup per CU
and many k-vectors) and by scalar loads: against the oracle on both sides of the rule, the same
bits from both, and the time of a small launch with many k-vectors."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype)


# 128 k-vectors and 256 workgroups of 64 atoms are the last without and with the stage, which
# holds 512 k-vectors
@pytest.mark.parametrize("n,P", [(4097, 128), (4097, 129), (5000, 512), (5000, 513), (16384, 200),
                                 (16385, 200), (16384, 1025)])
def test_forces_against_oracle(n, P):
    import oracle
    from copy_gpu_amd import force as FM

    rng = np.random.default_rng(n + P)
    Lb, alpha = np.array([31.0, 22.5, 40.0]), 0.1
    pos = rng.uniform(0, 1, (3, n)) * Lb[:, None]
    q = rng.uniform(-1, 1, n)
    g = np.stack(np.meshgrid(*[np.arange(-6, 7)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[(g != 0).any(1)]
    m = g[rng.permutation(len(g))[:P]].astype(np.int32)
    w = rng.uniform(0.5, 2.0, P)
    F0 = rng.normal(0, 1, (3, n)).astype(np.float32)
    F = [_dev(a, torch.float32) for a in F0]
    FM.kspace_compute(tuple(Lb), alpha, *[_dev(a) for a in pos], _dev(q),
                      _dev(m.reshape(-1), torch.int32), _dev(w), *F, precision=32)
    Fk, _ = oracle.kspace_forces(*pos, q, Lb, alpha, m, w)
    re, im = oracle.rho(*pos, q, Lb, m)
    # a component is a sum of P terms of at most |q| 4 pi w |k| |rho| / (V k^2), each with a sine
    # of 1.3e-7 and a structure factor of 1e-6 sum |q|; the sum is rounded onto F0
    k = 2 * np.pi * m / Lb
    term = np.abs(q).max() * (4 * np.pi * w / (Lb.prod() * np.sqrt((k * k).sum(1))) *
                              (np.hypot(re, im) + np.abs(q).sum())).sum()
    out = np.stack([a.double().cpu().numpy() for a in F]) - F0
    assert np.abs(out.T - Fk).max() <= 1e-6 * term + 2.4e-7 * np.abs(F0).max()


@pytest.mark.parametrize("R", [2, 6])
def test_batch_and_single_run_same_bits(gpu, R):
    """Six replicas of 3,000 ions fill more than one workgroup per CU (scalar loads); two, or one
    alone, do not (LDS stage).  First with 100 k-vectors, which none stages, then with 200."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce, systems
    from copy_gpu_amd.batch import ReplicaBatch

    n, P = 3000, 200
    x, y, z, q, L = systems.random_ions(n, 0.3, 0.8, seed=21)
    v = systems.velocities(n, 1.0, seed=21)
    cfg = ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=5.0, alpha=0.5, skin=0.3,
                      kspace="RBE", coulomb_sample_num=P, precision=32, n_max=n)
    b = ReplicaBatch([cfg] * R)
    single = LJCutCoulKspaceForce(cfg)
    states = []
    for f in [*b.replicas, single]:
        f.Init(_dev(q))
        st = [_dev(a) for a in (x, y, z, *v)] + \
            [torch.zeros(n, device="cuda") for _ in range(3)] + \
            [torch.zeros(3 * n, device="cuda", dtype=torch.int32)]
        states.append(st)
    for P, step0 in ((100, 1), (200, 7)):
        for f, st in zip([*b.replicas, single], states):
            f.sample_kvectors(P, 5, 0)
            f.Execute(*st[:3], *st[6:9])
        b.md_run([tuple(st) for st in states[:R]], dt=0.002, nsteps=6, seeds=[5] * R, step0=step0)
        st = states[R]
        single.md_run(*st[:9], dt=0.002, nsteps=6, seed=5, step0=step0, img=st[9])
    torch.cuda.synchronize()
    for s in states[:R]:
        for a, c in zip(s, st):
            assert torch.equal(a, c)


def test_time_of_many_kvectors_at_few_atoms(gpu):
    """2,000 ions, 8,000 k-vectors: an FP32 sine and product take a fraction of the FP64 ones, and
    the wait for the coefficients must not make up for it."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    n, m, L = 2000, 13, 19.5
    g = np.random.default_rng(3).permutation(m ** 3)[:n]
    pos = [_dev(a) for a in (np.stack([g % m, g // m % m, g // m ** 2]) + 0.5) * 1.5]
    us = {}
    for precision in (32, 64):
        f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=1.0, coulomb_cut=1.0,
                                             alpha=0.5, kspace="RBE", coulomb_sample_num=8000,
                                             precision=precision, n_max=n))
        f.Init(_dev(np.where(g % 2, 1.0, -1.0)))
        f.sample_kvectors(8000, 5, 0)
        F = [torch.zeros(n, device="cuda", dtype=f.fdtype) for _ in range(3)]
        for _ in range(3):
            f.Execute(*pos, *F)
        f.set_timing(True)
        for _ in range(20):
            f.Execute(*pos, *F)
        us[precision] = 1e3 * f.timing("kforce")[0]
    print(f"k-space force: FP32 {us[32]:.1f} us, FP64 {us[64]:.1f} us", flush=True)
    assert us[32] < 0.47 * us[64]
