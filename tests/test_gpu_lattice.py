"""Structure factors of a whole lattice box by FP64 matrix products, against the direct
FP64 sum over atoms: box edges and atom counts around the tile, stage and slice sizes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _direct(pos, q, m, lo, L):
    """rho(m) in extended precision (numpy long double phases)."""
    s = (pos.astype(np.longdouble) - np.longdouble(lo)[:, None]) / np.longdouble(L)[:, None]
    re, im = np.zeros(len(m)), np.zeros(len(m))
    for a in range(0, len(m), 512):
        ph = m[a:a + 512].astype(np.longdouble) @ s
        ph = (2.0 * np.pi * (ph - np.rint(ph)).astype(np.float64))
        re[a:a + 512], im[a:a + 512] = np.cos(ph) @ q, np.sin(ph) @ q
    return re, im


# rows (2Mg+1)^2 and columns 2Mg: below and just past one 256-row block (7, 8), one to five
# 16-column tiles and two column blocks (33); n around a 32-atom stage and several slices
@pytest.mark.parametrize("Mg,n", [(1, 1), (1, 31), (2, 33), (7, 64), (8, 257), (12, 1000),
                                  (16, 129), (24, 2049), (33, 300)])
def test_spectrum_against_direct_sum(Mg, n):
    from copy_gpu_amd import proposal as PR

    rng = np.random.default_rng(100 * Mg + n)
    lo, L = np.array([-1.0, 2.0, 0.5]), np.array([9.0, 11.0, 7.5])
    # two snapshots, positions in and out of the box (images are equivalent)
    snaps = [lo[:, None] + L[:, None] * rng.uniform(-0.5, 1.5, (3, n)) for _ in range(2)]
    q = rng.uniform(-1.5, 1.5, n)
    dev = [tuple(torch.as_tensor(a.copy()).cuda() for a in s) for s in snaps]
    S2 = PR.spectrum(dev, torch.as_tensor(q).cuda(), tuple(L), 0.5, Mg, box_lo=tuple(lo))
    m = PR.lattice_grid(Mg)
    ref, bound = np.zeros(len(m)), np.zeros(len(m))
    # per term: phase rounding of about 4 Mg 2^-53 turns from (x - lo) alone, and a few
    # roundings of the products; |rho| error <= n |q| (2 pi 4 Mg + 16) 2^-53
    for s in snaps:
        re, im = _direct(s, q, m, lo, L)
        ref += re * re + im * im
        e = np.abs(q).sum() * (2 * np.pi * 4 * Mg + 16 + n / 8) * 2.0 ** -53
        bound += 2 * np.hypot(re, im) * e + e * e + 1e-15 * (re * re + im * im)
    ref[len(m) // 2] = 0.0
    assert S2[len(m) // 2] == 0.0
    assert np.array_equal(S2, S2[::-1])
    err = np.abs(S2 - ref / 2) - bound
    assert (err <= 0).all(), (int(err.argmax()), m[err.argmax()], S2[err.argmax()],
                              ref[err.argmax()] / 2)


def test_spectrum_refuses_what_it_cannot_take():
    from copy_gpu_amd import proposal as PR

    q = torch.ones(8, device="cuda", dtype=torch.float64)
    x = torch.zeros(8, device="cuda", dtype=torch.float64)
    for kw in ({"Mg": 0}, {"alpha": 0.0}, {"box_len": (1.0, 9.0, 9.0)}):
        a = {"box_len": (9.0, 9.0, 9.0), "alpha": 0.5, "Mg": 4, **kw}
        with pytest.raises(PR.RBMDError):
            PR.spectrum([(x, x, x)], q, a["box_len"], a["alpha"], a["Mg"])
    with pytest.raises(AssertionError):
        PR.spectrum([(x[:4], x, x)], q, (9.0, 9.0, 9.0), 0.5, 4)
    assert not PR.spectrum([], q, (9.0, 9.0, 9.0), 0.5, 4).any()


# full Ewald in FP64 through the lattice box: 64-column blocks (1 to 3), a wide row basis, and
# atom counts around a wave's 16 and a workgroup's 64
@pytest.mark.parametrize("L,n", [((6.0, 7.0, 6.5), 2), ((6.0, 7.0, 6.5), 17), ((9.0, 7.0, 25.0), 64),
                                 ((7.0, 60.0, 9.0), 300), ((7.0, 9.0, 60.0), 257),
                                 ((31.0, 6.0, 8.0), 65)])
def test_ewald_against_oracle(L, n):
    import oracle
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(n)
    Lb, lo = np.array(L), np.array([0.5, -1.0, 0.0])
    alpha, tol = 0.5, 1e-12
    # a jittered lattice: no pair much closer than its spacing
    g = np.ceil((n / Lb.prod()) ** (1 / 3) * Lb).astype(int) + 1
    cell = np.stack(np.meshgrid(*[np.arange(k) for k in g], indexing="ij"), -1).reshape(-1, 3)
    pick = cell[rng.permutation(len(cell))[:n]]
    pos = lo + (pick + 0.5 + rng.uniform(-0.15, 0.15, (n, 3))) * (Lb / g)
    x, y, z = (np.ascontiguousarray(pos[:, d]) for d in range(3))
    q = rng.uniform(-1.0, 1.0, n)
    f = LJCutCoulKspaceForce(ForceConfig(box_len=L, box_lo=tuple(lo), cut_off=2.5, coulomb_cut=2.9,
                                         skin=0.3, alpha=alpha, kspace="EWALD", precision=64,
                                         ewald_tol=tol, n_max=n + 7))
    dev = lambda a: torch.as_tensor(a).cuda()  # noqa: E731
    f.Init(dev(q))
    X, F = [dev(a) for a in (x, y, z)], [torch.zeros(n, device="cuda", dtype=torch.float64)
                                         for _ in range(3)]
    for _ in range(2):  # the second evaluation finds the first's sums and coefficients
        f.Execute(*X, *F, energy_virial=True)
    m, w, re, im = f.kspace()
    got = torch.stack(F, 1).cpu().numpy()
    Fk, evk = oracle.kspace_forces(x - lo[0], y - lo[1], z - lo[2], q, Lb, alpha, m, w)
    Fp, _ = oracle.pair_forces(x, y, z, q, lo, Lb, 2.5, 2.9, alpha)
    # the pair part agrees to 1e-12 of itself elsewhere; the k-space part is judged on its own
    assert np.linalg.norm(got - Fp - Fk) <= 1e-12 * (np.linalg.norm(Fp) + np.linalg.norm(Fk))
    r, i = _direct(pos.T, q, m, lo, Lb)
    bound = np.abs(q).sum() * (2 * np.pi * 4 * np.abs(m).max() + 16 + n / 8) * 2.0 ** -53
    assert np.abs(re - r).max() <= bound and np.abs(im - i).max() <= bound
    assert abs(f.energy_virial()["e_kspace"] - evk[0]) <= 1e-12 * abs(evk[0])


# the handle-free k-space step at most / above 4,096 atoms (no scratch / scratch), one atom,
# with and without weights, more k-vectors than one LDS stage (512)
@pytest.mark.parametrize("n,P,weights,precision", [
    (1, 1, True, 64), (255, 7, False, 64), (257, 600, True, 64), (4096, 124, True, 32),
    (4097, 124, True, 64), (4097, 65, False, 32)])
def test_kspace_compute_against_oracle(n, P, weights, precision):
    import oracle
    from copy_gpu_amd import force as FM
    from copy_gpu_amd import systems

    rng = np.random.default_rng(n + P)
    Lb, alpha = np.array([11.0, 12.5, 10.0]), 0.1
    pos = rng.uniform(0, 1, (3, n)) * Lb[:, None]
    q = rng.uniform(-1, 1, n)
    g = np.stack(np.meshgrid(*[np.arange(-5, 6)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[(g != 0).any(1)]
    m = g[rng.permutation(len(g))[:P]].astype(np.int32)
    w = rng.uniform(0.5, 2.0, P) if weights else None
    dt = torch.float32 if precision == 32 else torch.float64
    dev = lambda a, t=torch.float64: torch.as_tensor(np.ascontiguousarray(a)).cuda().to(t)  # noqa: E731
    F0 = rng.normal(0, 1, (3, n))
    F = [dev(a, dt) for a in F0]
    F0 = np.stack([a.double().cpu().numpy() for a in F])
    rho, ev = FM.kspace_compute(tuple(Lb), alpha, *[dev(a) for a in pos], dev(q),
                                dev(m.reshape(-1), torch.int32), None if w is None else dev(w),
                                *F, precision=precision)
    if w is None:
        _, S = systems.sample_kvectors_host(alpha, Lb, 1, 1, 0)
        w = np.full(P, S / P)
    Fk, evk = oracle.kspace_forces(*pos, q, Lb, alpha, m, w)
    re, im = oracle.rho(*pos, q, Lb, m)
    # FP32: sines of 1.3e-7, products and sums of 16 of them; FP64 as the oracle's own
    tol = 1e-6 if precision == 32 else 1e-12
    got = rho.cpu().numpy()
    s = np.abs(q).sum()
    assert np.abs(got - np.stack([re, im], 1)).max() <= tol * s
    k = 2 * np.pi * m / Lb
    k2 = (k * k).sum(1)
    V = Lb.prod()
    # each force component is a sum of P terms of at most |q| 4 pi w |k| |rho| / (V k^2), each
    # with its own sine and structure factor
    term = np.abs(q).max() * (4 * np.pi * w / (V * np.sqrt(k2)) * (np.hypot(re, im) + s)).sum()
    out = np.stack([a.double().cpu().numpy() for a in F], 0) - F0
    eps = 1.2e-7 if precision == 32 else 2.3e-16
    assert np.abs(out.T - Fk).max() <= tol * term + 2 * eps * np.abs(F0).max()
    e = (w * 2 * np.pi / V * (np.hypot(re, im) + tol * s) ** 2 / k2 * (4 + k2 / alpha)).sum()
    assert np.abs(ev.cpu().numpy() - evk).max() <= 4 * tol * (e + (w * s * s / k2).sum() / V * 2 * np.pi)


# the last and first calls without and with scratch: 2^24 (FP64: 2^25) atoms times k-vectors,
# 16,384 k-vectors
@pytest.mark.parametrize("n,P,precision", [(4096, 4096, 32), (4096, 4097, 32), (4096, 8192, 64),
                                           (4096, 8193, 64), (60, 16384, 64), (60, 16385, 64)])
def test_kspace_compute_either_side_of_scratch(n, P, precision):
    """Both sides against the oracle, with the error model of the test above; the call on the
    fixed scratch gives the same bits."""
    import oracle
    from copy_gpu_amd import force as FM

    rng = np.random.default_rng(n + P)
    Lb, alpha = np.array([31.0, 42.5, 30.0]), 0.1
    pos = rng.uniform(0, 1, (3, n)) * Lb[:, None]
    q = rng.uniform(-1, 1, n)
    g = np.stack(np.meshgrid(*[np.arange(-13, 14)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[(g != 0).any(1)]
    m = g[rng.permutation(len(g))[:P]].astype(np.int32)
    w = rng.uniform(0.5, 2.0, P)
    dt = torch.float32 if precision == 32 else torch.float64
    dev = lambda a, t=torch.float64: torch.as_tensor(np.ascontiguousarray(a)).cuda().to(t)  # noqa: E731
    args = [tuple(Lb), alpha, *[dev(a) for a in pos], dev(q), dev(m.reshape(-1), torch.int32), dev(w)]
    F = [torch.zeros(n, device="cuda", dtype=dt) for _ in range(3)]
    rho, ev = FM.kspace_compute(*args, *F, precision=precision)
    Fk, _ = oracle.kspace_forces(*pos, q, Lb, alpha, m, w)
    re, im = oracle.rho(*pos, q, Lb, m)
    tol = 1e-6 if precision == 32 else 1e-12
    s = np.abs(q).sum()
    assert np.abs(rho.cpu().numpy() - np.stack([re, im], 1)).max() <= tol * s
    k = 2 * np.pi * m / Lb
    term = np.abs(q).max() * (4 * np.pi * w / (Lb.prod() * np.sqrt((k * k).sum(1))) *
                              (np.hypot(re, im) + s)).sum()
    out = np.stack([a.double().cpu().numpy() for a in F])
    assert np.abs(out.T - Fk).max() <= tol * term
    if P <= 8192:
        G = [torch.zeros(n, device="cuda", dtype=dt) for _ in range(3)]
        rho2, ev2 = FM.kspace_compute(*args, *G, precision=precision, noalloc=True)
        torch.cuda.synchronize()
        assert torch.equal(rho, rho2) and torch.equal(ev, ev2)
        assert all(torch.equal(a, b) for a, b in zip(F, G))


def test_handles_and_spectra_of_unequal_boxes():
    """Kernels' limit of dynamic LDS: a full Ewald handle and a spectrum that need more than 64 KiB
    still run after smaller ones have been made and run."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce
    from copy_gpu_amd import proposal as PR

    rng = np.random.default_rng(5)
    n = 200
    q = rng.uniform(-1, 1, n)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()  # noqa: E731

    def handle(L):
        m = np.ceil(np.array(L) / 1.2).astype(int)
        g = rng.permutation(m.prod())[:n]
        p = (np.stack([g % m[0], g // m[0] % m[1], g // (m[0] * m[1])]) + 0.5) * (L / m)[:, None]
        f = LJCutCoulKspaceForce(ForceConfig(box_len=tuple(L), cut_off=2.5, coulomb_cut=3.0,
                                             alpha=0.5, kspace="EWALD", ewald_tol=1e-10,
                                             precision=64, n_max=n))
        f.Init(dev(q))
        return f, [dev(a) for a in p]

    def evaluate(f, p):
        F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
        f.Execute(*p, *F)
        return torch.stack(F)

    big = handle(np.array([8.0, 70.0, 8.0]))
    mmax = np.abs(big[0].kspace()[0]).max(0)
    # the y and x tables of 64 atoms, 80 doubles between rows
    assert (2 * (mmax[1] + 1) + 16) * 80 * 8 > 65536 and mmax[1] <= 103
    first = evaluate(*big)
    small = handle(np.array([8.0, 8.0, 9.0]))
    evaluate(*small)
    assert torch.equal(evaluate(*big), first)

    X = [dev(rng.uniform(0, 20, n)) for _ in range(3)]
    spectrum = lambda Mg: PR.spectrum([tuple(X)], dev(q), (20.0,) * 3, 0.5, Mg)  # noqa: E731
    first = spectrum(60)
    spectrum(2)
    assert np.array_equal(spectrum(60), first)
    c = slice(58, 63)
    cube = first.reshape(121, 121, 121)[c, c, c].ravel()
    assert np.abs(cube - spectrum(2)).max() <= 1e-12 * cube.max()


# 118, 784 and 802 k-vectors: single k-vectors below 800, the lattice box from there
@pytest.mark.parametrize("tol,P", [(1e-3, 118), (3e-11, 784), (2e-11, 802)])
def test_ewald_of_few_kvectors(tol, P):
    import oracle
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(P)
    n, Lb = 60, np.array([6.0, 7.0, 6.5])
    m = rng.permutation(125)[:n]
    pos = (np.stack([m % 5, m // 5 % 5, m // 25]) + 0.5 + rng.uniform(-0.1, 0.1, (3, n))) * Lb[:, None] / 5
    q = rng.uniform(-1.0, 1.0, n)
    f = LJCutCoulKspaceForce(ForceConfig(box_len=tuple(Lb), cut_off=2.5, coulomb_cut=2.9, skin=0.3,
                                         alpha=0.5, kspace="EWALD", precision=64, ewald_tol=tol,
                                         n_max=n))
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()  # noqa: E731
    f.Init(dev(q))
    assert f.stats()["ewald_k"] == P
    F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
    for _ in range(2):
        f.Execute(*[dev(a) for a in pos], *F, energy_virial=True)
    mm, w, re, im = f.kspace()
    Fk, evk = oracle.kspace_forces(*pos, q, Lb, 0.5, mm, w)
    Fp, _ = oracle.pair_forces(*[np.ascontiguousarray(a) for a in pos], q, np.zeros(3), Lb, 2.5, 2.9, 0.5)
    got = torch.stack(F, 1).cpu().numpy()
    assert np.linalg.norm(got - Fp - Fk) <= 1e-12 * (np.linalg.norm(Fp) + np.linalg.norm(Fk))
    r, i = _direct(pos, q, mm, np.zeros(3), Lb)
    bound = np.abs(q).sum() * (2 * np.pi * 4 * np.abs(mm).max() + 16 + n / 8) * 2.0 ** -53
    assert np.abs(re - r).max() <= bound and np.abs(im - i).max() <= bound
    assert abs(f.energy_virial()["e_kspace"] - evk[0]) <= 1e-12 * abs(evk[0])


def test_time_of_few_kvectors():
    """20,000 ions and 46 k-vectors in FP64: a full Ewald evaluation takes no more than 1.3 times
    that of as many sampled k-vectors."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    n, m = 20000, 28
    g = np.random.default_rng(1).permutation(m ** 3)[:n]
    L = 1.5 * m
    X = [torch.as_tensor(a).cuda() for a in (np.stack([g % m, g // m % m, g // m ** 2]) + 0.5) * 1.5]
    q = torch.as_tensor(np.where(g % 2, 1.0, -1.0)).cuda()
    us = {}
    for kind in ("RBE", "EWALD"):
        # |m| <= 2.9 at a tolerance of 1e-4
        alpha = (2 * np.pi * 2.9 / L) ** 2 / (4 * np.log(1e4))
        f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=5.0,
                                             alpha=alpha, kspace=kind, coulomb_sample_num=46,
                                             ewald_tol=1e-4, precision=64, n_max=n))
        f.Init(q)
        if kind == "RBE":
            f.sample_kvectors(46, 1, 0)
        else:
            assert f.stats()["ewald_k"] == 46
        F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        for _ in range(5):
            f.Execute(*X, *F)
        t[0].record()
        for _ in range(30):
            f.Execute(*X, *F)
        t[1].record()
        torch.cuda.synchronize()
        us[kind] = 1e3 * t[0].elapsed_time(t[1]) / 30
    print(f"evaluation: {us}", flush=True)
    assert us["EWALD"] < 1.3 * us["RBE"]
