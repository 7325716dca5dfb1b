"""Verlet rows across the shapes of the list build: candidate blocks (up to 2048 and up to
4096 staged candidates, several blocks per tile, tiles beyond the LDS stage), groups of
home atoms, and pairs at the criterion's small-distance bound.  The rows must equal the
oracle's neighbour sets, bit for bit."""
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SEED = 20261202


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype)


# (cutoff, cells per axis, density): tile candidates about 27 density (cutoff + 0.3)^3
@pytest.mark.parametrize("rc,cells,rho,stage", [
    (1.3, 4, 0.3, 0),     # about 35 candidates, a home cell of one or two atoms
    (2.5, 4, 0.8, 0),     # 470 candidates, 18 home atoms
    (5.0, 3, 0.3, 0),     # 1,200 candidates, 45 home atoms
    (6.4, 3, 0.3, 0),     # 2,440: 32-bit masks, five groups of home atoms
    (7.9, 3, 0.3, 0),     # 4,470: staged in LDS, two blocks
    (8.4, 3, 0.3, 0),     # 5,300: beyond the LDS stage, blocks staged in turn
    (5.0, 3, 0.3, 208),   # blocks of 208 candidates
    (5.0, 2, 0.3, 0),     # two cells per axis: images
])
def test_rows_equal_oracle_sets(orc, gpu, rc, cells, rho, stage):
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce, systems

    r_list = rc + 0.3
    L = 1.013 * cells * r_list
    n = int(rho * L ** 3)
    print(f"case: rc {rc}, {cells} cells per axis, {n} ions, stage {stage}", flush=True)
    sys.stdout.flush()
    x, y, z, q, Lb_ = systems.random_ions(n, n / L ** 3, 0.8, seed=SEED)
    # two pairs astride the smallest accepted distance (d^2 > 1e-4), one on the diagonal
    x[1], y[1], z[1] = x[0] + 0.0099, y[0], z[0]
    x[3], y[3], z[3] = x[2] + 0.0101, y[2], z[2]
    x[5], y[5], z[5] = x[4] + 0.0058, y[4] - 0.0058, z[4] + 0.0058
    f = LJCutCoulKspaceForce(ForceConfig(box_len=(Lb_,) * 3, cut_off=min(rc, 2.5),
                                         coulomb_cut=rc, alpha=0.5, kspace="NONE", n_max=n,
                                         tile_stage=stage))
    f.Init(_dev(q))
    F = [torch.zeros(n, device="cuda") for _ in range(3)]
    f.Execute(_dev(x), _dev(y), _dev(z), *F)
    torch.cuda.synchronize()
    st = f.stats()
    assert st["cells"] == cells ** 3 and st["overflow_rows"] == 0
    assert (st["big_tiles"] > 0) == (st["largest_tile"] >= st["tile_stage"])
    Lb = np.array([Lb_] * 3)
    xw, yw, zw = orc.wrap(x, y, z, np.zeros(3), Lb)
    oo, io = orc.neighbors_images(xw, yw, zw, Lb, r_list)
    og, ig = f.neighbors()
    assert og[-1] == oo[-1]
    for i in range(n):
        assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i
    # rows in their order: the entries within the LJ range come first
    d = np.stack([xw, yw, zw], 1)
    j, i = ig, np.repeat(np.arange(n), np.diff(og))
    dd = d[j] - d[i]
    dd -= Lb * np.round(dd / Lb)
    inner = (dd * dd).sum(1) < (min(rc, 2.5) + 0.3) ** 2
    if cells > 2:
        assert st["inner_entries"] == int(inner.sum())


# random batch rows: one block, blocks staged in turn (208 candidates), two and more blocks of
# 4,096; rows whose hits fit, and rows of which only the kept entries would
@pytest.mark.parametrize("rc,stage,cap,overflow", [
    (5.0, 0, 0, False), (5.0, 208, 0, False), (7.9, 0, 0, False), (8.4, 0, 0, False),
    (5.0, 0, 128, True), (5.0, 208, 128, True)])
def test_random_batch_rows_over_blocks(orc, gpu, rc, stage, cap, overflow):
    """FP64 forces equal the oracle's for the same draws."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce, systems

    L = 1.013 * 3 * (rc + 0.3)
    n, pice, seed = int(0.3 * L ** 3), 3, 78
    print(f"case: random batch rows, rc {rc}, {n} ions, stage {stage}, capacity {cap}", flush=True)
    x, y, z, q, Lb_ = systems.random_ions(n, n / L ** 3, 0.8, seed=SEED + 1)
    Lb = np.array([Lb_] * 3)
    f = LJCutCoulKspaceForce(ForceConfig(box_len=(Lb_,) * 3, cut_off=2.5, coulomb_cut=rc,
                                         alpha=0.5, kspace="NONE", precision=64, n_max=n,
                                         tile_stage=stage, list_capacity=cap,
                                         neighbor_type="RBL", r_core=2.5, rbl_pice=pice,
                                         rbl_seed=seed))
    f.Init(_dev(q))
    F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
    f.Execute(_dev(x), _dev(y), _dev(z), *F)
    torch.cuda.synchronize()
    st = f.stats()
    assert st["builds"] == 1 and (st["overflow_rows"] > 0) == overflow
    assert (st["big_tiles"] > 0) == (st["largest_tile"] >= st["tile_stage"])
    xw, yw, zw = orc.wrap(x, y, z, np.zeros(3), Lb)
    Fo, _ = orc.rbl_forces(xw, yw, zw, q, np.zeros(3), Lb, 2.5, rc, 0.5, 2.5, pice, seed, 1)
    G = np.stack([t.cpu().numpy() for t in F], 1)
    assert np.linalg.norm(G - Fo) < 1e-12 * np.linalg.norm(Fo)


# tiles of at most 64 candidates take one wave per row: n atoms in 27 cells make n candidates of
# every tile, in one cell 27 n, in 2 x 2 x 3 cells 12 cells' atoms up to three times each
@pytest.mark.parametrize("cells,n", [((3, 3, 3), 2), ((3, 3, 3), 63), ((3, 3, 3), 64),
                                     ((3, 3, 3), 65), ((1, 1, 1), 2), ((1, 1, 1), 3),
                                     ((2, 2, 3), 28)])
@pytest.mark.parametrize("neighbors", ["VERLET-LIST", "RBL"])
def test_rows_of_few_candidates(orc, gpu, cells, n, neighbors):
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(n)
    rc, skin = 2.0, 0.3
    # a grid of 12 points per cell edge of 1.1 list radii, so that pairs at every distance occur
    Lb = np.array(cells) * 1.1 * (rc + skin)
    m = 12 * np.array(cells)
    g = rng.permutation(m.prod())[:n]
    p = (np.stack([g % m[0], g // m[0] % m[1], g // (m[0] * m[1])]) + 0.5) * (Lb / m)[:, None]
    if n > 4:  # pairs astride the smallest accepted distance
        p[:, 1] = p[:, 0] + [0.0099, 0, 0]
        p[:, 3] = p[:, 2] + [0, 0.0101, 0]
    f = LJCutCoulKspaceForce(ForceConfig(box_len=tuple(Lb), cut_off=1.0, coulomb_cut=rc, skin=skin,
                                         alpha=0.5, kspace="NONE", precision=64, n_max=n,
                                         neighbor_type=neighbors, r_core=1.0, rbl_pice=1))
    f.Init(_dev(rng.uniform(-1, 1, n)))
    F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
    f.Execute(*[_dev(a) for a in p], *F)
    st = f.stats()
    assert st["cells"] == np.prod(cells) and st["overflow_rows"] == 0
    assert cells != (3, 3, 3) or st["largest_tile"] == n
    w = [np.ascontiguousarray(a) for a in orc.wrap(*p, np.zeros(3), Lb)]
    oo, io = orc.neighbors_images(*w, Lb, rc + skin)
    og, ig = f.neighbors()
    assert og[-1] == oo[-1]
    for i in range(n):
        assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i
    if neighbors == "VERLET-LIST" and min(cells) > 2:
        d = np.stack(w, 1)
        dd = d[ig] - d[np.repeat(np.arange(n), np.diff(og))]
        dd -= Lb * np.round(dd / Lb)
        assert st["inner_entries"] == int(((dd * dd).sum(1) < (1.0 + skin) ** 2).sum())


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("stage", [0, 208])
def test_position_that_is_not_a_number(gpu, sign, stage):
    """An atom at NaN (of either sign bit) is nobody's neighbour: it has no row, and the others
    have the forces of the system without it."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce, systems

    n = 1500
    x, y, z, q, L = systems.random_ions(n, 0.3, 0.8, seed=SEED + 2)
    forces = []
    for bad in (True, False):
        p = np.stack([x, y, z])
        keep = np.arange(n) != 700
        if bad:
            p[0, 700] = np.copysign(np.nan, sign)
        else:
            p = p[:, keep]
        m = p.shape[1]
        f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=5.0,
                                             alpha=0.5, kspace="NONE", precision=64, n_max=m,
                                             tile_stage=stage))
        f.Init(_dev(q if bad else q[keep]))
        F = [torch.zeros(m, device="cuda", dtype=torch.float64) for _ in range(3)]
        f.Execute(*[_dev(a) for a in p], *F)
        st = f.stats()
        assert st["overflow_rows"] == 0
        G = np.stack([t.cpu().numpy() for t in F])
        forces.append(G[:, keep] if bad else G)
        if bad:
            og, _ = f.neighbors()
            assert og[701] == og[700]
    # the same terms in another order: a few hundred, none above the largest force by much
    assert np.abs(forces[0] - forces[1]).max() <= 1e-12 * np.abs(forces[1]).max()


# the longest rows of eight row buffers, of seven, and the longest accepted; one more is refused
@pytest.mark.parametrize("neighbors,cap", [("VERLET-LIST", 8192), ("VERLET-LIST", 8256),
                                           ("VERLET-LIST", 9600), ("VERLET-LIST", 9664),
                                           ("RBL", 9472), ("RBL", 9536), ("RBL", 9600)])
def test_longest_rows(orc, gpu, neighbors, cap):
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce
    from copy_gpu_amd.force import RBMDError

    rng = np.random.default_rng(cap)
    n, L = 1200, 2.5  # one cell: 32,400 candidates of 27 images, rows of some 4,190 n / 1000
    m = 11
    g = rng.permutation(m ** 3)[:n]
    p = (np.stack([g % m, g // m % m, g // m ** 2]) + rng.uniform(0.3, 0.7, (3, n))) * (L / m)
    cfg = ForceConfig(box_len=(L,) * 3, cut_off=2.0, coulomb_cut=2.0, skin=0.45, alpha=0.5,
                      kspace="NONE", n_max=n, list_capacity=cap, neighbor_type=neighbors,
                      r_core=1.0, rbl_pice=1)
    # 159,744 bytes hold 24 (RBL: 28) a candidate for 256 candidates and 16 an entry
    if cap > (9536 if neighbors == "RBL" else 9600):
        with pytest.raises(RBMDError):
            LJCutCoulKspaceForce(cfg)
        return
    f = LJCutCoulKspaceForce(cfg)
    f.Init(_dev(rng.uniform(-1, 1, n)))
    F = [torch.zeros(n, device="cuda") for _ in range(3)]
    f.Execute(*[_dev(a) for a in p], *F)
    st = f.stats()
    assert st["cap"] == cap and st["overflow_rows"] == 0 and st["cells"] == 1
    Lb = np.array([L] * 3)
    w = [np.ascontiguousarray(a) for a in orc.wrap(*p, np.zeros(3), Lb)]
    oo, io = orc.neighbors_images(*w, Lb, 2.45)
    og, ig = f.neighbors()
    assert og[-1] == oo[-1] and np.diff(og).max() > 4096
    for i in range(n):
        assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i
