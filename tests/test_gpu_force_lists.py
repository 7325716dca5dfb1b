"""The force pass's cell bins and sort: chunked prefix sums (more than 16,384 cells), a cell
beyond its bucket, one atom, atoms outside the box; positions that move with and without a
rebuild.  The rows must equal the oracle's neighbour sets and the forces a fresh handle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a)).to(device="cuda", dtype=dtype)


def _system(kind, rng):
    """positions [3][n], box edge, cutoff"""
    if kind == "chunked":  # 26^3 cells
        n, L = 4001, 28.7
        g = rng.permutation(28 ** 3)[:n]
        pos = np.stack([g % 28, g // 28 % 28, g // 784]) + 0.5 + rng.uniform(-0.1, 0.1, (3, n))
        return pos, L, 1.0
    if kind == "bucket":  # 27 cells, one of them with 700 of 764 atoms
        L = 9.6
        g = rng.permutation(9 ** 3)[:700]
        a = np.stack([g % 9, g // 9 % 9, g // 81]) * 0.35 + 0.1 + rng.uniform(-0.02, 0.02, (3, 700))
        b = np.stack(np.meshgrid(*[np.arange(4)] * 3)).reshape(3, -1) * 1.4 + 3.6
        return np.concatenate([a, b], 1), L, 2.9
    if kind == "one":
        return np.full((3, 1), 4.2), 9.6, 2.9
    n = 500  # images outside the box
    g = rng.permutation(8 ** 3)[:n]
    pos = (np.stack([g % 8, g // 8 % 8, g // 64]) + 0.5) * 1.3 + rng.uniform(-0.1, 0.1, (3, n))
    return pos + 10.4 * rng.integers(-1, 2, (3, n)), 10.4, 2.9


@pytest.mark.parametrize("kind", ["chunked", "bucket", "one", "outside"])
def test_bins_and_sort(orc, gpu, kind):
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(11)
    pos, L, rc = _system(kind, rng)
    n = pos.shape[1]
    q = rng.uniform(-1, 1, n)
    skin = 0.1 if kind == "chunked" else 0.3
    cfg = ForceConfig(box_len=(L,) * 3, cut_off=rc, coulomb_cut=rc, alpha=0.5, skin=skin,
                      kspace="RBE", coulomb_sample_num=70, precision=64, n_max=n)

    def evaluate(f, p):
        f.sample_kvectors(70, 5, 0)
        F = [torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
        f.Execute(*[_dev(a) for a in p], *F)
        return torch.stack(F).cpu().numpy()

    f = LJCutCoulKspaceForce(cfg)
    f.Init(_dev(q))
    builds = 0
    # the start, a step within half the skin (no rebuild), one beyond it
    for step, move in enumerate((0.0, 0.2 * skin, 2.0 * skin)):
        p = pos + move / np.sqrt(3.0)
        F = evaluate(f, p)
        st = f.stats()
        builds += step != 1
        assert st["builds"] == builds
        if st["overflow_rows"]:
            # the crowded cell's rows are longer than the mean density's: the forces are exact
            # all the same, and the next evaluation builds longer rows
            assert kind == "bucket" and step == 0
            again = evaluate(f, p)
            assert np.abs(F - again).max() <= 1e-10 * np.abs(again).max()
            st = f.stats()
            builds += 1
            assert st["builds"] == builds and st["overflow_rows"] == 0
        if step != 1:
            w = [np.ascontiguousarray(a) for a in orc.wrap(*p, np.zeros(3), np.array([L] * 3))]
            oo, io = orc.neighbors_images(*w, np.array([L] * 3), rc + skin)
            og, ig = f.neighbors()
            assert og[-1] == oo[-1]
            for i in range(n):
                assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i
        # rounding: positions of about L in steps of 2^-53 L against steep pairs
        fresh = LJCutCoulKspaceForce(cfg)
        fresh.Init(_dev(q))
        G = evaluate(fresh, p)
        assert np.abs(F - G).max() <= 1e-10 * max(np.abs(G).max(), 1e-300)


# cells of exactly their bucket, of up to three atoms in a list beyond it, of as many as the
# sort ranks at once and of one more; the others hold three
CROWDED = (64, 65, 96, 97, 129, 1024, 1025)


def test_cells_beyond_their_bucket(orc, gpu):
    """Rows equal the oracle's sets and forces a second handle's bit for bit, at each of
    several builds (the lists of the atoms beyond a bucket start empty every time)."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(12)
    edge, cells = 2.2, 9
    L = 1.0001 * edge * cells
    crowd = {(1, 1, 1 + k): c for k, c in enumerate(CROWDED)}
    pos = []
    for c in np.ndindex(cells, cells, cells):
        m = crowd.get(c, 3 if min(c) > 0 and max(c) < 8 and c[0] > 3 else 0)
        g = rng.permutation(12 ** 3)[:m]
        p = (np.stack([g % 12, g // 12 % 12, g // 144]) + 0.5) * (0.8 * edge / 12) + 0.1 * edge
        pos.append(p + np.array(c)[:, None] * L / cells)
    pos = np.concatenate(pos, 1)
    pos = pos[:, rng.permutation(pos.shape[1])]
    n = pos.shape[1]
    q = rng.uniform(-1, 1, n)
    cfg = ForceConfig(box_len=(L,) * 3, cut_off=2.0, coulomb_cut=2.0, skin=0.2, alpha=0.5,
                      kspace="NONE", precision=64, n_max=n, list_capacity=2560)
    assert 4 * n / cells ** 3 + 32 <= 64  # the smallest bucket
    f = LJCutCoulKspaceForce(cfg)
    f.Init(_dev(q))
    for build, move in enumerate((0.0, 0.15, 0.0), 1):
        p = pos + move
        F, G = ([torch.zeros(n, device="cuda", dtype=torch.float64) for _ in range(3)]
                for _ in range(2))
        f.Execute(*[_dev(a) for a in p], *F)
        st = f.stats()
        assert st["builds"] == build and st["overflow_rows"] == 0
        w = [np.ascontiguousarray(a) for a in orc.wrap(*p, np.zeros(3), np.array([L] * 3))]
        oo, io = orc.neighbors_images(*w, np.array([L] * 3), 2.2)
        og, ig = f.neighbors()
        assert og[-1] == oo[-1]
        for i in range(n):
            assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i
        h = LJCutCoulKspaceForce(cfg)
        h.Init(_dev(q))
        h.Execute(*[_dev(a) for a in p], *G)
        for a, b in zip(F, G):
            assert torch.equal(a, b)


def test_sort_time_of_a_droplet(gpu):
    """100,000 ions in a 27th of their box, most cells beyond their bucket: the cell sort of a
    rebuild takes no more than four times that of the same ions in a box of their own."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    n, m = 100000, 47
    g = np.random.default_rng(13).permutation(m ** 3)[:n]
    pos = (np.stack([g % m, g // m % m, g // m ** 2]) + 0.5) * 1.5
    us = []
    for L in (1.5 * m, 3 * 1.5 * m):
        f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=6.0,
                                             alpha=0.5, kspace="NONE", n_max=n))
        f.Init(_dev(np.where(g % 2, 1.0, -1.0)))
        X = [[_dev(a + d) for a in pos] for d in (0.0, 0.2)]
        F = [torch.zeros(n, device="cuda") for _ in range(3)]
        for k in range(4):
            f.Execute(*X[k % 2], *F)
        torch.cuda.synchronize()
        b0 = f.stats()["builds"]
        f.set_timing(True)
        for k in range(10):
            f.Execute(*X[k % 2], *F)
        us.append(1e3 * f.timing("cellsort")[0])
        assert f.stats()["builds"] == b0 + 10
    print(f"cell sort: {us[0]:.1f} us, droplet {us[1]:.1f} us", flush=True)
    assert us[1] < 4 * us[0]


# every earlier cell counted (no chunk counts) at a number of cells that four does not divide,
# and three waves per cell: workgroups that begin within a cell
@pytest.mark.parametrize("cells,n", [((25, 25, 25), 5000), ((1, 1, 5), 850)])
def test_starts_of_cells(orc, gpu, cells, n):
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    rng = np.random.default_rng(14)
    rc, skin = 2.0, 0.2
    L = np.array(cells) * 1.0001 * (rc + skin)
    m = np.ceil(L / (0.9 * (L.prod() / n) ** (1 / 3))).astype(int)
    g = rng.permutation(m.prod())[:n]
    pos = np.stack([g % m[0], g // m[0] % m[1], g // (m[0] * m[1])]) + rng.uniform(0.3, 0.7, (3, n))
    pos *= (L / m)[:, None]
    f = LJCutCoulKspaceForce(ForceConfig(box_len=tuple(L), cut_off=rc, coulomb_cut=rc, skin=skin,
                                         alpha=0.5, kspace="NONE", n_max=n, list_capacity=1024))
    f.Init(_dev(rng.uniform(-1, 1, n)))
    F = [torch.zeros(n, device="cuda") for _ in range(3)]
    f.Execute(*[_dev(a) for a in pos], *F)
    st = f.stats()
    assert st["cells"] == np.prod(cells) and st["overflow_rows"] == 0
    w = [np.ascontiguousarray(a) for a in orc.wrap(*pos, np.zeros(3), L)]
    oo, io = orc.neighbors_images(*w, L, rc + skin)
    og, ig = f.neighbors()
    assert og[-1] == oo[-1]
    for i in range(n):
        assert np.array_equal(np.sort(ig[og[i]:og[i + 1]]), np.sort(io[oo[i]:oo[i + 1]])), i


def test_sort_time_of_many_cells(gpu):
    """A thin gas of 4,000 ions: the cell sort of 15,625 cells takes no more than four times
    that of 512."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    n, m = 4000, 16
    g = np.random.default_rng(15).permutation(m ** 3)[:n]
    us = []
    for cells in (8, 25):
        L = 5.35 * cells
        pos = (np.stack([g % m, g // m % m, g // m ** 2]) + 0.5) * (L / m)
        f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=5.0,
                                             alpha=0.5, kspace="NONE", n_max=n))
        f.Init(_dev(np.where(g % 2, 1.0, -1.0)))
        X = [[_dev(a + d) for a in pos] for d in (0.0, 0.2)]
        F = [torch.zeros(n, device="cuda") for _ in range(3)]
        for k in range(4):
            f.Execute(*X[k % 2], *F)
        torch.cuda.synchronize()
        assert f.stats()["cells"] == cells ** 3
        f.set_timing(True)
        for k in range(20):
            f.Execute(*X[k % 2], *F)
        us.append(1e3 * f.timing("cellsort")[0])
    print(f"cell sort: 512 cells {us[0]:.1f} us, 15,625 cells {us[1]:.1f} us", flush=True)
    assert us[1] < 4 * us[0]


def test_empty_tiles_of_a_rebuild(gpu):
    """4,000 ions in 64,000 cells: a rebuild costs the tiles without home atoms nothing, so its
    tile pass takes at most 1.25 times that of an evaluation that keeps its list."""
    from copy_gpu_amd import ForceConfig, LJCutCoulKspaceForce

    n, m, L = 4000, 16, 5.35 * 40
    g = np.random.default_rng(16).permutation(m ** 3)[:n]
    pos = (np.stack([g % m, g // m % m, g // m ** 2]) + 0.5) * (L / m)
    f = LJCutCoulKspaceForce(ForceConfig(box_len=(L,) * 3, cut_off=2.5, coulomb_cut=5.0,
                                         alpha=0.5, kspace="NONE", n_max=n))
    f.Init(_dev(np.where(g % 2, 1.0, -1.0)))
    X = [[_dev(a + d) for a in pos] for d in (0.0, 0.2)]
    F = [torch.zeros(n, device="cuda") for _ in range(3)]
    us = []
    for move in (0, 1):
        for k in range(4):
            f.Execute(*X[move * (k % 2)], *F)
        torch.cuda.synchronize()
        b0 = f.stats()["builds"]
        f.set_timing(True)
        for k in range(20):
            f.Execute(*X[move * (k % 2)], *F)
        us.append(1e3 * f.timing("pair")[0])
        f.set_timing(False)
        assert f.stats()["builds"] == b0 + 20 * move
    print(f"tile pass: {us[0]:.1f} us, with a rebuild {us[1]:.1f} us", flush=True)
    assert us[1] < 1.25 * us[0]
