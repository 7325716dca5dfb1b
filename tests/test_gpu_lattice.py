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
