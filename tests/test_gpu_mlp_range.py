"""The proposal network at activations far from zero, and at batches around a tile and beyond
one tile per wave."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _chain():
    """A network whose first unit alone acts: z = silu(silu(f_0))."""
    from copy_gpu_amd.proposal import ProposalMLP

    p = np.zeros(4545, np.float32)
    p[0] = p[320] = p[4480] = 1.0
    net = ProposalMLP(seed=1)
    net.set_params(p)
    return net, p


# around the argument where e^-x reaches the bound of the kernel's exponential, and out to the
# largest FP32 values
XS = np.array([-3e38, -1e30, -1e20, -1e6, -1e3, -100, -89, -88, -87.5, -87, -86.5, -40, -5, -1, 0,
               1, 5, 40, 86.5, 87, 88, 100, 1e3, 1e6], np.float32)


def test_forward():
    from oracle import mlp as omlp

    net, p = _chain()
    f = np.zeros((XS.size, 4), np.float32)
    f[:, 0] = XS
    h = net.forward(f).double().cpu().numpy()
    with np.errstate(over="ignore"):
        ref, _ = omlp.forward(p.astype(np.float64), f.astype(np.float64))
    assert np.all(np.abs(h - ref) <= 1e-6 + 2e-5 * np.abs(ref))


@pytest.mark.parametrize("x", XS[XS < 10])
def test_gradient(x):
    """Of one sample; far below zero the first layer's gradient is zero, whatever the feature."""
    from oracle import mlp as omlp

    net, p = _chain()
    f = np.zeros((1, 4), np.float32)
    f[0, 0] = x
    y, w = np.array([0.5], np.float32), np.array([1.0], np.float32)
    loss, g = net.loss_grad(f, y, w)
    with np.errstate(over="ignore"):
        lref, gref = omlp.loss_grad(p.astype(np.float64), f.astype(np.float64),
                                    y.astype(np.float64), w.astype(np.float64))
    assert abs(loss - lref) <= 1e-5 * lref
    # silu' is kept to 1.5e-36, times the feature
    assert np.all(np.abs(g - gref) <= 2e-5 * np.abs(gref).max() + 2e-36 * min(abs(x), 100.0))


# one sample, a tile of 16 and its neighbours, a wave more than one workgroup's, and batches that
# give some waves a second tile (above 32,768 samples) and all of them several
@pytest.mark.parametrize("B", [1, 15, 16, 17, 129, 35937, 120001])
def test_batches(B):
    from copy_gpu_amd.proposal import ProposalMLP
    from oracle import mlp as omlp

    net = ProposalMLP(seed=11)
    p = omlp.bf16_round(net.params())
    rng = np.random.default_rng(B)
    f = rng.uniform(0, 3, (B, 4)).astype(np.float32)
    y = rng.normal(0, 1, B).astype(np.float32)
    w = rng.uniform(0.1, 1, B).astype(np.float32)
    w /= w.sum()
    f64 = f.astype(np.float64)
    h = net.forward(f).double().cpu().numpy()
    href, _ = omlp.forward(p, f64)
    assert np.all(np.abs(h - href) <= 1e-6 + 2e-5 * np.abs(href))
    loss, g = net.loss_grad(f, y, w)
    lref, gref = omlp.loss_grad(p, f64, y.astype(np.float64), w.astype(np.float64))
    # the tolerances of the FP32 network's other tests
    assert abs(loss - lref) <= 1e-5 * lref
    assert np.abs(g - gref).max() <= 2e-5 * np.abs(gref).max()
    for lo, hi in [(0, 256), (256, 320), (320, 4416), (4416, 4480), (4480, 4544), (4544, 4545)]:
        assert np.linalg.norm(g[lo:hi] - gref[lo:hi]) <= 1e-4 * np.linalg.norm(gref[lo:hi]) + 1e-9
