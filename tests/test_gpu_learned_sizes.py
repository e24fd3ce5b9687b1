"""The network's loss and gradient at sizes off the kernels' tiles.

The dense kernels work 16 cells a tile and 128 a block, the weight gradients
64 cells a stage and 256 a block:
cell counts below one tile, one past a stage, a block, and a batch of many
blocks, against the CPU statement of the network.  Tolerances as in
test_gpu_learned.py: loss 1e-3, each gradient tensor 2e-2 (relative L2).  A
batch of copies of one sample has that sample's loss and gradient; only the
order of the FP32 sums differs: 1e-3.
"""
import numpy as np
import pytest

import or_mpnn as om
import systems

fs = pytest.importorskip("flowsolversourcecode_amd")
learn = pytest.importorskip("flowsolversourcecode_amd.learn")
pytestmark = pytest.mark.gpu


def network(shape, count, layers=3):
    fam = [systems.pressure_like(*shape, 40 + k, shift=0.1) for k in range(count)]
    rng = np.random.default_rng(3)
    n = len(fam[0][2])
    x = [np.linalg.solve(systems.dense(*f[:4]), f[4]) if n < 2000 else rng.standard_normal(n) for f in fam]
    net = learn.Mpnn(fam[0][0], layers=layers, seed=1, capacity=count)
    net.add_samples(np.stack([f[4] for f in fam]), np.stack(x), np.stack([f[2] for f in fam]),
                    np.stack([f[3] for f in fam]), rng.uniform(0.5, 1.5, (count, n)))
    theta = om.init_params(5) + 0.01
    net.set_params(theta)
    return net, theta


def oracle(net, theta, ids):
    nbr0 = net.nbr.astype(np.int64) - 1
    samples = []
    for k in ids:
        s = net.sample(k)
        X0, e, t, _, _ = om.features(nbr0, s["b"], s["ac"], s["anb"], s["vol"], s["x"], None)
        samples.append((nbr0, X0, e, t))
    loss, caches, _ = om.forward(theta, samples)
    return loss, om.backward(theta, samples, caches)


@pytest.mark.parametrize("shape, ids", [((3, 2, 2), [0]), ((5, 13, 1), [1, 0]), ((5, 7, 3), [0, 1, 2]),
                                        ((13, 11, 9), [2, 0, 1])])
def test_gradient_off_the_tiles(shape, ids):
    net, theta = network(shape, 3)
    loss, g = net.loss_grad(ids)
    lo, go = oracle(net, theta, ids)
    assert abs(loss - lo) <= 1e-3 * lo
    o = 0
    for name, dims in om.param_layout():
        k = int(np.prod(dims))
        a, b = g[o:o + k], go[o:o + k]
        if name != "bd":  # the mean-free output does not depend on bd
            assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b) + 1e-12, name
        o += k


@pytest.mark.parametrize("copies", [2, 51, 105])
def test_copies_have_the_samples_gradient(copies):
    net, theta = network((13, 11, 9), 1)
    loss, g = net.loss_grad([0])
    lc, gc = net.loss_grad([0] * copies)
    assert abs(loss - lc) <= 1e-6 * loss
    assert np.linalg.norm(g[:-1] - gc[:-1]) <= 1e-3 * np.linalg.norm(g[:-1])


@pytest.mark.parametrize("first, then, grad", [(105, 101, True), (110, 102, False), (160, 4, True)])
def test_smaller_batch_after_a_larger_one(first, then, grad):
    """A network keeps its largest batch's workspaces: what a smaller batch
    gives there is, bit for bit, what it gives on a fresh network."""
    net, theta = network((13, 11, 9), 1)
    net.loss_grad([0] * first, grad=grad)
    loss, g = net.loss_grad([0] * then)
    fresh, _ = network((13, 11, 9), 1)
    lf, gf = fresh.loss_grad([0] * then)
    assert loss == lf and np.array_equal(g, gf)
