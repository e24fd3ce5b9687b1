"""Records the warm-start network's losses and gradients on an MI355X:

    python tests/golden/make_mpnn_golden.py [OUT.npz]

mpnn_gradients.npz holds, per entry of CASES, the loss (FP64) and the gradient
(FP32) of one batch of samples.  Every sum of a step runs over fixed partials
in a fixed order, so a batch has one gradient, to the bit, and a training run
can be repeated; tests/test_gpu_learned_golden.py holds the device to it.
Inputs are uniform numbers: the same on every machine.
"""
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.dirname(os.path.dirname(HERE))]

# name: mesh shape, layers, batch (sample ids)
CASES = {
    "tile": ((5, 7, 3), 1, [1]),           # 105 cells: less than one block of the gradient kernels
    "blocks": ((13, 11, 9), 2, [2, 0, 1]),  # 3861 cells: 16 blocks, the last of 21 cells
    "many": ((64, 64, 1), 1, [0, 1, 2] * 7),  # 86016 cells: 336 blocks
    "large": ((64, 64, 1), 1, [0, 1, 2] * 11),  # 135168 cells: 528 blocks
}
SAMPLES = 3


def box_neighbours(nx, ny, nz):
    """(6, N) neighbours of a box of cells, 1-based, 0 = none, no gaps."""
    n = nx * ny * nz
    i = np.arange(n)
    x, y, z = i % nx, i // nx % ny, i // (nx * ny)
    out = np.zeros((6, n), dtype=np.int32)
    fill = np.zeros(n, dtype=int)
    for ok, k in ((x > 0, i - 1), (x < nx - 1, i + 1), (y > 0, i - nx), (y < ny - 1, i + nx), (z > 0, i - nx * ny),
                  (z < nz - 1, i + nx * ny)):
        out[fill[ok], i[ok]] = k[ok] + 1
        fill[ok] += 1
    return out


def network(shape, layers, seed=11):
    from flowsolversourcecode_amd import learn
    nbr = box_neighbours(*shape)
    w, n = nbr.shape
    rng = np.random.default_rng(seed)
    b, x = rng.uniform(-1, 1, (SAMPLES, n)), rng.uniform(-1, 1, (SAMPLES, n))
    ac, vol = rng.uniform(5, 7, (SAMPLES, n)), rng.uniform(0.5, 1.5, (SAMPLES, n))
    anb = np.where(nbr > 0, -rng.uniform(0.5, 1.5, (SAMPLES, w, n)), 0.0)
    net = learn.Mpnn(nbr, layers=layers, seed=1, capacity=SAMPLES)
    net.add_samples(b, x, ac, anb, vol)
    net.set_params(rng.uniform(-0.2, 0.2, net.P))
    return net


def run(name):
    shape, layers, ids = CASES[name]
    loss, g = network(shape, layers).loss_grad(ids)
    return loss, g.astype(np.float32)


if __name__ == "__main__":
    out = {}
    for name in CASES:
        loss, g = run(name)
        again, h = run(name)
        assert loss == again and np.array_equal(g, h), name
        out[name + "_loss"], out[name + "_grad"] = np.float64(loss), g
        print(name, loss, np.abs(g).max(), flush=True)
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else os.path.join(HERE, "mpnn_gradients.npz"), **out)
