"""The network's kernels at the edges of their tiles (16 x 16 outputs, 16-deep
groups of K, 16 x 64 parameters, 64 batch rows per step) against the FP64 oracle.

Tolerances as in test_gpu_initializer.py (FP32 sums of at most a few hundred
terms, relative to the largest magnitude: forward 1e-5, gradient 1e-4).  The
first Adam step moves a parameter by lr g / (|g| + 1e-8): exact to the rounding
of the parameter (2^-24 relative, and of the quotient, 4 of them) wherever the
gradient's sign is beyond its own error."""
import ctypes

import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

# (nIn, nHidden, nHiddenLayers, nOut), rows
EDGES = [((1, 1, 1, 1), 1), ((3, 5, 0, 2), 4), ((15, 16, 1, 17), 16), ((16, 17, 2, 15), 17), ((17, 64, 1, 65), 63),
         ((31, 33, 16, 3), 64), ((512, 15, 1, 1), 65), ((129, 48, 2, 63), 130), ((775, 64, 1, 176), 64),
         # from 2048 tiles of an output on a workgroup takes four of them
         ((1, 128, 2, 128), 16 * 256), ((100, 33, 2, 130), 16 * 1024 + 1), ((20, 513, 1, 16), 63 * 16 + 47)]


@pytest.mark.parametrize("shape,rows", EDGES)
def test_edges(gpu, shape, rows):
    from rootpwa_amd.mlp import MLP
    rng = np.random.default_rng(rows)
    net = MLP(*shape, seed=2)
    p = (rng.normal(size=net.nParams()) / np.sqrt(max(shape[0], shape[1]))).astype(np.float32)
    x = rng.normal(size=(rows, shape[0])).astype(np.float32)
    t = rng.normal(size=(rows, shape[3])).astype(np.float32)
    net.setParams(p)
    layers = M.unpack(p.astype(np.float64), *shape)
    y, _ = M.forward(layers, x)
    assert np.max(np.abs(net.forward(x) - y)) <= 1e-5 * np.max(np.abs(y))
    loss, g = net.lossGrad(x, t)
    lref, gref = M.loss_grad(layers, x, t)
    assert abs(loss - lref) <= 1e-5 * lref
    assert np.max(np.abs(g - gref)) <= 1e-4 * np.max(np.abs(gref))
    # one batch holding all rows, one step
    lr = 0.01
    net.train(x, t, batchSize=rows, epochs=1, lr=lr, seed=1)
    q = net.params().astype(np.float64)
    big = np.abs(gref) > 1e-3 * np.max(np.abs(gref))
    want = p - lr * gref / (np.abs(gref) + 1e-8)
    err = np.abs(q - want)[big]
    # relative: 1e-8 / |g| changes by at most the gradient's 10 % error there
    tol = (2.0 ** -24 * (np.abs(want) + 4 * lr) + lr * 0.1 * 1e-8 / np.abs(gref))[big]
    assert np.all(err <= tol)


def test_set_params_starts_the_optimiser_anew(gpu):
    """After setParams a network trains as a new one with these parameters does,
    bit for bit, however many steps it has taken before: the moments are zero when
    the next step reads them."""
    from rootpwa_amd.mlp import MLP
    rng = np.random.default_rng(11)
    shape, rows = (775, 512, 2, 176), 128
    x = rng.normal(size=(rows, shape[0])).astype(np.float32)
    t = rng.normal(size=(rows, shape[3])).astype(np.float32)
    fresh = MLP(*shape, seed=4)
    p = fresh.params()
    loss = fresh.train(x, t, batchSize=32, epochs=2, lr=1e-3, seed=9)
    net = MLP(*shape, seed=5)
    for _ in range(4):
        net.train(x, t, batchSize=16, epochs=3, lr=1e-2, seed=1)
        net.setParams(p)
        assert np.array_equal(net.train(x, t, batchSize=32, epochs=2, lr=1e-3, seed=9), loss)
        assert np.array_equal(net.params(), fresh.params())


def test_device_memory_held(gpu):
    """What a network holds after its calls: the activations of the largest call, 4
    bytes x (nIn + 2 x hidden units + 2 x nOut) a row, and a training set of up to
    16 MB (32 MB of slack, with the allocator's granularity)."""
    from rootpwa_amd.mlp import MLP

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert gpu.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0  # of the library's runtime
        return a.value

    slack = 32 << 20
    net = MLP(512, 256, 8, 64, seed=1)
    start = free()
    x, t = np.zeros((60000, 512), np.float32), np.zeros((60000, 64), np.float32)
    net.train(x, t, batchSize=64, epochs=1)  # a set of 138 MB
    assert start - free() <= slack
    acts = 60000 * 4 * (512 + 2 * 8 * 256 + 2 * 64)
    net.forward(x)
    net.lossGrad(x, t)
    assert start - free() <= acts + slack


def test_more_tiles_than_one_launch(gpu):
    """An output of more than 2^31 values (2^21 + 16 rows x 1024 hidden units: 2^23 + 64
    tiles, 17 GB of activations) takes several launches; a row's result does not
    depend on the rows beside it."""
    from rootpwa_amd.mlp import MLP
    rows = (1 << 21) + 16
    net = MLP(1, 1024, 1, 1, seed=3)
    x = np.linspace(-3, 3, rows, dtype=np.float32)[:, None]
    y = net.forward(x)
    for first in (0, (1 << 16) - 8, (1 << 20) - 8, rows - 16):
        assert np.array_equal(net.forward(x[first:first + 16]), y[first:first + 16])


def _mix64(x):
    m = (1 << 64) - 1
    x = (x + 0x9E3779B97F4A7C15) & m
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & m
    return x ^ (x >> 31)


def _adam(p, state, shape, x, t, batch, epochs, lr, seed):
    """FP64 Adam over the documented shuffle; state: both moments and the step count."""
    m1, m2, k = state
    losses = []
    for epoch in range(epochs):
        perm = list(range(len(x)))
        for i in range(len(x) - 1, 0, -1):
            j = _mix64(seed ^ _mix64((epoch << 32) + i)) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        total = 0.0
        for b in range(len(x) // batch):
            at = perm[b * batch:(b + 1) * batch]
            loss, g = M.loss_grad(M.unpack(p, *shape), x[at], t[at])
            k += 1
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            p = p - lr * (m1 / (1 - 0.9 ** k)) / (np.sqrt(m2 / (1 - 0.999 ** k)) + 1e-8)
            total += loss
        losses.append(total / (len(x) // batch))
    return p, (m1, m2, k), losses


@pytest.mark.parametrize("shape", [(13, 24, 2, 5), (40, 33, 1, 70)])
def test_training_steps(gpu, shape):
    """Batches smaller than a set that is no multiple of them, several epochs, and a
    second call that goes on with the optimiser's state, against FP64 Adam.  Of the
    parameters' whole change (2-norm) FP64 Adam's differs by 6e-5 with errors of
    1e-6 of the largest component in every gradient (the FP32 sums' are below), and
    by 0.1 where the second call forgets the moments; allowed 5e-4.  Losses 1e-5."""
    from rootpwa_amd.mlp import MLP
    rng = np.random.default_rng(1)
    net = MLP(*shape, seed=1)
    p0 = (rng.normal(size=net.nParams()) / np.sqrt(24)).astype(np.float32)
    x = rng.normal(size=(150, shape[0])).astype(np.float32)
    t = rng.normal(size=(150, shape[3])).astype(np.float32)
    net.setParams(p0)
    p, state = p0.astype(np.float64), (0.0, 0.0, 0)
    for epochs, seed in ((3, 5), (2, 6)):
        loss = net.train(x, t, batchSize=32, epochs=epochs, lr=1e-3, seed=seed)
        p, state, ref = _adam(p, state, shape, x.astype(np.float64), t.astype(np.float64), 32, epochs, 1e-3, seed)
        assert np.max(np.abs(loss / np.array(ref) - 1)) <= 1e-5
        assert np.linalg.norm(net.params() - p) <= 5e-4 * np.linalg.norm(p - p0)
