"""Loss, gradient and training steps of the rate network at batch sizes around its tiles of 16 samples, its groups of
32 tiles and its 1024 wavefronts, against the CPU restatement (oracle/mlp.py)."""
import numpy as np
import pytest

from oracle import mlp as R

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def mix(z):
    z = (z + 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def samples(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, (n, 7)).astype(np.float32), rng.normal(size=(n, 5)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 511, 513, 1024 * 16 + 5])
def test_gradient_at_ragged_batches(n):
    from proteuscfd_amd import gpu

    net = gpu.MLP(seed=0)
    p = R.init(9).astype(np.float32)
    net.params = p
    x, t = samples(n, n)
    print(f"[mlp batches] n={n}", flush=True)
    lg, gg = net.loss_grad(x, t)
    lo, go = R.loss_grad(p, x, t)
    # the restatement rounds to BF16 where the kernels do; a value at the edge of two may go either way, 2^-9 of it
    assert abs(lg - lo) <= 2.0**-9 * lo
    for name in ["W1", "b1", "W2", "b2", "W3", "b3"]:
        a, b = R.unpack(gg)[name].astype(float), R.unpack(go)[name]
        assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b), name
    net.close()


@pytest.mark.parametrize("batch", [1, 17, 500, 4096])
def test_training_draws_its_batches_in_order(batch):
    """With a step size that moves no weight by a BF16 rounding, the loss of every step is that of the batch the
    index stream draws for it."""
    from proteuscfd_amd import gpu

    n, steps, seed = 5003, 6, 12345
    net = gpu.MLP(seed=0)
    p = R.init(9).astype(np.float32)
    net.params = p
    x, t = samples(n, 3)
    print(f"[mlp batches] train batch={batch}", flush=True)
    hist = net.train(x, t, steps=steps, batch=batch, lr=1e-9, seed=seed)
    s = seed
    for it in range(steps):
        idx = []
        for _ in range(batch):
            s = mix(s)
            idx.append(s % n)
        lo, _ = R.loss_grad(p, x[idx], t[idx])
        # BF16 roundings that go the other way, as above
        assert abs(hist[it] - lo) <= 2.0**-9 * lo, it
    net.close()


def test_calls_share_a_network():
    """Calls of growing and shrinking batches on one network, among them one whose index lists it does not keep
    (above 1 MiB): every step's loss is its own batch's."""
    from proteuscfd_amd import gpu

    n, steps = 140001, 3
    net = gpu.MLP(seed=0)
    p = R.init(9).astype(np.float32)
    x, t = samples(n, 4)
    net.params = p
    for k, batch in enumerate([1, 300, 140000, 17]):
        print(f"[mlp batches] shared batch={batch}", flush=True)
        hist = net.train(x, t, steps=steps, batch=batch, lr=1e-9, seed=70 + k)
        s = 70 + k
        for it in range(steps):
            idx = []
            for _ in range(batch):
                s = mix(s)
                idx.append(s % n)
            lo, _ = R.loss_grad(p, x[idx], t[idx])
            assert abs(hist[it] - lo) <= 2.0**-9 * lo, (batch, it)
    net.close()


@pytest.mark.parametrize("steps", [1, 4095, 4096, 4097])
def test_long_calls_keep_every_loss(steps):
    """A step size that moves no weight: the losses of one call are those of calls of at most 1,000 steps that
    draw on from where the one before stopped, to the bit, on both sides of the 4,096 losses a network keeps."""
    from proteuscfd_amd import gpu

    n, batch = 97, 3
    net = gpu.MLP(seed=0)
    net.params = R.init(5).astype(np.float32)
    x, t = samples(n, 6)
    whole = net.train(x, t, steps=steps, batch=batch, lr=1e-30, seed=8)
    s, parts = 8, []
    for k in range(0, steps, 1000):
        m = min(1000, steps - k)
        parts.append(net.train(x, t, steps=m, batch=batch, lr=1e-30, seed=s))
        for _ in range(m * batch):
            s = mix(s)
    assert np.all(whole > 0) and np.array_equal(whole, np.concatenate(parts))
    net.close()
