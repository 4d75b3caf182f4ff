"""The training kernel at the edges of its workgroups (64 samples) and of its
sample draw, which reduces a 64-bit Philox value modulo the sample count."""
import numpy as np
import pytest

from oracle import oracle as orc
from readdygpu_amd import Simulation, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 15, 16, 17, 63, 64, 65, 127, 200, 1000])
def test_loss_grad_against_bf16_oracle(m):
    """Relative L2 <= 2e-3 against the FP64 oracle rounding to BF16 where the
    kernel does (the bound of the gradient check at 4,096 samples; a batch of
    one has no averaging, hence 4e-3 below 64)."""
    spec, pieces, xyz, types = workloads.learned_slab(n=64, n_pieces=4)
    rng = np.random.default_rng(m)
    x = rng.uniform(-1, 1, (m, 3)).astype(np.float32)
    t = rng.normal(size=(m, 3)).astype(np.float32)
    with Simulation(spec, xyz, types) as sim:
        sim.surrogate_init(3)
        w = sim.surrogate_weights()
        loss, g = sim.surrogate_loss_grad(x, t)
    lr, gr = orc.mlp_loss_grad(w, x, t, True)
    assert abs(loss - lr) <= 2e-3 * abs(lr)
    assert np.linalg.norm(g - gr) <= (2e-3 if m >= 64 else 4e-3) * np.linalg.norm(gr)


@pytest.mark.parametrize("samples,batch", [(64, 64), (1000, 100), (4097, 192)])
def test_first_step_draws_the_samples(samples, batch):
    """The loss of the first optimiser step equals the loss of the samples that
    Philox(seed, step 0, c) mod m names, up to the sum's rounding."""
    spec, pieces, xyz, types = workloads.learned_slab(n=64, n_pieces=4)
    seed = 77
    idx = []
    for c in range(batch):
        q = orc.philox([c, 0, 0, 0x5452414E], [seed, 0])
        idx.append(((int(q[1]) << 32) | int(q[0])) % samples)
    lo, hi = np.zeros(3), np.asarray(spec.box_hi)
    with Simulation(spec, xyz, types) as sim:
        sim.set_composite(pieces)
        sim.surrogate_init(3)
        sim.surrogate_make_data(samples, seed=5)
        curve = sim.surrogate_train(1, batch=batch, seed=seed)
        sim.surrogate_init(3)
        gs = sim.surrogate_norm()[2]
        pos = []
        for i in idx:
            q = orc.philox([i, 0, 0x44415441, 0x53555247], [5, 0])
            pos.append([(int(v) >> 8) * 2.0 ** -24 for v in q[:3]])
        pos = (np.array(pos) * (hi - lo)).astype(np.float32)
        g, _ = sim.composite_eval(pos)
        xn = (pos * np.float32(1.0) * (2.0 / hi).astype(np.float32) - np.float32(1.0)).astype(np.float32)
        loss, _ = sim.surrogate_loss_grad(xn, g / np.float32(gs))
    assert abs(curve[0] - loss) <= 1e-4 * abs(loss)
