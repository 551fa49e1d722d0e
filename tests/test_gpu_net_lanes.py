"""Training spreads a batch's crops over several streams, each with its own
gradient part.  With one snapshot of the crop's size every crop is the same,
so a batch of any size has the gradient of one crop times the batch, its mean
loss is that crop's, and Adam's first step, lr g / (|g| + 1e-8), moves every
weight with |g| >= 99e-8 by the same amount to within lr / 99 (for a factor m:
|g / (|g| + e) - m g / (m |g| + e)| <= e / |g|).  The gradient is summed in a
fixed order, so a run repeats bit for bit."""
import numpy as np
import pytest

from turbins_amd import Net, Solver, abi, workload as W

pytestmark = pytest.mark.gpu

LR = 1e-3


@pytest.mark.parametrize("shape", [(32, 16, 16), (36, 12, 20)])
def test_batches_over_lanes(shape):
    nx, ny, nz = shape
    c = W.case("bump_small", nx=nx, ny=ny, nz=nz)
    g = Solver(W.config_for(c, pois_mode=abi.POIS_MIXED_IR))
    g.setup_geometry(W.topography(c))
    for k, v in W.initial_fields(c, [g.flags(q) for q in range(4)]).items():
        g.upload(k, v)
    net = Net(seed=3)
    net.reserve(1, nx, ny, nz)
    g.record_snapshots(net)
    for _ in range(2):
        g.step(c["dt"])
    g.close()
    assert net.snapshot_count() == 1
    w0 = net.get_weights()
    runs = {}
    for batch in (1, 2, 3, 4, 5, 9):
        for rep in range(2):
            net.set_weights(w0)
            l0, l1 = net.train(1, batch, shape, lr=LR, seed=batch)
            w = net.get_weights()
            if rep:
                assert np.array_equal(w, runs[batch][1]) and l0 == runs[batch][0]
            runs[batch] = (l0, w)
    l1, w1 = runs[1]
    big = np.abs(w1 - w0) >= 0.99 * LR
    print("lanes", shape, "weights with a large gradient", big.mean())
    assert big.mean() > 0.1
    for batch, (l, w) in runs.items():
        assert abs(l - l1) <= 1e-12 * l1
        # the step itself is rounded to the weight's FP32
        assert np.max(np.abs(w - w1)[big]) <= LR / 99 + 1e-6
    net.close()
