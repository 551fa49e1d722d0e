"""The network on a grid with enough voxels for the convolutions' large boxes
against a corner of it by itself, which takes the small ones.

An output depends on inputs at most 20 voxels away (one voxel per convolution
of the finest level, 2 and 4 of the others, and the pooling's alignment), so
away from the cut the two grids' outputs are formed from the same numbers in
the same order: equal bits.  With a target that differs from the output near
the corner only, both have the same weight gradient up to the mean's divisor
(a power of two here, exact through the BF16 roundings) and the order of the
FP32 sums: about 1e-5 relative for 3e4 terms of either sign, 1e-4 allowed."""
import numpy as np
import pytest

from turbins_amd import Net

pytestmark = pytest.mark.gpu

REACH = 20


@pytest.mark.parametrize("whole,crop", [((64, 64, 96), (36, 28, 44)), ((36, 60, 132), (28, 40, 24)),
                                        ((64, 64, 64), (32, 32, 32))])
def test_corner_of_a_large_grid(whole, crop):
    print("net boxes", whole, crop, flush=True)
    net = Net(seed=5)
    rng = np.random.default_rng(sum(whole))
    in3 = rng.standard_normal((*whole, 3)).astype(np.float32)
    cut = tuple(slice(0, n) for n in crop)
    small = np.ascontiguousarray(in3[cut])
    a, b = net.forward(in3), net.forward(small)
    keep = tuple(slice(0, n - REACH) for n in crop)
    assert np.array_equal(a[keep], b[keep])
    if whole == (64, 64, 64):
        ta, tb = a.copy(), b.copy()
        near = tuple(slice(0, 8) for _ in crop)
        d = rng.standard_normal((8, 8, 8)).astype(np.float32)
        ta[near] += d
        tb[near] = ta[near]
        ga, gb = net.gradient(in3, ta)[1], net.gradient(small, tb)[1]
        scale = np.prod(whole) / np.prod(crop)
        err = np.linalg.norm(ga.astype(np.float64) * scale - gb) / np.linalg.norm(gb)
        print("gradient", err)
        assert err <= 1e-4
    net.close()
