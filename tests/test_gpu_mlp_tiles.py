"""Gradient of the learned bound (k_mlp_train, csrc/mlp.hip) at the edges of its
64-point tiles and with more tiles than workgroups."""
import numpy as np
import pytest

from snch_lbvh_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 33, 63, 64, 65, 1000, 64 * 256 - 1, 64 * 256 + 1])
def test_gradient_tiles(n):
    import snch_lbvh_amd as S
    from oracle import mlp_oracle as M

    V, _ = W.cut_torus(64, 32)
    lo, hi = (b.astype(np.float32) for b in W.padded_box(V))
    pts = W.uniform_points(n, lo, hi, n)
    d = np.random.default_rng(n).uniform(0.0, 0.02, n).astype(np.float32)
    mlp = S.LearnedBound(lo, hi, sigma=4.0, seed=3)
    th, four, frame = mlp.params()
    g, loss = mlp.gradient(pts, d)
    lref, gref = M.loss_and_grad(th, pts, d, four, frame, bf16_weights=True)
    assert abs(loss - lref) <= 2e-2 * lref
    assert np.linalg.norm(g - gref) < 5e-2 * np.linalg.norm(gref)
    # four times the same points: the deltas, scaled by a power of two, round to
    # BF16 alike, each point's share is the same wherever it lies in a tile, and
    # only the order of FP32 sums differs (<= 2^17 terms of 2^-24 each, adding up
    # like a random walk)
    g4, loss4 = mlp.gradient(np.tile(pts, (4, 1)), np.tile(d, 4))
    assert abs(loss4 - loss) <= 2e-5 * loss
    assert np.linalg.norm(g4 - g) < 2e-5 * np.linalg.norm(g)
