"""2D rays and segments longer than 1: a segment is hit up to 1e-3 of its length
past an end, which is outside its box.  The hit found is the per-thread search's
(dev_ray)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(6))
def test_hits_past_the_ends(seed):
    import test_device_api as A

    import snch_lbvh_amd as S

    r = np.random.default_rng(seed)
    m, n = 330 + 150 * seed, 2000000
    a = r.uniform(-1, 1, (m, 2))
    b = a + 10 * np.exp(r.uniform(np.log(1e-3), 0, (m, 1))) * r.normal(size=(m, 2))
    V = np.stack([a, b], 1).reshape(-1, 2).astype(np.float32)
    F = np.arange(2 * m, dtype=np.int32).reshape(-1, 2)
    lo, hi = V.min(0), V.max(0)
    o = r.uniform(lo, hi, (n, 2)).astype(np.float32)
    o[::2] = V[F[r.integers(0, m, n // 2)]].mean(1) + r.normal(size=(n // 2, 2)).astype(np.float32)
    d = r.normal(size=(n, 2))
    along = F[r.integers(0, m, n)]
    d[::3] = (V[along[:, 1]] - V[along[:, 0]] + 1e-3 * r.normal(size=(n, 2)))[::3]
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    tmax = np.full(n, np.inf, np.float32)
    sc = S.Scene2D(V, F).build_bvh()
    one = np.ones((n, 3), np.float32)
    want = A._run(A._lib(), S, sc, 0, o, d, tmax, one[:, 0], 0.5 * one, False)
    hit, t, uv, idx = (x.cpu().numpy() for x in sc.ray_intersect(o, d))
    np.testing.assert_array_equal(hit, want["hit"].astype(bool))
    np.testing.assert_array_equal(t, want["t"])
    np.testing.assert_array_equal(idx[hit], want["ray_idx"][hit])
