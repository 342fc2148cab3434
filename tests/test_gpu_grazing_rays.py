"""Rays that graze slivers from afar: the computed hit can lie well before the
entry of its own box, and the hit found is the per-thread search's (dev_ray)
all the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(r, n, d):
    """Triangles in [-1, 1]^3: slivers, triangles that nearly hold the direction d, and others."""
    T = r.uniform(-1, 1, (n, 3, 3))
    k = np.arange(n) % 3
    log = lambda lo, m: np.exp(r.uniform(np.log(lo), 0, (m, 1)))  # noqa: E731
    s = k == 0
    m = s.sum()
    T[s, 2] = T[s, 0] + r.uniform(-0.1, 1.1, (m, 1)) * (T[s, 1] - T[s, 0]) + 0.3 * log(1e-9, m) * r.uniform(-1, 1, (m, 3))
    s = k == 1
    m = s.sum()
    e = r.uniform(-1, 1, (m, 3))
    T[s, 1] = T[s, 0] + r.uniform(-1, 1, (m, 1)) * d + log(1e-3, m) * e
    T[s, 2] = T[s, 0] + r.uniform(-1, 1, (m, 1)) * d + log(1e-3, m) * e + 1e-2 * log(1e-4, m) * r.uniform(-1, 1, (m, 3))
    return T.astype(np.float32)


@pytest.mark.parametrize("lo,hi,seed", [(2, 10, 1), (10, 1000, 2), (1000, 100000, 3)])
def test_hits_of_grazing_rays(lo, hi, seed):
    import test_device_api as A

    import snch_lbvh_amd as S

    r = np.random.default_rng(seed)
    lib = A._lib()
    n = 100000
    one = np.ones((n, 3), np.float32)
    tmax = np.full(n, np.inf, np.float32)
    for k in range(40):
        d0 = r.normal(size=3)
        d0 /= np.linalg.norm(d0)
        T = _scene(r, 3 + int(r.integers(60)), d0)
        V, F = np.ascontiguousarray(T.reshape(-1, 3)), np.arange(3 * len(T), dtype=np.int32).reshape(-1, 3)
        o = np.tile(np.float32(-d0 * np.exp(r.uniform(np.log(lo), np.log(hi)))), (n, 1))
        to = (r.dirichlet([1, 1, 1], n)[..., None] * T[r.integers(0, len(T), n)]).sum(1)
        d = to - o
        d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
        sc = S.Scene(V, F).build_bvh()
        want = A._run(lib, S, sc, 0, o, d, tmax, one[:, 0], 0.5 * one, False)
        hit, t, uv, idx = (x.cpu().numpy() for x in sc.ray_intersect(o, d))
        np.testing.assert_array_equal(hit, want["hit"].astype(bool))
        np.testing.assert_array_equal(t, want["t"])
        np.testing.assert_array_equal(idx[hit], want["ray_idx"][hit])
