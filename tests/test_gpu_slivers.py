"""Closest point where a triangle's computed distance is far above what its box
promises: slivers, and degenerate triangles whose distance may be NaN.  A
closed mesh hides these (a neighbour on the same edge answers), so the meshes
here are soups.  The answers are the per-thread search's (dev_nearest), which
takes no bound from boxes but the reference's own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the distance to this triangle from P comes out as 0.966, its box says 0.734 at most
SLIVER = np.float32([[0.824123621, 0.401569724, 0.514788389], [1.70230901, -0.242001653, -0.0885771513],
                     [1.64838266, -0.202482164, -0.0515265465]])
P = np.float32([[1.063833, 0.108649611, 0.600390971]])


def _mesh(T):
    return np.ascontiguousarray(T.reshape(-1, 3)), np.arange(3 * len(T), dtype=np.int32).reshape(-1, 3)


def _soup(kind, n, seed):
    r = np.random.default_rng(seed)
    a = r.uniform(-1, 1, (n, 3))
    size = np.where(r.random(n) < 0.5, 1.0, np.exp(r.uniform(np.log(1e-3), 0, n)))[:, None]
    b = a + size * r.uniform(-1, 1, (n, 3))
    thin = np.exp(r.uniform(np.log(1e-9), np.log(0.3), n))[:, None]
    c = a + r.uniform(-0.1, 1.1, (n, 1)) * (b - a) + size * thin * r.uniform(-1, 1, (n, 3))
    T = np.stack([a, b, c], 1).astype(np.float32)
    T = T[np.arange(n)[:, None], r.permuted(np.tile(np.arange(3), (n, 1)), axis=1)]
    if kind == "degenerate":  # repeated vertices, points, and vertices on the opposite edge
        k = np.arange(n) % 5
        T[k == 0, 1] = T[k == 0, 0]
        T[k == 1, 2] = T[k == 1, 0]
        T[k == 2, 2] = T[k == 2, 1]
        T[k == 3, 1:] = T[k == 3, :1]
        T[k == 4, 2] = 0.5 * (T[k == 4, 0] + T[k == 4, 1])
    return _mesh(T)


def _points(V, F, n, seed):
    r = np.random.default_rng(seed)
    T = V[F[r.integers(0, len(F), n)]]
    w = r.dirichlet([1, 1, 1], n)[..., None]
    far = np.exp(r.uniform(np.log(1e-6), np.log(10), (n, 1)))
    q = (w * T).sum(1) + far * r.uniform(-1, 1, (n, 3))
    q[::4] = r.uniform(V.min(0) - 0.1, V.max(0) + 0.1, (len(q[::4]), 3))
    return q.astype(np.float32)


def _per_thread(S, sc, mesh, q):
    import test_device_api as A

    n = len(q)
    one = np.ones((n, 3), np.float32)
    g = A._run(A._lib(), S, sc, mesh, q, one, one[:, 0], one[:, 0], 0.5 * one, False)
    return g["cp_idx"], g["cp_dist"]


def test_the_only_triangle_near():
    import snch_lbvh_amd as S

    V, F = _mesh(np.stack([SLIVER, SLIVER[[0, 1, 1]] + np.float32(50) * np.eye(3, dtype=np.float32)]))
    sc = S.Scene(V, F).build_bvh()
    for n in (1, 64, 1000):
        i, d = (x.cpu().numpy() for x in sc.closest_point(np.tile(P, (n, 1))))
        assert np.all(i == 0) and np.all(np.abs(d - 0.966) < 1e-3)


@pytest.mark.parametrize("kind", ["slivers", "degenerate"])
@pytest.mark.parametrize("leaf_size", [1, 8])
def test_soups(kind, leaf_size):
    """24 soups, each alone, and all in one batch."""
    import snch_lbvh_amd as S

    meshes = [_soup(kind, 2 + (7 * k) % 61, k) for k in range(24)]
    q = [_points(V, F, 20000, 100 + k) for k, (V, F) in enumerate(meshes)]
    batch = S.BatchScene(meshes).build_bvh(leaf_size=leaf_size)
    off = np.arange(25) * 20000
    bi, bd = (x.cpu().numpy() for x in batch.closest_point(np.concatenate(q), off))
    for k, (V, F) in enumerate(meshes):
        s = slice(off[k], off[k + 1])
        want_i, want_d = _per_thread(S, batch, k, q[k])
        sc = S.Scene(V, F).build_bvh(leaf_size=leaf_size)
        for i, d in ((bi[s], bd[s]), tuple(x.cpu().numpy() for x in sc.closest_point(q[k]))):
            np.testing.assert_array_equal(d, want_d)
            np.testing.assert_array_equal(i, want_i)
