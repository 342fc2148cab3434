"""Closest silhouettes of meshes with triangles of very uneven sizes and shapes
(convex hulls of random points), near and far: the oracle's distances bit for
bit.  Many of their leaves own no edges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hull(n, seed, stretched):
    from scipy.spatial import ConvexHull

    r = np.random.default_rng(seed)
    p = r.normal(size=(n, 3))
    if stretched:
        p[:, 0] *= np.exp(1.5 * r.normal(size=n))
    p /= np.linalg.norm(p, axis=1, keepdims=True)
    T = ConvexHull(p).simplices.copy()
    a, b, c = (p[T[:, k]] for k in range(3))
    inward = (np.cross(b - a, c - a) * a).sum(1) < 0
    T[inward] = T[inward][:, [0, 2, 1]]
    return p.astype(np.float32), T.astype(np.int32)


@pytest.mark.parametrize("n,seed,stretched", [(9000, 1, False), (9000, 1, True), (3000, 3, False), (3000, 3, True)])
def test_hulls(oracle, n, seed, stretched):
    import snch_lbvh_amd as S

    V, F = _hull(n, seed, stretched)
    r = np.random.default_rng(7)
    m = 400000
    q = r.uniform(-1.5, 1.5, (m, 3)).astype(np.float32)
    far = np.exp(r.uniform(np.log(1e-3), 0, (m // 2, 1)))
    q[::2] = V[F[r.integers(0, len(F), m // 2)]].mean(1) + (2 * far * r.normal(size=(m // 2, 3))).astype(np.float32)
    sc, tr = S.Scene(V, F).build_bvh(), oracle.build_tree(V, F)
    d = sc.closest_silhouette(q)[1].cpu().numpy()
    np.testing.assert_array_equal(d, oracle.closest_silhouette(tr, q)[1])
