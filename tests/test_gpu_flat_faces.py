"""Axis-parallel faces, where half of the answers' distances round below their
boxes' bounds, near the origin and far from it: the answers of the per-thread
searches (device header), also where faces, edges and vertices tie."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(lo, hi):
    V = np.array([[x, y, z] for x in (lo[0], hi[0]) for y in (lo[1], hi[1]) for z in (lo[2], hi[2])], np.float32)
    F = np.int32([[0, 1, 3], [0, 3, 2], [4, 6, 7], [4, 7, 5], [0, 4, 5], [0, 5, 1], [2, 3, 7], [2, 7, 6], [0, 2, 6],
                  [0, 6, 4], [1, 5, 7], [1, 7, 3]])
    return V, F


def _scene(far):
    """A floor of 32 x 32 cells, boxes on it, some of them side by side."""
    k = np.arange(33)
    V = [np.stack(np.meshgrid(k / 2, k / 2, [0.0], indexing="ij"), -1).reshape(-1, 3).astype(np.float32)]
    c = (np.arange(32)[:, None] * 33 + np.arange(32)).ravel()
    F = [np.concatenate([np.c_[c, c + 33, c + 34], np.c_[c, c + 34, c + 1]]).astype(np.int32)]
    r = np.random.default_rng(1)
    for x, y in [(3, 3), (4, 3), (3, 4), *r.integers(0, 15, (12, 2))]:
        v, f = _box((x, y, 0), (x + 1, y + 1, int(r.integers(1, 4))))
        F.append(f + sum(map(len, V)))
        V.append(v)
    V = np.concatenate(V) + (np.float32([100, 50, 7]) if far else np.float32([-8, -8, 0]))
    return V.astype(np.float32), np.concatenate(F)


@pytest.mark.parametrize("far", [False, True])
@pytest.mark.parametrize("leaf_size", [1, 4])
def test_flat_faces(far, leaf_size):
    import snch_lbvh_amd as S
    import test_device_api as A

    V, F = _scene(far)
    r = np.random.default_rng(2)
    n = 200000
    lo, hi = V.min(0), V.max(0)
    q = r.uniform(lo - 1, hi + 1, (n, 3)).astype(np.float32)
    k = r.random(n)
    q[k < 0.5] = np.round(2 * q[k < 0.5]) / 2  # on the planes, edges and vertices, and straight above them
    d = r.normal(size=(n, 3))
    d[k < 0.2] = np.eye(3)[r.integers(0, 3, (k < 0.2).sum())] * r.choice([-1, 1], ((k < 0.2).sum(), 1))
    d[(k > 0.5) & (k < 0.6), 2] *= 1e-3
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    tmax = np.where(r.random(n) < 0.7, np.inf, 5 * r.random(n)).astype(np.float32)
    one = np.ones((n, 3), np.float32)
    sc = S.Scene(V, F).build_bvh(leaf_size=leaf_size)
    for flip in (False, True):
        want = A._run(A._lib(), S, sc, 0, q, d, tmax, one[:, 0], 0.5 * one, flip)
        i, dist = (x.cpu().numpy() for x in sc.closest_point(q))
        np.testing.assert_array_equal(dist, want["cp_dist"])
        np.testing.assert_array_equal(i, want["cp_idx"])
        for hint in (None, np.float32(0.5) * want["sil_dist"], np.float32(1.1) * want["sil_dist"]):
            i, dist = (x.cpu().numpy() for x in sc.closest_silhouette(q, flip=flip, seed_radius=hint))
            np.testing.assert_array_equal(dist, want["sil_dist"])
            np.testing.assert_array_equal(i, want["sil_idx"])
    hit, t, uv, idx = (x.cpu().numpy() for x in sc.ray_intersect(q, d, tmax))
    np.testing.assert_array_equal(hit, want["hit"].astype(bool))
    np.testing.assert_array_equal(t[hit], want["t"][hit])
    np.testing.assert_array_equal(idx[hit], want["ray_idx"][hit])
