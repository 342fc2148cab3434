"""The pooled wave searches at the edges of their launch shapes: answers do not
depend on how many queries share a wave, on the pool's size or on leaf runs,
also where a mesh far from the origin makes box bounds and distances round
differently (many candidates within a few units in the last place)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _meshes():
    from snch_lbvh_amd import workloads as W

    V, F = W.icosphere(3, 0.02, seed=1)
    B, sides, caps = W.slab_box(12)  # axis-aligned, coplanar triangles
    return {
        "ico": (V, F),
        "ico_far": (V + np.float32([96.0, -40.0, 7.0]), F),
        "box_far": (B + np.float32([24.0, 3.0, 0.0]), np.concatenate([sides, caps])),
        "two": (V[F[:2].ravel()], np.arange(6, dtype=np.int32).reshape(2, 3)),
    }


def _points(V, n, seed):
    from snch_lbvh_amd import workloads as W

    lo, hi = W.padded_box(V, 0.3)
    q = W.uniform_points(n, lo, hi, seed)
    # exact ties: points straight above vertices and on them
    r = np.random.default_rng(seed)
    at = V[r.integers(0, len(V), n // 8)]
    q[: n // 16] = at[: n // 16] * np.float32([1, 1, 1]) + np.float32([0, 0, 0.25])
    q[n // 16: n // 8] = at[n // 16: n // 8]
    return q[r.permutation(n)]


@pytest.mark.parametrize("name", ["ico", "ico_far", "box_far", "two"])
@pytest.mark.parametrize("leaf_size", [1, 3, 8])
def test_closest_point_does_not_depend_on_the_launch(name, leaf_size):
    import oracle
    import snch_lbvh_amd as S

    V, F = _meshes()[name]
    q = _points(V, 70000, 11)
    sc = S.Scene(V, F).build_bvh(leaf_size=leaf_size)
    i0, d0 = (x.cpu().numpy() for x in sc.closest_point(q))  # the default launch
    for n in (1, 2, 8, 9, 63, 64, 65, 1000):
        i1, d1 = (x.cpu().numpy() for x in sc.closest_point(q[:n]))
        np.testing.assert_array_equal(d1, d0[:n])
        np.testing.assert_array_equal(i1, i0[:n])
    for kw in ({"block_size": 512}, {"block_size": 128, "stack_depth": 8}, {"coherent": 2}):
        i1, d1 = (x.cpu().numpy() for x in sc.closest_point(q, **kw))
        np.testing.assert_array_equal(d1, d0)
        np.testing.assert_array_equal(i1, i0)
    # FP32 rounding of a distance between points of this size: a few units in
    # the last place of the coordinates
    ref = oracle.bf_closest_point(V, F, q[:2000])[1]
    assert np.abs(d0[:2000] - ref).max() <= 8 * np.spacing(np.abs(q).max())


@pytest.mark.parametrize("name", ["ico", "ico_far", "box_far", "two"])
@pytest.mark.parametrize("leaf_size", [1, 8])
def test_closest_silhouette_does_not_depend_on_the_launch(name, leaf_size):
    import snch_lbvh_amd as S

    V, F = _meshes()[name]
    q = _points(V, 70000, 12)
    sc = S.Scene(V, F).build_bvh(leaf_size=leaf_size)
    np_ = lambda r: tuple(x.cpu().numpy() for x in r)  # noqa: E731
    for flip in (False, True):
        e0, d0 = np_(sc.closest_silhouette(q, flip=flip))
        for n in (1, 2, 20, 21, 63, 64, 65, 1000):
            e1, d1 = np_(sc.closest_silhouette(q[:n], flip=flip))
            np.testing.assert_array_equal(d1, d0[:n])
            np.testing.assert_array_equal(e1, e0[:n])
        for kw in ({"block_size": 512}, {"block_size": 128, "stack_depth": 8}, {"stack_depth": 32}, {"coherent": 2}):
            e1, d1 = np_(sc.closest_silhouette(q, flip=flip, **kw))
            np.testing.assert_array_equal(d1, d0)
            np.testing.assert_array_equal(e1, e0)
        # hints too small, about right, too large, zero and none
        r = np.random.default_rng(3)
        seed = np.where(np.isfinite(d0), d0, 1.0) * r.choice([0.0, 0.5, 1.0, 1.25, 1e30], len(d0))
        for n in (65, len(q)):
            e1, d1 = np_(sc.closest_silhouette(q[:n], flip=flip, seed_radius=seed[:n].astype(np.float32)))
            np.testing.assert_array_equal(d1, d0[:n])
            np.testing.assert_array_equal(e1, e0[:n])
        # a hard cap: the answer where it lies within, else something farther
        cap = (np.where(np.isfinite(d0), d0, 1.0) * r.choice([0.5, 1.25], len(d0))).astype(np.float32)
        e1, d1 = np_(sc.closest_silhouette(q, flip=flip, seed_radius=cap, seed_is_cap=True))
        within = d0 <= cap
        np.testing.assert_array_equal(d1[within], d0[within])
        np.testing.assert_array_equal(e1[within], e0[within])
        assert np.all(d1[~within] > cap[~within])


@pytest.mark.parametrize("name", ["ico", "ico_far", "box_far", "two"])
@pytest.mark.parametrize("leaf_size", [1, 8])
def test_rays_do_not_depend_on_the_launch(name, leaf_size):
    import oracle
    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = _meshes()[name]
    n = 70000
    o, d = _points(V, n, 13), W.unit_directions(n, 14)
    d[::7] = np.eye(3, dtype=np.float32)[np.arange(len(d[::7])) % 3]  # along the axes: infinite reciprocals
    r = np.random.default_rng(4)
    tmax = r.choice(np.float32([np.inf, 0.5, 0.0, -1.0, np.nan]), n, p=[0.5, 0.3, 0.1, 0.05, 0.05])
    sc = S.Scene(V, F).build_bvh(leaf_size=leaf_size)
    for tm in (None, tmax):
        cut = lambda k: None if tm is None else tm[:k]  # noqa: E731
        full = [x.cpu().numpy() for x in sc.ray_intersect(o, d, cut(n))]
        for k in (1, 2, 31, 32, 33, 64, 65, 1000):
            part = [x.cpu().numpy() for x in sc.ray_intersect(o[:k], d[:k], cut(k))]
            for a, b in zip(part, full):
                np.testing.assert_array_equal(a, b[:k])
            any_hit = sc.ray_intersect(o[:k], d[:k], cut(k), any_hit=True)[0].cpu().numpy()
            np.testing.assert_array_equal(any_hit, full[0][:k])
        if leaf_size == 1:  # the oracle visits a node's children in the same order
            hit, t = oracle.ray(oracle.build_tree(V, F), o[:4000], d[:4000], cut(4000))[:2]
            np.testing.assert_array_equal(full[0][:4000], hit.astype(bool))
            np.testing.assert_array_equal(full[1][:4000], t)
