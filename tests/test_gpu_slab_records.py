"""The edge slabs that a build leaves in its cone records, at the sizes where
the refit changes its ways (rounds that use all threads of a workgroup and
rounds that use half, one subtree, mid sets, the nodes above): every edge of a
child lies within its slab, every face normal within its cone and the slab's
excess, and nearly all narrow cones have a slab."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _View(ctypes.Structure):
    _fields_ = [(k, ctypes.c_uint32) for k in ("dim", "n_leaves", "flags", "qbase")] + \
               [(k, ctypes.c_void_p) for k in ("tnode", "tcone", "tleaf", "tedge", "nbox", "ncone", "V", "F")]


def _cone_records(S, sc):
    v = _View()
    assert S.lib().snch_scene_device_view(sc._h, 0, ctypes.byref(v)) == 0
    rec = np.empty((v.n_leaves - 1, 16), np.float32)
    assert S.lib().hipMemcpy(ctypes.c_void_p(rec.ctypes.data), ctypes.c_void_p(v.tcone),
                             ctypes.c_size_t(rec.nbytes), 2) == 0
    return rec


def _check(V, F, g, slots, owned, rec, every=1):
    n = len(F)
    V = V.astype(np.float64)
    left, right = g["nodes"][: n - 1, 1].astype(int), g["nodes"][: n - 1, 2].astype(int)
    span = np.zeros((2 * n - 1, 2), int)  # sorted positions of a node's leaves
    span[n - 1:] = np.arange(n)[:, None]
    order, todo = [], [0]
    while todo:
        i = todo.pop()
        order.append(i)
        todo += [c for c in (left[i], right[i]) if c < n - 1]
    for i in reversed(order):
        span[i] = span[left[i], 0], span[right[i], 1]
    a, b, o0, o1 = V[slots[:, 1]], V[slots[:, 2]], V[slots[:, 0]], V[slots[:, 3]]
    with np.errstate(all="ignore"):
        unit = lambda x: x / np.linalg.norm(x, axis=1, keepdims=True)  # noqa: E731
        # slots are (opp1, lo, hi, opp0)
        normals = np.stack([unit(np.cross(b - a, o1 - a)), unit(np.cross(a - b, o0 - b))], 1)
    narrow = held = 0
    for i in range(0, n - 1, every):
        for side, c in ((0, left[i]), (1, right[i])):
            axis, ha, radius = g["cones"][c, :3].astype(np.float64), float(g["cones"][c, 3]), float(g["cones"][c, 4])
            e = owned[g["sorted_idx"][span[c, 0]: span[c, 1] + 1]].ravel()
            e = e[e >= 0]
            if not 0 <= ha < 0.75 or len(e) == 0:
                continue
            word = int(rec[i, 8 * side + 7].view(np.uint32))
            narrow += 1
            excess = (word >> 13) & 63
            if excess < 63:
                nn = normals[e].reshape(-1, 3)
                angle = np.arctan2(np.linalg.norm(np.cross(axis, nn), axis=1), nn @ axis)
                assert angle.max() <= ha + 1e-4 * excess + 64 * 5e-6 + 1e-6
            if word >= 0xFFF80000:
                continue
            held += excess < 63
            lo, hi = g["boxes"][c, :3], g["boxes"][c, 3:]
            centre = ((hi + lo) * np.float32(0.5)).astype(np.float64)
            mid = ((word & 0x1FFF) ^ 0x1000) - 0x1000
            h = (np.concatenate([a[e], b[e]]) - centre) @ axis
            tol = 1e-6 * np.abs(g["boxes"][c]).max()
            assert np.abs(h - mid * radius / 4095).max() <= (word >> 19) * radius / 8191 + tol
    return narrow, held


@pytest.mark.parametrize("n", [2, 3, 700, 1023, 1024, 1025, 3000])
def test_torus(n):
    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(64, 32)
    F = np.ascontiguousarray(F[:n])
    sc = S.Scene(V, F).build_bvh()
    narrow, held = _check(V, F, sc.export(), *sc.silhouettes(), _cone_records(S, sc))
    assert held >= 0.9 * narrow


@pytest.mark.parametrize("layout", ["auto", "memory", "climb"])
@pytest.mark.parametrize("noise", [0.0, 0.001])
def test_sphere(layout, noise):
    """20,480 triangles: cuts, mid sets and nodes above them."""
    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.icosphere(5, noise, seed=1)
    sc = S.Scene(V, F).build_bvh(top_layout=layout)
    rec = _cone_records(S, sc)
    narrow, held = _check(V, F, sc.export(), *sc.silhouettes(), rec, every=7)
    assert narrow > 2000 and held >= 0.9 * narrow
    # the layout does not change a record
    np.testing.assert_array_equal(rec.view(np.uint32), _cone_records(S, S.Scene(V, F).build_bvh()).view(np.uint32))
