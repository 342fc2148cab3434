"""A rebuild that reports an earlier call's error has still built the tree: the
scene answers from it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _raise_sticky_word(lib):
    """Sets the device's traversal error word from the host."""
    word = lib._ZN4snch20traversal_error_wordEv
    word.restype = ctypes.c_void_p
    one = ctypes.c_uint32(1)
    assert lib.hipMemcpy(ctypes.c_void_p(word()), ctypes.byref(one), ctypes.c_size_t(4), 1) == 0


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("first,then", [(1, 8), (8, 1)])
def test_queries_after_a_failed_rebuild(batch, first, then):
    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(48, 24)
    lo, hi = W.padded_box(V, 0.2)
    q = W.uniform_points(3000, lo, hi, 3)
    off = (np.array([0, len(q)]),) if batch else ()
    new = lambda: S.BatchScene([(V, F)]) if batch else S.Scene(V, F)  # noqa: E731
    ask = lambda s: [x.cpu().numpy() for f in (s.closest_point, s.closest_silhouette) for x in f(q, *off)]  # noqa: E731
    want = ask(new().build_bvh())
    sc = new().build_bvh(leaf_size=first)
    _raise_sticky_word(S.lib())
    with pytest.raises(Exception):
        sc.build_bvh(leaf_size=then)
    for a, b in zip(ask(sc), want):
        np.testing.assert_array_equal(a, b)
    for a, b in zip(ask(sc.build_bvh(leaf_size=then)), want):  # the word is clear again
        np.testing.assert_array_equal(a, b)
