"""The batch tuner does not choose between options that launch the same thing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_depth_8_is_no_choice():
    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(300, 150)
    b = S.BatchScene([(V, F)]).build_bvh()
    lo, hi = W.padded_box(V, 0.2)
    n = 200000
    q = W.uniform_points(n, lo, hi, 7)
    for kind in ("silhouette", "point"):
        for _ in range(10):  # (noise alone prefers one of two equal launches half of the time)
            assert b.autotune(q, np.array([0, n], np.uint32), kind=kind)["stack_depth"] != 8
