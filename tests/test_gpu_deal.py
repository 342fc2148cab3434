"""How a launch deals its queries to waves (runs of 1 to 64 neighbours), and the
largest wave pools: answers are those of small launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [393215, 393217, 800001, 1600001, 3200001])
@pytest.mark.parametrize("coherent", [0, 2])
def test_runs(n, coherent):
    import torch

    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(24, 12)
    lo, hi = W.padded_box(V, 0.2)
    sc = S.Scene(V, F).build_bvh()
    q = torch.from_numpy(W.uniform_points(n, lo, hi, n)).cuda()
    d = torch.nn.functional.normalize(q.roll(1, 0) - 0.5, dim=1)
    parts = [slice(a, min(n, a + 60000)) for a in range(0, n, 60000)]
    for f in (lambda s: sc.closest_point(q[s], coherent=coherent),
              lambda s: sc.closest_silhouette(q[s], coherent=coherent),
              lambda s: sc.ray_intersect(q[s], d[s])[:2]):
        whole = f(slice(0, n))
        small = [f(s) for s in parts]
        for k, x in enumerate(whole):
            assert torch.equal(x, torch.cat([s[k] for s in small]))


@pytest.mark.parametrize("block_size", [64, 512])
@pytest.mark.parametrize("cap", [False, True])
def test_largest_pools(block_size, cap):
    """Eight waves of 1,280 pending nodes (and, with a cap, their bounds) share
    one workgroup's LDS."""
    import torch

    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(64, 32)
    lo, hi = W.padded_box(V, 0.2)
    sc = S.Scene(V, F).build_bvh()
    q = torch.from_numpy(W.uniform_points(20000, lo, hi, 5)).cuda()
    e0, d0 = sc.closest_silhouette(q)
    if cap:
        e1, d1 = sc.closest_silhouette(q, seed_radius=torch.full((20000,), 10.0, device="cuda"), seed_is_cap=True,
                                       block_size=block_size, stack_depth=32)
    else:
        e1, d1 = sc.closest_silhouette(q, block_size=block_size, stack_depth=32)
    assert torch.equal(d0, d1) and torch.equal(e0, e1)


@pytest.mark.parametrize("sizes", [(1, 70, 1), (5001, 0, 63), (450001, 10, 129)])
@pytest.mark.parametrize("queries_per_wave", [64, 256])
def test_batch(sizes, queries_per_wave):
    import torch

    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    meshes = [W.cut_torus(24, 12), W.cut_torus(8, 6), (W.icosphere(2, 0.05, seed=2))]
    lo, hi = W.padded_box(meshes[0][0], 0.2)
    q = torch.from_numpy(W.uniform_points(sum(sizes), lo, hi, 7)).cuda()
    off = np.cumsum([0, *sizes])
    b = S.BatchScene(meshes).build_bvh()
    tune = {"block_size": 128, "stack_depth": 8, "queries_per_wave": queries_per_wave}
    for name in ("closest_point", "closest_silhouette"):
        i, d = getattr(b, name)(q, off, tune=tune)
        for m, (V, F) in enumerate(meshes):
            s = slice(int(off[m]), int(off[m + 1]))
            if sizes[m]:
                i1, d1 = getattr(S.Scene(V, F).build_bvh(), name)(q[s])
                assert torch.equal(d[s], d1) and torch.equal(i[s], i1)
