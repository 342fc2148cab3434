"""Hints and hard caps of the closest silhouette on launches whose waves take
several chunks each (more queries than 64 per resident wave)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [393217, 800001])
@pytest.mark.parametrize("flip", [False, True])
def test_large_hinted_and_capped(n, flip):
    import torch

    import snch_lbvh_amd as S
    from snch_lbvh_amd import workloads as W

    V, F = W.cut_torus(24, 12)
    lo, hi = W.padded_box(V, 0.2)
    sc = S.Scene(V, F).build_bvh()
    q = torch.from_numpy(W.uniform_points(n, lo, hi, n)).cuda()
    e0, d0 = sc.closest_silhouette(q, flip=flip)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    near = torch.where(torch.isfinite(d0), d0, torch.ones_like(d0))
    # too small, exact, too large and none
    scale = torch.tensor([0.0, 0.5, 1.0, 1.25, float("inf")], device="cuda")[
        torch.randint(0, 5, (n,), generator=g, device="cuda")]
    hint = torch.where(torch.isfinite(scale), near * scale, scale)
    e1, d1 = sc.closest_silhouette(q, flip=flip, seed_radius=hint)
    assert torch.equal(d0, d1) and torch.equal(e0, e1)
    cap = near * torch.where(torch.rand(n, generator=g, device="cuda") < 0.5, 0.5, 1.25)
    e2, d2 = sc.closest_silhouette(q, flip=flip, seed_radius=cap, seed_is_cap=True)
    within = d0 <= cap
    assert torch.equal(d2[within], d0[within]) and torch.equal(e2[within], e0[within])
    assert bool((d2[~within] > cap[~within]).all())
