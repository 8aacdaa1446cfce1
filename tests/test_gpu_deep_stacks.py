"""Walks whose traversal stacks grow past the levels held in LDS: large overlapping triangles,
so that a ray enters most boxes it tests. Per-ray walk against the oracle's, and camera rays by
one walk per wave (64 frames per pixel) against one walk per ray."""
import numpy as np
import pytest

from scene_cases import hit_test_rays, soup_scene

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("n,size", [(300, 2.0), (4000, 1.5), (20000, 0.7)])
def test_overlapping_triangles(oracle, n, size):
    import torch
    from axomae_amd.nova_hip import HipEngine, RENDER_PER_RAY_TRAVERSAL
    sc = soup_scene(n, 900 + n, size=size)
    e = HipEngine(0)
    e.upload(sc)
    info = e.build_bvh()
    rays = hit_test_rays(sc, "soup", 6000)
    print(f"[stack] {n} triangles of size {size}: wide depth {info.wide_depth}, {len(rays)} rays", flush=True)
    prim, tuv = e.closest_hit(rays)
    oprim, otuv = oracle.OracleScene(sc).closest_hit(rays)
    np.testing.assert_array_equal(prim.cpu().numpy(), oprim)
    np.testing.assert_array_equal(tuv.cpu().numpy(), otuv)
    wave = e.render(24, 18, 64, 1)[1]
    ray = e.render(24, 18, 64, 1, flags=RENDER_PER_RAY_TRAVERSAL)[1]
    assert torch.equal(wave, ray)
    e.close()
