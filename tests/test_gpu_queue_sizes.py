"""Walks and queues at the edges of their shares: ray and pixel counts around a run of 256, around
the shards of a bounce's queue, and past the lanes of a launch (where lanes refill)."""
import numpy as np
import pytest

from axomae_amd import scenes
from conftest import rel_rmse
from scene_cases import BVH_SCENES

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from axomae_amd.nova_hip import HipEngine
    e = HipEngine(0)
    yield e
    e.close()


@gpu
@pytest.mark.parametrize("n", [786431, 786432, 786433, 1200077])
def test_closest_hit_of_many_rays_equals_its_slices(engine, n):
    """One call over n rays (refilled from a share per workgroup) and calls over slices (a ray per lane)."""
    import torch
    engine.upload(BVH_SCENES["terrain_spheres"]())
    engine.build_bvh()
    g = torch.Generator().manual_seed(n)
    rays = torch.rand(n, 6, generator=g) * 8 - 4
    rays = rays.cuda()
    print(f"[hits] {n} rays", flush=True)
    prim, tuv = engine.closest_hit(rays)
    for a in range(0, n, 200003):
        p, t = engine.closest_hit(rays[a:a + 200003].contiguous())
        assert torch.equal(prim[a:a + 200003], p) and torch.equal(tuv[a:a + 200003], t)
    assert (prim >= 0).any() and (prim < 0).any()


@gpu
@pytest.mark.parametrize("w,h", [(1, 1), (255, 1), (67, 43), (1031, 517)])
def test_passes_match_oracle(oracle, engine, w, h):
    """Pixel by pixel as at the ordinary sizes; a final image over the accumulated one included."""
    import ctypes as C

    import torch
    from axomae_amd import nova_hip as nh
    sc = BVH_SCENES["box_room"]()
    engine.upload(sc)
    engine.build_bvh()
    osc = oracle.OracleScene(sc)
    for pass_, flag in [(1, nh.INTEGRATOR_NORMAL), (2, nh.INTEGRATOR_DEPTH), (3, nh.INTEGRATOR_EMISSIVE)]:
        print(f"[passes] {w}x{h} pass {pass_}", flush=True)
        final, _ = engine.render(w, h, frames=1, max_depth=2, integrator_flags=nh.INTEGRATOR_PATH | flag, z_near=0.1, z_far=50.0)
        ref, _ = osc.render_pass(w, h, 1, pass_, z_near=0.1, z_far=50.0)
        assert np.all(final.cpu().numpy() == ref, axis=2).mean() >= 0.999
        both = torch.zeros_like(final)
        params = nh.render_params(sc, w, h, frames=1, max_depth=2, integrator_flags=nh.INTEGRATOR_PATH | flag, z_near=0.1, z_far=50.0)
        engine._check(engine.L.nova_hip_render_frames(engine.ctx, C.byref(params), both.data_ptr(), both.data_ptr(), None,
                                                      torch.cuda.current_stream().cuda_stream), "render_frames")
        assert torch.equal(both, final)


@gpu
@pytest.mark.parametrize("w,h,frames", [(1, 1, 1), (257, 1, 1), (2048, 1, 1), (2049, 1, 1), (683, 3, 3)])
def test_paths_match_oracle(oracle, engine, w, h, frames):
    sc = scenes.box_room()
    engine.upload(sc)
    engine.build_bvh()
    print(f"[paths] {w}x{h}x{frames}", flush=True)
    final, _ = engine.render(w, h, frames, 4)
    ref, _ = oracle.OracleScene(sc).render(w, h, frames, 4)
    assert rel_rmse(final.cpu().numpy(), ref) <= 1e-3
