"""Few-path batches walk with the next node's words ahead, large ones without: one call of 9 frames
(7,077,888 paths, past the line between the two) and 9 calls of one frame give the same image bit
for bit, as every ray takes the same steps."""
import numpy as np
import pytest

from scene_cases import BVH_SCENES

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("scene", ["terrain_spheres", "box_room"])
def test_large_batch_equals_single_frames(scene):
    from axomae_amd import nova_hip as nh
    eng = nh.HipEngine(0)
    try:
        eng.upload(BVH_SCENES[scene]())
        eng.build_bvh()
        one, acc = eng.render(1024, 768, 9, 4, flags=nh.RENDER_PER_RAY_TRAVERSAL)
        accum = None
        for f in range(9):
            final, accum = eng.render(1024, 768, 1, 4, frame_start=f, accum=accum, flags=nh.RENDER_PER_RAY_TRAVERSAL)
        np.testing.assert_array_equal(accum.cpu().numpy(), acc.cpu().numpy())
        np.testing.assert_array_equal(final.cpu().numpy(), one.cpu().numpy())
    finally:
        eng.close()
