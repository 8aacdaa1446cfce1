"""Bakes at the sizes where the sampled kernel's groups of 2x2 texels, its 16x8 blocks and its
256-sample rounds have remainders: outputs of odd sizes, fewer samples than lanes, one sample
more than a round; 3- and 4-channel maps of odd sizes. Against the oracle, whose bakes take each
texel's samples one after another: the same directions (both compute them with the same float
operations up to sincospi's rounding), so what remains is rounding and, where a direction lies on
a texel's edge, the neighbouring texel. The bakes' tolerance, relative RMSE 1e-3."""
import numpy as np
import pytest

from axomae_amd import scenes

gpu = pytest.mark.gpu


def rel_rmse(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@gpu
@pytest.mark.parametrize("ow,oh", [(1, 1), (2, 3), (15, 9), (17, 8), (33, 17)])
@pytest.mark.parametrize("samples", [1, 63, 257])
def test_sampled_bakes_at_edge_sizes(oracle, ow, oh, samples):
    from axomae_amd import nova_hip as nh
    env = scenes.sky_envmap(61, 37, (0.3, 0.8, 0.2))
    jobs = [(env, ow, oh, nh.BAKE_IRRADIANCE, 0.0), (env, ow, oh, nh.BAKE_IRRADIANCE_SOBOL, 0.0), (env, ow, oh, nh.BAKE_PREFILTER, 0.6),
            (env, ow, oh, nh.BAKE_PREFILTER, 0.0), (None, ow, oh, nh.BAKE_BRDF_LUT, 0.0)]
    refs = [oracle.bake_irradiance(env, ow, oh, samples), oracle.bake_irradiance(env, ow, oh, samples, sobol=True),
            oracle.bake_prefilter(env, ow, oh, 0.6, samples), oracle.bake_prefilter(env, ow, oh, 0.0, samples), oracle.bake_brdf_lut(ow, oh, samples)]
    for job, out, ref in zip(jobs, nh.bake_batch(jobs, samples), refs):
        assert rel_rmse(out, ref) <= 1e-3, (job[1:], samples)


@gpu
@pytest.mark.parametrize("w,h", [(1, 1), (3, 2), (61, 37)])
def test_gl_bakes_of_odd_maps(oracle, w, h):
    """Lookups that wrap on both axes, maps of one texel among them."""
    from axomae_amd import nova_hip as nh
    rs = np.random.RandomState(w)
    env = scenes.Texture(w, h, 4, rs.rand(w * h * 4).astype(np.float32))
    cube, irr = nh.bake_batch([(env, 5, 5, nh.BAKE_CUBEMAP, 0.0), (env, 3, 2, nh.BAKE_IRRADIANCE_RIEMANN, 0.0)], 1)
    assert rel_rmse(cube, oracle.bake_cubemap(env, 5)) <= 1e-3
    assert rel_rmse(irr, oracle.bake_irradiance_riemann(env, 3, 2)) <= 1e-3
