"""The GPU build at the primitive counts where it changes kernels (16-lane rows, waves, whole
workgroups, one workgroup per node, many workgroups per node): primitive order, node count,
depth, leaves and boxes as the reference builder's."""
import numpy as np
import pytest

from scene_cases import soup_scene

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from axomae_amd.nova_hip import HipEngine
    e = HipEngine(0)
    yield e
    e.close()


def _boxes(nodes):
    return sorted(tuple(np.concatenate([n["min"], n["max"]]).tolist()) + (int(n["count"]),) for n in nodes)


@gpu
@pytest.mark.parametrize("n,scale", [(2, 1.0), (3, 1.0), (16, 1.0), (17, 1.0), (64, 1.0), (65, 1.0), (512, 1.0), (513, 1.0), (4097, 1.0), (16384, 1.0),
                                     (16385, 1.0), (40000, 1.0), (600, 4000.0), (20000, 4000.0), (70000, 4000.0)])
def test_build_equals_the_reference_builder(oracle, engine, n, scale):
    """scale 4000: every cost of the upper nodes exceeds float(INT_MAX), so they split at x < 0."""
    sc = soup_scene(n, 100 + n, lo=-scale, hi=scale, size=0.05 * scale, duplicate=n // 50)
    print(f"[build] {n} triangles, scale {scale}", flush=True)
    engine.upload(sc)
    info = engine.build_bvh()
    prim, nodes = engine.bvh_arrays()
    oprim, onodes = oracle.OracleScene(sc).bvh_arrays()
    np.testing.assert_array_equal(prim, oprim)
    assert info.binary_nodes == len(onodes) and info.leaves == int((onodes["count"] > 0).sum())
    assert _boxes(nodes) == _boxes(onodes)
    depth = np.zeros(len(onodes), dtype=int)
    for k, nd in enumerate(onodes):  # the reference's children follow their parent
        if nd["count"] == 0:
            depth[nd["left"]] = depth[nd["left"] + 1] = depth[k] + 1
    assert info.binary_depth == depth.max() + 1
