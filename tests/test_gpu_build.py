"""Builds whose result must not depend on the order in which threads run:
repeated builds, and hierarchies deeper than the levels queued at once,
against the CPU builder (byte-identical) and the CPU traversal."""

import numpy as np
import pytest

from ordinarylight_amd import workloads
from ordinarylight_amd.renderers.hip import DeviceContext, DeviceScene
from oracle import native as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(hip_device):
    c = DeviceContext(hip_device)
    yield c
    c.close()


def chain(clustered, seed):
    """One triangle per power of two of the 30-bit Morton code, so that every
    binary level of the chain splits one off, and a cluster in the first cell."""
    rng = np.random.default_rng(seed)
    cells = np.zeros((32, 3))
    for k in range(30):
        cells[k, k % 3] = 2 ** (k // 3)
    cells[31] = 1023.0
    centre = np.concatenate(((cells + 0.5) / 1024.0, np.full((clustered, 3), 0.5 / 1024.0)
                             + rng.uniform(-1e-4, 1e-4, (clustered, 3))))
    size = np.concatenate((np.full(32, 2e-4), np.full(clustered, 2e-5)))
    corner = rng.normal(0.0, 1.0, (len(centre), 3, 3))
    corner -= corner.mean(1, keepdims=True)
    return (centre[:, None] + size[:, None, None] * corner).astype(np.float32).reshape(-1, 3)


@pytest.mark.parametrize("triangles, repeats", [(2, 20), (1000, 100), (62_500, 400)])
def test_repeated_builds_are_identical(ctx, triangles, repeats):
    # A subtree's box read before it had arrived gave a node too small a box
    # in about one of 200 builds of the largest size.
    scene, _ = workloads.tessellated_room(1, triangles)
    first = None
    for k in range(repeats):
        ds = DeviceScene(ctx, scene, 2)
        nodes, tri = ds.bvh_arrays()
        if first is None:
            ref = oracle.lbvh_build(ds.packed.positions, ds.packed.indices, 2)
            first = ref["nodes"], ref["tri"].view(np.uint32)
        ds.close()
        assert np.array_equal(nodes, first[0]), f"build {k}"
        assert np.array_equal(tri.view(np.uint32), first[1]), f"build {k}"


@pytest.mark.parametrize("clustered, depth", [(0, 10), (1, 10), (4096, 13), (70_000, 13)])
def test_deep_hierarchies(ctx, clustered, depth):
    from ordinarylight_amd.scene import Scene
    verts = chain(clustered, 7)
    scene = Scene()
    scene.add_mesh(verts, np.arange(len(verts), dtype=np.uint32).reshape(-1, 3))
    ds = DeviceScene(ctx, scene, leaf_size=1)
    nodes, tri = ds.bvh_arrays()
    ref = oracle.lbvh_build(ds.packed.positions, ds.packed.indices, 1)
    assert ds.info.bvh_depth == ref["depth"] >= depth
    assert np.array_equal(nodes, ref["nodes"])
    rng = np.random.default_rng(3)
    n = 20_000
    aim = ds.packed.positions[ds.packed.indices].mean(1)[rng.integers(0, len(ds.packed.indices), n)]
    o = rng.uniform(-0.1, 0.1, (n, 3)).astype(np.float32)
    d = (aim - o).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    got, want = ds.trace(o, d, 0.0, 1e30), oracle.OracleScene(ds.packed).trace(o, d, 0.0, 1e30)
    assert (got[3] != 0xFFFFFFFF).mean() > 0.5
    # Identical but where two triangles' distances round alike (as in the
    # closest-hit comparison over whole scenes).
    assert (got[3] == want[3]).mean() >= 0.9999
    ds.close()
