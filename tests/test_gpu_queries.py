"""Ray queries and downloads at the sizes where they change their route:
pinned buffers up to 4096 rays, then pieces of 768 KB through a ring of two."""

import numpy as np
import pytest

from ordinarylight_amd import workloads
from ordinarylight_amd.renderers.hip import DeviceContext, DeviceScene

pytestmark = pytest.mark.gpu

RAY = 16  # bytes per ray of a hit download


@pytest.fixture(scope="module")
def scene(hip_device):
    ctx = DeviceContext(hip_device)
    built, _ = workloads.tessellated_room(1, 2000)
    ds = DeviceScene(ctx, built, 2)
    yield ds
    ds.close()
    ctx.close()


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, (256 << 10) // RAY - 1, (256 << 10) // RAY + 1, (2 << 20) // RAY,
                               (2 << 20) // RAY + 1, (10 << 20) // RAY + 3, (768 << 10) // RAY - 1, (768 << 10) // RAY,
                               (768 << 10) // RAY + 1, 2 * (768 << 10) // RAY + 1, 3 * (768 << 10) // RAY + 1])
def test_hits_do_not_depend_on_the_size_of_the_call(scene, n):
    rng = np.random.default_rng(n)
    o = rng.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    whole = scene.trace(o, d, 0.001, 1e30)
    for k in list(range(0, n, 4096))[:: max(1, n // 4096 // 24)] + [max(0, n - 4096)]:
        part = scene.trace(o[k:k + 4096], d[k:k + 4096], 0.001, 1e30)
        for a, b in zip(whole, part):
            assert np.array_equal(a[k:k + 4096], b), f"rays from {k}"
    again = scene.trace(o, d, 0.001, 1e30)
    assert all(np.array_equal(a, b) for a, b in zip(whole, again))
