"""Texel wrapping and channel decoding of the texture pass at the smallest
textures (one period is one or two texels, so a bilinear footprint leaves it
on both sides), in every wrap mode, against the CPU oracle."""

import numpy as np
import pytest

from ordinarylight_amd import cameras, packing, workloads
from ordinarylight_amd.renderers.hip import HipPathTracer
from ordinarylight_amd.scene import Material, Texture, TextureTransform
from oracle import native as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wrap", ["repeat", "clamp", "mirror"])
@pytest.mark.parametrize("size", [(1, 1), (1, 2), (2, 1), (3, 5)])
@pytest.mark.parametrize("linear", [True, False])
def test_smallest_textures_match_oracle(hip_device, wrap, size, linear):
    rng = np.random.default_rng(11)
    scene, cam = workloads.box_room(0)
    pixels = rng.integers(0, 256, (*size, 4)).astype(np.uint8)
    floor_v, floor_i = workloads._quad((-1, 0.01, -1), (-1, 0.01, 1), (1, 0.01, 1), (1, 0.01, -1))
    texture = Texture(pixels, wrap_s=wrap, wrap_t=wrap, linear_filter=linear)
    material = Material(base_color=(0.9, 0.9, 0.9), roughness=0.8, base_color_texture=texture,
                        base_color_transform=TextureTransform(offset=(-0.7, 0.4), scale=(2.5, 3.5)),
                        metallic_roughness_texture=texture)
    scene.add_mesh(floor_v, floor_i, material, texcoords=workloads._planar_uv(floor_v[:, [0, 2, 1]], 1.0))
    r = HipPathTracer(max_bounces=3, samples_per_pixel=2)
    img = r.render_frame(scene, cam, 64, 48)[..., :3]
    r.close()
    orc = oracle.OracleScene(packing.pack_scene(scene))
    ref = orc.render(cameras.camera_basis(cam), cameras.camera_projection(cam), 64, 48, 2, 0, max_bounces=3)[..., :3]
    orc.close()
    # The bound of the textured-scene comparison: 1e-3 relative on 99.9 % of
    # pixels (mismatches are path divergences at edges).
    ok = np.all(np.abs(img - ref) <= 1e-6 + 1e-3 * np.maximum(np.abs(img), np.abs(ref)), axis=-1)
    assert ok.mean() >= 0.999
