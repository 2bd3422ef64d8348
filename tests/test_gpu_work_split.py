"""The split of a launch's queue over blocks and waves, at the sizes where it changes: frames of one path, of a wave
and a block and one more or less, of one strip per block of the grid and one more, all bit for bit the fp32 oracle's."""
import numpy as np
import pytest

import oracle
from rayna_amd import Renderer, presets

pytestmark = pytest.mark.gpu

# (width, height, samples): paths below, at and above a wave (64), a block (256), the shade grid (16 blocks of 256 per
# CU: 2^20 paths on 256 CUs), where the strips grow from one to two waves' positions
SIZES = [(1, 1, 1), (63, 1, 1), (64, 1, 1), (13, 5, 1), (255, 1, 1), (257, 1, 1), (41, 25, 1), (1024, 1024, 1),
         (1025, 1024, 1)]


@pytest.mark.parametrize("width,height,samples", SIZES)
def test_spheres_equal_the_oracle(gpu, width, height, samples):
    scene, cam, opts = presets.sphere_colours((0.5, 0.7, 0.9), -3.0, width=width, height=height, samples=samples,
                                              ray_depth=3)
    with Renderer(scene, cam, opts) as r:
        out = r.render(layout="rowmajor")
    ref, segments, _, _ = oracle.TwinScene(scene).render(cam, opts, precision=32, box_mode=oracle.BOX_TIGHT)
    assert np.array_equal(out.img, ref)
    assert out.stats.segments == segments


@pytest.mark.parametrize("width,height,samples", [(1, 1, 1), (9, 7, 1), (16, 16, 1), (57, 9, 2), (91, 53, 3)])
def test_marched_scene_equals_the_oracle(gpu, width, height, samples):
    scene, cam, opts = presets.sdf_volume(width=width, height=height, samples=samples, ray_depth=4, max_iterations=64)
    with Renderer(scene, cam, opts) as r:
        out = r.render(layout="rowmajor")
    ref, segments, _, _ = oracle.TwinScene(scene).render(cam, opts, precision=32, box_mode=oracle.BOX_TIGHT)
    assert np.array_equal(out.img, ref)
    assert out.stats.segments == segments
