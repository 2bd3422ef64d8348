"""Paths traced to their ends in one launch against one launch per depth: validation keeps a frame on the latter (and
changes no pixel), so every scene's two frames and closest-hit counts must be equal, whatever the depth limit, the
samples per pixel (below and from 16 on, where the camera rays are packets) and the number of chunks."""
import numpy as np
import pytest

from rayna_amd import Renderer, presets

pytestmark = pytest.mark.gpu

SCENES = {"mesh": lambda **k: presets.triangle_mesh(subdiv=3, **k), "spheres": presets.random_spheres,
          "cornell": presets.cornell, "rttnw": lambda **k: presets.rttnw(balls=50, **k),
          "textured": presets.textured, "transformed": presets.transformed_mix,
          "inverse": lambda **k: presets.inverse_spheres(**k)[:3]}


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("width,height,samples,depth,chunk", [(1, 1, 1, 6, 0), (37, 23, 15, 0, 0), (37, 23, 16, 0, 0),
                                                             (37, 23, 17, 1, 0), (64, 64, 3, 7, 0), (33, 65, 40, 5, 0),
                                                             (64, 33, 40, 4, 64 * 33 * 17)])
def test_one_launch_equals_one_per_depth(gpu, scene, width, height, samples, depth, chunk):
    sc, cam, opts = SCENES[scene](width=width, height=height, samples=samples, ray_depth=depth)
    frames = []
    for validate in (False, True):
        with Renderer(sc, cam, opts) as r:
            r.set_tuning(chunk_slots=chunk)
            r.set_validate(validate)
            for _ in range(2):  # the second frame: another RNG key, the queues and counters used again
                out = r.render(layout="rowmajor")
                frames.append((out.img, out.stats.segments))
    for a, b in zip(frames[:2], frames[2:]):
        assert np.array_equal(a[0], b[0])
        assert a[1] == b[1]
