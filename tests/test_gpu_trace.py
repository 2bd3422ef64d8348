"""Paths traced to their ends in one launch against one launch per depth: validation keeps a frame on the latter (and
changes no pixel), so every scene's two frames and closest-hit counts must be equal, whatever the depth limit, the
samples per pixel (below and from 16 on, where the camera rays are packets), the number of chunks and, with unbounded
objects, the number of paths (from 128 * 128 on the camera rays get launches of their own).  Up to 2^17 paths, for the
largest trees 2^20, a path has four lanes, beyond that one."""
import numpy as np
import pytest

import oracle
from rayna_amd import Camera, Renderer, RenderOpts, Scene, presets
from rayna_amd.batch import BatchRenderer, Request
from tests.test_stack_bound import deep_scene

pytestmark = pytest.mark.gpu

SCENES = {"mesh": lambda **k: presets.triangle_mesh(subdiv=3, **k), "spheres": presets.random_spheres,
          "cornell": presets.cornell, "rttnw": lambda **k: presets.rttnw(balls=50, **k),
          "textured": presets.textured, "transformed": presets.transformed_mix,
          "inverse": lambda **k: presets.inverse_spheres(**k)[:3], "mixed": presets.mixed_primitives,
          "sdf": lambda **k: presets.sdf_volume(max_iterations=64, **k)}


@pytest.mark.parametrize("scene", sorted(SCENES))
@pytest.mark.parametrize("width,height,samples,depth,chunk", [(1, 1, 1, 6, 0), (37, 23, 15, 0, 0), (37, 23, 16, 0, 0),
                                                             (37, 23, 17, 1, 0), (64, 64, 3, 7, 0), (33, 65, 40, 5, 0),
                                                             (64, 33, 40, 4, 64 * 33 * 17),
                                                             (128, 127, 1, 4, 0), (128, 128, 1, 4, 0),
                                                             (363, 361, 1, 5, 0), (1025, 1024, 1, 3, 0),
                                                             (257, 256, 16, 4, 0)])
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


@pytest.mark.parametrize("scene", ["cornell", "mixed", "rttnw", "sdf", "textured"])
@pytest.mark.parametrize("samples", [3, 16])
def test_adjoint_equals_the_oracle(gpu, scene, samples):
    """The replay in one launch, on scenes with instances, media, textures and unbounded objects: the oracle's gradient
    up to the order of its float64 sums."""
    sc, cam, opts = SCENES[scene](width=24, height=16, samples=samples, ray_depth=5)
    d = np.random.default_rng(3).standard_normal((16, 24, 3)).astype(np.float32)
    with Renderer(sc, cam, opts) as r:
        g, _ = r.adjoint(d, layout="rowmajor")
    ref, _, _ = oracle.TwinScene(sc).adjoint(cam, opts, d, precision=32)
    assert np.linalg.norm(g - ref) <= 1e-9 * np.linalg.norm(ref)


@pytest.mark.parametrize("first,last", [(64, 1), (40, 25), (64, 17)])
def test_camera_ray_time_of_unequal_chunks(gpu, first, last):
    """A frame's chunks may differ in the depths that get launches of their own (here 2 and 0, 2 and 1, 2 and 1): the
    time of the camera rays is the sum of their own launches.  They are about a sixth of the time here, alone as in chunks
    (0 and two thirds were reported)."""
    sc, cam, opts = presets.triangle_mesh(subdiv=5, width=960, height=540, samples=first + last)
    with Renderer(sc, cam, opts) as r:
        r.set_tuning(chunk_slots=960 * 540 * first)
        shares = []
        for _ in range(3):
            s = r.render(to_host=False).stats
            shares.append(s.extend_camera_ms / s.extend_ms)
        assert s.extend_launches == 2 * (opts.ray_depth + 1)
    assert 0.02 < np.median(shares) < 0.4


@pytest.mark.parametrize("width,height,samples", [(1, 1, 1), (37, 23, 3), (150, 120, 7)])
def test_quad_stacks_past_their_lds_share(gpu, width, height, samples):
    """Four lanes to a path (up to 2^17 of them) on a tree that takes 55 stack entries, 44 of them in LDS; and with 16
    samples to a pixel the first bounce from the camera-ray packets' hits."""
    scene = deep_scene()
    cam = Camera(pos=(0.2, 0.0, 0.0), fwd=(1.0, 0.0, 0.0), v_fov=60.0, focus_dist=1.0)
    for spp in (samples, 16):
        opts = RenderOpts(width, height, spp, 4)
        with Renderer(scene, cam, opts) as r:
            out = r.render(layout="rowmajor")
        ref, segments, _, _ = oracle.TwinScene(scene).render(cam, opts, precision=32, box_mode=oracle.BOX_TIGHT)
        assert np.array_equal(out.img, ref)
        assert out.stats.segments == segments


@pytest.mark.parametrize("scene,width,height,samples,knob", [("mixed", 640, 360, 64, "refill_lanes"),
                                                            ("cornell", 360, 360, 1, "wave_batch")])
def test_tuning_reaches_the_whole_path_launches(gpu, scene, width, height, samples, knob):
    """Scenes with unbounded objects heed refill_lanes and paths with four lanes wave_batch: one lane, or one path, at a
    time takes far longer than the default (1.6 and 2.2 times; a fifth is asked for), and no value changes the image."""
    sc, cam, opts = SCENES[scene](width=width, height=height, samples=samples)
    times, images = [], []
    with Renderer(sc, cam, opts) as r:
        for v in (0, 1, 64 if knob == "refill_lanes" else 4096):
            r.set_tuning(**{knob: v})
            r.clear_accumulation()
            images.append(r.render(layout="rowmajor").img)
            times.append(np.median([r.render(to_host=False).stats.kernel_ms for _ in range(7)]))
    assert all(np.array_equal(images[0], i) for i in images[1:])
    assert times[1] > 1.2 * times[0]


@pytest.mark.parametrize("width,samples,depth,apart", [(40, 1, 0, True), (40, 1, 1, True), (40, 1, 2, False),
                                                       (1449, 1, 2, True), (1449, 1, 3, True), (1448, 1, 3, True),
                                                       (200, 6, 2, True), (200, 6, 0, True)])
@pytest.mark.parametrize("scene", ["two sets of blobs", "bulb and blobs", "blobs"])
def test_scenes_of_marches(gpu, scene, width, samples, depth, apart):
    """Scenes of nothing but marches: several unbounded objects' depths get launches of their own in frames of few vertices
    to a path and from 2^21 paths on (1449 * 1449; with a Mandelbulb from 3 * 2^23), between 2^14 paths and those the
    camera rays do; the frames equal those of a launch per depth."""
    sc, cam, opts = presets.sdf_volume(width=width, height=width, samples=samples, ray_depth=depth, max_iterations=48)
    bulb, blobs = sc.objects[:2]
    moved, _, _ = presets.sdf_volume(seed=9, max_iterations=48)
    sc = Scene({"two sets of blobs": [blobs, moved.objects[1]], "bulb and blobs": [bulb, blobs], "blobs": [blobs]}[scene],
               sc.skybox)
    with Renderer(sc, cam, opts) as r:
        out = r.render(layout="rowmajor")
        r.clear_accumulation()
        r.set_validate(True)
        ref = r.render(layout="rowmajor")
    assert np.array_equal(out.img, ref.img) and out.stats.segments == ref.stats.segments
    if scene == "blobs":
        apart = depth == 0 or 1 << 14 <= width * width * samples < 1 << 21
    elif scene == "bulb and blobs" and width == 1449 and depth == 3:
        apart = False
    assert (out.stats.shade_ms > 0.0) == apart


@pytest.mark.parametrize("scene,width,samples,apart", [("mesh", 1024, 16, 2), ("mesh", 1023, 16, 1), ("inverse", 1024, 16, 2),
                                                       ("cornell", 1024, 16, 1), ("rttnw", 1024, 64, 2),
                                                       ("rttnw", 1023, 64, 0)])
def test_first_bounce_of_large_frames(gpu, scene, width, samples, apart):
    """From 2^24 paths on, the first bounce gets launches of its own in trees of some size and in scenes with media or
    instances (without camera-ray packets from 2^26 on); the frames equal those of a launch per depth."""
    sc, cam, opts = SCENES[scene](width=width, height=width, samples=samples, ray_depth=3)
    with Renderer(sc, cam, opts) as r:
        out = r.render(layout="rowmajor")
        r.set_validate(True)
        r.clear_accumulation()
        ref = r.render(layout="rowmajor")
    assert np.array_equal(out.img, ref.img) and out.stats.segments == ref.stats.segments
    with BatchRenderer([sc]) as b:
        imgs, st = b.render([Request(0, cam, opts)])
    assert np.array_equal(imgs[0], ref.img)
    assert st.launches == 3 + 2 * apart + 1 + 3 + 1
