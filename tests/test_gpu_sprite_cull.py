"""The depth-sprite pass with its sample and hidden-tile test: the image equals
the oracle's bit for bit around the particle count where the sample begins, from
outside and inside the cloud, with background, ragged sizes, large and tiny
sprites, and with matrices that switch the test off."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from pmarch import scenes
from pmarch.camera import make_camera

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 4095, 4096, 4113, 20000])
@pytest.mark.parametrize("size", [(8, 8), (67, 41), (256, 161)])
@pytest.mark.parametrize("radius", [0.003, 0.04, 0.3])
def test_sprites_equal_oracle(marcher, n, size, radius):
    rng = np.random.default_rng(n)
    xyz = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32) * np.float32([1, 0.6, 1.4])
    print(f"sprites n={n} {size} R={radius}", flush=True)
    marcher.set_frame(70, xyz, 0.1)
    for eye, target in (((1.1, 0.8, -1.6), (0, 0, 0)), ((0.05, 0.02, -0.1), (0.1, 0.1, 0.8)), ((0, 0, -90.0), (0, 0, 0))):
        cam = make_camera(eye, target, *size)
        assert np.array_equal(marcher.depth_sprites(70, cam, radius), O.depth_sprites(xyz, cam, radius))


@pytest.mark.parametrize("entry", [(8, 0.05), (2, 0.02), (10, -1.0), (15, 0.5)])
def test_sprites_other_matrices(marcher, entry):
    """Projections whose depth leaves the view z (or falls with it), a scaled
    View: no sprite may be left out."""
    rng = np.random.default_rng(1)
    xyz = rng.uniform(-0.5, 0.5, (6000, 3)).astype(np.float32)
    marcher.set_frame(70, xyz, 0.1)
    cam = make_camera((1.1, 0.8, -1.6), (0, 0, 0), 131, 77)
    proj, view = cam.proj.copy(), cam.view.copy()
    proj[entry[0]] = np.float32(entry[1])
    view[[0, 4, 8]] *= np.float32(1.5)
    print(f"sprites other matrices {entry}", flush=True)
    for c in (dataclasses.replace(cam, proj=proj), dataclasses.replace(cam, view=view)):
        assert np.array_equal(marcher.depth_sprites(70, c, 0.05), O.depth_sprites(xyz, c, 0.05))


@pytest.mark.parametrize("n,radius", [(n, r) for n in (16383, 16384, 20011, 270000) for r in (0.004, 0.02, 0.06, 0.3)
                                      if n * r < 20000])
def test_sprites_sampled(marcher, n, radius):
    """Around the particle count where the sample begins and, beyond 262,144, where
    its small sprites take eight lanes each: footprints of a pixel to most of the
    image, drawn by a lane, by pairs or by a wave, hidden or not."""
    rng = np.random.default_rng(n)
    xyz = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32) * np.float32([1, 0.6, 1.4])
    print(f"sprites sampled n={n} R={radius}", flush=True)
    marcher.set_frame(70, xyz, 0.1)
    for size in ((97, 60), (211, 131)):
        for eye, target in (((1.1, 0.8, -1.6), (0, 0, 0)), ((0.05, 0.02, -0.1), (0.1, 0.1, 0.8))):
            cam = make_camera(eye, target, *size)
            assert np.array_equal(marcher.depth_sprites(70, cam, radius), O.depth_sprites(xyz, cam, radius))


@pytest.mark.parametrize("entry", [(8, 0.05), (2, 0.02), (10, -1.0), (15, 0.5)])
def test_sprites_sampled_other_matrices(marcher, entry):
    """As test_sprites_other_matrices, with enough particles for a sample."""
    rng = np.random.default_rng(1)
    xyz = rng.uniform(-0.5, 0.5, (20000, 3)).astype(np.float32)
    marcher.set_frame(70, xyz, 0.1)
    cam = make_camera((1.1, 0.8, -1.6), (0, 0, 0), 131, 77)
    proj, view = cam.proj.copy(), cam.view.copy()
    proj[entry[0]] = np.float32(entry[1])
    view[[0, 4, 8]] *= np.float32(1.5)
    print(f"sprites sampled, other matrices {entry}", flush=True)
    for c in (cam, dataclasses.replace(cam, proj=proj), dataclasses.replace(cam, view=view)):
        assert np.array_equal(marcher.depth_sprites(70, c, 0.1), O.depth_sprites(xyz, c, 0.1))
