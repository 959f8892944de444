"""A refused frame: what was set before stays, whole and usable, and a frame that
was never set is still not set."""
import numpy as np
import pytest

from pmarch import PmError, scenes

pytestmark = pytest.mark.gpu


def _refused(kind, n):
    """More particles than the frame holds, refused for one reason."""
    xyz = np.random.default_rng(1).uniform(0, 1, (n, 3)).astype(np.float32)
    if kind == "inf":
        xyz[n // 2, 1] = np.inf
    elif kind == "nan":              # one coordinate among many
        xyz[n // 2, 1] = np.nan
    elif kind == "far":              # every key beyond an int32
        xyz += np.float32(3.0e8)
    elif kind == "grid":             # cells of h
        xyz[0] = -2.0e4
    elif kind == "march grid":       # cells of h/2 alone: 700^3 and 1400^3
        xyz[0] = -69.0
    elif kind == "product":          # 2^64 cells of h, a product that wraps to 0
        xyz[0] = (-0.1 * (2 ** 22 - 12), -0.1 * (2 ** 21 - 12), -0.1 * (2 ** 21 - 12))
    return xyz


@pytest.mark.parametrize("stream", [False, True])
@pytest.mark.parametrize("kind", ["inf", "nan", "far", "grid", "march grid", "product"])
def test_refused_frame(marcher, kind, stream):
    sc = scenes.lattice_cube(2, n_side=8, spacing=0.05, width=48, height=32)
    c = sc.cameras[0]
    print(f"refused frame {kind} stream {stream}", flush=True)
    marcher.set_frame(61, sc.xyz, sc.h)
    st = sc.settings(skip_mode=4)
    view = (st, c.inv_pv, c.eye, c.width, c.height)
    marcher.batch_set(st, [(61, c.width, c.height, c.inv_pv, c.eye)])
    want, grid = marcher.march(61, *view), marcher.grid(61)
    bad = _refused(kind, 5 * len(sc.xyz))
    build = marcher.set_frame_stream if stream else marcher.set_frame
    for frame in (61, 9000):
        with pytest.raises(PmError):
            build(frame, bad, sc.h)
    info = marcher.frame_info(61)
    assert info.n == len(sc.xyz) and list(info.dims) == list(grid[0].dims)
    with pytest.raises(PmError):
        marcher.frame_info(9000)
    with pytest.raises(PmError):
        marcher.march(9000, *view)
    with pytest.raises(PmError):
        marcher.depth_sprites(9000, c, 0.05)
    for a, b in zip(marcher.grid(61)[1:], grid[1:]):
        assert np.array_equal(a, b)
    for a, b in zip(marcher.march(61, *view)[:3], want[:3]):
        assert np.array_equal(a, b)
    marcher.batch_run()
    marcher.wait()
    for a, b in zip(marcher.batch_download(0), want[:3]):
        assert np.array_equal(a, b)
    sc2 = scenes.lattice_cube(3, n_side=9, spacing=0.05)
    assert build(61, sc2.xyz, sc2.h).n == len(sc2.xyz)
