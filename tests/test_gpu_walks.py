"""The candidate-list walk and the skip distance field at their edges: lists that
fit, fill up between planes, or are shorter than one plane or one row of the
stencil; rays that cross many clear cells at once.  Images and counters equal
the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle as O
from pmarch import scenes

pytestmark = pytest.mark.gpu

KEYS = dict(O.Settings._fields_)
COUNTERS = ("rays", "rays_in_aabb", "hits", "samples", "march_samples", "march_cand")


def _check(marcher, sc, counters=COUNTERS, **kw):
    c = sc.cameras[0]
    st = sc.settings(**kw)
    pos, nrm, t, got = marcher.march(60, st, c.inv_pv, c.eye, c.width, c.height)
    o = O.march(O.Grid(sc.xyz, sc.h), O.make_settings(**{k: v for k, v in st.items() if k in KEYS}), c.inv_pv, c.eye,
                c.width, c.height)
    assert np.array_equal(pos, o[0]) and np.array_equal(nrm, o[1]) and np.array_equal(t, o[2])
    for k in counters:
        assert got[k] == o[3][k], (k, got[k], o[3][k])
    return got


@pytest.mark.parametrize("per_cell", [1, 3, 9, 40])
@pytest.mark.parametrize("compensated", [0, 1])
def test_list_walk_fill(marcher, per_cell, compensated):
    """per_cell particles in each h/2 cell: a 25-cell plane holds up to 25, 75,
    225 and 1,000 candidates, a 5-cell row up to 200, against 36 list slots."""
    rng = np.random.default_rng(per_cell)
    h = 0.1
    base = np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij"), -1).reshape(-1, 1, 3) * (h / 2)
    xyz = (base + rng.uniform(0, h / 2, (base.shape[0], per_cell, 3))).reshape(-1, 3).astype(np.float32)
    sc = scenes.tiny_scene(xyz, h, eye=(0.9, 0.8, -0.7), target=(0.22, 0.22, 0.22), width=44, height=37)
    sc.iso *= per_cell
    print(f"list walk, {per_cell} per cell, compensated {compensated}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    for skip in (0, 1, 4):
        got = _check(marcher, sc, skip_mode=skip, compensated=compensated)
        assert got["hits"] > 100


@pytest.mark.parametrize("gap", [1, 2, 9, 40])
def test_skip_over_clear_cells(marcher, gap):
    """Three small clusters `gap` cells apart, so rays cross clear regions of
    every radius up to and beyond the field's largest; a grid side not a
    multiple of anything."""
    rng = np.random.default_rng(gap)
    h = 0.1
    centres = np.array([[0, 0, 0], [gap + 4, 0.4, 0.3], [0.2, gap + 4, gap + 3]]) * h
    xyz = np.concatenate([c + rng.uniform(-1.6 * h, 1.6 * h, (300, 3)) for c in centres]).astype(np.float32)
    mid = xyz.mean(0)
    ext = float((xyz.max(0) - xyz.min(0)).max())
    sc = scenes.tiny_scene(xyz, h, eye=mid + np.array([0.9, 0.7, -1.1]) * ext, target=mid, width=71, height=53)
    print(f"skip over {gap} clear cells", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    for boxes in (0, 1):
        got = _check(marcher, sc, skip_mode=4, bound_boxes=boxes)
        assert got["hits"] > 10


@pytest.mark.parametrize("eps,bisect,fp64", [(0.1 / 32, 8, 1), (0.02, 8, 1), (0.1 / 32, 0, 0), (0.1 / 32, 3, 0),
                                             (-0.1 / 32, 2, 1), (0.0, 8, 1)])
@pytest.mark.parametrize("step", [0.0125, 0.04, 0.3])
def test_finish_list(marcher, eps, bisect, fp64, step):
    """A hit's samples from one list: short steps (the list), steps and offsets
    whose box spans more cells than the list takes (the walk for each sample),
    no bisection, an offset of zero or below it; hits at the grid's edge."""
    sc = scenes.lattice_cube(3, n_side=9, spacing=0.05, width=61, height=43)
    sc.step, sc.normal_eps = step, eps
    print(f"finish list eps {eps} bisect {bisect} fp64 {fp64} step {step}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    for comp in (0, 1):
        got = _check(marcher, sc, skip_mode=4, bisect_iters=bisect, final_fp64=fp64, compensated=comp)
        assert got["hits"] > 50


@pytest.mark.parametrize("size", [(9, 7), (64, 40), (333, 207)])
@pytest.mark.parametrize("aniso", [0, 1])
@pytest.mark.parametrize("normal_mode", [0, 1])
def test_reference_groups(marcher, size, aniso, normal_mode):
    """The reference march in lane groups: few, some and many active tiles, a
    MaxSteps that no group size divides, every skip, both normals; and the
    anisotropic configured march and its finish at the same sizes."""
    from parity import depth_in_front
    sc = scenes.lattice_cube(5, n_side=12, spacing=0.05, width=size[0], height=size[1])
    c = sc.cameras[0]
    print(f"reference groups {size} aniso {aniso} normals {normal_mode}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    G = O.Grid(sc.xyz, sc.h)
    depth = depth_in_front(c, G.bmin, G.bmax, 0.01).astype(np.float32)
    extra = dict(scenes.ANISO_SETTINGS, iso=1.0) if aniso else dict(iso=sc.iso)
    for skip, steps in ((0, 37), (2, 101), (3, 1)):
        st = dict(mode=1, max_steps=steps, step=0.013, normal_mode=normal_mode, normal_eps=sc.normal_eps,
                  skip_mode=skip, compensated=skip & 1, **extra)
        pos, nrm, t, got = marcher.march(60, st, c.inv_pv, c.eye, c.width, c.height, depth=depth)
        o = O.march(G, O.make_settings(**st), c.inv_pv, c.eye, c.width, c.height, depth=depth)
        assert np.array_equal(pos, o[0]) and np.array_equal(t, o[2])
        assert np.array_equal(nrm, o[1], equal_nan=True)
        for k in ("rays_in_aabb", "hits", "samples", "cand", "march_samples"):
            assert got[k] == o[3][k], (k, got[k], o[3][k])
    if aniso:
        _check(marcher, sc, counters=("rays", "hits", "samples", "cand", "march_samples"), skip_mode=4,
               normal_mode=normal_mode, **extra)


@pytest.mark.parametrize("tiles", [(7, 9), (8, 8), (13, 5), (47, 17), (25, 32), (25, 33)])
@pytest.mark.parametrize("per_cell", [1, 12])
def test_tile_list_and_group_finish(marcher, tiles, per_cell):
    """Tile counts around a mask's 64 (63, 64, 65) and around the finish rule's
    line for sparse frames (799, 800, 825), ragged right and lower edges; 12 per
    h/2 cell is a dense frame, whose small images all finish in lane groups.
    Both normals, offsets that leave the list, no bisection, no FP64 step."""
    rng = np.random.default_rng(per_cell)
    h = 0.1
    base = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 1, 3) * (h / 2)
    xyz = (base + rng.uniform(0, h / 2, (base.shape[0], per_cell, 3))).reshape(-1, 3).astype(np.float32)
    sc = scenes.tiny_scene(xyz, h, eye=(0.9, 0.8, -0.7), target=(0.2, 0.2, 0.2), width=8 * tiles[0] - 3,
                           height=8 * tiles[1] - 5)
    sc.iso *= per_cell
    print(f"tile list and group finish, {tiles} tiles, {per_cell} per cell", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    for kw in (dict(normal_mode=0), dict(normal_mode=1), dict(normal_eps=0.03, final_fp64=0, bisect_iters=5),
               dict(normal_eps=-0.004, bisect_iters=0), dict(bisect_iters=1, compensated=1)):
        # the empty-cell skip counts every sample's whole stencil; the differences' box counts
        # are the oracle's where the offset is the scene's own
        keys = COUNTERS if "normal_mode" in kw and kw["normal_mode"] or "normal_eps" in kw else COUNTERS + ("cand",)
        got = _check(marcher, sc, counters=keys, skip_mode=1, **kw)
        assert got["hits"] > 100


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("away", ["none", "some", "all"])
def test_batch_tile_list(marcher, use_graph, away):
    """The batch's tile list: views of one pixel, one ragged tile and many tiles,
    views that look away from the particles, no active tile at all; each image
    equals the oracle's, run after run."""
    sc = scenes.lattice_cube(4, n_side=10, spacing=0.05, width=32, height=32)
    print(f"batch tile list graph {use_graph} away {away}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    st = sc.settings(skip_mode=4)
    G = O.Grid(sc.xyz, sc.h)
    cams = []
    for i, (w, h) in enumerate(((1, 1), (7, 5), (130, 67), (8, 8))):
        off = away == "all" or (away == "some" and i % 2 == 0)
        eye = np.array([0.5, 0.6, 2.2])
        cams.append(scenes.make_camera(eye, np.array([0.5, 0.6, 9.0]) if off else np.array([0.5, 0.5, 0.5]), w, h))
    marcher.batch_set(st, [(60, c.width, c.height, c.inv_pv, c.eye) for c in cams], use_graph=use_graph)
    ref = [O.march(G, O.make_settings(**st), c.inv_pv, c.eye, c.width, c.height) for c in cams]
    assert (sum(o[3]["hits"] for o in ref) > 0) == (away != "all")
    for _ in range(3):
        marcher.batch_run()
        marcher.wait()
        for v, o in enumerate(ref):
            for got, want in zip(marcher.batch_download(v), o[:3]):
                assert np.array_equal(got, want.reshape(got.shape)), v
        for k in ("rays", "hits", "samples", "march_samples"):
            assert marcher.stats()[k] == sum(o[3][k] for o in ref), k


@pytest.mark.parametrize("size", [(61, 43), (333, 207)])
@pytest.mark.parametrize("iso", [0.0, 1e-6, 0.004])
def test_finish_list_low_iso(marcher, size, iso):
    """Hits beside and on the edges of the padded particle box, whose segments'
    cells reach the grid's last rows: iso 0 (every ray that enters hits on the
    box) and a small part of the rest density, with few and many tiles, and as a
    batch."""
    sc = scenes.lattice_cube(3, n_side=9, spacing=0.05, width=size[0], height=size[1])
    sc.iso *= iso
    c = sc.cameras[0]
    print(f"finish list low iso {iso} {size}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    for normal_mode in (0, 1) if iso else (0,):       # (a box hit has no particle to take gradients from)
        got = _check(marcher, sc, skip_mode=0, normal_mode=normal_mode)
        assert got["hits"] > 100
    st = sc.settings(skip_mode=0)
    pos, nrm, t, _ = marcher.march(60, st, c.inv_pv, c.eye, c.width, c.height)
    marcher.batch_set(st, [(60, c.width, c.height, c.inv_pv, c.eye)])
    marcher.batch_run()
    marcher.wait()
    for got, want in zip(marcher.batch_download(0), (pos, nrm, t)):
        assert np.array_equal(got, want)


@pytest.mark.parametrize("size", [(61, 43), (333, 207)])
@pytest.mark.parametrize("eps", [float("nan"), 1e5])
def test_finish_offset_without_box(marcher, size, eps):
    """An offset that is not a number, or far beyond the grid, leaves the hits'
    points as they are: zero normals, as the one-ray-per-lane schedule's."""
    sc = scenes.lattice_cube(3, n_side=9, spacing=0.05, centre=(0, 0, 0), width=size[0], height=size[1])
    c = sc.cameras[0]
    print(f"finish offset {eps} {size}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    st = sc.settings(skip_mode=1, normal_eps=eps)
    got = marcher.march(60, st, c.inv_pv, c.eye, *size)
    plain = marcher.march(60, dict(st, schedule=1), c.inv_pv, c.eye, *size)
    assert got[3]["hits"] > 100 and got[3]["samples"] == plain[3]["samples"]
    for a, b in zip(got[:3], plain[:3]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("tiles", [(25, 31), (25, 33)])
@pytest.mark.parametrize("eps", [0.02, 0.03, 0.06])
def test_candidates_of_wide_offsets(marcher, tiles, eps):
    """The candidates counted for the central differences do not depend on which
    finish the image's size selects (775 and 825 tiles), also for boxes of seven
    rows and more."""
    sc = scenes.lattice_cube(3, n_side=9, spacing=0.05, width=8 * tiles[0], height=8 * tiles[1])
    sc.normal_eps = eps
    print(f"candidates of offset {eps}, {tiles} tiles", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    got = _check(marcher, sc, counters=COUNTERS + ("cand",), skip_mode=1)
    assert got["hits"] > 1000


@pytest.mark.parametrize("extra,dist,groups", [(0, 2.6, 1), (0, 1.5, 1), (0, 1.1, 0), (0, 0.7, 0), (40, 1.1, 1), (40, 0.7, 0)])
@pytest.mark.parametrize("learned", [0, 1])
def test_group_finish_by_hits(marcher, extra, dist, groups, learned):
    """The finish of a dense frame in an image of 4,800 tiles: four lanes per hit
    up to 81,920 (1 + (most / (8 mean))^2) hits, at most four times 81,920, most the
    fullest h/2 cell's particles (83,200 here, and 185,000 with `extra` in one cell),
    a lane per hit beyond, chosen on the device; images and counters are those of the
    one-ray-per-lane schedule."""
    from pmarch import train
    rng = np.random.default_rng(12)
    h = 0.1
    base = np.stack(np.meshgrid(*[np.arange(14)] * 3, indexing="ij"), -1).reshape(-1, 1, 3) * (h / 2)
    xyz = (base + rng.uniform(0, h / 2, (base.shape[0], 5, 3))).reshape(-1, 3)
    xyz = np.concatenate([xyz, h * (7 + rng.uniform(0.01, 0.49, (extra, 3)))]).astype(np.float32)
    mid = np.full(3, 0.35)
    d = np.array([0.7, 0.6, -0.4]) / np.linalg.norm([0.7, 0.6, -0.4])
    sc = scenes.tiny_scene(xyz, h, eye=mid + dist * d, target=mid, width=640, height=480)
    sc.iso *= 5
    c = sc.cameras[0]
    print(f"group finish by hits, {extra} in a cell, distance {dist} learned {learned}", flush=True)
    if learned:
        marcher.mlp_set(train.load()[0])
    marcher.set_frame(60, sc.xyz, sc.h)
    st = sc.settings(skip_mode=4)
    plain = marcher.march(60, dict(st, schedule=1), c.inv_pv, c.eye, c.width, c.height)
    for _ in range(2):
        got = marcher.march(60, dict(st, learned=learned), c.inv_pv, c.eye, c.width, c.height)
        for a, b in zip(got[:3], plain[:3]):
            assert np.array_equal(a, b)
        for k in ("rays", "rays_in_aabb", "hits") + (() if learned else ("samples", "march_samples")):
            assert got[3][k] == plain[3][k], k
        most = 185000 if extra else 83200
        assert (got[3]["hits"] < 0.97 * most if groups else got[3]["hits"] > 1.03 * most) and got[3]["hits"] > 15000


@pytest.mark.parametrize("size", [(4096, 4096), (4099, 4096), (4224, 4083)])
def test_tile_list_of_large_images(marcher, size):
    """4,096 masks of 64 tiles, from which on they are summed in a launch of their
    own, a few more, and 4,216 (not a multiple of 64): images and counters are
    those of the one-ray-per-lane schedule."""
    sc = scenes.lattice_cube(3, n_side=7, spacing=0.05, width=size[0], height=size[1])
    c = sc.cameras[0]
    print(f"tile list of {size}", flush=True)
    marcher.set_frame(60, sc.xyz, sc.h)
    st = sc.settings(skip_mode=4, bisect_iters=2)
    got = marcher.march(60, st, c.inv_pv, c.eye, *size)
    plain = marcher.march(60, dict(st, schedule=1), c.inv_pv, c.eye, *size)
    for a, b in zip(got[:3], plain[:3]):
        assert np.array_equal(a, b)
    for k in ("rays", "rays_in_aabb", "hits", "samples"):
        assert got[3][k] == plain[3][k], k
    assert got[3]["hits"] > 100000
