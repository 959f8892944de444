"""Batched views x frames in one persistent launch (plain and learned), with
and without hipGraph capture: every view equals the single-view march of the
same frame and camera and the oracle's march, bit for bit, and graph replays
equal the eager run."""
import numpy as np
import pytest

import oracle as O
import pmarch
from pmarch import scenes, train

pytestmark = pytest.mark.gpu


def _frames(marcher, base_id=60, n=3, with_xyz=False):
    sc = scenes.dam_break(7, nx=30, ny=60, nz=30)
    frames = scenes.displaced_frames(sc, n, seed=3, spacing=0.005)
    for i, xyz in enumerate(frames):
        marcher.set_frame(base_id + i, xyz, sc.h)
    ids = [base_id + i for i in range(n)]
    if with_xyz:
        return sc, ids, {base_id + i: xyz for i, xyz in enumerate(frames)}
    return sc, ids


def _views(sc, fids, n, seed):
    rng = np.random.default_rng(seed)
    cams = scenes.random_views(rng, (0.075, 0.15, 0.075), n, 40, 300, 30, 200, radius=(0.35, 0.6))
    return [(fids[i % len(fids)], c.width, c.height, c.inv_pv, c.eye) for i, c in enumerate(cams)]


def _check_views(marcher, sc, views, settings, frames=None):
    """Every view against the single-view march; with the frames' positions,
    also against the oracle's (plain) march of the same frame and camera."""
    keys = dict(O.Settings._fields_)
    osettings = O.make_settings(**{k: v for k, v in sc.settings().items() if k in keys})
    grids = {}
    for i, (f, W, H, ipv, eye) in enumerate(views):
        b = marcher.batch_download(i)
        s = marcher.march(f, settings, ipv, eye, W, H)
        for x, y in zip(b, s[:3]):
            assert np.array_equal(x, y), f"view {i} ({W}x{H}, frame {f}) differs"
        if frames is not None:
            if f not in grids:
                grids[f] = O.Grid(frames[f], sc.h)
            o = O.march(grids[f], osettings, ipv, eye, W, H)
            for x, y in zip(b, o[:3]):
                assert np.array_equal(x, y), f"view {i} ({W}x{H}, frame {f}) differs from the oracle"


@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_plain_matches_single_views(marcher, use_graph):
    sc, fids, xyz = _frames(marcher, with_xyz=True)
    views = _views(sc, fids, 12, seed=1)
    st = sc.settings(skip_mode=4)
    print(f"batch plain graph={use_graph} views={len(views)}", flush=True)
    marcher.batch_set(st, views, use_graph=use_graph)
    marcher.batch_run()
    marcher.wait()
    bs = marcher.stats()
    assert bs["rays"] == sum(W * H for _, W, H, _, _ in views)
    _check_views(marcher, sc, views, st, frames=xyz)


def test_batch_graph_replays_match_eager(marcher):
    sc, fids = _frames(marcher)
    views = _views(sc, fids, 8, seed=2)
    st = sc.settings(skip_mode=4)
    print("batch graph replays", flush=True)
    marcher.batch_set(st, views, use_graph=False)
    marcher.batch_run()
    marcher.wait()
    eager = [marcher.batch_download(i) for i in range(len(views))]
    eager_stats = marcher.stats()
    marcher.batch_set(st, views, use_graph=True)
    for rep in range(3):
        marcher.batch_run()
        marcher.wait()
        s = marcher.stats()
        for k in ("rays", "hits", "samples", "march_cand", "march_samples"):
            assert s[k] == eager_stats[k], (rep, k)
        for i in range(len(views)):
            for x, y in zip(marcher.batch_download(i), eager[i]):
                assert np.array_equal(x, y), f"replay {rep} view {i}"
        # eager work between replays on the same stream
        f, W, H, ipv, eye = views[rep]
        marcher.march(f, st, ipv, eye, W, H)


def test_batch_learned_matches_single_views(marcher):
    if not train.WEIGHTS.exists():
        pytest.skip("no trained network checkpoint")
    params, _ = train.load()
    marcher.mlp_set(params)
    sc, fids, xyz = _frames(marcher, with_xyz=True)
    views = _views(sc, fids, 10, seed=4)
    st = sc.settings(learned=1)
    print("batch learned", flush=True)
    marcher.batch_set(st, views, use_graph=True)
    marcher.batch_run()
    marcher.wait()
    assert marcher.stats()["mlp_evals"] > 0
    _check_views(marcher, sc, views, st, frames=xyz)


def test_batch_invalidated_by_frame_update(marcher):
    sc, fids = _frames(marcher, base_id=70, n=2)
    views = _views(sc, fids, 3, seed=5)
    marcher.batch_set(sc.settings(skip_mode=4), views, use_graph=True)
    marcher.set_frame(fids[0], sc.xyz, sc.h)
    with pytest.raises(pmarch.PmError):
        marcher.batch_run()


def test_batch_rejects_bad_views(marcher):
    sc, fids = _frames(marcher, base_id=72, n=1)
    with pytest.raises(pmarch.PmError):
        marcher.batch_set(sc.settings(), [(999, 64, 64, np.eye(4), np.zeros(3))])
    with pytest.raises(pmarch.PmError):
        marcher.batch_set(sc.settings(), [(fids[0], 0, 64, np.eye(4), np.zeros(3))])
    with pytest.raises(pmarch.PmError):
        marcher.batch_set(sc.settings(mode=1), [(fids[0], 64, 64, np.eye(4), np.zeros(3))])


def test_batch_download_into_pinned_memory():
    """Views into memory the caller pinned are copied there directly: no staging,
    so the shared copy's workers are not started; one pageable image among them
    is copied too."""
    import ctypes
    import os

    hip = ctypes.CDLL("libamdhip64.so")

    def pin(shape):
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * int(np.prod(shape))), 0) == 0
        return np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), shape)

    print("batch download into pinned memory", flush=True)
    m = pmarch.Marcher(0)
    sc = scenes.lattice_cube(4, n_side=10, spacing=0.05, width=640, height=480)
    c = sc.cameras[0]
    m.set_frame(0, sc.xyz, sc.h)
    st = sc.settings(skip_mode=4)
    m.batch_set(st, [(0, c.width, c.height, c.inv_pv, c.eye), (0, 16, 8, c.inv_pv, c.eye)])
    m.batch_run()
    m.wait()
    shapes = [(c.height, c.width, 4), (c.height, c.width, 4), (c.height, c.width)]
    pinned, other = [pin(s) for s in shapes], [pin(s) for s in shapes]
    small = [pin((8, 16, 4)), pin((8, 16, 4)), pin((8, 16))]
    assert m.L.pm_batch_download(m.ctx, 1, *(p.ctypes.data for p in small)) == 0
    before = len(os.listdir("/proc/self/task"))
    for _ in range(2):
        assert m.L.pm_batch_download(m.ctx, 0, *(p.ctypes.data for p in pinned)) == 0
    assert len(os.listdir("/proc/self/task")) == before
    plain = m.batch_download(0)
    other[1] = np.zeros(shapes[1], np.float32)
    assert m.L.pm_batch_download(m.ctx, 0, *(p.ctypes.data for p in other)) == 0
    for a, b, want in zip(pinned, other, plain):
        assert np.array_equal(a, want) and np.array_equal(b, want)
    assert (plain[0][..., 3] > 0).sum() > 1000
    for p in pinned + [other[0], other[2]] + small:
        assert hip.hipHostFree(ctypes.c_void_p(p.ctypes.data)) == 0
    m.close()


@pytest.mark.parametrize("dense", [(0, 1), (1, 1), (0, 0)])
@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_of_dense_frames(marcher, dense, use_graph):
    """A batch over sparse and dense frames (1 and 12 particles per h/2 cell): one
    dense frame among them and all hits walk for each sample, none and they share
    lists; each view equals the oracle's."""
    rng = np.random.default_rng(3)
    h = 0.1
    base = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 1, 3) * (h / 2)
    print(f"batch of dense frames {dense} graph {use_graph}", flush=True)
    views, want = [], []
    st = None
    for f, d in enumerate(dense):
        per = 12 if d else 1
        xyz = (base + rng.uniform(0, h / 2, (base.shape[0], per, 3))).reshape(-1, 3).astype(np.float32)
        sc = scenes.tiny_scene(xyz, h, eye=(0.9, 0.8, -0.7), target=(0.2, 0.2, 0.2), width=71, height=50)
        st = st or sc.settings(skip_mode=4)
        marcher.set_frame(60 + f, sc.xyz, sc.h)
        G, c = O.Grid(sc.xyz, sc.h), sc.cameras[0]
        views.append((60 + f, c.width, c.height, c.inv_pv, c.eye))
        want.append(O.march(G, O.make_settings(**st), c.inv_pv, c.eye, c.width, c.height))
    marcher.batch_set(st, views, use_graph=use_graph)
    for _ in range(3):
        marcher.batch_run()
        marcher.wait()
        for v, o in enumerate(want):
            for a, b in zip(marcher.batch_download(v), o[:3]):
                assert np.array_equal(a, b.reshape(a.shape)), v
        got = marcher.stats()
        for k in ("rays", "hits", "samples", "march_samples"):
            assert got[k] == sum(o[3][k] for o in want), k
    assert any(o[3]["hits"] > 200 for o in want)
