"""Performance cases of the particle-fluid ray marcher, through pmarch.Marcher.

Each case is one thing a program built on the library does over and over: march
a resident frame into its own images, run the reference renderer's passes, bring
in the next frame, smooth a depth image, replay a batch of views, take a
training step of the step-proposal network.  Sizes follow the workloads the
library is benchmarked on (pmarch.scenes); `draw` spreads over their ranges.
`exact` restates every result in 64 bits with plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "bachelor-thesis_amd"))
from pmarch import Marcher, scenes, train  # noqa: E402
from pmarch.camera import make_camera, orbit_eye  # noqa: E402

DEV = "cuda"


def _view(name, kind, scene, side, width, height, skip="bound", learned=False, aniso=False):
    d = dict(kind=kind, scene=scene, side=side, width=width, height=height, skip=skip, learned=learned,
             anisotropic=aniso)
    return dict(name=name, **d) if name else d


def listed():
    return [
        # a thumbnail / picking view of a small cloud: launches and latency
        _view("view_lattice10_96x64", "view", "lattice", 10, 96, 64),
        # the ordinary hand-off of the renderer: images into host memory
        _view("host_lattice32_640x480", "host", "lattice", 32, 640, 480),
        # the headline view: 1,024,000 particles at 1920x1080, device images
        _view("view_dam80_1920x1080", "view", "dam", 80, 1920, 1080),
        # the learned-step march, at an odd size
        _view("view_dam64_learned_1283x721", "view", "dam", 64, 1283, 721, learned=True),
        # the largest: 4,000,000 unevenly dense particles at 3840x2160
        _view("view_pool4M_3840x2160", "view", "pool", 4_000_000, 3840, 2160),
        # the reference renderer's passes on the GPU: depth sprites, then its march
        _view("reference_dam80_1920x1080", "reference", "dam", 80, 1920, 1080, skip="box"),
        # the same with the reference's default, the anisotropic kernel
        _view("reference_aniso_dam80_1920x1080", "reference", "dam", 80, 1920, 1080, skip="box", aniso=True),
        # the configured march with the anisotropic kernel
        _view("aniso_dam80_1920x1080", "view", "dam", 80, 1920, 1080, aniso=True),
        # autoplay: the next frame arrives from the host, is built and marched once
        _view("stream_dam80_1920x1080", "stream", "dam", 80, 1920, 1080),
        # screen-space smoothing of the sprite depths (N = 8 is the renderer's default)
        dict(name="smooth_1920x1080_n8", kind="smooth", width=1920, height=1080, taps=8),
        # a replayed batch of uneven views over two resident frames, images fetched
        dict(name="batch_dam40_2x4", kind="batch", side=40, frames=2, views=4),
        # one training step's gradient of the step-proposal network (batch of train.py)
        dict(name="step_grad_4096", kind="grad", rows=4096),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "host", "reference", "stream", "smooth", "batch", "grad"])
    w = _logint(rng, 64, 1920)
    h = max(33, min(1080, int(w * rng.uniform(0.45, 0.9))))
    if kind == "smooth":
        return dict(kind=kind, width=w, height=h, taps=rng.choice([8, 8, 3, 5, 12]))
    if kind == "batch":
        return dict(kind=kind, side=_logint(rng, 12, 40), frames=rng.randint(1, 3), views=rng.randint(2, 4))
    if kind == "grad":
        return dict(kind=kind, rows=64 * _logint(rng, 1, 1024))
    if kind == "reference":
        aniso = rng.random() < 0.3
        return _view(None, kind, "dam", _logint(rng, 16, 80), w, h, aniso=aniso,
                     skip=rng.choice(["box", "cons"] if aniso else ["box", "cons", "none"]))
    if kind == "stream":
        return _view(None, kind, "dam", _logint(rng, 16, 80), w, h)
    scene = rng.choice(["lattice", "dam", "dam", "pool"])
    side = {"lattice": lambda: _logint(rng, 8, 48), "dam": lambda: _logint(rng, 16, 80),
            "pool": lambda: _logint(rng, 30_000, 1_000_000)}[scene]()
    if kind == "view" and scene == "dam" and rng.random() < 0.3:
        return _view(None, kind, scene, side, w, h, aniso=True)
    return _view(None, kind, scene, side, w, h, skip=rng.choice(["bound", "bound", "bound", "empty", "none"]),
                 learned=rng.random() < 0.25)


# ------------------------------------------------------------------- inputs --

def _orbit(rng, target, radius, width, height):
    """A camera near the workload's own (30 degrees up, 45 degrees round), seeded."""
    eye = orbit_eye(target, radius * rng.uniform(0.95, 1.1), rng.uniform(25.0, 35.0), rng.uniform(30.0, 60.0))
    return make_camera(eye, target, width, height)


def _scene(case, seed):
    """(scene, camera): particles and a view of them."""
    rng = np.random.default_rng(1000 + seed)
    side, W, H = case["side"], case["width"], case["height"]
    if case["scene"] == "lattice":
        sc = scenes.lattice_cube(seed, n_side=side, spacing=1.6 / side)
        return sc, _orbit(rng, (0.5, 0.5, 0.5), 2.0, W, H)
    if case["scene"] == "pool":
        sc = scenes.clustered_pool(seed, n_total=side, r=0.003 * (4.0e6 / side) ** (1.0 / 3.0))
        return sc, _orbit(rng, (0.5, 0.3, 0.2), 1.7, W, H)
    sp = 0.4 / side
    kw = dict(nx=side, ny=2 * side, nz=side, spacing=sp, jitter_sigma=0.4 * sp)
    if case["anisotropic"]:        # the anisotropic kernel is tuned for h = 0.1
        k = 0.05 / sp
        sc = scenes.dam_break_aniso(seed, scale=k, **kw)
        return sc, _orbit(rng, tuple(k * c for c in scenes.COLUMN_CENTRE), 1.3 * k, W, H)
    return scenes.dam_break(seed, **kw), _orbit(rng, scenes.COLUMN_CENTRE, 1.3, W, H)


def _settings(case, sc):
    if case["kind"] == "reference":
        skip = {"none": 0, "box": 2, "cons": 3}[case["skip"]]
        st = dict(mode=1, max_steps=128, step=float(np.float32(0.009 * sc.h / 0.1)), normal_mode=1, skip_mode=skip,
                  compensated=0)
        if case["anisotropic"]:
            return dict(st, iso=1.0, **scenes.ANISO_SETTINGS)
        return dict(st, iso=sc.iso)
    skip = {"none": 0, "empty": 1, "bound": 4}[case["skip"]]
    if case["anisotropic"]:
        return scenes.aniso_settings(sc, skip_mode=skip)
    return sc.settings(skip_mode=skip, learned=int(case["learned"]), bound_boxes=int(case["kind"] == "stream"))


def _batch(case, seed):
    """(frames, h, settings, [(frame, camera)]): every view over every frame."""
    side, sp = case["side"], 0.4 / case["side"]
    sc = scenes.dam_break(seed, nx=side, ny=2 * side, nz=side, spacing=sp, jitter_sigma=0.4 * sp)
    frames = scenes.displaced_frames(sc, case["frames"], seed, spacing=sp)
    sizes, rng = np.random.default_rng(side), np.random.default_rng(2000 + seed)
    cams = []
    for _ in range(case["views"]):
        W, H = int(sizes.integers(128, 641)), int(sizes.integers(128, 361))
        cams += scenes.random_views(rng, scenes.COLUMN_CENTRE, 1, wmin=W, wmax=W, hmin=H, hmax=H)
    return frames, sc.h, sc.settings(skip_mode=4), [(f, c) for f in range(len(frames)) for c in cams]


def _depth_image(case, seed):
    """A sprite depth image: smooth rolling surface over part of the view, 1.0
    elsewhere, with sprite-sized bumps."""
    g = torch.Generator().manual_seed(seed)
    W, H = case["width"], case["height"]
    a, b, c = (torch.rand(3, generator=g) * 3.0).tolist()
    y, x = torch.meshgrid(torch.linspace(0, 1, H), torch.linspace(0, 1, W), indexing="ij")
    s = 0.93 + 0.02 * torch.sin(6 * x + a) * torch.cos(5 * y + b) + 0.002 * torch.rand(H, W, generator=g)
    return torch.where((x - 0.5) ** 2 + (y - 0.5) ** 2 + 0.02 * torch.sin(9 * x + c) < 0.16, s, torch.ones(())).float()


def _rows(case, seed):
    """(params, x, target): network rows spread as the trace logger's features."""
    rng = np.random.default_rng(3000 + seed)
    n = case["rows"]
    x = np.empty((n, 24), np.float32)
    x[:, :8] = rng.binomial(16, rng.uniform(0, 0.6, (n, 1)), (n, 8)) * 0.125
    x[:, 8:16] = rng.uniform(0, 2.0, (n, 8)) * (rng.random((n, 8)) < 0.6)
    d = rng.normal(size=(n, 3))
    x[:, 16:19] = d / np.linalg.norm(d, axis=1, keepdims=True)
    x[:, 19] = rng.uniform(0, 2.0, n)
    x[:, 20] = rng.uniform(0, 1.0, n) ** 3
    x[:, 21] = rng.uniform(0, 1.0, n) ** 2
    x[:, 22] = rng.uniform(0, 2.0, n)
    x[:, 23] = rng.uniform(0, 1.6, n)
    t = np.log2(1.0 + rng.exponential(6.0, n)).astype(np.float32)
    return train.he_init(seed), x, t


# ---------------------------------------------------------------- prepare/run --

def prepare(case, seed):
    kind = case["kind"]
    if kind == "smooth":
        img = _depth_image(case, seed).to(DEV)
        return dict(kind=kind, case=case, m=Marcher(0), depth=img, out=torch.zeros_like(img))
    if kind == "grad":
        p, x, t = _rows(case, seed)
        m = Marcher(0)
        m.mlp_set(p)
        return dict(kind=kind, m=m, x=x, t=t)
    if kind == "batch":
        frames, h, st, views = _batch(case, seed)
        m = Marcher(0)
        for f, xyz in enumerate(frames):
            m.set_frame(f, xyz, h)
        m.batch_set(st, [(f, c.width, c.height, c.inv_pv, c.eye) for f, c in views])
        return dict(kind=kind, m=m, views=len(views))
    sc, cam = _scene(case, seed)
    m = Marcher(0)
    if case["learned"]:
        m.mlp_set(train.load()[0])
    if kind != "stream":
        m.set_frame(0, sc.xyz, sc.h)
    s = dict(kind=kind, m=m, xyz=sc.xyz, h=sc.h, cam=cam, settings=_settings(case, sc))
    if kind != "host":
        W, H = cam.width, cam.height
        s.update(pos=torch.zeros(H, W, 4, device=DEV), nrm=torch.zeros(H, W, 4, device=DEV),
                 t=torch.zeros(H, W, device=DEV), depth=torch.zeros(H, W, device=DEV))
    return s


def run(state):
    kind, m = state["kind"], state["m"]
    if kind == "smooth":
        W, H = state["case"]["width"], state["case"]["height"]
        m.depth_smooth_device(state["depth"].data_ptr(), state["out"].data_ptr(), W, H, state["case"]["taps"],
                              stream=torch.cuda.current_stream().cuda_stream)
        return state["out"]
    if kind == "grad":
        loss, grad = m.mlp_grad(state["x"], state["t"], train.W_OVER)
        return {"loss": loss, "grad": grad}
    if kind == "batch":
        m.batch_run()
        m.wait()
        return [dict(zip(("positions", "normals", "t"), m.batch_download(v))) for v in range(state["views"])]
    cam = state["cam"]
    W, H = cam.width, cam.height
    if kind == "host":
        pos, nrm, t, _ = m.march(0, state["settings"], cam.inv_pv, cam.eye, W, H)
        return {"positions": pos, "normals": nrm, "t": t}
    pos, nrm, t, depth = state["pos"], state["nrm"], state["t"], state["depth"]
    if kind == "stream":
        m.set_frame(0, state["xyz"], state["h"])
    d_depth = 0
    if kind == "reference":
        d_depth = depth.data_ptr()
        m.depth_sprites_device(0, cam, state["h"], d_depth)
    m.march_device(0, state["settings"], cam.inv_pv, cam.eye, W, H, pos.data_ptr(), nrm.data_ptr(), t.data_ptr(),
                   d_depth=d_depth)
    out = {"positions": pos, "normals": nrm, "t": t}
    if kind == "reference":
        out["depth"] = depth
    return out


def work(case):
    """Inputs read once, outputs written once; per covered pixel the crossing
    sample, 8 bisection samples and 6 normal samples (reference mode: the sample
    and its gradient) of about 33 particles within h at 25 operations each (the
    anisotropic density: about 270 within 2h at 40)."""
    kind = case["kind"]
    if kind == "smooth":
        px = case["width"] * case["height"]
        return {"bytes": 8 * px, "flops": 2 * (2 * case["taps"] + 1) ** 2 * px}
    if kind == "grad":
        return {"bytes": 100 * case["rows"] + 8 * 6338, "flops": 6 * 5825 * case["rows"]}
    if kind == "batch":
        n, px = 2 * case["side"] ** 3, 384 * 244 * case["views"] * case["frames"]
        return {"bytes": 12 * n * case["frames"] + 36 * px, "flops": 0.1 * px * 15 * 33 * 25}
    n = {"lattice": case["side"] ** 3, "dam": 2 * case["side"] ** 3, "pool": case["side"]}[case["scene"]]
    px = case["width"] * case["height"]
    hits = px * {"lattice": 0.4, "dam": 0.12, "pool": 0.25}[case["scene"]]
    per = (270 * 40 if case["anisotropic"] else 33 * 25) * (2 if kind == "reference" else 15)
    sprites = kind == "reference"
    return {"bytes": 12 * n + (40 if sprites else 36) * px, "flops": hits * per + (60 * n if sprites else 0)}


# ------------------------------------------------------- the results in 64 bits --

class _Cloud:
    """Particles in cells of h (x fastest), on the GPU in 64 bits."""

    def __init__(self, xyz, h, s):
        self.h, self.s = float(np.float32(h)), s
        x = torch.from_numpy(np.ascontiguousarray(xyz, np.float32)).to(DEV).double()
        self.pmin, self.pmax = x.amin(0), x.amax(0)
        self.bmin, self.bmax = self.pmin - self.h, self.pmax + self.h
        self.lo = torch.floor(self.pmin / self.h).long() - 3
        self.n = torch.floor(self.pmax / self.h).long() - self.lo + 4
        c = self._lin(torch.floor(x / self.h).long() - self.lo)
        order = torch.argsort(c, stable=True)
        self.x = x[order]
        total = int(self.n.prod())
        self.start = torch.zeros(total + 1, dtype=torch.long, device=DEV)
        self.start[1:] = torch.cumsum(torch.bincount(c, minlength=total), 0)

    def _lin(self, k):
        return k[..., 0] + self.n[0] * (k[..., 1] + self.n[1] * k[..., 2])

    def _rows(self, q, R):
        """Per (dz, dy) row of the cells within R: (indices [nq, J], valid [nq, J])."""
        k = torch.floor(q / self.h).long() - self.lo
        inside = ((k >= R) & (k < self.n - R)).all(-1)
        k = torch.where(inside[:, None], k, torch.full_like(k, R))
        off = torch.zeros(3, dtype=torch.long, device=DEV)
        for dz in range(-R, R + 1):
            for dy in range(-R, R + 1):
                off[0], off[1], off[2] = -R, dy, dz
                b = self._lin(k + off)
                b, e = self.start[b], self.start[b + 2 * R + 1]
                e = torch.where(inside, e, b)
                J = int((e - b).amax()) if len(q) else 0
                if J == 0:
                    continue
                j = b[:, None] + torch.arange(J, device=DEV)
                yield torch.minimum(j, torch.full_like(j, len(self.x) - 1)), j < e[:, None]

    def _spline(self, q, sig):
        return torch.where(q >= 0.5, sig * 2 * (1 - q) ** 3, sig * (6 * (q ** 3 - q * q) + 1)).where(
            q < 1, torch.zeros((), dtype=torch.float64, device=DEV))

    def _slope(self, q, sig):
        return torch.where(q >= 0.5, -sig * 6 * (1 - q) ** 2, sig * 6 * (3 * q * q - 2 * q)).where(
            q < 1, torch.zeros((), dtype=torch.float64, device=DEV))

    def _G(self, q):
        """The clamped inverse covariance (h G), its determinant, and the neighbours' count."""
        s = self.s
        hx = float(np.float32(s["ext_mult"])) * self.h
        W = torch.zeros(len(q), dtype=torch.float64, device=DEV)
        N, S1, S2 = W.clone(), W.new_zeros(len(q), 3), W.new_zeros(len(q), 3, 3)
        for j, ok in self._rows(q, 2):
            r = self.x[j] - q[:, None]
            d = r.norm(dim=-1)
            ok = ok & (d < hx)
            w = torch.where(ok, 1 - (d / hx) ** 3, torch.zeros_like(d))
            W += w.sum(1)
            N += ok.sum(1)
            wr = w[..., None] * r
            S1 += wr.sum(1)
            S2 += (wr.unsqueeze(-1) * r.unsqueeze(-2)).sum(1)
        Wn = W.clamp_min(1e-300)[:, None]
        m = S1 / Wn
        C = S2 / Wn[..., None] - m[:, :, None] * m[:, None, :]
        V = torch.eye(3, dtype=torch.float64, device=DEV).expand(len(q), 3, 3).clone()
        for _ in range(8):                                   # cyclic Jacobi, batched
            for a, b in ((0, 1), (0, 2), (1, 2)):
                apq = C[:, a, b]
                small = apq.abs() < 1e-300
                th = (C[:, b, b] - C[:, a, a]) / (2 * torch.where(small, torch.ones_like(apq), apq))
                t = torch.where(th < 0, -1.0, 1.0) / (th.abs() + torch.sqrt(th * th + 1))
                t = torch.where(small, torch.zeros_like(t), t)
                c = 1 / torch.sqrt(t * t + 1)
                s_ = t * c
                J = torch.eye(3, dtype=torch.float64, device=DEV).repeat(len(q), 1, 1)
                J[:, a, a], J[:, b, b], J[:, a, b], J[:, b, a] = c, c, s_, -s_
                mul = lambda A, B: (A.unsqueeze(-1) * B.unsqueeze(-3)).sum(-2)  # noqa: E731
                C = mul(mul(J.transpose(1, 2).contiguous(), C), J)
                V = mul(V, J)
        lam = torch.diagonal(C, dim1=1, dim2=2)
        lam = torch.maximum(lam, lam.amax(1, keepdim=True) / s["k_r"]) * s["k_s"]
        lam = torch.where((N <= s["n_eps"])[:, None], torch.full_like(lam, s["k_n"]), lam).clamp_min(1e-300)
        G = ((V / lam[:, None, :]).unsqueeze(2) * V.unsqueeze(1)).sum(-1)
        return G / self.h, 1 / lam.prod(1) / self.h ** 3, N

    def field(self, q, grad=False):
        """rho at q [nq, 3], or the reference's sum of gradW (with its extra 1 / |r|)."""
        aniso = self.s.get("anisotropic", 0)
        out = torch.zeros(len(q), 3 if grad else 1, dtype=torch.float64, device=DEV)
        per = max(1024, int(2.0e7 / max(1, self.occupancy(5 if aniso else 3))))
        for i in range(0, len(q), per):
            p = q[i:i + per]
            G = det = None
            sig = 8 / math.pi / (1 if aniso else self.h ** 3)
            if aniso:
                G, det, N = self._G(p)
            for j, ok in self._rows(p, 1):
                r = self.x[j] - p[:, None]
                ok = ok & ((r * r).sum(-1) < self.h ** 2)
                if aniso:
                    r = (G[:, None] * r.unsqueeze(-2)).sum(-1)
                d = r.norm(dim=-1)
                u = d / self.h
                if grad:
                    g = self._slope(u, sig) / (d * d * self.h)
                    g = torch.where(ok & (u < 1), g, torch.zeros_like(g))
                    out[i:i + per] += (g[..., None] * torch.where(ok[..., None], r, torch.zeros_like(r))).sum(1) * (
                        det[:, None] if aniso else 1)
                else:
                    w = torch.where(ok, self._spline(u, sig), torch.zeros_like(u)).sum(1)
                    out[i:i + per, 0] += w * (det if aniso else 1)
        return out if grad else out[:, 0]

    def occupancy(self, cells):
        """Most particles in `cells` consecutive cells of a row."""
        if not hasattr(self, "_occ"):
            self._occ = {}
        if cells not in self._occ:
            self._occ[cells] = int((self.start[cells:] - self.start[:-cells]).amax())
        return self._occ[cells]


def _rays(cam, z=None):
    """(eye, directions [H W, 3], points at depth z): pixel-corner rays."""
    W, H = cam.width, cam.height
    M = torch.from_numpy(cam.inv_pv.astype(np.float64)).to(DEV).reshape(4, 4)       # [col][row]
    eye = torch.from_numpy(cam.eye.astype(np.float64)).to(DEV)
    y, x = torch.meshgrid(torch.arange(H, device=DEV).double(), torch.arange(W, device=DEV).double(), indexing="ij")
    cx, cy = (x * 2 / W - 1).reshape(-1), (y * 2 / H - 1).reshape(-1)
    zz = torch.ones_like(cx) if z is None else z.reshape(-1)
    w = cx[:, None] * M[0] + cy[:, None] * M[1] + zz[:, None] * M[2] + M[3]
    p = w[:, :3] / w[:, 3:]
    d = p - eye
    return eye, d / d.norm(dim=1, keepdim=True), p


def _images(cam, hit, x, n, t):
    """Whole images from the hits' values."""
    H, W = cam.height, cam.width
    pos = torch.zeros(H * W, 4, dtype=torch.float64, device=DEV)
    nrm, tt = pos.clone(), torch.full((H * W,), -1.0, dtype=torch.float64, device=DEV)
    pos[hit, :3], pos[hit, 3], nrm[hit, :3], nrm[hit, 3], tt[hit] = x, 1.0, n, 1.0, t
    return {"positions": pos.reshape(H, W, 4), "normals": nrm.reshape(H, W, 4), "t": tt.reshape(H, W)}


def _march64(cloud, cam, s):
    """The configured march: AABB entry, fixed step, first sample at or above
    iso, 8 bisections, central differences."""
    eye, d, _ = _rays(cam)
    step, iso, eps = (float(np.float32(s[k])) for k in ("step", "iso", "normal_eps"))
    t0, t1 = (cloud.bmin - eye) / d, (cloud.bmax - eye) / d
    tn, tf = torch.minimum(t0, t1).amax(1).clamp_min(0), torch.maximum(t0, t1).amin(1)
    ray = torch.nonzero(tn <= tf).reshape(-1)
    k_hit = torch.full((len(d),), -1, dtype=torch.long, device=DEV)
    k = 0
    while len(ray):
        t = tn[ray] + k * step
        ray, t = ray[t <= tf[ray]], t[t <= tf[ray]]
        above = cloud.field(eye + t[:, None] * d[ray]) >= iso
        k_hit[ray[above]] = k
        ray = ray[~above]
        k += 1
    hit = torch.nonzero(k_hit >= 0).reshape(-1)
    dh, kh = d[hit], k_hit[hit].double()
    hi = tn[hit] + kh * step
    lo = torch.where(kh > 0, hi - step, hi)
    for _ in range(s["bisect_iters"]):
        mid = (lo + hi) / 2
        above = cloud.field(eye + mid[:, None] * dh) >= iso
        lo, hi = torch.where(above, lo, mid), torch.where(above, mid, hi)
    t = torch.where(kh > 0, (lo + hi) / 2, hi)
    x = eye + t[:, None] * dh
    g = torch.zeros_like(x)
    for a in range(3):
        e = torch.zeros(3, dtype=torch.float64, device=DEV)
        e[a] = eps
        g[:, a] = cloud.field(x - e) - cloud.field(x + e)
    return _images(cam, hit, x, g / g.norm(dim=1, keepdim=True).clamp_min(1e-300), t)


def _sprites64(cloud, cam):
    """The depth-sprite image: the least fragment depth of every pixel."""
    W, H, R = cam.width, cam.height, cloud.h
    M, V, P = (torch.from_numpy(a.astype(np.float64)).to(DEV).reshape(4, 4).T.contiguous()
               for a in (cam.inv_pv, cam.view, cam.proj))
    eye = torch.from_numpy(cam.eye.astype(np.float64)).to(DEV)
    depth = torch.ones(H * W, dtype=torch.float64, device=DEV)
    PV = P @ V
    one = lambda p: torch.cat([p, torch.ones_like(p[..., :1])], -1)  # noqa: E731
    mul = lambda A, p: (A * p.unsqueeze(-2)).sum(-1)  # noqa: E731
    ax, ay = V[0, :3], V[1, :3]
    corner = [mul(PV, one(cloud.x + R * (sx * ax + sy * ay))) for sx in (-1, 1) for sy in (-1, 1)]
    c = torch.stack([v[:, :2] / v[:, 3:] for v in corner])
    f = (c + 1) * 0.5 * torch.tensor([W, H], device=DEV)
    lo = torch.ceil(f.amin(0) - 0.5).clamp_min(0)
    hi = torch.minimum(torch.floor(f.amax(0) - 0.5), torch.tensor([W - 1.0, H - 1.0], dtype=torch.float64, device=DEV))
    ok = (torch.stack([v[:, 3] for v in corner]) > 0).all(0) & (lo <= hi).all(1)
    x, lo, hi = cloud.x[ok], lo[ok].long(), hi[ok].long()
    if not len(x):
        return depth.reshape(H, W)
    bw, bh = ((hi - lo).amax(0) + 1).tolist()
    off = torch.stack(torch.meshgrid(torch.arange(bw, device=DEV), torch.arange(bh, device=DEV), indexing="xy"),
                      -1).reshape(-1, 2)
    per = max(1, 4_000_000 // len(off))
    n = torch.linalg.cross(ax, ay)
    for i in range(0, len(x), per):
        q, px = x[i:i + per, None], lo[i:i + per, None] + off
        ok = (px <= hi[i:i + per, None]).all(-1)
        ndc = (px + 0.5) * torch.tensor([2.0 / W, 2.0 / H], dtype=torch.float64, device=DEV) - 1
        w = mul(M, torch.cat([ndc, torch.ones_like(ndc[..., :1]), torch.ones_like(ndc[..., :1])], -1))
        d = w[..., :3] - eye * w[..., 3:]
        X = eye + (((q - eye) * n).sum(-1) / (d * n).sum(-1))[..., None] * d
        r = X - q
        l2 = ((r * ax).sum(-1) / R) ** 2 + ((r * ay).sum(-1) / R) ** 2
        v = mul(V, one(X))
        cp = mul(P, v)
        zp = cp[..., 2] / cp[..., 3]
        v[..., 2] -= R * torch.cos(math.pi / 2 * l2.clamp(0, 1).sqrt())
        cp = mul(P, v)
        z = (cp[..., 2] / cp[..., 3]).clamp(0, 1)
        ok &= (l2 <= 1) & (zp >= 0) & (zp <= 1)
        depth.scatter_reduce_(0, (px[..., 1] * W + px[..., 0])[ok], z[ok], "amin")
    return depth.reshape(H, W)


def _reference64(cloud, cam, s):
    """Depth sprites, then the march from them: MaxSteps samples, the
    DensityGrid's cleared nodes skipped, normalize(sum gradW)."""
    depth = _sprites64(cloud, cam)
    eye, d, p = _rays(cam, depth)
    step, iso = float(np.float32(s["step"])), float(np.float32(s["iso"]))
    ray = torch.nonzero(depth.reshape(-1) != 1).reshape(-1)
    dims = torch.ceil((cloud.bmax - cloud.bmin) / cloud.h).long()
    flag = torch.zeros(tuple(dims.tolist()), dtype=torch.bool, device=DEV)
    u, R = (cloud.x - cloud.bmin) / cloud.h, 1.5 if s["skip_mode"] == 3 else 1.0
    for i in range(27):                                       # nodes whose centre is nearer than R cells
        k = torch.floor(u).long() + torch.tensor([i % 3 - 1, i // 3 % 3 - 1, i // 9 - 1], device=DEV)
        ok = ((u - (k + 0.5)).abs() < R).all(1) & (k >= 0).all(1) & (k < dims).all(1)
        flag[tuple(k[ok].T)] = True
    point = {}
    for _ in range(s["max_steps"]):
        if not len(ray):
            break
        st = step * d[ray]
        p[ray] += st
        q = p[ray]
        todo = torch.arange(len(ray), device=DEV) if s["skip_mode"] else ray[:0]
        while len(todo):
            k = torch.floor((q[todo] - cloud.bmin) / cloud.h).long()
            ok = (k >= 0).all(1) & (k < dims).all(1)
            todo, k = todo[ok], k[ok]
            ok = ~flag[tuple(k.T)]
            todo, k = todo[ok], k[ok]
            lo = cloud.bmin + k * cloud.h
            ta, tb = (lo - q[todo]) / st[todo], (lo + cloud.h - q[todo]) / st[todo]
            tn, tf = torch.minimum(ta, tb).amax(1), torch.maximum(ta, tb).amin(1)
            t = torch.where(tn < tf, tf, tn)
            q[todo] += st[todo] * (torch.where(t >= 0, t, torch.zeros_like(t)) + 1)[:, None]
        p[ray] = q
        above = cloud.field(q) >= iso
        point[len(point)] = ray[above]
        ray = ray[~above]
    hit = torch.cat(list(point.values())) if point else ray[:0]
    x = p[hit]
    g = cloud.field(x, grad=True)
    img = _images(cam, hit, x, g / g.norm(dim=1, keepdim=True), (x - eye).norm(dim=1))
    return dict(img, depth=depth)


def _grad64(p, x, t):
    P = torch.from_numpy(p).double().requires_grad_(True)
    W1, b1, W2, b2, w3, b3 = torch.split(P, [2048, 64, 4096, 64, 64, 1])
    act = lambda z: z * torch.sigmoid(1.702 * z)  # noqa: E731
    h = act(torch.from_numpy(x).double() @ W1.reshape(64, 32)[:, :24].T + b1)
    y = act(h @ W2.reshape(64, 64).T + b2) @ w3 + b3
    d = y - torch.from_numpy(t).double()
    loss = (torch.where(d > 0, train.W_OVER, 1.0) * d * d).mean()
    loss.backward()
    return {"loss": loss.item(), "grad": P.grad.numpy()}


def _smooth64(img, N):
    i = torch.arange(-N, N + 1, dtype=torch.float64)
    k = torch.exp(-0.5 * i * i)
    k = k / k.sum()
    p = torch.nn.functional.pad(img.double()[None, None], (N, N, N, N), mode="replicate")[0, 0].to(DEV)
    H, W = img.shape
    p = sum(k[a].item() * p[a:a + H] for a in range(2 * N + 1))
    return sum(k[a].item() * p[:, a:a + W] for a in range(2 * N + 1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "smooth":
        return _smooth64(_depth_image(case, seed), case["taps"])
    if kind == "grad":
        return _grad64(*_rows(case, seed))
    if kind == "batch":
        frames, h, st, views = _batch(case, seed)
        clouds = [_Cloud(xyz, h, st) for xyz in frames]
        return [_march64(clouds[f], c, st) for f, c in views]
    if case["scene"] == "pool" and case["side"] * case["width"] * case["height"] > 1.0e11:
        return None                                           # dense clusters: minutes in plain torch
    sc, cam = _scene(case, seed)
    s = _settings(case, sc)
    cloud = _Cloud(sc.xyz, sc.h, s)
    return _reference64(cloud, cam, s) if kind == "reference" else _march64(cloud, cam, s)
