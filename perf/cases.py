"""The work that programs built on this framework have it do, as measurable cases.

A case is one call (or the calls that belong together) through the public
Python interface: whole frames, tiles of the offline engine, single rays of the
integrator, batches of jobs, the learned guide's evaluation and training
gradient, and frames that sample a frozen guide.  Scenes and sizes are those of
narvalengine_amd.configs and of the tests, or the same generators at other
sizes.  Every case is seeded: a scene's grid or mesh, its camera position and
the render's random streams come from the seed alone.

Online training inside a render is not a case of its own: its gradients are
summed by floating-point atomics, so two runs of the same render take different
paths.  Its expensive part is the `guide_grad` kind here.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from narvalengine_amd import abi, configs
from narvalengine_amd.engine import OfflineEngine, SceneSettings
from narvalengine_amd.runtime import Batch, Context, Guide
from narvalengine_amd.scene import Camera, Scene

_CTX = None


def _ctx() -> Context:
    """A program holds one context per device and renders everything on it."""
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
    return _CTX


# ---- cases --------------------------------------------------------------------------
def listed():
    return [
        # Integrator::Li as a program calls it for single rays (picking, light
        # probes): the smallest call, all latency.
        dict(name="li_pick", kind="li", scene="fbm", res=64, n=4, bounces=16),
        # Li for a probe grid: 256 camera rays x 256 estimates through a cloud.
        dict(name="li_probes", kind="li", scene="cloud", res=256, n=65536, bounces=64),
        # OfflineEngine.renderTile, the engine's unit of work: one of the 40 x 10
        # tiles of a 1280 x 720 frame of a volume (32 x 72 pixels).
        dict(name="tile_volume", kind="tile", scene="fbm", res=128, width=1280, height=720, spp=32, bounces=16),
        # An interactive look at a mesh scene: few samples, a small frame.
        dict(name="preview_mesh", kind="frame", scene="box", res=5, width=640, height=360, spp=4, bounces=8),
        # The volume128 workload: 512 x 512, 64 spp, 16 bounces.
        dict(name="volume128", kind="frame", scene="fbm", res=128, width=512, height=512, spp=64, bounces=16),
        # The cloud512 workload, the framework's headline frame (the largest):
        # 1920 x 1080, 256 spp, up to 128 bounces.
        dict(name="cloud512", kind="frame", scene="cloud", res=512, width=1920, height=1080, spp=256, bounces=128),
        # The surface1m workload (1.3 M triangles) at a quarter of its samples.
        dict(name="surface1m", kind="frame", scene="box", res=8, width=1024, height=1024, spp=64, bounces=8),
        # Surfaces and a grid volume in one scene, an odd frame size.
        dict(name="room_fog", kind="frame", scene="room", res=96, width=857, height=481, spp=32, bounces=12),
        # A batch of uneven jobs on the wavefront executor, read back linear.
        dict(name="batch8", kind="batch", jobs=8, table=3, spp=32, bounces=16, executor=abi.NE_BATCH_WAVEFRONT),
        # The converged-reference mode: FP64 paths, linear FP64 film.
        dict(name="reference64", kind="fp64", scene="fbm", res=64, width=160, height=120, spp=16, bounces=16),
        # A frame that samples a frozen guide's tabulated proposal.
        dict(name="guided_cloud", kind="guided", scene="cloud", res=256, width=960, height=540, spp=16, bounces=64,
             log2_table=14, cache_res=16),
        # The gradient of one default-size training batch.
        dict(name="guide_grad", kind="guide_grad", n=65536, log2_table=15),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: every kind alike often, sizes spread
    over their logarithm, none kept to round numbers."""
    kind = rng.choice(["li", "tile", "frame", "frame", "frame", "batch", "fp64", "guided", "guide_grad", "guide_eval"])
    if kind == "li":
        scene = rng.choice(["fbm", "cloud", "box"])
        res = _log(rng, 3, 7) if scene == "box" else _log(rng, 32, 256)
        return dict(kind=kind, scene=scene, res=res, n=_log(rng, 1, 262144), bounces=rng.randint(4, 64))
    if kind == "tile":
        scene = rng.choice(["fbm", "cloud", "box", "room"])
        res = rng.randint(3, 6) if scene == "box" else _log(rng, 32, 192)
        h = _log(rng, 240, 1080)
        return dict(kind=kind, scene=scene, res=res, width=int(h * rng.uniform(1.0, 1.8)), height=h,
                    spp=_log(rng, 4, 256), bounces=rng.randint(4, 64))
    if kind == "frame":
        scene = rng.choice(["fbm", "cloud", "box", "room", "envmap"])
        res = rng.randint(3, 8) if scene == "box" else _log(rng, 32, 256)
        h = _log(rng, 90, 1080)
        w = int(h * rng.uniform(0.8, 1.8))
        most = 6.0e7 if scene in ("box", "room", "envmap") else 2.0e8  # paths
        return dict(kind=kind, scene=scene, res=res, width=w, height=h,
                    spp=max(1, min(_log(rng, 1, 256), int(most / (w * h)))),
                    bounces=rng.randint(2, 128 if scene == "cloud" else 24))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 12), table=rng.randint(0, 1000), spp=_log(rng, 4, 64),
                    bounces=rng.randint(4, 32),
                    executor=rng.choice([abi.NE_BATCH_PERSISTENT, abi.NE_BATCH_WAVEFRONT]))
    if kind == "fp64":
        scene = rng.choice(["fbm", "cloud", "box"])
        res = rng.randint(3, 6) if scene == "box" else _log(rng, 32, 128)
        return dict(kind=kind, scene=scene, res=res, width=_log(rng, 48, 256), height=_log(rng, 48, 256), spp=_log(rng, 1, 64),
                    bounces=rng.randint(2, 24))
    if kind == "guided":
        h = _log(rng, 120, 720)
        return dict(kind=kind, scene="cloud", res=_log(rng, 48, 256), width=int(h * rng.uniform(1.0, 1.8)), height=h,
                    spp=_log(rng, 2, 64), bounces=rng.randint(4, 96), log2_table=rng.randint(12, 16),
                    cache_res=rng.choice([0, 8, 16, 24]))
    if kind == "guide_grad":
        return dict(kind=kind, n=_log(rng, 1000, 65536), log2_table=rng.randint(12, 17))
    return dict(kind="guide_eval", n=_log(rng, 16, 262144), log2_table=rng.randint(12, 19))


# ---- scenes -------------------------------------------------------------------------
def _scene(case, rng):
    """(scene, camera) of a case; the seed picks the grid or mesh and moves the camera."""
    kind, res = case["scene"], case["res"]
    gseed = int(rng.integers(1, 1 << 30))
    jit = rng.uniform(-0.08, 0.08, 3)
    aspect = case.get("width", 1) / case.get("height", 1)
    if kind == "fbm":
        s = configs.volume_scene(configs.fbm_grid.__wrapped__(res, gseed))
        cam = Camera(position=tuple(np.array([0.0, 0.25, -1.8]) + jit), look_at=(0, 0, 0), vfov=45.0, aspect=aspect)
    elif kind == "cloud":
        s = configs.cloud_scene(configs.cumulus_grid.__wrapped__(res, gseed), maj_res=16)
        cam = Camera(position=tuple(np.array([0.0, 0.05, -1.45]) + jit), look_at=(0, 0, 0), vfov=40.0, aspect=aspect)
    elif kind == "envmap":  # a volume over a floor under an importance-sampled map, as the tests light it
        s = Scene()
        s.set_volume(configs.fbm_grid.__wrapped__(res, gseed), 12.0, (0.95,) * 3, (0.05,) * 3, 0.7, maj_res=4)
        s.add_rectangle(s.add_glossy((0.6, 0.55, 0.5), 0.5), position=(0, -0.5, 0), rotation=(90, 0, 0),
                        scale=(6, 6, 1))
        m = rng.gamma(0.8, 0.3, (128, 256, 3)).astype(np.float32)
        m[24:36, 80:104] *= 60.0
        s.set_env_map(m)
        s.set_sun(-np.array([1.0, 2.0, -0.7]), (0.5, 0.5, 0.5))
        cam = Camera(position=tuple(np.array([0.0, 0.25, -1.8]) + jit), look_at=(0, 0, 0), vfov=45.0, aspect=aspect)
    else:  # "box": the surface1m box with an icosphere of `res` subdivisions; "room": with fog of `res` voxels an edge
        s = Scene()
        mats = [s.add_glossy(rng.uniform(0.1, 0.9, 3), float(rng.uniform(0.05, 0.8))) for _ in range(9)]
        s.add_rectangle(mats[0], position=(0, 0, 0), rotation=(90, 0, 0), scale=(2, 2, 1))
        s.add_rectangle(mats[1], position=(0, 2, 0), rotation=(-90, 0, 0), scale=(2, 2, 1))
        s.add_rectangle(mats[2], position=(0, 1, 1), rotation=(0, 0, 0), scale=(2, 2, 1))
        s.add_rectangle(mats[3], position=(-1, 1, 0), rotation=(0, 90, 0), scale=(2, 2, 1))
        s.add_rectangle(mats[4], position=(1, 1, 0), rotation=(0, -90, 0), scale=(2, 2, 1))
        s.add_rectangle(s.add_emitter((15.0, 15.0, 15.0)), position=(0, 1.98, 0.1), rotation=(-90, 0, 0),
                        scale=(0.6, 0.6, 1))
        s.add_sphere((-0.6, 0.3, -0.3), 0.3, mats[5])
        s.add_sphere((0.62, 0.35, -0.1), 0.35, mats[6])
        s.add_sphere((-0.15, 0.2, -0.75), 0.2, mats[7])
        sub = min(res, 8) if kind == "box" else 5
        v, t = configs.icosphere.__wrapped__(sub, gseed, 0.1)
        xf = np.eye(4)
        xf[:3, :3] *= 0.45
        xf[:3, 3] = (0.0, 0.55, 0.35)
        s.add_mesh(v, t, mats[8], xf)
        if kind == "room":
            s.set_volume(configs.fbm_grid.__wrapped__(res, gseed), 3.0, (0.9,) * 3, (0.1,) * 3, 0.6,
                         position=(0, 0.9, 0), scale=(1.8, 1.6, 1.8), maj_res=4)
            s.set_env(abi.NE_ENV_SKY, c0=(0.2, 0.3, 0.6), c1=(0.6, 0.6, 0.6), c2=(0.1, 0.1, 0.1))
        cam = Camera(position=tuple(np.array([0.0, 1.0, -3.2]) + jit), look_at=(0, 1, 0), vfov=40.0, aspect=aspect)
    return s, cam


def _rays(case, rng, cam):
    """Camera-like rays: from the camera position towards points of the unit cube around its target."""
    o = np.asarray(cam.position, np.float64)
    d = np.asarray(cam.look_at, np.float64) + rng.uniform(-0.45, 0.45, (case["n"], 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([np.broadcast_to(o, d.shape), d], 1).astype(np.float32)


# ---- the guide's inputs -------------------------------------------------------------
_IN, _OUT = (48, 64, 64, 64, 64), (64, 64, 64, 64, 48)


def _guide_params(log2_table, rng):
    """Parameters of a trained guide's size and spread (hash features of a few
    tenths, distinct lobes; padding rows and columns zero)."""
    table = rng.uniform(-0.3, 0.3, 16 * (1 << log2_table) * 2).astype(np.float32)
    w = []
    for l in range(5):
        m = rng.uniform(-1.0, 1.0, (_IN[l], _OUT[l])) * 0.7 * math.sqrt(6.0 / (35 if l == 0 else 64))
        if l == 0:
            m[35:] = 0.0
        if l == 4:
            m[:, 40:] = 0.0
        w.append(m.reshape(-1))
    b = [rng.uniform(0.0, 0.5, o) if l < 4 else rng.uniform(-1.5, 1.5, o) for l, o in enumerate(_OUT)]
    b[4][40:] = 0.0
    return table, np.concatenate(w + b).astype(np.float32)


def _guide_inputs(case, seed):
    """(table, mlp, samples): unit-cube positions, incoming directions, sampled
    directions about them or, for most, about one light, and positive weights of
    a long-tailed distribution."""
    rng = np.random.default_rng([seed, 77])
    table, mlp = _guide_params(case["log2_table"], rng)
    n = case["n"]
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    lit = rng.uniform(size=(n, 1)) < 0.7
    w = np.where(lit, np.array([0.5, 0.8, -0.3]) + 0.4 * rng.normal(size=(n, 3)), d + 0.5 * rng.normal(size=(n, 3)))
    w /= np.linalg.norm(w, axis=1, keepdims=True)
    r = rng.lognormal(-1.0, 1.0, (n, 1))
    return table, mlp, np.concatenate([rng.uniform(0.0, 1.0, (n, 3)), d, w, r], 1).astype(np.float32)


def _levels():
    growth = math.exp((math.log(512.0) - math.log(16.0)) / 15)
    return [int(math.floor(16.0 * growth ** l + 1e-6)) for l in range(16)]


# ---- prepare and run ----------------------------------------------------------------
def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    rng = np.random.default_rng([seed, 5])
    st = dict(kind=kind, ctx=ctx, seed=int(seed) & 0xFFFFFFFF, case=case)
    if kind in ("guide_grad", "guide_eval"):
        table, mlp, smp = _guide_inputs(case, seed)
        g = Guide(ctx, log2_table=case["log2_table"], batch=65536)
        g.set_params(table, mlp)
        st.update(guide=g, samples=smp, queries=np.ascontiguousarray(smp[:, :6]))
        return st
    if kind == "batch":
        pick = np.random.default_rng([case["table"], 48])
        jobs = []
        for j in range(case["jobs"]):
            res = [64, 96, 128][int(pick.integers(3))]
            w, h = [(256, 256), (512, 288), (333, 250)][int(pick.integers(3))]
            spp = max(1, case["spp"] // [1, 2, 4][int(pick.integers(3))])
            s, cam = _scene(dict(scene="fbm", res=res, width=w, height=h), rng)
            jobs.append(dict(scene=ctx.upload(s), camera=cam, width=w, height=h, spp=spp,
                             max_bounces=case["bounces"], seed=st["seed"], job=j))
        st.update(batch=Batch(ctx, jobs), cfg=(8, 8, 4, case["executor"]))
        return st
    s, cam = _scene(case, rng)
    if kind == "tile":
        eng = OfflineEngine(cam, SceneSettings((case["width"], case["height"]), case["spp"], case["bounces"]), s,
                            ctx=ctx, seed=st["seed"])
        st.update(engine=eng, camera=cam, index=int(rng.integers(4, 6)) * 40 + int(rng.integers(14, 26)))
        return st
    st.update(scene=ctx.upload(s), camera=cam)
    if kind == "li":
        st["rays"] = _rays(case, rng, cam)
        return st
    st["film"] = ctx.film(case["width"], case["height"])
    if kind == "guided":
        g = Guide(ctx, log2_table=case["log2_table"], cache_res=case["cache_res"])
        g.set_params(*_guide_params(case["log2_table"], rng))
        st["guide"] = g
    return st


def run(st):
    kind, c, ctx = st["kind"], st["case"], st["ctx"]
    if kind == "li":
        return ctx.li(st["scene"], st["rays"], c["bounces"], st["seed"])
    if kind == "tile":
        st["engine"].renderTile(st["camera"], st["index"])
        return st["engine"].pixels
    if kind == "frame" or kind == "guided":
        film = st["film"]
        film.clear()
        ctx.render(st["scene"], st["camera"], film, spp=c["spp"], max_bounces=c["bounces"], seed=st["seed"],
                   guide=st.get("guide"))
        return film.tonemap(c["spp"])
    if kind == "fp64":
        film = st["film"]
        film.clear()
        ctx.render(st["scene"], st["camera"], film, spp=c["spp"], max_bounces=c["bounces"], seed=st["seed"],
                   precision=abi.NE_FP64)
        return film.read()
    if kind == "batch":
        st["batch"].run(st["cfg"])
        return [st["batch"].read(k) for k in range(c["jobs"])]
    if kind == "guide_grad":
        loss = st["guide"].train_step(st["samples"], update=False)
        table_grad, mlp_grad = st["guide"].grads()
        return dict(loss=np.float32(loss), table_grad=table_grad, mlp_grad=mlp_grad)
    return st["guide"].eval(st["queries"])


# ---- what a pass cannot do without ----------------------------------------------------
def _scene_bytes(scene, res):
    if scene == "box":
        return 20 * 4 ** min(res, 8) * (48 + 20)  # triangles and their share of the nodes
    return 4 * res ** 3 + (20 * 4 ** 5 * 68 if scene == "room" else 0)


def work(case):
    """Bytes: the scene or the parameters read once, the outputs written once.
    Flops: for renders, the arithmetic of the mean number of path vertices of
    each scene (free flight, light sample, shadow ray, scattering: about 800
    operations a vertex in a volume, 1500 with a BVH in the way)."""
    kind = case["kind"]
    mlp = 2 * (35 * 64 + 3 * 64 * 64 + 64 * 40)
    if kind == "guide_eval":
        return dict(bytes=case["n"] * (24 + 160 + 512), flops=case["n"] * (mlp + 16 * 8 * 10))
    if kind == "guide_grad":
        return dict(bytes=case["n"] * (40 + 512) + 16 * (1 << case["log2_table"]) * 12,
                    flops=case["n"] * (3 * mlp + 2 * 16 * 8 * 10))
    per = dict(fbm=(1.5, 800), cloud=(1.3, 800), envmap=(2.5, 1500), box=(4.0, 1500), room=(4.0, 1500))
    if kind == "batch":
        pick = np.random.default_rng([case["table"], 48])
        nb = fl = 0.0
        for _ in range(case["jobs"]):
            res = [64, 96, 128][int(pick.integers(3))]
            w, h = [(256, 256), (512, 288), (333, 250)][int(pick.integers(3))]
            spp = max(1, case["spp"] // [1, 2, 4][int(pick.integers(3))])
            nb += 4 * res ** 3 + w * h * 24
            fl += w * h * spp * 1.5 * 800
        return dict(bytes=nb, flops=fl)
    v, f = per[case["scene"]]
    if kind == "li":
        return dict(bytes=min(_scene_bytes(case["scene"], case["res"]), case["n"] * 1024) + case["n"] * 36,
                    flops=case["n"] * v * f)
    px = case["width"] * case["height"]
    if kind == "tile":
        px = (case["width"] // 40) * (case["height"] // 10)
    paths = px * case["spp"]
    return dict(bytes=min(_scene_bytes(case["scene"], case["res"]), paths * 1024) + px * 12, flops=paths * v * f)


# ---- 64-bit values --------------------------------------------------------------------
def _encode64(p, table, log2_table):
    """Multiresolution hash encoding in FP64 (torch, so that gradients flow to the table)."""
    T = 1 << log2_table
    tab = table.reshape(16, T, 2)
    out = []
    for l, res in enumerate(_levels()):
        s = p * res
        f = torch.clamp(torch.floor(s), max=res - 1)
        t = s - f
        fi = f.to(torch.int64)
        e = 0
        for k in range(8):
            bit = torch.tensor([k & 1, (k >> 1) & 1, (k >> 2) & 1])
            x, y, z = (fi + bit).unbind(1)
            w = torch.where(bit == 1, t, 1.0 - t).prod(1)
            if (res + 1) ** 3 <= T:
                idx = x + (res + 1) * (y + (res + 1) * z)
            else:
                idx = (x ^ ((y * 2654435761) & 0xFFFFFFFF) ^ ((z * 805459861) & 0xFFFFFFFF)) & (T - 1)
            e = e + w[:, None] * tab[l, idx]
        out.append(e)
    return torch.cat(out, 1)


def _network64(q, table, mlp, log2_table):
    """Mixture parameters: weights (n, 8), unit means (n, 8, 3), kappa (n, 8)."""
    n = len(q)
    x = torch.cat([_encode64(q[:, :3].clamp(0.0, 1.0), table, log2_table), q[:, 3:6],
                   torch.zeros(n, 13, dtype=torch.float64)], 1)
    off, boff = 0, sum(i * o for i, o in zip(_IN, _OUT))
    for l in range(5):
        h = x @ mlp[off:off + _IN[l] * _OUT[l]].reshape(_IN[l], _OUT[l]) + mlp[boff:boff + _OUT[l]]
        x = torch.relu(h) if l < 4 else h
        off += _IN[l] * _OUT[l]
        boff += _OUT[l]
    y = x[:, :40].reshape(n, 8, 5)
    mean = y[:, :, 1:4]
    return (torch.softmax(y[:, :, 0], 1), mean / mean.norm(dim=2, keepdim=True).clamp_min(1e-12),
            torch.exp(y[:, :, 4].clamp(-10.0, 8.0)))


def exact(case, seed):
    """The guide's outputs in FP64.  Images and radiance are Monte Carlo
    estimates along the framework's own random streams: in other arithmetic a
    path takes other turns, so they have no such value."""
    if case["kind"] not in ("guide_grad", "guide_eval"):
        return None
    table, mlp, smp = (torch.from_numpy(a).to(torch.float64) for a in _guide_inputs(case, seed))
    if case["kind"] == "guide_eval":
        with torch.no_grad():
            pi, mu, kap = _network64(smp[:, :6], table, mlp, case["log2_table"])
            return torch.cat([pi[:, :, None], mu, kap[:, :, None]], 2).reshape(-1, 40)
    table.requires_grad_(True)
    mlp.requires_grad_(True)
    pi, mu, kap = _network64(smp[:, :6], table, mlp, case["log2_table"])
    c = (mu * smp[:, None, 6:9]).sum(2)
    vmf = kap / (2.0 * math.pi * -torch.expm1(-2.0 * kap)) * torch.exp(kap * (c - 1.0))
    loss = -(smp[:, 9] * torch.log((pi * vmf).sum(1))).sum() / smp[:, 9].sum()
    loss.backward()
    return dict(loss=loss.detach(), table_grad=table.grad, mlp_grad=mlp.grad)
