"""Workloads of the renderer, each one pass through its public entry points.

  rays     Context.trace on host rays: picking, probes, bakers
  device   yn_trace_noalloc on device rays: tracing inside a caller's own loop
  frame    Context.pathtracer: one frame of a progressive view on device
           images, as an interactive front end calls it
  render   Job.render of several frames, then Job.read: a finished image
  serve    Context.submit / serve: several jobs sharing the wavefront
  tonemap  Context.tonemap on a device image

Scenes are the repository's procedural ones (the Cornell box and icosphere
rooms); cameras, rays, images and frame seeds come from the seed.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
import random

import numpy as np
import torch

import yune_amd as Y

SCENE_SEED = 2024           # the rooms' geometry, as the benchmark's large scene
RAY_LEN = 100.0             # longer than any room: a ray without a hit ends here


def listed():
    return [
        # picking under a cursor, autofocus, a few probes: a call's latency
        dict(name="pick", call="rays", scene="room", spheres=8, subdiv=5, n=200, shadow=False),
        # a baker's batch of hemisphere rays from random points (odd count)
        dict(name="rays_1m", call="rays", scene="room", spheres=24, subdiv=4, n=1_000_003, shadow=False),
        # visibility between point pairs: ambient occlusion, light-map shadows
        dict(name="visibility", call="rays", scene="room", spheres=24, subdiv=4, n=150_001, shadow=True),
        # closest hits inside a caller's GPU loop: rays and results stay in device memory
        dict(name="device_rays", call="device", scene="room", spheres=8, subdiv=4, n=200_003),
        # an editor's material thumbnail, the kernels' shipped parameters
        dict(name="thumb", call="frame", scene="cornell", w=97, h=61, mode=0, mis=0, depth=0, on=0),
        # one frame of an interactive view of a mid-size scene
        dict(name="frame_720p", call="frame", scene="room", spheres=48, subdiv=4, w=1280, h=720, mode=0, mis=1,
             depth=8, on=0),
        # the Cornell box at ordinary quality
        dict(name="cornell_512", call="render", scene="cornell", w=512, h=512, frames=64, mode=0, mis=1, depth=8,
             on=1, overlap=0),
        # final-quality frames of a large scene, the largest work
        dict(name="room_1m", call="render", scene="room", spheres=48, subdiv=5, w=1920, h=1080, frames=32, mode=0,
             mis=1, depth=8, on=0, overlap=1),
        # interactive bidirectional preview
        dict(name="bdpt_frame", call="frame", scene="cornell", w=640, h=360, mode=1, mis=1, depth=5, on=0),
        # bidirectional image at ordinary quality
        dict(name="bdpt_720p", call="render", scene="cornell", w=1280, h=720, frames=8, mode=1, mis=1, depth=5,
             on=0, overlap=0),
        # a render service's queue: jobs of several sizes and scenes at once
        dict(name="serve", call="serve", jobs=12, spheres=12, subdiv=4, most_px=512, most_spp=48),
        # the display pass of a full-HD view
        dict(name="tonemap", call="tonemap", w=1920, h=1080, op=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _room(rng, most):
    """A scene of up to about `most` triangles."""
    if rng.random() < 0.25:
        return dict(scene="cornell")
    subdiv = rng.choice((3, 4, 5))
    return dict(scene="room", spheres=_log(rng, 1, max(1, min(48, most // (20 * 4 ** subdiv)))), subdiv=subdiv)


def draw(rng):
    call = rng.choice(("rays", "rays", "device", "frame", "frame", "render", "bdpt", "serve", "tonemap"))
    if call == "rays":
        return dict(call="rays", n=_log(rng, 64, 1_000_000), shadow=rng.random() < 0.4, **_room(rng, 200_000))
    if call == "device":
        return dict(call="device", n=_log(rng, 64, 262_144), **_room(rng, 200_000))
    if call == "tonemap":
        return dict(call="tonemap", w=_log(rng, 64, 3840), h=_log(rng, 48, 2160), op=rng.choice((0, 1)))
    if call == "serve":
        return dict(call="serve", jobs=rng.randint(2, 12), spheres=_log(rng, 1, 16), subdiv=rng.choice((3, 4)),
                    most_px=rng.choice((128, 256, 512)), most_spp=_log(rng, 8, 48))
    if call == "bdpt":
        c = dict(mode=1, mis=rng.choice((0, 1)), depth=rng.choice((3, 5)), on=0, **_room(rng, 20_000))
        if rng.random() < 0.5:
            return dict(call="frame", w=_log(rng, 64, 1280), h=_log(rng, 48, 720), **c)
        return dict(call="render", w=_log(rng, 64, 640), h=_log(rng, 48, 480), frames=_log(rng, 2, 16), overlap=0, **c)
    mis = rng.choice((0, 1, 1))
    c = dict(mode=0, mis=mis, depth=rng.choice((0, 2, 5, 8)), on=rng.choice((0, 1)), **_room(rng, 250_000))
    if call == "frame":
        return dict(call="frame", w=_log(rng, 64, 1920), h=_log(rng, 48, 1080), **c)
    return dict(call="render", w=_log(rng, 64, 1024), h=_log(rng, 48, 768), frames=_log(rng, 2, 64),
                overlap=rng.choice((0, 0, 1)), **c)


# ------------------------------------------------------------------ inputs

@functools.lru_cache(maxsize=8)
def _scene(scene, spheres=0, subdiv=0):
    """The geometry a program has loaded, with the reference's BVH."""
    s = Y.gen_cornell() if scene == "cornell" else Y.gen_icosphere_room(SCENE_SEED, spheres, subdiv)
    s.bvh()
    return s


@functools.lru_cache(maxsize=None)
def _context(overlap=0, graph=0):
    """A program has one context for all it does."""
    return Y.Context(trace_overlap=overlap, graph=graph)


def _case_scene(case):
    return _scene(case["scene"], case.get("spheres", 0), case.get("subdiv", 0))


def _params(mode, mis, depth, on):
    if mode == 1:
        return Y.params_reference(1, mis=mis, bdpt_bounces=depth)
    if depth == 0:          # the shipped kernel: no bounce limit, roulette after bounce 6
        return Y.params_reference(0, mis=mis, oren_nayar=on)
    return Y.params_reference(0, mis=mis, max_bounces=depth, rr_threshold=2, oren_nayar=on)


def _camera(rng, scene, s):
    """A viewer somewhere inside a room; the Cornell box keeps its own view."""
    if scene == "cornell":
        return s.cam
    eye = rng.uniform(-4, 4, 3)
    look = rng.uniform(-4, 4, 3) - eye
    look /= np.linalg.norm(look)
    side = np.cross(look, (0.0, 1.0, 0.0))
    side /= np.linalg.norm(side)
    return Y.camera(side, np.cross(side, look), look, eye, 60.0)


def _rays(case, seed):
    """Rays from random points in the scene's box, in random directions;
    shadow rays run to another random point."""
    s = _case_scene(case)
    rng = np.random.default_rng(seed)
    v = s.tris["v1"][:, :3]
    lo, hi = v.min(0), v.max(0)
    n = case["n"]
    r = np.zeros((n, 8), np.float32)
    r[:, :3] = rng.uniform(lo, hi, (n, 3))
    if case.get("shadow"):
        d = rng.uniform(lo, hi, (n, 3)) - r[:, :3]
        length = np.linalg.norm(d, axis=1)
        r[:, 3] = length
        r[:, 7] = 1.0
    else:
        d = rng.normal(size=(n, 3))
        length = np.linalg.norm(d, axis=1)
        r[:, 3] = RAY_LEN
    r[:, 4:7] = d / length[:, None]
    return s, r


class State:
    """What a program holds between calls; gives it back when dropped."""

    def __init__(self, case, ctx):
        self.case, self.ctx, self.sids, self.job = case, ctx, [], None

    def __del__(self):
        if self.job is not None:
            self.job.release()
        for sid in self.sids:
            self.ctx.release_scene(sid)


def prepare(case, seed):
    call = case["call"]
    st = State(case, _context(case.get("overlap", 0), 1 if call == "serve" else 0))
    ctx = st.ctx
    if call == "tonemap":
        g = torch.Generator(device="cuda").manual_seed(seed)
        img = torch.exp(torch.randn((case["h"], case["w"], 4), generator=g, device="cuda") - 1.0)
        img[..., 3] = 64.0                              # frames accumulated
        st.img, st.out = img, torch.empty_like(img)
        return st
    if call == "serve":
        rng = np.random.default_rng(seed)
        scenes = [_scene("cornell"), _scene("room", case["spheres"], case["subdiv"]), _scene("room", 2, 3)]
        st.sids = [ctx.scene(s) for s in scenes]
        st.jobs = []
        mix = random.Random(case["jobs"])                # sizes and scenes of the queue's jobs
        for _ in range(case["jobs"]):
            k = mix.randrange(3)
            px = mix.choice([p for p in (96, 128, 256, 512) if p <= case["most_px"]])
            spp = _log(mix, 4, case["most_spp"])
            st.jobs.append((st.sids[k], _camera(rng, "cornell" if k == 0 else "room", scenes[k]), px, px,
                            _params(0, 1, 8, 0), spp, int(rng.integers(1, 1 << 30))))
        return st
    if call in ("rays", "device"):
        s, st.rays = _rays(case, seed)
        st.sids = [ctx.scene(s)]
        if call == "device":
            n = case["n"]
            st.rays = torch.from_numpy(st.rays).cuda()
            st.tri = torch.empty(n, dtype=torch.int32, device="cuda")
            st.light = torch.empty(n, dtype=torch.int32, device="cuda")
            st.t = torch.empty(n, dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
        return st
    s = _case_scene(case)
    st.sids = [ctx.scene(s)]
    rng = np.random.default_rng(seed)
    st.cam = _camera(rng, case["scene"], s)
    st.params = _params(case["mode"], case["mis"], case["depth"], case["on"])
    if call == "render":
        st.job = ctx.job(st.sids[0], st.cam, case["w"], case["h"], st.params, base_seed=int(rng.integers(1, 1 << 30)))
    else:
        st.rand = random.Random(seed)
        st.frame = 0
        st.img = [torch.zeros((case["h"], case["w"], 4), device="cuda") for _ in range(2)]
    return st


def run(st):
    case, ctx = st.case, st.ctx
    call = case["call"]
    if call == "rays":
        tri, light, t = ctx.trace(st.sids[0], st.rays)
        if case["shadow"]:
            # which occluder a shadow ray meets is left open; that it meets one, or the light, is not
            return {"blocked": (tri >= 0).astype(np.uint8), "light": light}
        return {"tri": tri, "light": light, "t": t}
    if call == "device":
        Y.check(Y.lib().yn_trace_noalloc(
            ctx._p, st.sids[0], C.c_void_p(st.rays.data_ptr()), case["n"], C.c_void_p(st.tri.data_ptr()),
            C.c_void_p(st.light.data_ptr()), C.c_void_p(st.t.data_ptr())), ctx._p)
        return {"tri": st.tri, "light": st.light, "t": st.t}
    if call == "frame":
        out, prev = st.img[st.frame & 1], st.img[1 - (st.frame & 1)]
        ctx.pathtracer(out, prev, st.cam, st.sids[0], case["w"], case["h"], st.params, 1, 1 if st.frame == 0 else 0,
                       st.rand.getrandbits(32))
        st.frame += 1
        return out
    if call == "render":
        st.job.render(case["frames"])
        return st.job.read()
    if call == "serve":
        jobs = [ctx.submit(sid, cam, w, h, p, spp, seed) for sid, cam, w, h, p, spp, seed in st.jobs]
        while ctx.serve(16):
            pass
        imgs = [j.read() for j in jobs]
        for j in jobs:
            j.release()
        return imgs
    ctx.tonemap(st.out, st.img, case["w"], case["h"], case["op"])
    return st.out


# -------------------------------------------------------------------- work

def _tris(case):
    return 36 if case.get("scene") == "cornell" else case["spheres"] * 20 * 4 ** case["subdiv"] + 14


def _ray_flops(n_tri):
    """A ray through a good tree of n_tri triangles: about log2(n) nodes of
    four boxes (an FMA per plane and the min / max of each) and a few
    triangle tests."""
    return 0.85 * math.log2(n_tri) * 4 * 24 + 5 * 50


def work(case):
    call = case["call"]
    if call == "tonemap":
        px = case["w"] * case["h"]
        return {"bytes": 32.0 * px, "flops": 4 * 60.0 * px}
    if call in ("rays", "device"):
        n = _tris(case)
        # 32 B in and 12 B out per ray; the tree and triangles that n rays can touch, at most once each
        return {"bytes": 44.0 * case["n"] + min(160.0 * n, 2500.0 * case["n"]), "flops": case["n"] * _ray_flops(n)}
    if call == "serve":
        px = case["jobs"] * (0.4 * case["most_px"]) ** 2
        spp = 0.4 * case["most_spp"]
        n = case["spheres"] * 20 * 4 ** case["subdiv"]
        return {"bytes": 16.0 * px + 224.0 * n, "flops": px * spp * 7 * (_ray_flops(n) + 300)}
    px = case["w"] * case["h"]
    samples = px * case.get("frames", 1)
    n = _tris(case)
    rays = 8.0 if case["mode"] == 1 else 4.0 + 4.0 * case["mis"]
    return {"bytes": 32.0 * px + 224.0 * n, "flops": samples * rays * (_ray_flops(n) + 300)}


# ------------------------------------------------------------------- exact

def _xyz(a):
    return torch.from_numpy(np.ascontiguousarray(a[:, :3]).astype(np.float64)).cuda()


def _exact_t(case, seed):
    """Hit distances over all triangles and the light quad, in 64 bits."""
    s, r = _rays(case, seed)
    v1, v2, v3 = (_xyz(s.tris[k]) for k in ("v1", "v2", "v3"))
    rays = torch.from_numpy(r.astype(np.float64)).cuda()
    q = s.light
    vec = lambda x: torch.tensor([float(x[i]) for i in range(3)], dtype=torch.float64, device="cuda")  # noqa: E731
    pos, nrm, el, ew = vec(q.pos), vec(q.normal), vec(q.edge_l), vec(q.edge_w)
    out = torch.empty(case["n"], dtype=torch.float64, device="cuda")
    e1, e2 = v2 - v1, v3 - v1
    fn, m = torch.linalg.cross(e1, e2), torch.linalg.cross(v1, e1)
    m2 = torch.linalg.cross(e2, v1)
    step = max(1, int(2e8) // len(v1))
    for i in range(0, case["n"], step):
        o, length, d = rays[i:i + step, :3], rays[i:i + step, 3], rays[i:i + step, 4:7]
        # Cramer's rule with the products of each ray and triangle as matrix products:
        # det = -d.n, u = det[o - v1, e2, d], v = det[o - v1, d, e1], t = (o - v1).n
        det = -(d @ fn.T)
        od = torch.linalg.cross(o, d)
        u = (od @ e2.T - d @ m2.T) / det
        v = -(od @ e1.T + d @ m.T) / det
        t = (o @ fn.T - (v1 * fn).sum(1)) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0) & (t < length[:, None])
        best = torch.where(ok, t, torch.inf).amin(1)
        dn = d @ nrm
        tq = ((pos - o) @ nrm) / dn
        h = o + d * tq[:, None] - pos
        a, b = el.norm(), ew.norm()
        pa, pb = (h @ el) / a, (h @ ew) / b
        hit = (dn.abs() > 1e-4) & (tq > 0) & (tq < length) & (pa >= 0) & (pa <= a) & (pb >= 0) & (pb <= b)
        best = torch.minimum(best, torch.where(hit, tq, torch.inf))
        out[i:i + step] = torch.minimum(best, length)
    return out


def exact(case, seed):
    """Distances of traced rays and tonemapped images; a rendered image is
    one draw of a random estimator, which 64 bits do not repeat."""
    if case["call"] in ("rays", "device") and not case.get("shadow"):
        if case["n"] * _tris(case) > 1.3e11:
            return None
        return {"tri": None, "light": None, "t": _exact_t(case, seed)}
    if case["call"] == "tonemap":
        g = torch.Generator(device="cuda").manual_seed(seed)
        img = torch.exp(torch.randn((case["h"], case["w"], 4), generator=g, device="cuda") - 1.0)
        img[..., 3] = 64.0
        c = img.double()
        if case["op"] == 1:
            x = c
            ldr = (x * (0.15 * x + 0.05) + 0.004) / (x * (0.15 * x + 0.50) + 0.06) - 0.02 / 0.30
        else:
            lum = 0.212671 * c[..., 0:1] + 0.715160 * c[..., 1:2] + 0.072169 * c[..., 2:3] + 0.001
            ldr = (c / lum) * (lum * (1 + lum) / (1 + lum))
        return ldr ** (1 / 2.2)
    return None
