"""The wavefront at sizes where it runs, and the variants of the whole-path
launches that ordinary scenes do not reach.

Batches of more than 4M paths run in the wavefront until 8M rays are left;
bidirectional ones of more than 1M paths and a tree above 4 MB to the end.  The settings of its launches must not change an image, which is
compared with the counting wavefront's (other template instances) and, on a
tile, with the oracle's.
"""
import dataclasses
import functools

import numpy as np
import pytest

import yune_amd as Y
from oracle import pyoracle as O
from test_gpu_pt import comb_scene, identical, mre, ocam, oscene

pytestmark = pytest.mark.gpu

PT = dict(mode=0, W=1024, H=1024, F=9, kw=dict(mis=1, max_bounces=8, rr_threshold=2), max_paths=1 << 24, room=(9, 2))
BD = dict(mode=1, W=1040, H=1024, F=1, kw=dict(mis=1, bdpt_bounces=5), max_paths=1 << 21, room=(24, 4))
SETTINGS = [dict(), dict(trace_overlap=1, lds_stack=8), dict(graph=1), dict(graph=1, trace_overlap=1), dict(trace_xcd=1),
            dict(trace_xcd=3, trace_refill=1), dict(trace_refill=-1), dict(trace_refill=64, lds_stack=12),
            dict(shade_waves=2), dict(shade_waves=3, lds_stack=32)]


def bits(img):
    return img.view(np.int32)


@functools.lru_cache(maxsize=None)
def scene(spheres=9, subdiv=2, seed=3):
    return Y.gen_icosphere_room(seed, spheres, subdiv)


def render(c, sid, s, k, seed=23, calls=1, counting=False):
    job = c.job(sid, s.cam, k["W"], k["H"], Y.params_reference(k["mode"], **k["kw"]), base_seed=seed)
    job.set_counting(counting)
    for _ in range(calls):
        job.render(k["F"])
    st = job.stats()
    assert st.iterations > 0            # the wavefront ran
    out = bits(job.read()), (st.rays_ext, st.rays_shadow, st.samples)
    job.release()
    return out


@pytest.fixture(scope="module")
def counted():
    """The images of the counting wavefront, of one call and of two."""
    out = {}
    for name, k in (("pt", PT), ("bdpt", BD)):
        s = scene(*k["room"])
        with Y.Context(max_paths=k["max_paths"]) as c:
            sid = c.scene(s)
            assert name == "pt" or c.scene_info(sid).node_bytes > 4 << 20
            out[name] = {n: render(c, sid, s, k, calls=n, counting=True) for n in (1, 2)}
    return out


@pytest.mark.parametrize("name,k", [("pt", PT), ("bdpt", BD)])
@pytest.mark.parametrize("opts", SETTINGS, ids=lambda o: "-".join(f"{a}{b}" for a, b in o.items()) or "default")
def test_settings_keep_large_images(name, k, opts, counted):
    s = scene(*k["room"])
    with Y.Context(max_paths=k["max_paths"], **opts) as c:
        got = render(c, c.scene(s), s, k)
    assert got[1] == counted[name][1][1]
    assert np.array_equal(got[0], counted[name][1][0])


@pytest.mark.parametrize("name,k", [("pt", PT), ("bdpt", BD)])
def test_graph_follows_its_arguments(name, k, counted):
    """Two scenes and sizes in turn (captured again each time) and two calls
    of one job (replayed), with ray queries and small batches between them."""
    s, other = scene(*k["room"]), scene(*((22, 4, 5) if k["mode"] else (4, 3, 5)))
    ko = dict(k, W=k["W"] + 24)
    rays = np.zeros((9000, 8), np.float32) + np.float32((0, 0, 4, 1e9, 0, 0, -1, 0))
    with Y.Context(max_paths=k["max_paths"]) as c:
        want = render(c, c.scene(other), other, ko, calls=2)
    with Y.Context(max_paths=k["max_paths"], graph=1) as c:
        a, b = c.scene(s), c.scene(other)
        for _ in range(2):
            got = render(c, a, s, k, calls=2)
            assert got[1] == counted[name][2][1] and np.array_equal(got[0], counted[name][2][0])
            c.trace(a, rays)
            got = render(c, b, other, ko, calls=2)
            assert got[1] == want[1] and np.array_equal(got[0], want[0])
            small = c.job(a, s.cam, 20, 20, Y.params_reference(k["mode"], **k["kw"]))
            small.render(2)
            small.release()


@pytest.mark.parametrize("name,k", [("pt", PT), ("bdpt", BD)])
def test_large_images_match_the_oracle_on_a_tile(name, k, counted):
    s = scene(*k["room"])
    x0, y0, n = 500, 300, 40
    oimg, _, _, _ = oscene(s, s.bvh()).render(ocam(s.cam), k["W"], k["H"], O.params(k["mode"], **k["kw"]),
                                              O.mt19937(23, k["F"]), rect=(x0, y0, x0 + n, y0 + n), threads=8)
    g = counted[name][1][0].view(np.float32)[y0:y0 + n, x0:x0 + n]
    o = oimg[y0:y0 + n, x0:x0 + n]
    assert np.array_equal(g[..., 3], o[..., 3])
    assert identical(g, o) >= 0.999
    assert mre(g, o)[0] <= 0.01


def two(c, jobs, serve):
    """Images of (sid, cam, W, H, params, frames) jobs, alone or in a round."""
    out = []
    if serve:
        js = [c.submit(sid, cam, w, h, p, f, 31 + i) for i, (sid, cam, w, h, p, f) in enumerate(jobs)]
        while c.serve(8):
            pass
        return [bits(j.read()) for j in js]
    for i, (sid, cam, w, h, p, f) in enumerate(jobs):
        j = c.job(sid, cam, w, h, p, base_seed=31 + i)
        j.set_counting(True)
        j.render(f)
        out.append(bits(j.read()))
    return out


@pytest.mark.parametrize("serve_mode", [0, 1])
@pytest.mark.parametrize("mode", [0, 1], ids=["pt", "bdpt"])
@pytest.mark.parametrize("copies", [1, 60])
def test_more_materials_than_lds_holds(mode, copies, serve_mode):
    """More than 256 materials of one scene, and of all scenes together:
    whole paths then read them from memory."""
    cornell, room = Y.gen_cornell(), scene()
    n = len(cornell.mats)
    wide = dataclasses.replace(cornell, tris=cornell.tris.copy(), mats=np.tile(cornell.mats, copies * 300 // n + 1),
                               nodes=None)
    wide.tris["matID"] += n * (len(wide.mats) // n - 1)        # the last copy
    kw = dict(bdpt_bounces=4) if mode else dict(mis=1, max_bounces=8, rr_threshold=2)
    p = Y.params_reference(mode, **kw)
    with Y.Context(max_paths=1 << 18, serve_mode=serve_mode) as c:
        sw, sc, sr = c.scene(wide), c.scene(cornell), c.scene(room)
        jobs = [(sw, cornell.cam, 65, 40, p, 2), (sr, room.cam, 33, 50, p, 3)]
        for js in (jobs, jobs[:1]):
            for a, b in zip(two(c, js, True), two(c, js, False)):
                assert np.array_equal(a, b)
        # alone, uncounted, and the image of the box itself
        j = c.job(sw, cornell.cam, 65, 40, p, base_seed=31)
        j.render(2)
        assert j.stats().iterations == 0
        assert np.array_equal(bits(j.read()), two(c, [(sc, cornell.cam, 65, 40, p, 2)], False)[0])


@pytest.mark.parametrize("mode", [0, 1], ids=["pt", "bdpt"])
def test_whole_paths_on_a_deep_tree(mode):
    """Camera rays down a comb-shaped tree: deeper than the 12 entries that
    whole paths keep in LDS, both with the tree as kernel argument and in a
    round with another scene."""
    s = comb_scene(60)
    s.cam = Y.camera((1, 0, 0), (0, 1, 0), (0, 0, -1), (0, 0, 0), 6.0)
    s.light = Y.light_quad((-0.5, -0.5, 0.5), (0, 0, -1), (5, 5, 5), (1, 0, 0), (0, 1, 0))     # behind the camera
    s.mats["ke"][:, :3] = (0.1, 0.2, 0.3)
    flat = Y.gen_cornell()
    kw = dict(bdpt_bounces=4) if mode else dict(mis=1, max_bounces=6, rr_threshold=2)
    p = Y.params_reference(mode, **kw)
    with Y.Context(max_paths=1 << 16, hoist_frac=-1, leaf_max=10, bvh_build=2, serve_mode=1) as c:
        a, b = c.scene(s, s.nodes), c.scene(flat)
        assert c.scene_info(a).max_depth > 16
        want = two(c, [(a, s.cam, 40, 30, p, 2), (b, flat.cam, 20, 20, p, 1)], False)
        assert np.array_equal(two(c, [(a, s.cam, 40, 30, p, 2), (b, flat.cam, 20, 20, p, 1)], True)[0], want[0])
        j = c.job(a, s.cam, 40, 30, p, base_seed=31)
        j.render(2)
        assert j.stats().iterations == 0
        img = j.read()
        assert np.array_equal(bits(img), want[0])
    oimg, _, _, _ = oscene(s, s.nodes).render(ocam(s.cam), 40, 30, O.params(mode, **kw), O.mt19937(31, 2), threads=8)
    assert identical(img, oimg) >= 0.999
    assert len(np.unique(img[..., :3])) > 3         # the triangles and the background
