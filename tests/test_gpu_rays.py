"""Caller's rays in one launch (k_rays): calls of every size give each ray
the result it has in a call of its own block.

Small calls read and write pinned host memory, larger ones the samples
buffer; up to one ray per lane a wave takes an equal share of the rays,
beyond that the lanes are refilled.  The blocks of 1,000 rays that the
results are compared with are themselves compared with the oracle by
test_trace_matches_oracle.
"""
import ctypes as C

import numpy as np
import pytest

import yune_amd as Y
from yune_amd._lib import lib

pytestmark = pytest.mark.gpu

LANES12, LANES16 = 256 * 7 * 256, 256 * 6 * 256        # rays a grid holds at 12 and 16 stack entries


def mixed_rays(n, seed):
    rng = np.random.default_rng(seed)
    r = np.zeros((n, 8), np.float32)
    r[:, :3] = rng.uniform(-4.9, 4.9, (n, 3))
    r[:, 4:7] = rng.normal(size=(n, 3))
    r[:, 7] = rng.uniform(size=n) < 0.3
    r[:, 3] = np.where(r[:, 7] != 0, rng.uniform(0.05, 6.0, n), np.inf)
    r[::97, 4] = 0.0                    # axis-parallel, NaN, infinite and empty rays among them
    r[::101, 5] = np.nan
    r[::103, 3] = 0.0
    r[::107, 0] = np.inf
    return r


def same(a, b):
    return all(np.array_equal(x.view(np.int32), y.view(np.int32)) for x, y in zip(a, b))


@pytest.fixture(scope="module")
def room():
    return Y.gen_icosphere_room(11, 12, 4)


@pytest.mark.parametrize("opts", [dict(), dict(bvh_width=2), dict(lds_stack=12, trace_xcd=3), dict(trace_refill=-1)],
                         ids=["default", "width2", "lds12-xcd3", "norefill"])
def test_call_sizes_give_the_same_results(room, opts):
    rays = mixed_rays(LANES12 + 70_001, 5)
    with Y.Context(max_paths=1 << 20, **opts) as c:
        sid = c.scene(room)
        # any-hit occluders depend on nothing but the tree, so all three arrays compare
        want = [np.concatenate(x) for x in zip(*(c.trace(sid, rays[i:i + 1000]) for i in range(0, 12_000, 1000)))]
        full = c.trace(sid, rays)
        assert same([x[:12_000] for x in full], want)
        for n in (1, 2, 63, 64, 65, 1000, 8191, 8192, 8193, LANES16 - 1, LANES16, LANES16 + 1, LANES12, LANES12 + 1):
            assert same(c.trace(sid, rays[:n]), [x[:n] for x in full]), n


@pytest.mark.parametrize("brute", [False, True])
def test_device_rays_at_any_alignment(brute):
    torch = pytest.importorskip("torch")
    s = Y.gen_cornell()
    n = 5003
    rays = mixed_rays(n, 8)
    rays[:, :3] = rays[:, :3] * 0.2 + np.float32([0, 0, -3])
    with Y.Context(max_paths=1 << 16) as c:
        sid = c.scene(s, brute=brute)
        want = c.trace(sid, rays)
        for off in (0, 1, 2, 3, 4):     # floats
            d = torch.zeros(n * 8 + 8, device="cuda")
            d[off:off + n * 8] = torch.from_numpy(rays.reshape(-1)).cuda()
            out = [torch.full((n + 3,), -7, dtype=t, device="cuda") for t in (torch.int32, torch.int32, torch.float32)]
            torch.cuda.synchronize()
            p = [C.c_void_p(o.data_ptr() + 4) for o in out]
            assert lib().yn_trace_noalloc(c._p, sid, C.c_void_p(d.data_ptr() + 4 * off), n, *p) == 0
            got = [o.cpu().numpy() for o in out]
            assert same([g[1:n + 1] for g in got], want), off
            assert all((g[0] == -7) and (g[n + 1:] == -7).all() for g in got)


def test_traversal_beyond_the_fixed_stack_is_refused():
    """yn_trace_noalloc's stack ends at 32 entries beyond the LDS part: a
    deeper traversal is an error, and the next call works."""
    torch = pytest.importorskip("torch")
    from test_gpu_pt import comb_scene
    deep, flat = comb_scene(60), Y.gen_cornell()
    rays = np.zeros((64, 8), np.float32)
    rays[:, 0] = np.linspace(-0.01, 0.01, 64)
    rays[:, 3] = np.inf
    rays[:, 6] = -1.0
    d = torch.from_numpy(rays).cuda()
    out = [torch.zeros(64, dtype=t, device="cuda") for t in (torch.int32, torch.int32, torch.float32)]
    torch.cuda.synchronize()
    with Y.Context(bvh_width=2, max_paths=1 << 12, hoist_frac=-1, leaf_max=10, bvh_build=2) as c:
        a, b = c.scene(deep, deep.nodes), c.scene(flat)
        assert c.scene_info(a).max_depth > 48
        p = [C.c_void_p(o.data_ptr()) for o in out]
        call = lambda sid: lib().yn_trace_noalloc(c._p, sid, C.c_void_p(d.data_ptr()), 64, *p)  # noqa: E731
        assert (c.trace(a, rays)[0] == 0).all()         # its stack follows the scene
        assert call(a) == -2
        assert call(b) == 0
        assert same([o.cpu().numpy() for o in out], c.trace(b, rays))


@pytest.mark.parametrize("lds,fits,deep", [(32, 60, 80), (16, 44, 60), (12, 40, 60), (8, 36, 60), (0, 44, 60)])
def test_fixed_stack_for_every_lds_size(lds, fits, deep):
    """yn_trace_noalloc takes traversals of 32 entries beyond the configured
    LDS part, whatever of it the kernel keeps in LDS."""
    torch = pytest.importorskip("torch")
    from test_gpu_pt import comb_scene
    rays = np.zeros((64, 8), np.float32)
    rays[:, 0] = np.linspace(-0.01, 0.01, 64)
    rays[:, 3] = np.inf
    rays[:, 6] = -1.0
    d = torch.from_numpy(rays).cuda()
    out = [torch.zeros(64, dtype=t, device="cuda") for t in (torch.int32, torch.int32, torch.float32)]
    torch.cuda.synchronize()
    with Y.Context(bvh_width=2, max_paths=1 << 12, hoist_frac=-1, leaf_max=10, bvh_build=2, lds_stack=lds) as c:
        for n, rc in ((fits, 0), (deep, -2)):
            s = comb_scene(n)
            sid = c.scene(s, s.nodes)
            p = [C.c_void_p(o.data_ptr()) for o in out]
            assert lib().yn_trace_noalloc(c._p, sid, C.c_void_p(d.data_ptr()), 64, *p) == rc, n
            if rc == 0:
                assert same([o.cpu().numpy() for o in out], c.trace(sid, rays))


@pytest.mark.parametrize("opts", [dict(trace_grid=1), dict(trace_grid=7, trace_block=64, trace_xcd=16),
                                  dict(trace_grid=20000)])
def test_configured_grid(room, opts):
    """Caller's rays keep to trace_grid blocks of trace_block threads: fewer
    of them take longer, for the same results."""
    import time

    def timed(c, sid):
        c.trace(sid, rays)
        best = 1e9
        for _ in range(3):
            t0 = time.perf_counter()
            r = c.trace(sid, rays)
            best = min(best, time.perf_counter() - t0)
        return r, best

    rays = mixed_rays(60_001, 6)
    with Y.Context(max_paths=1 << 16) as c:
        want, t = timed(c, c.scene(room))
    with Y.Context(max_paths=1 << 16, **opts) as c:
        got, tc = timed(c, c.scene(room))
    assert same(got, want)
    if opts["trace_grid"] < 20:
        assert tc > 4 * t               # at most 1,792 of 393,216 lanes


@pytest.mark.parametrize("shift", [0, 5, -5])
@pytest.mark.parametrize("deep", [False, True])
def test_results_over_the_device_rays(room, deep, shift):
    """Results may be written where the rays lie: every ray is read first.
    A deep tree's stacks leave room for fewer lanes than there are rays."""
    torch = pytest.importorskip("torch")
    from test_gpu_pt import comb_scene
    n = 262_143
    rays = mixed_rays(n, 12)
    opts = dict(bvh_width=2, hoist_frac=-1, leaf_max=10, bvh_build=2, lds_stack=32) if deep else {}
    s = comb_scene(80) if deep else room
    if deep:                            # short ways through the comb, one triangle each
        rng = np.random.default_rng(3)
        i = rng.integers(0, 80, n)
        rays[:, 0], rays[:, 1], rays[:, 2] = 0.0, -0.03, -1.0 - 0.1 * i + 0.05
        rays[:, 3], rays[:, 7] = rng.uniform(0.01, 5.0, n), 0.0
        rays[:, 4], rays[:, 5], rays[:, 6] = rng.uniform(-0.6, 0.6, n), 0.0, -1.0
    with Y.Context(max_paths=1 << 18, **opts) as c:
        sid = c.scene(s, s.nodes) if deep else c.scene(s)
        want = c.trace(sid, rays)
        assert not deep or 0.2 < (want[0] >= 0).mean() < 1.0
        d = torch.zeros(n * 8 + 16, device="cuda")
        d[8:8 + n * 8] = torch.from_numpy(rays.reshape(-1)).cuda()
        torch.cuda.synchronize()
        at = [d.data_ptr() + 4 * (8 + shift + k * n) for k in range(3)]
        assert lib().yn_trace_noalloc(c._p, sid, C.c_void_p(d.data_ptr() + 32), n, *(C.c_void_p(a) for a in at)) == 0
        got = [d[8 + shift + k * n:8 + shift + (k + 1) * n].cpu().numpy() for k in range(3)]
        assert same(got, want)


def test_reciprocal_rounds_as_division():
    """x_rcp against IEEE division over every exponent and both signs.  A ray
    straight at the plane of one right triangle of unit legs has the
    determinant s (its direction's length along the plane's normal) and the
    distance 1 / s exactly: both are reported bit for bit, and so is a hit that
    1 / s = inf, or 0, rules out."""
    s = Y.gen_cornell()
    s.tris = np.zeros(1, dtype=Y.TRI_DTYPE)
    s.tris["v1"], s.tris["v2"], s.tris["v3"] = (0, 0, 0, 1), (1, 0, 0, 1), (0, 1, 0, 1)
    for k in ("vn1", "vn2", "vn3"):
        s.tris[k] = (0, 0, 1, 0)
    s.mats = s.mats[:1]
    s.light = Y.light_quad((50, 50, 50), (0, -1, 0), (1, 1, 1), (0.1, 0, 0), (0, 0, 0.1))
    rng = np.random.default_rng(7)
    m = np.concatenate([rng.integers(0, 1 << 23, 2000), np.arange(24), (1 << 23) - 1 - np.arange(24),
                        (1 << 22) + np.arange(-8, 8)]).astype(np.uint32)
    x = ((np.arange(1, 255, dtype=np.uint32)[:, None] << 23) | m).reshape(-1).view(np.float32)
    rays = np.zeros((2 * len(x), 8), np.float32)
    rays[:, :2] = 0.25
    rays[:, 3] = np.inf
    rays[:len(x), 2], rays[:len(x), 6] = 1.0, -x        # det = x
    rays[len(x):, 2], rays[len(x):, 6] = -1.0, x        # det = -x
    with np.errstate(all="ignore"):
        inv = np.float32(1) / x
        u = (x * np.float32(0.25)) * inv                # both coordinates
        want = np.where((u >= 0) & (u + u <= 1) & (inv > 0) & (inv < np.inf), inv, np.float32(np.inf))
    with Y.Context(max_paths=1 << 21) as c:
        tri, light, t = c.trace(c.scene(s, brute=True), rays)
    assert (light == -1).all()
    for part in (slice(0, len(x)), slice(len(x), None)):
        assert np.array_equal(t[part].view(np.int32), want.view(np.int32))
        assert np.array_equal(tri[part] == 0, np.isfinite(want))
    assert np.isfinite(want).mean() > 0.99
