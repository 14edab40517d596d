"""Whole paths in one launch (k_paths) against the wavefront.

A job with counting on always runs in the wavefront; without, small batches
run in k_paths and large ones are finished by it.  Each path's arithmetic is
the same, so images and ray counts must be equal bit for bit.
"""
import numpy as np
import pytest

import yune_amd as Y

pytestmark = pytest.mark.gpu


def render(ctx, sid, cam, w, h, frames, params, counting):
    j = ctx.job(sid, cam, w, h, params, base_seed=9)
    j.set_counting(counting)
    j.render(frames)
    img, st = j.read(), j.stats()
    j.release()
    return img.view(np.int32), (st.rays_ext, st.rays_shadow, st.samples)


PARAMS = {"mis": dict(mis=1, max_bounces=8, rr_threshold=2), "shipped": dict(), "direct": dict(gi=0),
          "fix": dict(mis=1, fix_mis=1, oren_nayar=1)}


@pytest.mark.parametrize("kind", sorted(PARAMS))
@pytest.mark.parametrize("scene", ["cornell", "room", "brute"])
def test_paths_equal_wavefront(scene, kind):
    """Sizes around a wave, a block and one path per wave, and more paths
    than lanes (taken from the queue as others end)."""
    s = Y.gen_icosphere_room(7, 6, 3) if scene == "room" else Y.gen_cornell()
    params = Y.params_reference(0, **PARAMS[kind])
    with Y.Context(max_paths=1 << 20) as ctx:
        sid = ctx.scene(s, brute=scene == "brute")
        for w, h, f in ((1, 1, 1), (9, 7, 1), (64, 1, 1), (13, 5, 3), (64, 65, 1), (97, 61, 2), (640, 500, 3)):
            a = render(ctx, sid, s.cam, w, h, f, params, False)
            b = render(ctx, sid, s.cam, w, h, f, params, True)
            assert np.array_equal(a[0], b[0]), (w, h, f)
            assert a[1] == b[1], (w, h, f)


def test_wavefront_finished_by_paths():
    """More paths than k_paths takes from the start: the wavefront hands its
    last rays over, and the image is that of the frames rendered one by one."""
    s = Y.gen_cornell()
    params = Y.params_reference(0, mis=1)
    with Y.Context() as ctx:
        sid = ctx.scene(s)
        a = render(ctx, sid, s.cam, 1000, 1000, 9, params, False)
        j = ctx.job(sid, s.cam, 1000, 1000, params, base_seed=9)
        for _ in range(9):
            j.render(1)
        b = j.read().view(np.int32), (j.stats().rays_ext, j.stats().rays_shadow, j.stats().samples)
        c = render(ctx, sid, s.cam, 1000, 1000, 9, params, True)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[0], c[0])
    assert a[1] == b[1] == c[1]


def test_paths_over_several_scenes():
    """A scheduler round with jobs of several scenes against each job alone."""
    scenes = [Y.gen_cornell(), Y.gen_icosphere_room(3, 4, 3), Y.gen_icosphere_room(5, 2, 2)]
    params = Y.params_reference(0, mis=1, max_bounces=8, rr_threshold=2)
    with Y.Context(max_paths=1 << 20, serve_mode=1) as ctx:
        sids = [ctx.scene(s) for s in scenes]
        jobs = [ctx.submit(sid, s.cam, 65 + 7 * k, 33, params, 3, 4 + k)
                for k, (sid, s) in enumerate(zip(sids, scenes))]
        while ctx.serve(4):
            pass
        for k, (j, sid, s) in enumerate(zip(jobs, sids, scenes)):
            alone = ctx.job(sid, s.cam, 65 + 7 * k, 33, params, base_seed=4 + k)
            alone.set_counting(True)
            alone.render(3)
            assert np.array_equal(j.read().view(np.int32), alone.read().view(np.int32)), k


@pytest.mark.parametrize("kw", [dict(mis=1, bdpt_bounces=5), dict(mis=0, bdpt_bounces=1), dict(),
                                dict(mis=1, bdpt_bounces=40, fix_mis=1)], ids=["mis5", "one", "shipped", "40"])
@pytest.mark.parametrize("scene", ["cornell", "room", "brute"])
def test_bidirectional_paths_equal_wavefront(scene, kw):
    s = Y.gen_icosphere_room(7, 6, 2) if scene == "room" else Y.gen_cornell()
    params = Y.params_reference(1, **kw)
    with Y.Context(max_paths=1 << 20) as ctx:
        sid = ctx.scene(s, brute=scene == "brute")
        for w, h, f in ((1, 1, 1), (9, 7, 1), (64, 65, 1), (97, 61, 2), (640, 500, 1)):
            a = render(ctx, sid, s.cam, w, h, f, params, False)
            b = render(ctx, sid, s.cam, w, h, f, params, True)
            assert np.array_equal(a[0], b[0]), (w, h, f)
            assert a[1] == b[1], (w, h, f)


@pytest.mark.parametrize("mode", [0, 1], ids=["pt", "bdpt"])
def test_frames_in_the_arguments(mode):
    """Launches of up to 16 frames take their seeds as arguments, longer ones
    from memory; ray queries between them use the same counters."""
    s = Y.gen_cornell()
    params = Y.params_reference(mode, mis=1, bdpt_bounces=3)
    rays = np.zeros((400000, 8), np.float32) + np.float32((0, 0, 9, 1e9, 0, 0, -1, 0))     # more than lanes
    with Y.Context(max_paths=1 << 19) as ctx:
        sid = ctx.scene(s)
        j = ctx.job(sid, s.cam, 33, 21, params, base_seed=9)
        ref = ctx.job(sid, s.cam, 33, 21, params, base_seed=9)
        ref.set_counting(True)
        for f in (1, 2, 15, 16, 17, 33, 1):
            j.render(f)
            if f & 1:
                ctx.trace(sid, rays)
            ref.render(f)
            assert np.array_equal(j.read().view(np.int32), ref.read().view(np.int32)), f
            a, b = j.stats(), ref.stats()
            assert (a.rays_ext, a.rays_shadow, a.samples) == (b.rays_ext, b.rays_shadow, b.samples), f


@pytest.mark.parametrize("size,frames", [(9, 1), (64, 3), (1500, 4)])
def test_continuous_jobs_end_in_one_launch(size, frames):
    """Jobs of two scenes, few enough for one launch or (9M paths) a wavefront
    first, with submissions between the calls, against each job alone."""
    scenes = [Y.gen_cornell(), Y.gen_icosphere_room(3, 4, 3)]
    params = Y.params_reference(0, mis=1)
    with Y.Context(serve_mode=0) as ctx:
        sids = [ctx.scene(s) for s in scenes]
        jobs = []
        for k in range(4):
            jobs.append((ctx.submit(sids[k % 2], scenes[k % 2].cam, size + k, size, params, frames, 4 + k), k))
            if k & 1:
                ctx.serve(1)
        while ctx.serve(4):
            pass
        for j, k in jobs:
            alone = ctx.job(sids[k % 2], scenes[k % 2].cam, size + k, size, params, base_seed=4 + k)
            alone.set_counting(True)
            alone.render(frames)
            assert np.array_equal(j.read().view(np.int32), alone.read().view(np.int32)), k
            alone.release()


@pytest.mark.parametrize("mode", [0, 1], ids=["pt", "bdpt"])
def test_whole_path_launches_report_their_time(mode):
    s = Y.gen_cornell()
    with Y.Context(max_paths=1 << 18) as ctx:
        j = ctx.job(ctx.scene(s), s.cam, 320, 200, Y.params_reference(mode, mis=1, bdpt_bounces=3), base_seed=2)
        j.render(2)
        st = j.stats()
        assert st.iterations == 0 and st.ms_trace_ext == 0
        assert 0 < st.ms_other <= st.ms_total
        one = st.ms_other
        j.render(2)
        assert j.stats().ms_other > one


@pytest.mark.parametrize("room,vertices,w,h,whole", [
    ((7, 6, 3), 8, 1200, 1000, True), ((7, 24, 4), 5, 640, 400, True), ((7, 24, 4), 5, 1200, 1000, False),
    ((7, 24, 4), 3, 1200, 1000, True), ((7, 24, 4), 3, 1500, 1500, False), ((7, 24, 4), 12, 1200, 1000, False)])
def test_large_bidirectional_batches_of_large_trees_run_in_the_wavefront(room, vertices, w, h, whole):
    """One launch of whole paths takes 1.2 times as long and more there."""
    s = Y.gen_icosphere_room(*room)
    params = Y.params_reference(1, mis=1, bdpt_bounces=vertices)
    with Y.Context(max_paths=1 << 22) as ctx:
        j = ctx.job(ctx.scene(s), s.cam, w, h, params, base_seed=9)
        j.render(1)
        assert (j.stats().iterations == 0) == whole
