"""Paths that reach the bounce limit of a launch (k_paths) before they end."""
import time

import numpy as np
import pytest

import yune_amd as Y
from mirror_box import mirror_box

pytestmark = pytest.mark.gpu
ENDLESS = dict(max_bounces=1 << 30, rr_threshold=1 << 30)


def bits(a):
    return np.asarray(a).view(np.int32)


def test_frames_that_fail_leave_their_images():
    """A frame with a path that does not end is an error, and what the image
    held stays: samples that were never written are not folded into it."""
    torch = pytest.importorskip("torch")
    box, cornell = mirror_box(), Y.gen_cornell()
    p, ok = Y.params_reference(**ENDLESS), Y.params_reference(mis=1, max_bounces=4)
    with Y.Context(max_paths=1 << 12) as c:
        a, b = c.scene(box), c.scene(cornell)

        def good():                     # also leaves its samples in the buffer
            j = c.job(b, cornell.cam, 16, 16, ok, base_seed=3)
            j.render(2)
            img = j.read()
            j.release()
            return img

        first = good()
        prev = torch.arange(2 * 3 * 4, dtype=torch.float32, device="cuda").reshape(2, 3, 4) + 5
        out = torch.full_like(prev, -7)
        torch.cuda.synchronize()
        with pytest.raises(Y.YuneError):
            c.pathtracer(out, prev, box.cam, a, 3, 2, p, 1, 0, 99)
        assert np.array_equal(bits(out.cpu()), bits(prev.cpu()))
        job = c.job(a, box.cam, 3, 2, p, base_seed=4)
        with pytest.raises(Y.YuneError):
            job.render(3)
        assert not job.read().any()
        assert np.array_equal(bits(good()), bits(first))


def test_rounds_that_fail_leave_their_images():
    box, cornell = mirror_box(), Y.gen_cornell()
    with Y.Context(max_paths=1 << 12, serve_mode=1) as c:
        a, b = c.scene(box), c.scene(cornell)
        warm = c.job(b, cornell.cam, 16, 16, Y.params_reference(mis=1), base_seed=3)
        warm.render(2)                  # samples in the buffer
        fine = c.submit(b, cornell.cam, 8, 8, Y.params_reference(mis=1), 2, base_seed=5)
        bad = c.submit(a, box.cam, 3, 2, Y.params_reference(**ENDLESS), 2, base_seed=5)
        fine_was, bad_was = bits(fine.read()), bits(bad.read())
        with pytest.raises(Y.YuneError):
            c.serve(1)
        assert np.array_equal(bits(fine.read()), fine_was) and np.array_equal(bits(bad.read()), bad_was)


@pytest.mark.parametrize("graph", [0, 1])
def test_an_endless_job_is_served_beside_others(graph):
    """Continuous serving: a job whose paths do not end stays pending, and
    the others are rendered as if it were not there: one with paths of several
    launches, small ones, and, submitted later, one of more work than fits
    (so that the wavefront goes on with the endless paths in it)."""
    box, cornell = mirror_box(), Y.gen_cornell()
    ok = Y.params_reference(mis=1)
    specs = [(0, 3, 2, Y.params_reference(**ENDLESS), 2), (0, 5, 3, Y.params_reference(max_bounces=3000, rr_threshold=1 << 30), 2),
             (1, 16, 12, ok, 3), (1, 64, 64, ok, 5), (0, 7, 1, Y.params_reference(max_bounces=511, rr_threshold=1 << 30), 1),
             (1, 9, 9, ok, 1)]
    got = []
    with Y.Context(max_paths=1 << 12, serve_mode=0, graph=graph) as c:
        sids = [c.scene(box), c.scene(cornell)]
        cams = [box.cam, cornell.cam]
        jobs = []

        def submit(k):
            scene, w, h, p, frames = specs[k]
            jobs.append(c.submit(sids[scene], cams[scene], w, h, p, frames, 11 + k))

        def serve():
            for _ in range(4000):
                if c.serve(1) == 1:
                    return
            raise AssertionError("the other jobs did not end")

        for k in (0, 1, 2):
            submit(k)
        serve()
        for k in (3, 4):
            submit(k)
        serve()
        submit(5)
        serve()
        assert not jobs[0].status()["done"]
        got = [bits(j.read()) for j in jobs]
    with Y.Context(max_paths=1 << 14) as c:
        sids = [c.scene(box), c.scene(cornell)]
        for k, (scene, w, h, p, frames) in enumerate(specs):
            if k:
                alone = c.job(sids[scene], cams[scene], w, h, p, base_seed=11 + k)
                alone.set_counting(True)        # in the wavefront
                alone.render(frames)
                assert np.array_equal(got[k], bits(alone.read())), k


def test_a_large_round_that_fails_leaves_its_images():
    """More paths than one launch takes: the wavefront's last paths, several
    scenes' among them, do not end."""
    box, cornell = mirror_box(), Y.gen_cornell()
    with Y.Context(max_paths=1 << 23, serve_mode=1) as c:
        a, b = c.scene(box), c.scene(cornell)
        fine = c.submit(b, cornell.cam, 1024, 1024, Y.params_reference(mis=1), 5, base_seed=5)
        bad = c.submit(a, box.cam, 3, 2, Y.params_reference(**ENDLESS), 1, base_seed=5)
        fine_was, bad_was = bits(fine.read()), bits(bad.read())
        with pytest.raises(Y.YuneError):
            c.serve(1)
        assert c.serve_stats().iterations > 0
        assert np.array_equal(bits(fine.read()), fine_was) and np.array_equal(bits(bad.read()), bad_was)
        bad.release()
        while c.serve(1):
            pass
        assert fine.read()[..., 3].min() == 5


def test_a_released_endless_job_is_dropped():
    """Once the job is released, other calls need not wait for its paths."""
    box, cornell = mirror_box(), Y.gen_cornell()
    rays = np.zeros((100, 8), np.float32) + np.float32((0, 0, -3, 1e9, 0.1, 0.2, -1, 0))
    p = Y.params_reference(mis=1)

    def use(c, b):
        j = c.job(b, cornell.cam, 16, 16, p, base_seed=3)
        j.render(2)
        return [bits(a) for a in (*c.trace(b, rays), j.read())]

    with Y.Context(max_paths=1 << 12) as c:
        want = use(c, c.scene(cornell))
    with Y.Context(max_paths=1 << 12, serve_mode=0) as c:
        a, b = c.scene(box), c.scene(cornell)
        for _ in range(2):
            endless = c.submit(a, box.cam, 3, 2, Y.params_reference(**ENDLESS), 2)
            fine = c.submit(b, cornell.cam, 16, 16, p, 2, base_seed=3)
            while c.serve(1) > 1:
                pass
            c.serve(2)
            endless.release()
            t0 = time.perf_counter()
            got = use(c, b)
            assert time.perf_counter() - t0 < 2
            assert all(np.array_equal(x, y) for x, y in zip(got, want))
            assert np.array_equal(bits(fine.read()), want[-1])
        c.release_scene(a)
