"""The scoring workspace and the pinned staging over calls of different sizes
on one context: scorings of few, many and few poses on different solves,
between runs and batches of many solves and of few;
every result equals the same call's on a context of its own."""
import numpy as np
import pytest

import qpso
import workloads as W
from helpers import assert_same_f32, assert_same_i32

pytestmark = pytest.mark.gpu


def same_result(a, b):
    assert_same_f32(np.array(a.pose[:], np.float32), np.array(b.pose[:], np.float32), "pose")
    assert_same_f32(np.float32(a.fit), np.float32(b.fit), "fitness")
    assert (a.raster_px, a.visit_px, a.n_degenerate, a.status) == (b.raster_px, b.visit_px, b.n_degenerate, b.status)


def poses_of(scene, n, seed):
    rng = np.random.default_rng(seed)
    gt = scene.objects[0][1]
    q = gt[3:, None] + rng.normal(0, 0.1, (4, n))
    out = np.empty((7, n), np.float32)
    out[:3] = gt[:3, None] * 1e-3 + rng.normal(0, 0.02, (3, n))
    out[3:] = q / np.linalg.norm(q, axis=0)
    return out


def alone(scene, params, call):
    with qpso.Context(0) as ctx:
        m = ctx.upload_mesh(scene.mesh_m())
        with ctx.solve(m, scene.cluster(), params) as s:
            r = call(s)
        ctx.release_mesh(m)
    return r


def test_sizes_in_turn_on_one_context():
    s0, p0 = W.config0(0)
    s1, p1 = W.config1(0, n_particles=2048, n_iters=2)
    p0.n_iters = 3
    few0, many1, few1 = poses_of(s0, 6, 1), poses_of(s1, 2048, 2), poses_of(s1, 6, 3)
    with qpso.Context(0) as ctx:
        m0, m1 = ctx.upload_mesh(s0.mesh_m()), ctx.upload_mesh(s1.mesh_m())
        a, b = ctx.solve(m0, s0.cluster(), p0), ctx.solve(m1, s1.cluster(), p1)
        got = [a.eval_poses(few0), b.run(), b.eval_poses(many1), a.run()]
        small = [ctx.solve(m0, s0.cluster(), p0) for _ in range(70)]
        batch = ctx.run_batch(small)
        got += [b.eval_poses(few1), ctx.run_batch(small[:3]), a.eval_poses(few0), b.eval_poses(many1)]
        for s in [a, b, *small]:
            s.close()
        ctx.release_mesh(m0)
        ctx.release_mesh(m1)
    r0 = alone(s0, p0, lambda s: s.run())
    r1 = alone(s1, p1, lambda s: s.run())
    e0 = alone(s0, p0, lambda s: s.eval_poses(few0))
    e1 = alone(s1, p1, lambda s: s.eval_poses(many1))
    e2 = alone(s1, p1, lambda s: s.eval_poses(few1))
    for g, want in ((got[0], e0), (got[2], e1), (got[4], e2), (got[6], e0), (got[7], e1)):
        assert_same_f32(g[0], want[0], "scores")
        assert_same_i32(g[1], want[1], "boxes")
    same_result(got[1], r1)
    same_result(got[3], r0)
    for r in [*batch, *got[5]]:
        same_result(r, r0)
