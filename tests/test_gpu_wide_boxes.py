"""Particles whose boxes leave the packed cache's 16-bit range: meshes drawn in
windows whose faces the later bits do not hold (their coordinates clamped to
the halves) and meshes whose faces they hold (every face from its corner
table), by the fast and the general projection, one band and several;
bit-exact against the oracle, and no slower than the same mesh in
boxes that fit."""
import numpy as np
import pytest

import oracle as O
import qpso
import workloads as W
from helpers import assert_same_f32, assert_same_i32

pytestmark = pytest.mark.gpu


def scene_of(faces, extent):
    z = 700.0
    a = extent * z / W.CAM[0] / 2.0
    sl, st = W.uv_dims(faces)
    mesh = qpso.mesh_uv_ellipsoid(sl, st, a, a * 0.9, a * 0.7, 2, 0.1 * a, 0.2 * a, 0)
    pose = np.array([4.0, -3.0, z, *qpso.random_quat(60)], np.float32)
    depth, labels = qpso.scene_render([(mesh, pose)], W.CAM, 1300.0, 2.0, 0.05, 6)
    return W.Scene([(mesh, pose)], depth, labels), a * 1e-3


def wide(b):
    return max(b[1] - b[0], b[3] - b[2]) > 2046 or min(b[0], b[2]) < -2047 or max(b[1], b[3]) > 2046


# 45k faces take 1,408 words of later bits, over an eighth of 10,112 words; 90k
# take 2,814, over an eighth of 20,224
@pytest.mark.parametrize("cfg,faces,extent", [(4, 45000, 60), (4, 45000, 300), (2, 90000, 120), (3, 90000, 300),
                                              (2, 45000, 120), (0, 9000, 120), (0, 45000, 120)])
@pytest.mark.parametrize("general", [False, True])
def test_wide_boxes_match_oracle(cfg, faces, extent, general):
    scene, a = scene_of(faces, extent)
    c = scene.clusters[0]
    mesh = scene.mesh_m().reshape(9, -1)
    if general:  # a corner beyond the fast projection's mesh bound, far ahead
        mesh[[2, 5, 8], -1] = (0.0, 0.0, 2e6)
    mesh = np.ascontiguousarray(mesh).reshape(-1)
    n = 6
    poses = np.zeros((7, n), np.float32)
    poses[3] = 1.0
    poses[2] = a * np.array([0.78, 0.783, 0.81, 0.795, 0.83, 0.95])
    poses[0] = a * np.array([0.0, 0.02, -0.4, 0.1, 0.6, 0.0])
    poses[1] = a * np.array([0.0, -0.05, 0.02, 0.1, 0.0, 0.1])
    if not general:
        poses[4:, 2::3] = 0.01  # and turned a little
    want, boxes = [], []
    for i in range(n):
        fr, info = O.render(mesh, poses[:, i], W.CAM, c["rect"])
        assert not info.degenerate
        boxes.append(list(info.aabb))
        want.append(O.fitness(info, c["rect"], c["num_points"], fr, c["depth"])[0])
    assert sum(wide(b) for b in boxes) >= 3 and not wide(boxes[-1])
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        m = ctx.upload_mesh(mesh)
        with ctx.solve(m, scene.cluster(), qpso.make_params(n, 1, cam=W.CAM)) as s:
            fit, aabb, _ = s.eval_poses(poses)
            fit2, aabb2, frames = s.eval_poses(poses, frames=True)
        ctx.release_mesh(m)
    assert_same_i32(aabb, np.array(boxes, np.int32), "aabb")
    assert_same_f32(fit, np.array(want, np.float32), "fitness")
    assert_same_i32(aabb2, np.array(boxes, np.int32), "aabb of the frame dump")
    assert_same_f32(fit2, np.array(want, np.float32), "fitness of the frame dump")
    fr, _ = O.render(mesh, poses[:, 0], W.CAM, c["rect"])
    assert_same_i32(frames[0], fr, "frame")


# 150k faces: more than the bits hold. One iteration from random orientations at
# one place; boxes too wide to pack took 1.5 times as long as boxes that
# fit when each band projected every face anew, 0.55 and 0.70 times since.
@pytest.mark.parametrize("cfg", [3, 4])
def test_wide_boxes_keep_the_cache(cfg):
    scene, a = scene_of(150000, 300)
    c = scene.clusters[0]

    def launch_ms(ctx, m, z):
        cl = qpso.make_cluster(c["rect"], (0.0, 0.0, z * 1e3), c["num_points"], c["depth"])
        with ctx.solve(m, cl, qpso.make_params(64, 1, cam=W.CAM, t_bound=0.0, t_bound_z=0.0)) as s:
            return min(s.run_timed()[1].ms_render_fitness for _ in range(10))

    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        m = ctx.upload_mesh(scene.mesh_m())
        t_wide, t_fit = launch_ms(ctx, m, 1.015 * a), launch_ms(ctx, m, 1.6 * a)
        ctx.release_mesh(m)
    assert t_wide < t_fit
