"""The fast vertex projection outside its range: poses whose coordinates
overflow, in X and Y alone (a rotation about the view axis) or in all three,
and meshes with vertices that do; bit-exact against the oracle."""
import numpy as np
import pytest

import oracle as O
import qpso
import workloads as W
from helpers import assert_same_f32, assert_same_i32

pytestmark = pytest.mark.gpu


def check(mesh, poses, cfg):
    scene = W.config0()[0]
    c = scene.clusters[0]
    n = poses.shape[1]
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        mid = ctx.upload_mesh(mesh)
        with ctx.solve(mid, scene.cluster(), qpso.make_params(n, 1, cam=W.CAM)) as s:
            fit, aabb, _ = s.eval_poses(poses)
        ctx.release_mesh(mid)
    want, boxes = [], []
    for i in range(n):
        fr, info = O.render(mesh, poses[:, i], W.CAM, c["rect"])
        # a box beyond the guard's limit is nobody's (the particle scores NaN)
        boxes.append(list(aabb[i] if info.degenerate else info.aabb))
        want.append(O.fitness(info, c["rect"], c["num_points"], fr, c["depth"])[0])
    assert_same_i32(aabb, np.array(boxes, np.int32), "aabb")
    assert_same_f32(fit, np.array(want, np.float32), "fitness")


def poses_of(v):
    gt = np.array([0.0, 0.0, 0.7, 1, 0, 0, 0], np.float32)
    out = np.repeat(gt[:, None], 9, axis=1)
    out[3:, :4] = 0
    for i in range(4):
        out[3 + i, i] = v     # one component of the quaternion
        if i:
            out[3 + i, 3 + i] = v  # beside a real part of 1
    out[0, 7], out[1, 8] = v, v    # the position
    return out


# meshes kept whole, and drawn in windows
@pytest.mark.parametrize("cfg,faces", [(0, 60), (2, 60), (4, 12000)])
@pytest.mark.parametrize("v", [1e12, 1e19, 1e20, 3e38, np.inf, -np.inf, np.nan])
def test_overflowing_poses(cfg, faces, v):
    sl, st = W.uv_dims(faces)
    check(qpso.mesh_uv_ellipsoid(sl, st, 40.0, 30.0, 25.0, 2, 4.0, 8.0, 0), poses_of(np.float32(v)), cfg)


@pytest.mark.parametrize("v", [1e20, 2e37, 3e38, np.inf])
def test_overflowing_vertices(v):
    # a few vertices' x and y far out, under rotations about the view axis
    # (not unit quaternions: one product overflows either way, X is inf - inf
    # while Z is a number)
    sl, st = W.uv_dims(60)
    mesh = qpso.mesh_uv_ellipsoid(sl, st, 40.0, 30.0, 25.0, 2, 4.0, 8.0, 0).reshape(9, -1)
    mesh[:2, ::7] = np.float32(v)
    poses = np.zeros((7, 6), np.float32)
    poses[2] = 0.7
    for i in range(6):
        a, m = 0.6 * (i % 3), (1.0, 4.0)[i // 3]
        poses[3, i], poses[6, i] = m * np.cos(a / 2), m * np.sin(a / 2)
    check(mesh.reshape(-1), poses, 0)
