"""The boxes of poses and meshes whose coordinates overflow, held against a
restatement of the general projection (main.h:309-369, 514-545, 1326-1353) in
numpy: the particle scores NaN, but its box is reported, and the fast
projection must leave it to the general one.  The meshes have fewer vertices
than a workgroup has threads, so that the extremes of a wrapped coordinate do
not depend on which vertices share a thread."""
import numpy as np
import pytest

import qpso
import workloads as W
from helpers import assert_same_i32

pytestmark = pytest.mark.gpu

F, D = np.float32, np.float64


def fma(a, b, c):
    return F(D(a) * D(b) + D(c))


def box_of(mesh, pose):
    """AABB (minX, maxX, minY, maxY) of every vertex, with the sentinels."""
    m = mesh.reshape(3, -1).astype(F)  # x, y, z of all corners
    vx, vy, vz = m
    t, q0, q1, q2, q3 = pose[:3], *pose[3:]
    two = F(2)
    t0 = two * fma(q2, vz, -(q3 * vy))
    t1 = two * -fma(q1, vz, -(q3 * vx))
    t2 = two * fma(q1, vy, -(q2 * vx))
    k0 = fma(q2, t2, -(q3 * t1))
    k1 = -fma(q1, t2, -(q3 * t0))
    k2 = fma(q1, t1, -(q2 * t0))
    px, py, pz = (fma(q0, a, v) + k + d for a, v, k, d in ((t0, vx, k0, t[0]), (t1, vy, k1, t[1]), (t2, vz, k2, t[2])))
    r = F(1) / pz
    fx, fy, cx, cy = W.CAM
    out = []
    for v, f, c in ((px * r, fx, cx), (py * r, fy, cy)):
        x = np.rint(F(16) * F(f * D(v) + c)).astype(D)
        x = np.where(np.isnan(x), 0, np.clip(x, -2.0 ** 31, 2.0 ** 31 - 1)).astype(np.int64)
        b = ((x + 15 + 2 ** 31) % 2 ** 32 - 2 ** 31) >> 4  # 32-bit, wrapping
        out += [min(50000, int(b.min())), max(-1, int(b.max()))]
    return out


def check(mesh, poses, cfg):
    scene = W.config0()[0]
    n = poses.shape[1]
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        m = ctx.upload_mesh(mesh)
        with ctx.solve(m, scene.cluster(), qpso.make_params(n, 1, cam=W.CAM)) as s:
            _, aabb, _ = s.eval_poses(poses)
        ctx.release_mesh(m)
    with np.errstate(all="ignore"):
        want = [box_of(mesh, poses[:, i]) for i in range(n)]
    assert_same_i32(aabb, np.array(want, np.int32), "aabb")


def small_mesh():
    sl, st = W.uv_dims(60)
    return qpso.mesh_uv_ellipsoid(sl, st, 40.0, 30.0, 25.0, 2, 4.0, 8.0, 0)


@pytest.mark.parametrize("cfg", [0, 2, 4])
@pytest.mark.parametrize("v", [1.0, 1e12, 1e19, 1e20, 3e38, np.inf, -np.inf, np.nan])
def test_boxes_of_overflowing_poses(cfg, v):
    poses = np.repeat(np.array([[0.0, 0.0, 0.7, 1, 0, 0, 0]], F).T, 9, axis=1)
    poses[3:, :4] = 0
    for i in range(4):
        poses[3 + i, i] = v     # one component of the quaternion
        if i:
            poses[3 + i, 3 + i] = v  # beside a real part of 1
    poses[0, 7], poses[1, 8] = v, v    # the position
    check(small_mesh(), poses, cfg)


@pytest.mark.parametrize("cfg", [0, 4])
@pytest.mark.parametrize("axes", [(0, 1), (0,), (1,), (2,)])
@pytest.mark.parametrize("v", [1e20, 2e37, 3e38, np.inf, np.nan])
def test_boxes_of_overflowing_vertices(cfg, axes, v):
    # a few vertices far out, under rotations about the view axis (some not
    # unit quaternions: one product overflows either way and X is inf - inf
    # while Z is a number)
    mesh = small_mesh().reshape(3, 3, -1)
    for a in axes:
        mesh[a, 0, ::7] = F(v)
    poses = np.zeros((7, 6), F)
    poses[2] = 0.7
    for i in range(6):
        ang, m = 0.6 * (i % 3), (1.0, 4.0)[i // 3]
        poses[3, i], poses[6, i] = m * np.cos(ang / 2), m * np.sin(ang / 2)
    check(mesh.reshape(-1), poses, cfg)
