"""The packed vertex cache and the cull's faces-reaching-below bits at the
edges of their ranges: meshes kept whole in LDS and drawn window by window,
regions of one, two and several bands, more faces than the bits hold, boxes
too wide for packed coordinates; bit-exact against the oracle."""
import numpy as np
import pytest

import oracle as O
import qpso
import workloads as W
from helpers import assert_same_f32, assert_same_i32

pytestmark = pytest.mark.gpu


def scene_of(faces, extent, seed=0):
    z = 700.0
    a = extent * z / W.CAM[0] / 2.0
    sl, st = W.uv_dims(faces)
    mesh = qpso.mesh_uv_ellipsoid(sl, st, a, a * 0.9, a * 0.7, 2, 0.1 * a, 0.2 * a, seed)
    pose = np.array([4.0, -3.0, z, *qpso.random_quat(seed + 60)], np.float32)
    depth, labels = qpso.scene_render([(mesh, pose)], W.CAM, 1300.0, 2.0, 0.05, seed + 6)
    return W.Scene([(mesh, pose)], depth, labels)


def poses_of(scene, near=False):
    rng = np.random.default_rng(5)
    gt = scene.objects[0][1]
    out = np.zeros((7, 6), np.float32)
    for i in range(6):
        t = gt[:3] * 1e-3 + rng.normal(0, 0.01, 3) * (i > 0)
        if near:  # boxes of up to and beyond 2,046 pixels, reaching off the frame
            t = np.array([0.02 * (i - 2), 0.0, 0.085 + 0.012 * i])
        q = gt[3:] + rng.normal(0, 0.1, 4) * (i > 0)
        out[:3, i], out[3:, i] = t, q / np.linalg.norm(q)
    return out


def check(scene, cfg, poses, face_cap=0):
    p = qpso.make_params(6, 1, cam=W.CAM, face_cap=face_cap)
    c = scene.clusters[0]
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        mid = ctx.upload_mesh(scene.mesh_m())
        with ctx.solve(mid, scene.cluster(), p) as s:
            fit, aabb, _ = s.eval_poses(poses)
        ctx.release_mesh(mid)
    want, boxes = [], []
    for i in range(6):
        fr, info = O.render(scene.mesh_m(), poses[:, i], W.CAM, c["rect"], face_cap=face_cap)
        boxes.append(list(info.aabb))
        want.append(O.fitness(info, c["rect"], c["num_points"], fr, c["depth"])[0])
    assert_same_i32(aabb, np.array(boxes, np.int32), "aabb")
    assert_same_f32(fit, np.array(want, np.float32), "fitness")
    return boxes


# vertices about half the faces: beside a 60 px rect a 40,448-word tile holds
# up to about 32k of them, a 20,224-word one 13k, a 10,112-word one 5k
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("faces", [2500, 9000, 21000, 60000])
def test_cache_sizes(cfg, faces):
    check(scene_of(faces, 60), cfg, poses_of(scene_of(faces, 60)))


# two bands and more; 45k faces need 1,407 words of bits (beyond an eighth of
# the 10,112-word tile), 170k faces 5,313 (beyond an eighth of the largest)
@pytest.mark.parametrize("cfg,faces", [(0, 9000), (0, 45000), (2, 9000), (2, 45000), (4, 4000), (4, 45000), (0, 170000)])
def test_bands(cfg, faces):
    scene = scene_of(faces, 300)
    check(scene, cfg, poses_of(scene))


@pytest.mark.parametrize("cfg", [0, 2, 4])
@pytest.mark.parametrize("faces,cap", [(1500, 0), (12000, 7001), (60000, 0)])
def test_wide_boxes(cfg, faces, cap):
    scene = scene_of(faces, 120)
    boxes = check(scene, cfg, poses_of(scene, near=True), cap)
    assert max(max(b[1] - b[0], b[3] - b[2]) for b in boxes) > 2046
