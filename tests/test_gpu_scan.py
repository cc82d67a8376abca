"""The fitness scan's pairs of consecutive pixels: rects whose left edge lies
on, just left and just right of the rendered box's (the union box's first
column, where the fp32 row index skips and doubles pixels, inside the scanned
region or not), odd and even widths from one pixel up, quirk widths, and the
frame's right and bottom edges; every tile configuration, bit-exact against
the oracle."""
import numpy as np
import pytest

import oracle as O
import qpso
import workloads as W
from helpers import assert_same_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4])
def test_scan_pairs_at_rect_edges(cfg):
    scene, params = W.config0(0)
    params.n_particles = 6
    gt = scene.objects[0][1]
    rng = np.random.default_rng(3)
    poses = np.zeros((7, 6), np.float32)
    for i in range(6):
        poses[:3, i] = gt[:3] * 1e-3 + rng.normal(0, 0.004, 3) * (i > 0)
        q = gt[3:] + rng.normal(0, 0.05, 4) * (i > 0)
        poses[3:, i] = q / np.linalg.norm(q)
    cam = (params.cam.fx, params.cam.fy, params.cam.cx, params.cam.cy)
    mesh = scene.mesh_m()
    depth = np.asarray(scene.depth, np.uint16)
    c0 = scene.clusters[0]["rect"]
    boxes = [list(O.render(mesh, poses[:, i], cam, c0)[1].aabb) for i in range(6)]
    ax0, ax1, ay0, ay1 = boxes[0]
    rects = []
    for d in (-2, -1, 0, 1, 2, 3):            # left edge around the box's
        for w in (1, 2, 3, 40, 41):
            rects.append([ax0 + d, ay0 + 5, ax0 + d + w, ay1 - 3])
    for w in (121, 123, 242):                 # widths with short rows, the box inside
        rects.append([ax0, ay0 - 7, ax0 + w, ay1 + 9])
    rects += [[ax0, ay0, ax0 + 1, ay0 + 1], [ax0, ay1 - 1, ax1, ay1], [0, 0, 640, 480],
              [ax0, ay0, 640, ay1], [ax0, ay0, ax1, 480], [ax1 - 1, ay0, ax1 + 4, ay1]]
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 128)
        mid = ctx.upload_mesh(mesh)
        for rect in rects:
            assert 0 <= rect[0] < rect[2] <= 640 and 0 <= rect[1] < rect[3] <= 480
            crop = np.zeros_like(depth)
            crop[rect[1]:rect[3], rect[0]:rect[2]] = depth[rect[1]:rect[3], rect[0]:rect[2]]
            with ctx.solve(mid, qpso.make_cluster(rect, scene.clusters[0]["centroid_mm"], 77, crop), params) as s:
                fit, _, _ = s.eval_poses(poses)
            want = []
            for i in range(6):
                fr, info = O.render(mesh, poses[:, i], cam, rect)
                want.append(O.fitness(info, rect, 77, fr, crop)[0])
            assert_same_f32(fit, np.array(want, np.float32), f"fitness, rect {rect}")
        ctx.release_mesh(mid)
