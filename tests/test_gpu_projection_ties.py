"""The fast vertex projection where a product of the rotation is denormal and
decides a rounding tie: its box and fitness are the general projection's
(the oracle's), bit for bit.

The quaternion (1, 0, 1 + 2^-23, 2^-100) turns a vertex (0, y, 1.5) to
x = 2 (q2 * 1.5 - q3 * y) with q2 * 1.5 halfway between two floats.  A y of 0.4 *
2^-49 leaves q3 * y below half of the least denormal, so the product is 0 and
the tie goes to the even neighbour; twice that product is not."""
import numpy as np
import pytest

import oracle as O
import qpso
import workloads as W
from helpers import assert_same_f32, assert_same_i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("cfg", [0, 4])
def test_denormal_product_at_a_tie(cfg, swap):
    scene = W.config0()[0]
    c = scene.clusters[0]
    fx, ratio = 2.0 ** 26, 3.0000004768371582 / 6.499999046325684
    mid = (c["rect"][0] + c["rect"][2]) / 2.0
    cam = (fx, 300.0, mid - fx * ratio, 239.5)
    y = 0.4 * 2.0 ** -49
    tri = [(0.0, y, 1.5), (0.0, -0.4, 1.5), (0.0, 0.4, 1.5)]
    if swap:
        tri[1], tri[2] = tri[2], tri[1]
    # one face, x, y and z of its three corners
    mesh = np.array([[v[k] for v in tri] for k in range(3)], np.float32).reshape(-1)
    pose = np.array([[0, 0, 8.0, 1, 0, 1 + 2.0 ** -23, 2.0 ** -100]], np.float32).T
    with qpso.Context(0) as ctx:
        ctx.set_tuning(cfg, 96)
        m = ctx.upload_mesh(mesh)
        with ctx.solve(m, scene.cluster(), qpso.make_params(1, 1, cam=cam)) as s:
            fit, aabb, _ = s.eval_poses(pose)
        ctx.release_mesh(m)
    fr, info = O.render(mesh, pose[:, 0], cam, c["rect"])
    assert not info.degenerate
    # the tie decides which of the two columns the first vertex takes, and with
    # it the way the face looks
    assert info.aabb[1] - info.aabb[0] >= 2
    want, _ = O.fitness(info, c["rect"], c["num_points"], fr, c["depth"])
    assert_same_i32(aabb[0], np.array(info.aabb[:], np.int32), "aabb")
    assert_same_f32(fit, np.array([want], np.float32), "fitness")
