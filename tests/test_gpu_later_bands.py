"""What the later bands of a region cost with four waves a workgroup: a mesh
whose faces the later bits hold is not slower than a larger one without them
(a 300 px rect takes about a dozen bands of a 10,112-word tile)."""
import numpy as np
import pytest

import qpso
import workloads as W

pytestmark = pytest.mark.gpu


def launch_ms(ctx, faces):
    z = 700.0
    a = 300 * z / W.CAM[0] / 2.0
    sl, st = W.uv_dims(faces)
    mesh = qpso.mesh_uv_ellipsoid(sl, st, a, a * 0.9, a * 0.7, 2, 0.1 * a, 0.2 * a, 0)
    pose = np.array([4.0, -3.0, z, *qpso.random_quat(60)], np.float32)
    depth, labels = qpso.scene_render([(mesh, pose)], W.CAM, 1300.0, 2.0, 0.05, 6)
    scene = W.Scene([(mesh, pose)], depth, labels)
    c = scene.clusters[0]
    cl = qpso.make_cluster(c["rect"], (0.0, 0.0, z), c["num_points"], c["depth"])
    m = ctx.upload_mesh(scene.mesh_m())
    # one iteration from random orientations at one place
    with ctx.solve(m, cl, qpso.make_params(64, 1, cam=W.CAM, t_bound=0.0, t_bound_z=0.0)) as s:
        ms = min(s.run_timed()[1].ms_render_fitness for _ in range(10))
    ctx.release_mesh(m)
    return ms


def test_fewer_faces_take_less_time():
    # 30k faces: 938 words of bits, 45k: 1,408, over an eighth of the tile.  Drawn
    # by the bits the smaller mesh took 1.02 times the larger one's time, culled
    # from the cache 0.70 times
    with qpso.Context(0) as ctx:
        ctx.set_tuning(4, 96)
        t30, t45 = launch_ms(ctx, 30000), launch_ms(ctx, 45000)
    assert t30 < 0.85 * t45
