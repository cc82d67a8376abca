"""The PSO step inside the render launches and over several workgroups (plain
solves, two buffers) against the step as one workgroup per solve (batched
form, pinned against the oracle elsewhere): swarm sizes around a wave, a
workgroup, the number of CUs and the largest with two buffers; odd and even
iteration counts; a swarm without a single valid fitness."""
import numpy as np
import pytest

import qpso
import workloads as W

pytestmark = pytest.mark.gpu


def same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


def run_both(n, iters, centroid=None):
    scene, params = W.config0(0)
    params.n_particles, params.n_iters, params.seed = n, iters, 5
    c = scene.clusters[0]
    cl = qpso.make_cluster(c["rect"], centroid or c["centroid_mm"], c["num_points"], c["depth"])
    with qpso.Context(0) as ctx:
        mid = ctx.upload_mesh(scene.mesh_m())
        with ctx.solve(mid, cl, params, trace=True) as s:
            plain = s.run()
            t_plain = s.trace()
            batch = ctx.run_batch([s])[0]
            t_batch = s.trace()
            again = s.run()
            t_again = s.trace()
        once = ctx.estimate_pose(mid, cl, params)
        ctx.release_mesh(mid)
    for r in (batch, again, once):
        assert list(r.pose) == list(plain.pose) and (r.raster_px, r.visit_px) == (plain.raster_px, plain.visit_px)
        assert np.float32(r.fit).view(np.uint32) == np.float32(plain.fit).view(np.uint32)
    same(t_plain, t_batch)
    same(t_plain, t_again)
    return plain, t_plain


@pytest.mark.parametrize("iters", [1, 2, 5])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 511, 513, 4096, 4097])
def test_plain_equals_batched(n, iters):
    run_both(n, iters)


@pytest.mark.parametrize("n", [5, 300])
def test_behind_camera(n):
    # mirrored boxes that start far off the rect
    run_both(n, 3, centroid=[0.0, 0.0, -5000.0])


@pytest.mark.parametrize("n", [5, 300])
def test_no_valid_fitness(n):
    # a thousand kilometres off: every coordinate beyond the fixed-point range, every
    # fitness NaN, no best ever found
    r, t = run_both(n, 3, centroid=[1e9, 0.0, 800.0])
    assert np.isnan(t["fit_trace"]).all() and (t["argmin_trace"] == 0).all()
    assert r.fit == np.float32(1e10)
