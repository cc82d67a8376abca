"""Performance cases of the pose search: what a program that uses the library
has it do, through the public calls of q-pso_amd/qpso.py.

A case is one object scene (a mesh, a ray-cast depth frame, the object's
cluster) or one frame of several, a swarm size, an iteration count, and the
call that searches it:

  plain    Solve.run of a solve that the program keeps (tuned once)
  traced   the same, with the per-iteration traces and the final swarm read back
  call     Context.estimate_pose, one call per cluster: upload, search, result
  batch    Context.run_batch over the solves of one frame
  serve    every cluster of some frames submitted to the server, then awaited
  score    Solve.eval_poses: fitness and bounding box of given poses
"""
import math
import os
import sys
import weakref

import numpy as np

sys.path.insert(0, os.path.join(os.getcwd(), "q-pso_amd"))

import qpso  # noqa: E402
import workloads as W  # noqa: E402

FACES = (500, 100000)   # meshes of the 16-object frame up to the stress mesh
EXTENT = (40, 320)      # cluster extents in pixels
PARTICLES = (16, 2048)
ITERS = (10, 200)


def listed():
    return [
        # a small tracked object between two frames: 1,280 faces, 32 particles;
        # launches and latency count
        {"name": "plain_1k_n32", "call": "plain", "scene": "small", "faces": 1280, "extent": 60, "n": 32, "iters": 30},
        # the benchmark's headline: one object, 10k faces, a 220 px cluster
        {"name": "plain_10k_n256", "call": "plain", "scene": "head", "faces": 10336, "extent": 220, "n": 256,
         "iters": 100},
        # one object of a served stream searched on its own, 50k faces
        {"name": "plain_50k_n128", "call": "plain", "scene": "object", "faces": 50000, "extent": 100, "n": 128,
         "iters": 60},
        # a search whose convergence the program looks at: traces read back
        {"name": "traced_5k_n64", "call": "traced", "scene": "object", "faces": 5304, "extent": 91, "n": 64,
         "iters": 60},
        # the reference program's own call and defaults (1,024 particles, 20
        # iterations, 3,072-face cap), everything uploaded in the call
        {"name": "call_reference", "call": "call", "scene": "reference", "faces": 10336, "extent": 220, "n": 1024,
         "iters": 20, "cap": 3072},
        # a frame of the served stream without the server: one call per
        # cluster, 1k to 50k faces
        {"name": "call_frame_8", "call": "call", "scene": "stream", "frames": 1, "n": 128, "iters": 60},
        # one 16-object frame (500 to 20,000 faces, 40 to 250 px, 64 to 512
        # particles) in one batch
        {"name": "batch_frame_16", "call": "batch", "scene": "frame", "objects": 16, "iters": 60},
        # eight frames of the stream submitted at once to the server
        {"name": "serve_64", "call": "serve", "scene": "stream", "frames": 8, "n": 128, "iters": 60},
        # the largest search: 100k faces, 2,048 particles, 200 iterations,
        # noisy depth
        {"name": "plain_100k_n2048", "call": "plain", "scene": "stress", "faces": 100000, "extent": 235, "n": 2048,
         "iters": 200},
        # an object cut by the frame edge in the reference-faithful mode
        {"name": "traced_edge_n64", "call": "traced", "scene": "edge", "faces": 1280, "extent": 60, "n": 64,
         "iters": 12},
        # scoring a handful of candidate poses, and a whole swarm of them
        {"name": "score_1k_32", "call": "score", "scene": "small", "faces": 1280, "extent": 60, "n": 32, "iters": 1},
        {"name": "score_10k_512", "call": "score", "scene": "head", "faces": 10336, "extent": 220, "n": 512,
         "iters": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["plain", "plain", "plain", "traced", "call", "call", "batch", "serve", "score", "edge"])
    if call == "batch":
        return {"call": "batch", "scene": "frame", "objects": rng.randint(2, 16), "iters": _log(rng, 20, 100)}
    if call == "serve":
        return {"call": "serve", "scene": "stream", "frames": rng.randint(1, 8), "n": _log(rng, 64, 256),
                "iters": _log(rng, 20, 100)}
    if call == "edge":
        return {"call": "traced", "scene": "edge", "faces": 1280, "extent": 60, "n": _log(rng, 16, 128),
                "iters": _log(rng, 5, 20)}
    while True:
        c = {"call": call, "scene": "object", "faces": _log(rng, *FACES), "extent": _log(rng, *EXTENT),
             "n": _log(rng, *PARTICLES), "iters": 1 if call == "score" else _log(rng, *ITERS)}
        if call == "call" and rng.random() < 0.3:
            c["cap"] = 3072
        # at most a fifth of the largest listed case
        if c["n"] * c["iters"] * _ops(c["faces"], c["extent"]) <= 0.2 * 2048 * 200 * _ops(100000, 235):
            return c


def _ops(faces, extent):
    """Operations of one particle in one iteration: per face the projection of
    its half vertex (45 each) and the facing test (10), for the half that
    faces the camera the edge set-up (40); per cluster pixel a depth (8) and
    the error term (6), the cluster about 0.7 as high as wide."""
    return 52 * faces + 14 * 0.7 * extent * extent


def _stream_sizes():
    return [int(round(math.exp(math.log(1000) + i * math.log(50) / 7))) for i in range(8)]


def _frame_sizes(k):
    """faces, extents (px) and particles of a k-object frame."""
    f = [int(round(500 * 40 ** ((i + 0.5) / k))) for i in range(k)]
    e = [40 * 6.25 ** ((i * 7 % k + 0.5) / k) for i in range(k)]
    # the frame holds 640 x 480 pixels: sixteen such objects fill about half
    return [(f[i], e[i] * min(1.0, 9.0 / k + 0.3), (64, 128, 256, 512)[i * 5 % 4]) for i in range(k)]


def work(case):
    if case["scene"] == "frame":
        jobs = [(f, e, n) for f, e, n in _frame_sizes(case["objects"])]
    elif case["scene"] == "stream":
        jobs = [(f, 65, case["n"]) for f in _stream_sizes()] * case["frames"]
    else:
        jobs = [(case["faces"], case["extent"], case["n"])]
    it, by, ops = case["iters"], 0.0, 0.0
    for f, e, n in jobs:
        f = min(f, case.get("cap", f))
        # mesh, cluster crop; random numbers (or the given poses) in, the
        # result (or every pose's fitness and box) out
        by += 36 * f + 2 * 0.7 * e * e + (48 * n if case["call"] == "score" else 48 * (it + 1) * n + 64)
        ops += n * it * _ops(f, e)
    if case["call"] == "traced":
        by += 4 * it * n + 36 * it + 88 * case["n"]
    return {"bytes": by, "flops": ops}


# ---------------------------------------------------------------- scenes
def _object_scene(seed, faces, extent, sigma=2.0, holes=0.05):
    rng = np.random.default_rng(7000 + seed)
    z = rng.uniform(650.0, 1000.0)
    a = extent * z / W.CAM[0] / 2.0
    sl, st = W.uv_dims(max(12, faces - 24))
    mesh = qpso.mesh_uv_ellipsoid(sl, st, a, a * 0.7, a * 0.5, 2, 0.1 * a, 0.2 * a, seed)
    room = [max(0.0, (px / 2.0 - extent / 2.0 - 8) * z / W.CAM[0]) for px in (640, 480)]
    t = [rng.uniform(-1, 1) * min(100.0, r) for r in room]
    pose = np.array(t + [z] + list(qpso.random_quat(7000 + seed)), np.float32)
    depth, labels = qpso.scene_render([(mesh, pose)], W.CAM, 1300.0, sigma, holes, seed + 6)
    return W.Scene([(mesh, pose)], depth, labels)


def _placed(seed, specs):
    """A frame of (mesh, extent px) objects that do not overlap."""
    rng = np.random.default_rng(9000 + seed)
    k = 1.0
    while True:
        trans = W._place(rng, len(specs), [k * e / 2.0 + 4 for _, e in specs], W.CAM, (600, 1200))
        if trans is not None:
            break
        k *= 0.97
    objects = []
    for i, (make, e) in enumerate(specs):
        mesh = make(k * e * trans[i][2] / W.CAM[0] / 2.0)
        objects.append((mesh, np.array(list(trans[i]) + list(qpso.random_quat(9000 + seed * 31 + i)), np.float32)))
    depth, labels = qpso.scene_render(objects, W.CAM, 1500.0, 2.0, 0.05, seed + 3)
    return W.Scene(objects, depth, labels)


def _frame_scene(seed, k):
    sizes = sorted(_frame_sizes(k), key=lambda s: -s[1])

    def maker(faces, i):
        sl, st = W.uv_dims(max(12, faces - 24))
        return lambda a: qpso.mesh_uv_ellipsoid(sl, st, a, a * 0.7, a * 0.5, 2, 0.1 * a, 0.2 * a, seed * 100 + i)
    return _placed(seed, [(maker(f, i), e) for i, (f, e, _) in enumerate(sizes)]), [n for _, _, n in sizes]


def _params(case):
    return qpso.make_params(case["n"], case["iters"], w=0.7, c1=1.5, c2=1.5, cam=W.CAM, seed=0,
                            face_cap=case.get("cap", 0))


def _one(case, seed):
    """The scene of a one-object case and its solve parameters."""
    kind, n, it = case["scene"], case["n"], case["iters"]
    if kind == "small":
        scene, p = W.config0(seed)
    elif kind == "head":
        scene, p = W.config1(seed)
    elif kind == "reference":
        scene, p = W.reference_config(seed)
    elif kind == "stress":
        scene, p = W.config4(seed)
    elif kind == "edge":
        scene, p = W.edge_config(seed)
    else:
        scene, p = _object_scene(seed, case["faces"], case["extent"]), _params(case)
    p.n_particles, p.n_iters = n, it  # random-table seed 0 throughout, as the reference program
    return scene, p


def _poses(scene, n, seed):
    """Candidate poses around the object's own: half of them close, half
    spread over the search's bounds."""
    rng = np.random.default_rng(11000 + seed)
    gt = scene.objects[0][1].astype(np.float64)
    s = np.where(np.arange(n) % 2 == 0, 0.01, 0.15)
    t = gt[:3, None] * 1e-3 + rng.uniform(-1, 1, (3, n)) * s
    q = gt[3:, None] + rng.normal(0, 1, (4, n)) * np.where(np.arange(n) % 2 == 0, 0.03, 0.7)
    q /= np.linalg.norm(q, axis=0)
    q *= np.where(q[0] < 0, -1.0, 1.0)
    return np.ascontiguousarray(np.concatenate([t, q]), np.float32)


# ---------------------------------------------------------------- what a program keeps
_ctx = None
_server = None  # weak: the server ends with the last state that uses it


def _context():
    global _ctx
    if _ctx is None:
        _ctx = qpso.Context(0)
    return _ctx


class _Served:
    def __init__(self, ctx):
        self.sv = qpso.Server(ctx, 32 << 30)
        self.sv.set_slots(8192)

    def __del__(self):
        self.sv.close()


class State:
    def __init__(self, call):
        self.call, self.ctx, self.meshes, self.solves, self.jobs, self.served = call, _context(), [], [], [], None

    def mesh(self, soa):
        self.meshes.append(self.ctx.upload_mesh(soa))
        return self.meshes[-1]

    def __del__(self):
        self.served = None
        for s in self.solves:
            s.close()
        for m in self.meshes:
            self.ctx.release_mesh(m)


def prepare(case, seed):
    global _server
    st = State(case["call"])
    ctx = st.ctx
    ctx.set_tuning(0, 128)  # a context's own default
    if case["scene"] == "frame":
        scene, ns = _frame_scene(seed, case["objects"])
        for i, n in enumerate(ns):
            if scene.clusters[i] is not None:
                p = _params({"n": n, "iters": case["iters"]})
                st.solves.append(ctx.solve(st.mesh(scene.mesh_m(i)), scene.cluster(i), p))
        ctx.autotune(st.solves, iters=3)
        return st
    if case["scene"] == "stream":
        meshes = W.config3_meshes(0)  # the objects the program knows
        ids = [st.mesh((m * np.float32(1e-3)).astype(np.float32)) for m, _ in meshes]
        for f in range(case["frames"]):
            specs = [(lambda a, m=m: m, 2 * a * W.CAM[0] / 900.0) for m, a in meshes]
            scene = _placed(seed * 100 + f, specs)
            for i, mid in enumerate(ids):
                if scene.clusters[i] is not None:
                    st.jobs.append((mid, scene.cluster(i), _params(case)))
        if case["call"] == "serve":
            sample = [ctx.solve(*j) for j in st.jobs[:16]]
            ctx.autotune(sample, iters=min(20, case["iters"]))
            for s in sample:
                s.close()
            st.served = _server() if _server is not None else None
            if st.served is None:
                st.served = _Served(ctx)
                _server = weakref.ref(st.served)
        return st
    scene, p = _one(case, seed)
    mid = st.mesh(scene.mesh_m())
    if case["call"] == "call":
        st.jobs.append((mid, scene.cluster(), p))
        return st
    st.solves.append(ctx.solve(mid, scene.cluster(), p, trace=case["call"] == "traced"))
    if case["call"] == "score":
        st.poses = _poses(scene, case["n"], seed)
    elif not p.offframe:
        ctx.autotune(st.solves, iters=3)
    return st


def _result(r):
    return {"pose": np.array(r.pose[:], np.float32), "fit": np.float32(r.fit), "raster_px": int(r.raster_px),
            "visit_px": int(r.visit_px), "n_degenerate": int(r.n_degenerate), "status": int(r.status)}


def _stack(rs):
    """The results of several solves, one array per field."""
    return {k: np.array([_result(r)[k] for r in rs]) for k in ("pose", "fit", "raster_px", "visit_px", "status")}


def run(st):
    if st.call == "plain":
        return _result(st.solves[0].run())
    if st.call == "traced":
        r = st.solves[0].run()
        return {"result": _result(r), "trace": st.solves[0].trace()}
    if st.call == "call":
        return _stack([st.ctx.estimate_pose(*j) for j in st.jobs])
    if st.call == "batch":
        return _stack(st.ctx.run_batch(st.solves))
    if st.call == "serve":
        sv = st.served.sv
        return _stack([sv.wait(t) for t in [sv.submit(*j) for j in st.jobs]])
    fit, aabb, _ = st.solves[0].eval_poses(st.poses)
    return {"fit": fit, "aabb": aabb}


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    """Fitness of given poses in 64 bits.  A search has no such value: its
    swarm follows the rounding of every fitness before."""
    if case["call"] != "score" or case["n"] * case["faces"] > 1e6:
        return None
    scene, p = _one(case, seed)
    c, poses = scene.clusters[0], _poses(scene, case["n"], seed).astype(np.float64)
    soa = scene.mesh_m().astype(np.float64).reshape(3, 3, -1)  # [coordinate][corner][face]
    return {"fit": np.array([_fitness(poses[:, i], soa, c, p) for i in range(case["n"])]), "aabb": None}


def _fitness(pose, soa, c, p):
    q0, q = pose[3], pose[4:]
    v = soa.reshape(3, -1)
    t = 2.0 * np.cross(q, v, axis=0)
    w = v + q0 * t + np.cross(q, t, axis=0) + pose[:3, None]
    X = np.rint(16.0 * (p.cam.cx + p.cam.fx * w[0] / w[2])).astype(np.int64).reshape(3, -1)
    Y = np.rint(16.0 * (p.cam.cy + p.cam.fy * w[1] / w[2])).astype(np.int64).reshape(3, -1)
    Z = (1000.0 * w[2]).reshape(3, -1)
    x0, x1, y0, y1 = ((f(a, axis=0) + 15) >> 4 for a, f in ((X, np.min), (X, np.max), (Y, np.min), (Y, np.max)))
    rect = c["rect"]
    bx0, bx1 = min(int(x0.min()), rect[0]), max(int(x1.max()), rect[2])
    by0, by1 = min(int(y0.min()), rect[1]), max(int(y1.max()), rect[3])
    # the depth buffer of the union box: every front-facing face fills its
    # whole bounding box with the depth its edge functions weigh (scaled by
    # 1/16 and 1/256), the smallest rounded depth stays
    buf = np.full((by1 - by0 + 1, bx1 - bx0), 60000.0)
    area = (X[0] - X[1]) * (Y[2] - Y[0]) - (X[2] - X[0]) * (Y[0] - Y[1])
    for f in np.flatnonzero((area > 0) & (x1 > x0) & (y1 > y0)):
        xs, ys = np.arange(x0[f], x1[f]), np.arange(y0[f], y1[f])[:, None]
        w2, w3 = (_edge(X[a, f], Y[a, f], X[b, f], Y[b, f], xs, ys) for a, b in ((1, 2), (2, 0)))
        d = Z[0, f] + w2 * ((Z[1, f] - Z[0, f]) / area[f]) + w3 * ((Z[2, f] - Z[0, f]) / area[f])
        b = buf[y0[f] - by0:y1[f] - by0, x0[f] - bx0:x1[f] - bx0]
        np.minimum(b, np.rint(d), out=b)
    # the scan over t = 0 .. T-1: its row is a product in float32 by definition
    Wb, Hb = bx1 - bx0, by1 - by0
    T = (Wb * Hb + 1023) // 1024 * 1024
    tt = np.arange(T)
    yy = (tt.astype(np.float32) * (np.float32(1) / np.float32(Wb))).astype(np.int64)
    xx = tt % Wb
    px, py = xx + bx0, yy + by0
    ok = (py <= by1) & (px >= 0) & (px < 640) & (py >= 0) & (py < 480)
    zr = buf[yy[ok], xx[ok]]
    zk = c["depth"].astype(np.float64)[py[ok], px[ok]]
    r, o = zr < 60000.0, zk > 0
    n = max(int(r.sum()), 1)
    e = np.where(r & o, (zr - zk) * 0.001, 0.0)
    return 0.05 * ((o & ~r).sum() / c["num_points"] + (r & ~o).sum() / n) + (e * e).sum() / n


def _edge(xa, ya, xb, yb, xs, ys):
    """An edge function at pixels, 28.4 coordinates, with the top-left bias and
    the reference's shifted depth weight (cx + 15) >> 8."""
    dx, dy = xa - xb, ya - yb
    cy = dy * xa - dx * ya + (1 if dy < 0 or (dy == 0 and dx > 0) else 0)
    return (cy + dx * 16 * ys - dy * 16 * xs + 15) >> 8
