"""Performance cases: the calls that programs built on this package make, over
the range of sizes and options they use.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) what a program holds before the call, on the GPU
run(state)          one pass through the public classes, and its outputs
work(case)          bytes and operations one pass cannot do without
exact(case, seed)   the outputs in 64 bits (plain numpy / torch), where they
                    have such a value

Kinds of case:
  frame   Session.process_frame: one live frame of one camera (track, integrate,
          raycast), the latency a robot or a hand-held scanner sees.
  serve   Server.run: whole short reconstructions of many cameras, batched.
  fuse    TsdfVolume.IntegrateScan with known poses and a rendered view of the
          result (motion capture, replay of a recorded trajectory).
  render  TsdfVolume.Raycast: depth, vertices, normals and colour of a finished map.
  mesh    MeshExtractor.ExtractMesh: marching cubes of a finished map, as many
          triangles as the program's mesh holds (the rooms have more).
  track   Session.source_maps and icp_track: tracking alone against given model
          maps (gnSolver::solve's use).
  filter  bilateral_filter and depth_pyramid of a raw depth image.
  graph   DefGraph from a mesh, its neighbours, and one blended mesh: the start of
          a non-rigid tracking.
  warp    NonRigidICP.solve (one graph) or NonRigidBatch.solve (several), then the
          warped mesh: one live frame of a deforming object.
"""
import math

import numpy as np
import torch

import dynamap_amd as dm
from dynamap_amd import _native as N
from dynamap_amd import configs


def listed():
    return [
        # the smallest live camera of the workloads: launch and wait latency count most
        dict(name="frame-320x240-2cm", kind="frame", rows=240, cols=320, voxel_mm=20.0, rgb=False, filt=0, frames=12),
        # the reference's default camera, photometric term and the depth filter on
        dict(name="frame-640x480-8mm", kind="frame", rows=480, cols=640, voxel_mm=8.0, rgb=True, filt=3, frames=12),
        # the benchmark's serving mix, from fresh sessions to their 16th frame
        dict(name="serve-16", kind="serve", n2cm=8, n8mm=8, frames=16),
        # the large multi-room map at its finest voxel size, poses known
        dict(name="fuse-640x480-4mm", kind="fuse", rows=480, cols=640, voxel_mm=4.0, scene=5, rgb=True, frames=4),
        # a view of a finished map at a ragged image size
        dict(name="render-421x517-8mm", kind="render", rows=421, cols=517, voxel_mm=8.0, scene=1, rgb=True, frames=10),
        # preview mesh of a part of a coarse map
        dict(name="mesh-2cm-box", kind="mesh", rows=240, cols=320, voxel_mm=20.0, scene=1, rgb=False, frames=10,
             box=1.1, triangles=12000),
        # the benchmark's mesh: every block of an 8 mm room (about 240 000 triangles are there)
        dict(name="mesh-8mm", kind="mesh", rows=480, cols=640, voxel_mm=8.0, scene=1, rgb=True, frames=30, box=0.0,
             triangles=180000),
        # tracking alone, both residual terms
        dict(name="track-640x480", kind="track", rows=480, cols=640, rgb=True),
        # depth preprocessing of a VGA frame
        dict(name="filter-640x480", kind="filter", rows=480, cols=640, radius=3, levels=3),
        # the deformation graph of the 200k-vertex cylinder at its 4048 nodes
        dict(name="graph-200k", kind="graph", n_theta=500, n_y=400, radius_mm=13.3, dgw_mm=25.0),
        # one deforming object per frame at that graph
        dict(name="warp-4048", kind="warp", n_theta=500, n_y=400, radius_mm=13.3, dgw_mm=25.0, graphs=1, rows=480,
             cols=640, gn=5, pcg=40),
        # several smaller objects at once, 2.5 cm grid
        dict(name="warp-batch-4", kind="warp", n_theta=300, n_y=240, radius_mm=25.0, dgw_mm=50.0, graphs=4, rows=480,
             cols=640, gn=5, pcg=40),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo=100, hi=480):
    rows = int(_log(rng, lo, hi))
    return rows, int(rows * rng.uniform(1.15, 1.4))


def draw(rng):
    kind = rng.choice(["frame", "frame", "serve", "fuse", "render", "mesh", "track", "filter", "graph", "warp"])
    if kind == "frame":
        r, c = _size(rng)
        return dict(kind=kind, rows=r, cols=c, voxel_mm=round(_log(rng, 8, 25), 2), rgb=rng.random() < 0.5,
                    filt=rng.choice([0, 0, 2, 3, 5]), frames=rng.randint(6, 12))
    if kind == "serve":
        a = rng.randint(0, 8)
        return dict(kind=kind, n2cm=a, n8mm=rng.randint(0 if a else 1, 7), frames=rng.randint(5, 15))
    if kind == "fuse":
        r, c = _size(rng)
        return dict(kind=kind, rows=r, cols=c, voxel_mm=round(_log(rng, 4, 20), 2), scene=rng.choice([1, 5]),
                    rgb=rng.random() < 0.7, frames=rng.randint(2, 5))
    if kind == "render":
        r, c = _size(rng)
        return dict(kind=kind, rows=r, cols=c, voxel_mm=round(_log(rng, 5, 25), 2), scene=rng.choice([1, 5]),
                    rgb=rng.random() < 0.5, frames=rng.randint(3, 10))
    if kind == "mesh":
        r, c = _size(rng, 160, 480)
        voxel = round(_log(rng, 8, 25), 2)
        return dict(kind=kind, rows=r, cols=c, voxel_mm=voxel, scene=1, rgb=rng.random() < 0.5,
                    frames=rng.randint(3, 20), box=rng.choice([0.0, 0.0, round(rng.uniform(1.0, 1.5), 3)]),
                    triangles=int(75000 * (8.0 / voxel) ** 2))
    if kind == "track":
        r, c = _size(rng)
        return dict(kind=kind, rows=r, cols=c, rgb=rng.random() < 0.6)
    if kind == "filter":
        r, c = _size(rng, 90, 720)
        return dict(kind=kind, rows=r, cols=c, radius=rng.randint(1, 7), levels=rng.randint(2, 5))
    mesh = dict(n_theta=int(_log(rng, 120, 500)), n_y=int(_log(rng, 100, 400)))
    radius = round(_log(rng, 13.3, 40), 2)
    if kind == "graph":
        return dict(kind=kind, radius_mm=radius, dgw_mm=round(2 * radius, 2), **mesh)
    r, c = _size(rng, 200, 480)
    return dict(kind=kind, radius_mm=max(radius, 15.0), dgw_mm=round(2 * radius, 2), graphs=rng.choice([1, 1, 2, 3]),
                rows=r, cols=c, gn=rng.randint(2, 5), pcg=rng.randint(10, 40), **mesh)


# ------------------------------------------------------------------ inputs
def _seed(seed, salt):
    return (configs.SEED_BASE + 7919 * int(seed) + 104729 * salt) & 0x7fffffffffff


def _sensor(rows, cols):
    """Field of view of the workloads' cameras (fx = 262.5 at 320 columns)."""
    f = cols * 262.5 / 320.0
    return dict(rows=rows, cols=cols, fx=f, fy=f, cx=(cols - 1) / 2.0, cy=(rows - 1) / 2.0)


def _tsdf(voxel_mm, scene=1):
    """The workloads' tables at their own voxel sizes; between them a pool for
    twice the scene's volume."""
    named = {20.0: configs.TSDF_2CM, 8.0: configs.TSDF_8MM, 4.0: configs.TSDF_4MM}
    if voxel_mm in named:
        return dict(named[voxel_mm])
    vs = voxel_mm / 1000.0
    volume = 36.0 if scene == 1 else 192.0
    pool = 1 << 13
    while pool < min(2.0 * volume / (8 * vs) ** 3, 1 << 20):
        pool <<= 1
    return dict(configs.TSDF_8MM, voxel_size=vs, num_blocks=pool, num_buckets=4 * pool,
                truncation_distance=max(3.0 * vs, 0.02))


def _sequence(scene, sensor, n, seed, rgb):
    """n frames of a seeded room along a seeded trajectory, with sensor noise."""
    sc = configs.Scene(scene, _seed(seed, 1))
    poses = sc.trajectory(n, _seed(seed, 2))
    frames = [sc.render(poses[f], sensor, _seed(seed, 3) + f, noise=True, rgb=True) for f in range(n)]
    return [d for d, _ in frames], [c if rgb else None for _, c in frames], poses


def _turn(state):
    """The next frame of a sequence played forwards and backwards in turn."""
    n = state["n"]
    k = state["k"] % max(1, 2 * n - 2)
    state["k"] += 1
    return k if k < n else 2 * n - 2 - k


def _cylinder(case):
    V = np.zeros((case["n_theta"] * case["n_y"], 3), np.float32)
    Nn = np.zeros_like(V)
    N.synth().dms_cylinder_mesh(case["n_theta"], case["n_y"], N.ptr(V), N.ptr(Nn))
    return V, Nn


def _graph_inputs(case, seed):
    """The mesh, jittered by 0.2 mm (no two graphs alike), and a smooth field
    of small rigid motions evaluated at its nodes."""
    V, Nn = _cylinder(case)
    rng = np.random.default_rng(_seed(seed, 4))
    V = (V + rng.uniform(-2e-4, 2e-4, V.shape)).astype(np.float32)
    return V, Nn, rng.uniform(0.5, 1.5, 6)


def _field(P, a):
    """Rigid motions at points P (n,3): rotations up to ~0.2 rad, 5 cm shifts."""
    w = 0.12 * np.stack([np.sin(4 * a[0] * P[:, 1]), np.cos(3 * a[1] * P[:, 0]), np.sin(5 * a[2] * P[:, 2])], 1)
    t = 0.03 * np.stack([np.cos(4 * a[3] * P[:, 1]), np.sin(3 * a[4] * P[:, 0]), np.cos(5 * a[5] * P[:, 2])], 1)
    th = np.linalg.norm(w, axis=1)[:, None, None]
    K = np.zeros((len(P), 3, 3))
    K[:, 0, 1], K[:, 0, 2], K[:, 1, 2] = -w[:, 2], w[:, 1], -w[:, 0]
    K -= K.transpose(0, 2, 1)
    T = np.tile(np.eye(4), (len(P), 1, 1))
    T[:, :3, :3] += np.sinc(th / np.pi) * K + 0.5 * np.sinc(th / (2 * np.pi)) ** 2 * (K @ K)
    T[:, :3, 3] = t
    return T


def _track_inputs(case, seed):
    """A noisy live frame, the noise-free maps of the pose before it at the
    three pyramid levels."""
    s = _sensor(case["rows"], case["cols"])
    sc = configs.Scene(1, _seed(seed, 1))
    poses = sc.trajectory(2, _seed(seed, 2))
    depth, rgb = sc.render(poses[1], s, _seed(seed, 3), noise=True, rgb=True)
    md, mc = sc.render(poses[0], s, 0, noise=False, rgb=True)
    maps = []
    for l in range(3):
        r, c = s["rows"] >> l, s["cols"] >> l
        k = 1 << l
        d = md[::k, ::k][:r, :c].astype(np.float64)
        i = (mc[::k, ::k][:r, :c].astype(np.float64) @ [0.2126, 0.7152, 0.0722]) / 255.0
        u, v = np.meshgrid(np.arange(c), np.arange(r))
        P = np.stack([(u - s["cx"] / k) * d / (s["fx"] / k), (v - s["cy"] / k) * d / (s["fy"] / k), d], -1)
        n = np.full_like(P, np.nan)
        g = np.cross(P[1:-1, 2:] - P[1:-1, :-2], P[2:, 1:-1] - P[:-2, 1:-1])
        with np.errstate(invalid="ignore", divide="ignore"):
            n[1:-1, 1:-1] = g / np.linalg.norm(g, axis=-1, keepdims=True)
        n[d <= 0] = np.nan
        maps.append((P.astype(np.float32), n.astype(np.float32), i.astype(np.float32)))
    return s, depth, (rgb if case["rgb"] else None), maps


def _icp(case):
    return configs.ICP_RGBD if case["rgb"] else configs.ICP_DEPTH


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_frame(case, seed):
    s = _sensor(case["rows"], case["cols"])
    depth, rgb, poses = _sequence(1, s, case["frames"], seed, case["rgb"])
    ses = dm.Session(_tsdf(case["voxel_mm"]), _icp(case), s, poses[0])
    ses.set_depth_filter(case["filt"])
    for k in range(case["frames"]):  # the map of the room is there
        ses.process_frame(depth[k], rgb[k])
    return dict(kind="frame", session=ses, depth=depth[::-1], rgb=rgb[::-1], n=case["frames"], k=1)


def _prepare_serve(case, seed):
    names = ["rigid-320x240-2cm"] * case["n2cm"] + ["rigid-640x480-8mm"] * case["n8mm"]
    srv = dm.Server(len(names), 480, 640, hbm_budget_bytes=64 << 30)
    for j, name in enumerate(names):
        w = configs.WORKLOADS[name]
        depth, rgb, poses = _sequence(1, w["sensor"], case["frames"], 64 * seed + j, w["rgb"])
        srv.add_trace(w["tsdf"], w["icp"], w["sensor"], poses[0], np.stack(depth), np.stack(rgb) if w["rgb"] else None)
    return dict(kind="serve", server=srv, frames=case["frames"])


def _volume(case, seed):
    s = _sensor(case["rows"], case["cols"])
    depth, rgb, poses = _sequence(case["scene"], s, case["frames"], seed, case["rgb"])
    vol = dm.TsdfVolume(_tsdf(case["voxel_mm"], case["scene"]), s["rows"], s["cols"])
    for f in range(case["frames"]):
        vol.IntegrateScan(depth[f], rgb[f], s, poses[f].astype(np.float32))
    return s, depth, rgb, poses, vol


def _prepare_fuse(case, seed):
    s, depth, rgb, poses, vol = _volume(case, seed)
    return dict(kind="fuse", volume=vol, sensor=s, depth=depth, rgb=rgb, poses=poses.astype(np.float32),
                n=case["frames"], k=0)


def _prepare_render(case, seed):
    s, _, _, poses, vol = _volume(case, seed)
    view = poses[case["frames"] // 2].copy()
    view[:3, 3] += [0.05, -0.03, -0.08]  # a view that no camera frame had
    return dict(kind="render", volume=vol, sensor=s, pose=view.astype(np.float32))


def _prepare_mesh(case, seed):
    s, depth, _, poses, vol = _volume(case, seed)
    box = None
    if case["box"] > 0:  # around the point that the middle of the first frame sees
        v, u = s["rows"] // 2, s["cols"] // 2
        d = float(np.median(depth[0][v - 8:v + 9, u - 8:u + 9]))
        c = poses[0][:3, :3] @ [(u - s["cx"]) / s["fx"] * d, (v - s["cy"]) / s["fy"] * d, d] + poses[0][:3, 3]
        box = (c - case["box"], c + case["box"])
    return dict(kind="mesh", volume=vol, extractor=dm.MeshExtractor(case["triangles"]), box=box)


def _prepare_track(case, seed):
    s, depth, rgb, maps = _track_inputs(case, seed)
    ses = dm.Session(dict(configs.TSDF_2CM), _icp(case), s, np.eye(4))
    for l, m in enumerate(maps):
        ses.set_model_maps(l, *m)
    return dict(kind="track", session=ses, depth=depth, rgb=rgb)


def _prepare_filter(case, seed):
    s = _sensor(case["rows"], case["cols"])
    depth, _, _ = _sequence(1, s, 1, seed, False)
    return dict(kind="filter", depth=depth[0], radius=case["radius"], levels=case["levels"])


def _prepare_graph(case, seed):
    V, Nn, a = _graph_inputs(case, seed)
    return dict(kind="graph", vertices=V, normals=Nn, a=a, radius=case["radius_mm"] / 1000.0,
                dgw=case["dgw_mm"] / 1000.0)


def _prepare_warp(case, seed):
    V, Nn = _cylinder(case)
    s = dict(_sensor(case["rows"], case["cols"]))
    S = N.synth()
    n, K = 6, case["graphs"]
    poses = np.zeros((n, 4, 4))
    S.dms_cylinder_trajectory(n, _seed(seed, 5), N.ptr(poses))
    frames = [np.zeros((s["rows"], s["cols"]), np.float32) for _ in range(n)]
    for f in range(n):
        S.dms_cylinder_render(float(f), N.ptr(poses[f].copy()), s["rows"], s["cols"], s["fx"], s["fy"], s["cx"],
                              s["cy"], _seed(seed, 6) + f, 1, N.ptr(frames[f]))
    gs = [dm.DefGraph(V, Nn, case["radius_mm"] / 1000.0, case["dgw_mm"] / 1000.0, max_nodes=8192) for _ in range(K)]
    solver = dm.NonRigidICP(gn_iterations=case["gn"], pcg_iterations=case["pcg"])
    return dict(kind="warp", graphs=gs, solver=solver, batch=solver.batch(gs) if K > 1 else None, sensor=s,
                frames=frames, poses=poses, n=n, k=0)


_PREPARE = dict(frame=_prepare_frame, serve=_prepare_serve, fuse=_prepare_fuse, render=_prepare_render,
                mesh=_prepare_mesh, track=_prepare_track, filter=_prepare_filter, graph=_prepare_graph,
                warp=_prepare_warp)


# ------------------------------------------------------------------ run
def run(state):
    return _RUN[state["kind"]](state)


def _run_frame(st):
    f = _turn(st)
    pose = st["session"].process_frame(st["depth"][f], st["rgb"][f])
    return dict(pose=pose, increment=st["session"].icp_increment())


def _run_serve(st):
    return st["server"].run(N.DM_RUN_BATCHED, 0, st["frames"], want_poses=True)["poses"]


def _run_fuse(st):
    f = _turn(st)
    vol = st["volume"]
    vol.IntegrateScan(st["depth"][f], st["rgb"][f], st["sensor"], st["poses"][f])
    depth, vertex, normal, rgb = vol.Raycast(st["poses"][f], st["sensor"])
    return dict(depth=depth, vertex=vertex, normal=normal, rgb=rgb, blocks=vol.GetNumAllocatedBlocks())


def _run_render(st):
    depth, vertex, normal, rgb = st["volume"].Raycast(st["pose"], st["sensor"])
    return dict(depth=depth, vertex=vertex, normal=normal, rgb=rgb)


def _run_mesh(st):
    m = st["extractor"].ExtractMesh(st["volume"], *(st["box"] or (None, None)))
    return dict(triangles=m.triangles, colors=m.colors, edges=m.edge_ids.view(np.int64), count=m.num_triangles_)


def _run_track(st):
    v, n, i = st["session"].source_maps(st["depth"], st["rgb"], 0)
    return dict(vertex=v, normal=n, intensity=i, increment=st["session"].icp_track())


def _run_filter(st):
    smooth = dm.bilateral_filter(st["depth"], st["radius"])
    return dict(smooth=smooth, pyramid=dm.depth_pyramid(st["depth"], levels=st["levels"]))


def _run_graph(st):
    g = dm.DefGraph(st["vertices"], st["normals"], st["radius"], st["dgw"], max_nodes=8192)
    vid, nbr, nbr_w = g.nodes()
    ids, w = g.vertex_neighbours()
    g.set_transforms(_field(st["vertices"][vid].astype(np.float64), st["a"]))
    v, n = dm.DqBlender(g).blendMesh()
    return dict(node_vertices=vid, node_neighbours=nbr, node_weights=nbr_w, neighbours=ids, weights=w, vertices=v,
                normals=n, blocks=g.num_blocks())


def _run_warp(st):
    f = _turn(st)
    gs, n = st["graphs"], st["n"]
    if st["batch"] is None:
        stats = [st["solver"].solve(gs[0], st["frames"][f], st["sensor"], st["poses"][f])]
    else:
        pick = [(f + j) % n for j in range(len(gs))]
        stats = st["batch"].solve([st["frames"][i] for i in pick], st["sensor"], [st["poses"][i] for i in pick])
    out = []
    for g in gs:
        v, nr = dm.DqBlender(g).blendMesh()
        out.append(dict(transforms=g.transforms(), vertices=v, normals=nr))
    return dict(graphs=out, residuals=[s["residuals"] for s in stats])


_RUN = dict(frame=_run_frame, serve=_run_serve, fuse=_run_fuse, render=_run_render, mesh=_run_mesh, track=_run_track,
            filter=_run_filter, graph=_run_graph, warp=_run_warp)


# ------------------------------------------------------------------ work
def _visible(rows, cols, voxel_mm):
    """Blocks a frame of the room touches: the frustum from the camera to
    walls about 2 m away, filled with blocks of 8 voxels."""
    fov = (320.0 / 262.5) * (rows / cols * 320.0 / 262.5)
    return fov * 2.0 ** 3 / 3.0 / (8e-3 * voxel_mm) ** 3


def _frame_work(rows, cols, voxel_mm, rgb, track):
    """depth (and colour) read, the frustum's voxels read and written, the
    model maps written; tracking: about 6 linearisations over 64 B a pixel at
    the three levels' sizes."""
    P, B = rows * cols, _visible(rows, cols, voxel_mm)
    byts = P * (4 + (3 if rgb else 0)) + B * 512 * 8 * 2 + P * 31
    flops = B * 512 * 60 + P * 400
    if track:
        byts += 6 * 64 * P * 0.3
        flops += 6 * 250 * P * 0.3
    return byts, flops


def work(case):
    k = case["kind"]
    if k == "frame":
        b, f = _frame_work(case["rows"], case["cols"], case["voxel_mm"], case["rgb"], True)
        if case["filt"]:
            P = case["rows"] * case["cols"]
            b, f = b + 8 * P, f + 12 * P * (2 * case["filt"] + 1) ** 2
    elif k == "serve":
        a, c = _frame_work(240, 320, 20.0, False, True), _frame_work(480, 640, 8.0, True, True)
        b, f = (case["frames"] * (case["n2cm"] * a[i] + case["n8mm"] * c[i]) for i in (0, 1))
    elif k == "fuse":
        b, f = _frame_work(case["rows"], case["cols"], case["voxel_mm"], case["rgb"], False)
    elif k == "render":
        P = case["rows"] * case["cols"]
        b, f = P * 31 + _visible(case["rows"], case["cols"], case["voxel_mm"]) * 512 * 4 * 0.2, P * 1500
    elif k == "mesh":
        # voxels of the room's blocks read, triangles of 96 B written
        blocks = _visible(case["rows"], case["cols"], case["voxel_mm"]) * 1.3
        b, f = blocks * 512 * 8 + case["triangles"] * 96, blocks * 512 * 30
    elif k == "track":
        P = case["rows"] * case["cols"]
        b, f = P * (4 + (3 if case["rgb"] else 0)) + P * 1.31 * 32 + P * 28 + 6 * 64 * P * 0.3, P * 900
    elif k == "filter":
        P = case["rows"] * case["cols"]
        b, f = P * 4 * (2 + 1 + 4 / 3), P * (12 * (2 * case["radius"] + 1) ** 2 + 50)
    else:
        nv = case["n_theta"] * case["n_y"]
        nodes = 2 * math.pi * 0.15 * 0.6 / (case["radius_mm"] / 1000.0) ** 2 * 1.2
        if k == "graph":
            b, f = nv * (24 + 32 + 24) + nodes * (20 + 128), nv * 30 * 9 + nv * 150
        else:
            blocks = 7 * nodes
            it = (2 * blocks - nodes) * (36 * 4 + 8) + 6 * nodes * 8 * 18 + 36 * nodes * 8
            lin = nv * (24 + 32 + 32) + nv * 10 * 12 + blocks * 144
            P = case["rows"] * case["cols"]
            b = case["graphs"] * (P * 4 + case["gn"] * (lin + case["pcg"] * it) + nv * 24 + nodes * 128)
            f = case["graphs"] * case["gn"] * (nv * (400 + 10 * 72) + case["pcg"] * 2 * blocks * 72)
    return dict(bytes=float(b), flops=float(f))


# ------------------------------------------------------------------ exact
def exact(case, seed):
    """In 64 bits: tracking, depth filters, neighbour weights and blending.
    None for the others: a rendered view, a mesh or a pose after integration
    follows from which voxel and which pixel single-precision rounding picks
    (the volume's own definition), and the sliding motions of a deforming
    surface are not observable, so they have no value of their own."""
    f = dict(track=_exact_track, filter=_exact_filter, graph=_exact_graph).get(case["kind"])
    return None if f is None else f(case, seed)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _f64(x):
    return torch.as_tensor(np.asarray(x), dtype=torch.float64, device=_dev())


def _source_maps(depth, rgb, s, level):
    """Vertex, normal (NaN where undefined) and intensity of one pyramid level."""
    k, r, c = 1 << level, s["rows"] >> level, s["cols"] >> level
    d = _f64(depth[::k, ::k][:r, :c])
    fx, fy, cx, cy = (float(np.float32(s[q])) / k for q in ("fx", "fy", "cx", "cy"))
    u = torch.arange(c, device=d.device, dtype=torch.float64)[None]
    v = torch.arange(r, device=d.device, dtype=torch.float64)[:, None]
    P = torch.stack([(u - cx) * d / fx, (v - cy) * d / fy, d], -1)
    P[~(d > 0)] = 0.0
    F = P.reshape(-1, 3)
    i = torch.arange(r * c, device=d.device)
    n = r * c
    L, R = torch.where(i - 2 < 0, i, i - 2), torch.where(i + 2 >= n, i, i + 2)
    U, D = torch.where(i - c <= 0, i, i - c), torch.where(i + c >= n, i, i + c)
    g = torch.linalg.cross(F[R] - F[L], F[D] - F[U])
    nn = g / torch.linalg.norm(g, dim=1, keepdim=True)
    bad = (F[L, 2] == 0) | (F[R, 2] == 0) | (F[U, 2] == 0) | (F[D, 2] == 0) | (F[:, 2] == 0)
    nn[bad] = float("nan")
    if rgb is None:
        it = torch.zeros(r, c, dtype=torch.float64, device=d.device)
    else:
        it = (_f64(rgb[::k, ::k][:r, :c]) * _f64([0.2126, 0.7152, 0.0722])).sum(-1) / 255.0
    return P, nn.reshape(r, c, 3), it


def _se3(xi):
    w, t = xi[:3], xi[3:]
    K = np.array([[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]])
    th = np.linalg.norm(w)
    if th < 1e-5:
        a, b, c = 1 - th ** 2 / 6, 0.5 - th ** 2 / 24, 1 / 6 - th ** 2 / 120
    else:
        a, b, c = np.sin(th) / th, (1 - np.cos(th)) / th ** 2, (th - np.sin(th)) / th ** 3
    T = np.eye(4)
    T[:3, :3] += a * K + b * K @ K
    T[:3, 3] = (np.eye(3) + b * K + c * K @ K) @ t
    return T


def _icp_system(p, n, it, model, s, T, pr):
    """A = sum J J^T and b = sum J r of one linearisation at increment T."""
    r, c = s["rows"], s["cols"]
    Q, NT, mi = model
    T = _f64(T)
    dmin, dmax, dist = (float(np.float32(pr[q])) for q in ("min_depth", "max_depth", "dist_max"))
    usable = lambda a: torch.isfinite(a).all(-1) & (a != 0).any(-1)  # noqa: E731
    ok = (p[:, 2] >= dmin) & (p[:, 2] <= dmax) & usable(n)
    p, n, it = p[ok], n[ok], it[ok]
    x = p @ T[:3, :3].T + T[:3, 3]
    away = lambda a: torch.trunc(a + torch.copysign(torch.full_like(a, 0.5), a))  # noqa: E731
    u = away(s["fx"] * x[:, 0] / x[:, 2] + s["cx"])
    v = away(s["fy"] * x[:, 1] / x[:, 2] + s["cy"])
    ok = (u >= 0) & (v >= 0) & (u < c) & (v < r)
    x, n, it, u, v = x[ok], n[ok], it[ok], u[ok].long(), v[ok].long()
    j = v * c + u
    q, nt = Q[j], NT[j]
    ok = (q[:, 2] >= dmin) & (q[:, 2] <= dmax) & usable(nt)
    ok &= ((n @ T[:3, :3].T * nt).sum(1).abs() > math.cos(math.pi / 10)) & (torch.linalg.norm(x - q, dim=1) <= dist)
    x, q, nt, it, u, v, j = x[ok], q[ok], nt[ok], it[ok], u[ok], v[ok], j[ok]
    J = torch.cat([torch.linalg.cross(x, nt), nt], 1)
    res = ((x - q) * nt).sum(1)
    A, b = J.T @ J, J.T @ res
    wp = float(np.float32(pr["photo_weight"]))
    if wp > 0:
        ok = (u >= 1) & (v >= 1) & (u < c - 1) & (v < r - 1)
        x, it, j = x[ok], it[ok], j[ok]
        gx, gy = (mi[j + 1] - mi[j - 1]) / 2, (mi[j + c] - mi[j - c]) / 2
        z = 1 / x[:, 2]
        G = torch.stack([gx * s["fx"] * z, gy * s["fy"] * z,
                         -(gx * s["fx"] * x[:, 0] + gy * s["fy"] * x[:, 1]) * z * z], 1)
        Jp = torch.cat([torch.linalg.cross(x, G), G], 1)
        A, b = A + wp * Jp.T @ Jp, b + wp * Jp.T @ (mi[j] - it)
    return A.cpu().numpy(), b.cpu().numpy()


def _exact_track(case, seed):
    s, depth, rgb, maps = _track_inputs(case, seed)
    pr = _icp(case)
    T, acc, prev = np.eye(4), np.zeros(6), np.zeros(6)
    for l in (2, 1, 0):
        P, n, it = (a.reshape(-1, 3) if a.dim() == 3 else a.reshape(-1) for a in _source_maps(depth, rgb, s, l))
        model = tuple(_f64(m).reshape(-1, 3) if m.ndim == 3 else _f64(m).reshape(-1) for m in maps[l])
        sl = {q: float(np.float32(s[q])) / (1 << l) for q in ("fx", "fy", "cx", "cy")}
        sl.update(rows=s["rows"] >> l, cols=s["cols"] >> l)
        for k in range(1, pr["lvl_iterations"][l] + 1):
            A, b = _icp_system(P, n, it, model, sl, T, pr)
            sc = 1 / A.max()
            lam = float(np.float32(pr["regularization"])) * (A * sc).max() / k
            xi = np.linalg.solve(A * sc + lam * np.eye(6), -b * sc)
            T, acc = _se3(xi) @ T, acc + xi
            if np.linalg.norm(acc - prev) <= float(np.float32(pr["min_increment"])):
                break
            prev = acc.copy()
    if not np.isfinite(acc.sum()) or acc.sum() >= float(np.float32(pr["max_increment"])):
        T = np.eye(4)
    v, n, it = _source_maps(depth, rgb, s, 0)
    return dict(vertex=v, normal=n, intensity=it, increment=T)


def _exact_filter(case, seed):
    depth = _f64(_prepare_filter(case, seed)["depth"])
    R, C = depth.shape
    r = case["radius"]
    pad = torch.nn.functional.pad(depth, (r, r, r, r))
    sw, sd = torch.zeros_like(depth), torch.zeros_like(depth)
    for j in range(2 * r + 1):
        for i in range(2 * r + 1):
            q = pad[j:j + R, i:i + C]
            w = torch.exp(-(q - depth) ** 2 / (2 * 0.03 ** 2) - ((i - r) ** 2 + (j - r) ** 2) / (2 * 2.0 ** 2)) * (q > 0)
            sw, sd = sw + w, sd + w * q
    smooth = torch.where(depth > 0, sd / sw, torch.zeros_like(sd))
    levels, d = [depth], depth
    for _ in range(1, case["levels"]):
        rr, cc = d.shape[0] // 2, d.shape[1] // 2
        center = d[0:2 * rr:2, 0:2 * cc:2]
        pad = torch.nn.functional.pad(d, (2, 3, 2, 3))
        sw, sd = torch.zeros_like(center), torch.zeros_like(center)
        for j, bj in enumerate((1., 4., 6., 4., 1.)):
            for i, bi in enumerate((1., 4., 6., 4., 1.)):
                q = pad[j:j + 2 * rr:2, i:i + 2 * cc:2]
                w = bi * bj * ((q > 0) & ((q - center).abs() < 0.09))
                sw, sd = sw + w, sd + w * q
        d = torch.where(center > 0, sd / sw, torch.zeros_like(sd))
        levels.append(d)
    return dict(smooth=smooth, pyramid=levels)


def _exact_graph(case, seed):
    V32, N32, a = _graph_inputs(case, seed)
    r = np.float32(case["radius_mm"] / 1000.0)
    # the vertex closest to the centre of each occupied cell, in vertex order
    # (which vertices are nodes is defined on single-precision cells)
    cell = np.floor(V32 / r)
    e = V32 - (cell + np.float32(0.5)) * r
    d2 = (e[:, 0] * e[:, 0] + e[:, 1] * e[:, 1]) + e[:, 2] * e[:, 2]
    key = (cell.astype(np.int64) + (1 << 20)) @ np.array([1 << 42, 1 << 21, 1])
    order = np.lexsort((np.arange(len(V32)), d2, key))
    first = np.concatenate([[True], key[order][1:] != key[order][:-1]])
    vid = np.sort(order[first])
    V, G = _f64(V32), _f64(V32[vid])
    dgw = float(np.float32(case["dgw_mm"] / 1000.0))

    def near(X, own):
        ids, ds = [], []
        for k in range(0, len(X), 1 << 14):
            x = X[k:k + (1 << 14)]
            d = torch.stack([(x[:, None, q] - G[None, :, q]) ** 2 for q in range(3)]).sum(0).sqrt()
            if own:
                rows = torch.arange(len(x), device=x.device)
                d[rows, k + rows] = float("inf")
            dd, ii = torch.topk(d, 4, dim=1, largest=False)
            ids.append(ii), ds.append(dd)
        d = torch.cat(ds).clamp(min=1e-4)
        return torch.cat(ids), torch.exp(-(d / dgw) ** 2)

    _, nbr_w = near(G, True)
    ids, w = near(V, False)
    T = _f64(_field(V32[vid].astype(np.float64), a))
    # unit quaternion (w, x, y, z) of each node, w >= 0 (small rotations), and its dual part
    R = T[:, :3, :3]
    qw = torch.sqrt(1 + R[:, 0, 0] + R[:, 1, 1] + R[:, 2, 2]) / 2
    qv = torch.stack([R[:, 2, 1] - R[:, 1, 2], R[:, 0, 2] - R[:, 2, 0], R[:, 1, 0] - R[:, 0, 1]], 1) / (4 * qw[:, None])
    t = T[:, :3, 3]
    dw = -0.5 * (t * qv).sum(1)
    dv = 0.5 * (qw[:, None] * t + torch.linalg.cross(t, qv))
    dq = torch.cat([qw[:, None], qv, dw[:, None], dv], 1)
    b = (w[..., None] * dq[ids]).sum(1)  # rotations within a right angle: no sign to choose
    own = torch.as_tensor(vid, device=b.device)
    b[own] = dq
    b = b / torch.linalg.norm(b[:, :4], dim=1, keepdim=True)
    rw, rv, dw, dv = b[:, :1], b[:, 1:4], b[:, 4:5], b[:, 5:]

    def turn(x):
        return x + 2 * torch.linalg.cross(rv, torch.linalg.cross(rv, x) + rw * x)

    shift = 2 * (dv * rw - rv * dw + torch.linalg.cross(rv, dv))
    return dict(node_vertices=None, node_neighbours=None, node_weights=nbr_w, neighbours=None, weights=w,
                vertices=turn(V) + shift, normals=turn(_f64(N32)), blocks=None)
