"""Kernels at the sizes where their tiles, windows and lists end, against the
oracle or an independent numpy statement of the same thing."""
import numpy as np
import pytest

import dynamap_amd as dm
from dynamap_amd import configs
from test_gpu_volume import SENS, mirror, small_tsdf

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room():
    depth, _, poses = configs.make_sequence("rigid-320x240-2cm", 3)
    return depth, poses


def shifted(poses, shift):
    off = np.eye(4)
    off[:3, 3] = shift
    return np.stack([off @ p for p in poses])


# The raycast's empty-space bits lie in bricks of 4^3 blocks over a window of
# 512^3 blocks: the room moved so that it straddles the window's upper and
# lower face on each axis (block 256 starts at 40.96 m at 2 cm voxels) and by
# odd numbers of blocks (every alignment of block, brick and coarse cell).
# Bounds as in test_gpu_volume.test_raycast_on_identical_volume: 1e-5 m at the
# origin, 3e-5 m where a float coordinate is spaced 3.8e-6 m.
@pytest.mark.parametrize("shift", [(0.16, 0.48, -0.8), (0.0, 40.2, 0.0), (0.0, -40.4, 0.0), (0.0, 0.0, 39.5),
                                   (-39.5, 0.0, -40.0)])
def test_raycast_empty_space_bits(room, shift):
    depth, poses = room
    P = shifted(poses, shift)
    props = small_tsdf()
    vol = dm.TsdfVolume(props, SENS["rows"], SENS["cols"])
    for f in range(3):
        vol.IntegrateScan(depth[f], None, SENS, P[f].astype(np.float32))
    Tf = P[2].astype(np.float32)
    gd = vol.Raycast(Tf, SENS)[0]
    od = mirror(vol, props).raycast(Tf.astype(np.float64), SENS)[0]
    hit = od > 0
    assert hit.mean() > 0.8 and np.mean((gd > 0) == hit) >= 0.999
    tol = 1e-5 if max(np.abs(shift)) < 8 else 3e-5
    assert np.mean(np.abs(gd - od)[hit & (gd > 0)] <= tol) >= 0.999


# The wavefront's shared first steps and the workgroup's shared block pointers
# at image sizes that leave partial tiles and at a field of view so wide that
# the bundle bound ends the shared steps early (fx = 40 at 96 columns), close
# and far minimum depths.  Same bounds as above.
@pytest.mark.parametrize("rows,cols,fx,dmin", [(1, 1, 60.0, 0.3), (7, 9, 12.0, 0.3), (17, 33, 30.0, 0.1),
                                              (96, 97, 40.0, 0.3), (130, 63, 400.0, 1.2)])
def test_raycast_ragged_views(room, rows, cols, fx, dmin):
    depth, poses = room
    props = small_tsdf(min_sensor_depth=dmin)
    vol = dm.TsdfVolume(props, SENS["rows"], SENS["cols"])
    for f in range(3):
        vol.IntegrateScan(depth[f], None, SENS, poses[f].astype(np.float32))
    sens = dict(rows=rows, cols=cols, fx=fx, fy=fx, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    Tf = poses[1].astype(np.float32)
    gd = vol.Raycast(Tf, sens)[0]
    od = mirror(vol, props).raycast(Tf.astype(np.float64), sens)[0]
    hit = od > 0
    assert np.mean((gd > 0) == hit) >= 0.999
    both = hit & (gd > 0)
    assert both.sum() == 0 or np.mean(np.abs(gd - od)[both] <= 1e-5) >= 0.999


# One linearisation record per 1024 pixels, 16 records per ticket group, 256
# leaves in the sum of the records: frames of 1, 16, 17, 256 and 257 records at
# level 0.  The host path sums the same records in the same order and takes the
# same FP64 step, so the increments agree to FP64 rounding (sin and cos of the
# two sides may differ in the last bit).
@pytest.mark.parametrize("variant", ["shuffle", "mfma"])
@pytest.mark.parametrize("rows,cols", [(24, 40), (128, 128), (130, 128), (512, 512), (513, 512)])
def test_icp_step_record_counts(rows, cols, variant):
    f = 0.82 * cols
    sens = dict(rows=rows, cols=cols, fx=f, fy=f, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    sc = configs.Scene(1, configs.SEED_BASE + 1002)
    poses = sc.trajectory(2, configs.SEED_BASE + 1002)
    frames = [sc.render(p, sens, 7, noise=False)[0] for p in poses]
    s = dm.Session(small_tsdf(), configs.ICP_DEPTH, sens, np.eye(4))
    for l in range(3):
        v, n, i = s.source_maps(frames[0], None, l)
        s.set_model_maps(l, v, n, i)
    s.source_maps(frames[1], None, 0)
    s.set_icp_reduce(variant)
    dev = [s.icp_track(solve_on_host=False) for _ in range(3)]
    host = s.icp_track(solve_on_host=True)
    assert np.linalg.norm(host[:3, 3]) > 1e-4
    for T in dev:
        np.testing.assert_allclose(T, host, rtol=0, atol=1e-12)


# The integration's wavefronts take chunks of the pool: one workgroup (64
# blocks per wavefront and round), an odd number, and more wavefronts than
# blocks give the same poses, bit for bit.
def test_integration_chunks():
    depth, _, poses = configs.make_sequence("rigid-320x240-2cm", 4)
    w = configs.WORKLOADS["rigid-320x240-2cm"]
    got = []
    for wg in (1, 3, 2048, 4096):
        srv = dm.Server(1, 240, 320)
        srv.add_trace(w["tsdf"], w["icp"], w["sensor"], poses[0], depth)
        srv.set_shapes(integrate_workgroups=wg)
        got.append(srv.run(0, 0, 4, want_poses=True)["poses"])
        srv.close()
    for g in got[1:]:
        np.testing.assert_array_equal(g, got[0])


# Integration against the FP32 transcription where the straight code's range
# ends: a camera turned about its own axis inside blocks it has mapped (blocks
# that cross the camera plane), and voxels of 2e-9 m and 1e4 m, whose squared
# distances leave the range at one end.
@pytest.mark.parametrize("scale", [1.0, 1e-7, 5e5])
def test_integration_operand_range(room, scale):
    import oracle_lib as O
    depth, poses = room
    base = small_tsdf()
    props = dict(base, voxel_size=base["voxel_size"] * scale, truncation_distance=base["truncation_distance"] * scale,
                 max_sensor_depth=base["max_sensor_depth"] * scale, min_sensor_depth=base["min_sensor_depth"] * scale)
    vol = dm.TsdfVolume(props, SENS["rows"], SENS["cols"])
    ora = O.OracleVolume(props, 32)
    for f, yaw in enumerate((0.0, 0.7, -0.9)):
        c, s = np.cos(yaw), np.sin(yaw)
        R = np.eye(4)
        R[:3, :3] = [[c, 0, s], [0, 1, 0], [-s, 0, c]]
        T = (poses[0] @ R).astype(np.float64)
        T[:3, 3] *= scale
        Tf, d = T.astype(np.float32), (depth[f] * np.float32(scale)).astype(np.float32)
        vol.IntegrateScan(d, None, SENS, Tf)
        ora.integrate_scan(d, None, SENS, Tf.astype(np.float64))
    gx, gs, _, gw = vol.blocks()
    ox, os_, _, ow = ora.blocks()
    gi, oi = np.lexsort(gx.T[::-1]), np.lexsort(ox.T[::-1])
    np.testing.assert_array_equal(gx[gi], ox[oi])
    np.testing.assert_array_equal(gw[gi], ow[oi])
    np.testing.assert_array_equal(gs[gi], os_[oi].astype(np.float32))
    assert (gw > 0).any()


# Host results pass in chunks of half the frame's pinned buffer: images from
# one pixel up, smaller than the volume's frame and as large, with the smallest
# chunk (a frame of 200x166) and a larger one; every output and fewer of them.
@pytest.mark.parametrize("rows,cols,frame", [(1, 1, (240, 320)), (3, 5, (240, 320)), (33, 31, (240, 320)),
                                            (240, 320, (240, 320)), (166, 200, (166, 200)), (2, 1, (2, 1))])
def test_raycast_outputs_in_chunks(room, rows, cols, frame):
    import ctypes as C
    from dynamap_amd import _native as N
    depth, poses = room
    vol = dm.TsdfVolume(small_tsdf(), *frame)
    view = dict(SENS, rows=min(frame[0], SENS["rows"]), cols=min(frame[1], SENS["cols"]))
    vol.IntegrateScan(np.ascontiguousarray(depth[0][:view["rows"], :view["cols"]]), None, view,
                      poses[0].astype(np.float32))
    sens = dict(rows=rows, cols=cols, fx=0.8 * cols + 1, fy=0.8 * cols + 1, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    Tf = np.ascontiguousarray(poses[0], np.float32)
    d, v, n, c = vol.Raycast(Tf, sens)
    np.testing.assert_array_equal(v[..., 2], d)  # a vertex's z is its depth, 0 without a surface
    assert np.array_equal(np.isnan(n[..., 0]), np.isnan(n[..., 2]))
    only = np.full((rows, cols, 3), 7, np.float32)
    N.check(N.lib().dm_volume_raycast(vol._h, N.ptr(Tf), C.byref(configs.sensor(sens)), None, None, N.ptr(only), None))
    np.testing.assert_array_equal(only, n)


# One Gauss-Newton step against the FP64 oracle on random clouds (normals in
# every direction, so that every motion is observable and the step is unique):
# 5 nodes, 16 (one workgroup of the PCG), 17 (one node in a second), 32 and 33
# (the same of the preconditioner), and 300,
# some of whose rows have more than 16 blocks.  PCG runs to its tolerance.  The GPU
# stores the blocks in FP32 (6e-8 relative); with the damping and the weights
# here the systems' condition numbers stay below 1e4, so 1e-3 of the largest
# motion bounds the difference.
@pytest.mark.parametrize("nodes", [5, 16, 17, 32, 33, 300])
def test_nonrigid_step_node_counts(nodes):
    import oracle_lib as O
    from test_oracle_nonrigid import random_cloud
    V, Nn = random_cloud(6000, 11)
    ids = np.linspace(0, len(V) - 1, nodes).astype(np.int32)
    lo, hi = V.min(0), V.max(0)
    size = float((hi - lo).max())
    dgw = 2.0 * size / nodes ** (1 / 3)
    g = dm.DefGraph(V, Nn, dgw=dgw, node_ids=ids)
    o = O.OracleGraph(V, Nn, dgw=dgw, bits=64, node_ids=ids)
    shift = 0.004 * np.stack([np.sin(V[:, 1] / size * 3), np.cos(V[:, 2] / size * 3), np.sin(V[:, 0] / size * 3)], 1)
    target = (V + shift).astype(np.float32)
    kw = dict(gn_iterations=1, pcg_iterations=400, pcg_tol=1e-9, damping=1.0)
    dm.NonRigidICP(**kw).solve_mesh(g, target, Nn, np.eye(4))
    o.solve_mesh(target, Nn, np.eye(4), **kw)
    Tg, To = g.transforms(), o.transforms().reshape(-1, 4, 4)
    moved = np.abs(To - np.eye(4)).max()
    assert moved > 1e-4
    assert np.abs(Tg - To).max() <= 1e-3 * moved
    if nodes == 300:  # the longest row, from the vertices' node pairs, has more than 16 blocks
        nn = g.vertex_neighbours()[0]
        pairs = np.unique(np.concatenate([nn[:, [a, b]] for a in range(4) for b in range(4)]), axis=0)
        assert np.bincount(pairs[:, 0]).max() > 16


# Nearest nodes where a query's lanes change in number (8 below 65536 queries,
# then 1) and where the nodes fill, miss and pass a tile of 1024
# and a group of 32.
# Whole coordinates: squared distances are exact and full of ties, which go to
# the lower index.
@pytest.mark.parametrize("nodes,verts", [(5, 16383), (1023, 16384), (1025, 65535), (1024, 65536), (2049, 300),
                                         (5, 65537), (33, 65536), (1087, 68000)])
def test_nearest_nodes_lanes_and_ties(nodes, verts):
    rng = np.random.default_rng(nodes + verts)
    cell = rng.permutation(41 ** 3)[:max(verts, nodes)]
    V = np.stack([cell // 1681, cell // 41 % 41, cell % 41], 1).astype(np.float32)
    Nn = np.tile(np.float32([0, 0, 1]), (len(V), 1))
    ids = rng.permutation(len(V))[:nodes].astype(np.int32)
    g = dm.DefGraph(V, Nn, dgw=20.0, node_ids=ids)
    vid, nbr, _ = g.nodes()
    P, Q = V.astype(np.int64), V[vid].astype(np.int64)

    def expect(rows, own):
        key = (((rows[:, None] - Q[None]) ** 2).sum(2)) * nodes + np.arange(nodes)
        if own is not None:
            key[np.arange(len(rows)), own] = 1 << 40
        return np.sort(np.partition(key, 3, 1)[:, :4], 1) % nodes

    np.testing.assert_array_equal(nbr, expect(Q, np.arange(nodes)))
    vnn = g.vertex_neighbours()[0]
    for a in range(0, len(P), 8192):
        np.testing.assert_array_equal(vnn[a:a + 8192], expect(P[a:a + 8192], None))


# Marching cubes at the origin, across it, and where float coordinates are so
# coarse (0.0078 m at 80 km, voxels of 0.02 m) that a cell's samples leave the
# voxels around it or change weight; caps that end inside a block.  Same order and the same bits as
# the FP32 restatement.
@pytest.mark.parametrize("shift,irregular", [((0.0, 0.0, 0.0), False), ((-1.3, 0.9, -2.1), False),
                                            ((80000.0, 0.0, 0.0), True), ((0.0, -80000.0, 0.0), False),
                                            ((0.0, 0.0, 81000.0), True)])
def test_mesh_cells_near_and_far(room, shift, irregular):
    import oracle_lib as O
    from test_gpu_mesh import check_same, mirror as mirror_slots
    depth, poses = room
    P = shifted(poses, shift)
    vol = dm.TsdfVolume(small_tsdf(), SENS["rows"], SENS["cols"])
    vol.props = small_tsdf()
    for f in range(3):
        vol.IntegrateScan(depth[f], None, SENS, P[f].astype(np.float32))
    vs, half = np.float32(vol.props["voxel_size"]), np.float32(0.5)
    g = np.arange(8) + 8 * vol.blocks()[0][:, int(np.argmax(np.abs(shift))), None]
    moved = False  # an index or a weight of a cell's samples, in the kernel's float operations
    for sign in (0, 1):
        p = g.astype(np.float32) * vs + (vs / 2 if sign else -vs / 2)
        q = (p - vs / 2) / vs
        w = p / vs - np.floor(p / vs)
        moved |= bool(((np.trunc(q + np.sign(q) * half) != g - 1 + sign) | (w < 0.25) | (w > 0.75)).any())
    assert moved == irregular
    o = O.mc_extract(mirror_slots(vol))
    m = vol.ExtractMesh(max_triangles=1 << 20)
    assert irregular or len(m) > 1000
    check_same((m.triangles, m.colors, m.edge_ids), o)
    for cap in (1, 2, 67, 130):
        c = dm.MeshExtractor(cap).ExtractMesh(vol)
        assert c.num_triangles_ == len(m) and len(c) == min(cap, len(m))
        check_same((c.triangles, c.colors, c.edge_ids), tuple(a[:cap] for a in o))


# Allocation where a workgroup's lists end: one pixel, ragged tiles, and a 16x16
# image of rays so far apart that one tile notes more keys than its list (1024)
# and its set of handled blocks hold; a window face crossed; a table with full buckets
# next.  The slots' keys and the dropped keys equal the oracle's after each
# of several frames, the same frame twice among them.
@pytest.mark.parametrize("rows,cols,fx,props,shift", [
    (1, 1, 10.0, {}, 0.0), (17, 33, 30.0, {}, 0.0), (16, 16, 5.0, dict(voxel_size=0.008), 0.0),
    (16, 16, 5.0, dict(voxel_size=0.008), 15.9), (16, 16, 5.0, dict(voxel_size=0.008, num_buckets=1024), 0.0),
    (9, 11, 9.0, dict(voxel_size=0.02, num_blocks=512), 0.0)])
def test_allocation_lists(room, rows, cols, fx, props, shift):
    import oracle_lib as O
    from test_gpu_volume import table_keys
    depth, poses = room
    sens = dict(rows=rows, cols=cols, fx=fx, fy=fx, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    P = shifted(poses, (shift, 0, 0))
    props = small_tsdf(**{"num_buckets": 1 << 15, "num_blocks": 1 << 15, **props})
    vol = dm.TsdfVolume(props, rows, cols)
    ora = O.OracleVolume(props, 32)
    most = 0
    for f, oy in ((0, 0), (0, 0), (1, 60), (2, 120)):
        d = np.ascontiguousarray(depth[f][oy:oy + rows, 40:40 + cols])
        Tf = P[f].astype(np.float32)
        before = vol.GetNumAllocatedBlocks()
        vol.AllocateFromDepth(d, sens, Tf)
        ora.allocate(d, sens, Tf.astype(np.float64))
        most = max(most, vol.GetNumAllocatedBlocks() - before)
        np.testing.assert_array_equal(table_keys(vol.GetHashEntries()), ora.table()[0])
        c, o = vol.counters(), ora.dropped()
        assert c["dropped_bucket"] == o["bucket"] and c["dropped_pool"] == o["pool"] and c["dropped_keyset"] == 0
    if fx == 5.0:
        assert most > 2048
    assert (ora.dropped()["pool"] > 0) == (props["num_blocks"] == 512)


# More new keys in one frame than the frame's list holds (4096): the list is
# filled, the rest is counted and taken in by a later frame as far as there is room.
def test_allocation_list_overflow(room):
    import oracle_lib as O
    from test_gpu_volume import table_keys
    depth, poses = room
    sens = dict(rows=32, cols=32, fx=9.0, fy=9.0, cx=15.5, cy=15.5)
    d, Tf = np.ascontiguousarray(depth[0][:32, :32]), poses[0].astype(np.float32)
    ora = O.OracleVolume(small_tsdf(voxel_size=0.008, num_buckets=1 << 16, num_blocks=1 << 16), 32)
    ora.allocate(d, sens, Tf.astype(np.float64))
    assert ora.num_alloc() > 5000
    vol = dm.TsdfVolume(small_tsdf(voxel_size=0.008, num_buckets=1 << 16, num_blocks=4096), 32, 32)
    vol.AllocateFromDepth(d, sens, Tf)
    c = vol.counters()
    assert c["allocated"] == 4096 and c["dropped_keyset"] >= ora.num_alloc() - 4096 and c["dropped_pool"] == 0
    vol.AllocateFromDepth(d, sens, Tf)
    c = vol.counters()
    assert c["allocated"] == 4096 and c["dropped_pool"] > 0
    xyz = vol.blocks()[0]
    full = {tuple(k) for k in ora.blocks()[0]}
    assert len({tuple(k) for k in xyz}) == 4096 and all(tuple(k) in full for k in xyz)


# Every filter radius, and pyramid levels down to nothing, at sizes that leave
# parts of a tile and of the window outside the image; pixels without depth and
# depth edges included.  The exponentials of the GPU and host libraries may
# differ in the last bit, so 2e-6 of the largest depth.
@pytest.mark.parametrize("radius", range(8))
@pytest.mark.parametrize("rows,cols", [(1, 1), (17, 33), (50, 39)])
def test_depth_filters_ragged(room, radius, rows, cols):
    import oracle_lib as O
    d = room[0][0][40:40 + rows, 100:100 + cols].copy()
    d.flat[::7] = 0.0
    d.flat[3::11] *= np.float32(1.05)
    g, o = dm.bilateral_filter(d, radius, 0.03, 2.5), O.bilateral(d, radius, 0.03, 2.5, bits=32)
    np.testing.assert_array_equal(g == 0, o == 0)
    assert np.abs(g - o).max() <= 2e-6 * np.abs(o).max()
    levels = dm.depth_pyramid(d, 0.01 * (radius + 1), 4)
    for l in range(1, 4):
        assert levels[l].shape == (rows >> l, cols >> l)
        if levels[l].size:
            o = O.pyr_down(levels[l - 1], 0.01 * (radius + 1), bits=32)
            assert np.abs(levels[l] - o).max() <= 2e-6 * np.abs(o).max()


# Sessions taken from the server's pool and cleared on the device: runs after
# the first equal it bit for bit, batched and frame by frame, with pools and
# tables of sizes that are no multiple of the clear's words, and bucket records
# of one and several lines.
@pytest.mark.parametrize("props", [dict(num_blocks=9999), dict(num_blocks=6007, num_buckets=5003, bucket_size=3),
                                   dict(bucket_size=25)])
def test_server_sessions_cleared(props):
    N = dm._native
    w = configs.WORKLOADS["rigid-320x240-2cm"]
    srv = dm.Server(4, 240, 320)
    for k in range(3):
        d, c, g = configs.make_sequence("rigid-320x240-2cm", 4, session=k)
        srv.add_trace(small_tsdf(**props), w["icp"], w["sensor"], g[0], d, c)
    first = srv.run(N.DM_RUN_BATCHED, 0, 4, want_poses=True)["poses"]
    assert np.abs(first[:, 1:, :3, 3] - first[:, :1, :3, 3]).max() > 1e-3
    for mode in (N.DM_RUN_BATCHED, N.DM_RUN_PER_FRAME_DEV, N.DM_RUN_BATCHED):
        np.testing.assert_array_equal(srv.run(mode, 0, 4, want_poses=True)["poses"], first)
    srv.close()


# The shared first steps' bound with mirrored axes (a focal length below zero,
# which the server takes): a camera rolled by 45 degrees, so that the two axes'
# shares of the bound are equal in size, before a wall at 1 m with an opening in
# front of the middle of every wavefront, behind which there is nothing the
# tracking may use.  The bundle's middle ray runs free through the opening; the
# rays beside it must find the wall, or the second frame cannot be tracked.
@pytest.mark.parametrize("sx,sy", [(1, 1), (1, -1), (-1, 1), (-1, -1)])
def test_raycast_shared_steps_mirrored_sensor(sx, sy):
    import oracle_lib as O
    n, near = 32, (1.0, 0.97)
    icp = dict(configs.ICP_DEPTH, max_depth=1.5)
    props = dict(configs.TSDF_2CM, voxel_size=0.01, truncation_distance=0.03, num_buckets=1 << 18, num_blocks=1 << 18)
    sens = dict(rows=n, cols=n, fx=5.0 * sx, fy=5.0 * sy, cx=(n - 1) / 2, cy=(n - 1) / 2)
    c = np.sqrt(0.5)
    pose = np.eye(4)
    pose[:2, :2] = [[c, -c], [c, c]]
    mid = (np.arange(n) % 8 >= 2) & (np.arange(n) % 8 < 6)
    D = np.stack([np.where(mid[:, None] & mid[None], z + 1.5, z) for z in near]).astype(np.float32)
    o = O.OraclePipeline(props, icp, sens, pose, bits=64)
    To = np.stack([o.process_frame(d, None) for d in D])
    assert To[1, 2, 3] > 0.025  # of the 0.03 m between the frames
    srv = dm.Server(1, n, n)
    srv.add_trace(props, icp, sens, pose, D)
    Tg = srv.run(0, 0, 2, want_poses=True)["poses"][0]
    srv.close()
    assert np.abs(Tg - To).max() < 1e-3  # a tenth of a voxel


# A minimum depth below zero: the rays begin behind the camera, where they lie
# as far apart as in front.  The map is made while the camera turns, so that
# surfaces stand on both sides.  Bounds as in test_raycast_ragged_views.
@pytest.mark.parametrize("n,fx", [(33, 20.0), (64, 40.0), (40, 12.0)])
@pytest.mark.parametrize("dmin", [-1.5, -3.0])
def test_raycast_negative_minimum_depth(n, fx, dmin):
    def turned(a):
        c, s = np.cos(a), np.sin(a)
        R = np.eye(4)
        R[:3, :3] = [[c, 0, s], [0, 1, 0], [-s, 0, c]]
        return pose @ R

    sc = configs.Scene(1, configs.SEED_BASE + 1002)
    pose = sc.trajectory(1, configs.SEED_BASE + 1002)[0]
    props = small_tsdf(min_sensor_depth=dmin)
    vol = dm.TsdfVolume(props, SENS["rows"], SENS["cols"])
    for a in np.arange(9) * 0.7:
        vol.IntegrateScan(sc.render(turned(a), SENS, 7, noise=False)[0], None, SENS, turned(a).astype(np.float32))
    sens = dict(rows=n, cols=n, fx=fx, fy=fx, cx=(n - 1) / 2, cy=(n - 1) / 2)
    Tf = turned(0.35).astype(np.float32)
    gd = vol.Raycast(Tf, sens)[0]
    od = mirror(vol, props).raycast(Tf.astype(np.float64), sens)[0]
    hit = od > 0
    assert 0 < hit.sum() < hit.size  # some rays end at a surface behind the camera
    assert np.mean((gd > 0) == hit) >= 0.999
    assert np.mean(np.abs(gd - od)[hit & (gd > 0)] <= 1e-5) >= 0.999


# Vertices, some of them nodes, that are not finite or so far away that squared
# distances overflow: their empty neighbour slots (-1) add nothing.  The other
# vertices' and nodes' neighbours, the block pattern, the blended mesh and a
# Gauss-Newton step are those of the graph without them (bound of the step as in
# test_nonrigid_step_node_counts).
def test_graph_empty_neighbour_slots():
    from test_oracle_nonrigid import random_cloud
    V, Nn = random_cloud(3000, 5)
    bad = np.float32([[np.nan, 0, 0], [0, np.inf, 0], [0, 0, 1e30], [np.nan] * 3, [-np.inf, 0, np.inf], [3e25, 0, 0]])
    ids = np.linspace(0, len(V) - 1, 40).astype(np.int32)
    V2, N2 = np.concatenate([V, bad]), np.concatenate([Nn, np.tile(np.float32([0, 0, 1]), (len(bad), 1))])
    ids2 = np.concatenate([ids, len(V) + np.arange(3, dtype=np.int32)])
    size = float((V.max(0) - V.min(0)).max())
    kw = dict(dgw=2.0 * size / len(ids) ** (1 / 3))
    g, h = dm.DefGraph(V, Nn, node_ids=ids, **kw), dm.DefGraph(V2, N2, node_ids=ids2, **kw)
    (_, nbr, nw), (_, nbr2, nw2) = g.nodes(), h.nodes()
    np.testing.assert_array_equal(nbr2[:40], nbr)
    np.testing.assert_array_equal(nw2[:40], nw)
    assert (nbr2[40:] == -1).all() and (nw2[40:] == 0).all()
    (vnn, vw), (vnn2, vw2) = g.vertex_neighbours(), h.vertex_neighbours()
    np.testing.assert_array_equal(vnn2[:3000], vnn)
    np.testing.assert_array_equal(vw2[:3000], vw)
    want = np.full((6, 4), -1)
    want[2, 0] = 42  # the third is a node and finite: its own nearest
    np.testing.assert_array_equal(vnn2[3000:], want)
    assert h.num_blocks() == g.num_blocks() + 3  # the three nodes' own
    T = np.tile(np.eye(4), (43, 1, 1))
    T[:, :3, 3] = np.random.default_rng(1).normal(0, 0.01, (43, 3))
    g.set_transforms(T[:40])
    h.set_transforms(T)
    for a, b in zip(dm.DqBlender(g).blendMesh(), dm.DqBlender(h).blendMesh()):
        np.testing.assert_array_equal(b[:3000], a)
    g.set_transforms(np.tile(np.eye(4), (40, 1, 1)))
    h.set_transforms(np.tile(np.eye(4), (43, 1, 1)))
    target = (V + 0.004 * np.sin(V[:, [1, 2, 0]] / size * 3)).astype(np.float32)
    kw = dict(gn_iterations=1, pcg_iterations=400, pcg_tol=1e-9, damping=1.0)
    s = dm.NonRigidICP(**kw).solve_mesh(g, target, Nn, np.eye(4))
    # no target for the others: a zero normal
    s2 = dm.NonRigidICP(**kw).solve_mesh(h, np.concatenate([target, np.zeros((6, 3), np.float32)]),
                                        np.concatenate([Nn, np.zeros((6, 3), np.float32)]), np.eye(4))
    assert s2["residuals"] == s["residuals"] > 2000
    moved = np.abs(g.transforms() - np.eye(4)).max()
    assert moved > 1e-4
    assert np.abs(h.transforms()[:40] - g.transforms()).max() <= 1e-3 * moved
    np.testing.assert_array_equal(h.transforms()[40:], np.tile(np.eye(4), (3, 1, 1)))
    h.defGraphUpdateNodes()
    np.testing.assert_array_equal(h.vertex_neighbours()[0], vnn2)


# Nodes without coordinates among those that the one-lane search looks at first
# (65536 queries or more): they are nobody's neighbours and change nobody's.
# Whole coordinates as in test_nearest_nodes_lanes_and_ties.
@pytest.mark.parametrize("nodes,verts", [(1087, 68000), (2049, 66000)])
def test_nearest_nodes_without_coordinates(nodes, verts):
    rng = np.random.default_rng(nodes)
    cell = rng.permutation(41 ** 3)[:verts]
    V = np.stack([cell // 1681, cell // 41 % 41, cell % 41], 1).astype(np.float32)
    ids = rng.permutation(verts)[:nodes].astype(np.int32)
    Q = V[ids].astype(np.int64)
    lost = np.arange(0, nodes, 32)[1::2]
    V[ids[lost]] = np.nan
    g = dm.DefGraph(V, np.tile(np.float32([0, 0, 1]), (verts, 1)), dgw=20.0, node_ids=ids)
    vnn = g.vertex_neighbours()[0]
    for a in range(0, verts, 8192):
        P = V[a:a + 8192]
        key = ((np.nan_to_num(P).astype(np.int64)[:, None] - Q[None]) ** 2).sum(2) * nodes + np.arange(nodes)
        key[:, lost] = 1 << 40
        want = np.sort(np.partition(key, 3, 1)[:, :4], 1) % nodes
        want[np.isnan(P[:, 0])] = -1
        np.testing.assert_array_equal(vnn[a:a + 8192], want)


# The initial pose is read before the session's creation returns: the caller's
# array is changed right after it.
def test_session_reads_initial_pose_before_return(room):
    import ctypes as C
    from dynamap_amd import _native as N
    depth, poses = room
    w = configs.WORKLOADS["rigid-320x240-2cm"]
    for _ in range(4):
        T = np.array(poses[1], np.float64)  # its own copy: the fixture's stays
        keep, h = T.copy(), C.c_void_p()
        N.check(N.lib().dm_session_create(C.byref(configs.tsdf_props(small_tsdf())), C.byref(configs.icp_props(w["icp"])),
                                          C.byref(configs.sensor(SENS)), N.ptr(T), C.byref(h)))
        T[:] = np.nan
        got = np.zeros((4, 4))
        d = np.ascontiguousarray(depth[1])
        N.check(N.lib().dm_session_process_frame(h, N.ptr(d), None, 0, N.ptr(got)))
        N.lib().dm_session_destroy(h)
        np.testing.assert_array_equal(got, keep)


# Results that need no packed copy on the device take no memory for one: 448 MB
# at 4000x4000 pixels.
def test_depth_render_takes_no_map_memory():
    import ctypes as C
    from dynamap_amd import _native as N
    n = 4000
    sens = dict(rows=n, cols=n, fx=3000.0, fy=3000.0, cx=2000.0, cy=2000.0)
    vol = dm.TsdfVolume(small_tsdf(), n, n)
    T, d, v = np.eye(4, dtype=np.float32), np.ones((n, n), np.float32), np.ones((n, n, 3), np.float32)
    rt = C.CDLL("libamdhip64.so.7")  # the runtime that the library links

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert rt.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def taken(vertex):
        before = free()
        N.check(N.lib().dm_volume_raycast(vol._h, N.ptr(T), C.byref(configs.sensor(sens)), N.ptr(d), vertex, None, None))
        return before - free()

    taken(None)  # whatever a first launch takes
    vol.close()
    vol = dm.TsdfVolume(small_tsdf(), n, n)
    assert taken(None) < 28 * n * n / 2
    assert not d.any()
    assert taken(N.ptr(v)) >= 28 * n * n / 2
    assert not v.any()


@pytest.fixture(scope="module")
def room_8mm():
    depth, _, poses = configs.make_sequence("rigid-640x480-8mm", 2)
    return depth, poses


# The keys that a workgroup may hold back before it lists them: 109, 13, 6 and 4
# in each of 1200 workgroups, of a first frame's 11 000 new blocks (the list is as
# long as the pool; at 4 the second frame's blocks pass it).  The same slots and
# drops as the oracle's.
@pytest.mark.parametrize("num_blocks", [1 << 18, 1 << 15, 1 << 14, 11000])
def test_allocation_room_of_workgroups(room_8mm, num_blocks):
    import oracle_lib as O
    from test_gpu_volume import table_keys
    depth, poses = room_8mm
    w = configs.WORKLOADS["rigid-640x480-8mm"]
    props = dict(w["tsdf"], num_buckets=1 << 16, num_blocks=num_blocks)
    vol, ora = dm.TsdfVolume(props, 480, 640), O.OracleVolume(props, 32)
    for f in range(2):
        Tf = poses[f].astype(np.float32)
        vol.AllocateFromDepth(depth[f], w["sensor"], Tf)
        ora.allocate(depth[f], w["sensor"], Tf.astype(np.float64))
        np.testing.assert_array_equal(table_keys(vol.GetHashEntries()), ora.table()[0])
        assert vol.counters()["dropped_pool"] == ora.dropped()["pool"]


# A scene far beyond the pool: each frame's 250 000 new blocks against a list and a
# pool of 4096 and 32768.  Every frame ends within 0.1 s (5 ms here; 0.45 and 1.6 s
# when the keys held back filled the frame's set) and the pool fills.
@pytest.mark.parametrize("num_blocks", [1 << 12, 1 << 15])
def test_allocation_far_beyond_the_pool(num_blocks):
    import time
    w = configs.WORKLOADS["large-640x480-4mm"]
    depth, _, poses = configs.make_sequence("large-640x480-4mm", 1)
    vol = dm.TsdfVolume(dict(w["tsdf"], num_buckets=1 << 18, num_blocks=num_blocks), 480, 640)
    Tf, took = poses[0].astype(np.float32), []
    for _ in range(4):
        t = time.perf_counter()
        vol.AllocateFromDepth(depth[0], w["sensor"], Tf)
        took.append(time.perf_counter() - t)
    c = vol.counters()
    assert c["allocated"] == num_blocks and c["dropped_keyset"] > 4 * 200000 and c["dropped_pool"] == 3 * num_blocks
    assert min(took[1:]) < 0.1


# The other change of a query's lanes in number (64 below 12288 queries, then 8),
# of vertices and of nodes.
@pytest.mark.parametrize("nodes,verts", [(1025, 12287), (1025, 12288), (12287, 12400), (12289, 12400)])
def test_nearest_nodes_few_queries(nodes, verts):
    test_nearest_nodes_lanes_and_ties(nodes, verts)


# Camera coordinates far below the range that the integration's shared division
# is exact in: a camera moved by less than 1e-20 m beside voxels at x = y = 0,
# with the principal point on a pixel's centre and on its edge, against the FP32
# transcription.
@pytest.mark.parametrize("t", [0.0, 1e-20, -1e-30, 1e-41])
@pytest.mark.parametrize("c", [0.0, -0.5, 7.5, 8.0])
def test_integration_tiny_numerators(t, c):
    import oracle_lib as O
    sens = dict(rows=16, cols=16, fx=20.0, fy=20.0, cx=c, cy=c)
    props = small_tsdf()
    vol, ora = dm.TsdfVolume(props, 16, 16), O.OracleVolume(props, 32)
    T = np.eye(4, dtype=np.float32)
    T[0, 3], T[1, 3] = t, -t
    d = np.full((16, 16), 1.0, np.float32)
    d[1:] = 1.03  # a voxel's pixel shows in its value
    for _ in range(2):
        vol.IntegrateScan(d, None, sens, T)
        ora.integrate_scan(d, None, sens, T.astype(np.float64))
    gx, gs, _, gw = vol.blocks()
    ox, os_, _, ow = ora.blocks()
    gi, oi = np.lexsort(gx.T[::-1]), np.lexsort(ox.T[::-1])
    np.testing.assert_array_equal(gx[gi], ox[oi])
    np.testing.assert_array_equal(gw[gi], ow[oi])
    np.testing.assert_array_equal(gs[gi], os_[oi].astype(np.float32))
    assert (gw > 0).any()


# The shared first steps have their own pixels per wavefront for each tile width:
# the same poses bit for bit at all four, batched at frame sizes that are no
# multiple of the tiles, with a narrow and a wide field of view; the poses are
# the oracle's within 1e-3 m.
@pytest.mark.parametrize("rows,cols,fx", [(97, 131, 90.0), (66, 70, 30.0), (75, 203, 260.0)])
def test_raycast_tile_widths(rows, cols, fx):
    import oracle_lib as O
    sens = dict(rows=rows, cols=cols, fx=fx, fy=fx, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    sc = configs.Scene(1, configs.SEED_BASE + 1002)
    poses = sc.trajectory(5, configs.SEED_BASE + 1002)
    D = np.stack([sc.render(p, sens, 7, noise=False)[0] for p in poses])
    got = []
    for width in (16, 8, 32, 64):
        srv = dm.Server(2, 120, 220)  # frames smaller than the launch
        srv.add_trace(small_tsdf(), configs.ICP_DEPTH, sens, poses[0], D)
        srv.add_trace(small_tsdf(voxel_size=0.03, truncation_distance=0.09), configs.ICP_DEPTH, sens, poses[0], D)
        srv.set_shapes(ray_tile_width=width)
        got.append(srv.run(0, 0, 5, want_poses=True)["poses"])
        srv.close()
    for g in got[1:]:
        np.testing.assert_array_equal(g, got[0])
    o = O.OraclePipeline(small_tsdf(), configs.ICP_DEPTH, sens, poses[0], bits=64)
    To = np.stack([o.process_frame(d, None) for d in D])
    assert np.abs(To[-1, :3, 3] - To[0, :3, 3]).max() > 1e-3
    assert np.abs(got[0][0] - To).max() < 1e-3


# test_raycast_ragged_views where the oracle must see the room, so that the
# comparison cannot pass on two empty images.
@pytest.mark.parametrize("rows,cols,fx,dmin", [(1, 1, 60.0, 0.3), (7, 9, 12.0, 0.3), (17, 33, 30.0, 0.1),
                                              (96, 97, 40.0, 0.3), (130, 63, 400.0, 1.2)])
def test_raycast_ragged_views_see_the_room(room, rows, cols, fx, dmin):
    depth, poses = room
    props = small_tsdf(min_sensor_depth=dmin)
    vol = dm.TsdfVolume(props, SENS["rows"], SENS["cols"])
    for f in range(3):
        vol.IntegrateScan(depth[f], None, SENS, poses[f].astype(np.float32))
    sens = dict(rows=rows, cols=cols, fx=fx, fy=fx, cx=(cols - 1) / 2, cy=(rows - 1) / 2)
    Tf = poses[1].astype(np.float32)
    gd = vol.Raycast(Tf, sens)[0]
    od = mirror(vol, props).raycast(Tf.astype(np.float64), sens)[0]
    hit = od > 0
    assert hit.any() and np.mean((gd > 0) == hit) >= 0.999
    assert np.mean(np.abs(gd - od)[hit & (gd > 0)] <= 1e-5) >= 0.999
