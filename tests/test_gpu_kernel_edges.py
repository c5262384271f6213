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
