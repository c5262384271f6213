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
