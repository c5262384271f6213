"""The marching-cubes tables of the build (product library and oracle) are
Bourke's tables as the reference uses them
(include/geometry/mesh/meshExtractor/lookupTables.h): compared through the
digests and per-case triangle counts in tests/golden/mc_tables.json."""
import ctypes
import hashlib
import json
import os

import numpy as np
import pytest

import oracle_lib as O
from dynamap_amd import _native as N

GOLD = json.load(open(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "mc_tables.json")))


def decode(words):
    rows = []
    for w in words:
        w = int(w)
        r = [(w >> (4 * k)) & 0xF for k in range(16)]
        r = [e if e != 0xF else -1 for e in r]
        k = r.index(-1) if -1 in r else 16
        rows.append(r[:k] + [-1] * (16 - k))
    return rows


def check(words):
    rows = decode(words)
    flat = [x for r in rows for x in r]
    assert hashlib.sha256(",".join(map(str, flat)).encode()).hexdigest() == GOLD["tri_sha256"]
    edge = [sum(1 << e for e in set(x for x in r if x >= 0)) for r in rows]
    assert hashlib.sha256(",".join(map(str, edge)).encode()).hexdigest() == GOLD["edge_sha256"]
    assert [sum(1 for x in r if x >= 0) // 3 for r in rows] == GOLD["triangles_per_case"]


def test_oracle_table():
    check(O.mc_table(32))


def test_product_table():
    lib = N.lib()
    out = np.zeros(256, np.uint64)
    assert lib.dm_mc_tri_table(out.ctypes.data_as(ctypes.c_void_p)) == 0
    check(out)


@pytest.mark.parametrize("vs", [0.02, 0.05, 0.003])
def test_cells_sample_their_own_block(vs):
    """The extraction leaves a block without observed voxels at once: whatever
    the rounding at large coordinates, on each axis a cell's corner samples have
    a voxel index in the cell's own block (here at every cell coordinate of the
    block keys' range, in the kernel's FP32 operations)."""
    f, vs = np.float32, np.float32(vs)
    for lo in range(-(1 << 23), 1 << 23, 1 << 21):
        g = np.arange(lo, lo + (1 << 21))
        own = np.zeros(len(g), bool)
        for off in (-vs / f(2), vs / f(2)):
            dual = (g.astype(f) * vs + f(0) + off) - vs / f(2)
            for q in (dual / vs, (dual + vs) / vs):
                own |= np.trunc(q + np.sign(q) * f(0.5)).astype(np.int64) >> 3 == g >> 3
        assert own.all()
