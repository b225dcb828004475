"""Wavefronts as work items of the coherent amplitude kernels and tiles of 1 to 8
shells on their own phases: every amplitude goes through the same operations
on the same atom ranges whatever the tile, so results are equal to the bit."""
import numpy as np
import pytest

from sassena_amd import synth
from sassena_amd.device import ScatterDevice

pytestmark = pytest.mark.gpu


def trajectory(na, nf, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(0.0, 30.0, size=(3, na, 1)) + np.cumsum(rng.normal(0.0, 0.1, size=(3, na, nf)), axis=2)
    return xyz.astype(np.float32), rng.choice([-3.74, 6.65, 5.80], size=na), rng


# shells on either side of a tile, orientations on either side of a workgroup (2 a wavefront, 4 wavefronts)
@pytest.mark.parametrize("ns,nm,na,nf", [(1, 1, 65, 70), (2, 9, 130, 64), (3, 8, 64, 65), (4, 7, 70, 129), (5, 17, 100, 30),
                                         (9, 3, 64, 66), (11, 16, 33, 100), (14, 5, 200, 65), (21, 33, 90, 70), (25, 2, 64, 64)])
@pytest.mark.parametrize("factors", [False, True])
def test_shell_tiles(ns, nm, na, nf, factors):
    xyz, b, rng = trajectory(na, nf, ns + nm)
    qlen, u = np.sort(rng.uniform(0.1, 4.0, size=ns)), synth.orientations(rng, nm)
    bs = rng.uniform(-2.0, 4.0, size=(ns, na)) if factors else None
    out = []
    for shape in (1, 3):
        with ScatterDevice("all", atom_split=2, tile_shape=shape) as dev:
            dev.stage(xyz, layout="soa")
            dev.set_factors(b)
            out.append(dev.compute_oriented(qlen, u, b_shell=bs))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("nv,na,nf,split", [(1, 64, 64, 1), (7, 65, 70, 2), (8, 100, 129, 3), (31, 64, 65, 1), (33, 130, 200, 2),
                                            (200, 70, 100, 1)])
def test_vector_blocks(nv, na, nf, split):
    xyz, b, rng = trajectory(na, nf, nv)
    qv = 1.7 * synth.orientations(rng, nv)
    out = []
    for block in (4, 8, 16):
        with ScatterDevice("all", "square", atom_split=split, vector_block=block) as dev:
            dev.stage(xyz, layout="soa")
            dev.set_factors(b)
            out.append(dev.compute_shell(qv))
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert np.array_equal(x, y)
