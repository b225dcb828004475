"""Frame-major blocks through both tile heights of the staging transpose (16
frames while tiles of 64 are fewer than 512) and the largest coordinate's
reduction: the same results, to the bit, as the block staged by rows, which
needs no transpose."""
import numpy as np
import pytest

from sassena_amd import ScatterDevice, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nf", [(1, 1), (63, 15), (64, 16), (65, 17), (130, 63), (64, 65), (1000, 200), (16385, 129)])
def test_layouts(na, nf):
    rng = np.random.default_rng(na + nf)
    frames = rng.uniform(-20.0, 20.0, size=(nf, na, 3)).astype(np.float32)
    b, u = rng.uniform(-2.0, 4.0, size=na), synth.orientations(rng, 3)
    qlen = synth.linear_shells(0.1, 2.0, 4)
    out = []
    for layout, xyz in (("frames", frames), ("soa", np.ascontiguousarray(frames.transpose(2, 1, 0)))):
        with ScatterDevice("all", "square") as dev:
            dev.stage(xyz, layout=layout)
            dev.set_factors(b)
            out.append(dev.compute_oriented(qlen, u))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("na,nf", [(1, 1), (64, 64), (77, 300), (3000, 65)])
@pytest.mark.parametrize("at", [0.0, 0.5, 1.0])
def test_infinite_coordinate_is_found(na, nf, at):
    xyz = np.zeros((3, na, nf), np.float32)
    xyz.reshape(-1)[int(at * (xyz.size - 1))] = -np.inf
    with ScatterDevice("all") as dev:
        with pytest.raises(RuntimeError, match="non-finite"):
            dev.stage(xyz, layout="soa")
