"""Blocks staged one after the other through one device, of as many and of
other numbers of frames (the FFT tables are kept while the number stays), with
a refused block between them: the same results, to the bit, as a new device's."""
import numpy as np
import pytest

from sassena_amd import ScatterDevice, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["all", "self"])
def test_blocks_in_turn(kind):
    rng = np.random.default_rng(5)
    u, qlen = synth.orientations(rng, 3), np.array([0.4, 1.1])
    with ScatterDevice(kind) as dev:
        for na, nf, layout in [(40, 100, "frames"), (40, 100, "atoms"), (70, 100, "soa"), (20, 1300, "frames"),
                               (20, 1, "frames"), (33, 100, "frames"), (64, 128, "atoms")]:
            shape = {"frames": (nf, na, 3), "atoms": (na, nf, 3), "soa": (3, na, nf)}[layout]
            xyz = rng.uniform(0.0, 20.0, size=shape).astype(np.float32)
            b = rng.uniform(1.0, 5.0, size=na)
            bad = np.full((2, 5, 3), np.inf, np.float32)
            with pytest.raises(RuntimeError, match="non-finite"):
                dev.stage(bad, layout="frames")
            dev.stage(xyz, layout=layout)
            dev.set_factors(b)
            got = dev.compute_oriented(qlen, u)
            with ScatterDevice(kind) as new:
                new.stage(xyz, layout=layout)
                new.set_factors(b)
                ref = new.compute_oriented(qlen, u)
            for x, y in zip(got, ref):
                assert np.array_equal(x, y)
