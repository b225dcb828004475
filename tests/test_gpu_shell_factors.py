"""One factor per shell and atom (X-ray form factors), read as the shells'
factors of an atom, against one call per shell with that shell's factors: the
same direct phases and sums, so equal to one FP32 rounding of an amplitude."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -22


@pytest.mark.parametrize("NA,NF,ns,NM,shape", [(1, 64, 1, 1, 0), (65, 70, 7, 9, 1), (64, 64, 8, 8, 1), (130, 65, 9, 17, 2),
                                               (40, 100, 21, 3, 3), (77, 66, 17, 5, 4), (300, 64, 41, 12, 5),
                                               (200, 3, 23, 64, 0)])
def test_factors_per_shell(NA, NF, ns, NM, shape):
    from sassena_amd import ScatterDevice, synth
    rng = np.random.default_rng(ns * NA)
    xyz = synth.random_walk(rng, NA, NF, 12.0, 0.1)
    u = synth.orientations(rng, NM)
    qlen = np.sort(rng.uniform(0.1, 4.0, ns))
    bs = rng.uniform(-3, 7, size=(ns, NA))
    with ScatterDevice("all", atom_split=1, tile_shape=shape) as dev:
        dev.stage(xyz)
        fqt, fq, fq2 = dev.compute_oriented(qlen, u, b_shell=bs)
        for s in range(ns):
            dev.set_factors(bs[s])
            r, rq, rq2 = dev.compute_oriented(qlen[s:s + 1], u)
            f0 = abs(r[0, 0])
            assert np.max(np.abs(fqt[s] - r[0])) < TOL * f0
            assert abs(fq[s] - rq[0]) < TOL * f0
            assert abs(fq2[s] - rq2[0]) < 2 * TOL * f0 ** 2 * NM
