"""dsp square and plain over many frames: where a vector's frames go to a whole
workgroup (from 256 frames, or from 65 where its chunk has fewer than four
vectors) and on both sides of these lines, against the amplitudes of one vector
at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NF,ns,NM", [(64, 2, 3), (65, 2, 1), (130, 2, 9), (255, 400, 8), (255, 300, 10), (256, 2, 5),
                                      (257, 1, 3), (1000, 2, 4), (5000, 1, 2), (256, 1024, 70)])
@pytest.mark.parametrize("dsp", ["square", "plain"])
def test_series_means(NF, ns, NM, dsp):
    from sassena_amd import ScatterDevice
    rng = np.random.default_rng(NF + NM)
    xyz = rng.uniform(0, 9, size=(3, 20, NF)).astype(np.float32)
    qv = rng.normal(size=(ns, NM, 3))
    with ScatterDevice("all", "plain", atom_split=1) as one, ScatterDevice("all", dsp, atom_split=1) as dev:
        for d in (one, dev):
            d.stage(xyz)
            d.set_factors(np.ones(20))
        A = one.compute_shells(qv.reshape(ns * NM, 1, 3))[0].reshape(ns, NM, NF)
        fqt, fq, fq2 = dev.compute_shells(qv)
    S = np.abs(A) ** 2 if dsp == "square" else A
    a = S.mean(axis=2)
    # FP64 sums over at most NM vectors or NF frames
    tol = 4 * np.finfo(float).eps * (NM + NF) * np.max(np.abs(S))
    assert np.max(np.abs(fqt - S.mean(axis=1))) < tol
    assert np.max(np.abs(fq - a.mean(axis=1))) < tol
    assert np.max(np.abs(fq2 - (np.abs(a) ** 2).mean(axis=1))) < 2 * tol * np.max(np.abs(S))
