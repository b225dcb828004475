"""The FP64 chain from amplitudes to F(q,t): power spectra, their sums over
chunks of vectors and the back-transform, against numpy on the same amplitudes
(dsp "plain" of one vector at a time returns them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NF,NM", [(1, 1), (2, 3), (63, 5), (64, 17), (65, 70), (511, 2), (513, 130), (2000, 33),
                                   (10241, 2)])
def test_back_transform_of_the_same_amplitudes(NF, NM):
    from sassena_amd import ScatterDevice
    rng = np.random.default_rng(NF + NM)
    NA = 40
    xyz = (rng.uniform(0, 12, size=(3, NA, 1)) + np.cumsum(rng.normal(0, 0.2, size=(3, NA, NF)), axis=2))
    xyz = xyz.astype(np.float32)
    b = rng.choice([-3.74, 6.65, 5.8], size=NA)
    qv = rng.normal(size=(2, NM, 3))
    with ScatterDevice("all", "plain", atom_split=1) as dev:
        dev.stage(xyz)
        dev.set_factors(b)
        A = np.array([[dev.compute_shell(q[m:m + 1])[0] for m in range(NM)] for q in qv])
    with ScatterDevice("all", atom_split=1) as dev:
        dev.stage(xyz)
        dev.set_factors(b)
        fqt, fq, fq2 = dev.compute_shells(qv)
    X = np.fft.fft(A, 2 * NF, axis=2)
    C = np.fft.ifft(np.abs(X) ** 2, axis=2)[:, :, :NF] / np.arange(NF, 0, -1)
    a = C.mean(axis=2)
    ref = C.mean(axis=1)
    # rounding of FP64 transforms, log2(2 NF) passes each way, over the NF - tau products of a lag
    tol = 16 * np.finfo(float).eps * NF * np.log2(4 * NF)
    f0 = np.abs(ref[:, :1])
    assert np.max(np.abs(fqt - ref) / f0) < tol
    assert np.max(np.abs(fq - a.mean(axis=1)) / f0[:, 0]) < tol
    s2 = (np.abs(a) ** 2).mean(axis=1)
    assert np.max(np.abs(fq2 - s2) / f0[:, 0] ** 2) < 2 * tol * NM
