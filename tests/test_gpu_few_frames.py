"""Trajectories of few frames, one orientation a lane, against the form with
one frame a lane (which the allocation-free call keeps): the same operations on
the same groups of atoms, so amplitudes differ by at most one FP32 rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -22


@pytest.mark.parametrize("NA,NF,ns,NM,split,scan,per_shell", [
    (1, 1, 1, 64, 1, "list", False), (63, 1, 4, 65, 1, "scan", False), (700, 1, 41, 130, 2, "scan", False),
    (640, 2, 9, 64, 3, "exact", False), (1500, 7, 17, 100, 1, "scan", False), (300, 31, 8, 128, 1, "list", True),
    (321, 47, 21, 512, 1, "scan", False), (2000, 3, 20, 64, 16, "exact", True)])
@pytest.mark.parametrize("dsp", ["autocorrelate", "square", "plain"])
def test_few_frames(NA, NF, ns, NM, split, scan, per_shell, dsp):
    from sassena_amd import ScatterDevice, synth
    rng = np.random.default_rng(NA + NF)
    xyz = synth.random_walk(rng, NA, NF, (NA / 0.1) ** (1 / 3), 0.1)
    b = synth.scattering_lengths(rng, NA)
    u = synth.orientations(rng, NM)
    qlen = {"list": np.sort(rng.uniform(0.1, 4.0, ns)), "scan": synth.linear_shells(0.1, 4.0, ns),
            "exact": synth.exact_linear_shells(0.1, 4.0, ns)}[scan]
    bs = np.abs(b)[None] * np.exp(-0.05 * qlen[:, None] ** 2) if per_shell else None
    with ScatterDevice("all", dsp, atom_split=split) as dev:
        dev.stage(xyz)
        dev.set_factors(b)
        fqt, fq, fq2 = dev.compute_oriented(qlen, u, b_shell=bs)
        rfqt, rfq, rfq2 = dev.compute_oriented(qlen, u, b_shell=bs, noalloc=True)
    # the scale of a shell: the largest |F(q,t)| and, for amplitudes that cancel, their mean square
    f0 = np.maximum(np.abs(rfqt).max(axis=1), np.sqrt(np.abs(rfq2)))
    assert np.max(np.abs(fqt - rfqt) / f0[:, None]) < TOL
    assert np.max(np.abs(fq - rfq) / f0) < TOL
    assert np.max(np.abs(fq2 - rfq2) / f0 ** 2) < 2 * TOL


@pytest.mark.parametrize("NF,NM", [(1, 3), (5, 33), (16, 7), (33, 40), (64, 20), (130, 9)])
@pytest.mark.parametrize("dsp", ["square", "plain"])
def test_series_sums(NF, NM, dsp):
    """dsp square and plain over vectors, from the amplitudes of one vector at a time."""
    from sassena_amd import ScatterDevice
    rng = np.random.default_rng(NF * NM)
    xyz = rng.uniform(0, 9, size=(3, 50, NF)).astype(np.float32)
    qv = rng.normal(size=(2, NM, 3))
    with ScatterDevice("all", "plain", atom_split=1) as one, ScatterDevice("all", dsp, atom_split=1) as dev:
        for d in (one, dev):
            d.stage(xyz)
            d.set_factors(np.ones(50))
        A = np.array([[one.compute_shell(q[m:m + 1])[0] for m in range(NM)] for q in qv])
        fqt, fq, fq2 = dev.compute_shells(qv)
    S = np.abs(A) ** 2 if dsp == "square" else A
    a = S.mean(axis=2)
    # FP64 sums over at most NM vectors or NF frames
    tol = 4 * np.finfo(float).eps * (NM + NF) * np.max(np.abs(S))
    assert np.max(np.abs(fqt - S.mean(axis=1))) < tol
    assert np.max(np.abs(fq - a.mean(axis=1))) < tol
    assert np.max(np.abs(fq2 - (np.abs(a) ** 2).mean(axis=1))) < 2 * tol * np.max(np.abs(S))
