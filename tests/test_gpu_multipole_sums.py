"""The sphere average as sums of radial times angular factors against the
kernel that runs every recurrence per moment (multipole_terms = 3): both in
FP64 over the same atom ranges, so the amplitudes differ by at most one FP32
rounding, 2^-23 relative in F."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -22


def walk(NA, NF, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(-9, 9, size=(3, NA, 1)) + np.cumsum(rng.normal(0, 0.3, size=(3, NA, NF)), axis=2)
    return xyz.astype(np.float32), rng.choice([-3.74, 0.0, 6.65, 5.80], size=NA)


def both(kind, xyz, b, qv, moments, split, b_shell=None, axis=(0.0, 0.0, 1.0)):
    from sassena_amd import ScatterDevice
    out = []
    for terms in (0, 3):
        with ScatterDevice("all", atom_split=split, multipole_terms=terms) as dev:
            dev.stage(xyz)
            dev.set_factors(b)
            out.append(dev.compute_multipole(kind, qv, moments, b_shell=b_shell, axis=axis))
    return out


def check(a, b):
    f0 = np.abs(b[0][:, :1])
    assert np.all(np.isfinite(a[0]))
    assert np.max(np.abs(a[0] - b[0]) / f0) < TOL
    assert np.max(np.abs(a[1] - b[1]) / f0[:, 0]) < TOL
    assert np.max(np.abs(a[2] - b[2]) / f0[:, 0] ** 2) < 2 * TOL * a[0].shape[1]


@pytest.mark.parametrize("lmax,ns,NA,NF,split", [(0, 1, 1, 1, 1), (1, 3, 5, 63, 1), (3, 6, 33, 64, 1), (4, 8, 64, 65, 2),
                                                 (6, 7, 70, 100, 1), (7, 6, 200, 70, 3), (8, 4, 130, 30, 1),
                                                 (10, 5, 300, 40, 2), (10, 11, 129, 129, 1), (12, 3, 90, 64, 1),
                                                 (14, 4, 100, 50, 1), (16, 2, 65, 64, 1)])
def test_sphere_sums(lmax, ns, NA, NF, split):
    xyz, b = walk(NA, NF, lmax + ns)
    b[0] = 6.65
    xyz[:, 0, 0] = 0.0   # r = 0
    qv = np.stack([np.zeros(ns), np.linspace(0.0, 2.5, ns) if ns > 1 else np.array([0.7]), np.zeros(ns)], 1)
    moments = [(l, m) for l in range(lmax + 1) for m in range(-l, l + 1)]
    check(*both("sphere", xyz, b, qv, moments, split))


@pytest.mark.parametrize("moments", [[(5, -3)], [(16, 16), (16, -16), (0, 0)], [(9, 4), (2, 1), (9, 4), (9, -4), (3, 0)],
                                     [(l, m) for l in (13, 2, 7) for m in (2, -2, 1)]])
def test_sphere_sums_of_partial_lists(moments):
    """Lists with gaps, repeats and any order, per-shell factors."""
    xyz, b = walk(77, 90, 3)
    qv = np.array([[0.0, 0.3, 0.0], [1.0, -0.4, 0.8], [4.0, 0.0, 0.1]])
    moments = [mo for mo in moments if abs(mo[1]) <= mo[0]]
    bs = np.random.default_rng(1).uniform(-2, 4, size=(3, 77))
    check(*both("sphere", xyz, b, qv, moments, 1, b_shell=bs))


@pytest.mark.parametrize("lmax,ns,NA,NF,split,axis", [
    (0, 1, 1, 1, 1, (0, 0, 1)), (1, 3, 5, 63, 1, (0, 0, 1)), (2, 2, 33, 64, 1, (0.3, -0.2, 0.9)), (3, 5, 64, 65, 2, (0, 1, 0)),
    (4, 4, 70, 100, 1, (0, 0, 1)), (6, 7, 200, 70, 3, (1, 2, -1)), (8, 3, 130, 30, 1, (0, 0, 1)), (10, 5, 300, 40, 2, (0, 0, -1)),
    (12, 4, 90, 64, 1, (0, 0, 1)), (13, 2, 129, 129, 1, (0.1, 0.1, 0.5)), (16, 6, 65, 64, 1, (0, 0, 1))])
def test_cylinder_sums(lmax, ns, NA, NF, split, axis):
    """q_r r from 0 through the leading terms, Miller's recurrence and the
    asymptotic start, shells along the axis and across it."""
    xyz, b = walk(NA, NF, 100 + lmax + ns)
    b[0] = 6.65
    xyz[:, 0, 0] = 0.0   # r = 0
    if NA > 3:
        b[1:4] = 5.8
        xyz[:, 1] *= 1e-7
        xyz[:, 2] *= 8.0
        xyz[:2, 3] = 0.0
    a = np.asarray(axis, float) / np.linalg.norm(axis)
    q = np.linspace(0.05, 3.0, ns)
    qv = q[:, None] * np.array([0.5, -0.2, 0.8])
    qv[0] = 1.1 * a
    moments = [(0, 0)] + [(l, m) for l in range(1, lmax + 1) for m in range(4)]
    check(*both("cylinder", xyz, b, qv, moments, split, axis=axis))


def test_cylinder_sums_of_partial_lists():
    """A list with gaps and repeats in any order, per-shell factors."""
    xyz, b = walk(77, 90, 5)
    qv = np.array([[0.2, 0.3, 0.0], [1.0, -0.4, 0.8], [4.0, 0.0, 0.1]])
    bs = np.random.default_rng(1).uniform(-2, 4, size=(3, 77))
    check(*both("cylinder", xyz, b, qv, [(7, 2), (1, 1), (0, 0), (7, 2), (11, 3), (4, 0)], 1, b_shell=bs))
