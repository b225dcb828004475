"""Multipole lists of few moments and calls of few atoms: sphere lists of at most
eight pairs of orders, whose factors start at their lowest degree and order, and
cylinder ranges cut into parts of eight atoms, against the kernel that runs every
recurrence per moment (multipole_terms = 3): the same atom ranges in FP64, so
amplitudes differ by at most one FP32 rounding, 2^-23 relative in F."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2.0 ** -22


def compare(kind, moments, ns, NA, NF, split, axis=(0.0, 0.0, 1.0)):
    from sassena_amd import ScatterDevice
    rng = np.random.default_rng(NA + NF + ns)
    xyz = rng.uniform(-9, 9, size=(3, NA, 1)) + np.cumsum(rng.normal(0, 0.3, size=(3, NA, NF)), axis=2)
    xyz = xyz.astype(np.float32)
    b = rng.choice([-3.74, 0.0, 6.65, 5.80], size=NA)
    b[0] = 6.65
    if NA > 3:
        b[1:3] = 5.8
        xyz[:, 1, 0] = 0.0    # r = 0
        xyz[:, 2] *= 1e-4     # every degree in the downward recurrence
    qv = np.linspace(0.2, 3.0, ns)[:, None] * np.array([0.48, 0.6, 0.64])
    out = []
    for terms in (0, 3):
        with ScatterDevice("all", atom_split=split, multipole_terms=terms) as dev:
            dev.stage(xyz)
            dev.set_factors(b)
            out.append(dev.compute_multipole(kind, qv, moments, axis=axis))
    a, r = out
    f0 = np.abs(r[0][:, :1])
    assert np.all(np.isfinite(a[0]))
    assert np.max(np.abs(a[0] - r[0]) / f0) < TOL
    assert np.max(np.abs(a[1] - r[1]) / f0[:, 0]) < TOL
    assert np.max(np.abs(a[2] - r[2]) / f0[:, 0] ** 2) < 2 * TOL * a[0].shape[1]


@pytest.mark.parametrize("moments", [[(0, 0)], [(1, 0)], [(1, -1)], [(2, 2), (2, -2)], [(16, 0)], [(16, -16)], [(15, 15), (16, 15)],
                                     [(3, 2), (5, 3), (4, -2)], [(12, 5), (0, 0)], [(l, 8) for l in range(9, 17)],
                                     [(l, m) for l in range(4) for m in range(-l, l + 1)]])
@pytest.mark.parametrize("ns,NA,NF,split", [(1, 1, 1, 1), (3, 33, 64, 1), (4, 300, 70, 2)])
def test_sphere_lists_of_few_pairs(moments, ns, NA, NF, split):
    compare("sphere", moments, ns, NA, NF, split)


@pytest.mark.parametrize("moments", [[(0, 0)], [(1, 2)], [(16, 0)], [(10, 1), (11, 3)], [(8, 2), (0, 0), (1, 1)],
                                     [(l, m) for l in range(1, 17) for m in range(4)]])
@pytest.mark.parametrize("ns,NA,NF,split", [(1, 1, 1, 1), (1, 9, 3, 1), (3, 15, 64, 1), (2, 65, 65, 1), (5, 200, 70, 3)])
def test_cylinder_parts(moments, ns, NA, NF, split):
    compare("cylinder", moments, ns, NA, NF, split, axis=(0.2, -0.1, 0.9))
