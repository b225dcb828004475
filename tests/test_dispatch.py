"""Which kernels a call launches, on both sides of the rules that choose them:
what the comparisons of one path with another rely on (host side only)."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(__file__))
from fakehip import fake_run  # noqa: E402,F401

SETUP = """
rng = np.random.default_rng(0)
def staged(NA, NF, *args, **cfg):
    dev = ScatterDevice("all", *args, **cfg)
    dev.stage(rng.uniform(-9, 9, size=(3, NA, NF)).astype(np.float32))
    dev.set_factors(np.ones(NA))
    launches()
    return dev
def units(n):
    u = rng.normal(size=(n, 3))
    return u / np.linalg.norm(u, axis=1)[:, None]
"""


def test_multipole_sums(fake_run):  # noqa: F811
    fake_run(SETUP + """
full = {"sphere": lambda L: [(l, m) for l in range(L + 1) for m in range(-l, l + 1)],
        "cylinder": lambda L: [(0, 0)] + [(l, m) for l in range(1, L + 1) for m in range(4)]}
for kind in full:
    for NA, NF, ns, split in ((1, 1, 1, 1), (33, 64, 3, 1), (77, 90, 3, 1), (300, 129, 11, 3), (300, 40, 5, 0)):
        for moments in ([full[kind](L) for L in (0, 1, 4, 10, 16)] + [[(16, 0)], [(7, 2), (0, 0), (7, 2)], [(12, 1), (3, 3)]]):
            with staged(NA, NF, atom_split=split) as dev:
                dev.compute_multipole(kind, rng.normal(size=(ns, 3)), moments, axis=(0, 0, 1))
            names = launches()
            assert ran(names, kind + "_sums_kernel") and not ran(names, "16multipole_kernel"), (kind, NA, moments, names)
    # one degree more, and the option that keeps the moments' own recurrences
    for L, terms in ((17, 0), (4, 3), (4, 2)):
        with staged(77, 90, multipole_terms=terms) as dev:
            dev.compute_multipole(kind, rng.normal(size=(3, 3)), full[kind](L), axis=(0, 0, 1))
        names = launches()
        assert ran(names, "16multipole_kernel") and not ran(names, "_sums_kernel"), (kind, L, terms, names)
""")


def test_few_frames(fake_run):  # noqa: F811
    fake_run(SETUP + """
q = np.linspace(0.1, 4.0, 9)
for NF, NM, few in ((1, 1, 0), (1, 2, 1), (1, 64, 1), (1, 65, 1), (2, 64, 1), (3, 64, 1), (7, 100, 1), (16, 22, 1), (16, 21, 0),
                    (31, 128, 1), (47, 512, 1), (48, 64, 1), (49, 64, 0), (48, 512, 1), (49, 512, 0), (64, 512, 0),
                    (65, 512, 0)):
    for bs in (None, np.ones((9, 300))):
        with staged(300, NF) as dev:
            dev.compute_oriented(q, units(NM), b_shell=bs)
            assert ran(launches(), "amp_few") == bool(few), (NF, NM)
            dev.compute_oriented(q, units(NM), b_shell=bs, noalloc=True)
            assert not ran(launches(), "amp_few"), (NF, NM)
""")


def test_direct_tiles(fake_run):  # noqa: F811
    """As wide as the shells fill: 21 shells in three tiles of 7."""
    fake_run(SETUP + """
for ns, VS in ((1, 1), (3, 3), (7, 7), (8, 8), (9, 5), (15, 8), (21, 7), (40, 8)):
    with staged(300, 100) as dev:
        dev.compute_oriented(np.sort(rng.uniform(0.1, 4.0, ns)), units(20), b_shell=np.ones((ns, 300)))
    names = launches()
    assert ran(names, f"amp_direct_kernelILi{VS}ELb1E"), (ns, names)
""")
