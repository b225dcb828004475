"""Host tables that a call copies to the device stay as they are until the copies
are made: copies are made at the next synchronisation here, freed memory is
overwritten at once, and no source may have changed in between."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(__file__))
from fakehip import fake_run  # noqa: E402,F401

SETUP = """
rng = np.random.default_rng(0)
NA, NF = 500, {NF}
u = rng.normal(size=(70, 3))
u /= np.linalg.norm(u, axis=1)[:, None]
q = np.linspace(0.3, 3.0, 21)
bs = rng.normal(size=(21, NA))
dev = ScatterDevice({kind!r}, "square")
dev.stage(rng.uniform(-9, 9, size=(3, NA, NF)).astype(np.float32))
dev.set_factors(np.ones(NA))
{call}
assert fake.fake_launches() > 0
assert fake.fake_stale() == 0, fake.fake_stale()
"""


@pytest.mark.parametrize("NF", [3, 100])
@pytest.mark.parametrize("kind,call", [
    ("all", "dev.compute_oriented(q, u)"),
    ("all", "dev.compute_oriented(np.sort(rng.uniform(0.3, 3.0, 21)), u)"),
    ("all", "dev.compute_oriented(q, u, b_shell=bs)"),
    ("all", "dev.compute_shells(q[:, None, None] * u, b_shell=bs)"),
    ("all", "dev.compute_multipole('sphere', q[:, None] * u[:21], [(l, m) for l in range(7) for m in range(-l, l + 1)])"),
    ("all", "dev.compute_multipole('sphere', q[:, None] * u[:21], [(20, 3)], b_shell=bs)"),
    ("all", "dev.compute_multipole('cylinder', q[:, None] * u[:21], [(0, 0), (5, 1)], axis=(0, 0, 1))"),
    ("self", "dev.compute_oriented(q, u)"),
    ("self", "dev.compute_oriented(q, u, b_shell=bs)")])
def test_sources_of_queued_copies(fake_run, NF, kind, call):  # noqa: F811
    fake_run(SETUP.format(NF=NF, kind=kind, call=call))
