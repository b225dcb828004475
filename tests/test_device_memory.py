"""Which kernels a call takes when device memory is short, and that nothing that
ran is refused (host side only, no kernel runs)."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(__file__))
from fakehip import fake_run  # noqa: E402,F401

SETUP = """
GB = 1 << 30
rng = np.random.default_rng(0)
def units(n):
    u = rng.normal(size=(n, 3))
    return u / np.linalg.norm(u, axis=1)[:, None]
def staged(NA, NF, **cfg):
    dev = ScatterDevice("all", **cfg)
    dev.stage(rng.uniform(-9, 9, size=(3, NA, NF)).astype(np.float32))
    dev.set_factors(np.ones(NA))
    return dev
"""

CYLINDER = SETUP + """
fake.fake_memory(64 * GB)
dev = staged(2000, 1024, atom_split=1)
qv = rng.normal(size=(30, 3))
moments = [(0, 0)] + [(l, m) for l in range(1, 17) for m in range(4)]
def call():
    launches()
    dev.compute_multipole("cylinder", qv, moments, axis=(0, 0, 1))
    return launches()
"""


def test_cylinder_call_repeats_with_little_memory_left(fake_run):  # noqa: F811
    """A second call needs nothing more than the first one's buffers."""
    fake_run(CYLINDER + """
assert ran(call(), "cylinder_sums")
fake.fake_memory(fake.fake_used())
names = call()
assert ran(names, "cylinder_sums"), names
""")


def test_cylinder_parts_are_halved_before_the_sums_are_given_up(fake_run):  # noqa: F811
    """From memory for every part of the ranges down to memory for one: the
    sums run, in fewer parts, and leave the margin of 4 GB."""
    fake_run(CYLINDER + """
MB = 1 << 20
staged_only = fake.fake_used()
call()
full = fake.fake_used() - staged_only
grids = []
for room in range(full // MB + 8, 120, -8):
    dev.close()
    fake.fake_memory(64 * GB)
    dev = staged(2000, 1024, atom_split=1)
    fake.fake_memory(fake.fake_used() + 4 * GB + room * MB)
    launches()
    dev.compute_multipole("cylinder", qv, moments, axis=(0, 0, 1))
    i = [i for i in range(fake.fake_launches()) if b"cylinder_sums" in fake.fake_name(i)]
    assert i, (room, launches())
    grids.append(fake.fake_grid(i[0], 0))
assert grids == sorted(grids, reverse=True), grids
assert grids[0] // grids[-1] == 17 and len(set(grids)) == 5, grids   # 17, 8, 4, 2, 1 parts
""")


FEW = SETUP + """
q, u = np.linspace(0.3, 3.0, 40), units(500)
def call(dev, q=q, u=u):
    launches()
    dev.compute_oriented(q, u)
    return launches()
"""


def test_few_frames_without_room_for_the_packed_atoms(fake_run):  # noqa: F811
    """40 frames: the packed copy and its parts would not fit beside the staged
    block; the kernel of a frame a lane runs as it did."""
    fake_run(FEW + """
fake.fake_memory(8 * GB)
dev = staged(200000, 40, dsp="square")
assert ran(call(dev, q[:4]), "amp_few")
dev.close()
dev = staged(200000, 40, dsp="square")
fake.fake_memory(fake.fake_used() + 100 * (1 << 20))
names = call(dev, q[:4])
assert ran(names, "amp_direct") or ran(names, "amp_oriented"), names
assert not ran(names, "amp_few")
""")


def test_stage_reuses_the_memory_of_packed_atoms(fake_run):  # noqa: F811
    """A larger block than before where only the packed copy stands in the way."""
    fake_run(FEW + """
fake.fake_memory(8 * GB)
dev = staged(200000, 40, dsp="square")
assert ran(call(dev, q[:4]), "amp_few")
# the block grows by 100,000 atoms x 64 frames x 12 B; most of it is in the copy (128 MB)
fake.fake_memory(fake.fake_used() + 100 * (1 << 20))
dev.stage(np.zeros((3, 300000, 40), np.float32))
dev.set_factors(np.ones(300000))
fake.fake_memory(16 * GB)
assert ran(call(dev, q[:4]), "amp_few")
""")
