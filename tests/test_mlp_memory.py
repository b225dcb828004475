"""The network's device buffers after an allocation that failed (host side only)."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(__file__))
from fakehip import fake_run  # noqa: E402,F401

SETUP = """
from sassena_amd.mlp import MLP
rng = np.random.default_rng(0)
def rows(n):
    return rng.normal(size=(n, 16)).astype(np.float32), rng.normal(size=n).astype(np.float32)
def pointers(kernel):
    "Device pointers of the last launch of the step kernel: x, t, fragments, parameters, y, partials."
    i = max(i for i in range(fake.fake_launches()) if kernel in fake.fake_name(i).decode())
    a = ctypes.cast(fake.fake_arg(i), ctypes.POINTER(ctypes.c_uint64))
    return {"x": a[0], "t": a[1], "y": a[8], "partial": a[9]}
net = MLP(seed=1)
small = rows(64)
"""


def test_partials_after_a_failed_call(fake_run):  # noqa: F811
    fake_run(SETUP + """
net.train(*small, steps=1, batch=64)
assert all(pointers("mlp_step")[k] for k in ("x", "t", "partial"))
fake.fake_memory(1 << 30)
try:
    net.gradients(*rows(1 << 20))     # 1.2 GB of partials
    raise SystemExit("enough memory after all")
except SxError as e:
    assert e.code == -4, e
fake.fake_forget()
net.train(*small, steps=1, batch=64)
p = pointers("mlp_step")
assert p["x"] and p["t"] and p["partial"], p
""")


@pytest.mark.parametrize("limit", [60, 68, 71])
def test_rows_after_a_failed_call(fake_run, limit):  # noqa: F811
    """Inputs, targets or outputs (64 + 4 + 4 MiB) find no room."""
    fake_run(SETUP + f"""
net.predict(small[0])
x = rows(1 << 20)[0]
fake.fake_memory({limit} << 20)
try:
    net.predict(x)
    raise SystemExit("enough memory after all")
except SxError as e:
    assert e.code == -4, e
fake.fake_forget()
net.predict(small[0])
p = pointers("mlp_step")
assert p["x"] and p["y"], p
net.train(*small, steps=1, batch=64)
p = pointers("mlp_step")
assert p["x"] and p["t"] and p["partial"], p
""")
