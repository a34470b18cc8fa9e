"""Copies between host arrays and the device: which route they take, and what they give back. Run on the CPU
(tests/host_hip.py)."""
from tests.host_hip import host_hip  # noqa: F401


def test_every_pinned_buffer_is_used(host_hip):
    """A copy of many chunks goes through all of the pinned memory that the device object holds."""
    host_hip("""
f = gpu.Film(dev, 2048, 1500)
before = H.host_hip_pinned()
for _ in range(4): f.read()
held = H.host_hip_pinned() - before
assert held == 12 * MB, held
""")
