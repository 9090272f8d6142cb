"""A batch of HRTEM images that fails on the way leaves no copy into the caller's arrays behind.
Host code only, on stand-ins of the HIP calls (tests/hipstub)."""
import pytest

from tests import hipstub

PROGRAM = """
n, B = 64, 1100                                   # three chunks of images
g = np.arange(n * n, dtype=np.float64).reshape(n, n)
ai = np.zeros((B, 21))
def call():
    return engine.hrtem_images(n, 2.5e-3, 0.1, 1.0, 1.0, 1, g, g, g.astype(complex), np.zeros(49), np.zeros(21), ai)
call()
assert stub.stub_pending() == 0
stub.stub_fail_copy(%d)
try:
    call()
except engine.TotemError:
    pass
else:
    raise SystemExit("the failing copy went unnoticed")
print("pending", stub.stub_pending())
stub.hipGetLastError()
call()                                            # the scratch is usable again
assert stub.stub_pending() == 0
"""


@pytest.mark.parametrize("copy", [1, 2, 3])       # copy 0 is the parameter rows'
def test_failed_batch_leaves_no_copy_behind(tmp_path, copy):
    assert "pending 0" in hipstub.run(tmp_path, PROGRAM % copy)


MANY_CHUNKS = """
n, B = 1536, 70                                   # an image of 18 MiB is above a chunk's size
g = np.zeros((n, n))
engine.hrtem_images(n, 2.5e-3, 0.1, 1.0, 1.0, 1, g, g, g.astype(complex), np.zeros(49), np.zeros(21), np.zeros((B, 21)))
print("events", stub.stub_events())
assert stub.stub_events() <= 64 and stub.stub_pending() == 0
"""


def test_events_kept_are_bounded(tmp_path):
    """A batch of any size leaves in at most 64 chunks: the events kept for them stay few."""
    hipstub.run(tmp_path, MANY_CHUNKS)
