"""Device memory of a myProjectfun call, on stand-ins of the HIP calls (tests/hipstub): its FP64 staging
is given back before the scan's batch is sized by the free memory."""
import pytest

from tests import hipstub

PROGRAM = """
from totem_amd import stem, specimen
n, M, P = %d, %d, %d
a, S = 3.905, 2
cfg = stem.StemConfig(atoms=specimen.perovskite(2, 2, 1, a=a), np_side=P, dx=2 * a / P, n=n, kv=200.0, alpha_mrad=20.0,
                      slice_thickness=a / 2, n_slices=S, slice_origin=-a / 8, detectors_mrad=((60.0, 200.0),),
                      width_red=2, hight_red=1, focal_members=M, focal_rms_nm=3.0 if M > 1 else 0.0)
inp = stem.prepare(cfg)
assert len(inp.gfsf) == M
stem.run(inp)
kept = 8 * S * P * P + 8 * M * n * n + 8 * n * n + 8 * n * n + 8 * 2 * M    # t, probes, propagator, mask, sums
builder = stub.stub_in_use()                                              # what the call leaves is the builder's
stem.run(inp)                                                             # the builder's scratch is there now
print("staged", stub.stub_in_use_at_info() - builder - kept)
assert stub.stub_in_use() == builder
"""


@pytest.mark.parametrize("n,members,side", [(64, 1, 128), (256, 9, 512), (1024, 5, 1536)])
def test_staging_is_given_back(tmp_path, n, members, side):
    assert "staged 0" in hipstub.run(tmp_path, PROGRAM % (n, members, side))
