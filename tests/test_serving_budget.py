"""Admission of served requests counts the potential builder's scratch, once (CPU)."""
import numpy as np
import pytest

from totem_amd import serve, specimen, stem
from tests import hipstub

A = 3.905


def _config(n, slices, flag="l", **kw):
    atoms = specimen.perovskite(6, 6, max(1, slices // 2), a=A)
    return stem.StemConfig(atoms=atoms, np_side=n, dx=6 * A / n, n=n, kv=200.0, alpha_mrad=20.0, slice_thickness=A / 2,
                           n_slices=slices, slice_origin=-A / 8, paraflag=flag, width_red=2, hight_red=2, **kw)


def test_second_request_waits_for_the_scratch():
    cfg = _config(512, 20)
    fp, scratch = serve.footprint_bytes(cfg), serve.scratch_bytes(cfg)
    assert scratch > 0
    room = serve.Admission(2 * fp + scratch)
    assert room.fits(cfg)
    room.take(cfg)
    assert room.fits(cfg)                       # the scratch is counted once
    room.take(cfg)
    assert not room.fits(cfg)
    room.release(cfg)
    assert room.fits(cfg)
    tight = serve.Admission(2 * fp + scratch - 1)
    tight.take(cfg)
    assert not tight.fits(cfg)                  # both footprints alone would fit
    assert tight.peak == fp


USED = """
from totem_amd import serve, stem, specimen
import tests.test_serving_budget as case
cfg = case._config(%d, %d, "%s"%s)
inp = stem.prepare(cfg)
corr = cfg.paraflag == "n"
stub.stub_reset_peak()
before = stub.stub_in_use()
engine.build_transmission(cfg.paraflag, cfg.np_side, cfg.n_slices, inp.series_n, inp.ele_n, inp.gx, inp.gy, inp.s2,
                          inp.aper_true, inp.sigma, inp.parameter, 1 << 40,
                          series_n_corr=inp.series_n_corr if corr else None,
                          ele_n_corr=inp.ele_n_corr if corr else None, corr_info_matrix=inp.corr_matrix if corr else None)
inputs = 8 * 2 * cfg.np_side ** 2 + (inp.corr_matrix.nbytes if corr else 0)     # s2, AperTrue, correction tables
print(stub.stub_peak() - before - inputs, serve.scratch_bytes(cfg))
"""


@pytest.mark.parametrize("n,slices,flag,extra", [(256, 4, "l", ""), (512, 20, "l", ""), (512, 20, "n", ""),
                                                 (1024, 40, "n", ""), (512, 8, "p", ", multiceng=1")])
def test_bound_covers_a_build(tmp_path, n, slices, flag, extra):
    """The scratch a build takes, measured on stand-ins of the HIP calls, is within the bound (1 MiB of
    term lists and twiddles beside it)."""
    used, bound = map(int, hipstub.run(tmp_path, USED % (n, slices, flag, extra)).split())
    print("  n=%d slices=%d %s: %.1f MiB of %.1f" % (n, slices, flag, used / 2**20, bound / 2**20))
    assert np.isfinite(used) and used <= bound + (1 << 20)
