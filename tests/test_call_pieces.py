"""A myProjectfun call whose probes pass through the conversion's staging in more than one piece (4 Mi
values): the images are those of a resident run on probes rounded on the host, bit for bit."""
import numpy as np
import pytest

from totem_amd import optics, specimen, stem

pytestmark = pytest.mark.gpu


def test_probes_in_two_pieces(engine):
    import torch
    n, side, members, S = 1024, 1536, 5, 2
    print("case call pieces n=%d members=%d" % (n, members), flush=True)
    assert n * n * members > 4 << 20
    a, dz = 3.905, 3.905 / 2
    cfg = stem.StemConfig(atoms=specimen.perovskite(4, 4, 1, a=a), np_side=side, dx=4 * a / side, n=n, kv=200.0,
                          alpha_mrad=20.0, slice_thickness=dz, n_slices=S, slice_origin=-dz / 4,
                          detectors_mrad=((60.0, 200.0),), width_red=2, hight_red=1, step=7, focal_members=members,
                          focal_rms_nm=3.0)
    inp = stem.prepare(cfg)
    inp.probe = inp.probe * (1 + np.arange(members))[:, None, None]      # no two probes alike
    call = stem.run(inp)[0]
    t = torch.empty((S, side, side), dtype=torch.complex64, device="cuda")
    st = torch.cuda.Stream()
    engine.build_transmission("l", side, S, inp.series_n, inp.ele_n, inp.gx, inp.gy, inp.s2, inp.aper_true, inp.sigma,
                              inp.parameter, t.data_ptr(), stream=st.cuda_stream)
    probes = torch.tensor(inp.probe.astype(np.complex64), device="cuda")
    prop = torch.tensor(optics.unit_complex64(inp.psf), device="cuda")
    aper = torch.tensor(inp.aper, device="cuda")
    M, D = len(inp.gfsf), cfg.depth
    det = torch.zeros((1, 1, M * D), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    job = engine.stem_job(n, side, S, t.data_ptr(), probes.data_ptr(), M, prop.data_ptr(), aper.data_ptr(), 1, D,
                          cfg.width_red, cfg.step, cfg.begin_row - 1, cfg.begin_col - 1, det.data_ptr())
    engine.stem_run(job, M * D, stream=st.cuda_stream)
    torch.cuda.synchronize()
    d = det.cpu().numpy()[0].reshape(1, M, D)
    want = np.zeros((1, D))
    for m in range(M):
        want += d[:, m] * inp.gfsf[m]
    assert np.array_equal(call.T, want)
