"""myProjectfun's device conversion of the double probes and propagator: the call's images are those of
a resident run with the host's rounding (optics.unit_complex64 for the propagator), bit for bit, for
propagators with unit-modulus, scaled, zero and axis values."""
import numpy as np
import pytest

from totem_amd import optics, stem
from totem_amd import specimen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,members", [(64, 1), (64, 3), (128, 1)])
def test_call_equals_resident_run(engine, n, members):
    import torch
    print("case call conversion n=%d members=%d" % (n, members), flush=True)
    a, dz = 3.905, 3.905 / 2
    cfg = stem.StemConfig(atoms=specimen.perovskite(2, 2, 2, a=a), np_side=256, dx=2 * a / 256, n=n, kv=200.0,
                          alpha_mrad=20.0, slice_thickness=dz, n_slices=4, slice_origin=-dz / 4, paraflag="l",
                          detectors_mrad=((60.0, 200.0), (0.0, 30.0)), width_red=3, hight_red=2, step=5, begin_row=9,
                          begin_col=14, focal_members=members, focal_rms_nm=3.0 if members > 1 else 0.0)
    inp = stem.prepare(cfg)
    rng = np.random.default_rng(n)
    h = np.exp(1j * rng.uniform(-np.pi, np.pi, (n, n)))
    h[rng.random((n, n)) < 0.3] = 0.0
    h[0, :8] = [1, -1, 1j, -1j, np.sqrt(0.5) * (1 + 1j), 0.5, 0.25j, 0]
    inp.psf = h
    call = stem.run(inp)[0]
    t = torch.empty((cfg.n_slices, 256, 256), dtype=torch.complex64, device="cuda")
    st = torch.cuda.Stream()
    engine.build_transmission("l", 256, cfg.n_slices, inp.series_n, inp.ele_n, inp.gx, inp.gy, inp.s2, inp.aper_true,
                              inp.sigma, inp.parameter, t.data_ptr(), stream=st.cuda_stream)
    probes = torch.tensor(inp.probe.astype(np.complex64), device="cuda")
    prop = torch.tensor(optics.unit_complex64(h), device="cuda")
    aper = torch.tensor(inp.aper, device="cuda")
    M, D = len(inp.gfsf), cfg.depth
    det = torch.zeros((1, 2, M * D), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    job = engine.stem_job(n, 256, cfg.n_slices, t.data_ptr(), probes.data_ptr(), M, prop.data_ptr(), aper.data_ptr(), 2,
                          D, cfg.width_red, cfg.step, cfg.begin_row - 1, cfg.begin_col - 1, det.data_ptr())
    engine.stem_run(job, M * D, stream=st.cuda_stream)
    torch.cuda.synchronize()
    d = det.cpu().numpy()[0].reshape(2, M, D)
    want = np.zeros((2, D))
    for m in range(M):
        want += d[:, m] * inp.gfsf[m]
    assert np.array_equal(call.T, want)
