"""The propagation passes at every compiled grid side and plan against a complex128 multislice in numpy:
exit waves of a short stack with a propagator of random phases inside the 2/3 band.  An exit wave's
FP32 error grows by about 5e-8 relative L2 a slice (41 slices of 512^2: 1.8e-6), so 1e-6 leaves a
factor of five over the four slices here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 128, 256, 320, 512, 768, 1024, 1536, 2048])
def test_exit_waves_match_numpy(engine, n):
    import torch
    rng = np.random.default_rng(n)
    S, D = 4, 3 if n <= 512 else 2
    np_side = n if n > 1024 else 2 * n if n in (64, 128, 256, 512) else n
    wrap = np_side == n
    step = 7 if wrap else 3
    t = np.exp(1j * rng.normal(0.0, 0.7, (S, np_side, np_side))).astype(np.complex64)
    probe = (rng.standard_normal((1, n, n)) + 1j * rng.standard_normal((1, n, n))).astype(np.complex64)
    k = np.fft.fftfreq(n)
    inside = k[:, None] ** 2 + k[None, :] ** 2 <= 1.0 / 9.0
    prop = (np.exp(1j * rng.uniform(-np.pi, np.pi, (n, n))) * inside).astype(np.complex64)
    ref = []
    for d in range(D):
        rows, cols = (5 + np.arange(n)) % np_side, (2 + d * step + np.arange(n)) % np_side
        psi = probe[0].astype(np.complex128)
        for s in range(S):
            psi = np.fft.fft2(psi * t[s][np.ix_(rows, cols)].astype(np.complex128)) * prop.astype(np.complex128)
            if s + 1 < S:
                psi = np.fft.ifft2(psi)
        ref.append(psi)
    td, pd, hd = (torch.tensor(a, device="cuda") for a in (t, probe, prop))
    aper = torch.ones((1, n, n), dtype=torch.float64, device="cuda")
    before = engine.plan(n)[0]
    try:
        for plan in range(engine.plan_count(n)):
            print("case passes n=%d np=%d plan=%d" % (n, np_side, plan), flush=True)
            engine.set_plan(n, plan)
            det = torch.zeros((1, 1, D), dtype=torch.float64, device="cuda")
            out = torch.zeros((D, n, n), dtype=torch.complex64, device="cuda")
            job = engine.stem_job(n, np_side, S, td.data_ptr(), pd.data_ptr(), 1, hd.data_ptr(), aper.data_ptr(), 1,
                                  D, D, step, 5, 2, det.data_ptr(), wrap=wrap, exit_ptr=out.data_ptr())
            engine.stem_run(job, 2, stream=torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            for d in range(D):
                e = np.linalg.norm(out[d].cpu().numpy() - ref[d]) / np.linalg.norm(ref[d])
                full = float(det[0, 0, d]) / (np.abs(ref[d]) ** 2).sum() - 1
                print("  position %d: rel L2 %.2e, total %.1e" % (d, e, full))
                assert e <= 1e-6 and abs(full) <= 1e-6
    finally:
        engine.set_plan(n, before)
