"""Detector sums over the column groups of bands that start and end anywhere (one column, inside the
grid, wrapped, whole grid): each image pixel is the masked sum of the run's own exit wave.  Squares of
FP32 values in at least FP32 (1.2e-7 relative, all terms positive) leave 1e-6 a factor of eight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 320, 512, 1024, 1536])
def test_detector_sums_of_any_band(engine, n):
    import torch
    rng = np.random.default_rng(n)
    D, S = 2, 2
    t = np.exp(1j * rng.normal(0.0, 0.7, (S, n, n))).astype(np.complex64)
    probe = (rng.standard_normal((1, n, n)) + 1j * rng.standard_normal((1, n, n))).astype(np.complex64)
    masks = np.stack([np.ones((n, n)), (rng.random((n, n)) < 0.5).astype(np.float64)])
    td, pd, ad = (torch.tensor(a, device="cuda") for a in (t, probe, masks))
    for lo, length in ((0, n), (5, 1), (n // 3, n // 2), (n - n // 3, 2 * n // 3 + 1), (n - 3, 4)):
        print("case detector sums n=%d band [%d, +%d)" % (n, lo, length), flush=True)
        prop = np.zeros((n, n), np.complex64)
        cols = (lo + np.arange(length)) % n
        prop[:, cols] = np.exp(1j * rng.uniform(-np.pi, np.pi, (n, length)))
        hd = torch.tensor(prop, device="cuda")
        det = torch.zeros((1, 2, D), dtype=torch.float64, device="cuda")
        out = torch.zeros((D, n, n), dtype=torch.complex64, device="cuda")
        job = engine.stem_job(n, n, S, td.data_ptr(), pd.data_ptr(), 1, hd.data_ptr(), ad.data_ptr(), 2, D, D, 3, 1, 2,
                              det.data_ptr(), wrap=True, exit_ptr=out.data_ptr())
        engine.stem_run(job, D, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        power = np.abs(out.cpu().numpy().astype(np.complex128)) ** 2
        for a in range(2):
            for d in range(D):
                want = (power[d] * np.fft.ifftshift(masks[a])).sum()  # masks are centred
                assert abs(float(det[0, a, d]) - want) <= 1e-6 * want
