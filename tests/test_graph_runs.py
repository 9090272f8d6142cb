"""Runs that replay a captured slice loop (eight full batches and more) and runs just below that:
bit-identical to plain launches, on repeated calls with other work between them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,batch", [(7, 1), (8, 1), (17, 2), (24, 3), (25, 3)])
def test_graph_runs_equal_plain_runs(engine, depth, batch):
    import torch
    print("case graph depth=%d batch=%d" % (depth, batch), flush=True)
    n, S = 64, 5
    rng = np.random.default_rng(depth)
    t = torch.tensor(np.exp(1j * rng.normal(0, 0.5, (S, n, n))).astype(np.complex64), device="cuda")
    probe = torch.tensor((rng.standard_normal((1, n, n)) + 1j * rng.standard_normal((1, n, n))).astype(np.complex64),
                         device="cuda")
    k = np.fft.fftfreq(n)
    inside = k[:, None] ** 2 + k[None, :] ** 2 <= 1 / 9
    prop = torch.tensor((np.exp(1j * rng.uniform(-3, 3, (n, n))) * inside).astype(np.complex64), device="cuda")
    aper = torch.tensor(rng.random((2, n, n)), device="cuda")
    det = torch.zeros((1, 2, depth), dtype=torch.float64, device="cuda")
    job = engine.stem_job(n, n, S, t.data_ptr(), probe.data_ptr(), 1, prop.data_ptr(), aper.data_ptr(), 2, depth, depth,
                          3, 1, 2, det.data_ptr(), wrap=True)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    engine.stem_run(job, batch, stream=st.cuda_stream)
    torch.cuda.synchronize()
    want = det.cpu().numpy().copy()
    assert want.all()
    for _ in range(3):
        det.zero_()
        torch.cuda.synchronize()
        engine.stem_run(job, batch, graph=True, stream=st.cuda_stream)
        torch.cuda.synchronize()
        assert np.array_equal(det.cpu().numpy(), want)
