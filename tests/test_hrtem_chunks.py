"""Batches of HRTEM images that leave for the host in several chunks (16 MiB of images each): every image
is bit for bit that of a batch of one chunk, first calls and repeated ones with other draws alike."""
import numpy as np
import pytest

from totem_amd import hrtem

pytestmark = pytest.mark.gpu


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    lam = 0.00417552
    f = (np.arange(n) - n // 2) / (n * 0.01)
    U, V = np.meshgrid(f, f)
    wave = np.fft.fftshift(np.fft.fft2(np.exp(1j * rng.uniform(-0.5, 0.5, (n, n)))))
    pp2 = np.zeros(49)
    pp2[0], pp2[1], pp2[2], pp2[8] = lam, 10.0, 10.0, 1.0e3
    mrr = np.abs(rng.normal(0.0, 5.0, 21)) + 1.0
    return {"lambda": lam, "alafa": 3e-4, "delta_yita": 2.0, "gfsf": 0.9, "mtotal": 1}, pp2, mrr, U, V, wave


@pytest.mark.parametrize("n,chunk,counts", [
    (320, 20, (45, 21, 40)),       # 20 + 20 + 5; 20 + 1; two whole chunks
    (128, 128, (300, 129)),
    (1536, 1, (3,)),               # an image above the chunk size is a chunk of its own
])
def test_chunked_batch_equals_small_batches(engine, n, chunk, counts):
    assert max(1, (16 << 20) // (8 * n * n)) == chunk
    for k, count in enumerate(counts):
        print("case hrtem chunks n=%d count=%d" % (n, count), flush=True)
        fixed = _inputs(n, 10 + k)
        ai = np.random.default_rng(20 + k).random((count, 21))
        img, paras = hrtem.images(*fixed, ai)
        for at in range(0, count, chunk):
            part, rows = hrtem.images(*fixed, ai[at:at + chunk])
            assert np.array_equal(img[at:at + chunk], part)
            assert np.array_equal(paras[at:at + chunk], rows)
