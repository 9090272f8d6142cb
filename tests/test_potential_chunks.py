"""Potential stacks whose phase tables take several chunks (384 MiB each), against FP64 sums formed
slice by slice: term offsets beyond the first chunk, an empty slice, corrections that repeat their
atoms' terms; and a slice of more runs than are searched for repetitions.

Tolerance: the engine's contract, 1e-6 relative L2 of V.  (A chain model, rms error
sqrt((2e-7)^2 + (2.5e-8)^2 n / 16) for n terms of a class, gives 7e-7 at the 10 500 here.)"""
import numpy as np
import pytest

from oracle import potential as opot
from totem_amd import optics

pytestmark = pytest.mark.gpu

N, DX = 1024, 0.08
COUNTS = (16000, 0, 9000, 21000, 3000)       # no corrections: chunks of slices 0-3 and 4; with them, of 0-1, 2, 3 and 4


def _slice_v(rows, kind, gx, gy, factors, par):
    """V of one slice in FP64: sum over classes of factor x (ey^T ex), on the GPU with real products."""
    import torch
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), device="cuda")
    vk = torch.zeros((N, N), dtype=torch.complex128, device="cuda")
    for c, f in enumerate(factors):
        q = rows[kind == c]
        fx, fy = 2 * np.pi * np.outer(gx[0], q[:, 0]), 2 * np.pi * np.outer(gy[:, 0], q[:, 1])     # [N, terms]
        bc, bs = dev(np.cos(fx) * q[:, 2]).T.contiguous(), dev(-np.sin(fx) * q[:, 2]).T.contiguous()
        ac, as_ = dev(np.cos(fy)), dev(-np.sin(fy))
        vk += torch.complex(ac @ bc - as_ @ bs, ac @ bs + as_ @ bc) * dev(f)
    return (torch.fft.ifft2(torch.fft.ifftshift(vk * par)) * N * N).cpu().numpy()


@pytest.mark.parametrize("corrected", [False, True])
def test_stack_of_several_chunks(engine, corrected):
    import torch
    print("case chunks corrected=%s" % corrected, flush=True)
    assert 16 * 528 * sum(COUNTS) > 384 << 20
    rng = np.random.default_rng(5)
    gx, gy, s2 = optics.reciprocal_grids(N, DX)
    par, sigma = optics.potential_parameter(N, DX), optics.interaction_sigma(200.0)
    J, S = sum(COUNTS), len(COUNTS)
    rows = np.zeros((J, 13))
    rows[:, :2] = rng.uniform(0, N * DX, (J, 2))
    rows[:, 2] = rng.uniform(0.5, 1.0, J)
    kind = rng.integers(0, 2, J)
    coeff = np.zeros((2, 10))
    coeff[:, :4] = [[1.0, 0.5, 0.4, 0.02], [0.8, 0.3, 0.6, 0.05]]
    rows[:, 3:] = coeff[kind]
    factors = [a * np.exp(-b * s2) + c * np.exp(-d * s2) for a, b, c, d in coeff[:, :4]]
    series = np.array(COUNTS, dtype=np.float64)
    kw = {}
    if corrected:
        corr = np.zeros((J, 5))
        corr[:, :2], corr[:, 3], corr[:, 4] = rows[:, :2], rows[:, 2], 1 + kind
        table = np.stack([0.3 * np.exp(-s2), 0.1 / (1 + s2)])
        factors = [f + table[c] for c, f in enumerate(factors)]
        kw = dict(series_n_corr=series, ele_n_corr=corr, corr_info_matrix=table)
    t = torch.empty((S, N, N), dtype=torch.complex64, device="cuda")
    vre, vim = engine.build_transmission("n", N, S, series, rows, gx, gy, s2, np.ones_like(s2), sigma, par, t.data_ptr(),
                                         want_v=True, stream=torch.cuda.current_stream().cuda_stream, **kw)
    off = np.concatenate([[0], np.cumsum(COUNTS)])
    for s in range(S):
        got = vre[s] + 1j * vim[s]
        if COUNTS[s] == 0:
            assert not got.any()
            continue
        V = _slice_v(rows[off[s]:off[s + 1]], kind[off[s]:off[s + 1]], gx, gy, factors, par)
        e = np.linalg.norm(got - V) / np.linalg.norm(V)
        print("  slice %d, %d atoms: V %.2e" % (s, COUNTS[s], e), flush=True)
        assert e <= 1e-6


def test_slice_of_many_runs_with_corrections(engine):
    """600 rows with coefficients of their own (600 runs, not searched) beside a slice whose corrections
    repeat its atoms."""
    import torch
    print("case many runs", flush=True)
    rng = np.random.default_rng(6)
    n, counts = 64, (600, 40)
    gx, gy, s2 = optics.reciprocal_grids(n, DX)
    par, sigma = optics.potential_parameter(n, DX), optics.interaction_sigma(200.0)
    J = sum(counts)
    rows, corr = np.zeros((J, 13)), np.zeros((J, 5))
    rows[:, :2] = rng.uniform(0, n * DX, (J, 2))
    rows[:, 2] = rng.uniform(0.5, 1.0, J)
    rows[:, 3:] = np.abs(rng.normal(1.0, 0.4, (J, 10)))          # no two rows alike
    kind = rng.integers(0, 2, J)
    rows[600:, 3:] = rows[[0, 1]][kind[600:], 3:]
    corr[:, :2], corr[:, 3], corr[:, 4] = rows[:, :2], rows[:, 2], 1 + kind
    table = np.stack([0.3 * np.exp(-s2), 0.1 / (1 + s2)])
    series = np.array(counts, dtype=np.float64)
    kw = dict(ele_n_corr=corr, series_n_corr=series)
    stats = engine.potential_plan_stats("n", n, 2, series, rows, gx, gy, s2, np.ones_like(s2), sigma, par,
                                        corr_info_matrix=table, **kw)
    assert stats["classes"] > 512 and not stats["split"]
    t = torch.empty((2, n, n), dtype=torch.complex64, device="cuda")
    vre, vim = engine.build_transmission("n", n, 2, series, rows, gx, gy, s2, np.ones_like(s2), sigma, par, t.data_ptr(),
                                         want_v=True, corr_info_matrix=table,
                                         stream=torch.cuda.current_stream().cuda_stream, **kw)
    V, _ = opot.potential_slices(n, rows, None, None, None, series, None, s2, gx, gy, sigma, par, np.ones_like(s2), "n",
                                 corr_matrix=table, **kw)
    for s in range(2):
        e = np.linalg.norm(vre[s] + 1j * vim[s] - V[s]) / np.linalg.norm(V[s])
        print("  slice %d: V %.2e" % (s, e))
        assert e <= 1e-6
