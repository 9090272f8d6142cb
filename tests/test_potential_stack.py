"""Potential stacks built several slices per launch, against the FP64 oracle (1e-6 relative L2 of V
and t, the engine's contract): grid sides with one, partial and many tiles, paired and unpaired
frequencies, tabulated (real and complex) and per-slice form factors, a slice without atoms."""
import numpy as np
import pytest

from oracle import potential as opot
from totem_amd import optics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_side,counts,absorptive,shift", [
    (64, (5,), False, 0.0),               # one slice: form factors evaluated in the accumulation
    (64, (3, 0, 9, 1), False, 0.0),       # tabulated; an empty slice
    (128, (40, 33, 0, 31, 65), True, 0.0),  # complex table
    (128, (17, 8), True, 0.25),           # unpaired: every tile
    (320, (7, 129, 2), False, 0.0),       # np/64 odd
    (320, (12,), True, 0.25),
    (512, (64, 1, 20), False, 0.0),
])
def test_stack_matches_oracle(engine, np_side, counts, absorptive, shift):
    import torch
    print("case stack np=%d counts=%s absorptive=%s shift=%g" % (np_side, counts, absorptive, shift), flush=True)
    rng = np.random.default_rng(np_side + len(counts))
    dx, S, J = 0.08, len(counts), sum(counts)
    gx, gy, s2 = optics.reciprocal_grids(np_side, dx)
    gx = gx + shift * (gx[0, 1] - gx[0, 0])
    aper = (rng.random(s2.shape) > 0.1).astype(np.float64)
    two = np.abs(rng.normal(1.0, 0.4, (2, 10)))          # two classes of Lobato rows
    rows = np.zeros((J, 14))
    rows[:, :2] = rng.uniform(0, np_side * dx, (J, 2))
    rows[:, 2] = rng.uniform(0.5, 1.0, J)
    kind = rng.integers(0, 2, J)
    rows[:, 3:13] = two[kind]
    rows[:, 13] = 0.4
    ab = np.abs(rng.normal(0.02, 0.01, (2, 10)))[kind] * np.tile([1.0, 60.0], 5) if absorptive else None
    series = np.array(counts, dtype=np.float64)
    par, sigma = optics.potential_parameter(np_side, dx), optics.interaction_sigma(200.0)
    t = torch.empty((S, np_side, np_side), dtype=torch.complex64, device="cuda")
    args = ("l", np_side, S, series, rows, gx, gy, s2, aper, sigma, par, t.data_ptr())
    engine.build_transmission(*args, absorp_n=ab, stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = t.cpu().numpy().astype(np.complex128)
    vre, vim = engine.build_transmission(*args, absorp_n=ab, want_v=True,
                                         stream=torch.cuda.current_stream().cuda_stream)
    V, tt = opot.potential_slices(np_side, rows, ab, None, None, series, None, s2, gx, gy, sigma, par, aper, "l")
    for s in range(S):
        v = vre[s] + 1j * vim[s]
        if counts[s] == 0:
            assert not v.any() and (got[s] == 1).all()
            continue
        ev = np.linalg.norm(v - V[s]) / np.linalg.norm(V[s])
        et = np.linalg.norm(got[s] - tt[s]) / np.linalg.norm(tt[s])
        print("  slice %d: V %.2e t %.2e" % (s, ev, et))
        assert ev <= 1e-6 and et <= 1e-6


@pytest.mark.parametrize("change", ["none", "weight", "order", "shorter", "place"])
def test_corrections_that_repeat_their_atoms(engine, change):
    """Correction rows at their atoms' places and weights share the atoms' structure-factor sums; rows that
    differ in one weight, in order, in number or in one place have sums of their own."""
    import torch
    print("case repeated runs change=%s" % change, flush=True)
    rng = np.random.default_rng(11)
    np_side, dx, counts = 128, 0.08, (37, 300, 5)
    gx, gy, s2 = optics.reciprocal_grids(np_side, dx)
    par, sigma = optics.potential_parameter(np_side, dx), optics.interaction_sigma(200.0)
    J, S = sum(counts), len(counts)
    coeff = np.abs(rng.normal(1.0, 0.4, (2, 10)))
    rows, corr = np.zeros((J, 13)), np.zeros((J, 5))
    rows[:, :2] = rng.uniform(0, np_side * dx, (J, 2))
    rows[:, 2] = rng.uniform(0.5, 1.0, J)
    kind = rng.integers(0, 2, J)
    rows[:, 3:13] = coeff[kind]
    corr[:, :2], corr[:, 3], corr[:, 4] = rows[:, :2], rows[:, 2], 1 + kind
    series = np.array(counts, dtype=np.float64)
    series_c = series.copy()
    if change == "weight":
        corr[40, 3] *= 0.5
    elif change == "order":
        corr[37:337] = corr[37:337][::-1]
    elif change == "shorter":
        corr, series_c = np.delete(corr, 100, axis=0), series - np.array([0, 1, 0])
    elif change == "place":
        corr[200, 0] += 0.3
    table = np.stack([0.3 * np.exp(-s2), 0.1 / (1 + s2)])
    aper = np.ones_like(s2)
    t = torch.empty((S, np_side, np_side), dtype=torch.complex64, device="cuda")
    V, _ = opot.potential_slices(np_side, rows, None, None, None, series, None, s2, gx, gy, sigma, par, aper, "n",
                                 ele_n_corr=corr, corr_matrix=table, series_n_corr=series_c)
    vre, vim = engine.build_transmission("n", np_side, S, series, rows, gx, gy, s2, aper, sigma, par, t.data_ptr(),
                                         series_n_corr=series_c, ele_n_corr=corr, corr_info_matrix=table, want_v=True,
                                         stream=torch.cuda.current_stream().cuda_stream)
    for s in range(S):
        ev = np.linalg.norm(vre[s] + 1j * vim[s] - V[s]) / np.linalg.norm(V[s])
        print("  slice %d: V %.2e" % (s, ev))
        assert ev <= 1e-6
