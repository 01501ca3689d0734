"""The sampler's choice of the rank-th candidate, at the edges of its bins.

The kernel counts values into 512 equal bins over at most 16 below the maximum
and orders the selected bin's candidates by comparison where they are at most
64, by index where they are more and all equal, by radix passes otherwise and
where the rank lies further down than the bins. Which path a row takes may not show: the token is the rank-th legal
candidate by (value descending, index ascending), with the kernel's own
support, exactly.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import ppk
from helpers import SEED

pytestmark = pytest.mark.gpu
F32 = np.float32


def rows(kind, choices, batch, rng):
    x = (rng.standard_normal((batch, choices)) * 0.5).astype(F32)
    if kind == "crowded":  # runs of equal values around the list's 64 entries
        x[:] = np.linspace(0, 1, choices, dtype=F32)
        for b in range(batch):
            n = min(choices, 60 + b)
            at = rng.permutation(choices)[:n]
            x[b, at] = F32(0.5)
    elif kind == "outlier":  # one value stretches the range: nearly all in bin 0
        x[:, choices // 2] = -1e6
    elif kind == "equal":  # no range, both zeros
        x[:] = 0.0
        x[:, ::3] = -0.0
    elif kind == "tiny":  # the bins' scale overflows
        x = (rng.integers(0, 3, (batch, choices)) * 1e-44).astype(F32)
    elif kind == "wide":  # the range itself overflows
        x[:, 0] = -3e38
        x[:, -1] = 3e38
    elif kind == "neighbours":  # consecutive floats
        x = (np.full((batch, choices), 4.0, F32).view(np.int32) + rng.integers(0, 2000, (batch, choices), dtype=np.int32)).view(F32)
    return x


@pytest.mark.parametrize("choices", [2, 63, 64, 65, 255, 257, 1000, 2047, 2048])
@pytest.mark.parametrize("kind", ["normal", "crowded", "outlier", "equal", "tiny", "wide", "neighbours"])
def test_rank_names_the_sorted_candidate(device, kind, choices):
    rng = np.random.default_rng(SEED + choices)
    batch = 40
    x = rows(kind, choices, batch, rng)
    start = (np.arange(batch) % 3 % choices).astype(np.uint32)
    count = (choices - start).astype(np.uint32)
    uniform = np.linspace(0, 0.999, batch, dtype=F32)
    uniform[-1] = F32(0.99999994)
    tok, val, sup = ppk.sampling.sample(
        torch.from_numpy(x).to(device), torch.from_numpy(uniform.reshape(-1, 1)).to(device),
        torch.from_numpy(np.stack([start, count], 1).view(np.int32)).to(device), 3.5, 1.0, 1, 5)
    tok, val, sup = (t.reshape(-1).cpu().numpy().view(np.uint32) for t in (tok, val, sup))
    assert np.all(val == 1)
    for b in range(batch):
        legal = x[b, start[b]:start[b] + count[b]]
        assert 1 <= sup[b] <= count[b]
        rank = min(int(F32(uniform[b] * F32(sup[b]))), int(sup[b]) - 1)
        want = 5 + start[b] + np.argsort(-legal.astype(np.float64), kind="stable")[rank]
        assert tok[b] == want, (kind, choices, b, rank, sup[b])


@pytest.mark.parametrize("choices", [2, 65, 300, 2048])
@pytest.mark.parametrize("kind", ["masked", "few_values", "crowded_unequal", "below_the_bins"])
def test_beyond_the_bins_and_crowded_bins(device, kind, choices):
    rng = np.random.default_rng(SEED + 3 * choices)
    batch, alpha = 40, 3.5
    x = (rng.standard_normal((batch, choices)) * 0.5).astype(F32)
    if kind == "masked":  # most values far below, at one value and at several
        x[rng.random((batch, choices)) < 0.9] = -1e4
        x[: batch // 2, ::3] = -60.0
    elif kind == "few_values":  # bins of equal values, zeros of both signs among them
        x = rng.choice(np.array([0.0, -0.0, 0.25, -3.0, -40.0], F32), (batch, choices))
    elif kind == "crowded_unequal":  # more than 64 unequal values in one bin, stretched by one at 15 below
        x = (x * 1e-3).astype(F32)
        x[:, -1] = -15.0
    else:  # alpha next to 1: the entropy's rounding makes supports of all sizes, ranks past the bins among them
        x[:] = np.linspace(0, -200, choices, dtype=F32)[rng.permutation(choices)]
        alpha = float(np.nextafter(F32(1), F32(2)))
    count = np.full(batch, choices, np.uint32)
    uniform = np.linspace(0, 0.999, batch, dtype=F32)
    bounds = np.stack([np.zeros(batch, np.uint32), count], 1)
    tok, val, sup = ppk.sampling.sample(
        torch.from_numpy(x).to(device), torch.from_numpy(uniform.reshape(-1, 1)).to(device),
        torch.from_numpy(bounds.view(np.int32)).to(device), alpha, 1.0, 1, 5)
    tok, val, sup = (t.reshape(-1).cpu().numpy().view(np.uint32) for t in (tok, val, sup))
    assert np.all(val == 1)
    below = 0
    for b in range(batch):
        rank = min(int(F32(uniform[b] * F32(sup[b]))), int(sup[b]) - 1)
        order = np.argsort(-x[b].astype(np.float64), kind="stable")
        assert tok[b] == 5 + order[rank], (kind, choices, b, rank, sup[b])
        below += x[b, order[rank]] < x[b].max() - 16
    if kind == "below_the_bins" and choices == 2048:  # (smaller supports may round to none)
        assert below > 0, "no rank past the bins"
