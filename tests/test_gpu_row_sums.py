"""Sums of a subdomain's chunk rows: the error does not grow with the number of
chunks it is cut into.  The rows are added in double and rounded once, so a
sum is within half an ulp of exact (and 2^-40 of the terms' magnitudes for the
additions in double)."""

import numpy as np
import pytest
import torch

from fbpinns_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1], [7, 8, 9], [1, 64, 1000], [5000]])
def test_rows_are_summed_to_half_an_ulp(counts):
    P, n = 97, sum(counts)
    rng = np.random.default_rng(n)
    part = (rng.standard_normal((n, P)) * 10.0 ** rng.uniform(-3, 3, (n, 1)) + 3.0).astype(np.float32)
    rcs = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32)
    rows = torch.arange(len(counts), dtype=torch.int32)
    g = torch.zeros((len(counts), P), device="cuda")
    ops.reduce_rows(torch.tensor(part).cuda(), rows.cuda(), rcs.cuda(), g)
    got = g.cpu().numpy().astype(np.float64)
    for k, (a, b) in enumerate(zip(rcs[:-1].tolist(), rcs[1:].tolist())):
        want = part[a:b].astype(np.float64).sum(0)
        size = np.abs(part[a:b].astype(np.float64)).sum(0)
        assert (np.abs(got[k] - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -40 * size).all(), counts[k]
