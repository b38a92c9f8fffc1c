"""The work-list builder's counting sort where it counts several windows of 1,536
subdomains (blocks of 1,024 points then, 512 otherwise): point counts around one
block and around the eight that the dies are dealt, two and three windows; all
arrays equal to the numpy restatement, bit for bit."""

import numpy as np
import pytest
import torch

from test_gpu_worklist import _ap_from_boxes, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1537, 3073])
@pytest.mark.parametrize("n", [1, 127, 129, 1023, 1024, 1025, 8191, 8192, 8193, 9217])
def test_windows_and_blocks(n, m):
    print(f"[windows] n={n} m={m}", flush=True)
    r = np.random.default_rng(n + m)
    xd = 1 + (n + m) % 3
    x = r.uniform(0, 1, (n, xd)).astype(np.float32)
    c = r.uniform(0, 1, (m, xd)).astype(np.float32)
    half = (r.uniform(0.3, 1.0, (m, xd)) * {1: 0.002, 2: 0.03, 3: 0.08}[xd]).astype(np.float32)
    ap = _ap_from_boxes(c - half, c + half, r.integers(0, 2, m))
    for active in (np.ones(m, dtype=int), r.integers(0, 3, m)):
        _check(ap, torch.tensor(x), active, [(64, None, None), (None, 5, 3)])
