"""The counting sort of the work-list builder around its 512-point blocks and
their deal to eight dies (a grid of a multiple of eight workgroups, some of them
past the last block): all arrays equal to the numpy restatement, bit for bit."""

import numpy as np
import pytest
import torch

from test_gpu_worklist import _ap_from_boxes, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,xd", [(63, 5, 1), (511, 40, 2), (512, 40, 3), (513, 7, 1), (4095, 33, 2), (4096, 9, 1),
                                    (4097, 64, 3), (4609, 1536, 2), (8193, 12, 1)])
def test_blocks_and_dies(n, m, xd):
    print(f"[blocks] n={n} m={m} xd={xd}", flush=True)
    r = np.random.default_rng(n)
    x = r.uniform(0, 1, (n, xd)).astype(np.float32)
    c = r.uniform(0, 1, (m, xd)).astype(np.float32)
    half = r.uniform(0.02, 0.25, (m, xd)).astype(np.float32)
    ap = _ap_from_boxes(c - half, c + half, r.integers(0, 2, m))
    _check(ap, torch.tensor(x), np.ones(m, dtype=int), [(64, None, None), (None, 5, 3)])
