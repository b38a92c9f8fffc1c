"""The work-list builder at the edges of its kernels' blocks: point counts
around the tile (1,024 points), wave (128) and workgroup (256) sizes, subdomain
counts around the 32-box groups of the inside test and the 1,536-subdomain
window of the counting sort, several levels per point; all arrays equal to the
numpy restatement (integer work, bit for bit)."""

import numpy as np
import pytest
import torch

from fbpinns_amd import ops

from test_gpu_worklist import _ap_from_boxes, _check

pytestmark = pytest.mark.gpu

# points, boxes, dimensions, levels
SIZES = [(1, 1, 1, 1), (127, 31, 2, 1), (128, 32, 3, 1), (129, 33, 1, 2), (255, 64, 2, 3), (257, 65, 3, 1),
         (1023, 40, 2, 1), (1024, 97, 1, 1), (1025, 1535, 2, 1), (2047, 1536, 1, 2), (2500, 1537, 2, 1),
         (1100, 3100, 3, 1)]


@pytest.mark.parametrize("n,m,xd,levels", SIZES)
def test_block_edges(n, m, xd, levels):
    print(f"[edges] n={n} m={m} xd={xd} levels={levels}", flush=True)
    r = np.random.default_rng(n + m)
    x = r.uniform(0, 1, (n, xd)).astype(np.float32)
    c = r.uniform(0, 1, (m, xd)).astype(np.float32)
    half = r.uniform(0.02, 0.25, (m, xd)).astype(np.float32)
    lo, hi = c - half, c + half
    k = min(n, m)
    lo[:k:3, 0] = x[:k:3, 0]        # points exactly on box edges (inclusive)
    hi[:, 0] = np.maximum(hi[:, 0], lo[:, 0])
    ap = _ap_from_boxes(lo, hi, r.integers(0, levels, m))
    for active in (np.ones(m, dtype=int), r.integers(0, 3, m)):
        _check(ap, torch.tensor(x), active, [(64, None, None), (None, 5, 3)])
    # the masked count and fill (inside_models)
    mask = (r.integers(0, 2, m)).astype(np.uint8)
    nt, mt, counts = ops.inside_takes(torch.tensor(x).cuda(), torch.tensor(lo).cuda(), torch.tensor(hi).cuda(),
                                      torch.tensor(mask).cuda())
    want = ((x[:, None] >= lo) & (x[:, None] <= hi)).all(2) & (mask > 0)
    wn, wm = np.nonzero(want)
    assert np.array_equal(nt.cpu().numpy(), wn) and np.array_equal(mt.cpu().numpy(), wm)
    assert np.array_equal(counts.cpu().numpy(), want.sum(1))
