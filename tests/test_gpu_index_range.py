"""Work lists whose last pairs lie at the end of the int32 index range, where the
kernels' look-ahead (up to 1,024 pairs past a chunk, four pair rows past a
segment) passes it: values and gradients equal those of the same pairs at the
start of a list, bit for bit.  Only the last pairs of the large arrays are
touched."""

import numpy as np
import pytest
import torch

from fbpinns_amd import ops
from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu

PAIRS = 2 ** 31 - 3     # the largest list the builder makes
POINTS, EACH = 107, 3   # three pairs per point, in two chunks


@pytest.mark.parametrize("ls", [[1, 16, 1], [1, 16, 16, 1], [1, 64, 64, 1]], ids=["one", "h16", "h64"])
def test_last_pairs_of_the_range(ls):
    if torch.cuda.mem_get_info()[0] < 48 << 30:
        pytest.skip("needs 48 GiB of free GPU memory")
    dec_cls, ap = setups.build((2,), (-1.0,), (1.0,), 2.5, ls, seed=1)
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    x = setups.uniform_points(POINTS, (-1.0,), (1.0,), seed=2).cuda()
    net = eng.net0.with_schema(0, 0)
    k = POINTS * EACH
    point = np.tile(np.arange(POINTS), EACH)                  # pair order: pass after pass over the points
    slot = (np.arange(k) % POINTS) * EACH + np.arange(k) // POINTS   # a point's pairs are consecutive slots
    cut = [0, 2 * POINTS, k]                                  # subdomain 0 twice per point, subdomain 1 once
    out = []
    for n in (k, PAIRS):
        off = n - k

        def tail(values):
            t = torch.empty(n, dtype=torch.int32, device="cuda")
            t[off:] = torch.as_tensor(values, dtype=torch.int32, device="cuda")
            return t

        def i32(values):
            return torch.as_tensor(np.asarray(values), dtype=torch.int32, device="cuda")
        t = {"pair_point": tail(point), "pair_seg": tail(point), "pair_slot": tail(slot + off),
             "chunk_model": i32([0, 1]), "chunk_start": i32([off + c for c in cut]),
             "point_seg_start": i32(np.arange(POINTS + 1)), "seg_pair_start": i32(off + EACH * np.arange(POINTS + 1)),
             "fbin_chunk_start": i32([0, 1, 2]), "bbin_chunk_start": i32([0, 1, 2])}
        wl = ops.Worklist(t, {"n_pairs": n, "n_chunks": 2, "n_points": POINTS, "n_segs": POINTS, "npou": 1,
                              "n_fbins": 2, "n_bbins": 2})
        wsum = torch.empty((POINTS, 1), device="cuda")
        plan = ops.Plan(net, eng.dom, x, wl, wsum, torch.ones(2, dtype=torch.uint8, device="cuda"), i32([0, 1]),
                        i32([0, 1, 2]), eng.m)
        print(f"[range] {ls} {n} pairs", flush=True)
        ops.pou_prepare(net.as_list(), eng.dom, x, wl.tensor_list(), wl.size_list(), plan.pairbuf, wsum)
        th = eng.theta.detach().requires_grad_(True)
        u = FBPINNJets.apply(th, plan)
        r = torch.randn(u.shape, generator=torch.Generator().manual_seed(3)).cuda()
        g, = torch.autograd.grad(u, th, r)
        out.append((wsum.clone(), u.detach(), g))
        del t, wl, plan
        torch.cuda.empty_cache()
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and a.abs().max() > 0 and torch.equal(a, b)
