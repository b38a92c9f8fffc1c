"""Chunk lengths of the two-layer kernels around the edges of their pair rows:
a wave's 16-pair sub-tiles, the four sub-tiles whose per-pair values it forms
at once (256 pairs of a workgroup) and their refills, against the same pairs in
chunks of 64 (one sub-tile per wave, no refill)."""
import pytest
import torch

from fbpinns_amd import autotune
from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu

# layer sizes, schema
NETS = [([1, 16, 16, 1], (1, 1)), ([2, 32, 32, 1], (3, 3)), ([3, 64, 64, 1], (7, 7)), ([2, 64, 64, 1], (0, 0))]


@pytest.mark.parametrize("n", [1, 17, 64, 65, 255, 256, 257, 512, 529, 1100])
@pytest.mark.parametrize("net", NETS, ids=["-".join(map(str, n[0])) for n in NETS])
def test_chunk_lengths(net, n, monkeypatch):
    """The forward's arithmetic per pair does not depend on the chunk: equal
    bit for bit.  The gradient rows are the same terms, each within 2^-20 of
    exact (split f16 products with float32 sums), added in another order: at
    most 2^-20 plus n ulp of a row of the terms' magnitudes, 1e-4 of its
    largest element with the cancellation of signed terms."""
    ls, (d1, d2) = net
    xd = ls[0]
    lo, hi = (-1.0,) * xd, (1.0,) * xd
    dec_cls, ap = setups.build((1,) * xd, lo, hi, 2.5, ls, seed=2, unnorm=(0.1, 1.3))
    x = setups.uniform_points(n, lo, hi, seed=7).cuda()
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    out = []
    for chunk in (2048, 64):
        monkeypatch.setattr(autotune, "plan_chunk", lambda s, n_cu, chunk=chunk: chunk)
        plan, _ = eng.make_plan(x, schema=(d1, d2))
        th = eng.theta.detach().requires_grad_(True)
        ujet = FBPINNJets.apply(th, plan)
        r = torch.rand(ujet.shape, generator=torch.Generator().manual_seed(n)).cuda() + 0.1
        g, = torch.autograd.grad(ujet, th, r)
        out.append((plan.wl.n_chunks, ujet.detach(), g))
    (c0, u0, g0), (c1, u1, g1) = out
    print(f"[rows] {ls} n={n} chunks {c0} {c1}", flush=True)
    assert c0 == 1 and c1 == (n + 63) // 64
    assert torch.equal(u0, u1)
    assert torch.isfinite(g0).all() and g0.abs().max() > 0
    assert (g0 - g1).abs().max() <= 1e-4 * g1.abs().max()
