"""Memory of a plan: the per-chunk gradient rows come with the first backward."""

import pytest
import torch

from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu


def test_gradient_rows_are_allocated_by_the_backward():
    lo, hi = (-1.0, -1.0), (1.0, 1.0)
    dec_cls, ap = setups.build((4, 4), lo, hi, 1.9, [2, 64, 64, 1], seed=0)
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    x = setups.uniform_points(20000, lo, hi, seed=1).cuda()
    eng.make_plan(x)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    plan, takes = eng.make_plan(x)
    rows = 4 * plan.wl.n_chunks * plan.net.P
    held = torch.cuda.memory_allocated() - before
    assert plan.wl.n_chunks > 16 and held < 256 * plan.wl.n_pairs + rows // 2
    th = eng.theta.detach().requires_grad_(True)
    before = torch.cuda.memory_allocated()
    u = FBPINNJets.apply(th, plan)
    assert torch.cuda.memory_allocated() - before < rows // 2
    g, = torch.autograd.grad(u, th, torch.ones_like(u))
    first = plan.partial.data_ptr()
    g2, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, torch.ones_like(u))
    assert plan.partial.data_ptr() == first and torch.equal(g, g2) and g.abs().max() > 0
