"""An upstream gradient whose negative bit is set (autograd hands one on from a
conjugated imaginary part) gives the gradients of its value."""

import torch
import pytest

from fbpinns_amd import ops
from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu


def test_jets_gradient():
    lo, hi = (-1.0, -1.0), (1.0, 1.0)
    dec_cls, ap = setups.build((2, 2), lo, hi, 1.9, [2, 16, 16, 1], seed=0)
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    plan, _ = eng.make_plan(setups.uniform_points(200, lo, hi, seed=1).cuda(), schema=(3, 0))
    th = eng.theta.detach().requires_grad_(True)
    r = torch.randn(3, 200, generator=torch.Generator().manual_seed(2)).cuda()
    want, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, r)
    neg = torch._neg_view(-r)
    assert neg.is_neg() and torch.equal(neg, r)
    got, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, neg)
    assert torch.equal(got, want) and want.abs().max() > 0


def test_residual_loss_of_a_conjugate():
    """d |conj(i loss)| = d loss for a positive loss."""
    u = torch.randn(500, 1, generator=torch.Generator().manual_seed(3)).cuda()
    coef, done = torch.tensor([1.5], device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    grads = []
    for conj in (False, True):
        v = u.clone().requires_grad_(True)
        loss = ops.ResidualLoss.apply(coef, 0.5, [0], [-1], done, v)
        if conj:
            torch.complex(torch.zeros_like(loss), loss).conj().abs().backward()
        else:
            loss.backward()
        grads.append(v.grad)
    assert grads[0].abs().max() > 0
    assert (grads[0] - grads[1]).abs().max() <= 2.0 ** -22 * grads[0].abs().max()   # the modulus' rounding


def test_zero_tensor_is_refused():
    """A zero tensor of autograd's has no memory: an error before any launch."""
    z = torch._efficientzerotensor(3, device="cuda")
    seg = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device="cuda")
    perm = torch.arange(3, dtype=torch.int32, device="cuda")
    with pytest.raises(ops.FbpxError):
        ops.segment_sum(seg, perm, z, torch.empty(3, device="cuda"))
