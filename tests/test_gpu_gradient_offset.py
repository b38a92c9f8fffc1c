"""Gradients summed over very many pairs whose upstream gradients differ in sign:
an offset that every pair's terms share (rounding to one side) would grow with
their number N, the gradient only with its root.

One subdomain of half-width 1 (normalised points and windows exact), 2^20 points,
upstream gradients +1 or -1.  A pair's terms carry independent relative errors of
a few 2^-23 (float32 rounding, the tanh's 2.5e-7), and their sum as much of the
root of the sum of their squares: 2^-20 of it is allowed.  An offset of 5e-9 of a
term comes to 5e-6 of it."""

import pytest
import torch

from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu

N = 1 << 20


@pytest.mark.parametrize("h", [16, 32, 64])
def test_no_offset(h):
    dec_cls, ap = setups.build((1,), (-1.0,), (1.0,), 1.0, [1, h, h, 1], seed=4)
    gen = torch.Generator().manual_seed(h)
    x = torch.rand((N, 1), generator=gen) * 2 - 1
    r = torch.randint(0, 2, (1, N), generator=gen).float() * 2 - 1
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    plan, _ = eng.make_plan(x.cuda(), schema=(0, 0))
    th = eng.theta.detach().requires_grad_(True)
    g, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, r.cuda())
    (W0, b0), (W1, b1), (W2, b2) = [(W[0].detach().cpu().double(), b[0].detach().cpu().double())
                                    for W, b in ap["trainable"]["network"]["subdomain"]["layers"]]
    x, r = x.double(), r.t().double()
    h1 = torch.tanh(x @ W0.t() + b0)
    h2 = torch.tanh(h1 @ W1.t() + b1)
    d2 = r * W2 * (1 - h2 * h2)          # the pairs' terms of the hidden layers' biases
    d1 = d2 @ W1 * (1 - h1 * h1)
    got, off = g[0].detach().cpu().double(), 0
    for name, d, a in (("W0", d1, x), ("b0", d1, None), ("W1", d2, h1), ("b1", d2, None), ("W2", r, h2),
                       ("b2", r, None)):
        a = torch.ones_like(r) if a is None else a
        want, terms = d.t() @ a, torch.sqrt((d * d).t() @ (a * a))
        e = ((got[off:off + want.numel()] - want.reshape(-1)).norm() / terms.norm()).item()
        off += want.numel()
        print(f"[offset] h={h} {name} {e:.2e}", flush=True)
        assert e <= 2.0 ** -20, (name, e)
