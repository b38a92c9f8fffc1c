"""The split-f16 hidden-layer products at the ends of float32's range, where the
powers of two that scale their operands meet it, against the float64 oracle.
Tolerances: those of tests/test_gpu_jets.py (1e-5 per column, 1e-4 per layer
tensor of the gradient)."""

import numpy as np
import pytest
import torch

from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.ops import FBPINNJets
from fbpinns_amd.problems import Problem

import setups
from oracle import model as om

pytestmark = pytest.mark.gpu


def _setup(ls, nsub, unnorm=(0.1, 1.3), n=333):
    lo, hi = (-1.0,) * ls[0], (1.0,) * ls[0]
    dec_cls, ap = setups.build(nsub, lo, hi, 1.9, ls, seed=1, unnorm=unnorm)
    return dec_cls, ap, setups.uniform_points(n, lo, hi, seed=5)


def _engine(dec_cls, ap):
    return FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)


@pytest.mark.parametrize("sd", [1e6, 1e9, 1e20])
@pytest.mark.parametrize("ls,nsub,d", [([1, 16, 16, 1], (5,), (1, 1)), ([2, 32, 32, 1], (3, 2), (3, 1)),
                                       ([3, 64, 64, 1], (2, 2, 2), (7, 7)), ([2, 64, 64, 1], (2, 2), (0, 0))])
def test_zero_gradients_of_a_large_output_scale(ls, nsub, d, sd):
    """Outputs unnormalised by sd, upstream gradients zero on one half of the
    domain: its subdomains' gradients are exactly zero, the others' finite."""
    print(f"[limits] {ls} {d} sd={sd}", flush=True)
    dec_cls, ap, x = _setup(ls, nsub, unnorm=(0.1, sd))
    eng = _engine(dec_cls, ap)
    plan, _ = eng.make_plan(x.cuda(), schema=d)
    th = eng.theta.detach().requires_grad_(True)
    u = FBPINNJets.apply(th, plan)
    r = torch.randn(u.shape, generator=torch.Generator().manual_seed(0)).cuda()
    g, = torch.autograd.grad(u, th, torch.zeros_like(r))
    assert (g == 0).all()
    r[:, x[:, 0].cuda() < 0] = 0
    g, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, r / sd)
    assert torch.isfinite(g).all()
    right = ap["static"]["decomposition"]["subdomain"]["params"][1][:, 0].cuda() > 0   # reaches x > 0
    assert (g[~right] == 0).all() and (g[right].abs().amax(1) > 0).all()


def _compare(eng, ap, x, xd, d, gscale):
    """Columns of the jets and every layer's gradient against the oracle."""
    plan, _ = eng.make_plan(x.cuda(), schema=d)
    th = eng.theta.detach().requires_grad_(True)
    u = FBPINNJets.apply(th, plan)
    r = torch.randn(u.shape, generator=torch.Generator().manual_seed(0)) * gscale
    g, = torch.autograd.grad(u, th, r.cuda())
    ref, _, _ = setups.oracle_jets(ap, x, xd, *d)
    assert (setups.col_rel_err(u, ref) <= 1e-5).all()
    takes, all_ims, layers, dom, _ = setups.oracle_view(ap, x)
    layers = [(W.requires_grad_(True), b.requires_grad_(True)) for W, b in layers]
    ujs = om.fbpinn_forward(layers, dom, x.double(), takes, om.identity_constraint,
                            om.get_jmaps(setups.schema_request(xd, *d)))
    og = torch.autograd.grad((torch.cat(ujs, 1).T * r.double()).sum(), [t for W, b in layers for t in (W, b)])
    got, off = g.detach().cpu().double()[all_ims], 0
    assert torch.isfinite(got).all()
    for t in og:
        a, b = got[:, off:off + t[0].numel()], t.reshape(len(all_ims), -1)
        off += t[0].numel()
        e = ((a - b).abs().max() / b.abs().max().clamp_min(1e-300)).item()
        print(f"  {tuple(t.shape)} rel err {e:.2e}", flush=True)
        assert e <= 1e-4


@pytest.mark.parametrize("ls,nsub", [([1, 16, 16, 1], (5,)), ([2, 32, 32, 1], (3, 2)), ([3, 64, 64, 1], (2, 2, 2))])
def test_largest_weights(ls, nsub):
    """Hidden weights up to 2^120, which saturate every unit: values and
    gradients of the value."""
    print(f"[limits] {ls} weights", flush=True)
    dec_cls, ap, x = _setup(ls, nsub)
    layers = ap["trainable"]["network"]["subdomain"]["layers"]
    W = layers[1][0]
    layers[1] = (W * (2.0 ** 120 / W.abs().max()), layers[1][1])
    _compare(_engine(dec_cls, ap), ap, x, ls[0], (0, 0), 1.0)


@pytest.mark.parametrize("ls,nsub,d", [([1, 16, 16, 1], (5,), (1, 1)), ([2, 32, 32, 1], (3, 2), (3, 1)),
                                       ([3, 64, 64, 1], (2, 2, 2), (7, 7)), ([3, 64, 64, 1], (2, 2, 2), (0, 0))])
def test_largest_gradients(ls, nsub, d):
    """Upstream gradients of 1e33: the bound the scale is chosen from comes near
    or passes float32's largest value, the gradients do not."""
    print(f"[limits] {ls} {d} gradients", flush=True)
    dec_cls, ap, x = _setup(ls, nsub)
    _compare(_engine(dec_cls, ap), ap, x, ls[0], d, 1e33)


@pytest.mark.parametrize("h", [16, 32, 64])
def test_bits_of_a_weight(h):
    """The first layer's bias gradient where it is one weight per unit: at x = 0
    with zero biases every tanh is 0 and its derivative 1, and with output
    weights of 1 and one hidden weight per column the gradient of u for unit u
    is that weight.  Three f16 pieces (h = 16) hold a float32 whole, two hold it
    to 2^-23 of itself."""
    dec_cls, ap = setups.build((1,), (-1.0,), (1.0,), 1.0, [1, h, h, 1], seed=4)
    gen = torch.Generator().manual_seed(h)
    w = torch.rand(h, generator=gen) + 0.5
    W = torch.zeros(1, h, h)
    W[0, torch.randperm(h, generator=gen), torch.arange(h)] = w
    layers = ap["trainable"]["network"]["subdomain"]["layers"]
    zero = [torch.zeros_like(b) for _, b in layers]
    layers[0], layers[1] = (layers[0][0], zero[0]), (W, zero[1])
    layers[2] = (torch.ones_like(layers[2][0]), zero[2])
    eng = _engine(dec_cls, ap)
    plan, _ = eng.make_plan(torch.zeros(1, 1).cuda(), schema=(0, 0))
    th = eng.theta.detach().requires_grad_(True)
    g, = torch.autograd.grad(FBPINNJets.apply(th, plan), th, torch.ones(1, 1).cuda())
    got = g[0, h:2 * h].cpu()
    err = ((got.double() - w.double()) / w.double()).abs().max().item()
    print(f"[limits] h={h} weight error {err:.2e}", flush=True)
    assert err <= (0.0 if h == 16 else 2.0 ** -23)
