"""The split-f16 hidden-layer products of the two-hidden-layer kernels over the
range of magnitudes their per-chunk scales have to follow: hidden weights from
zero to five times their initial size, upstream gradients from 1e-20 to 1e15
and spread over six decades between the points, against the float64 oracle.

Tolerances: the jets' (1e-5 per column) and the gradients' (1e-4 per layer
tensor) of tests/test_gpu_jets.py, times the factor on the hidden weights: a
relative rounding error of z = W2 h grows with |z|, and the tanh derivatives
turn it into that relative error of their own."""

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

# layer sizes, subdomains, schema
NETS = [([1, 16, 16, 1], (5,), (1, 1)), ([2, 32, 32, 1], (3, 2), (3, 1)), ([2, 64, 64, 1], (2, 2), (3, 0)),
        ([3, 64, 64, 1], (2, 2, 2), (7, 7)), ([3, 16, 16, 1], (2, 2, 2), (7, 3)), ([3, 64, 64, 1], (2, 2, 2), (0, 0))]
SCALES = [(1.0, 1e-20), (1.0, 1e15), (1e-4, 1.0), (5.0, 1.0), (0.0, 1.0), (1.0, 0.0)]


def _setup(net, wscale, n=333):
    ls, nsub, (d1, d2) = net
    lo, hi = (-1.0,) * ls[0], (1.0,) * ls[0]
    dec_cls, ap = setups.build(nsub, lo, hi, 1.9, ls, seed=1, unnorm=(0.1, 1.3))
    layers = ap["trainable"]["network"]["subdomain"]["layers"]
    layers[1] = (layers[1][0] * wscale, layers[1][1])
    x = setups.uniform_points(n, lo, hi, seed=5)
    eng = FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)
    return eng, ap, x


@pytest.mark.parametrize("wscale,gscale", SCALES)
@pytest.mark.parametrize("net", NETS, ids=["-".join(map(str, n[0])) + f"_{n[2][0]}{n[2][1]}" for n in NETS])
def test_scales(net, wscale, gscale):
    print(f"[split] {net} weights x {wscale} gradients x {gscale}", flush=True)
    xd, (d1, d2) = net[0][0], net[2]
    eng, ap, x = _setup(net, wscale)
    plan, _ = eng.make_plan(x.cuda(), schema=(d1, d2))
    th = eng.theta.detach().requires_grad_(True)
    ujet = FBPINNJets.apply(th, plan)
    rng = np.random.default_rng(3)
    r = rng.standard_normal(tuple(ujet.shape)) * 10.0 ** rng.uniform(-6, 0, (1, len(x))) * gscale
    r = torch.tensor(r, dtype=torch.float32)
    g, = torch.autograd.grad(ujet, th, r.cuda())
    factor = max(1.0, wscale)
    ref, _, all_ims = setups.oracle_jets(ap, x, xd, d1, d2)
    err = setups.col_rel_err(ujet, ref)
    print("  columns", err.tolist(), flush=True)
    assert (err <= 1e-5 * factor).all()
    assert torch.isfinite(g).all()
    if gscale == 0.0:
        assert (g == 0).all()
        return
    takes, all_ims, layers, dom, _ = setups.oracle_view(ap, x)
    layers = [(W.requires_grad_(True), b.requires_grad_(True)) for W, b in layers]
    ujs = om.fbpinn_forward(layers, dom, x.double(), takes, om.identity_constraint,
                            om.get_jmaps(setups.schema_request(xd, d1, d2)))
    L = (torch.cat(ujs, 1).T * r.double()).sum()
    og = torch.autograd.grad(L, [t for W, b in layers for t in (W, b)])
    ref_rows = torch.cat([t.reshape(len(all_ims), -1) for t in og], 1)
    got = g.detach().cpu().double()[all_ims]
    off = 0
    for t in og:
        k = t[0].numel()
        a, b = got[:, off:off + k], ref_rows[:, off:off + k]
        off += k
        e = ((a - b).abs().max() / b.abs().max().clamp_min(1e-300)).item()
        print(f"  {tuple(t.shape)} rel err {e:.2e}", flush=True)
        assert e <= 1e-4 * factor


def test_infinite_weight_stays_in_its_subdomain():
    """An infinite hidden weight makes its own subdomain's values NaN and
    leaves every point outside it unchanged, bit for bit."""
    net = NETS[3]
    eng, ap, x = _setup(net, 1.0)
    plan, _ = eng.make_plan(x.cuda(), schema=(0, 0))
    with torch.no_grad():
        u0 = FBPINNJets.apply(eng.theta, plan)
        eng.all_params["trainable"]["network"]["subdomain"]["layers"][1][0][0, 5, 7] = float("inf")
        u1 = FBPINNJets.apply(eng.theta, plan)
    boxes = ap["static"]["decomposition"]["subdomain"]["params"]
    inside0 = ((x >= boxes[0][0].cpu()) & (x <= boxes[1][0].cpu())).all(1).cuda()
    assert inside0.any() and not inside0.all()
    assert torch.equal(u0[:, ~inside0], u1[:, ~inside0])
    assert not torch.isfinite(u1[:, inside0]).any()
