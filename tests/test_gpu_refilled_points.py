"""FusedEngine.model on a buffer of points that is refilled in place, the way a
program evaluates one set of points after another: each call's values are those
of the points that the buffer holds then."""

import torch
import pytest

from fbpinns_amd.engine import FusedEngine
from fbpinns_amd.networks import FCN
from fbpinns_amd.problems import Problem

import setups

pytestmark = pytest.mark.gpu

LO, HI = (-1.0, -1.0), (1.0, 1.0)


def _engine():
    dec_cls, ap = setups.build((3, 3), LO, HI, 1.9, [2, 16, 16, 1], seed=0)
    return FusedEngine(Problem, dec_cls, FCN, ap, device="cuda:0", graph=False)


def _points(seed, n=300):
    return setups.uniform_points(n, LO, HI, seed=seed).cuda()


def test_refilled_buffer():
    eng = _engine()
    a, b = _points(1), _points(2)
    want = [_engine().model(v) for v in (a, b)]
    assert not torch.equal(*want)
    buf = a.clone()
    assert torch.equal(eng.model(buf), want[0])
    assert torch.equal(eng.model(buf), want[0])      # the kept plan
    buf.copy_(b)
    assert torch.equal(eng.model(buf), want[1])
    buf[:] = a
    assert torch.equal(eng.model(buf), want[0])
    big = torch.cat([a, b])                          # views share their base's version
    view = big[:300]
    assert torch.equal(eng.model(view), want[0])
    big[:300] = b
    assert torch.equal(eng.model(view), want[1])


def test_points_in_inference_mode():
    eng = _engine()
    a, b = _points(1), _points(2)
    want = [_engine().model(v) for v in (a, b)]
    with torch.inference_mode():
        buf = a.clone()
        u = eng.model(buf)
        buf.copy_(b)
        v = eng.model(buf)
    assert torch.equal(u, want[0]) and torch.equal(v, want[1])
