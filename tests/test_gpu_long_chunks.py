"""The jet kernels against the float64 oracle with chunks of many tiles, so
that what a wave carries from tile to tile is checked too: the pair rows and
their refills, the loads ahead, the sums of dW2 and of the per-unit and bias
gradients and their changes of sign.  Point counts leave a last tile of every
kind (one wave, an odd number of tiles, a full one).  Tolerances as in
tests/test_gpu_jets.py: 1e-5 per jet column, 1e-4 per layer tensor of the
gradient, each against its own largest value."""

import pytest
import torch

from fbpinns_amd import autotune

import setups
from test_gpu_split_limits import _compare, _engine

pytestmark = pytest.mark.gpu

NETS = [([1, 16, 16, 1], (1, 1)), ([2, 16, 16, 1], (3, 1)), ([3, 16, 16, 1], (7, 7)), ([2, 32, 32, 1], (3, 3)),
        ([3, 32, 32, 1], (7, 3)), ([2, 32, 32, 1], (0, 0)), ([2, 64, 64, 1], (3, 1)), ([3, 64, 64, 1], (7, 7)),
        ([3, 64, 64, 1], (7, 0)), ([2, 64, 64, 1], (0, 0)),
        # one hidden layer: loads one sub-tile ahead, or (64 units, six or seven jets) where they are used
        ([1, 16, 1], (1, 1)), ([2, 32, 1], (3, 3)), ([2, 64, 1], (3, 3)), ([3, 64, 1], (7, 0)), ([3, 64, 1], (7, 3)),
        ([3, 64, 1], (7, 7))]


@pytest.mark.parametrize("n", [450, 577, 1100])
@pytest.mark.parametrize("ls,d", NETS, ids=["-".join(map(str, n[0])) + "_%d%d" % n[1] for n in NETS])
def test_one_chunk_of_many_tiles(ls, d, n, monkeypatch):
    print(f"[long] {ls} {d} n={n}", flush=True)
    monkeypatch.setattr(autotune, "plan_chunk", lambda s, n_cu: 2048)
    lo, hi = (-1.0,) * ls[0], (1.0,) * ls[0]
    dec_cls, ap = setups.build((1,) * ls[0], lo, hi, 2.5, ls, seed=2, unnorm=(0.1, 1.3))
    x = setups.uniform_points(n, lo, hi, seed=n)
    eng = _engine(dec_cls, ap)
    assert eng.make_plan(x.cuda(), schema=d)[0].wl.n_chunks == 1
    _compare(eng, ap, x, ls[0], d, 1.0)


@pytest.mark.parametrize("chunk", [320, 2048])
@pytest.mark.parametrize("ls,nsub,d", [([2, 16, 16, 1], (2, 2), (3, 3)), ([2, 32, 32, 1], (3, 2), (3, 1)),
                                       ([3, 64, 64, 1], (2, 2, 2), (7, 7))])
def test_several_long_chunks(ls, nsub, d, chunk, monkeypatch):
    """Subdomains of several chunks of five tiles, or of one of up to 32, with
    the windows of more than one."""
    print(f"[long] {ls} {d} chunk={chunk}", flush=True)
    monkeypatch.setattr(autotune, "plan_chunk", lambda s, n_cu: chunk)
    lo, hi = (-1.0,) * ls[0], (1.0,) * ls[0]
    dec_cls, ap = setups.build(nsub, lo, hi, 1.9, ls, seed=3, unnorm=(0.1, 1.3))
    x = setups.uniform_points(2500, lo, hi, seed=6)
    _compare(_engine(dec_cls, ap), ap, x, ls[0], d, 1.0)
