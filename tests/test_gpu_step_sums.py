"""The sums that end a training step, at the edges of their launch shapes:
Adam over rows in 1,024- and 256-thread workgroups with the step count folded
in or not, the chunk rows' sum in batches of eight, and the residual loss over
the workgroups that finish their sum in one launch and over more of them.
Oracles in float64 on the CPU.
"""
import pytest
import torch

from fbpinns_amd import _lib, ops

pytestmark = pytest.mark.gpu
EPS32 = 2.0 ** -24


@pytest.mark.parametrize("n_rows,P,chunks", [
    (1, 1, 1), (1, 1023, 8), (1, 1025, 9), (320, 1024, 2), (320, 1025, 1), (327681, 1, 1), (37, 97, 17),
])
def test_adam_rows_partial_edges(n_rows, P, chunks):
    """chunks: rows r sums 1 + r % chunks chunk rows.  One update from zero
    moments: m = (1 - b1) g and v = (1 - b2) g^2 within the rounding of a sum
    of up to `chunks` floats and three products; the parameter moves by lr
    times a value in [-1, 1] with that relative error."""
    g = torch.Generator().manual_seed(n_rows + P)
    per = torch.arange(n_rows) % chunks + 1
    rcs = torch.zeros(n_rows + 1, dtype=torch.int32)
    rcs[1:] = per.cumsum(0)
    part = torch.rand(int(rcs[-1]), P, generator=g) + 0.5
    g64 = torch.zeros(n_rows, P, dtype=torch.float64)
    g64.index_add_(0, torch.repeat_interleave(torch.arange(n_rows), per), part.double())
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 1e-8
    dev = "cuda"
    rows = torch.arange(n_rows, dtype=torch.int32).flip(0).contiguous()   # row i of the list is subdomain rows[i]
    th0 = torch.rand(n_rows, P, generator=g)
    th, mu, nu = th0.to(dev), torch.zeros(n_rows, P, device=dev), torch.zeros(n_rows, P, device=dev)
    count = torch.zeros(1, dtype=torch.int32, device=dev)
    done = torch.zeros(1, dtype=torch.int32, device=dev)
    ops.adam_rows_partial(th, mu, nu, part.to(dev), rows.to(dev), rcs.to(dev), count, done, True, lr, b1, b2, eps)
    assert int(count.item()) == 1 and int(done.item()) == 0
    want = g64.flip(0)
    rel = (chunks + 8) * EPS32
    assert ((mu.cpu().double() - 0.1 * want).abs() <= (rel + 4 * EPS32 / 0.1) * 0.1 * want).all()
    assert ((nu.cpu().double() - 0.001 * want ** 2).abs() <= (2 * rel + 4 * EPS32 / 0.001) * 0.001 * want ** 2).all()
    # the bias-corrected first step is g / (|g| + eps) = 1 up to eps / |g|; the
    # corrections divide by 1 - b, which float32 holds to EPS32 / (1 - b)
    step = (th0.double() - th.cpu().double()) / lr
    tol = 2 * (2 * rel + EPS32 / 0.1 + EPS32 / 0.001) + 2 * EPS32 / lr + 2 * eps
    assert ((step - 1.0).abs() <= tol).all()


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("n", [1, 511, 512, 2048, 2049, 2048 * 256, 2048 * 256 + 1])
def test_residual_loss_grid_edges(n, accumulate):
    """loss = weight / n sum (2 a b - 0.5 a)^2; every summand is positive, so
    a float32 sum in any order with at most 40 additions per chain (points of
    a thread, wave, workgroup, grid) keeps a relative error of (40 + 8) ulp."""
    g = torch.Generator().manual_seed(n)
    a, b = torch.rand(n, generator=g) + 0.5, torch.rand(n, generator=g) + 0.5
    want = 0.7 / n * (2.0 * a.double() * b.double() - 0.5 * a.double()).pow(2).sum().item()
    dev = "cuda"
    ad, bd = a.to(dev), b.to(dev)
    coef = torch.tensor([2.0, -0.5], device=dev)
    r = torch.empty(n, device=dev)
    scratch = torch.full((_lib.FBPX_RESIDUAL_BLOCKS,), float("nan"), device=dev)
    done = torch.zeros(1, dtype=torch.int32, device=dev)
    for start in (3.0, 5.0):   # twice: the counter is left at 0
        loss = torch.tensor([start], device=dev)
        ops.residual_loss([ad, bd], [0, 0], [1, -1], coef, 0.7, r, scratch, loss, done, [], [], accumulate)
        total = want + (start if accumulate else 0.0)
        # the terms cancel by at most 2 a b / (2 a b - 0.5 a) <= 2: 4 ulp more on r, 8 on r^2
        assert abs(loss.item() - total) <= 64 * EPS32 * total
        assert int(done.item()) == 0
