"""The operators' direct path (ops._op): the same results as the registered
custom op, the same version counts, and the custom op wherever something
interposes on operators."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from fbpinns_amd import ops

pytestmark = pytest.mark.gpu


def _args(n=300):
    g = torch.Generator().manual_seed(0)
    seg = torch.tensor([0, 100, 100, n], dtype=torch.int32)
    perm = torch.randperm(n, generator=g).to(torch.int32)
    x = torch.randn(n, generator=g)
    return seg.cuda(), perm.cuda(), x.cuda(), torch.empty(3, device="cuda")


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_direct_call_equals_custom_op():
    seg, perm, x, out = _args()
    want = torch.empty_like(out)
    torch.ops.fbpx.segment_sum(seg, perm, x, want, None)
    v = out._version
    ops.segment_sum(seg, perm, x, out)
    assert torch.equal(out, want) and out._version == v + 1
    ops.segment_sum(seg, perm, x, out, scale=None)     # keywords
    assert torch.equal(out, want) and out._version == v + 2


def test_modes_and_inference_still_see_the_custom_op():
    seg, perm, x, out = _args()
    with _Seen() as seen:
        ops.segment_sum(seg, perm, x, out)
    assert any("fbpx.segment_sum" in s for s in seen.names)
    want = out.clone()
    with torch.inference_mode():
        out2 = torch.empty(3, device="cuda")
        ops.segment_sum(seg, perm, x, out2)
    assert torch.equal(out2, want)


def test_list_arguments_count_their_versions():
    net = [1, 32, 1, 1, 0]
    A, B, q = (torch.randn(2, 50, device="cuda") for _ in range(3))
    a, b = torch.empty(50, 1, device="cuda"), torch.empty(50, 1, device="cuda")
    c, d = torch.empty(50, 1, device="cuda"), torch.empty(50, 1, device="cuda")
    ops.affine_jets(net, 0, 50, A, B, q, [0, 1], [a, b])
    torch.ops.fbpx.affine_jets(net, 0, 50, A, B, q, [0, 1], [c, d])
    assert torch.equal(a, c) and torch.equal(b, d)
    assert (a._version, b._version) == (c._version, d._version)


def test_in_place_update_is_noticed_by_autograd():
    """A parameter updated by an operator between forward and backward is
    refused by autograd's version check, as with the custom op."""
    p = torch.randn(8, device="cuda")
    w = torch.randn(8, device="cuda", requires_grad=True)
    y = (w * p).sum()
    z = torch.zeros(8, device="cuda")
    count = torch.zeros(1, dtype=torch.int32, device="cuda")
    ops.adam_flat(p, z.clone(), z.clone(), torch.ones(8, device="cuda"), count, torch.zeros_like(count), True, 1e-3,
                  0.9, 0.999, 1e-8)
    with pytest.raises(RuntimeError, match="inplace operation"):
        y.backward()


def test_errors_are_the_same():
    seg, perm, x, out = _args()
    for bad in ((seg, perm, x[:-1], out), (seg.long(), perm, x, out), (seg.cpu(), perm, x, out)):
        with pytest.raises(ops.FbpxError):
            ops.segment_sum(*bad)
        with pytest.raises(ops.FbpxError):
            torch.ops.fbpx.segment_sum(*bad, None)
