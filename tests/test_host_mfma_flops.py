"""Matrix-core FLOPs per pair as counted from the kernels' instructions: a
v_mfma_f32_16x16x32_f16 does 2 * 16 * 16 * 32 FLOPs and serves one 16-pair
sub-tile (dW2 at h = 64: the four waves' 64 pairs)."""

import pytest

from fbpinns_amd.configs import mfma_flops_per_pair

INSTR = 2 * 16 * 16 * 32


@pytest.mark.parametrize("h,frag,dw2", [
    (16, 3, 2),                       # one 16-row block; two instructions per dW2 block
    (32, 2 * 3, 4 * 2),               # two row blocks, one K-step of three; four dW2 blocks
    (64, 4 * 2 * 3, 4 * 2 * 3)])      # four row blocks, two K-steps; four blocks of a quadrant, two K-steps, per wave
@pytest.mark.parametrize("n1,n2", [(0, 0), (2, 0), (2, 1), (3, 3)])
def test_counts(h, frag, dw2, n1, n2):
    columns = 1 + (n1 > 0) + n2       # Z_0, the transposed vector or s, one per second derivative
    fwd, bwd = columns * frag, columns * (2 * frag + dw2)
    assert mfma_flops_per_pair(h, 2, n1, n2) == (fwd * INSTR / 16, bwd * INSTR / 16)


def test_one_hidden_layer_has_none():
    assert mfma_flops_per_pair(32, 1, 1, 1) == (0, 0)
