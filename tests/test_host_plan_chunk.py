"""Chunk cap of the work lists that nobody times (autotune.plan_chunk) and the
small two-hidden-layer default that takes it."""

import pytest

from fbpinns_amd import autotune as A


@pytest.mark.parametrize("n_pairs,want", [(0, 64), (1, 64), (64 * 512, 64), (64 * 512 + 1, 128), (180_699, 384),
                                          (150_000, 320), (10 ** 9, 384)])
def test_plan_chunk(n_pairs, want):
    assert A.plan_chunk(n_pairs, 256) == want


def test_default_spec_of_small_two_layer_lists():
    assert A.default_spec(13_647, 2, 50, 256) == ("chunks", 64)
    assert A.default_spec(150_000, 2, 400, 256) == ("chunks", 320)
    assert A.default_spec(150_000, 2, 512, 256) == A.DEFAULT_SMALL   # two workgroups per CU already
    assert A.default_spec(13_647, 1, 50, 256) == A.DEFAULT_SMALL     # one hidden layer: its own rules
