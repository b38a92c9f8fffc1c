"""fbpx_pou_prepare refuses lists its kernels would read through null pointers, or
whose segments it would leave unwritten, before anything is launched."""

import ctypes

import pytest

from fbpinns_amd import _lib


def _call(scratch=8, wsum=8, dom=8, x=8, **wl):
    w = _lib.fbpx_worklist(**dict(dict(n_pairs=4, n_chunks=1, n_points=2, n_segs=2, npou=1, chunk_model=8, chunk_start=8,
                                       pair_point=8, pair_slot=8, point_seg_start=8, seg_pair_start=8), **wl))
    return _lib.lib().fbpx_pou_prepare(None, ctypes.byref(_lib.fbpx_net(1, 32, 1, 1, 1)), dom, x, ctypes.byref(w),
                                       scratch, wsum)


@pytest.mark.parametrize("bad", [dict(n_points=0), dict(point_seg_start=None), dict(seg_pair_start=None),
                                 dict(chunk_model=None), dict(chunk_start=None), dict(pair_slot=None),
                                 dict(scratch=None), dict(wsum=None), dict(dom=None), dict(x=None)])
def test_refused_before_the_launch(bad):
    assert _call(**bad) == -1
    assert "pou_prepare" in _lib.lib().fbpx_last_error().decode()
