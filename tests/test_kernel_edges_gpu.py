"""Kernels and dispatch branches at the sizes where they can go wrong: tile
and launch edges, remainders, the smallest and largest of their range."""
import ctypes

import numpy as np
import pytest
import torch

from aquagpusph_amd import _lib

pytestmark = pytest.mark.gpu


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _dp(t):
    return ctypes.c_void_p(t.data_ptr())


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("cells,cap", [(7, 7), (1000, 60_000_000),
                                       (524_288, 524_289),
                                       (1_100_003, 1_500_000)])
def test_ihoc_table_of_wide_grids(cuda, cells, cap):
    """The head-of-chain table of grids below, at and beyond one pass of the
    bounded launch (2048 x 256 cells), under a wider capacity: every cell in
    use is written, nothing past them."""
    rng = np.random.default_rng(cells)
    n = 5000
    ic = np.sort(rng.integers(0, cells, n)).astype(np.int32)
    ic[-1] = cells - 1
    want = np.full(cells, n, np.int32)
    first = np.r_[True, ic[1:] != ic[:-1]]
    want[ic[first]] = np.flatnonzero(first)
    ihoc = torch.full((cap,), -7, dtype=torch.int32, device="cuda")
    nc = _dev(np.array([cells, 1, 1, cells], np.int32))
    icd, st = _dev(ic), _dev(np.zeros(1, np.int32))
    _lib.call("aq_linklist_ihoc", _dp(icd), _dp(ihoc), n, _dp(nc), cap,
              _dp(st), _stream())
    got = ihoc.cpu().numpy()
    np.testing.assert_array_equal(got[:cells], want)
    assert (got[cells:] == -7).all()
