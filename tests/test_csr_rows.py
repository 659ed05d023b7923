"""The bound on even rows that the default SpMM launch order goes by (host side, no GPU)."""

import numpy as np
import pytest

import cacg_amd
from cacg_amd import problems as P


def bound(lens):
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    return cacg_amd.lib().cacg_csr_even_bound(len(lens), rp.ctypes.data)


@pytest.mark.parametrize("A,longest", [(P.laplacian_2d(16), 5), (P.laplacian_3d(8), 7)])
def test_stencil_rows_are_even(A, longest):
    assert bound(np.diff(A.rowptr)) == longest + 1


@pytest.mark.parametrize("lens,want", [([1] * 9, 2), ([0] * 9, 1), ([27] * 50 + [8], 28), ([600] * 9, 601),
                                       ([], 0)])
def test_even_lengths(lens, want):
    assert bound(np.array(lens, dtype=np.int64)) == want


@pytest.mark.parametrize("lens", [[5] * 63 + [200], [1, 9] * 40, [3] * 60 + [16] * 20, [5] * 999 + [300]])
def test_uneven_lengths_have_none(lens):
    """The default order must not count on even rows there, long rows or not."""
    assert bound(np.array(lens)) == 0
