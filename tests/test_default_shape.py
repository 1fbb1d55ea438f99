"""The default shape of a matrix struct that no call has filled (CPU only): the
lean path of the named kernel's lanes rule, as nothing is known of its rows."""
from __future__ import annotations

import pytest

from sptrsv_amd import _lib as L
from sptrsv_amd import interface as I


@pytest.mark.parametrize("k,variant", [(1, 1), (4, 0)])
def test_default_shape_of_a_bare_struct(k, variant):
    mat = L.SpMat()
    mat.nr = mat.nc = 1000
    mat.nnz = 9000
    cfg = I.default_config(mat, None, I.PREC_F64, k)
    assert (cfg.kernel, cfg.variant) == (I.KERNEL_SIMPLE, variant)
