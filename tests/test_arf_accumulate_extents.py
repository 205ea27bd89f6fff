"""Projections without pairs, into no pixels, or into more pixels than the binned sums index: they
take the direct kernel, or nothing, and are not refused."""
import ctypes as C

import pytest
import torch


@pytest.mark.parametrize("m,n_pix", [(10**6, 0), (0, 0), (10**6, 2**31 - 1), (10**6, 2**31), (10**6, 2**40), (0, 2**31)])
def test_the_direct_kernel_is_named(m, n_pix):
    from opengate_amd import _abi as A

    need = C.c_int64(-1)
    assert A.load_library().gh_arf_accumulate_workspace(m, 3, n_pix, 1, C.byref(need)) == 0
    assert need.value == 0


@pytest.mark.parametrize("windows", [3, 9])
@pytest.mark.parametrize("shape", [(0, 4, 4), (6, 4, 4), (2, 1, 1)])
def test_no_pairs(windows, shape):
    from opengate_amd.learn.arf import ArfModel

    arf = ArfModel(device="cpu", sizes=[3, 128, 128, windows + 1], windows=[(0.1, 0.2)] * windows)
    img = torch.zeros(shape, dtype=torch.float64)
    arf.project(None, 0, img)
    assert not img.any()
