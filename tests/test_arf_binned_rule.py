"""Which projections take the binned sums: only those that measured faster than one atomic per pair,
window and image (microseconds direct / binned in the comments)."""
import ctypes as C

import pytest


@pytest.mark.parametrize("m,n_win,heads,plane,squared,binned", [
    (10**6, 3, 1, 4096, True, False),     # 253 / 688: one bin
    (10**6, 1, 1, 4096, True, False),     # 88 / 677
    (10**6, 3, 1, 4096, False, False),    # 133 / 668
    (3 * 10**5, 3, 1, 4096, True, False),  # 80 / 231
    (10**6, 3, 1, 16384, True, True),     # 263 / 202: four bins
    (10**6, 1, 1, 16384, True, False),    # 91 / 192
    (10**6, 3, 1, 16384, False, False),   # 141 / 197
    (10**6, 1, 2, 16384, True, False),    # 92 / 111
    (10**6, 3, 2, 16384, True, True),     # 266 / 120
    (3 * 10**5, 3, 16, 16384, True, True),  # 84 / 46
    (10**5, 3, 16, 16384, True, False),   # 29 / 41
    (10**6, 3, 128, 16384, True, True),   # 268 / 112
    (0, 3, 1, 4096, True, False)])
def test_rule(m, n_win, heads, plane, squared, binned):
    from opengate_amd import _abi as A

    need = C.c_int64(-1)
    assert A.load_library().gh_arf_accumulate_workspace(m, n_win, heads * plane, int(squared), C.byref(need)) == 0
    assert (need.value > 0) == binned
