"""Sizes past one launch's grid are not refused: the checks of the C entry points, which run before anything is launched."""
import ctypes

import pytest

from yastn_amd import _lib as L


def test_reflectors_take_any_number_of_columns():
    columns = 16 * 65535
    for n in (columns, columns + 1, 4 * columns):
        L.call('yastn_hip_reflect_trailing', None, L.YH_F64, None, None, 0, 0, n, None)
        L.call('yastn_hip_svd_reflect', None, None, None, L.YH_C128, None, None, None, 0, n, None)
        L.call('yastn_hip_qr_reflect', None, L.YH_F64, None, 0, n, None)


def test_rounds_take_any_number_of_jobs():
    """A sweep of 70000 jobs in a round with a buffer for none of them: refused for the buffer, not for the round."""
    rounds = (ctypes.c_int64 * 2)(0, 70000)
    state = (ctypes.c_int32 * 64)()
    with pytest.raises(L.HipBackendError, match='Gram buffer'):
        L.call('yastn_hip_svd_panel_sweep', None, None, L.YH_F64, None, None, ctypes.addressof(rounds), 1, 16, 1, 1, None, 0,
               0, 60, ctypes.addressof(state), 64, None)
