"""Sizes past one launch's grid are not refused: the checks of the C entry points, which run before anything is launched."""
from yastn_amd import _lib as L


def test_reflectors_take_any_number_of_columns():
    columns = 16 * 65535
    for n in (columns, columns + 1, 4 * columns):
        L.call('yastn_hip_reflect_trailing', None, L.YH_F64, None, None, 0, 0, n, None)
        L.call('yastn_hip_svd_reflect', None, None, None, L.YH_C128, None, None, None, 0, n, None)
        L.call('yastn_hip_qr_reflect', None, L.YH_F64, None, 0, n, None)
