"""The triangular solve of the QR adjoint on both sides of the column count up to which its rows fit the LDS beside the
kernel's own arrays (480 complex, 1008 real), against the formula in numpy as for the other sizes."""
import pytest

from test_gpu_qr_adjoint_sizes import test_qr_adjoint_blocks as check_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('k', [479, 480, 481, 496, 497, 512])
def test_complex_rows_at_the_lds_limit(k):
    check_blocks(((k + 20, k), (33, 17)), True)


@pytest.mark.parametrize('k', [1008, 1009, 1024, 1025])
def test_real_rows_at_the_lds_limit(k):
    check_blocks(((k + 20, k),), False)
