"""QR of columns of very different size: the last column of a real square block has no reflector of its own, so its squares
need not be representable, and products of it with the other columns may leave the exponent range where the result does not."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


@pytest.mark.parametrize('n', [2, 20, 33, 64, 70, 200, 330, 600])
def test_last_column_of_another_scale(n):
    from yastn_amd import backend_hip as B
    print('qr scaled columns', n, flush=True)
    a = np.random.default_rng(n).standard_normal((n, n)) + 3 * np.sqrt(n) * np.eye(n)
    meta = (((0, n * n), (n, n), (0, n * n), (n, n), (0, n * n), (n, n)),)
    q0, r0 = np.linalg.qr(a)
    sign = np.sign(np.diag(r0))
    q0, r0 = q0 * sign, sign[:, None] * r0
    for scale, last in ((1.0, 1.0), (1e100, 1e250)):
        d = np.full(n, scale)
        d[-1] = last
        Q, R = (t.cpu().numpy().reshape(n, n)
                for t in B.qr(torch.as_tensor((a * d).ravel(), device=DEV), meta, (n * n, n * n)))
        # n reflectors, each orthogonal to a few eps, in a block whose condition is below 10
        assert np.max(np.abs(Q - q0)) <= 40 * 2.2e-16 * n
        assert np.linalg.norm(R / d - r0) <= 40 * 2.2e-16 * n * np.linalg.norm(r0)
