"""Decompositions of more columns or blocks than one launch's grid takes (65535 workgroups along y)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


@pytest.mark.parametrize('cplx', [False, True])
def test_qr_of_a_block_wider_than_the_grid(cplx):
    from yastn_amd import backend_hip as B
    m, n = 3, 16 * 65535 + 3 + 17  # two launches of the reflectors for the columns right of the only panel
    print('wide qr', m, n, cplx, flush=True)
    rng = np.random.default_rng(1)
    a = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0)
    meta = (((0, m * n), (m, n), (0, m * m), (m, m), (0, m * n), (m, n)),)
    Q, R = (t.cpu().numpy() for t in B.qr(torch.as_tensor(a.ravel(), device=DEV), meta, (m * m, m * n)))
    Q, R = Q.reshape(m, m), R.reshape(m, n)
    # three reflectors of length three: a few eps of each column
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(m))) <= 20 * 2.2e-16
    assert np.all(np.linalg.norm(Q @ R - a, axis=0) <= 40 * 2.2e-16 * np.linalg.norm(a, axis=0))
    assert np.max(np.abs(np.tril(R[:, :m], -1))) == 0 and np.all(np.diag(R).real > 0)
