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


def test_eigh_of_more_panels_than_the_grid():
    from yastn_amd import backend_hip as B
    nb, n = 21846, 33  # three panels each: 65538 in the round of every panel against itself
    print('many eigh blocks', nb, n, flush=True)
    a = torch.from_numpy(np.random.default_rng(2).standard_normal((nb, n, n))).to(DEV)
    a = a + a.transpose(1, 2)
    meta = tuple(((i * n * n, (i + 1) * n * n), (n, n), (i * n * n, (i + 1) * n * n), (n, n), (i * n, (i + 1) * n))
                 for i in range(nb))
    S, U = B.eigh(a.reshape(-1).contiguous(), meta, (nb * n, nb * n * n))
    S, U = S.reshape(nb, 1, n), U.reshape(nb, n, n)
    # about 32 rotations of a column a sweep and 10 sweeps, each orthogonal to about 4 eps: 4 eps sqrt(320) = 1.6e-14; the
    # iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
    norm = torch.linalg.vector_norm(a, dim=(1, 2))
    assert bool(((U.transpose(1, 2).contiguous() @ U - torch.eye(n, device=DEV, dtype=a.dtype)).abs() <= 5e-14).all())
    assert bool((torch.linalg.vector_norm(a @ U - U * S, dim=(1, 2)) <= 3e-13 * norm).all())
    ref = np.linalg.eigvalsh(a[-1].cpu().numpy())
    assert np.max(np.abs(S[-1, 0].cpu().numpy() - ref)) <= 3e-13 * float(norm[-1])
