"""Orthogonality of the singular vectors of large blocks, where most products of a sine and a cosine can be left over by a
last sweep that no other one verifies: random, graded and nearly repeated spectra, real and complex."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
EPS = 2.2e-16


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('kind', ['random', 'graded', 'near'])
@pytest.mark.parametrize('m,n', [(500, 500), (900, 640), (1100, 1100)])
def test_vectors_of_large_blocks(m, n, kind, cplx):
    from yastn_amd import backend_hip as B
    print('orthogonality', m, n, kind, cplx, flush=True)
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, n)) + (1j * rng.standard_normal((m, n)) if cplx else 0)
    if kind == 'graded':  # rows and columns over eight decades
        x = x * 10.0 ** np.linspace(0, -8, m)[:, None] * 10.0 ** np.linspace(0, -8, n)
    elif kind == 'near':  # the singular values of a perturbed isometry: close to each other, none equal
        q = np.linalg.qr(x)[0]
        x = q + 1e-6 * x / np.sqrt(m)
    meta = (((0, m * n), (m, n), (0, m * n), (m, n), (0, n), (0, n * n), (n, n)),)
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(x.ravel(), device=DEV), meta, (m * n, n, n * n)))
    U, V = U.reshape(m, n), V.reshape(n, n)
    # cosines of the iteration's columns: the tolerance eps sqrt(n) twice; vectors: at most n rotations a sweep and 20 sweeps,
    # each orthogonal to about 4 eps, adding like a random walk
    tol = 2 * EPS * np.sqrt(n) + 4 * EPS * np.sqrt(20 * n)
    assert np.max(np.abs(U.conj().T @ U - np.eye(n))) <= tol
    assert np.max(np.abs(V @ V.conj().T - np.eye(n))) <= tol
    assert np.linalg.norm(U * S @ V - x) <= tol * np.linalg.norm(x)
