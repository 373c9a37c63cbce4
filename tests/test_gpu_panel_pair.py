"""Panel pairs of the block Jacobi (16-column panels) where their shapes can go wrong: one panel, a lone last column,
odd and even panel counts, ragged last panels, several pairs and slices per round, columns at the ends of the
exponent range (where the rotation takes its long form), real and complex, SVD and eigh."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


def _svd_meta(shapes):
    meta, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    return tuple(meta), (u, s, v), a


# A column takes part in at most q - 1 rotations a sweep and these blocks converge in at most 16 sweeps; a rotation is
# orthogonal to about 4 eps and its errors add like a random walk: 4 eps sqrt(16 * 160) = 5e-14
TOL = 1e-13


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('shapes,scale', [
    (((17, 17),), 1.0), (((32, 32), (31, 40)), 1.0), (((33, 33), (70, 33), (33, 65)), 1.0), (((47, 49), (48, 48)), 1.0),
    (((97, 81), (16, 90), (130, 113), (64, 160)), 1.0), (((50, 40),) * 40, 1.0), (((40, 40),), 1e75), (((40, 40),), 1e-70)])
def test_svd_of_panel_pairs(shapes, scale, cplx):
    from yastn_amd import backend_hip as B
    print('panel pairs', shapes[:4], len(shapes), scale, cplx, flush=True)
    meta, sizes, n = _svd_meta(shapes)
    rng = np.random.default_rng(len(shapes))
    x = rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0)
    for sl, D, *_ in meta[1:]:  # decaying columns in all but the first block
        x[sl[0]:sl[1]] = (x[sl[0]:sl[1]].reshape(D) * 10.0 ** (-8 * np.arange(D[1]) / D[1])).ravel()
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(x * scale, device=DEV), meta, sizes))
    for sl, D, su, du, ss, sv, dv in meta:
        a = x[sl[0]:sl[1]].reshape(D)
        u, s, v = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]] / scale, V[sv[0]:sv[1]].reshape(dv)
        ref = np.linalg.svd(a, compute_uv=False)
        assert np.max(np.abs(s - ref)) <= TOL * ref[0]
        assert np.linalg.norm(u * s @ v - a) <= TOL * np.linalg.norm(a)
        assert np.max(np.abs(u.conj().T @ u - np.eye(len(s)))) <= TOL
        assert np.max(np.abs(v @ v.conj().T - np.eye(len(s)))) <= TOL


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('n', [97, 128, 145])
def test_eigh_of_panel_pairs(n, cplx):
    from yastn_amd import backend_hip as B
    print('panel pairs, eigh', n, cplx, flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0)
    a = x + x.conj().T
    meta = (((0, n * n), (n, n), (0, n * n), (n, n), (0, n)),)
    S, U = (t.cpu().numpy() for t in B.eigh(torch.as_tensor(a.ravel(), device=DEV), meta, (n, n * n)))
    U = U.reshape(n, n)
    norm = np.linalg.norm(a)
    # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
    assert np.max(np.abs(S - np.linalg.eigvalsh(a))) <= TOL * norm
    assert np.linalg.norm(U * S @ U.conj().T - a) <= 10 * TOL * norm
    assert np.max(np.abs(U.conj().T @ U - np.eye(n))) <= TOL
