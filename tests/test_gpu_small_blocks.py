"""Blocks of at most 32 columns (one workgroup each): the smallest sizes, both slot counts (16 and 32 columns) and their
edges, tall blocks up to the LDS limit, wide, rank-deficient and zero blocks, many at once, real and complex."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# at most 31 rotations of a column a sweep and 12 sweeps, each orthogonal to about 4 eps, adding like a random walk:
# 4 eps sqrt(12 * 31) = 1.7e-14; the sums over up to 900 rows add eps sqrt(900) = 7e-15
TOL = 5e-14


def _svd_meta(shapes):
    meta, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    return tuple(meta), (u, s, v), a


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('shapes', [
    ((1, 1), (1, 7), (5, 1), (2, 2), (3, 2)), ((15, 15), (16, 16), (16, 40), (200, 16)), ((17, 17), (31, 33), (32, 32)),
    ((32, 20), (17, 64), (130, 32), (32, 129)), ((900, 12), (9, 800), (33, 33)), ((24, 24),) * 60])
def test_svd_of_small_blocks(shapes, cplx):
    from yastn_amd import backend_hip as B
    print('small blocks', shapes[:5], len(shapes), cplx, flush=True)
    meta, sizes, n = _svd_meta(shapes)
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0)
    sl, D = meta[-1][:2]  # the last block: columns over nine decades
    x[sl[0]:sl[1]] = (x[sl[0]:sl[1]].reshape(D) * 10.0 ** (-9 * np.arange(D[1]) / D[1])).ravel()
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(x, device=DEV), meta, sizes))
    for sl, D, su, du, ss, sv, dv in meta:
        a = x[sl[0]:sl[1]].reshape(D)
        u, s, v = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]], V[sv[0]:sv[1]].reshape(dv)
        ref = np.linalg.svd(a, compute_uv=False)
        assert np.max(np.abs(s - ref)) <= TOL * ref[0]
        assert np.linalg.norm(u * s @ v - a) <= TOL * np.linalg.norm(a)
        assert np.max(np.abs(u.conj().T @ u - np.eye(len(s)))) <= TOL
        assert np.max(np.abs(v @ v.conj().T - np.eye(len(s)))) <= TOL


@pytest.mark.parametrize('m,n', [(20, 20), (40, 30), (12, 50)])
def test_svd_of_small_deficient_blocks(m, n):
    """Rank 3 and zero blocks: exact factors with orthonormal completions."""
    from yastn_amd import backend_hip as B
    print('small deficient blocks', m, n, flush=True)
    meta, sizes, size = _svd_meta(((m, n), (m, n)))
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, 3)) @ rng.standard_normal((3, n))
    x = np.concatenate([a.ravel(), np.zeros(m * n)])
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(x, device=DEV), meta, sizes))
    for (sl, D, su, du, ss, sv, dv), ref in zip(meta, (a, 0 * a)):
        u, s, v = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]], V[sv[0]:sv[1]].reshape(dv)
        scale = max(np.linalg.norm(ref), 1.0)
        assert np.linalg.norm(u * s @ v - ref) <= TOL * scale
        assert np.max(np.abs(u.T @ u - np.eye(len(s)))) <= TOL
        assert np.max(np.abs(v @ v.T - np.eye(len(s)))) <= TOL


@pytest.mark.parametrize('cplx', [False, True])
def test_eigh_of_small_blocks(cplx):
    from yastn_amd import backend_hip as B
    print('small blocks, eigh', cplx, flush=True)
    rng = np.random.default_rng(5)
    dims, meta, data, a_off, s_off = (1, 2, 3, 15, 16, 17, 31, 32, 33, 24, 24), [], [], 0, 0
    for n in dims:
        x = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0)
        data.append(x + x.conj().T)
        meta.append(((a_off, a_off + n * n), (n, n), (a_off, a_off + n * n), (n, n), (s_off, s_off + n)))
        a_off, s_off = a_off + n * n, s_off + n
    S, U = (t.cpu().numpy() for t in B.eigh(torch.as_tensor(np.concatenate([a.ravel() for a in data]), device=DEV),
                                            tuple(meta), (s_off, a_off)))
    for a, (sl, D, su, du, ss) in zip(data, meta):
        w, u = S[ss[0]:ss[1]], U[su[0]:su[1]].reshape(du)
        norm = np.linalg.norm(a)
        # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
        assert np.max(np.abs(w - np.linalg.eigvalsh(a))) <= 6 * TOL * norm
        assert np.linalg.norm(u * w @ u.conj().T - a) <= 6 * TOL * norm
        assert np.max(np.abs(u.conj().T @ u - np.eye(len(w)))) <= TOL
