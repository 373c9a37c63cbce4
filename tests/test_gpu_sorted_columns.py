"""SVDs whose columns (or, for wide blocks, rows) are reordered by norm before the preconditioning QR: ascending, equal,
zero and repeated columns, tall and wide blocks, one column more than a one-workgroup block takes, clustered and equal
singular values (where the last sweep may not be left out), real and complex."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# a column takes part in at most q - 1 rotations a sweep and 20 sweeps, each orthogonal to about 4 eps, adding like a
# random walk: 4 eps sqrt(20 * 300) = 7e-14; the sums over up to 2500 rows add eps sqrt(2500) = 1.1e-14
TOL = 1e-13


def _block(kind, m, n, cplx, rng):
    def normal(*s):
        return rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0)
    k = min(m, n)
    if kind == 'ascending':
        x = normal(m, n)
        return x * 10.0 ** np.linspace(-8, 0, n) * (10.0 ** np.linspace(-8, 0, m))[:, None]
    if kind == 'equal':  # orthogonal columns of one norm (rows for a wide block)
        x = np.linalg.qr(normal(max(m, n), k))[0]
        return x if m >= n else x.conj().T
    if kind == 'zero':  # every third column and row zero, two columns alike
        x = normal(m, n)
        x[:, ::3] = 0
        x[::3] = 0
        x[:, -1] = x[:, 1]
        return x
    w = {'cluster': 10.0 ** (-(np.arange(k) // 8)) * (1 + 1e-10 * np.arange(k)), 'repeated': 10.0 ** (-(np.arange(k) // 8) / 2)}
    u, v = np.linalg.qr(normal(m, k))[0], np.linalg.qr(normal(n, k))[0]
    return u * w[kind] @ v.conj().T


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('kind', ['ascending', 'equal', 'zero', 'cluster', 'repeated'])
@pytest.mark.parametrize('shapes', [((33, 33), (34, 40)), ((300, 50), (50, 300), (129, 130)), ((2500, 35), (35, 2500))])
def test_svd_of_sorted_columns(shapes, kind, cplx):
    from yastn_amd import backend_hip as B
    print('sorted columns', shapes, kind, cplx, flush=True)
    rng = np.random.default_rng(len(kind))
    meta, a, u, s, v, blocks = [], 0, 0, 0, 0, []
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
        blocks.append(_block(kind, m, n, cplx, rng))
    x = np.concatenate([b.ravel() for b in blocks])
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(x, device=DEV), tuple(meta), (u, s, v)))
    for blk, (_, _, su, du, ss, sv, dv) in zip(blocks, meta):
        ub, sb, vb = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]], V[sv[0]:sv[1]].reshape(dv)
        ref = np.linalg.svd(blk, compute_uv=False)
        assert np.all(np.diff(sb) <= 0)
        assert np.max(np.abs(sb - ref)) <= TOL * ref[0]
        assert np.linalg.norm(ub * sb @ vb - blk) <= TOL * np.linalg.norm(blk)
        assert np.max(np.abs(ub.conj().T @ ub - np.eye(len(sb)))) <= TOL
        assert np.max(np.abs(vb @ vb.conj().T - np.eye(len(sb)))) <= TOL
