"""The kernels behind the settings of the decompositions: panel widths other than 16 (YASTN_HIP_PANEL_WIDTH), blocks of more
columns in one workgroup (YASTN_HIP_SVD_LDS_MAX_Q, YASTN_HIP_EIGH_LDS_MAX_Q), fixed slices per panel pair and no QR before
the SVD's iteration, against numpy."""
import numpy as np
import pytest
import torch

from yastn_amd import plans as P

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# at most 150 rotations of a column a sweep and 13 sweeps, each orthogonal to about 4 eps, adding like a random walk:
# 4 eps sqrt(13 * 150) = 4e-14; sums over up to 300 rows add eps sqrt(300) = 4e-15
TOL = 8e-14
SETTINGS = [{'PANEL_WIDTH': 1}, {'PANEL_WIDTH': 5}, {'PANEL_WIDTH': 8}, {'PANEL_WIDTH': 12}, {'PANEL_WIDTH': 24},
            {'PANEL_WIDTH': 32}, {'PANEL_SLICES': 3}, {'PANEL_SLICES': 64}, {'PANEL_WIDTH': 32, 'PANEL_SLICES': 5},
            {'SVD_LDS_MAX_Q': 128, 'EIGH_LDS_MAX_Q': 128}, {'SVD_LDS_MAX_Q': 0, 'EIGH_LDS_MAX_Q': 0},
            {'SVD_LDS_MAX_Q': 20, 'EIGH_LDS_MAX_Q': 48}, {'PRECOND': False}, {'PRECOND': False, 'PANEL_WIDTH': 8}]


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('setting', SETTINGS, ids=str)
def test_decompositions_under_settings(monkeypatch, setting, cplx):
    from yastn_amd import backend_hip as B
    print('settings', setting, cplx, flush=True)
    for name, value in setting.items():
        monkeypatch.setattr(P, name, value)
    monkeypatch.setattr(P, '_CACHE', P._Cache())
    rng = np.random.default_rng(8)

    def normal(*s):
        return rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0)

    shapes = ((3, 3), (24, 24), (40, 33), (47, 90), (150, 150), (300, 65))
    meta, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    blocks = [normal(m, n) * 10.0 ** np.linspace(0, -4, n) for m, n in shapes]
    x = torch.as_tensor(np.concatenate([b.ravel() for b in blocks]), device=DEV)
    U, S, V = (t.cpu().numpy() for t in B.svd(x, tuple(meta), (u, s, v)))
    for blk, (_, _, su, du, ss, sv, dv) in zip(blocks, meta):
        ub, sb, vb = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]], V[sv[0]:sv[1]].reshape(dv)
        assert np.max(np.abs(sb - np.linalg.svd(blk, compute_uv=False))) <= TOL * sb[0]
        assert np.linalg.norm(ub * sb @ vb - blk) <= TOL * np.linalg.norm(blk)
        assert np.max(np.abs(ub.conj().T @ ub - np.eye(len(sb)))) <= TOL
        assert np.max(np.abs(vb @ vb.conj().T - np.eye(len(sb)))) <= TOL

    meta, a, s = [], 0, 0
    blocks = [b + b.conj().T for b in (normal(n, n) for n in (3, 24, 33, 60, 131))]
    for b in blocks:
        n = len(b)
        meta.append(((a, a + n * n), (n, n), (a, a + n * n), (n, n), (s, s + n)))
        a, s = a + n * n, s + n
    x = torch.as_tensor(np.concatenate([b.ravel() for b in blocks]), device=DEV)
    S, U = (t.cpu().numpy() for t in B.eigh(x, tuple(meta), (s, a)))
    for blk, (_, _, su, du, ss) in zip(blocks, meta):
        w, ub = S[ss[0]:ss[1]], U[su[0]:su[1]].reshape(du)
        # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
        tol = TOL * np.sqrt(len(w)) * np.linalg.norm(blk)
        assert np.max(np.abs(w - np.linalg.eigvalsh(blk))) <= tol
        assert np.linalg.norm(ub * w @ ub.conj().T - blk) <= tol
        assert np.max(np.abs(ub.conj().T @ ub - np.eye(len(w)))) <= TOL
