"""Which kernel decomposes the blocks of one workgroup each: lists on both sides of the rule's lines, with the kernel that
each is meant to take, against numpy."""
import numpy as np
import pytest
import torch

from yastn_amd import plans as P

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# at most 35 rotations of a column a sweep and 12 sweeps, each orthogonal to about 4 eps, adding like a random walk:
# 4 eps sqrt(12 * 35) = 1.8e-14; the sums over up to 2000 rows add eps sqrt(2000) = 1e-14
TOL = 5e-14


def _blocks(shapes, cplx, rng):
    return [rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0) for s in shapes]


@pytest.mark.parametrize('shapes, cplx, waves16', [
    (((4, 4),) * 700 + ((600, 3),), False, True), (((4, 4),) * 700 + ((5, 5),), False, False),
    (((9, 9),) * 256, False, True), (((9, 9),) * 257, True, False), (((9, 30), (30, 9), (2, 2)), True, True),
    (((10, 10), (9, 9)), False, False), (((320, 10), (10, 320), (9, 9)), False, True), (((319, 10),), False, False),
    (((320, 10),), True, False), (((448, 14), (480, 15)), False, False), (((448, 14),), False, True),
    (((2000, 8), (8, 1999)), False, True), (((2000, 8),), True, True)])
def test_svd_lists(shapes, cplx, waves16):
    from yastn_amd import backend_hip as B
    print('one workgroup, svd', shapes[:3], len(shapes), cplx, flush=True)
    meta, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    meta = tuple(meta)
    blocks = _blocks(shapes, cplx, np.random.default_rng(a))
    x = torch.as_tensor(np.concatenate([b.ravel() for b in blocks]), device=DEV)
    plan = P.svd_plan(meta, x.element_size(), a, (u, s, v), x.device)
    fits = sum((max(d) + min(d)) * min(d) * x.element_size() <= 131072 for d in shapes)
    assert (plan.n_small, plan.n_lds) == ((0, fits) if waves16 else (fits, 0))
    U, S, V = (t.cpu().numpy() for t in B.svd(x, meta, (u, s, v)))
    for blk, (_, _, su, du, ss, sv, dv) in zip(blocks, meta):
        ub, sb, vb = U[su[0]:su[1]].reshape(du), S[ss[0]:ss[1]], V[sv[0]:sv[1]].reshape(dv)
        assert np.max(np.abs(sb - np.linalg.svd(blk, compute_uv=False))) <= TOL * sb[0]
        assert np.linalg.norm(ub * sb @ vb - blk) <= TOL * np.linalg.norm(blk)
        assert np.max(np.abs(ub.conj().T @ ub - np.eye(len(sb)))) <= TOL
        assert np.max(np.abs(vb @ vb.conj().T - np.eye(len(sb)))) <= TOL


@pytest.mark.parametrize('dims, cplx, counts', [
    ((9, 4, 1), False, (0, 3, 0)), ((10, 4), True, (2, 0, 0)), ((33, 5, 20), False, (0, 3, 0)), ((33, 5, 20), True, (0, 3, 0)),
    ((36,) * 256, False, (0, 256, 0)), ((36,) * 257, False, (0, 0, 257)), ((33,) * 1024, True, (0, 1024, 0)),
    ((33,) * 1024 + (8,), True, (0, 1, 1024)), ((37, 33, 8), False, (0, 1, 2)), ((64, 12), True, (1, 0, 1))])
def test_eigh_lists(dims, cplx, counts):
    from yastn_amd import backend_hip as B
    print('one workgroup, eigh', dims[:3], len(dims), cplx, flush=True)
    meta, a, s = [], 0, 0
    for n in dims:
        meta.append(((a, a + n * n), (n, n), (a, a + n * n), (n, n), (s, s + n)))
        a, s = a + n * n, s + n
    meta = tuple(meta)
    blocks = [b + b.conj().T for b in _blocks([(n, n) for n in dims], cplx, np.random.default_rng(a))]
    x = torch.as_tensor(np.concatenate([b.ravel() for b in blocks]), device=DEV)
    plan = P.eigh_plan(meta, x.element_size(), a, (s, a), x.device)
    assert (plan.n_small, plan.n_lds, plan.n_big) == counts
    S, U = (t.cpu().numpy() for t in B.eigh(x, meta, (s, a)))
    for blk, (_, _, su, du, ss) in zip(blocks, meta):
        w, ub = S[ss[0]:ss[1]], U[su[0]:su[1]].reshape(du)
        # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
        tol = TOL * np.sqrt(len(w)) * np.linalg.norm(blk)
        assert np.max(np.abs(w - np.linalg.eigvalsh(blk))) <= tol
        assert np.linalg.norm(ub * w @ ub.conj().T - blk) <= tol
        assert np.max(np.abs(ub.conj().T @ ub - np.eye(len(w)))) <= 2 * TOL


def test_a_lower_cap_is_kept(monkeypatch):
    from yastn_amd import backend_hip as B
    n = 20
    monkeypatch.setattr(P, 'EIGH_LDS_MAX_Q', 16)
    monkeypatch.setattr(P, '_CACHE', P._Cache())
    a = _blocks([(n, n)], False, np.random.default_rng(n))[0]
    a = a + a.T
    meta = (((0, n * n), (n, n), (0, n * n), (n, n), (0, n)),)
    x = torch.as_tensor(a.ravel(), device=DEV)
    plan = P.eigh_plan(meta, 8, n * n, (n, n * n), x.device)
    assert (plan.n_small, plan.n_lds, plan.n_big) == (0, 0, 1)
    S, _ = B.eigh(x, meta, (n, n * n))
    assert np.max(np.abs(S.cpu().numpy() - np.linalg.eigvalsh(a))) <= TOL * np.sqrt(n) * np.linalg.norm(a)
