"""Householder panels in registers: rows at the edges of the instances (64 rows per register slot, passes of 32, 16 and 8
columns) and past the tallest one, where the panel is factored in place; last panels of one to 32 columns, dependent
and zero columns, entries near the ends of the exponent range, a NaN, real and complex."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# at most 96 reflectors, each orthogonal to about 4 eps, adding like a random walk: 4 eps sqrt(96) = 9e-15; sums over up
# to 3100 rows add eps sqrt(3100) = 1.2e-14
TOL = 5e-14


def _run(blocks, cplx):
    from yastn_amd import backend_hip as B
    meta, a, q, r = [], 0, 0, 0
    for x in blocks:
        m, n = x.shape
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (q, q + m * k), (m, k), (r, r + k * n), (k, n)))
        a, q, r = a + m * n, q + m * k, r + k * n
    x = np.concatenate([b.ravel() for b in blocks])
    Q, R = (t.cpu().numpy() for t in B.qr(torch.as_tensor(x, device=DEV), tuple(meta), (q, r)))
    return [(Q[sq[0]:sq[1]].reshape(dq), R[sr[0]:sr[1]].reshape(dr)) for _, _, sq, dq, sr, dr in meta]


def _normal(rng, cplx, *s):
    return rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0)


def _check(blk, qb, rb):
    scale = np.max(np.abs(blk)) or 1.0  # norms of scaled blocks, so that their squares stay in range
    assert np.linalg.norm(qb @ (rb / scale) - blk / scale) <= TOL * np.linalg.norm(blk / scale)
    assert np.max(np.abs(qb.conj().T @ qb - np.eye(qb.shape[1]))) <= TOL
    assert np.all(np.tril(rb, -1) == 0) and np.all(np.diagonal(rb).real >= 0)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('rows', [(33, 64, 65, 128, 129), (256, 257, 448, 449), (576, 577, 768, 769), (960, 961, 1152, 1153),
                                  (1472, 1473, 1920, 1921), (2944, 2945, 3100)])
def test_panel_heights(rows, cplx):
    rng = np.random.default_rng(rows[0])
    for group in (rows[:1], rows):  # one block, and blocks of several instances in one launch
        blocks = [_normal(rng, cplx, m, n) for m, n in zip(group, (33, 8, 9, 64, 41))]
        print('qr panels', [b.shape for b in blocks], cplx, flush=True)
        for blk, (qb, rb) in zip(blocks, _run(blocks, cplx)):
            _check(blk, qb, rb)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('m', [40, 300, 1100])
def test_special_columns(m, cplx):
    rng = np.random.default_rng(m)
    dep = _normal(rng, cplx, m, 40)
    dep[:, 5] = 0
    dep[:, 20:] = dep[:, :20] @ _normal(rng, cplx, 20, 20)
    tri = np.triu(_normal(rng, cplx, m, 34))  # zero tails: reflectors that are the identity
    for e in (-150, 150):  # squares near the ends of the exponent range
        blocks = [dep, np.zeros((m, 33), dep.dtype), tri, _normal(rng, cplx, m, 36) * 10.0 ** e]
        for blk, (qb, rb) in zip(blocks, _run(blocks, cplx)):
            _check(blk, qb, rb)


@pytest.mark.parametrize('m', [40, 300, 1100])
def test_nan_stays_behind_its_column(m):
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, 36))
    good = _run([x], False)[0][1]
    x[m // 2, 20] = np.nan
    (_, rb), (q2, r2) = _run([x, np.eye(5)], False)
    np.testing.assert_allclose(rb[:, :20], good[:, :20], rtol=0, atol=1e-12)
    assert np.isnan(rb[20, 20]) and np.array_equal(q2 @ r2, np.eye(5))
