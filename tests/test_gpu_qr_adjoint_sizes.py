"""The triangular solve and the core of the QR adjoint at the edges of their 16 x 16 blocks, with rows that fit the LDS and rows
that do not (more than 1000 real, 500 complex columns), against the formula in numpy: gA = (gQ + Q C) R^-H."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('dims', [((1, 1), (2, 2), (15, 15), (16, 16), (17, 17)), ((31, 31), (33, 32), (50, 33), (65, 65)),
                                  ((200, 97), (129, 128)), ((1030, 1030),)])
def test_qr_adjoint_blocks(dims, cplx):
    from yastn_amd import backend_hip as B
    print('qr adjoint', dims, cplx, flush=True)
    rng = np.random.default_rng(len(dims))
    normal = lambda *s: rng.standard_normal(s) + (1j * rng.standard_normal(s) if cplx else 0)
    meta, blocks, ao, qo, ro = [], [], 0, 0, 0
    for m, n in dims:
        # a well-conditioned block, so that the error of the solve is that of its arithmetic
        blocks.append(normal(m, n) / np.sqrt(m + n) + 3 * np.eye(m, n))
        meta.append(((ao, ao + m * n), (m, n), (qo, qo + m * n), (m, n), (ro, ro + n * n), (n, n)))
        ao, qo, ro = ao + m * n, qo + m * n, ro + n * n
    x = torch.as_tensor(np.concatenate([b.ravel() for b in blocks]), device=DEV).requires_grad_(True)
    gq, gr = normal(qo), normal(ro)
    Q, R = B.qr(x, tuple(meta), (qo, ro))
    torch.autograd.backward([Q, R], [torch.as_tensor(gq, device=DEV), torch.as_tensor(gr, device=DEV)])
    got, Q, R = x.grad.cpu().numpy(), Q.detach().cpu().numpy(), R.detach().cpu().numpy()
    for (sa, D, sq, _, sr, _), a in zip(meta, blocks):
        m, n = D
        q, r = Q[sq[0]:sq[1]].reshape(m, n), R[sr[0]:sr[1]].reshape(n, n)
        dq, dr = gq[sq[0]:sq[1]].reshape(m, n), gr[sr[0]:sr[1]].reshape(n, n)
        M = r @ dr.conj().T - dq.conj().T @ q
        C = np.tril(M, -1) + np.tril(M, -1).conj().T + np.diag(np.diag(M).real)
        ref = np.linalg.solve(r, (dq + q @ C).conj().T).conj().T
        # products of length n and a substitution of a triangle of condition about 4: eps sqrt(n) each, a few of them
        err = np.linalg.norm(got[sa[0]:sa[1]].reshape(m, n) - ref) / np.linalg.norm(ref)
        assert err <= 40 * 2.2e-16 * np.sqrt(n + 1), (D, err)
