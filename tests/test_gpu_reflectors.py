"""Block reflectors of the batched QR and of the preconditioned SVD, 16 columns per workgroup: widths at the edges of
slabs (16) and panels (32), a single row or column, tall and wide blocks, blocks of unequal numbers of panels together,
panels in and out of LDS, real and complex."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'
# at most 450 reflectors, each orthogonal to about 4 eps, adding like a random walk: 4 eps sqrt(450) = 1.9e-14; sums over
# up to 1400 rows add eps sqrt(1400) = 8e-15
TOL = 5e-14


def _data(shapes, cplx):
    n = sum(a * b for a, b in shapes)
    rng = np.random.default_rng(n)
    return rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('shapes', [
    ((1, 1), (1, 9), (9, 1), (2, 3)), ((31, 31), (32, 32), (33, 33), (32, 64)), ((47, 49), (48, 48), (49, 47), (64, 65)),
    ((31, 200), (200, 31), (33, 400), (97, 97)), ((1400, 40), (3, 3), (450, 450))])
def test_qr_reflectors(shapes, cplx):
    from yastn_amd import backend_hip as B
    print('qr', shapes, cplx, flush=True)
    meta, a, q, r = [], 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (q, q + m * k), (m, k), (r, r + k * n), (k, n)))
        a, q, r = a + m * n, q + m * k, r + k * n
    x = _data(shapes, cplx)
    Q, R = (t.cpu().numpy() for t in B.qr(torch.as_tensor(x, device=DEV), tuple(meta), (q, r)))
    for sl, D, sq, dq, sr, dr in meta:
        blk, qb, rb = x[sl[0]:sl[1]].reshape(D), Q[sq[0]:sq[1]].reshape(dq), R[sr[0]:sr[1]].reshape(dr)
        assert np.linalg.norm(qb @ rb - blk) <= TOL * np.linalg.norm(blk)
        assert np.max(np.abs(qb.conj().T @ qb - np.eye(dq[1]))) <= TOL
        assert np.all(np.tril(rb, -1) == 0) and np.all(np.diagonal(rb).real >= 0)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('shapes', [
    ((33, 33), (33, 34), (90, 47)), ((48, 48), (49, 130), (64, 64)), ((700, 34), (34, 700), (65, 65)),
    ((1400, 40), (40, 1400), (129, 97))])
def test_svd_reflectors(shapes, cplx):
    """The reflector launches against the same products as grouped GEMMs, the factors before and after them the same."""
    from yastn_amd import _functions as F, _lib as L, plans as P
    print('svd', shapes, cplx, flush=True)
    blocks, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        blocks.append((a, m, n, u, s, v))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    x = torch.as_tensor(_data(shapes, cplx), device=DEV)
    plan = P.SvdPlan(blocks, x.element_size(), 0, a, u, s, v, x.device)
    assert plan.n_pre == len(shapes)
    dt, st = F.dtype_code(x), F.stream_of(x)
    work = torch.zeros(plan.work_numel, dtype=x.dtype, device=DEV)
    floors = torch.zeros(plan.nblocks, dtype=torch.float64, device=DEV)
    L.call('yastn_hip_svd_precond_load', x.data_ptr(), work.data_ptr(), floors.data_ptr(), dt, plan.d_blocks.data_ptr(),
           plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(), plan.n_pre, st)
    for step, (d_ids, n, rest) in enumerate(plan.panel_steps):
        L.call('yastn_hip_svd_qr_panel', work.data_ptr(), dt, plan.d_qdesc.data_ptr(), d_ids.data_ptr(), n, step,
               plan.qr_rows, st)
        trail = plan.qr_steps[step][2]
        assert (trail is not None) == (rest > 0)
        if trail is None:
            continue
        ref = work.clone()
        for gp in trail:
            F.run_gemm(gp, (ref,), (ref,), dt, tune=False)
        L.call('yastn_hip_reflect_trailing', work.data_ptr(), dt, plan.d_qdesc.data_ptr(), d_ids.data_ptr(), n, step, rest,
               st)
        for p, q, w_off, *_ in plan.h_qdesc.tolist():
            assert (work[w_off:w_off + p * q] - ref[w_off:w_off + p * q]).abs().max() <= TOL * ref.abs().max()
    torch.manual_seed(7)
    U, Vh = (torch.randn(size, dtype=x.dtype, device=DEV) for size in (u, v))
    Ur, Vr, wr = U.clone(), Vh.clone(), work.clone()
    for h1, h2, h3 in plan.q_apply:
        F.run_gemm(h1, (wr,), (wr, Ur, Vr), dt, tune=False)
        F.run_gemm(h2, (wr,), (wr,), dt, tune=False)
        F.run_gemm(h3, (wr, Ur, Vr), (wr,), dt, tune=False)
    L.call('yastn_hip_svd_reflect', U.data_ptr(), Vh.data_ptr(), work.data_ptr(), dt, plan.d_blocks.data_ptr(),
           plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(), plan.n_pre, plan.qr_cols, st)
    assert (U - Ur).abs().max() <= TOL * Ur.abs().max()
    assert (Vh - Vr).abs().max() <= TOL * Vr.abs().max()
