"""Inputs with a NaN or an infinity in blocks of every path of the decompositions (one workgroup, panels, panels after a
QR; tall and wide): refused as in the small case, with the device in order afterwards."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


def _svd_meta(m, n):
    k = min(m, n)
    return (((0, m * n), (m, n), (0, m * k), (m, k), (0, k), (0, k * n), (k, n)),), (m * k, k, k * n)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('m,n', [(24, 24), (50, 24), (24, 50), (40, 40), (90, 40), (40, 90), (130, 130), (300, 130),
                                 (130, 300)])
def test_svd_refuses_nonfinite_blocks(m, n, cplx):
    from yastn_amd import backend_hip as B
    print('nonfinite svd', m, n, cplx, flush=True)
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal(m * n) + (1j * rng.standard_normal(m * n) if cplx else 0)
    meta, sizes = _svd_meta(m, n)
    for bad in (np.nan, np.inf, -np.inf):
        for at in (0, m * n // 2, m * n - 1):
            x = a.copy()
            x[at] = bad
            with pytest.raises(ValueError, match='infs or NaNs'):
                B.svd(torch.as_tensor(x, device=DEV), meta, sizes)
    x = np.full_like(a, np.nan)
    with pytest.raises(ValueError, match='infs or NaNs'):
        B.svd(torch.as_tensor(x, device=DEV), meta, sizes)
    U, S, V = (t.cpu().numpy() for t in B.svd(torch.as_tensor(a, device=DEV), meta, sizes))
    k, ref = min(m, n), a.reshape(m, n)
    # a few tens of rotations of every column, eps each: 50 eps sqrt(k)
    assert np.linalg.norm(U.reshape(m, k) * S @ V.reshape(k, n) - ref) <= 50 * 2.2e-16 * np.sqrt(k) * np.linalg.norm(ref)


@pytest.mark.parametrize('n', [24, 40, 130])
def test_eigh_refuses_nonfinite_blocks(n):
    from yastn_amd import backend_hip as B
    print('nonfinite eigh', n, flush=True)
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    a = a + a.T
    meta = (((0, n * n), (n, n), (0, n * n), (n, n), (0, n)),)
    for bad in (np.nan, np.inf):
        x = a.copy()
        x[n // 3, n // 2] = x[n // 2, n // 3] = bad
        with pytest.raises(ValueError, match='infs or NaNs'):
            B.eigh(torch.as_tensor(x.ravel(), device=DEV), meta, (n, n * n))
    S, _ = B.eigh(torch.as_tensor(a.ravel(), device=DEV), meta, (n, n * n))
    # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
    assert np.max(np.abs(S.cpu().numpy() - np.linalg.eigvalsh(a))) <= 50 * 2.2e-16 * n * np.linalg.norm(a)
