"""The sign convention of U and Vh, 16 columns per workgroup, at the edges of its columns and rows; and the words the host
reads after a decomposition: smallest and negative info words, an infinity or NaN anywhere in the input."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('shapes', [((1, 1), (1, 5), (5, 1)), ((15, 40), (16, 16), (17, 63), (64, 17)),
                                    ((33, 33), (65, 32), (130, 129)), ((3, 2),) * 600])
def test_signs(shapes, cplx):
    from yastn_amd import backend_hip as B
    rng = np.random.default_rng(len(shapes))
    meta, a, u, s, v = [], 0, 0, 0, 0
    for m, n in shapes:
        k = min(m, n)
        meta.append(((a, a + m * n), (m, n), (u, u + m * k), (m, k), (s, s + k), (v, v + k * n), (k, n)))
        a, u, s, v = a + m * n, u + m * k, s + k, v + k * n
    U, V = (rng.standard_normal(n) + (1j * rng.standard_normal(n) if cplx else 0) for n in (u, v))
    U2, V2 = (t.cpu().numpy() for t in B.fix_svd_signs(*(torch.as_tensor(x, device=DEV) for x in (U, V)), tuple(meta)))
    for _, _, su, du, _, sv, dv in meta:
        ub, vb = U[su[0]:su[1]].reshape(du), V[sv[0]:sv[1]].reshape(dv)
        piv = ub[np.argmax(np.floor(np.abs(ub) * 2.0 ** 40), axis=0), np.arange(du[1])]
        ph = piv / np.abs(piv)
        # one division and one complex product: a few roundings of entries of order one to five
        np.testing.assert_allclose(U2[su[0]:su[1]].reshape(du), ub * ph.conj(), rtol=0, atol=2e-14)
        np.testing.assert_allclose(V2[sv[0]:sv[1]].reshape(dv), vb * ph[:, None], rtol=0, atol=2e-14)


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('n', [0, 1, 255, 257, 70001, 1 << 20])
def test_result_words(n, cplx):
    from yastn_amd import _lib as L
    dt = torch.complex128 if cplx else torch.float64
    x = torch.ones(n, dtype=dt, device=DEV)
    out = torch.empty(3 + L.YH_CHECK_SCRATCH, dtype=torch.int32, device=DEV)
    st = torch.cuda.current_stream().cuda_stream

    def words(info):
        t = torch.tensor(info, dtype=torch.int32, device=DEV)
        L.call('yastn_hip_check_result', out.data_ptr(), out.numel(), t.data_ptr(), len(info), x.data_ptr(), n,
               L.YH_C128 if cplx else L.YH_F64, st)
        return out[:3].tolist()
    assert words([3]) == [3, 0, 0]
    assert words([5, -1, 7] * 200) == [-1, 200, 0]
    assert words([2] * 300 + [-3]) == [-3, 1, 0]
    for pos in {0, n // 2, n - 1} if n else ():
        for bad in (float('inf'), float('-inf'), float('nan')):
            x[pos] = complex(0, bad) if cplx else bad
            assert words([1, 2]) == [1, 0, 1]
        x[pos] = 1
    assert words([4]) == [4, 0, 0]
