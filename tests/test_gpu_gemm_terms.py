"""Grouped GEMM kernels on lists whose term index differs from the GEMM index (GEMMs of no, one and several terms),
at the edges of the column tiles, with entries small enough that every sum is exact: the results have to be equal."""
import numpy as np
import pytest
import torch

from yastn_amd import _functions as F
from yastn_amd import _lib as L
from yastn_amd import plans as P

pytestmark = pytest.mark.gpu

COLUMNS = (1, 63, 255, 256, 257, 511, 512, 513, 769)
DEPTHS = (1, 3, 4, 5, 8, 9, 16, 17, 39, 40, 41, 47, 48, 80, 81, 95, 96, 97)  # short and steady k loops, with remainders
ROWS = ((1, 2, 3, 4), (1, 4, 5, 16), (17, 64, 65, 130))
CASES = [(r, c) for r in ROWS for c in sorted(L.TILE_DIMS) if c != L.YH_TILE_SMALLM or max(r) <= L.TILE_DIMS[c][0]]


def _strides(rng, rows, cols):
    """(rs, cs) of a dense rows x cols matrix in either order."""
    return (cols, 1) if rng.integers(2) else (1, rows)


def _entries(rng, n, cplx):
    x = rng.integers(-4, 5, n).astype(np.float64)
    return x + 1j * rng.integers(-4, 5, n) if cplx else x


@pytest.mark.parametrize('cplx', [False, True])
@pytest.mark.parametrize('rows, cfg', CASES)
def test_terms_and_tile_edges(rows, cfg, cplx):
    rng = np.random.default_rng(100 * cfg + len(rows) + rows[-1] + cplx)
    gemms, terms, mats, na, nb, nc = [], [], [], 0, 0, 0
    for i, N in enumerate(COLUMNS):
        M, tc = rows[i % len(rows)], (1, 0, 3, 2)[i % 4]
        rs, cs = _strides(rng, M, N)
        gemms.append((M, N, nc, rs, cs, len(terms), tc, i % 2))
        for _ in range(tc):
            K = int(rng.choice(DEPTHS))
            (ars, acs), (brs, bcs) = _strides(rng, M, K), _strides(rng, K, N)
            flags = int(rng.integers(4)) if cplx else 0
            terms.append((na, ars, acs, nb, brs, bcs, K, flags | (1 << 16)))
            na, nb = na + M * K, nb + K * N
        nc += M * N
    A, B, C = _entries(rng, na, cplx), _entries(rng, nb, cplx), _entries(rng, nc, cplx)
    ref = C.copy()

    def view(x, off, rs, cs, m, n):
        return x[off + rs * np.arange(m)[:, None] + cs * np.arange(n)]

    for M, N, off, rs, cs, tb, tc, acc in gemms:
        out = view(C, off, rs, cs, M, N) if acc else np.zeros((M, N), dtype=C.dtype)
        for a_off, ars, acs, b_off, brs, bcs, K, fl in terms[tb:tb + tc]:
            a, b = view(A, a_off, ars, acs, M, K), view(B, b_off, brs, bcs, K, N)
            out = out + (a.conj() if fl & 1 else a) @ (b.conj() if fl & 2 else b)
        ref[off + rs * np.arange(M)[:, None] + cs * np.arange(N)] = out
    plan = P.GemmPlan(gemms, terms, (na, nb), (nc,), 'cuda', cfg=cfg)
    dA, dB, dC = (torch.from_numpy(x).cuda() for x in (A, B, C))
    F.run_gemm(plan, (dC,), (dA, dB), F.dtype_code(dC), tune=False)
    assert np.array_equal(dC.cpu().numpy(), ref)
