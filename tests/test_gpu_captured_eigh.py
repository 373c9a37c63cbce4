"""A captured eigendecomposition of blocks that fit one workgroup's LDS converges on replayed inputs that take more sweeps
than the eager calls before the capture did."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda:0'


@pytest.mark.parametrize('dims', [(40,), (64, 37, 12), (33, 20)])
def test_replay_takes_more_sweeps_than_the_warmup(dims):
    from yastn_amd import _functions as F
    from yastn_amd import backend_hip as B
    print('captured eigh', dims, flush=True)
    meta, a, s = [], 0, 0
    for n in dims:
        meta.append(((a, a + n * n), (n, n), (a, a + n * n), (n, n), (s, s + n)))
        a, s = a + n * n, s + n
    meta = tuple(meta)
    rng = np.random.default_rng(a)

    def matrices(kind):
        out = []
        for n in dims:
            x = np.diag(np.arange(1.0, n + 1)) if kind == 'diagonal' else rng.standard_normal((n, n))
            if kind == 'graded':
                x = x * 10.0 ** np.linspace(0, -6, n)[:, None] * 10.0 ** np.linspace(0, -6, n)
            out.append(x + x.T)
        return out

    data = torch.as_tensor(np.concatenate([x.ravel() for x in matrices('diagonal')]), device=DEV)
    B.eigh(data, meta, (s, a))
    torch.cuda.synchronize()
    graph, checks = torch.cuda.CUDAGraph(), F.deferred_checks()
    with checks, torch.cuda.graph(graph):
        S, U = B.eigh(data, meta, (s, a))
    for kind in ('random', 'graded', 'diagonal', 'random'):
        blocks = matrices(kind)
        data.copy_(torch.as_tensor(np.concatenate([x.ravel() for x in blocks])))
        eager = B.eigh(data.clone(), meta, (s, a))
        graph.replay()
        torch.cuda.synchronize()
        checks.check()
        assert torch.equal(S, eager[0]) and torch.equal(U, eager[1])
        for blk, (_, _, _, _, ss) in zip(blocks, meta):
            # the iteration runs on a + mu with mu the Gershgorin bound, at most sqrt(n) times the norm
            tol = 5e-14 * np.sqrt(len(blk)) * np.linalg.norm(blk)
            assert np.max(np.abs(S[ss[0]:ss[1]].cpu().numpy() - np.linalg.eigvalsh(blk))) <= tol
