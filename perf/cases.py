"""Performance cases of the block-sparse backend: what its users have it do, over the range they do it in.

Tensor-network programs call the backend in a few ways, and each is a kind of case here:

  transfer  one contraction of an MPS tensor with its conjugate (the step of every norm, overlap and transfer
            matrix), from a handful of elements, where the calls themselves cost, to 150 uneven sectors
  heff2     the two-site effective Hamiltonian of DMRG applied once (four contractions), the inner loop of
            Lanczos; called eagerly or replayed as a HIP graph, as a solver does with a fixed structure
  svd       a two-site tensor cut back to its bond (dimension and sector sizes) by a truncated block SVD
  eigh      the inverse square root of a positive Hermitian bond tensor by its block eigendecomposition
  qr        the block QR of a half-system, forward and backward
  ctmrg     a whole CTMRG step of an iPEPS with an observable, forward and backward, eager (two projector SVDs
            of a move one after the other) or captured (one HIP graph, both SVDs of a move in one call)
  corner    the product of two enlarged corners, forward and backward
  proj      the projectors between two half-systems (product, SVD, truncation, two products)

Blocks are seeded N(0, 1) numbers, scaled by a decaying bond spectrum where the real objects have one.
Charges follow the usual bell-shaped sector sizes, so odd and ragged block shapes are the rule.
"""
import itertools
import math

import numpy as np
import torch

DEVICE = 'cuda:0'


def _backend():
    from yastn_amd import backend_hip
    return backend_hip


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest contraction: a transfer step of a short MPS (45 000 flops), all latency
        {'name': 'transfer_78', 'kind': 'transfer', 'sym': 'U1', 'chi': 78, 'dtype': 'float64',
         'policy': 'fuse_contracted'},
        # the smallest truncation: nine blocks up to about 30 x 30
        {'name': 'svd_78', 'kind': 'svd', 'chi': 78, 'dtype': 'float64'},
        # many uneven sectors at once: two conserved charges, complex
        {'name': 'transfer_u1u1_2048', 'kind': 'transfer', 'sym': 'U1xU1', 'chi': 2048, 'dtype': 'complex128',
         'policy': 'fuse_contracted'},
        # DMRG at production size, the solver's inner loop replayed as a graph
        {'name': 'heff2_1024_graph', 'kind': 'heff2', 'chi': 1024, 'dtype': 'float64', 'policy': 'fuse_contracted',
         'graph': True},
        # DMRG / TDVP with complex tensors at an ordinary odd size, without leg fusion
        {'name': 'heff2_301_c128', 'kind': 'heff2', 'chi': 301, 'dtype': 'complex128', 'policy': 'no_fusion',
         'graph': False},
        # the truncation that follows it at production size: 27 blocks up to 198 x 198
        {'name': 'svd_1024', 'kind': 'svd', 'chi': 1024, 'dtype': 'float64'},
        # gauge fixing / canonical forms: 25 Hermitian blocks up to about 106 x 106
        {'name': 'eigh_1024', 'kind': 'eigh', 'chi': 1024, 'dtype': 'float64'},
        # QR-reduced projectors: 13 blocks from 4 to 440
        {'name': 'qr_6_64', 'kind': 'qr', 'D': 6, 'chi': 64, 'dtype': 'float64'},
        # one iPEPS optimisation step in the usual eager call pattern
        {'name': 'ctmrg_6_64', 'kind': 'ctmrg', 'D': 6, 'chi': 64, 'graph': False},
        # the same step captured once and replayed
        {'name': 'ctmrg_6_64_graph', 'kind': 'ctmrg', 'D': 6, 'chi': 64, 'graph': True},
        # the largest contractions: enlarged corners of a D = 8 complex iPEPS
        {'name': 'corner_8_128', 'kind': 'corner', 'D': 8, 'chi': 128, 'dtype': 'complex128'},
        # the largest decomposition: blocks up to 1134 x 1134, complex
        {'name': 'proj_8_128', 'kind': 'proj', 'D': 8, 'chi': 128, 'dtype': 'complex128'},
    ]


def draw(rng):
    def between(lo, hi):  # spread over the logarithm, odd sizes among them
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(('transfer', 'heff2', 'svd', 'eigh', 'qr', 'ctmrg', 'corner', 'proj'))
    dtype = rng.choice(('float64', 'complex128'))
    if kind == 'transfer':
        return {'kind': kind, 'sym': rng.choice(('U1', 'U1xU1')), 'chi': between(32, 2048), 'dtype': dtype,
                'policy': rng.choice(('fuse_contracted', 'fuse_to_matrix', 'no_fusion'))}
    if kind == 'heff2':
        return {'kind': kind, 'chi': between(32, 1024), 'dtype': dtype,
                'policy': rng.choice(('fuse_contracted', 'fuse_contracted', 'no_fusion')),
                'graph': rng.random() < 0.5}
    if kind in ('svd', 'eigh'):
        return {'kind': kind, 'chi': between(32, 1024), 'dtype': dtype}
    if kind == 'ctmrg':
        return {'kind': kind, 'D': rng.choice((3, 6)), 'chi': between(16, 48), 'graph': rng.random() < 0.5}
    return {'kind': kind, 'D': rng.choice((3, 4, 6, 8)), 'chi': between(24, 120), 'dtype': dtype}


# ------------------------------------------------------------------------------------------------ structures
# A leg is (signature, charges in ascending order (tuples), dimensions).

def _split(total, charges, weight):
    """Sector sizes proportional to the weight, at least 1, the rounding rest in the middle sector."""
    w = np.array([weight(q) for q in charges])
    D = np.maximum(1, np.round(total * w / w.sum())).astype(int)
    D[int(np.argmax(w))] += total - int(D.sum())
    return tuple(int(x) for x in D)


def _bond(chi, sym='U1'):
    """Charges and sector sizes of an MPS bond."""
    if sym == 'U1':
        qmax = max(2, min(12, int(2 * math.log2(chi) - 8)))
        var = 2 * (1 + qmax / 4) ** 2
        qs = list(range(-qmax, qmax + 1))
        return [(q,) for q in qs], _split(chi, qs, lambda q: math.exp(-q * q / var))
    n = max(5, min(150, round(chi / 13.65)))
    var = 2 * 9.0 * n / 150
    w = {c: math.exp(-(c[0] ** 2 + c[1] ** 2) / var) for c in itertools.product(range(-12, 13), repeat=2)}
    qs = sorted(sorted(w, key=lambda c: (-w[c], c))[:n])
    return qs, _split(chi, qs, w.get)


def _env(chi):
    """Charges and sector sizes of an environment leg."""
    qmax = 2 + min(4, chi // 32)
    qs = list(range(-qmax, qmax + 1))
    return [(q,) for q in qs], _split(chi, qs, lambda q: math.exp(-q * q / (2 * qmax - 2)))


def _env_of_step(chi):
    """The same for the environments that a CTMRG step is set up with: five charges unless chi is 64 or 128."""
    if chi in (64, 128):
        return _env(chi)
    qs = list(range(-2, 3))
    return [(q,) for q in qs], _split(chi, qs, lambda q: math.exp(-q * q / 4))


_SITE = {3: {-1: 1, 0: 1, 1: 1}, 4: {-1: 1, 0: 2, 1: 1}, 6: {-1: 2, 0: 2, 1: 2}, 8: {-2: 1, -1: 2, 0: 2, 1: 2, 2: 1}}


def _double(D):
    """Charges and sector sizes of a double-layer leg: ket charge minus bra charge."""
    d = {}
    for k, dk in _SITE[D].items():
        for b, db in _SITE[D].items():
            d[k - b] = d.get(k - b, 0) + dk * db
    qs = sorted(d)
    return [(q,) for q in qs], tuple(d[q] for q in qs)


def _blocks(legs):
    """Charge indices and shapes of the allowed blocks (total charge zero), in ascending charge order."""
    for idx in itertools.product(*(range(len(l[1])) for l in legs)):
        n = len(legs[0][1][0])
        if all(sum(l[0] * l[1][i][c] for l, i in zip(legs, idx)) == 0 for c in range(n)):
            yield idx, tuple(l[2][i] for l, i in zip(legs, idx))


def _size(legs):
    return sum(math.prod(shape) for _, shape in _blocks(legs))


def _normal(n, dtype, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n)
    return x + 1j * rng.standard_normal(n) if dtype == 'complex128' else x


def _config(sym='U1', policy='fuse_contracted'):
    from yastn_amd import blocksparse as bs
    return bs.make_config(_backend(), sym, device=DEVICE, tensordot_policy=policy)


def _tensor(config, legs, flat):
    from yastn_amd import blocksparse as bs
    return bs.from_flat(config, [bs.leg(config, s, t, D) for s, t, D in legs],
                        (0,) * len(legs[0][1][0]), flat)


# ------------------------------------------------------------------------------------------------ the inputs
# What a case's tensors are, as (legs, block buffer) pairs made from the seed alone.

def _mps(case, seed):
    if case['sym'] == 'U1':
        phys = ([(0,), (1,)], (1, 1))
    else:
        phys = ([(0, 0), (0, 1), (1, 0), (1, 1)], (1, 1, 1, 1))
    v = _bond(case['chi'], case['sym'])
    legs = [(1, *v), (1, *phys), (-1, *v)]
    return legs, _normal(_size(legs), case['dtype'], seed)


_SPIN = ([(-1,), (1,)], (1, 1))
_MPO = ([(-2,), (0,), (2,)], (1, 3, 1))


def _two_site(case, seed):
    """A two-site tensor whose bond spectra decay, as those of a state do."""
    v = _bond(case['chi'])
    legs = [(1, *v), (1, *_SPIN), (1, *_SPIN), (-1, *v)]
    x = _normal(_size(legs), case['dtype'], seed)
    o = 0
    for idx, shape in _blocks(legs):
        n = math.prod(shape)
        a, b = (10.0 ** (-3 * np.arange(k) / k) for k in (shape[0], shape[3]))
        block = x[o:o + n].reshape(shape)
        block *= a[:, None, None, None] * b
        o += n
    return legs, x


def _xxz():
    """The XXZ Hamiltonian's MPO tensor (bond, out, bond, in), bond basis ordered by charge."""
    eye, sz = np.eye(2), np.diag([-0.5, 0.5])
    up = np.array([[0.0, 0.0], [1.0, 0.0]])
    W = np.zeros((5, 2, 5, 2))
    for a, b, op in ((0, 0, eye), (1, 0, up), (2, 0, up.T), (3, 0, sz), (4, 1, up.T / 2), (4, 2, up / 2), (4, 3, sz),
                     (4, 4, eye)):
        W[a, :, b, :] = op
    W = W[[1, 0, 3, 4, 2]][:, :, [1, 0, 3, 4, 2]]
    legs = [(1, *_MPO), (1, *_SPIN), (-1, *_MPO), (-1, *_SPIN)]
    return legs, _flat(torch.from_numpy(W), legs, _allowed(legs)).numpy()


def _heff2_inputs(case, seed):
    v = _bond(case['chi'])
    AA = [(1, *v), (1, *_SPIN), (1, *_SPIN), (-1, *v)]
    FR = [(1, *v), (1, *_MPO), (-1, *v)]
    FL = [(-1, *v), (-1, *_MPO), (1, *v)]
    return [(legs, _normal(_size(legs), case['dtype'], 3 * seed + k)) for k, legs in enumerate((AA, FL, FR))] + [_xxz()]


def _density(case, seed):
    """A positive Hermitian bond tensor: X X^H of blocks twice as wide as high."""
    v = _bond(case['chi'])
    out = []
    rng = np.random.default_rng(seed)
    for n in v[1]:
        x = rng.standard_normal((n, 2 * n)) / math.sqrt(2 * n)
        if case['dtype'] == 'complex128':
            x = (x + 1j * rng.standard_normal((n, 2 * n)) / math.sqrt(2 * n)) / math.sqrt(2)
        out.append((x @ x.conj().T).ravel())
    return [(1, *v), (-1, *v)], np.concatenate(out)


def _corner_leg(D, chi):
    """Charges and sizes of a fused (environment, double-layer) leg."""
    e, d = _env(chi), _double(D)
    n = {}
    for (q,), a in zip(*e):
        for (p,), b in zip(*d):
            n[q + p] = n.get(q + p, 0) + a * b
    qs = sorted(n)
    return [(q,) for q in qs], tuple(n[q] for q in qs)


def _square(case, seed):
    v = _corner_leg(case['D'], case['chi'])
    legs = [(1, *v), (-1, *v)]
    return legs, _normal(_size(legs), case['dtype'], seed) / math.sqrt(max(v[1]))


def _half(case, seed, s):
    """A half-system (env, double, env', double'): random, with the decaying spectra of the environment legs."""
    e, d = _env(case['chi']), _double(case['D'])
    legs = [(s, *e), (s, *d), (-s, *e), (-s, *d)]
    x = _normal(_size(legs), case['dtype'], seed) / math.sqrt(case['chi'])
    o = 0
    for idx, shape in _blocks(legs):
        n = math.prod(shape)
        a, b = (10.0 ** (-2 * np.arange(k) / k) for k in (shape[0], shape[2]))
        block = x[o:o + n].reshape(shape)
        block *= a[:, None, None, None] * b[:, None]
        o += n
    return legs, x


# ------------------------------------------------------------------------------------------------ prepare and run

def _capture(fn):
    """fn captured as a HIP graph after warm-up passes on a side stream; (graph, output)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def prepare(case, seed):
    from yastn_amd import ctmrg as C, workloads as W
    kind, state = case['kind'], {'case': case}
    if kind == 'transfer':
        state['A'] = _tensor(_config(case['sym'], case['policy']), *_mps(case, seed))
    elif kind == 'heff2':
        config = _config(policy=case['policy'])
        state['args'] = [_tensor(config, *x) for x in _heff2_inputs(case, seed)]
        if case['graph']:
            with torch.no_grad():
                state['graph'], state['out'] = _capture(lambda: W.heff2(*state['args']))
    elif kind == 'svd':
        state['A'] = _tensor(_config(), *_two_site(case, seed))
        state['cut'] = {'D_total': case['chi'], 'D_block': dict(zip(*_bond(case['chi'])))}  # the sector sizes stay
    elif kind == 'eigh':
        state['A'] = _tensor(_config(), *_density(case, seed))
    elif kind == 'qr':
        legs, flat = _square(case, seed)
        state['A'] = _tensor(_config(), legs, flat)
        state['w'] = [torch.as_tensor(_normal(len(flat), case['dtype'], 7 * seed + k), device=DEVICE) for k in (1, 2)]
    elif kind == 'ctmrg':
        A, env, sz = C.setup(_config(), D=case['D'], chi=case['chi'], seed=seed)
        state['args'] = (A, env, sz, case['chi'])
        if case['graph']:
            state['step'], _ = C.captured_fwd_bwd(*state['args'], batch=True)
    elif kind == 'corner':
        config = _config()
        state['AB'] = [_tensor(config, *_square(case, 2 * seed + k)) for k in (0, 1)]
        legs, flat = _square(case, 2 * seed + 1000003)
        state['w'] = torch.as_tensor(flat, device=DEVICE)
    elif kind == 'proj':
        config = _config()
        state['r'] = [_tensor(config, *_half(case, 2 * seed + k, s)).fuse_legs(axes=((0, 1), (2, 3)))
                      for k, s in ((0, 1), (1, -1))]
        state['cut'] = {'D_block': dict(zip(*_env(case['chi'])))}
    return state


def run(state):
    from yastn_amd import blocksparse as bs, ctmrg as C, workloads as W
    case = state['case']
    kind = case['kind']
    if kind == 'ctmrg':
        if case['graph']:
            loss, grad = state['step'].replay()
        else:
            loss, grad = C.fwd_bwd(*state['args'])
        return {'loss': loss, 'grad': grad}
    if kind == 'qr':
        data = state['A'].data.detach().clone().requires_grad_(True)
        Q, R = bs.qr(state['A']._replace(data=data), axes=(0, 1), sQ=-1)
        torch.autograd.backward([Q.data, R.data], state['w'])
        return {'Q': Q.data, 'R': R.data, 'grad': data.grad}
    if kind == 'corner':
        a, b = (t.data.detach().requires_grad_(True) for t in state['AB'])
        c = state['AB'][0]._replace(data=a) @ state['AB'][1]._replace(data=b)
        ga, gb = torch.autograd.grad(c.data, (a, b), state['w'])
        return {'C': c.data, 'gA': ga, 'gB': gb}
    with torch.no_grad():
        if kind == 'transfer':
            return W.u1xu1_transfer(state['A']).data
        if kind == 'heff2':
            if case['graph']:
                state['graph'].replay()
                return state['out'].data
            return W.heff2(*state['args']).data
        if kind == 'svd':
            U, S, V = bs.svd_with_truncation(state['A'], axes=((0, 1), (2, 3)), fix_signs=True, **state['cut'])
            return {'U': U.data, 'S': S.data, 'V': V.data}
        if kind == 'eigh':
            S, U = bs.eigh(state['A'], axes=(0, 1))
            return {'S': S.data, 'rsqrt': (U @ S.rsqrt() @ U.conj().transpose((1, 0))).data}
        p0, p1 = C.proj_corners(*state['r'], case['chi'], svd_opts=state['cut'])
        return {'p0': p0.data, 'p1': p1.data}


# ------------------------------------------------------------------------------------------------ what a pass needs

def _sum(*legs):
    """{total charge: dimension} of several legs together."""
    n = {(0,) * len(legs[0][1][0]): 1}
    for s, t, D in legs:
        m = {}
        for q, a in n.items():
            for c, d in zip(t, D):
                k = tuple(x + s * y for x, y in zip(q, c))
                m[k] = m.get(k, 0) + a * d
        n = m
    return n


def _flip(leg):
    return (-leg[0], *leg[1:])


def _macs(left, inner, right):
    """Multiply-adds of a contraction over `inner` (legs of the left tensor): sum over sectors of M K N."""
    M, K, N = _sum(*left), _sum(*inner), _sum(*right)
    return sum(m * K.get(tuple(-x for x in q), 0) * N.get(tuple(-x for x in q), 0) for q, m in M.items())


def work(case):
    cplx = case.get('dtype') == 'complex128'
    item, mul = (16, 8) if cplx else (8, 2)  # bytes of an element, flops of a multiply-add
    kind = case['kind']
    if kind == 'transfer':
        legs, x = _mps(case, 0)
        macs = _macs([_flip(legs[2])], [_flip(legs[0]), _flip(legs[1])], [legs[2]])
        return {'bytes': item * (len(x) + sum(d * d for d in legs[2][2])), 'flops': mul * macs}
    if kind == 'heff2':
        (AA, a), (FL, l), (FR, r), (W, w) = _heff2_inputs(case, 0)
        v, m = AA[3], FR[1]
        macs = _macs(AA[:3], [v], [m, FR[2]])
        one = _macs([W[0], W[1]], [W[2], W[3]], [AA[0], AA[1], FR[2]])
        macs += 2 * one + _macs([FL[2]], [FL[0], FL[1]], [AA[1], AA[2], FR[2]])
        return {'bytes': item * (2 * len(a) + len(l) + len(r) + len(w)), 'flops': mul * macs}
    if kind == 'svd':
        v = _bond(case['chi'])
        m = _sum((1, *v), (1, *_SPIN))
        n = _sum((-1, *v), (1, *_SPIN))
        dims = [(a, n.get(tuple(-x for x in q), 0)) for q, a in m.items()]
        kept = 2 * case['chi'] * max(1, case['chi'] // len(v[1]))
        flops = sum(4 * a * b * min(a, b) + 8 * min(a, b) ** 3 for a, b in dims)
        return {'bytes': item * (sum(a * b for a, b in dims) + kept), 'flops': flops * mul / 2}
    if kind == 'eigh':
        dims = _bond(case['chi'])[1]
        return {'bytes': item * 2 * sum(d * d for d in dims), 'flops': sum((9 + 2) * d ** 3 for d in dims) * mul / 2}
    n = _corner_leg(case['D'], case['chi'])[1]
    n2, n3 = sum(d * d for d in n), sum(d ** 3 for d in n)
    if kind == 'qr':  # 4/3 n^3 each for R and Q, three products of the adjoint
        return {'bytes': item * 6 * n2, 'flops': (8 / 3 + 6) * n3 * mul / 2}
    if kind == 'corner':
        return {'bytes': item * 6 * n2, 'flops': 3 * mul * n3}
    if kind == 'proj':  # the product, the SVD, two thin products
        return {'bytes': item * 2 * n2, 'flops': (2 + 12) * n3 * mul / 2}
    e, d, s = (1, *_env_of_step(case['chi'])), (1, *_double(case['D'])), _SITE[case['D']]
    fused = _sum(e, d).values()
    n3 = sum(k ** 3 for k in fused)
    corner = _macs([e, e], [d, d], [d, d]) + 2 * _macs([e, d], [e], [e])
    edge = _macs([e, d], [e, d], [e]) + _macs([d, d], [d, d], [e, e]) + _macs([e], [e, d], [e, d])
    # per move four corners, two halves, two products, SVDs (with their adjoint) and projectors, six renormalised tensors
    move = 4 * corner + 4 * n3 + 2 * edge + 4 * _macs([e], [e], [e, d])
    svd = 2 * 12 * n3
    total = 2 * (2 * move + 5 * corner + n3) * 3 + 2 * svd + 2 * 2 * 8 * n3
    env = 4 * _size([e, _flip(e)]) + 4 * _size([e, d, _flip(e)])
    site = 2 * sum(s.values()) ** 4 // 3
    return {'bytes': 8 * (env + 2 * site), 'flops': total}


# ------------------------------------------------------------------------------------------------ exact values
# Plain dense arithmetic in 64 bits on the same inputs: legs laid out with their sectors in ascending charge.

def _offsets(leg):
    return [0, *itertools.accumulate(leg[2])]


def _allowed(legs):
    """Charge-level presence of the blocks allowed by the selection rule."""
    p = np.zeros([len(l[1]) for l in legs], dtype=bool)
    for idx, _ in _blocks(legs):
        p[idx] = True
    return p


def _dense(flat, legs, device=None):
    flat = torch.as_tensor(flat, device=device or DEVICE)
    x = torch.zeros([sum(l[2]) for l in legs], dtype=flat.dtype, device=flat.device)
    offs = [_offsets(l) for l in legs]
    o = 0
    for idx, shape in _blocks(legs):
        n = math.prod(shape)
        x[tuple(slice(f[i], f[i + 1]) for f, i in zip(offs, idx))] = flat[o:o + n].reshape(shape)
        o += n
    return x


def _flat(x, legs, present):
    offs = [_offsets(l) for l in legs]
    parts = [x[tuple(slice(f[i], f[i + 1]) for f, i in zip(offs, idx))].reshape(-1) for idx in np.argwhere(present)]
    return torch.cat(parts) if parts else x.new_zeros(0)


def _contract(X, Y, axes):
    """tensordot of (array, legs, presence) triples."""
    (x, lx, px), (y, ly, py) = X, Y
    rest = [l for i, l in enumerate(lx) if i not in axes[0]] + [l for i, l in enumerate(ly) if i not in axes[1]]
    p = np.tensordot(px.astype(np.int64), py.astype(np.int64), axes=axes) > 0
    return torch.tensordot(x, y, dims=axes), rest, p


def _labels(*legs):
    """Total charge of every dense index of the fused legs (one conserved charge)."""
    out = np.zeros(1, dtype=int)
    for s, t, D in legs:
        out = (out[:, None] + s * np.repeat([q[0] for q in t], D)[None, :]).ravel()
    return out


def _signed(u, v):
    """Singular vectors with the largest entry of each column of u (the first, in steps of 2^-40) made real positive."""
    piv = u[(u.abs() * 2.0 ** 40).floor().argmax(0), torch.arange(u.shape[1], device=u.device)]
    ph = piv / piv.abs()
    return u * ph.conj(), ph[:, None] * v


def _svd_blocks(blocks, keep):
    """{charge: (u, s, v)} of a dict of matrices in ascending charge, signs fixed, keep[charge] values each."""
    cut = {}
    for q, k in sorted(keep.items()):
        m = blocks.get(q)
        if m is not None and min(m.shape):
            u, s, v = torch.linalg.svd(m.cpu(), full_matrices=False)
            u, v = _signed(u, v)
            cut[q] = tuple(x.to(m.device) for x in (u[:, :k], s[:k], v[:k]))
    return cut


def _exact_svd(case, seed):
    legs, flat = _two_site(case, seed)
    x = _dense(flat, legs)
    m = x.reshape(x.shape[0] * 2, -1)
    rows, cols = _labels(*legs[:2]), -_labels(*legs[2:])
    blocks = {}
    for q in sorted(set(rows) & set(cols)):
        i, j = (torch.from_numpy(np.flatnonzero(a == q)).to(m.device) for a in (rows, cols))
        blocks[q] = (i, j, m[i][:, j])
    # a block's bond charge is the negative of its row charge
    cut = _svd_blocks({-q: b[2] for q, b in blocks.items()}, {q: k for (q,), k in zip(*_bond(case['chi']))})
    bond = ([(int(q),) for q in cut], tuple(len(s) for _, s, _ in cut.values()))
    U = m.new_zeros(m.shape[0], sum(bond[1]))
    V = m.new_zeros(sum(bond[1]), m.shape[1])
    o = 0
    for q, (u, s, v) in cut.items():
        i, j, _ = blocks[-q]
        U[i, o:o + len(s)] = u
        V[o:o + len(s)].index_copy_(1, j, v)
        o += len(s)
    lu, lv = [*legs[:2], (1, *bond)], [(-1, *bond), *legs[2:]]
    return {'U': _flat(U.reshape(x.shape[0], 2, -1), lu, _allowed(lu)), 'S': torch.cat([s for _, s, _ in cut.values()]),
            'V': _flat(V.reshape(-1, 2, x.shape[3]), lv, _allowed(lv))}


def _each(flat, dims):
    """The square diagonal blocks of a two-leg tensor."""
    flat = torch.as_tensor(flat)
    o = 0
    for n in dims:
        yield flat[o:o + n * n].reshape(n, n)
        o += n * n


def _exact_qr(case, seed):
    legs, flat = _square(case, seed)
    dims = legs[0][2]
    w = [_each(_normal(len(flat), case['dtype'], 7 * seed + k), dims) for k in (1, 2)]
    out = {'Q': [], 'R': [], 'grad': []}
    for a, wq, wr in zip(_each(flat, dims), *w):
        a = a.clone().requires_grad_(True)
        q, r = torch.linalg.qr(a)
        d = torch.diagonal(r).detach()
        ph = torch.where(d.real < 0, -torch.ones_like(d), torch.ones_like(d))
        q, r = q * ph, ph[:, None] * r
        torch.autograd.backward([q, r], [wq, wr])
        for k, x in zip(out, (q.detach(), r.detach(), a.grad)):
            out[k].append(x.reshape(-1))
    return {k: torch.cat(x) for k, x in out.items()}


def _exact_corner(case, seed):
    dims = _square(case, 0)[0][0][2]
    A, B, W = (_each(torch.as_tensor(_square(case, 2 * seed + k)[1], device=DEVICE), dims) for k in (0, 1, 1000003))
    out = {'C': [], 'gA': [], 'gB': []}
    for a, b, w in zip(A, B, W):
        for k, x in zip(out, (a @ b, w @ b.conj().T.contiguous(), a.conj().T.contiguous() @ w)):
            out[k].append(x.reshape(-1))
    return {k: torch.cat(x) for k, x in out.items()}


def _exact_proj(case, seed):
    e, d = _env(case['chi']), _double(case['D'])
    lab = _labels((1, *e), (1, *d))
    r = []
    for k, s in ((0, 1), (1, -1)):
        legs, flat = _half(case, 2 * seed + k, s)
        r.append(_dense(flat, legs).reshape(len(lab), -1))
    idx = {int(q): torch.from_numpy(np.flatnonzero(lab == q)).to(r[0].device) for q in sorted(set(lab))}
    sub = {q: [x[i][:, i] for x in r] for q, i in idx.items()}
    cut = _svd_blocks({q: a @ b.T.contiguous() for q, (a, b) in sub.items()}, {q: k for (q,), k in zip(*e)})
    bond = ([(q,) for q in cut], tuple(len(s) for _, s, _ in cut.values()))
    p = [r[0].new_zeros(len(lab), sum(bond[1])) for _ in (0, 1)]
    o = 0
    for q, (u, s, v) in cut.items():
        a, b = sub[q]
        p[0][idx[q], o:o + len(s)] = b.T.contiguous() @ (v.conj() / s.sqrt()[:, None]).T.contiguous()
        p[1][idx[q], o:o + len(s)] = a.T.contiguous() @ (u / s.sqrt()).conj()
        o += len(s)
    out = {}
    for name, x, s in (('p0', p[0], 1), ('p1', p[1], -1)):
        legs = [(s, *e), (s, *d), (-s, *bond)]
        out[name] = _flat(x.reshape(sum(e[1]), sum(d[1]), -1), legs, _allowed(legs))
    return out


class _Svd(torch.autograd.Function):
    """Real square SVD with fixed signs; its adjoint regularises x / (x^2 + 1e-12), as the usual iPEPS codes do."""

    @staticmethod
    def forward(ctx, m):
        u, s, v = torch.linalg.svd(m.cpu(), full_matrices=False)
        u, v = _signed(u, v)
        u, s, v = u.to(m.device), s.to(m.device), v.to(m.device)
        ctx.save_for_backward(u, s, v)
        return u, s, v

    @staticmethod
    def backward(ctx, gu, gs, gv):
        u, s, v = ctx.saved_tensors
        inv = lambda x: x / (x * x + 1e-12)
        F, G = inv(s[None, :] - s[:, None]), inv(s[None, :] + s[:, None])
        F.fill_diagonal_(0)
        G.fill_diagonal_(0)
        X, Y = u.T @ gu, v @ gv.T
        J = 0.5 * (F + G) * (X - X.T) + 0.5 * (F - G) * (Y - Y.T) + torch.diag(gs)
        return u @ J @ v


def _exact_ctmrg(case, seed):
    """The step on dense tensors whose legs carry charge labels, differentiated by torch."""
    D, chi = case['D'], case['chi']
    site, dbl, env = _SITE[D], _double(D), _env_of_step(chi)
    v = ([(q,) for q in sorted(site)], tuple(site[q] for q in sorted(site)))
    legs = [(-1, *v), (1, *v), (1, *v), (-1, *v), (1, [(0,), (1,)], (1, 1))]
    flat = torch.as_tensor(_normal(_size(legs), 'float64', seed) / math.sqrt(_size(legs)), device=DEVICE).requires_grad_(True)
    where = _dense(torch.arange(1, flat.numel() + 1), legs)
    A = torch.where(where > 0, flat[(where - 1).clamp(min=0)], torch.zeros((), dtype=torch.float64, device=DEVICE))
    one = np.repeat([q[0] for q in v[0]], v[1])
    pair = torch.from_numpy(np.argsort((one[:, None] - one[None, :]).ravel(), kind='stable')).to(A.device)

    def layer(op=None):  # double-layer site, each leg's (ket, bra) index sorted by charge
        a = torch.einsum('tlbrp,TLBRp->tTlLbBrR', A if op is None else torch.einsum('tlbrq,qp->tlbrp', A, op), A)
        a = a.reshape([len(one) ** 2] * 4)
        for i in range(4):
            a = a.index_select(i, pair)
        return a

    names = ('tl', 't', 'tr', 'r', 'br', 'b', 'bl', 'l')
    mid = {'t': 1, 'r': 1, 'b': -1, 'l': -1}
    E = {}
    for i, k in enumerate(names):
        ls = [(-1, *env), (mid[k], *dbl), (1, *env)] if k in mid else [(-1, *env), (1, *env)]
        E[k] = _dense(_normal(_size(ls), 'float64', seed + 10 + i), ls)
    td = torch.tensordot
    lab = np.repeat([q[0] for q in env[0]], env[1])  # charges of the environment legs, dense
    ld = np.repeat([q[0] for q in dbl[0]], dbl[1])
    split = {q: n for (q,), n in zip(*env)}

    def corners(E, a, first=None):
        def fuse(c, order):
            c = c.permute(order)
            return c.reshape(c.shape[0] * c.shape[1], -1)
        one_ = lambda x, y, z: td(td(x, y, dims=([2], [0])), z, dims=([2], [0]))
        tl = fuse(td(one_(E['l'], E['tl'], E['t']), a if first is None else first, dims=([2, 1], [0, 1])), (0, 2, 1, 3))
        tr = fuse(td(one_(E['t'], E['tr'], E['r']), a, dims=([1, 2], [0, 3])), (0, 2, 1, 3))
        br = fuse(td(one_(E['r'], E['br'], E['b']), a, dims=([2, 1], [2, 3])), (0, 2, 1, 3))
        bl = fuse(td(one_(E['b'], E['bl'], E['l']), a, dims=([2, 1], [1, 2])), (0, 3, 1, 2))
        return tl, tr, br, bl

    def projectors(r0, r1, left):
        """p0, p1 between r0 and r1; `left`: the charge labels of r0's rows, the negative of those r1's rows meet."""
        rr = td(r0, r1, dims=([1], [1]))
        factors = {}
        for q in sorted(set(left)):
            i = torch.from_numpy(np.flatnonzero(left == q)).to(rr.device)
            factors[q] = (i, *_Svd.apply(rr[i][:, i]))
        if case['graph']:
            keep = {q: min(n, factors[q][2].numel()) for q, n in split.items() if q in factors}
        else:
            ranked = sorted(((x, q) for q, f in factors.items() for x in f[2].tolist()), reverse=True)[:chi]
            keep = {}
            for x, q in ranked:
                if x > 0:
                    keep[q] = keep.get(q, 0) + 1
        p0, p1 = [], []
        for q, k in sorted(keep.items()):
            i, u, s, vh = factors[q]
            rs = s[:k].rsqrt()
            p0.append(r1[i].T @ (rs[:, None] * vh[:k]).T)
            p1.append(r0[i].T @ (u[:, :k] * rs))
        return [torch.cat(p, 1).reshape(len(lab), len(ld), -1) for p in (p0, p1)]

    unit = lambda t: t / t.abs().max()
    a = layer()
    # The first leg of an environment tensor carries the label -lab, the last +lab, the site's legs -ld, +ld, +ld, -ld;
    # rows of both half-systems that meet list the same charges in the same order, with opposite signs.
    flat_sum = lambda x, y: (x[:, None] + y[None, :]).ravel()
    tl, tr, br, bl = corners(E, a)
    tt, bb = tl @ tr, br @ bl
    hrb, hrt = projectors(tt, bb.T, flat_sum(-lab, ld))
    hlb, hlt = projectors(tt.T, bb, flat_sum(lab, ld))
    N = dict(E)
    N['l'] = unit(td(hlb, td(a, td(E['l'], hlt, dims=([2], [0])), dims=([0, 1], [2, 1])), dims=([0, 1], [2, 0])))
    N['tl'] = unit(td(hlb, td(E['tl'], E['t'], dims=([1], [0])), dims=([0, 1], [0, 1])))
    N['bl'] = unit(td(E['b'], td(E['bl'], hlt, dims=([1], [0])), dims=([2, 1], [0, 1])))
    N['r'] = unit(td(hrt, td(a, td(E['r'], hrb, dims=([2], [0])), dims=([2, 3], [2, 1])), dims=([0, 1], [2, 0])))
    N['tr'] = unit(td(E['t'], td(E['tr'], hrb, dims=([1], [0])), dims=([2, 1], [0, 1])))
    N['br'] = unit(td(hrt, td(E['br'], E['b'], dims=([1], [0])), dims=([0, 1], [0, 1])))
    E = N
    tl, tr, br, bl = corners(E, a)
    ll, rr = bl @ tl, tr @ br
    vtr, vtl = projectors(ll, rr.T, flat_sum(-lab, -ld))
    vbr, vbl = projectors(ll.T, rr, flat_sum(lab, -ld))
    N = dict(E)
    N['t'] = unit(td(td(td(vtl, E['t'], dims=([0], [0])), a, dims=([2, 0], [0, 1])), vtr, dims=([1, 3], [0, 1])))
    N['tl'] = unit(td(E['l'], td(E['tl'], vtr, dims=([1], [0])), dims=([2, 1], [0, 1])))
    N['tr'] = unit(td(vtl, td(E['tr'], E['r'], dims=([1], [0])), dims=([0, 1], [0, 1])))
    N['b'] = unit(td(td(td(vbr, E['b'], dims=([0], [0])), a, dims=([2, 0], [2, 3])), vbl, dims=([1, 3], [0, 1])))
    N['bl'] = unit(td(vbr, td(E['bl'], E['l'], dims=([1], [0])), dims=([0, 1], [0, 1])))
    N['br'] = unit(td(E['r'], td(E['br'], vbl, dims=([1], [0])), dims=([2, 1], [0, 1])))
    E = N
    tl, tr, br, bl = corners(E, a)
    sz = torch.tensor([[-0.5, 0.0], [0.0, 0.5]], dtype=torch.float64, device=DEVICE)
    tlo = corners(E, a, first=layer(sz))[0]
    rest = tr @ (br @ bl)
    loss = (tlo * rest.T).sum() / (tl * rest.T).sum()
    loss.backward()
    return {'loss': loss.detach(), 'grad': flat.grad}


def exact(case, seed):
    kind = case['kind']
    if kind == 'transfer':
        legs, flat = _mps(case, seed)
        x, p = _dense(flat, legs), _allowed(legs)
        y, out, q = _contract((x, legs, p), (x.conj().resolve_conj(), [_flip(l) for l in legs], p), ([0, 1], [0, 1]))
        return _flat(y, out, q)
    if kind == 'heff2':
        AA, FL, FR, W = [(_dense(f, legs), legs, _allowed(legs)) for legs, f in _heff2_inputs(case, seed)]
        W = (W[0].to(AA[0].dtype), *W[1:])
        tmp = _contract(AA, FR, ([3], [0]))
        tmp = _contract(W, tmp, ([2, 3], [3, 2]))
        tmp = _contract(W, tmp, ([2, 3], [0, 3]))
        return _flat(*_contract(FL, tmp, ([0, 1], [3, 0])))
    if kind == 'eigh':
        legs, flat = _density(case, seed)
        S, R = [], []
        for m in _each(flat, legs[0][2]):
            s, u = torch.linalg.eigh(m)
            S.append(s)
            R.append(((u * s.rsqrt()) @ u.conj().T).reshape(-1))
        # the eigenvalue tensor is sorted by the charge of its own leg, the negative of the row's
        return {'S': torch.cat(S[::-1]), 'rsqrt': torch.cat(R)}
    with torch.enable_grad():
        return {'svd': _exact_svd, 'qr': _exact_qr, 'corner': _exact_corner, 'proj': _exact_proj,
                'ctmrg': _exact_ctmrg}[kind](case, seed)
