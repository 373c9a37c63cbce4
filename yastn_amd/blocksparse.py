# Parts of this file restate the YASTN planner (yastn/tensor/_merging.py, _contractions.py, linalg.py) in
# the reference's statement order, because the metas it produces must be bit-identical to the reference's:
#   Copyright 2024 The YASTN Authors. All Rights Reserved.
#   Licensed under the Apache License, Version 2.0 (the "License"); you may not use this file except in
#   compliance with the License.  You may obtain a copy of the License at
#   https://www.apache.org/licenses/LICENSE-2.0
#   Unless required by applicable law or agreed to in writing, software distributed under the License is
#   distributed on an "AS IS" BASIS, WITHOUT WARRANTIES OR CONDITIONS OF ANY KIND, either express or
#   implied.  See the License for the specific language governing permissions and limitations under the
#   License.
"""Restated block-sparse planner and the tensor layer the workloads need (abelian U1 / U1xU1).

The backend never sees charges; it receives flat data buffers and integer meta tuples.  On a
machine without the reference package, this module produces those metas with the same block
order, offsets and fused-leg decompositions as the reference planner, so that the backend can be
driven through tensordot / fuse / unfuse / svd / truncation exactly as the reference drives it.
Golden vectors recorded from the reference pin every meta (tests/test_blocksparse.py).

Restated from (reference file: lines):
  data model            yastn/tensor/_auxiliary.py:26-50
  block creation order  yastn/tensor/_initialize.py:158-253
  merge to matrix       yastn/tensor/_merging.py:76-187 (+ no-change shortcuts 84-134)
  hard fusion           yastn/tensor/_merging.py:281-377, 488-549, 640-697
  tensordot             yastn/tensor/_contractions.py:57-346, 349-450 (no fusion), 453-528 (broadcast)
  masks                 yastn/tensor/_merging.py:554-583, _contractions.py:529-574
  svd / truncation      yastn/tensor/linalg.py:49-132, 135-380, 539-634 (multiplets), 637-735
  qr                    yastn/tensor/linalg.py:738-830
  eigh                  yastn/tensor/linalg.py:831-1010
Meta fusion (mfs), direct-sum fusion, leg-intersection masks and fermionic swap gates are not
restated: the workloads here do not use them.
"""
from __future__ import annotations

from functools import lru_cache
from itertools import accumulate, groupby, product
from numbers import Number
from operator import itemgetter
from typing import NamedTuple

import numpy as np


class BlockSparseError(Exception):
    """Structural error raised before the backend is called (the reference raises YastnError)."""


# ------------------------------------------------------------------ data model

# The planners below are cached by the structures of their operands.  Hashing the charges, sizes and slices of a few
# hundred blocks takes longer than anything else that a small contraction does on the host (75 of 160 us at 300 blocks),
# so Struct and Slices compute their hash once.
class _KeepHash:
    def __hash__(self):
        h = self.__dict__.get('_hash')
        if h is None:
            h = self.__dict__['_hash'] = tuple.__hash__(self)
        return h

    def __getstate__(self):  # pickles and copies carry the tuple alone
        return None


class _StructFields(NamedTuple):
    s: tuple = ()
    n: tuple = ()
    diag: bool = False
    t: tuple = ()
    D: tuple = ()
    size: int = 0


class Struct(_KeepHash, _StructFields):
    pass


class Slices(_KeepHash, tuple):
    """The Slc of every block, in the order of the blocks."""


class Slc(NamedTuple):
    slcs: tuple = ()
    D: tuple = ()
    Dp: int = 0


class Fusion(NamedTuple):
    tree: tuple = (1,)
    op: str = 'o'
    s: tuple = (1,)
    t: tuple = ()
    D: tuple = ()

    def conj(self):
        return self._replace(s=tuple(-x for x in self.s))


class _LegSlices(NamedTuple):
    t: tuple = ()
    D: tuple = ()
    dec: tuple = ()


class _Dec(NamedTuple):
    t: tuple = ()
    Dslc: tuple = (None, None)
    Dprod: int = 0
    Drsh: tuple = ()


class SymU1:
    SYM_ID = 'U1'
    NSYM = 1

    @classmethod
    def fuse(cls, charges, signatures, new_signature):
        return new_signature * np.einsum('kmn,m->kn', charges, np.asarray(signatures, dtype=np.int64))

    @classmethod
    def zero(cls):
        return (0,) * cls.NSYM

    @classmethod
    def add_charges(cls, *charges, signatures=None, new_signature=1):
        if not charges:
            return cls.zero()
        sg = (1,) * len(charges) if signatures is None else signatures
        c = np.array(charges, dtype=np.int64).reshape((1, len(charges), cls.NSYM))
        return tuple(cls.fuse(c, sg, new_signature).ravel().tolist())


class SymU1xU1(SymU1):
    SYM_ID = 'U1xU1'
    NSYM = 2


SYMS = {'U1': SymU1, 'U1xU1': SymU1xU1}


class Config(NamedTuple):
    backend: object = None
    sym: object = SymU1
    device: str = 'cpu'
    dtype: str = 'float64'
    tensordot_policy: str = 'fuse_contracted'


def make_config(backend, sym='U1', device='cpu', dtype='float64', tensordot_policy='fuse_contracted'):
    sym = SYMS[sym] if isinstance(sym, str) else sym
    return Config(backend=backend, sym=sym, device=device, dtype=dtype, tensordot_policy=tensordot_policy)


class Leg(NamedTuple):
    s: int
    t: tuple
    D: tuple

    def conj(self):
        return Leg(-self.s, self.t, self.D)


def leg(config, s, t, D):
    nsym = config.sym.NSYM
    t = tuple((x,) if isinstance(x, (int, np.integer)) else tuple(x) for x in t)
    t = tuple(tuple(int(y) for y in x) for x in t)
    if any(len(x) != nsym for x in t):
        raise BlockSparseError('charge length does not match the symmetry')
    return Leg(int(s), t, tuple(int(x) for x in D))


def _slices_of(Dps, Ds):
    return Slices(Slc(((stop - dp, stop),), ds, dp) for stop, dp, ds in zip(accumulate(Dps), Dps, Ds))


@lru_cache(maxsize=1024)
def _conj_struct(sym, struct):
    return struct._replace(s=tuple(-x for x in struct.s), n=sym.add_charges(struct.n, new_signature=-1))


# ------------------------------------------------------------------ tensor

class Tensor:
    """Block-sparse tensor: one flat data buffer of C-ordered blocks in ascending charge order."""

    def __init__(self, config, struct, slices, data, hfs=None, trans=None):
        self.config = config
        self.struct = struct
        self.slices = slices
        self._data = data
        self.hfs = tuple(hfs) if hfs is not None else tuple(Fusion(s=(x,)) for x in struct.s)
        self.trans = tuple(trans) if trans is not None else tuple(range(len(struct.s)))

    # -- bookkeeping
    def _replace(self, **kw):
        d = dict(config=self.config, struct=self.struct, slices=self.slices, data=self._data, hfs=self.hfs,
                 trans=self.trans)
        d.update(kw)
        return Tensor(**d)

    @property
    def data(self):
        return self._data

    @property
    def s(self):
        return tuple(self.struct.s[i] for i in self.trans)

    @property
    def n(self):
        return self.struct.n

    @property
    def isdiag(self):
        return self.struct.diag

    @property
    def ndim(self):
        return len(self.trans)

    @property
    def ndim_n(self):
        return len(self.struct.s)

    @property
    def size(self):
        return self.struct.size

    @property
    def yastn_dtype(self):
        return self.config.backend.get_yastn_dtype(self._data)

    def get_legs(self, axis):
        """Leg (s, t, D) of a native axis, from the existing blocks."""
        nsym = self.config.sym.NSYM
        ax = self.trans[axis]
        tD = {}
        for t, D in zip(self.struct.t, self.struct.D):
            tD[t[ax * nsym:(ax + 1) * nsym]] = D[ax]
        ks = sorted(tD)
        return Leg(self.struct.s[ax], tuple(ks), tuple(tD[k] for k in ks))

    def __repr__(self):
        return f"Tensor(s={self.s}, n={self.n}, blocks={len(self.struct.t)}, size={self.size})"

    # -- algebra
    def conj(self):
        return self._replace(struct=_conj_struct(self.config.sym, self.struct), hfs=tuple(h.conj() for h in self.hfs),
                             data=self.config.backend.conj(self._data))

    def transpose(self, axes):
        if sorted(axes) != list(range(self.ndim)):
            raise BlockSparseError('axes do not match tensor ndim')
        return self._replace(trans=tuple(self.trans[i] for i in axes))

    def moveaxis(self, source, destination):
        source = (source,) if isinstance(source, int) else tuple(source)
        destination = (destination,) if isinstance(destination, int) else tuple(destination)
        source = tuple(s % self.ndim for s in source)
        destination = tuple(d % self.ndim for d in destination)
        order = [n for n in range(self.ndim) if n not in source]
        for d, s in sorted(zip(destination, source)):
            order.insert(d, s)
        return self.transpose(tuple(order))

    def __matmul__(self, b):
        return tensordot(self, b, axes=(self.ndim - 1, 0))

    def __mul__(self, number):
        return self._replace(data=self._data * number)

    __rmul__ = __mul__

    def __truediv__(self, number):
        return self._replace(data=self._data / number)

    def __neg__(self):
        return self._replace(data=-self._data)

    def norm(self):
        return self.config.backend.norm(self._data, 'fro')

    def to_number(self):
        """Value of a rank-0 tensor (or the first element)."""
        if self.size == 0:
            return self.config.backend.zeros((), dtype='float64', device=self.config.device)
        return self._data.reshape(-1)[0]

    def rsqrt(self, cutoff=0):
        if not self.isdiag:
            raise BlockSparseError('rsqrt is defined for diagonal tensors')
        return self._replace(data=self.config.backend.rsqrt(self._data, cutoff=cutoff))

    def sqrt(self):
        return self._replace(data=self.config.backend.sqrt(self._data))

    def consume_transpose(self):
        return consume_transpose(self)

    def fuse_legs(self, axes, mode='hard'):
        return fuse_legs(self, axes)

    def unfuse_legs(self, axes):
        return unfuse_legs(self, axes)

    def svd_with_truncation(self, axes=(0, 1), **kw):
        return svd_with_truncation(self, axes=axes, **kw)

    def svd(self, axes=(0, 1), **kw):
        return svd(self, axes=axes, **kw)

    def to_dict(self, level=2):
        """Everything needed to rebuild the tensor (the fields of the reference's Tensor.to_dict,
        tensor/_output.py:35-110): at level 0 the structure objects as they are, at level >= 1 as basic
        Python data, at level 2 also the data as a numpy array."""
        nd = len(self.struct.s)
        if level >= 1:
            config = self.config._asdict()
            config['sym'] = self.config.sym.SYM_ID
            config['backend'] = getattr(self.config.backend, 'BACKEND_ID', None)
            struct = self.struct._asdict()
            slices = [tuple(x) for x in self.slices]
            hfs = tuple(h._asdict() for h in self.hfs)
        else:
            config, struct, slices, hfs = self.config, self.struct, self.slices, self.hfs
        data = self._data if level < 2 else self.config.backend.to_numpy(self._data)
        return {'type': 'Tensor', 'dict_ver': 2, 'level': level, 'config': config, 'data': data,
                'struct': struct, 'slices': slices, 'trans': self.trans, 'isdiag': self.isdiag, 'hfs': hfs,
                'mfs': ((1,),) * nd}

    @staticmethod
    def from_dict(d, config=None):
        """Inverse of to_dict (reference tensor/_initialize.py from_dict); a level >= 1 dictionary needs the
        config (its backend and symmetry) or takes the configuration's names from a passed config."""
        if d.get('level', 0) >= 1 or isinstance(d['struct'], dict):
            if config is None:
                raise BlockSparseError('from_dict of a level >= 1 dictionary needs a config')
            tup = lambda x: tuple(tup(y) for y in x) if isinstance(x, (list, tuple)) else x
            sd = d['struct']
            struct = Struct(s=tup(sd['s']), n=tup(sd['n']), diag=bool(sd['diag']), t=tup(sd['t']), D=tup(sd['D']),
                            size=int(sd['size']))
            slices = Slices(Slc(tup(x[0]), tup(x[1]), int(x[2])) for x in d['slices'])
            hfs = tuple(Fusion(**{k: (tup(v) if k != 'op' else v) for k, v in h.items()}) for h in d['hfs'])
            data = d['data']
            if isinstance(data, np.ndarray):
                dtype = 'complex128' if np.iscomplexobj(data) else ('bool' if data.dtype == np.bool_ else 'float64')
                data = config.backend.to_tensor(data, dtype=dtype, device=config.device)
            return Tensor(config, struct, slices, data, hfs=hfs, trans=tup(d['trans']))
        return Tensor(config or d['config'], d['struct'], d['slices'], d['data'], hfs=d['hfs'], trans=d['trans'])

    def to_dense(self):
        """Dense numpy array (legs in logical order, sectors in ascending charge)."""
        a = consume_transpose(self)
        nsym = a.config.sym.NSYM
        data = a.config.backend.to_numpy(a._data)
        legs = [a.get_legs(i) for i in range(a.ndim)]
        offs = [dict(zip(l.t, accumulate((0,) + l.D))) for l in legs]
        out = np.zeros(tuple(sum(l.D) for l in legs), dtype=data.dtype)
        for t, D, sl in zip(a.struct.t, a.struct.D, a.slices):
            if a.isdiag:
                continue
            idx = tuple(slice(offs[i][t[i * nsym:(i + 1) * nsym]], offs[i][t[i * nsym:(i + 1) * nsym]] + D[i])
                        for i in range(len(D)))
            out[idx] = data[sl.slcs[0][0]:sl.slcs[0][1]].reshape(D)
        return out


def _fill_struct(config, legs, n, isdiag=False):
    """All blocks allowed by the selection rule, sorted by charges (reference _initialize.py:158-253)."""
    sym, nsym = config.sym, config.sym.NSYM
    s = tuple(l.s for l in legs)
    n = sym.zero() if n is None else ((n,) if isinstance(n, (int, np.integer)) else tuple(n))
    combos_t = list(product(*(l.t for l in legs)))
    combos_D = list(product(*(l.D for l in legs)))
    if combos_t:
        ct = np.array(combos_t, dtype=np.int64).reshape(len(combos_t), len(legs), nsym)
        ok = np.all(sym.fuse(ct, s, 1) == np.array(n, dtype=np.int64), axis=1)
    else:
        ok = np.zeros(0, dtype=bool)
    meta = []
    for keep, t, D in zip(ok, combos_t, combos_D):
        if keep and all(d > 0 for d in D):
            meta.append((tuple(x for tt in t for x in tt), tuple(D)))
    meta.sort(key=itemgetter(0))
    ts = tuple(m[0] for m in meta)
    Ds = tuple(m[1] for m in meta)
    Dps = tuple(int(np.prod(D)) for D in Ds)
    if isdiag:
        Dps = tuple(D[0] for D in Ds)
    struct = Struct(s=s, n=tuple(n), diag=isdiag, t=ts, D=Ds, size=sum(Dps))
    return struct, _slices_of(Dps, Ds)


def zeros(config, legs, n=None, dtype=None):
    struct, slices = _fill_struct(config, legs, n)
    data = config.backend.zeros((struct.size,), dtype=dtype or config.dtype, device=config.device)
    return Tensor(config, struct, slices, data)


def from_flat(config, legs, n, flat):
    """Tensor whose block buffer (in the reference's block order) is ``flat`` (numpy or backend array)."""
    struct, slices = _fill_struct(config, legs, n)
    if len(flat) != struct.size:
        raise BlockSparseError(f"data has {len(flat)} elements, structure needs {struct.size}")
    if isinstance(flat, np.ndarray):
        dtype = 'complex128' if np.iscomplexobj(flat) else 'float64'
        flat = config.backend.to_tensor(flat, dtype=dtype, device=config.device)
    return Tensor(config, struct, slices, flat)


def from_blocks(config, s, n, t, D, flat, isdiag=False):
    """Tensor with the listed blocks (charges t, shapes D, in ascending charge order) and the block buffer
    ``flat`` (the layout of the reference's Tensor.from_dict, tensor/_output.py)."""
    t = tuple(tuple(x) for x in t)
    D = tuple(tuple(x) for x in D)
    if list(t) != sorted(set(t)):
        raise BlockSparseError('block charges must be unique and in ascending order')
    Dps = tuple(d[0] if isdiag else int(np.prod(d)) for d in D)
    struct = Struct(s=tuple(s), n=tuple(n), diag=isdiag, t=t, D=D, size=sum(Dps))
    if len(flat) != struct.size:
        raise BlockSparseError(f"data has {len(flat)} elements, structure needs {struct.size}")
    if isinstance(flat, np.ndarray):
        dtype = 'complex128' if np.iscomplexobj(flat) else ('bool' if flat.dtype == np.bool_ else 'float64')
        flat = config.backend.to_tensor(flat, dtype=dtype, device=config.device)
    return Tensor(config, struct, _slices_of(Dps, D), flat)


def split_data_and_meta(d, squeeze=False):
    """(data, meta) of a to_dict dictionary (the reference's yastn/_split_combine_dict.py:21-45): every
    'data' entry, visited in sorted key order through nested dictionaries, goes to the data tuple and is
    replaced in the meta copy by its position.  With ``squeeze``, a single data array is not wrapped."""
    data = []

    def walk(x):
        out = {}
        for k in sorted(x):
            if k == 'data':
                data.append(x[k])
                out[k] = len(data) - 1
            elif isinstance(x[k], dict):
                out[k] = walk(x[k])
            else:
                out[k] = x[k]
        return out
    meta = walk(d)
    return (data[0] if squeeze and len(data) == 1 else tuple(data)), meta


def combine_data_and_meta(data, meta):
    """Inverse of split_data_and_meta (reference _split_combine_dict.py:57-70)."""
    if not isinstance(data, (list, tuple)):
        data = [data]
    out = {}
    for k in sorted(meta):
        if k == 'data':
            out[k] = data[meta[k]]
        elif isinstance(meta[k], dict):
            out[k] = combine_data_and_meta(data, meta[k])
        else:
            out[k] = meta[k]
    return out


def seeded_normal(n, dtype, seed):
    """Block entries N(0,1) from np.random.default_rng(seed) over the flat buffer (complex: independent
    real and imaginary parts)."""
    rng = np.random.default_rng(seed)
    if dtype == 'complex128':
        re = rng.standard_normal(n)
        return re + 1j * rng.standard_normal(n)
    return rng.standard_normal(n)


def rand(config, legs, n=None, dtype='float64', seed=0, scale=1.0):
    struct, slices = _fill_struct(config, legs, n)
    return from_flat(config, legs, n, seeded_normal(struct.size, dtype, seed) * scale)


# ------------------------------------------------------------------ leg structures

def _leg_structure_merge(teff, tlegs, Deff, Dlegs):
    """Decomposition of a merged leg: effective charges sorted, sub-charges sorted within
    (reference _merging.py:681-694)."""
    rows = sorted(set(zip(teff, tlegs, Deff, Dlegs)))
    t, D, dec = [], [], []
    for te, grp in groupby(rows, key=itemgetter(0)):
        lo, recs = 0, []
        for _, tl, De, Dl in grp:
            recs.append(_Dec(tl, (lo, lo + De), De, Dl))
            lo += De
        t.append(te)
        D.append(lo)
        dec.append(tuple(recs))
    return _LegSlices(tuple(t), tuple(D), tuple(dec))


@lru_cache(maxsize=1024)
def _leg_structure_combine_charges_prod(sym, t_in, D_in, s_in, t_out, s_out):
    ct = list(product(*t_in))
    cD = list(product(*D_in))
    ct = np.array(ct, dtype=np.int64).reshape((len(ct), len(s_in), sym.NSYM))
    cD = np.array(cD, dtype=np.int64).reshape((len(cD), len(s_in)))
    teff = sym.fuse(ct, s_in, s_out)
    keep = np.array([i for i, te in enumerate(teff.tolist()) if tuple(te) in t_out], dtype=np.int64)
    cD, ct, teff = cD[keep], ct[keep], teff[keep]
    Deff = tuple(np.prod(cD, axis=1, dtype=np.int64).tolist())
    Dlegs = tuple(map(tuple, cD.tolist()))
    teff = tuple(map(tuple, teff.tolist()))
    tlegs = tuple(map(tuple, ct.reshape(len(ct), len(s_in) * sym.NSYM).tolist()))
    return _leg_structure_merge(teff, tlegs, Deff, Dlegs)


def _get_tD_legs(struct):
    lt, nd, nsym = len(struct.t), len(struct.s), len(struct.n)
    ts = np.array(struct.t, dtype=np.int64).reshape(lt, nd, nsym)
    Ds = np.array(struct.D, dtype=np.int64).reshape(lt, nd)
    legs = [sorted(set((tuple(t), D) for t, D in zip(ts[:, n, :].tolist(), Ds[:, n].tolist()))) for n in range(nd)]
    dicts = [dict(x) for x in legs]
    if any(len(a) != len(b) for a, b in zip(legs, dicts)):
        raise BlockSparseError('Bond dimensions related to some charge are not consistent.')
    return [tuple(d.keys()) for d in dicts], [tuple(d.values()) for d in dicts], dicts


@lru_cache(maxsize=1024)
def _leg_struct_trivial(struct, axis=0):
    nsym = len(struct.n)
    tD = sorted((tt[nsym * axis: nsym * (axis + 1)], DD[axis]) for tt, DD in zip(struct.t, struct.D))
    t = tuple(x[0] for x in tD)
    D = tuple(x[1] for x in tD)
    return _LegSlices(t, D, tuple((_Dec(tt, (0, DD), DD, (DD,)),) for tt, DD in zip(t, D)))


# ------------------------------------------------------------------ merge to matrix / fuse / unmerge

@lru_cache(maxsize=1024)
def _meta_merge_to_matrix(config, struct, slices, axes, inds):
    """reference _merging.py:137-187."""
    sym, nsym = config.sym, config.sym.NSYM
    s_eff = (struct.s[axes[0][0]] if axes[0] else 1, struct.s[axes[1][0]] if axes[1] else -1)
    t_old = struct.t if inds is None else [struct.t[i] for i in inds]
    D_old = struct.D if inds is None else [struct.D[i] for i in inds]
    sl_old = slices if inds is None else [slices[i] for i in inds]
    tset = np.array(t_old, dtype=np.int64).reshape((len(t_old), len(struct.s), nsym))
    Dset = np.array(D_old, dtype=np.int64).reshape((len(D_old), len(struct.s)))
    t, teff, ls = [], [], []
    for side in (0, 1):
        ta = tset[:, axes[side], :]
        Da = Dset[:, axes[side]]
        Deff = np.prod(Da, axis=1, dtype=np.int64).tolist()
        Da = [tuple(x) for x in Da.tolist()]
        s = tuple(struct.s[i] for i in axes[side])
        te = [tuple(x) for x in sym.fuse(ta, s, s_eff[side]).tolist()]
        ta = [tuple(x) for x in ta.reshape(len(ta), len(s) * nsym).tolist()]
        teff.append(te)
        t.append(ta)
        ls.append(_leg_structure_merge(te, ta, Deff, Da))
    rows = sorted((tl, tr, xl, xr, slo.slcs[0], Do) for tl, tr, xl, xr, slo, Do
                  in zip(teff[0], teff[1], t[0], t[1], sl_old, D_old))
    meta_mrg, t_new, D_new, sl_new, lo = [], [], [], [], 0
    for (tel, ter), grp in groupby(rows, key=itemgetter(0, 1)):
        i0, i1 = ls[0].t.index(tel), ls[1].t.index(ter)
        tn = tel + ter
        D0, D1 = ls[0].D[i0], ls[1].D[i1]
        t_new.append(tn)
        D_new.append((D0, D1))
        sl_new.append(Slc(((lo, lo + D0 * D1),), (D0, D1), D0 * D1))
        lo += D0 * D1
        grp = list(grp)
        k = 0
        for d0, d1 in product(ls[0].dec[i0], ls[1].dec[i1]):
            if k < len(grp) and d0.t == grp[k][2] and d1.t == grp[k][3]:
                meta_mrg.append((tn, grp[k][4], grp[k][5], (d0.Dslc, d1.Dslc), (d0.Dprod, d1.Dprod)))
                k += 1
    struct_new = struct._replace(t=tuple(t_new), D=tuple(D_new), s=s_eff, size=lo)
    return struct_new, Slices(sl_new), tuple(meta_mrg), ls[0], ls[1]


def _no_change_in_transpose_and_merge(meta_mrg, meta_new, Dsize):
    """reference _merging.py:92-111 (C-order layouts that coincide need no copy)."""
    if Dsize in (0, 1):
        return True
    lo = 0
    for _, slo, _, _, _ in meta_mrg:
        if slo[0] != lo:
            return False
        lo = slo[1]
    if lo != Dsize:
        return False
    for (_, Dn, _), (_, grp) in zip(meta_new, groupby(meta_mrg, key=itemgetter(0))):
        lo = 0
        for _, _, _, Dslc, _ in grp:
            if Dslc[0][0] != lo:
                return False
            lo = Dslc[0][1]
        if lo != Dn[0]:
            return False
    return True


def _transpose_and_merge(config, data, order, struct, slices, meta_mrg, inds=None):
    args = _merge_args(order, struct, slices, meta_mrg, inds, config.backend.get_size(data))
    return data if args is None else config.backend.transpose_and_merge(data, *args)


def _merge_args(order, struct, slices, meta_mrg, inds, size):
    """The arguments of the backend's transpose_and_merge after the data (of ``size`` elements), or None where the data
    is already in place."""
    meta_new = tuple((x, y, z.slcs[0]) for x, y, z in zip(struct.t, struct.D, slices))
    if inds is None and tuple(range(len(order))) == tuple(order) and struct.size == size \
            and _no_change_in_transpose_and_merge(meta_mrg, meta_new, struct.size):
        return None
    return order, meta_new, meta_mrg, struct.size


def _transpose_and_merge_pair(config, data_a, args_a, data_b, args_b):
    """transpose_and_merge of two operands (args: _merge_args); one backend call for both when both need a merge and the
    backend fuses such pairs (transpose_and_merge_pair)."""
    backend = config.backend
    if args_a is not None and args_b is not None:
        pair = getattr(backend, 'transpose_and_merge_pair', None)
        if pair is not None:
            return pair(data_a, *args_a, data_b, *args_b)
    return (data_a if args_a is None else backend.transpose_and_merge(data_a, *args_a),
            data_b if args_b is None else backend.transpose_and_merge(data_b, *args_b))


def _merge_to_matrix(a, axes, inds=None):
    order = axes[0] + axes[1]
    struct, slices, meta_mrg, ls_l, ls_r = _meta_merge_to_matrix(a.config, a.struct, a.slices, axes, inds)
    data = _transpose_and_merge(a.config, a._data, order, struct, slices, meta_mrg, inds)
    return data, struct, slices, ls_l, ls_r


def _no_change_in_unmerge(meta):
    """reference _merging.py:122-134."""
    low, Dn_last, sl_last, sln = 0, 0, (0, 0), (0, 0)
    for sln, Dn, slo, _, sub in meta:
        if slo != sl_last:
            if slo[0] != sl_last[1] or low != Dn_last:
                return False
            sl_last, Dn_last, low = slo, Dn[0], 0
        if low != sub[0][0]:
            return False
        low = sub[0][1]
    return sl_last[1] == sln[1]


def _unmerge(config, data, meta):
    Dsize = meta[-1][0][1] if meta else 0
    if config.backend.get_size(data) != Dsize:
        raise BlockSparseError('unmerge size mismatch')
    if _no_change_in_unmerge(meta):
        return data
    return config.backend.unmerge(data, meta)


@lru_cache(maxsize=1024)
def _meta_unmerge_matrix(config, struct, slices, ls0, ls1, snew):
    """reference _merging.py:528-549."""
    nsym = config.sym.NSYM
    rows = []
    for to, slo, Do in zip(struct.t, slices, struct.D):
        i0, i1 = ls0.t.index(to[:nsym]), ls1.t.index(to[nsym:])
        for d0, d1 in product(ls0.dec[i0], ls1.dec[i1]):
            rows.append((d0.t + d1.t, d0.Drsh + d1.Drsh, d0.Dprod * d1.Dprod, (d0.Dprod, d1.Dprod), slo.slcs[0], Do,
                         (d0.Dslc, d1.Dslc)))
    rows.sort(key=itemgetter(0))
    tnew = tuple(r[0] for r in rows)
    Dnew = tuple(r[1] for r in rows)
    Dp = tuple(r[2] for r in rows)
    struct_new = struct._replace(s=tuple(snew), t=tnew, D=Dnew, size=sum(Dp))
    sl_new = _slices_of(Dp, Dnew)
    meta = tuple((x.slcs[0], *r[3:]) for x, r in zip(sl_new, rows))
    return meta, struct_new, sl_new


@lru_cache(maxsize=1024)
def _meta_fuse_hard(config, struct, slices, axes, inds):
    """reference _merging.py:304-377."""
    sym, nsym = config.sym, config.sym.NSYM
    if inds is None:
        t_old, D_old, sl_old = struct.t, struct.D, slices
    else:
        t_old = tuple(struct.t[i] for i in inds)
        D_old = tuple(struct.D[i] for i in inds)
        sl_old = [slices[i] for i in inds]
        struct = struct._replace(t=t_old, D=D_old)
    lt, nd = len(t_old), len(struct.s)
    t_in, D_in, tD_dict = _get_tD_legs(struct)
    slegs = tuple(tuple(struct.s[n] for n in ax) for ax in axes)
    s_eff = [struct.s[ax[0]] if ax else -1 for ax in axes]
    if axes and not axes[0]:
        s_eff[0] = 1
    s_eff = tuple(s_eff)
    tset = np.array(t_old, dtype=np.int64).reshape(lt, nd, nsym)
    teff = np.zeros((lt, len(s_eff), nsym), dtype=np.int64)
    for n, ax in enumerate(axes):
        teff[:, n, :] = sym.fuse(tset[:, ax, :], slegs[n], s_eff[n]) if ax else sym.zero()
    lls = []
    for n, ax in enumerate(axes):
        if len(ax) > 1:
            tset_n = tuple(set(map(tuple, teff[:, n, :].tolist())))
            lls.append(_leg_structure_combine_charges_prod(sym, tuple(t_in[i] for i in ax), tuple(D_in[i] for i in ax),
                                                           slegs[n], tset_n, s_eff[n]))
        elif len(ax) == 1:
            t = tuple(tD_dict[ax[0]].keys())
            D = tuple(tD_dict[ax[0]].values())
            lls.append(_LegSlices(t, D, tuple((_Dec(tt, (0, DD), DD, (DD,)),) for tt, DD in zip(t, D))))
        else:
            lls.append(_LegSlices((sym.zero(),), (1,), ((_Dec((), (0, 1), 1, (1,)),),)))
    teff_split = [tuple(map(tuple, x)) for x in teff.tolist()]
    if axes:
        told = list(zip(*[tset[:, ax, :].reshape(lt, len(ax) * nsym).tolist() for ax in axes]))
        told = [tuple(map(tuple, x)) for x in told]
    else:
        told = list(t_old)
    teff_flat = list(map(tuple, teff.reshape(lt, len(axes) * nsym).tolist()))
    rows = sorted((tes, tn, tos, slo.slcs[0], Do) for tes, tn, tos, slo, Do
                  in zip(teff_split, teff_flat, told, sl_old, D_old))
    meta_mrg, t_new, D_new = [], [], []
    for (tes, tn), grp in groupby(rows, key=itemgetter(0, 1)):
        idx = tuple(ls.t.index(te) for ls, te in zip(lls, tes))
        decs = tuple(ls.dec[i] for ls, i in zip(lls, idx))
        t_new.append(tn)
        D_new.append(tuple(ls.D[i] for ls, i in zip(lls, idx)))
        grp = list(grp)
        k = 0
        for de in product(*decs):
            if k < len(grp) and tuple(d.t for d in de) == grp[k][2]:
                meta_mrg.append((tn, grp[k][3], grp[k][4], tuple(d.Dslc for d in de), tuple(d.Dprod for d in de)))
                k += 1
    Dp = np.prod(D_new, axis=1, dtype=np.int64).tolist() if D_new else []
    struct_new = struct._replace(t=tuple(t_new), D=tuple(D_new), s=s_eff, size=sum(Dp))
    return struct_new, _slices_of(Dp, D_new), meta_mrg, t_in, D_in


def _combine_hfs_prod(hfs, t_in, D_in, s_out, axes):
    """reference _merging.py:697-712."""
    tfl, Dfl, sfl, op = [], [], [s_out], 'p'
    tree = [sum(hfs[n].tree[0] for n in axes)]
    for n in axes:
        tfl.append(t_in[n])
        tfl.extend(hfs[n].t)
        Dfl.append(D_in[n])
        Dfl.extend(hfs[n].D)
        sfl.extend(hfs[n].s)
        tree.extend(hfs[n].tree)
        op += hfs[n].op
    return Fusion(tree=tuple(tree), op=op, s=tuple(sfl), t=tuple(tfl), D=tuple(Dfl))


def _unfuse_fusion(hf):
    """One layer of an unfuse (reference _merging.py:981-997)."""
    tt, DD, ss, hfs = [], [], [], []
    first, cum = 1, 0
    for n in range(1, len(hf.tree)):
        if cum == 0:
            cum = hf.tree[n]
        if hf.tree[n] == 1:
            cum -= 1
            if cum == 0:
                tt.append(hf.t[first - 1])
                DD.append(hf.D[first - 1])
                ss.append(hf.s[first])
                hfs.append(Fusion(tree=hf.tree[first:n + 1], op=hf.op[first:n + 1], s=hf.s[first:n + 1],
                                  t=hf.t[first:n], D=hf.D[first:n]))
                first = n + 1
    return tuple(tt), tuple(DD), tuple(ss), hfs


def fuse_legs(a, axes):
    """Hard fusion of groups of legs; e.g. axes=(0, (1, 2), 3) (reference _merging.py:202-301)."""
    if a.isdiag:
        raise BlockSparseError('Cannot fuse legs of a diagonal tensor.')
    axes = tuple((x,) if isinstance(x, int) else tuple(x) for x in axes)
    order = tuple(x for g in axes for x in g)
    if sorted(order) != list(range(a.ndim)):
        raise BlockSparseError('Provided axes do not match tensor ndim.')
    order = tuple(a.trans[ax] for ax in order)
    axes = tuple(tuple(a.trans[ax] for ax in g) for g in axes)
    struct, slices, meta_mrg, t_in, D_in = _meta_fuse_hard(a.config, a.struct, a.slices, axes, None)
    data = _transpose_and_merge(a.config, a._data, order, struct, slices, meta_mrg)
    hfs = []
    for n, g in enumerate(axes):
        if len(g) > 1:
            hfs.append(_combine_hfs_prod(a.hfs, t_in, D_in, struct.s[n], g))
        else:
            hfs.append(a.hfs[g[0]])
    return Tensor(a.config, struct, slices, data, hfs=hfs, trans=None)


@lru_cache(maxsize=1024)
def _meta_unfuse_hard(config, struct, slices, axes, hfs):
    """reference _merging.py:488-525."""
    sym, nsym = config.sym, config.sym.NSYM
    t_in, _, tD_dict = _get_tD_legs(struct)
    lls, hfs_new, snew, nlegs = [], [], [], []
    for n, hf in enumerate(hfs):
        if n in axes:
            t_part, D_part, s_part, hfs_part = _unfuse_fusion(hf)
            lls.append(_leg_structure_combine_charges_prod(sym, t_part, D_part, s_part, t_in[n], struct.s[n]))
            hfs_new.extend(hfs_part)
            nlegs.append(len(hfs_part))
            snew.extend(s_part)
        else:
            t, D = tuple(tD_dict[n].keys()), tuple(tD_dict[n].values())
            lls.append(_LegSlices(t, D, tuple((_Dec(tt, (0, DD), DD, (DD,)),) for tt, DD in zip(t, D))))
            hfs_new.append(hf)
            snew.append(struct.s[n])
    rows = []
    for to, slo, Do in zip(struct.t, slices, struct.D):
        idx = tuple(ls.t.index(to[n * nsym:(n + 1) * nsym]) for n, ls in enumerate(lls))
        for tt in product(*(ls.dec[i] for ls, i in zip(lls, idx))):
            rows.append((sum((x.t for x in tt), ()), sum((x.Drsh for x in tt), ()), tuple(x.Dprod for x in tt),
                         slo.slcs[0], Do, tuple(x.Dslc for x in tt)))
    rows.sort(key=itemgetter(0))
    tnew = tuple(r[0] for r in rows)
    Dnew = tuple(r[1] for r in rows)
    Dp = np.prod(np.array(Dnew, dtype=np.int64).reshape(len(Dnew), len(snew)), axis=1, dtype=np.int64).tolist()
    struct_new = struct._replace(s=tuple(snew), t=tnew, D=Dnew, size=sum(Dp))
    sl_new = _slices_of(Dp, Dnew)
    meta = tuple((x.slcs[0], *r[2:]) for x, r in zip(sl_new, rows))
    return meta, struct_new, sl_new, tuple(nlegs), tuple(hfs_new)


def unfuse_legs(a, axes):
    """Revert one layer of hard fusion of the given (logical) legs (reference _merging.py:380-485)."""
    axes = (axes,) if isinstance(axes, int) else tuple(axes)
    if a.isdiag:
        raise BlockSparseError('Cannot unfuse legs of a diagonal tensor.')
    haxes, uaxes = [], []
    for mi in range(a.ndim):
        hi = a.trans[mi]
        if mi in axes and a.hfs[hi].tree[0] > 1:
            if a.hfs[hi].op[0] != 'p':
                raise BlockSparseError('only product fusions can be unfused here')
            haxes.append(hi)
            uaxes.append(mi)
    if not haxes:
        return a
    meta, struct, slices, nlegs, hfs = _meta_unfuse_hard(a.config, a.struct, a.slices, tuple(haxes), tuple(a.hfs))
    data = _unmerge(a.config, a._data, meta)
    trans = list(a.trans)
    for unfused, n in zip(nlegs[::-1], uaxes[::-1]):
        trans = trans[:n] + [trans[n]] * unfused + trans[n + 1:]
    for ax in range(max(trans), -1, -1):
        newax = sum(i < ax for i in trans)
        ii = trans.index(ax)
        while ii < len(trans) and trans[ii] == ax:
            trans[ii] = newax
            newax += 1
            ii += 1
    return Tensor(a.config, struct, slices, data, hfs=hfs, trans=trans)


def consume_transpose(a):
    """Apply a pending logical transpose to the data (reference _single.py:316-346)."""
    if a.trans == tuple(range(a.ndim_n)):
        return a
    order = np.array(a.trans, dtype=np.int64)
    lt, nd, nsym = len(a.struct.t), len(a.struct.s), len(a.struct.n)
    ts = np.array(a.struct.t, dtype=np.int64).reshape(lt, nd, nsym)
    Ds = np.array(a.struct.D, dtype=np.int64).reshape(lt, nd)
    newt = tuple(map(tuple, ts[:, order, :].reshape(lt, nd * nsym).tolist()))
    newD = tuple(map(tuple, Ds[:, order].tolist()))
    rows = sorted(zip(newt, newD, a.slices), key=itemgetter(0))
    Dp = tuple(r[2].Dp for r in rows)
    slices = _slices_of(Dp, tuple(r[1] for r in rows))
    struct = a.struct._replace(s=tuple(a.struct.s[i] for i in a.trans), t=tuple(r[0] for r in rows),
                               D=tuple(r[1] for r in rows))
    meta = tuple((sn.slcs[0], sn.D, r[2].slcs[0], r[2].D) for sn, r in zip(slices, rows))
    data = a._data if a.isdiag else a.config.backend.transpose(a._data, a.trans, meta)
    return Tensor(a.config, struct, slices, data, hfs=tuple(a.hfs[i] for i in a.trans), trans=None)


# ------------------------------------------------------------------ tensordot

def _common_inds(t_a, t_b, nin_a, nin_b, ndim_a, ndim_b, nsym):
    """reference _contractions.py:250-278."""
    ta = np.array(t_a, dtype=np.int64).reshape((len(t_a), ndim_a, nsym))
    tb = np.array(t_b, dtype=np.int64).reshape((len(t_b), ndim_b, nsym))
    la = [tuple(x) for x in ta[:, nin_a, :].reshape(len(ta), len(nin_a) * nsym).tolist()]
    lb = [tuple(x) for x in tb[:, nin_b, :].reshape(len(tb), len(nin_b) * nsym).tolist()]
    sa, sb = set(la), set(lb)
    ia = tuple(i for i, x in enumerate(la) if x in sb)
    ib = tuple(i for i, x in enumerate(lb) if x in sa)
    return (None if len(ia) == len(la) else ia), (None if len(ib) == len(lb) else ib)


def _meta_tensordot_f2m(struct_a, slices_a, struct_b, slices_b):
    """reference _contractions.py:281-298."""
    nsym = len(struct_a.n)
    ra = sorted((t[nsym:], t, D, sl.slcs[0]) for t, D, sl in zip(struct_a.t, struct_a.D, slices_a))
    rb = [(t[:nsym], t, D, sl.slcs[0]) for t, D, sl in zip(struct_b.t, struct_b.D, slices_b)]
    rows = []
    for (tar, ta, Da, sla), (tbl, tb, Db, slb) in zip(ra, rb):
        if tar != tbl:
            raise BlockSparseError('block charges of the contracted legs do not pair up')
        rows.append((ta[:nsym] + tb[nsym:], (Da[0], Db[1]), sla, Da, slb, Db))
    rows.sort()
    t_c = tuple(r[0] for r in rows)
    D_c = tuple(r[1] for r in rows)
    Dp = tuple(D[0] * D[1] for D in D_c)
    slices_c = _slices_of(Dp, D_c)
    meta = tuple((sl.slcs[0], *r[1:]) for sl, r in zip(slices_c, rows))
    return meta, Struct(s=(struct_a.s[0], struct_b.s[1]), t=t_c, D=D_c, size=sum(Dp)), slices_c


def _meta_tensordot_fc(struct_a, slices_a, struct_b, slices_b):
    """reference _contractions.py:301-346."""
    nsym = len(struct_a.n)
    lta, nda = len(struct_a.t), len(struct_a.s)
    ta = np.array(struct_a.t, dtype=np.int64).reshape((lta, nda, nsym))
    Da = np.array(struct_a.D, dtype=np.int64).reshape((lta, nda))
    ra = sorted((tuple(tc), tuple(to), Dc, Dop, tuple(Do), sl.slcs[0]) for tc, to, Dc, Dop, Do, sl in zip(
        ta[:, -1, :].tolist(), ta[:, :-1, :].reshape(lta, (nda - 1) * nsym).tolist(), Da[:, -1].tolist(),
        np.prod(Da[:, :-1], axis=1, dtype=np.int64).tolist(), Da[:, :-1].tolist(), slices_a))
    ltb, ndb = len(struct_b.t), len(struct_b.s)
    tb = np.array(struct_b.t, dtype=np.int64).reshape((ltb, ndb, nsym))
    Db = np.array(struct_b.D, dtype=np.int64).reshape((ltb, ndb))
    rb = [(tuple(tc), tuple(to), Dc, Dop, tuple(Do), sl.slcs[0]) for tc, to, Dc, Dop, Do, sl in zip(
        tb[:, 0, :].tolist(), tb[:, 1:, :].reshape(ltb, (ndb - 1) * nsym).tolist(), Db[:, 0].tolist(),
        np.prod(Db[:, 1:], axis=1, dtype=np.int64).tolist(), Db[:, 1:].tolist(), slices_b)]
    rows = []
    for (tar, ga), (tbl, gb) in zip(groupby(ra, key=itemgetter(0)), groupby(rb, key=itemgetter(0))):
        if tar != tbl:
            raise BlockSparseError('block charges of the contracted legs do not pair up')
        for (_, toa, Dca, Dopa, Doa, sla), (_, tob, Dcb, Dopb, Dob, slb) in product(list(ga), list(gb)):
            rows.append((toa + tob, Doa + Dob, Dopa * Dopb, (Dopa, Dopb), sla, (Dopa, Dca), slb, (Dcb, Dopb)))
    rows.sort()
    t_c = tuple(r[0] for r in rows)
    D_c = tuple(r[1] for r in rows)
    Dp = tuple(r[2] for r in rows)
    slices_c = _slices_of(Dp, D_c)
    meta = tuple((sl.slcs[0], *r[3:]) for sl, r in zip(slices_c, rows))
    return meta, Struct(s=struct_a.s[:-1] + struct_b.s[1:], t=t_c, D=D_c, size=sum(Dp)), slices_c


def _meta_tensordot_nf(struct_a, slices_a, struct_b, slices_b, ind_a, ind_b, nout_a, nin_a, nin_b, nout_b):
    """No-fusion policy (reference _contractions.py:349-450).  Returns (meta_dot, reshape_a, reshape_b,
    struct_c, slices_c): reshape_* = (slice, block shape, rows, cols) of each participating block as the
    matrix its permutation gives; meta_dot lists per output block (slice, (rows, cols), [[ia, ib], ...]),
    the block products to sum.  The output blocks come in ascending charge order; the products of a
    block keep the order that the reference's (unstable) argsorts give them, which is reproduced by
    running the same numpy sorts on the same arrays, so summation order and metas are identical."""
    nsym = len(struct_a.n)

    def side(struct, slices, ind, nout, nin):
        sel = range(len(struct.t)) if ind is None else ind
        t = [struct.t[i] for i in sel]
        D = [struct.D[i] for i in sel]
        sl = [slices[i].slcs[0] for i in sel]
        nb, nd = len(t), len(struct.s)
        at = np.array(t, dtype=np.int64).reshape((nb, nd, nsym))
        aD = np.array(D, dtype=np.int64).reshape((nb, nd))
        t_out = at[:, nout, :].reshape(nb, len(nout) * nsym)
        t_in = at[:, nin, :].reshape(nb, len(nin) * nsym)
        D_out, D_in = aD[:, nout], aD[:, nin]
        sectors, inv, cnt = np.unique(np.hstack([t_in, D_in]), return_inverse=True, return_counts=True, axis=0)
        return dict(t=t, D=D, sl=sl, t_out=t_out, D_out=D_out,
                    Dp_out=np.prod(D_out, axis=1, dtype=np.int64), Dp_in=np.prod(D_in, axis=1, dtype=np.int64),
                    sectors=sectors, by_sector=np.argsort(inv), cnt=cnt)

    A = side(struct_a, slices_a, ind_a, nout_a, nin_a)
    B = side(struct_b, slices_b, ind_b, nout_b, nin_b)
    if not np.array_equal(A['sectors'], B['sectors']):
        raise BlockSparseError('Bond dimensions do not match.')
    reshape_a = tuple((sl, D, int(r), int(c)) for sl, D, r, c in zip(A['sl'], A['D'], A['Dp_out'], A['Dp_in']))
    reshape_b = tuple((sl, D, int(r), int(c)) for sl, D, r, c in zip(B['sl'], B['D'], B['Dp_in'], B['Dp_out']))
    # every (a block, b block) pair of a common contracted sector, a-major within the sector
    pa, pb, oa, ob = [], [], 0, 0
    for na, nb in zip(A['cnt'].tolist(), B['cnt'].tolist()):
        ia, ib = A['by_sector'][oa:oa + na], B['by_sector'][ob:ob + nb]
        pa.append(np.repeat(ia, nb))
        pb.append(np.tile(ib, na))
        oa, ob = oa + na, ob + nb
    pa = np.concatenate(pa) if pa else np.zeros(0, dtype=np.int64)
    pb = np.concatenate(pb) if pb else np.zeros(0, dtype=np.int64)
    tc = np.hstack([A['t_out'][pa], B['t_out'][pb]])
    t_c, first, inv, cnt = np.unique(tc, return_index=True, return_inverse=True, return_counts=True, axis=0)
    fa, fb = pa[first], pb[first]
    D_c = tuple(map(tuple, np.hstack([A['D_out'][fa], B['D_out'][fb]]).tolist()))
    Dp2 = tuple(map(tuple, np.column_stack([A['Dp_out'][fa], B['Dp_out'][fb]]).tolist()))
    Dp = [r * c for r, c in Dp2]
    offs = tuple(accumulate(Dp, initial=0))
    slc_c = tuple(zip(offs, offs[1:]))
    slices_c = Slices(Slc((sl,), D, dp) for sl, D, dp in zip(slc_c, D_c, Dp))
    pairs = np.column_stack([pa, pb])[np.argsort(inv)].tolist()
    bounds = tuple(accumulate(cnt.tolist(), initial=0))
    meta_dot = [(sl, d2, pairs[i:j]) for sl, d2, i, j in zip(slc_c, Dp2, bounds, bounds[1:])]
    s_c = tuple(struct_a.s[i] for i in nout_a) + tuple(struct_b.s[i] for i in nout_b)
    struct_c = Struct(s=s_c, t=tuple(map(tuple, t_c.tolist())), D=D_c, size=offs[-1])
    return meta_dot, reshape_a, reshape_b, struct_c, slices_c


def tensordot(a, b, axes, conj=(0, 0)):
    """Contract legs axes[0] of a with axes[1] of b (reference _contractions.py:57-125)."""
    if conj[0]:
        a = a.conj()
    if conj[1]:
        b = b.conj()
    in_a, in_b = ((x,) if isinstance(x, int) else tuple(x) for x in axes)
    in_a = tuple(x % a.ndim for x in in_a)
    in_b = tuple(x % b.ndim for x in in_b)
    if len(in_a) != len(in_b):
        raise BlockSparseError('axes[0] and axes[1] indicate different number of legs.')
    nin_a = tuple(a.trans[ax] for ax in in_a)
    nin_b = tuple(b.trans[ax] for ax in in_b)
    if not all(a.struct.s[i] == -b.struct.s[j] for i, j in zip(nin_a, nin_b)):
        raise BlockSparseError('Signatures do not match.')
    if a.isdiag:
        return _tensordot_diag(a, b, in_b, destination=(0,))
    if b.isdiag:
        return _tensordot_diag(b, a, in_a, destination=(-1,))
    if a.config.backend.BACKEND_ID != b.config.backend.BACKEND_ID:
        raise BlockSparseError('Two tensors have different backends.')
    for i, j in zip(nin_a, nin_b):
        if a.hfs[i].tree != b.hfs[j].tree:
            raise BlockSparseError('hard-fusion structures of contracted legs differ')
    nout_a = tuple(i for i in a.trans if i not in nin_a)
    nout_b = tuple(i for i in b.trans if i not in nin_b)
    hfs_c = tuple(a.hfs[i] for i in nout_a) + tuple(b.hfs[i] for i in nout_b)
    if a.config.tensordot_policy not in _TENSORDOT:
        raise BlockSparseError(f"tensordot policy {a.config.tensordot_policy} not restated")
    data, struct_c, slices_c = _TENSORDOT[a.config.tensordot_policy](a, b, nout_a, nin_a, nin_b, nout_b)
    return Tensor(a.config, struct_c, slices_c, data, hfs=hfs_c, trans=None)


@lru_cache(maxsize=1024)
def _plan_tensordot_f2m(config, struct_a, slices_a, size_a, struct_b, slices_b, size_b, nout_a, nin_a, nin_b, nout_b):
    nsym = config.sym.NSYM
    ind_a, ind_b = _common_inds(struct_a.t, struct_b.t, nin_a, nin_b, len(struct_a.s), len(struct_b.s), nsym)
    n_c = config.sym.add_charges(struct_a.n, struct_b.n)
    s_c = tuple(struct_a.s[i] for i in nout_a) + tuple(struct_b.s[i] for i in nout_b)
    struct_a, slices_a, mrg_a, ls_l, ls_ac = _meta_merge_to_matrix(config, struct_a, slices_a, (nout_a, nin_a), ind_a)
    struct_b, slices_b, mrg_b, ls_bc, ls_r = _meta_merge_to_matrix(config, struct_b, slices_b, (nin_b, nout_b), ind_b)
    if ls_ac != ls_bc:
        raise BlockSparseError('Bond dimensions do not match.')
    args_a = _merge_args(nout_a + nin_a, struct_a, slices_a, mrg_a, ind_a, size_a)
    args_b = _merge_args(nin_b + nout_b, struct_b, slices_b, mrg_b, ind_b, size_b)
    meta_dot, struct_c, slices_c = _meta_tensordot_f2m(struct_a, slices_a, struct_b, slices_b)
    size_dot = struct_c.size
    meta_un, struct_c, slices_c = _meta_unmerge_matrix(config, struct_c, slices_c, ls_l, ls_r, s_c)
    return args_a, args_b, meta_dot, size_dot, meta_un, struct_c._replace(n=n_c), slices_c


def _tensordot_f2m(a, b, nout_a, nin_a, nin_b, nout_b):
    size = a.config.backend.get_size
    args_a, args_b, meta_dot, size_dot, meta_un, struct_c, slices_c = _plan_tensordot_f2m(
        a.config, a.struct, a.slices, size(a._data), b.struct, b.slices, size(b._data), nout_a, nin_a, nin_b, nout_b)
    data_a, data_b = _transpose_and_merge_pair(a.config, a._data, args_a, b._data, args_b)
    data = a.config.backend.dot(data_a, data_b, meta_dot, size_dot)
    return _unmerge(a.config, data, meta_un), struct_c, slices_c


@lru_cache(maxsize=1024)
def _plan_tensordot_fc(config, struct_a, slices_a, size_a, struct_b, slices_b, size_b, nout_a, nin_a, nin_b, nout_b):
    nsym = config.sym.NSYM
    ind_a, ind_b = _common_inds(struct_a.t, struct_b.t, nin_a, nin_b, len(struct_a.s), len(struct_b.s), nsym)
    n_c = config.sym.add_charges(struct_a.n, struct_b.n)
    axes_a = tuple((x,) for x in nout_a) + (nin_a,)
    struct_a, slices_a, mrg_a, t_a, D_a = _meta_fuse_hard(config, struct_a, slices_a, axes_a, ind_a)
    axes_b = (nin_b,) + tuple((x,) for x in nout_b)
    struct_b, slices_b, mrg_b, t_b, D_b = _meta_fuse_hard(config, struct_b, slices_b, axes_b, ind_b)
    if not all(D_a[i] == D_b[j] for i, j in zip(nin_a, nin_b)):
        raise BlockSparseError('Bond dimensions do not match.')
    args_a = _merge_args(nout_a + nin_a, struct_a, slices_a, mrg_a, None, size_a)
    args_b = _merge_args(nin_b + nout_b, struct_b, slices_b, mrg_b, None, size_b)
    meta_dot, struct_c, slices_c = _meta_tensordot_fc(struct_a, slices_a, struct_b, slices_b)
    return args_a, args_b, meta_dot, struct_c._replace(n=n_c), slices_c


def _tensordot_fc(a, b, nout_a, nin_a, nin_b, nout_b):
    size = a.config.backend.get_size
    args_a, args_b, meta_dot, struct_c, slices_c = _plan_tensordot_fc(
        a.config, a.struct, a.slices, size(a._data), b.struct, b.slices, size(b._data), nout_a, nin_a, nin_b, nout_b)
    data_a, data_b = _transpose_and_merge_pair(a.config, a._data, args_a, b._data, args_b)
    return a.config.backend.dot(data_a, data_b, meta_dot, struct_c.size), struct_c, slices_c


@lru_cache(maxsize=1024)
def _plan_tensordot_nf(config, struct_a, slices_a, struct_b, slices_b, nout_a, nin_a, nin_b, nout_b):
    ind_a, ind_b = _common_inds(struct_a.t, struct_b.t, nin_a, nin_b, len(struct_a.s), len(struct_b.s),
                                config.sym.NSYM)
    meta_dot, reshape_a, reshape_b, struct_c, slices_c = _meta_tensordot_nf(
        struct_a, slices_a, struct_b, slices_b, ind_a, ind_b, nout_a, nin_a, nin_b, nout_b)
    n_c = config.sym.add_charges(struct_a.n, struct_b.n)
    return meta_dot, reshape_a, reshape_b, struct_c._replace(n=n_c), slices_c


def _tensordot_nf(a, b, nout_a, nin_a, nin_b, nout_b):
    """reference _contractions.py:186-246 (the transpose_dot_sum branch)."""
    meta_dot, reshape_a, reshape_b, struct_c, slices_c = _plan_tensordot_nf(
        a.config, a.struct, a.slices, b.struct, b.slices, nout_a, nin_a, nin_b, nout_b)
    data = a.config.backend.transpose_dot_sum(a._data, b._data, meta_dot, reshape_a, reshape_b, nout_a + nin_a,
                                              nin_b + nout_b, struct_c.size)
    return data, struct_c, slices_c


_TENSORDOT = {'fuse_to_matrix': _tensordot_f2m, 'fuse_contracted': _tensordot_fc, 'no_fusion': _tensordot_nf}


@lru_cache(maxsize=1024)
def _meta_broadcast(b_struct, b_slices, a_struct, a_slices, axis):
    """reference _contractions.py:502-528."""
    nsym = len(a_struct.n)
    ind_tb = tuple(x[axis * nsym:(axis + 1) * nsym] for x in b_struct.t)
    sl_a = {x[:nsym]: s for x, s in zip(a_struct.t, a_slices)}
    rows = tuple((tb, slb.slcs[0], Db, slb.Dp, sl_a[ib].slcs[0])
                 for tb, slb, Db, ib in zip(b_struct.t, b_slices, b_struct.D, ind_tb) if ib in sl_a)
    if any(Db[axis] != sla[1] - sla[0] for _, _, Db, _, sla in rows):
        raise BlockSparseError('Bond dimensions do not match.')
    if len(rows) < len(b_struct.t):
        Dp = tuple(r[3] for r in rows)
        c_slices = _slices_of(Dp, tuple(r[2] for r in rows))
        c_struct = b_struct._replace(t=tuple(r[0] for r in rows), D=tuple(r[2] for r in rows), size=sum(Dp))
    else:
        c_struct, c_slices = b_struct, b_slices
    meta = tuple((sn.slcs[0], slb, Db, sla) for (_, slb, Db, _, sla), sn in zip(rows, c_slices))
    return meta, c_struct, c_slices


def broadcast(a, b, axis):
    """Multiply leg ``axis`` of b by the diagonal tensor a."""
    ax = b.trans[axis % b.ndim]
    meta, struct, slices = _meta_broadcast(b.struct, b.slices, a.struct, a.slices, ax)
    if b.isdiag:
        meta = tuple((sln, slb, Db[0], sla) for sln, slb, Db, sla in meta)
        nd, ax = 1, 0
    else:
        nd = b.ndim_n
    data = b.config.backend.dot_diag(a._data, b._data, meta, struct.size, ax, nd)
    return b._replace(struct=struct, slices=slices, data=data)


def _tensordot_diag(a, b, in_b, destination):
    if len(in_b) != 1:
        raise BlockSparseError('contraction with a diagonal tensor over more than one leg is not restated')
    c = broadcast(a, b, in_b[0])
    return c.moveaxis(source=in_b, destination=destination)


# ------------------------------------------------------------------ masks

@lru_cache(maxsize=1024)
def _meta_mask(a_struct, a_slices, a_isdiag, mask_t, mask_D, axis):
    """reference _merging.py:554-583."""
    tD = {t: D for t, D in zip(mask_t, mask_D) if D > 0}
    nsym = len(a_struct.n)
    ind = tuple(x[axis * nsym:(axis + 1) * nsym] for x in a_struct.t)
    rows = tuple((ta, sla.slcs[0], Da, tm, tD[tm]) for ta, sla, Da, tm in zip(a_struct.t, a_slices, a_struct.D, ind)
                 if tm in tD)
    c_t = tuple(r[0] for r in rows)
    if a_isdiag:
        c_D = tuple((r[4], r[4]) for r in rows)
        c_Dp = tuple(r[4] for r in rows)
    else:
        c_D = tuple(r[2][:axis] + (r[4],) + r[2][axis + 1:] for r in rows)
        c_Dp = np.prod(c_D, axis=1, dtype=np.int64).tolist() if c_D else ()
    c_slices = _slices_of(c_Dp, c_D)
    c_struct = a_struct._replace(t=c_t, D=c_D, size=sum(c_Dp))
    if a_isdiag:
        meta = tuple((sn.slcs[0], Dn[0], sla, Da[0], tm) for sn, Dn, (_, sla, Da, tm, _) in zip(c_slices, c_D, rows))
        return meta, c_struct, c_slices, 0, 1
    meta = tuple((sn.slcs[0], Dn, sla, Da, tm) for sn, Dn, (_, sla, Da, tm, _) in zip(c_slices, c_D, rows))
    return meta, c_struct, c_slices, axis, len(a_struct.s)


def apply_mask(mask, *args, axes=0):
    """Keep the entries of legs ``axes`` of args where the diagonal boolean ``mask`` is True
    (reference _contractions.py:529-574)."""
    axes = tuple(axes) if hasattr(axes, '__iter__') else (axes,)
    nsym = mask.config.sym.NSYM
    be = mask.config.backend
    m = getattr(mask, 'host_index', None)  # a static mask knows its indices on the host
    if m is None:
        m = {t[:nsym]: be.to_mask(mask._data[sl.slcs[0][0]:sl.slcs[0][1]])
             for t, sl in zip(mask.struct.t, mask.slices)}
    mask_t = tuple(m.keys())
    mask_D = tuple(len(v) for v in m.values())
    out = []
    for b, ax in zip(args, axes):
        ax = b.trans[ax % b.ndim]
        meta, struct, slices, ax2, nd = _meta_mask(b.struct, b.slices, b.isdiag, mask_t, mask_D, ax)
        data = be.apply_mask(b._data, m, meta, struct.size, ax2, nd)
        out.append(b._replace(struct=struct, slices=slices, data=data))
    return out[0] if len(out) == 1 else out


# ------------------------------------------------------------------ decompositions

@lru_cache(maxsize=1024)
def _meta_svd(config, struct, slices, minD, sU, nU):
    """reference linalg.py:323-380."""
    sym, nsym = config.sym, config.sym.NSYM
    n0 = sym.zero()
    if any(D == 0 for D in minD):
        keep = [i for i, d in enumerate(minD) if d > 0]
        struct = struct._replace(t=tuple(struct.t[i] for i in keep), D=tuple(struct.D[i] for i in keep))
        slices = Slices(slices[i] for i in keep)
        minD = tuple(minD[i] for i in keep)
    if nU and sU == struct.s[1]:
        t_con = tuple(x[nsym:] for x in struct.t)
    elif nU:
        tc = np.array(struct.t, dtype=np.int64).reshape((len(struct.t), 2, nsym))
        t_con = tuple(map(tuple, sym.fuse(tc[:, 1:, :], (1,), -1).tolist()))
    elif sU == -struct.s[0]:
        t_con = tuple(x[:nsym] for x in struct.t)
    else:
        tc = np.array(struct.t, dtype=np.int64).reshape((len(struct.t), 2, nsym))
        t_con = tuple(map(tuple, sym.fuse(tc[:, :1, :], (1,), -1).tolist()))
    Un, Vn = (struct.n, n0) if nU else (n0, struct.n)
    Ut = tuple(x[:nsym] + y for x, y in zip(struct.t, t_con))
    St = tuple(y + y for y in t_con)
    Vt = tuple(y + x[nsym:] for y, x in zip(t_con, struct.t))
    UD = tuple((ds[0], dm) for ds, dm in zip(struct.D, minD))
    SD = tuple((dm, dm) for dm in minD)
    VD = tuple((dm, ds[1]) for dm, ds in zip(minD, struct.D))
    UDp = np.prod(UD, axis=1, dtype=np.int64).tolist() if UD else ()
    Usl = _slices_of(UDp, UD)
    rows = tuple(zip(slices, struct.D, Usl, UD, St, Vt, VD))
    St, Vt, SD, VD = zip(*sorted(zip(St, Vt, SD, VD))) if St else ((), (), (), ())
    SDp = tuple(d[0] for d in SD)
    VDp = np.prod(VD, axis=1, dtype=np.int64).tolist() if VD else ()
    Ssl = _slices_of(SDp, SD)
    Vsl = _slices_of(VDp, VD)
    Sd = {x: y.slcs[0] for x, y in zip(St, Ssl)}
    Vd = {x: y.slcs[0] for x, y in zip(Vt, Vsl)}
    meta = tuple((sl.slcs[0], d, su.slcs[0], du, Sd[ts], Vd[tv], dv) for sl, d, su, du, ts, tv, dv in rows)
    Us = Struct(s=(struct.s[0], sU), n=Un, diag=False, t=Ut, D=UD, size=sum(UDp))
    Ss = Struct(s=(-sU, sU), n=n0, diag=True, t=St, D=SD, size=sum(SDp))
    Vs = Struct(s=(-sU, struct.s[1]), n=Vn, diag=False, t=Vt, D=VD, size=sum(VDp))
    return meta, Us, Usl, Ss, Ssl, Vs, Vsl


def svd(a, axes=(0, 1), sU=1, nU=True, Uaxis=-1, Vaxis=0, fix_signs=False, **kwargs):
    """Blockwise thin SVD a = U S V (reference linalg.py:135-320, policy 'fullrank')."""
    out_l, out_r = ((x,) if isinstance(x, int) else tuple(x) for x in axes)
    out_hl = tuple(a.trans[ax] for ax in out_l)
    out_hr = tuple(a.trans[ax] for ax in out_r)
    data, struct, slices, ls_l, ls_r = _merge_to_matrix(a, (out_hl, out_hr))
    minD = tuple(min(ds) for ds in struct.D)
    meta, Ust, Usl, Sst, Ssl, Vst, Vsl = _meta_svd(a.config, struct, slices, minD, sU, nU)
    sizes = (Ust.size, Sst.size, Vst.size)
    be = a.config.backend
    Ud, Sd, Vd = be.svd(data, meta, sizes, diagnostics=kwargs.get('diagnostics', None))
    if fix_signs:
        Ud, Vd = be.fix_svd_signs(Ud, Vd, meta)
    ls_s = _leg_struct_trivial(Sst, axis=0)
    S = Tensor(a.config, Sst, Ssl, Sd, hfs=(Fusion(s=(-sU,)), Fusion(s=(sU,))))
    Us = tuple(a.struct.s[i] for i in out_hl) + (sU,)
    mu, Ust, Usl = _meta_unmerge_matrix(a.config, Ust, Usl, ls_l, ls_s, Us)
    U = Tensor(a.config, Ust, Usl, _unmerge(a.config, Ud, mu),
               hfs=tuple(a.hfs[i] for i in out_hl) + (Fusion(s=(sU,)),))
    Vs = (-sU,) + tuple(a.struct.s[i] for i in out_hr)
    mv, Vst, Vsl = _meta_unmerge_matrix(a.config, Vst, Vsl, ls_s, ls_r, Vs)
    V = Tensor(a.config, Vst, Vsl, _unmerge(a.config, Vd, mv),
               hfs=(Fusion(s=(-sU,)),) + tuple(a.hfs[i] for i in out_hr))
    return U.moveaxis(-1, Uaxis), S, V.moveaxis(0, Vaxis)


@lru_cache(maxsize=1024)
def _meta_qr(config, struct, slices, sQ):
    """Sector layout of Q and R for a = Q R (reference linalg.py:795-830): Q(s0, sQ) keeps the charge of a,
    R(-sQ, s1) has zero charge; the connecting leg of a sector carries the charge that lets R be charge-free.
    Meta rows: (slice of a, D of a, slice of Q, D of Q, slice of R, D of R); R's blocks are sorted by charge."""
    sym, nsym = config.sym, config.sym.NSYM
    if sQ == struct.s[1]:
        t_con = tuple(x[nsym:] for x in struct.t)
    else:
        tc = np.array(struct.t, dtype=np.int64).reshape((len(struct.t), 2, nsym))
        t_con = tuple(map(tuple, sym.fuse(tc[:, 1:, :], (1,), -1).tolist()))
    k = tuple(min(ds) for ds in struct.D)
    Qt = tuple(x[:nsym] + y for x, y in zip(struct.t, t_con))
    QD = tuple((ds[0], m) for ds, m in zip(struct.D, k))
    QDp = tuple(a * b for a, b in QD)
    Qsl = _slices_of(QDp, QD)
    Rrows = sorted((y + x[nsym:], (m, ds[1])) for y, x, m, ds in zip(t_con, struct.t, k, struct.D))
    Rt = tuple(r[0] for r in Rrows)
    RD = tuple(r[1] for r in Rrows)
    RDp = tuple(a * b for a, b in RD)
    Rsl = _slices_of(RDp, RD)
    where_R = {t: sl.slcs[0] for t, sl in zip(Rt, Rsl)}
    meta = tuple((sl.slcs[0], d, sq.slcs[0], dq, where_R[y + x[nsym:]], (dq[1], d[1]))
                 for sl, d, sq, dq, y, x in zip(slices, struct.D, Qsl, QD, t_con, struct.t))
    Qs = Struct(s=(struct.s[0], sQ), n=struct.n, diag=False, t=Qt, D=QD, size=sum(QDp))
    Rs = Struct(s=(-sQ, struct.s[1]), n=sym.zero(), diag=False, t=Rt, D=RD, size=sum(RDp))
    return meta, Qs, Qsl, Rs, Rsl


def qr(a, axes=(0, 1), sQ=1, Qaxis=-1, Raxis=0):
    """Blockwise reduced QR a = Q R with diag(R) >= 0 (reference linalg.py:738-792)."""
    out_l, out_r = ((x,) if isinstance(x, int) else tuple(x) for x in axes)
    out_hl = tuple(a.trans[ax] for ax in out_l)
    out_hr = tuple(a.trans[ax] for ax in out_r)
    data, struct, slices, ls_l, ls_r = _merge_to_matrix(a, (out_hl, out_hr))
    meta, Qst, Qsl, Rst, Rsl = _meta_qr(a.config, struct, slices, sQ)
    Qd, Rd = a.config.backend.qr(data, meta, (Qst.size, Rst.size))
    ls = _leg_struct_trivial(Rst, axis=0)
    mq, Qst, Qsl = _meta_unmerge_matrix(a.config, Qst, Qsl, ls_l, ls,
                                        tuple(a.struct.s[i] for i in out_hl) + (sQ,))
    Q = Tensor(a.config, Qst, Qsl, _unmerge(a.config, Qd, mq),
               hfs=tuple(a.hfs[i] for i in out_hl) + (Fusion(s=(sQ,)),))
    mr, Rst, Rsl = _meta_unmerge_matrix(a.config, Rst, Rsl, ls, ls_r,
                                        (-sQ,) + tuple(a.struct.s[i] for i in out_hr))
    R = Tensor(a.config, Rst, Rsl, _unmerge(a.config, Rd, mr),
               hfs=(Fusion(s=(-sQ,)),) + tuple(a.hfs[i] for i in out_hr))
    return Q.moveaxis(-1, Qaxis), R.moveaxis(0, Raxis)


def _cat(datas):
    """Concatenate flat data buffers (torch tensors or numpy arrays)."""
    if isinstance(datas[0], np.ndarray):
        return np.concatenate(datas)
    import torch
    return torch.cat(datas)


def svd_many(items, fix_signs=False, **kwargs):
    """Blockwise thin SVDs of several tensors in one backend call per data type.  ``items`` is a list of
    (a, axes, sU, nU).  Each tensor is merged to its sector matrices as in :func:`svd`; the blocks of all
    tensors of one data type are concatenated into one buffer with one meta (offsets shifted), so the
    backend batches every block of them into the same launches; the factors are split back per tensor.
    Returns a list of (U, S, V) as :func:`svd` would for each item (Uaxis = -1, Vaxis = 0)."""
    groups = {}
    for i, it in enumerate(items):
        groups.setdefault(str(it[0].data.dtype), []).append(i)
    out = [None] * len(items)
    for idx in groups.values():
        for i, r in zip(idx, _svd_many_same_dtype([items[i] for i in idx], fix_signs, **kwargs)):
            out[i] = r
    return out


def _svd_many_same_dtype(items, fix_signs=False, **kwargs):
    parts, datas, metas = [], [], []
    off = [0, 0, 0, 0]  # data, U, S, V
    for a, axes, sU, nU in items:
        out_l, out_r = ((x,) if isinstance(x, int) else tuple(x) for x in axes)
        out_hl = tuple(a.trans[ax] for ax in out_l)
        out_hr = tuple(a.trans[ax] for ax in out_r)
        data, struct, slices, ls_l, ls_r = _merge_to_matrix(a, (out_hl, out_hr))
        minD = tuple(min(ds) for ds in struct.D)
        meta, Ust, Usl, Sst, Ssl, Vst, Vsl = _meta_svd(a.config, struct, slices, minD, sU, nU)
        sh = lambda x, o: (x[0] + o, x[1] + o)
        metas.extend((sh(sl, off[0]), d, sh(su, off[1]), du, sh(ss, off[2]), sh(sv, off[3]), dv)
                     for sl, d, su, du, ss, sv, dv in meta)
        parts.append((a, tuple(off), (Ust, Usl, Sst, Ssl, Vst, Vsl), ls_l, ls_r, out_hl, out_hr, sU))
        datas.append(data)
        off = [off[0] + len(data), off[1] + Ust.size, off[2] + Sst.size, off[3] + Vst.size]
    cfg = items[0][0].config
    be = cfg.backend
    meta_all = tuple(metas)
    Ud, Sd, Vd = be.svd(_cat(datas), meta_all, tuple(off[1:]), diagnostics=kwargs.get('diagnostics', None))
    if fix_signs:
        Ud, Vd = be.fix_svd_signs(Ud, Vd, meta_all)
    out = []
    for a, o, (Ust, Usl, Sst, Ssl, Vst, Vsl), ls_l, ls_r, out_hl, out_hr, sU in parts:
        ls_s = _leg_struct_trivial(Sst, axis=0)
        S = Tensor(a.config, Sst, Ssl, Sd[o[2]:o[2] + Sst.size], hfs=(Fusion(s=(-sU,)), Fusion(s=(sU,))))
        Us = tuple(a.struct.s[i] for i in out_hl) + (sU,)
        mu, Ust2, Usl2 = _meta_unmerge_matrix(a.config, Ust, Usl, ls_l, ls_s, Us)
        U = Tensor(a.config, Ust2, Usl2, _unmerge(a.config, Ud[o[1]:o[1] + Ust.size], mu),
                   hfs=tuple(a.hfs[i] for i in out_hl) + (Fusion(s=(sU,)),))
        Vs = (-sU,) + tuple(a.struct.s[i] for i in out_hr)
        mv, Vst2, Vsl2 = _meta_unmerge_matrix(a.config, Vst, Vsl, ls_s, ls_r, Vs)
        V = Tensor(a.config, Vst2, Vsl2, _unmerge(a.config, Vd[o[3]:o[3] + Vst.size], mv),
                   hfs=(Fusion(s=(-sU,)),) + tuple(a.hfs[i] for i in out_hr))
        out.append((U, S, V))
    return out


def truncation_mask(S, tol=0, tol_block=0, D_block=float('inf'), D_total=float('inf'), truncate_multiplets=False,
                    mask_f=None, **kwargs):
    """Boolean diagonal mask of the kept singular values (reference linalg.py:637-735).

    The reference decides on the host from S, reading one count per block and the global one
    (``.item()``, a device round trip each) and sorting on the device.  Here S is read to the host once
    and the same rule runs in numpy (``np.argsort`` orders ties as the reference numpy backend does);
    the kept indices ride along as the mask's ``host_index``, so applying it reads nothing back."""
    if mask_f is not None:
        return mask_f(S)
    be = S.config.backend
    nsym = S.config.sym.NSYM
    Sh = np.asarray(be.to_numpy(be.detach(S._data))).real
    keep = np.ones(Sh.shape, dtype=bool)
    if truncate_multiplets:
        tol_block, D_block = 0, float('inf')
    tol_null = 0. if isinstance(tol_block, dict) else tol_block
    D_null = 0 if isinstance(D_block, dict) else D_block
    for t, sl in zip(S.struct.t, S.slices):
        t = t[:nsym]
        lo, hi = sl.slcs[0]
        tol_rel = tol_block[t] if isinstance(tol_block, dict) and t in tol_block else tol_null
        blk = Sh[lo:hi]
        D_tol = np.count_nonzero(blk > tol_rel * np.abs(blk).max()) if hi > lo else 0
        D_bl = D_block[t] if isinstance(D_block, dict) and t in D_block else D_null
        D_bl = min(D_bl, D_tol)
        if 0 < D_bl < sl.Dp:
            inds = np.argsort(blk)
            keep[lo:hi][inds[:-D_bl]] = False
        elif D_bl == 0:
            keep[lo:hi] = False
    tmp = Sh * keep
    D_tol = np.count_nonzero(tmp > tol * np.abs(tmp).max()) if tmp.size else 0
    D_total = min(D_total, D_tol)
    if D_total == 0:
        keep[:] = False
    else:
        inds = np.argsort(tmp)
        if truncate_multiplets and D_total < len(inds):
            gap = -1
            for p in range(D_total, len(inds)):
                gp = abs(Sh[inds[-p]] - Sh[inds[-p - 1]])
                if gp > gap:
                    D_total, gap = p, gp
                if gap > abs(Sh[inds[-p]]):
                    break
        keep[inds[:-D_total]] = False
    m = S._replace(data=be.to_tensor(keep, dtype='bool', device=S.config.device))
    m.host_index = {t[:nsym]: be.to_mask(keep[sl.slcs[0][0]:sl.slcs[0][1]]) for t, sl in zip(S.struct.t, S.slices)}
    return m


def truncation_mask_multiplets(S, tol=0, D_total=float('inf'), eps_multiplet=1e-13, hermitian=False, **kwargs):
    """Boolean mask keeping at most D_total of the largest values of the diagonal S above tol * max(S)
    without splitting a multiplet (reference linalg.py:539-634): values are ranked over all blocks, and
    the cut moves down to the nearest position whose relative gap |s_i - s_i+1| / (max(|s_i|, |s_i+1|) +
    1e-16) exceeds eps_multiplet (it stays where it is when there is none).  With ``hermitian``, blocks of
    opposite charges keep only the positions kept in both."""
    if not S.isdiag:
        raise BlockSparseError('truncation_mask_multiplets requires a diagonal tensor')
    be = S.config.backend
    vals = be.detach(S._data)
    keep = vals > float('inf')
    order = be.argsort(-vals)
    ranked = np.asarray(be.to_numpy(vals[order]))  # one host copy; the cut is decided on the host
    n_keep = min(int(np.sum(ranked > ranked[0] * tol)), D_total)
    if n_keep >= len(ranked):
        return S._replace(data=vals > -float('inf'))
    big = np.maximum(np.abs(ranked[:-1]), np.abs(ranked[1:])) + 1.0e-16
    rel_gap = np.abs(ranked[:-1] - ranked[1:]) / big
    for i in range(n_keep - 1, -1, -1):
        if rel_gap[i] > eps_multiplet:
            n_keep = i + 1
            break
    keep[order[:n_keep]] = True
    if hermitian:
        nsym = S.config.sym.NSYM
        where = {t: sl.slcs[0] for t, sl in zip(S.struct.t, S.slices)}
        for t in S.struct.t:
            lo, hi = where[t]
            if not bool(keep[lo:hi].any()):
                continue
            tc = np.array(t, dtype=np.int64).reshape((1, 1, -1))
            tn = tuple(S.config.sym.fuse(tc, (1,), -1).ravel().tolist())
            if tn == t:
                continue
            if tn not in where:
                raise BlockSparseError(f'no block {tn} opposite to {t}')
            lo2, hi2 = where[tn]
            k = min(hi - lo, hi2 - lo2)
            both = keep[lo:lo + k] & keep[lo2:lo2 + k]
            keep[lo:lo + k] = both
            keep[lo2:lo2 + k] = both
    return S._replace(data=keep)


_STATIC_MASKS = {}


def truncation_mask_static(S, D_block, check=None):
    """Mask keeping the first D_block[t] values of every block t of the diagonal S (the values of a block
    are in descending order), decided from the structure alone: S is not read on the host, so the mask
    (and the step around it) can be captured in a HIP graph and replayed.  Blocks absent from D_block
    keep nothing.  It equals truncation_mask(S, tol=0, D_block=D_block, D_total=sum(D_block)) whenever
    every kept value is positive.  With ``check`` (a device int64 tensor of two counters) the step adds, on
    the device, 1 to check[0] when a kept value is 0 (the eager rule would then keep fewer: the fixed
    structure is invalid) and 1 to check[1] when a dropped value exceeds the smallest kept one (the
    reference's global rule truncation_mask(S, D_total=sum) would pick another set)."""
    nsym = S.config.sym.NSYM
    be = S.config.backend
    norm_key = lambda k: (k,) if isinstance(k, (int, np.integer)) else tuple(k)
    want = {norm_key(k): int(v) for k, v in D_block.items()}
    key = (S.struct, S.slices, tuple(sorted(want.items())), str(S.config.device))
    hit = _STATIC_MASKS.get(key)
    if hit is None:
        keep = np.zeros(S.struct.size, dtype=bool)
        index = {}
        for t, sl in zip(S.struct.t, S.slices):
            lo, hi = sl.slcs[0]
            k = min(want.get(t[:nsym], 0), hi - lo)
            keep[lo:lo + k] = True
            index[t[:nsym]] = be.to_mask(keep[lo:hi])  # host index list, in the backend's mask type
        hit = (index, be.to_tensor(keep, dtype='bool', device=S.config.device))
        if len(_STATIC_MASKS) > 256:
            _STATIC_MASKS.clear()
        _STATIC_MASKS[key] = hit
    index, kept = hit
    if check is not None:
        import torch
        s = be.detach(S._data)
        inf = torch.full_like(s, float('inf'))
        kmin = torch.where(kept, s, inf).amin()
        dmax = torch.where(kept, -inf, s).amax()
        check.add_(torch.stack([(kmin <= 0), (dmax > kmin)]).to(check.dtype))
    m = S._replace(data=kept)
    m.host_index = index
    return m


def svd_with_truncation(a, axes=(0, 1), sU=1, nU=True, Uaxis=-1, Vaxis=0, fix_signs=False, tol=0, tol_block=0,
                        D_block=float('inf'), D_total=float('inf'), truncate_multiplets=False, mask_f=None, **kwargs):
    """reference linalg.py:49-132."""
    U, S, V = svd(a, axes=axes, sU=sU, nU=nU, fix_signs=fix_signs, **kwargs)
    mask = truncation_mask(S, tol=tol, tol_block=tol_block, D_block=D_block, D_total=D_total,
                           truncate_multiplets=truncate_multiplets, mask_f=mask_f)
    U, S, V = apply_mask(mask, U, S, V, axes=(-1, 0, 0))
    return U.moveaxis(-1, Uaxis), S, V.moveaxis(0, Vaxis)


@lru_cache(maxsize=1024)
def _meta_eigh(config, struct, slices, sU, minD):
    """reference linalg.py:963-1010."""
    sym, nsym = config.sym, config.sym.NSYM
    n0 = sym.zero()
    if sU == -struct.s[0]:
        t_con = tuple(x[:nsym] for x in struct.t)
    else:
        tc = np.array(struct.t, dtype=np.int64).reshape((len(struct.t), 2, nsym))
        t_con = tuple(map(tuple, sym.fuse(tc[:, :1, :], (1,), -1).tolist()))
    Ut = tuple(x[:nsym] + y for x, y in zip(struct.t, t_con))
    UD = tuple((ds[0], dm) for ds, dm in zip(struct.D, minD))
    UDp = np.prod(UD, axis=1, dtype=np.int64).tolist() if UD else ()
    Usl = _slices_of(UDp, UD)
    SD = tuple((dm, dm) for dm in minD)
    St = tuple(y + y for y in t_con)
    rows = tuple(zip(slices, struct.D, Usl, UD, St))
    St, SD = zip(*sorted(zip(St, SD))) if St else ((), ())
    SDp = tuple(d[0] for d in SD)
    Ssl = _slices_of(SDp, SD)
    Sd = {x: y.slcs[0] for x, y in zip(St, Ssl)}
    meta = tuple((sl.slcs[0], d, su.slcs[0], du, Sd[ts]) for sl, d, su, du, ts in rows)
    Us = Struct(s=(struct.s[0], sU), n=n0, diag=False, t=Ut, D=UD, size=sum(UDp))
    Ss = Struct(s=(-sU, sU), n=n0, diag=True, t=St, D=SD, size=sum(SDp))
    return meta, Ss, Ssl, Us, Usl


def eigh(a, axes, sU=1):
    """Blockwise Hermitian eigendecomposition a = U S U^H, eigenvalues ascending per block
    (reference linalg.py:831-960 with the default 'fullrank' policy, without the 'which' reordering)."""
    out_l, out_r = ((x,) if isinstance(x, int) else tuple(x) for x in axes)
    out_hl = tuple(a.trans[ax] for ax in out_l)
    out_hr = tuple(a.trans[ax] for ax in out_r)
    data, struct, slices, ls_l, ls_r = _merge_to_matrix(a, (out_hl, out_hr))
    minD = tuple(min(ds) for ds in struct.D)
    meta, Sst, Ssl, Ust, Usl = _meta_eigh(a.config, struct, slices, sU, minD)
    Sd, Ud = a.config.backend.eigh(data, meta, (Sst.size, Ust.size))
    ls_s = _leg_struct_trivial(Sst, axis=1)
    S = Tensor(a.config, Sst, Ssl, Sd, hfs=(Fusion(s=(-sU,)), Fusion(s=(sU,))))
    Us = tuple(a.struct.s[i] for i in out_hl) + (sU,)
    mu, Ust, Usl = _meta_unmerge_matrix(a.config, Ust, Usl, ls_l, ls_s, Us)
    U = Tensor(a.config, Ust, Usl, _unmerge(a.config, Ud, mu),
               hfs=tuple(a.hfs[i] for i in out_hl) + (Fusion(s=(sU,)),))
    return S, U


def vdot(a, b):
    """<a|b> summed over common blocks (a conjugated)."""
    nsym = a.config.sym.NSYM
    ib = {t: sl.slcs[0] for t, sl in zip(b.struct.t, b.slices)}
    meta = tuple((sl.slcs[0], ib[t]) for t, sl in zip(a.struct.t, a.slices) if t in ib)
    if a.trans != tuple(range(a.ndim_n)) or b.trans != tuple(range(b.ndim_n)):
        a, b = consume_transpose(a), consume_transpose(b)
        return vdot(a, b)
    return a.config.backend.vdot(a.config.backend.conj(a._data), b._data, meta)
