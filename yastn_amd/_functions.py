"""torch.autograd.Function wrappers of the C-ABI kernels (forward + setup_context style, so that
torch.func transforms and non-reentrant checkpoint recompute work as with the reference's
yastn/backend/_backend_torch_backwards.py).  Every forward and backward is one or a few grouped
HIP launches over all blocks of the call; nothing falls back to per-block torch ops.
"""
import functools
import os

import numpy as np
import torch

from . import _lib as L
from . import plans as P

SYNC_CHECKS = os.environ.get('YASTN_HIP_SYNC_CHECKS', '1') != '0'
# empirical tile autotuning of every new grouped-GEMM plan (skipped while a HIP graph is captured)
AUTOTUNE = os.environ.get('YASTN_HIP_AUTOTUNE', '1') != '0'


def _maybe_autotune(plan, run):
    if AUTOTUNE and not getattr(plan, 'tuned', False) and not torch.cuda.is_current_stream_capturing():
        plan.autotune(run)
MAX_SWEEPS = int(os.environ.get('YASTN_HIP_MAX_SWEEPS', '60'))
# Lorentzian broadening of the SVD adjoint: the reference fixes it to 1e-12 (torch_svd_gesdd.py:4-6,
# absolute, whatever ad_decomp_reg says).  set_ad_broadening(eps) changes it, e.g. to 1e-30 for an
# unbroadened adjoint in finite-difference checks.
AD_EPS = 1e-12


def set_ad_broadening(eps):
    global AD_EPS
    AD_EPS = float(eps)


def dtype_code(t):
    if t.dtype == torch.float64:
        return L.YH_F64
    if t.dtype == torch.complex128:
        return L.YH_C128
    raise TypeError(f"yastn_amd HIP kernels compute in float64 / complex128, got {t.dtype}")


def raw(t):
    """Materialise lazy conjugation / negation and make the buffer contiguous."""
    if t.is_conj():
        t = t.resolve_conj()
    if t.is_neg():
        t = t.resolve_neg()
    return t.contiguous()


def stream_of(t):
    if t.device.type != 'cuda':
        raise RuntimeError(f"yastn_amd backend needs GPU tensors, got a tensor on {t.device}")
    return _raw_stream(t.device.index)


def _stream_object(index):
    return torch.cuda.current_stream(index).cuda_stream


# the raw handle of the current stream without a Stream object (a tenth of its cost), where torch has the call
_raw_stream = getattr(torch._C, '_cuda_getCurrentRawStream', _stream_object)


def ptr(t):
    return t.data_ptr() if t is not None else None


def _real_dtype(t):
    return t.real.dtype if t.is_complex() else t.dtype


# ------------------------------------------------------------------ gather family

class _Opaque(torch.autograd.Function):
    """Runs fn on plain tensors: under torch.func transforms, apply() hands forward the unwrapped tensors.
    Used by the adjoints below, which launch kernels through raw device pointers; an adjoint is not
    differentiated again."""

    @staticmethod
    def forward(fn, *args):
        return fn(*args)

    @staticmethod
    def setup_context(ctx, inputs, output):
        pass

    @staticmethod
    def backward(ctx, *grads):
        raise RuntimeError("yastn_amd: the adjoint kernels are not differentiable again")


def host_array(t):
    """Host numpy copy of a tensor that carries no gradient (mask values, indices).  Under a torch.func
    transform such a tensor is wrapped and has no storage of its own; _Opaque hands its forward the
    plain tensor, and the copy is taken there."""
    if not _is_wrapped(t):
        return t.detach().cpu().numpy()
    box = []

    def grab(v):
        box.append(v.detach().cpu().numpy())
        return v.new_empty(0)

    _Opaque.apply(grab, t)
    return box[0]


class _CtxProxy:
    """The autograd context with its saved tensors replaced by plain ones."""

    def __init__(self, ctx, saved):
        self._ctx, self.saved_tensors = ctx, saved

    def __getattr__(self, name):
        return getattr(self._ctx, name)


def _is_wrapped(t):
    return torch.is_tensor(t) and torch._C._functorch.is_functorch_wrapped_tensor(t)


def _plain_backward(fn):
    """Decorator for the backward of a Function: when its saved tensors or incoming gradients are wrapped
    by a torch.func transform (the reference's fixed-point AD calls torch.func.vjp, fixed_pt.py:853), the
    backward runs inside _Opaque, which unwraps them; otherwise it runs as it is."""
    @functools.wraps(fn)
    def wrapper(ctx, *grads):
        saved = ctx.saved_tensors  # unpacked once (checkpointing allows no second unpack)
        if not any(_is_wrapped(t) for t in (*saved, *grads)):
            return fn(_CtxProxy(ctx, saved), *grads)
        ns, slots = len(saved), []

        def run(*ts):
            out = fn(_CtxProxy(ctx, ts[:ns]), *ts[ns:])
            slots[:] = [o is not None for o in out]
            return tuple(o for o in out if o is not None)
        res = _Opaque.apply(run, *saved, *grads)
        res = iter(res if isinstance(res, tuple) else (res,))
        return tuple(next(res) if s else None for s in slots)
    return wrapper


def run_gather(entry, plan, dst, src):
    L.call(entry, ptr(dst), dst.numel(), ptr(src), src.numel(), dtype_code(dst), *plan.args(), stream_of(dst))
    return dst


def run_gather_same(entry, plan, dst, src):
    L.call(entry, ptr(dst), ptr(src), dst.numel(), dtype_code(dst), *plan.args(), stream_of(dst))
    return dst


def _fast_apply_available():
    """The fast path of _Fn.apply relies on torch internals (torch 2.10): the C base class of
    autograd.Function, torch._C._are_functorch_transforms_active and
    torch._functorch.utils.unwrap_dead_wrappers.  Returns that helper, or None (then torch's public
    Function.apply runs on every call) when any of them is missing or has another shape."""
    try:
        from torch._functorch.utils import unwrap_dead_wrappers as unwrap
        import inspect
        if len(inspect.signature(unwrap).parameters) != 1:
            return None
        if not callable(getattr(torch._C, '_are_functorch_transforms_active', None)):
            return None
        base = getattr(torch._C, '_FunctionBase', None)
        if base is None or base not in torch.autograd.Function.__mro__ or not hasattr(base, 'apply'):
            return None
        return unwrap
    except Exception:
        return None


_UNWRAP_DEAD = _fast_apply_available()
FAST_APPLY = _UNWRAP_DEAD is not None and os.environ.get('YASTN_HIP_FAST_APPLY', '1') != '0'


class _Fn(torch.autograd.Function):
    """autograd.Function whose ``apply`` skips torch's per-call ``inspect.signature`` binding of default
    arguments (~30 us a call, ~200 calls per CTMRG step): every call in this package passes all forward
    arguments positionally, so the binding is the identity.  Under a torch.func transform, with keyword
    arguments, or when the torch internals it needs are absent (FAST_APPLY false), torch's own path runs."""

    @classmethod
    def apply(cls, *args, **kwargs):
        if not FAST_APPLY or kwargs or torch._C._are_functorch_transforms_active():
            return super().apply(*args, **kwargs)
        return super(torch.autograd.Function, cls).apply(*_UNWRAP_DEAD(args))


class TransposeAndMerge(_Fn):
    """A1 / A6 (reference _backend_torch_backwards.py:338-392)."""

    @staticmethod
    def forward(data, order, meta_new, meta_mrg, Dsize):
        data = raw(data)
        plan = P.merge_plan(tuple(order), meta_new, meta_mrg, Dsize, data.numel(), data.device)
        out = torch.empty(Dsize, dtype=data.dtype, device=data.device)
        return run_gather('yastn_hip_transpose_and_merge', plan, out, data)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, order, meta_new, meta_mrg, Dsize = inputs
        ctx.order, ctx.meta_new, ctx.meta_mrg, ctx.Dsize, ctx.src_numel = tuple(order), meta_new, meta_mrg, Dsize, data.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g)
        plan = P.merge_adjoint_plan(ctx.order, ctx.meta_new, ctx.meta_mrg, ctx.Dsize, ctx.src_numel, g.device)
        out = torch.empty(ctx.src_numel, dtype=g.dtype, device=g.device)
        return run_gather('yastn_hip_transpose_and_merge_adjoint', plan, out, g), None, None, None, None


class TransposeAndMergePair(_Fn):
    """A1 / A6 of both operands of one tensordot in one launch each way: the two reference
    kernel_transpose_and_merge calls (_backend_torch_backwards.py:338-392) of _tensordot_fc / f2m."""

    @staticmethod
    def forward(data_a, order_a, meta_new_a, meta_mrg_a, Dsize_a, data_b, order_b, meta_new_b, meta_mrg_b, Dsize_b):
        data_a, data_b = raw(data_a), raw(data_b)
        dev = data_a.device
        pa = P.merge_plan(tuple(order_a), meta_new_a, meta_mrg_a, Dsize_a, data_a.numel(), dev)
        pb = P.merge_plan(tuple(order_b), meta_new_b, meta_mrg_b, Dsize_b, data_b.numel(), dev)
        plan = P.pair_plan(pa, pb, dev)
        out_a = torch.empty(Dsize_a, dtype=data_a.dtype, device=dev)
        out_b = torch.empty(Dsize_b, dtype=data_b.dtype, device=dev)
        L.call('yastn_hip_transpose_and_merge_pair', ptr(out_a), Dsize_a, ptr(data_a), data_a.numel(), ptr(out_b),
               Dsize_b, ptr(data_b), data_b.numel(), dtype_code(out_a), *plan.args(), stream_of(out_a))
        return out_a, out_b

    @staticmethod
    def setup_context(ctx, inputs, output):
        data_a, order_a, meta_new_a, meta_mrg_a, Dsize_a, data_b, order_b, meta_new_b, meta_mrg_b, Dsize_b = inputs
        ctx.args_a = (tuple(order_a), meta_new_a, meta_mrg_a, Dsize_a, data_a.numel())
        ctx.args_b = (tuple(order_b), meta_new_b, meta_mrg_b, Dsize_b, data_b.numel())

    @staticmethod
    @_plain_backward
    def backward(ctx, ga, gb):
        ga, gb = raw(ga), raw(gb)
        dev = ga.device
        pa = P.merge_adjoint_plan(*ctx.args_a, dev)
        pb = P.merge_adjoint_plan(*ctx.args_b, dev)
        out_a = torch.empty(ctx.args_a[4], dtype=ga.dtype, device=dev)
        out_b = torch.empty(ctx.args_b[4], dtype=gb.dtype, device=dev)
        if ga.dtype == gb.dtype:
            plan = P.pair_plan(pa, pb, dev)
            L.call('yastn_hip_transpose_and_merge_adjoint_pair', ptr(out_a), out_a.numel(), ptr(ga), ga.numel(),
                   ptr(out_b), out_b.numel(), ptr(gb), gb.numel(), dtype_code(out_a), *plan.args(), stream_of(out_a))
        else:
            run_gather('yastn_hip_transpose_and_merge_adjoint', pa, out_a, ga)
            run_gather('yastn_hip_transpose_and_merge_adjoint', pb, out_b, gb)
        return out_a, None, None, None, None, out_b, None, None, None, None


class Unmerge(_Fn):
    """A2 / A8 (reference _backend_torch_backwards.py:395-426)."""

    @staticmethod
    def forward(data, meta):
        data = raw(data)
        plan = P.unmerge_plan(meta, data.numel(), data.device)
        out = torch.empty_like(data)
        return run_gather_same('yastn_hip_unmerge', plan, out, data)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, meta = inputs
        ctx.meta, ctx.numel = meta, data.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g)
        plan = P.unmerge_adjoint_plan(ctx.meta, ctx.numel, g.device)
        out = torch.empty(ctx.numel, dtype=g.dtype, device=g.device)
        return run_gather_same('yastn_hip_unmerge_adjoint', plan, out, g), None


class Transpose(_Fn):
    """backend.transpose (reference _backend_torch_backwards.py:313-335)."""

    @staticmethod
    def forward(data, axes, meta):
        data = raw(data)
        plan = P.transpose_plan(tuple(axes), meta, data.numel(), data.device)
        out = torch.empty_like(data)
        return run_gather_same('yastn_hip_transpose', plan, out, data)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, axes, meta = inputs
        ctx.axes, ctx.meta, ctx.numel = tuple(axes), meta, data.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g)
        inv = tuple(int(x) for x in np.argsort(ctx.axes))
        meta_inv = _inverse_transpose_meta(ctx.meta)
        plan = P.transpose_plan(inv, meta_inv, ctx.numel, g.device)
        out = torch.empty(ctx.numel, dtype=g.dtype, device=g.device)
        return run_gather_same('yastn_hip_transpose', plan, out, g), None, None


_INV_T = P._Cache(maxsize=1024)


def _inverse_transpose_meta(meta):
    return _INV_T.get(('inv_t', id(meta)), (meta,),
                      lambda: tuple((slo, Do, sln, Dn) for sln, Dn, slo, Do in meta))


def _mask_host(mask):
    """Host copy of a mask dict (charge -> kept indices).  A value may also be a ``slice`` (the
    reference's flip_charges embeds with {0: slice(None)}, tensor/_single.py:222-225); it is resolved
    against the masked dimension of each block when the plan is built.  The tensor values of one dtype
    and device are concatenated and copied in one transfer (each copy to the host waits for the device)."""
    def as_index(arr):
        if arr.dtype == np.bool_:
            arr = np.nonzero(arr.ravel())[0]
        return arr.astype(np.int64).ravel()
    vals, groups = {}, {}
    for k, v in mask.items():
        key = tuple(k) if isinstance(k, (list, tuple)) else k
        if isinstance(v, slice):
            vals[key] = v
        elif torch.is_tensor(v) and v.device.type == 'cpu' and not _is_wrapped(v):
            vals[key] = as_index(v.detach().numpy())
        elif torch.is_tensor(v):
            vals[key] = None
            groups.setdefault((v.dtype, v.device), []).append((key, v))
        else:
            vals[key] = as_index(np.asarray(v))
    for items in groups.values():
        if len(items) == 1:
            arrs = [host_array(items[0][1])]
        else:
            flat = host_array(torch.cat([v.reshape(-1) for _, v in items]))
            arrs = np.split(flat, np.cumsum([v.numel() for _, v in items])[:-1])
        for (key, _), arr in zip(items, arrs):
            vals[key] = as_index(arr)
    return vals


def _mask_key(mh):
    return tuple((k, ('slice', v.start, v.stop, v.step) if isinstance(v, slice) else v.tobytes())
                 for k, v in sorted(mh.items(), key=lambda kv: repr(kv[0])))


_SWAP = P._Cache(maxsize=1024)


def _swapped_mask_meta(meta):
    return _SWAP.get(('swap', id(meta)), (meta,),
                     lambda: tuple((sla, Da, sln, Dn, tm) for sln, Dn, sla, Da, tm in meta))


def _mask_gather(Adata, mh, key, meta, Dsize, axis, embed):
    plan = P.mask_plan(mh, meta, Dsize, Adata.numel(), axis, Adata.device, embed=embed, mask_key=key)
    out = torch.empty(Dsize, dtype=Adata.dtype, device=Adata.device)
    return run_gather('yastn_hip_embed_mask' if embed else 'yastn_hip_apply_mask', plan, out, Adata)


class ApplyMask(_Fn):
    """A12 apply_mask, adjoint = embed (reference _backend_torch_backwards.py:251-279)."""

    @staticmethod
    def forward(Adata, mask, meta, Dsize, axis, ndim):
        Adata = raw(Adata)
        mh = _mask_host(mask)
        return _mask_gather(Adata, mh, _mask_key(mh), meta, Dsize, axis, False)

    @staticmethod
    def setup_context(ctx, inputs, output):
        Adata, mask, meta, Dsize, axis, ndim = inputs
        ctx.mh = _mask_host(mask)
        ctx.meta, ctx.axis, ctx.size_a = meta, axis, Adata.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g)
        out = _mask_gather(g, ctx.mh, _mask_key(ctx.mh), _swapped_mask_meta(ctx.meta), ctx.size_a, ctx.axis, True)
        return out, None, None, None, None, None


class EmbedMask(_Fn):
    """A12 embed_mask, adjoint = apply (reference _backend_torch_backwards.py:282-310)."""

    @staticmethod
    def forward(Adata, mask, meta, Dsize, axis, ndim):
        Adata = raw(Adata)
        mh = _mask_host(mask)
        return _mask_gather(Adata, mh, _mask_key(mh), meta, Dsize, axis, True)

    @staticmethod
    def setup_context(ctx, inputs, output):
        Adata, mask, meta, Dsize, axis, ndim = inputs
        ctx.mh = _mask_host(mask)
        ctx.meta, ctx.axis, ctx.size_a = meta, axis, Adata.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g)
        out = _mask_gather(g, ctx.mh, _mask_key(ctx.mh), _swapped_mask_meta(ctx.meta), ctx.size_a, ctx.axis, False)
        return out, None, None, None, None, None


# ------------------------------------------------------------------ grouped GEMM

_Pointers = L.ctypes.c_void_p * L.YH_MAX_BUFS


def launch_plan(plan, outs, ins, dtype, stream):
    """One launch of a grouped-GEMM plan, followed by its split-K reduction when it has one (the
    partial products then live in a scratch buffer appended to the outputs)."""
    part = None
    if plan.part_numel:
        dev = next(t for t in outs if t is not None)
        part = torch.empty(plan.part_numel, dtype=dev.dtype, device=dev.device)
        outs = [*outs, *[None] * (plan.part_buf - len(outs)), part]
    po, pi = _Pointers(*map(ptr, outs)), _Pointers(*map(ptr, ins))  # the rest are null
    L.call('yastn_hip_grouped_gemm', po, pi, dtype, *plan.args(), stream)
    if part is not None:
        L.call('yastn_hip_splitk_reduce', po, ptr(part), dtype, plan.d_red.data_ptr(), len(plan.h_red), stream)


def run_gemm(plan, outs, ins, dtype, tune=True):
    dev = next(t for t in outs if t is not None)
    run = lambda: launch_plan(plan, outs, ins, dtype, stream_of(dev))
    if tune and plan.accumulates and AUTOTUNE and not getattr(plan, 'tuned', False) \
            and not torch.cuda.is_current_stream_capturing():
        # an accumulating plan is timed on copies of its outputs, so the real ones are written once
        scratch = [t.clone() if t is not None else None for t in outs]
        _maybe_autotune(plan, lambda: launch_plan(plan, scratch, ins, dtype, stream_of(dev)))
    elif tune:
        _maybe_autotune(plan, run)
    run()


class Dot(_Fn):
    """A3 / A7 (reference _backend_torch_backwards.py:98-138)."""

    @staticmethod
    def forward(Adata, Bdata, meta_dot, Dsize):
        dtype = torch.promote_types(Adata.dtype, Bdata.dtype)
        A = raw(Adata.to(dtype))
        B = raw(Bdata.to(dtype))
        plan = P.dot_plan(meta_dot, A.numel(), B.numel(), Dsize, A.device)
        out = (torch.empty if plan.covered == Dsize else torch.zeros)(Dsize, dtype=dtype, device=A.device)
        run = lambda: launch_plan(plan, (out,), (A, B), dtype_code(out), stream_of(out))
        _maybe_autotune(plan, run)
        run()
        return out

    @staticmethod
    def setup_context(ctx, inputs, output):
        Adata, Bdata, meta_dot, Dsize = inputs
        ctx.save_for_backward(Adata, Bdata)
        ctx.meta_dot = meta_dot

    @staticmethod
    @_plain_backward
    def backward(ctx, gC):
        Adata, Bdata = ctx.saved_tensors
        dtype = torch.promote_types(Adata.dtype, Bdata.dtype)
        A = raw(Adata.to(dtype))
        B = raw(Bdata.to(dtype))
        gC = raw(gC.to(dtype))
        plan = P.dot_adjoint_plan(ctx.meta_dot, A.numel(), B.numel(), gC.numel(), A.device)
        gA = (torch.zeros if plan.zero_a else torch.empty)(A.numel(), dtype=dtype, device=A.device)
        gB = (torch.zeros if plan.zero_b else torch.empty)(B.numel(), dtype=dtype, device=A.device)
        run = lambda: launch_plan(plan, (gA, gB), (A, B, gC), dtype_code(gA), stream_of(gA))
        _maybe_autotune(plan, run)
        run()
        if not Adata.is_complex() and gA.is_complex():
            gA = gA.real.contiguous()
        if not Bdata.is_complex() and gB.is_complex():
            gB = gB.real.contiguous()
        return gA, gB, None, None


class DotDiag(_Fn):
    """backend.dot_diag (reference backend_np.py:604-611, backend_torch.py:557-564): every output block
    is a dense block of B scaled along ``axis`` by a diagonal block of A, one launch.  The reference
    differentiates its torch ops; here gB = g conj(A) (the same kernel) and gA = the sum of g conj(B)
    along the other axes (one deterministic reduction launch)."""

    @staticmethod
    def forward(Adata, Bdata, meta, Dsize, axis, a_ndim):
        dtype = torch.promote_types(Adata.dtype, Bdata.dtype)
        A, B = raw(Adata.to(dtype)), raw(Bdata.to(dtype))
        plan = P.dot_diag_plan(meta, axis, a_ndim, A.numel(), B.numel(), Dsize, A.device)
        out = (torch.empty if plan.covered == Dsize else torch.zeros)(Dsize, dtype=dtype, device=A.device)
        L.call('yastn_hip_dot_diag', ptr(out), ptr(A), ptr(B), dtype_code(out), plan.d_jobs.data_ptr(), plan.njobs,
               plan.max_n, 0, stream_of(out))
        return out

    @staticmethod
    def setup_context(ctx, inputs, output):
        Adata, Bdata, meta, Dsize, axis, a_ndim = inputs
        ctx.save_for_backward(Adata, Bdata)
        ctx.meta, ctx.Dsize, ctx.axis, ctx.a_ndim = meta, Dsize, axis, a_ndim

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        Adata, Bdata = ctx.saved_tensors
        dtype = torch.promote_types(Adata.dtype, Bdata.dtype)
        A, B, g = raw(Adata.to(dtype)), raw(Bdata.to(dtype)), raw(g.to(dtype))
        plan = P.dot_diag_plan(ctx.meta, ctx.axis, ctx.a_ndim, A.numel(), B.numel(), ctx.Dsize, A.device)
        st, dt = stream_of(g), dtype_code(g)
        gA = gB = None
        if ctx.needs_input_grad[0]:
            gA = (torch.empty if plan.a_covered == A.numel() else torch.zeros)(A.numel(), dtype=dtype,
                                                                              device=A.device)
            L.call('yastn_hip_dot_diag_adjoint_a', ptr(gA), ptr(g), ptr(B), dt, plan.d_jobs.data_ptr(),
                   plan.d_groups.data_ptr(), plan.ngroups, plan.d_ids.data_ptr(), plan.max_D, st)
            if not Adata.is_complex() and gA.is_complex():
                gA = gA.real.contiguous()
        if ctx.needs_input_grad[1]:
            gB = (torch.empty if plan.b_covered == B.numel() else torch.zeros)(B.numel(), dtype=dtype,
                                                                              device=B.device)
            L.call('yastn_hip_dot_diag', ptr(gB), ptr(A), ptr(g), dt, plan.d_jobs_t.data_ptr(), plan.njobs,
                   plan.max_n, 1, st)
            if not Bdata.is_complex() and gB.is_complex():
                gB = gB.real.contiguous()
        return gA, gB, None, None, None, None


# ------------------------------------------------------------------ SVD / eigh

# while a HIP graph is captured the sweeps cannot stop on a host read: the captured SVD launches the most
# sweeps an eager call of the same plan used, plus this margin (the extra ones exit at once on the device;
# a replay that needed more reports non-convergence through the deferred checks).  Hermitian blocks whose matrices fit one
# workgroup iterate there until they have converged, whatever eager calls saw; those of them that run on the panel path, which is
# faster, get CAPTURE_EIGH_SWEEPS at least, twice what random and graded blocks take (about 110 us of launches
# that exit at once: one block of 64 columns 655 us a replay, 545 with the margin alone, 1878 in one workgroup).
CAPTURE_SWEEP_MARGIN = 3
CAPTURE_EIGH_SWEEPS = 20
_DEFERRED = []  # stack of lists collecting convergence flags to check later (deferred_checks)


class deferred_checks:
    """Within this context (and always while a HIP graph is being captured into it) the convergence flags
    of the Jacobi kernels are not read on the host after each call: they are collected, and ``check()``
    reads them all at once (one synchronisation), e.g. after each replay of a captured graph."""

    def __init__(self):
        self.flags = []

    def __enter__(self):
        _DEFERRED.append(self.flags)
        return self

    def __exit__(self, *exc):
        _DEFERRED.remove(self.flags)
        return False

    def check(self):
        for what, flags in self.flags:
            _raise_on_flags(flags, what)


def _raise_on_flags(flags, what):
    lo, bad, nonfinite = flags.tolist()
    if nonfinite:
        # as the reference, whose scipy SVD / eigh check the input (backend_np.py:281-286)
        raise ValueError(f"{what}: the input contains infs or NaNs")
    if lo == -3:
        raise L.HipBackendError(f"{what}: panel Jacobi plan smaller than a panel pair (LDS)")
    if bad:
        raise L.HipBackendError(f"{what}: Jacobi did not converge in {MAX_SWEEPS} sweeps for {bad} block(s)")


def _check_info(info, what, data, dt, st):
    """Convergence words of a decomposition of ``data`` and whether that is finite, checked now or deferred."""
    capturing = torch.cuda.is_current_stream_capturing()
    if not _DEFERRED and capturing:
        raise RuntimeError("yastn_amd: SVD/eigh captured in a HIP graph needs deferred_checks() around the capture")
    if info.numel() == 0 or not (_DEFERRED or SYNC_CHECKS):
        return
    out = torch.empty(3 + L.YH_CHECK_SCRATCH, dtype=torch.int32, device=info.device)
    L.call('yastn_hip_check_result', ptr(out), out.numel(), ptr(info), info.numel(), ptr(data), data.numel(), dt, st)
    if _DEFERRED:
        _DEFERRED[-1].append((what, out[:3]))
    else:
        _raise_on_flags(out[:3], what)


_SIDE = {}


def _side_stream(device):
    """A second stream per device (default priority), for work that overlaps the current stream."""
    key = torch.device(device).index
    if key not in _SIDE:
        _SIDE[key] = torch.cuda.Stream(device=device)
    return _SIDE[key]


def _householder_steps(plan, work, dt, st):
    """The panel steps of a batched Householder QR (plans.SvdPlan / QrPlan): the panels of all blocks in one launch,
    then their reflectors on the columns to their right in another."""
    for step, (d_ids, n, rest) in enumerate(plan.panel_steps):
        L.call('yastn_hip_svd_qr_panel', ptr(work), dt, plan.d_qdesc.data_ptr(), d_ids.data_ptr(), n, step, plan.qr_rows, st)
        if rest:
            L.call('yastn_hip_reflect_trailing', ptr(work), dt, plan.d_qdesc.data_ptr(), d_ids.data_ptr(), n, step, rest,
                   st)


def _run_jacobi(mode, plan, data, out_a, out_s, out_b):
    """LDS-resident blocks in one launch; larger blocks through the panel path (one launch per round of
    panel pairs, one host check per sweep).  mode 0: SVD (U, S, Vh); mode 1: eigh (S, U)."""
    dt = dtype_code(data)
    st = stream_of(data)
    work = torch.empty(max(plan.work_numel, 1), dtype=data.dtype, device=data.device)
    info = torch.empty(max(plan.nblocks, 1), dtype=torch.int32, device=data.device)
    joined, lds_st = None, st
    if plan.n_big and (plan.n_small or plan.n_lds) and not torch.cuda.is_current_stream_capturing():
        # the one-workgroup kernels (small blocks) run on a side stream, overlapping the panel path of the
        # large blocks, which occupies only part of the GPU; joined below
        cur = torch.cuda.current_stream(data.device)
        side = _side_stream(data.device)
        side.wait_stream(cur)
        lds_st = side.cuda_stream
        joined = (cur, side)
    try:
        order = plan.d_order.data_ptr()
        if plan.n_small:
            L.call('yastn_hip_jacobi_small', ptr(out_a), ptr(out_s), ptr(out_b), ptr(data), dt, mode,
                   plan.d_blocks.data_ptr(), order, plan.n_small, plan.small_bytes, ptr(info), MAX_SWEEPS, lds_st)
        order += plan.n_small * plan.d_order.element_size()
        if plan.n_lds and mode == 0:
            L.call('yastn_hip_svd', ptr(out_a), ptr(out_s), ptr(out_b), ptr(data), dt, plan.d_blocks.data_ptr(),
                   plan.n_lds, order, plan.n_lds, plan.lds_bytes, ptr(work), ptr(info), MAX_SWEEPS, lds_st)
        elif plan.n_lds:
            L.call('yastn_hip_eigh', ptr(out_s), ptr(out_a), ptr(data), dt, plan.d_blocks.data_ptr(), plan.n_lds,
                   order, plan.n_lds, plan.lds_bytes, ptr(work), ptr(info), MAX_SWEEPS, lds_st)
        if plan.n_big:
            mu = torch.empty(plan.nblocks, dtype=torch.float64, device=data.device)
            floors = torch.empty(plan.nblocks, dtype=torch.float64, device=data.device)
            if plan.n_plain:
                L.call('yastn_hip_svd_panel_init', ptr(data), ptr(work), ptr(mu), ptr(floors), dt, mode,
                       plan.d_blocks.data_ptr(), plan.d_plain.data_ptr(), plan.n_plain, st)
            if plan.n_pre:
                L.call('yastn_hip_svd_precond_load', ptr(data), ptr(work), ptr(floors), dt, plan.d_blocks.data_ptr(),
                       plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(), plan.n_pre, st)
                # W0 = Q R (Householder), then X = R^H
                _householder_steps(plan, work, dt, st)
                L.call('yastn_hip_svd_precond_init', ptr(work), dt, plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(),
                       plan.n_pre, st)
            # two launches per round (Gram partials, then inner sweep + update); a round of a sweep after one
            # that rotated nothing exits at once on the device, so under capture a fixed budget of sweeps is
            # recorded with no host read in between
            state = torch.zeros(4 + MAX_SWEEPS, dtype=torch.int32, device=data.device)
            part = torch.empty(max(plan.part_numel, 1), dtype=torch.float64, device=data.device)
            capturing = torch.cuda.is_current_stream_capturing()
            budget = MAX_SWEEPS
            if capturing and getattr(plan, 'sweeps_seen', None):
                budget = plan.sweeps_seen + CAPTURE_SWEEP_MARGIN
                if mode == 1 and plan.big_fits_lds:
                    budget = max(budget, CAPTURE_EIGH_SWEEPS)
                budget = min(MAX_SWEEPS, budget)
            launched = 0
            for sweep in range(budget):
                L.call('yastn_hip_svd_panel_sweep', ptr(work), ptr(floors), dt, plan.d_jblocks.data_ptr(),
                       plan.d_jobs.data_ptr(), plan.h_rounds.ctypes.data, len(plan.rounds), plan.panel_width,
                       plan.maxch_p, plan.panel_slices, ptr(part), part.numel(), sweep, MAX_SWEEPS, ptr(state),
                       state.numel(), st)
                launched += 1
                if not capturing and int(state[4 + sweep].item()) == 0:
                    plan.sweeps_seen = max(getattr(plan, 'sweeps_seen', 0) or 0, sweep + 1)
                    break
            L.call('yastn_hip_svd_panel_result', ptr(state), state.numel(), launched, st)
            d_sweeps = state.data_ptr() + 3 * state.element_size()
            done = 0
            if plan.n_plain:
                L.call('yastn_hip_svd_panel_finalize', ptr(out_a), ptr(out_s), ptr(out_b) if mode == 0 else None,
                       ptr(work), ptr(mu), dt, mode, plan.d_blocks.data_ptr(), plan.d_plain.data_ptr(), plan.n_plain,
                       ptr(info), done, d_sweeps, st)
            if plan.n_pre:
                L.call('yastn_hip_svd_precond_finalize', ptr(out_a), ptr(out_s), ptr(out_b), ptr(work), dt,
                       plan.d_blocks.data_ptr(), plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(), plan.n_pre, ptr(info),
                       done, d_sweeps, st)
                # p-side vectors: [V_J; 0] -> Q [V_J; 0], panels in reverse order
                L.call('yastn_hip_svd_reflect', ptr(out_a), ptr(out_b), ptr(work), dt, plan.d_blocks.data_ptr(),
                       plan.d_qdesc.data_ptr(), plan.d_pre.data_ptr(), plan.n_pre, plan.qr_cols, st)
    finally:
        # the side-stream launch reads data and writes the outputs: joined even when the panel path raises
        if joined is not None:
            joined[0].wait_stream(joined[1])
    _check_info(info[:plan.nblocks], 'svd' if mode == 0 else 'eigh', data, dt, st)


def svd_forward(data, meta, sizes):
    data = raw(data)
    plan = P.svd_plan(meta, data.element_size(), data.numel(), sizes, data.device)
    U = torch.empty(sizes[0], dtype=data.dtype, device=data.device)
    S = torch.empty(sizes[1], dtype=_real_dtype(data), device=data.device)
    V = torch.empty(sizes[2], dtype=data.dtype, device=data.device)
    _run_jacobi(0, plan, data, U, S, V)
    return U, S, V


class _SvdAdjointPlans:
    """Cached plans of the composed SVD adjoint for one svd meta."""

    def __init__(self, meta, dims, device):
        u_sz, s_sz, v_sz, a_sz = dims
        descs, kk, tt = [], 0, 0
        gx, tx, g2, t2, g3, t3 = [], [], [], [], [], []
        self.cover = 0
        for sl, D, slU, DU, slS, slV, DV in meta:
            m, n = D
            k = min(m, n)
            t_sz = m * k if m >= n else k * n
            descs.append((m, n, k, slU[0], slS[0], slV[0], kk, tt))
            # X = U^H gU  (ins: 0 U, 1 gU, 2 Vh, 3 gVh; outs: 0 X, 1 Y)
            gx.append((k, k, kk, k, 1, len(tx), 1, 0 << 8))
            tx.append((slU[0], 1, k, slU[0], k, 1, m, 1 | (0 << 8) | (1 << 16)))
            # Y = Vh gVh^H
            gx.append((k, k, kk, k, 1, len(tx), 1, 1 << 8))
            tx.append((slV[0], n, 1, slV[0], 1, n, n, 2 | (2 << 8) | (3 << 16)))
            # T += U J (m >= n)  or  T += J Vh (m < n)   (ins: 0 U, 1 J, 2 Vh; out 0 T)
            if m >= n:
                g2.append((m, k, tt, k, 1, len(t2), 1, 1))
                t2.append((slU[0], k, 1, kk, k, 1, k, (0 << 8) | (1 << 16)))
            else:
                g2.append((k, n, tt, n, 1, len(t2), 1, 1))
                t2.append((kk, k, 1, slV[0], n, 1, k, (1 << 8) | (2 << 16)))
            # gA = T Vh (m >= n) or U T (m < n)   (ins: 0 T, 1 Vh, 2 U; out 0 gA)
            if m >= n:
                g3.append((m, n, sl[0], n, 1, len(t3), 1, 0))
                t3.append((tt, k, 1, slV[0], n, 1, k, (0 << 8) | (1 << 16)))
            else:
                g3.append((m, n, sl[0], n, 1, len(t3), 1, 0))
                t3.append((slU[0], k, 1, tt, n, 1, k, (2 << 8) | (0 << 16)))
            kk += k * k
            tt += t_sz
            self.cover += m * n
        self.kk, self.tt = kk, tt
        self.nblocks = len(descs)
        self.h_descs = np.array(descs, dtype=np.int64).reshape(-1, 8)
        self.d_descs = torch.from_numpy(self.h_descs).to(device)
        self.p1 = P.GemmPlan(gx, tx, (u_sz, u_sz, v_sz, v_sz), (max(kk, 1), max(kk, 1)), device) if gx else None
        self.p2 = P.GemmPlan(g2, t2, (u_sz, max(kk, 1), v_sz), (max(tt, 1),), device) if g2 else None
        self.p3 = P.GemmPlan(g3, t3, (max(tt, 1), v_sz, u_sz), (a_sz,), device) if g3 else None
        self.zero_a = self.cover != a_sz


_SVD_ADJ = P._Cache()


def svd_backward(U, S, V, gU, gS, gV, meta, data_size):
    dims = (U.numel(), S.numel(), V.numel(), data_size)
    ap = _SVD_ADJ.get(('svd_adj', id(meta), dims, U.dtype, U.device.type, U.device.index), (meta,),
                      lambda: _SvdAdjointPlans(meta, dims, U.device))
    dt = dtype_code(U)
    dev = U.device
    gA = (torch.zeros if ap.zero_a else torch.empty)(data_size, dtype=U.dtype, device=dev)
    if ap.nblocks == 0:
        return gA
    U, S, V = raw(U), raw(S), raw(V)
    gU = raw(gU.to(U.dtype)) if gU is not None else None
    gV = raw(gV.to(U.dtype)) if gV is not None else None
    gS = raw(gS.to(S.dtype)) if gS is not None else None
    X = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
    Y = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
    J = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
    T = torch.empty(max(ap.tt, 1), dtype=U.dtype, device=dev)
    if gU is not None or gV is not None:
        # zero gradients are passed as the forward factors with the flag off; their products are unused
        run_gemm(ap.p1, (X, Y), (U, gU if gU is not None else U, V, gV if gV is not None else V), dt)
    L.call('yastn_hip_svd_adjoint_core', ptr(J), ptr(T), ptr(X), ptr(Y), ptr(S), ptr(gS if gS is not None else S),
           ptr(gU if gU is not None else U), ptr(gV if gV is not None else V), dt, ap.d_descs.data_ptr(),
           ap.nblocks, AD_EPS, int(gS is not None), int(gU is not None), int(gV is not None), stream_of(U))
    run_gemm(ap.p2, (T,), (U, J, V), dt)
    run_gemm(ap.p3, (gA,), (T, V, U), dt)
    return gA


class Svd(_Fn):
    """A4 / A9 (reference _backend_torch_backwards.py:26-66, linalg/torch_svd_gesdd.py)."""

    @staticmethod
    def forward(data, meta, sizes, fullrank_uv=False, ad_decomp_reg=1.0e-12, diagnostics=None):
        if fullrank_uv:
            raise NotImplementedError("yastn_amd svd computes the thin SVD (fullrank_uv=False)")
        return svd_forward(data, meta, sizes)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, meta, sizes = inputs[:3]
        U, S, V = output
        ctx.save_for_backward(U, S, V)
        ctx.meta, ctx.data_size = meta, data.numel()
        ctx.set_materialize_grads(False)

    @staticmethod
    @_plain_backward
    def backward(ctx, gU, gS, gV):
        U, S, V = ctx.saved_tensors
        gA = svd_backward(U, S, V, gU, gS, gV, ctx.meta, ctx.data_size)
        return gA, None, None, None, None, None


def eigh_forward(data, meta, sizes):
    data = raw(data)
    plan = P.eigh_plan(meta, data.element_size(), data.numel(), sizes, data.device)
    S = torch.zeros(sizes[0], dtype=_real_dtype(data), device=data.device)
    U = torch.zeros(sizes[1], dtype=data.dtype, device=data.device)
    _run_jacobi(1, plan, data, U, S, None)
    return S, U


class _EighAdjointPlans:
    def __init__(self, meta, dims, device):
        u_sz, s_sz, a_sz = dims
        descs, kk = [], 0
        g1, t1, g2, t2, g3, t3 = [], [], [], [], [], []
        self.cover = 0
        for sl, D, slU, DU, slS in meta:
            n = D[0]
            descs.append((n, slS[0], kk, 0, 0, 0, 0, 0))
            # X = U^H gU   (ins 0 U, 1 gU; out 0 X)
            g1.append((n, n, kk, n, 1, len(t1), 1, 0))
            t1.append((slU[0], 1, n, slU[0], n, 1, n, 1 | (0 << 8) | (1 << 16)))
            # T = U Xo      (ins 0 U, 1 Xo; out 0 T)
            g2.append((n, n, kk, n, 1, len(t2), 1, 0))
            t2.append((slU[0], n, 1, kk, n, 1, n, (0 << 8) | (1 << 16)))
            # gA = T U^H    (ins 0 T, 1 U; out 0 gA)
            g3.append((n, n, sl[0], n, 1, len(t3), 1, 0))
            t3.append((kk, n, 1, slU[0], 1, n, n, 2 | (0 << 8) | (1 << 16)))
            kk += n * n
            self.cover += n * n
        self.kk, self.nblocks = kk, len(descs)
        self.d_descs = torch.from_numpy(np.array(descs, dtype=np.int64).reshape(-1, 8)).to(device)
        self.p1 = P.GemmPlan(g1, t1, (u_sz, u_sz), (max(kk, 1),), device) if g1 else None
        self.p2 = P.GemmPlan(g2, t2, (u_sz, max(kk, 1)), (max(kk, 1),), device) if g2 else None
        self.p3 = P.GemmPlan(g3, t3, (max(kk, 1), u_sz), (a_sz,), device) if g3 else None
        self.zero_a = self.cover != a_sz


_EIGH_ADJ = P._Cache()


class Eigh(_Fn):
    """A5 / A10: Hermitian eigendecomposition with the (unbroadened) torch.linalg.eigh adjoint
    that the reference backend uses (backend_torch.py:378)."""

    @staticmethod
    def forward(data, meta, sizes):
        return eigh_forward(data, meta, sizes)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, meta, sizes = inputs
        S, U = output
        ctx.save_for_backward(S, U)
        ctx.meta, ctx.data_size = meta, data.numel()
        ctx.set_materialize_grads(False)

    @staticmethod
    @_plain_backward
    def backward(ctx, gS, gU):
        S, U = ctx.saved_tensors
        dims = (U.numel(), S.numel(), ctx.data_size)
        ap = _EIGH_ADJ.get(('eigh_adj', id(ctx.meta), dims, U.dtype, U.device.index), (ctx.meta,),
                           lambda: _EighAdjointPlans(ctx.meta, dims, U.device))
        dev, dt = U.device, dtype_code(U)
        gA = (torch.zeros if ap.zero_a else torch.empty)(ctx.data_size, dtype=U.dtype, device=dev)
        if ap.nblocks == 0:
            return gA, None, None
        U = raw(U)
        gU = raw(gU.to(U.dtype)) if gU is not None else None
        gS = raw(gS.to(S.dtype)) if gS is not None else None
        X = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
        Xo = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
        T = torch.empty(max(ap.kk, 1), dtype=U.dtype, device=dev)
        if gU is not None:
            run_gemm(ap.p1, (X,), (U, gU), dt)
        L.call('yastn_hip_eigh_adjoint_core', ptr(Xo), ptr(X), ptr(S), ptr(gS if gS is not None else S), dt,
               ap.d_descs.data_ptr(), ap.nblocks, int(gS is not None), int(gU is not None), stream_of(U))
        run_gemm(ap.p2, (T,), (U, Xo), dt)
        run_gemm(ap.p3, (gA,), (T, U), dt)
        return gA, None, None


# ------------------------------------------------------------------ fix_svd_signs

_SIGN_MAPS = P._Cache()


def _sign_maps(meta, device):
    """Per-block words of the sign kernels, and the dot_diag metas (reference layout (sln, slb, Db, sla)) that
    scale the columns of U and the rows of Vh by one phase per singular value."""
    def build():
        blocks, mu, mv = [], [], []
        for sl, D, slU, DU, slS, slV, DV in meta:
            blocks.append((sl[0], D[0], D[1], slU[0], slS[0], slV[0], 0, 0))
            mu.append((slU, slU, DU, slS))
            mv.append((slV, slV, DV, slS))
        h = np.array(blocks, dtype=np.int64).reshape(-1, L.YH_SVD_WORDS)
        return torch.from_numpy(h).to(device), len(blocks), tuple(mu), tuple(mv)
    return _SIGN_MAPS.get(('signs', id(meta), device.index), (meta,), build)


def fix_svd_signs(Udata, Vdata, meta):
    """A11: pivots from the HIP kernel; phases applied with differentiable tensor ops when a gradient
    is needed (as the reference torch backend does), else in place by the HIP kernel.  On the gradient
    route the phases scale U's columns and Vh's rows through dot_diag, whose adjoint sums each phase's
    contributions in a fixed order (deterministic, no sort)."""
    s_numel = max([slS[1] for _, _, _, _, slS, _, _ in meta], default=0)
    blocks, nb, mu, mv = _sign_maps(meta, Udata.device)
    dt = dtype_code(Udata)
    if not (torch.is_grad_enabled() and (Udata.requires_grad or Vdata.requires_grad)):
        U2 = raw(Udata).clone()
        V2 = raw(Vdata).clone()
        L.call('yastn_hip_fix_svd_signs', ptr(U2), ptr(V2), dt, blocks.data_ptr(), nb, stream_of(U2))
        return U2, V2
    def pivots(u):  # on plain tensors: under a torch.func transform _Opaque hands it the unwrapped U
        u = raw(u)
        piv = torch.empty(max(s_numel, 1), dtype=torch.int64, device=u.device)
        L.call('yastn_hip_svd_sign_pivots', ptr(u), ptr(piv), dt, blocks.data_ptr(), nb, stream_of(u))
        return piv
    U0 = Udata.detach()
    piv = _Opaque.apply(pivots, U0) if _is_wrapped(U0) else pivots(U0)
    # one pivot per column, all at distinct positions of U: the adjoint of the selection adds into each
    # position once
    ph = torch.index_select(Udata, 0, piv[:s_numel])
    ph = ph / ph.abs()
    return (DotDiag.apply(ph.conj(), Udata, mu, Udata.numel(), 1, 2),
            DotDiag.apply(ph, Vdata, mv, Vdata.numel(), 0, 2))

def qr_forward(data, meta, sizes, plan=None):
    """Batched Householder QR of every block (plan: plans.QrPlan)."""
    data = raw(data)
    if plan is None:
        plan = P.qr_plan(meta, data.element_size(), data.numel(), sizes, data.device)
    dt = dtype_code(data)
    st = stream_of(data)
    Q = torch.zeros(sizes[0], dtype=data.dtype, device=data.device)
    R = torch.zeros(sizes[1], dtype=data.dtype, device=data.device)
    if plan.nblocks == 0:
        return Q, R
    work = torch.empty(plan.work_numel, dtype=data.dtype, device=data.device)
    L.call('yastn_hip_qr_init', ptr(data), ptr(work), dt, plan.d_qdesc.data_ptr(), plan.d_qblocks.data_ptr(),
           plan.nblocks, st)
    _householder_steps(plan, work, dt, st)
    L.call('yastn_hip_qr_reflect', ptr(work), dt, plan.d_qdesc.data_ptr(), plan.nblocks, plan.max_k, st)
    L.call('yastn_hip_qr_finalize', ptr(Q), ptr(R), ptr(work), dt, plan.d_qdesc.data_ptr(),
           plan.d_qblocks.data_ptr(), plan.nblocks, st)
    return Q, R


def qr_backward(data, Q, R, gQ, gR, meta, sizes):
    """Adjoint of the batched QR: with R1 = R(:, :k), gQ' = gQ (+ A(:, k:) gR(:, k:)^H when m < n),
    C = copyltu(R1 gR1^H - gQ'^H Q), gA(:, :k) = (gQ' + Q C) R1^{-H} and gA(:, k:) = Q gR(:, k:)."""
    data = raw(data)
    if gQ is None:
        gQ = torch.zeros_like(Q)
    if gR is None:
        gR = torch.zeros_like(R)
    gQ, gR = gQ.contiguous(), gR.contiguous()
    plan = P.qr_adjoint_plan(meta, data.element_size(), data.numel(), sizes, data.device)
    dt = dtype_code(data)
    st = stream_of(data)
    gA = torch.zeros(data.numel(), dtype=data.dtype, device=data.device)
    if plan.nblocks == 0:
        return gA
    gQp = gQ.clone()
    if plan.gq is not None:
        run_gemm(plan.gq, (gQp,), (data, gR), dt, tune=False)
        run_gemm(plan.gy, (gA,), (Q, gR), dt, tune=False)
    M1 = torch.empty(plan.m_numel, dtype=data.dtype, device=data.device)
    M2 = torch.empty_like(M1)
    run_gemm(plan.m1, (M1,), (R, gR), dt, tune=False)
    run_gemm(plan.m2, (M2,), (gQp, Q), dt, tune=False)
    C = torch.empty_like(M1)
    L.call('yastn_hip_qr_adjoint_core', ptr(C), ptr(M1), ptr(M2), dt, plan.d_words.data_ptr(), plan.nblocks, st)
    B = gQp  # B = gQ' + Q C, accumulated in place
    run_gemm(plan.b, (B,), (Q, C), dt, tune=False)
    L.call('yastn_hip_qr_adjoint_trsm', ptr(gA), ptr(B), ptr(R), dt, plan.d_words.data_ptr(), plan.nblocks,
           plan.max_rows, plan.max_k, st)
    return gA


class Qr(_Fn):
    """Batched QR with its adjoint (the reference differentiates torch.linalg.qr through torch's autograd,
    backend_torch.py:475-484)."""

    @staticmethod
    def forward(data, meta, sizes, plan):
        return qr_forward(data, meta, sizes, plan)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, meta, sizes, _ = inputs
        Q, R = output
        ctx.save_for_backward(data, Q, R)
        ctx.meta, ctx.sizes = meta, sizes
        ctx.set_materialize_grads(False)

    @staticmethod
    @_plain_backward
    def backward(ctx, gQ, gR):
        data, Q, R = ctx.saved_tensors
        if gQ is None and gR is None:
            return None, None, None, None
        return qr_backward(data, Q, R, gQ, gR, ctx.meta, ctx.sizes), None, None, None


class PermutePack(_Fn):
    """Blocks of a flat buffer permuted into packed matrices (one box gather); the adjoint is the
    inverse gather into a zeroed buffer of the source's size."""

    @staticmethod
    def forward(data, fwd, bwd, packed_numel):
        data = raw(data)
        out = torch.empty(packed_numel, dtype=data.dtype, device=data.device)
        return run_gather('yastn_hip_block_gather', fwd, out, data)

    @staticmethod
    def setup_context(ctx, inputs, output):
        data, _, bwd, _ = inputs
        ctx.bwd, ctx.numel = bwd, data.numel()

    @staticmethod
    @_plain_backward
    def backward(ctx, g):
        g = raw(g).contiguous()
        out = torch.zeros(ctx.numel, dtype=g.dtype, device=g.device)
        return run_gather('yastn_hip_block_gather', ctx.bwd, out, g), None, None, None


class TdsCore(_Fn):
    """Output blocks as sums of products of packed matrices (one grouped GEMM); adjoint: two grouped
    GEMMs accumulating into the packed gradients."""

    @staticmethod
    def forward(At, Bt, plan, Dsize):
        At, Bt = raw(At), raw(Bt)
        C = torch.zeros(Dsize, dtype=At.dtype, device=At.device)
        if plan.dot.ngemms:
            run_gemm(plan.dot, (C,), (At, Bt), dtype_code(C))
        return C

    @staticmethod
    def setup_context(ctx, inputs, output):
        At, Bt, plan, _ = inputs
        ctx.save_for_backward(At, Bt)
        ctx.plan = plan

    @staticmethod
    @_plain_backward
    def backward(ctx, gC):
        At, Bt = ctx.saved_tensors
        gC = raw(gC).contiguous()
        plan = ctx.plan
        gA = torch.zeros_like(At)
        gB = torch.zeros_like(Bt)
        dt = dtype_code(gA)
        if plan.dot_a is not None and plan.dot_a.ngemms:
            run_gemm(plan.dot_a, (gA,), (gC, Bt), dt)
        if plan.dot_b is not None and plan.dot_b.ngemms:
            run_gemm(plan.dot_b, (gB,), (At, gC), dt)
        return gA, gB, None, None
