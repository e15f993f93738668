"""Fused ladder decode of QAD's fake-quantised Linears on MI355X, forward and backward.

Mirror of the reference's ``hi2/qad_kernel.py`` (``load`` 229-258, ``available`` 261-268,
``failure`` 271-272, ``_StoredDecode`` 275-318, ``_Transform`` 321-336, ``original`` 339-348,
``stored`` 351-370), backed by ``hi2x_qad_decode_fwd/bwd``, ``hi2x_qad_weights_fwd/bwd`` (the
decode with the transform) and ``hi2x_qad_wht_scale`` of ``libhi2x.so``.  ``load()`` returns an object with the
extension's three functions (``decode_fwd``, ``decode_bwd``, ``wht_scale``, same
arguments), so code written against the reference's extension runs unchanged.  The
calls never wait for the device: a group row outside the latent is skipped by the
kernels (nothing read or written; its byte gradients are 0) instead of being checked on
the host.

The stored values equal the torch graph of ``hi2.qad.FakeQuantLinear._group`` bit for
bit; the latent gradients too; the per-block byte gradients are sums in the reference
kernel's pairwise-tree order, and the transform is the reference kernel's butterfly.
``HI2_QAD_BACKEND=torch`` makes :func:`available` False (the caller then runs its own
torch graph, as in the reference); ``=kernel`` makes a missing library an error.
"""

import ctypes
import os

import torch

from . import _lib
from .gptq_kernel import kernel_dir, supported  # noqa: F401  (re-exported as in the reference)


def _check(t: torch.Tensor, dtype: torch.dtype, name: str) -> None:
    if not t.is_contiguous() or t.dtype != dtype:
        raise RuntimeError(f"{name} must be contiguous {dtype}")


def _full(t: torch.Tensor | None):
    """None in the place of an empty tensor (an absent vector, on whatever device it is)."""
    return None if t is None or t.numel() == 0 else t


def _opt(t: torch.Tensor | None):
    return _lib.ptr(_full(t))


def _group_args(latent, unit, lo_u, st_u, consts, rows, block):
    _check(latent, torch.float32, "latent")
    _check(lo_u, torch.float32, "lo_u")
    _check(st_u, torch.float32, "st_u")
    _check(consts, torch.float16, "consts")
    _check(rows, torch.int64, "rows")
    if unit is not None and unit.numel():
        _check(unit, torch.float32, "unit")
        if unit.shape != latent.shape:
            raise RuntimeError("unit must have the latent's shape")
    k, n = latent.shape[1], rows.shape[0]
    if block not in (16, 32, 64):
        raise RuntimeError("block must be 16, 32 or 64")
    if k % block or tuple(lo_u.shape) != (n, k // block) or tuple(st_u.shape) != (n, k // block):
        raise RuntimeError("lo_u / st_u must be [rows, K / block]")
    if tuple(consts.shape) != (n, 3):
        raise RuntimeError("consts must be [rows, 3]")
    return k, n


def _transform_args(flags, scale, k):
    """The rotation flags and smoothing vector as pointers, checked as ``wht_scale`` checks
    them (None without a transform)."""
    if flags is None:
        return None, None
    _check(flags, torch.uint8, "flags")
    if k % 16 or flags.numel() != k // 16:
        raise RuntimeError("K must be a multiple of 16 with one flag per 16 columns")
    if scale is not None and scale.numel():
        _check(scale, torch.float16, "scale")
        if scale.numel() != k:
            raise RuntimeError("scale must have K entries")
    return _lib.ptr(flags), _opt(scale)


def _group_table(latent, unit, meta, params, grads=None):
    """The groups of a tensor as the library's array (and its width), each checked as
    ``decode_fwd`` checks it; ``grads``: the byte gradients ``[lo, st]`` of every group."""
    tab = (_lib.QadGroup * max(len(meta), 1))()
    for gi, (rows, consts, nbits, block) in enumerate(meta):
        lo_u, st_u = params[2 * gi], params[2 * gi + 1]
        _lib.require_gpu(latent, lo_u, st_u, consts, rows)
        _, n = _group_args(latent, unit, lo_u, st_u, consts, rows, block)
        tab[gi] = _lib.QadGroup(
            lo_u.data_ptr(), st_u.data_ptr(), consts.data_ptr(), rows.data_ptr(), n, int(block),
            float(2 ** nbits - 1), *((g.data_ptr() for g in grads[2 * gi:2 * gi + 2])
                                     if grads else (None, None)))
    return tab


class _Kernels:
    """The three functions of the reference's extension (``hi2/qad_kernel.py:37-49``)."""

    @staticmethod
    def decode_fwd(latent, unit, lo_u, st_u, consts, rows, block, nmax, out):
        dev = _lib.require_gpu(latent, lo_u, st_u, consts, rows, out)
        k, n = _group_args(latent, unit, lo_u, st_u, consts, rows, block)
        _check(out, torch.float32, "out")
        if out.shape != latent.shape:
            raise RuntimeError("out must have the latent's shape")
        if n:
            _lib.call("hi2x_qad_decode_fwd", dev, _lib.ptr(latent), _opt(unit), _lib.ptr(lo_u),
                      _lib.ptr(st_u), _lib.ptr(consts), _lib.ptr(rows), n, latent.shape[0], k,
                      int(block), float(nmax), _lib.ptr(out))

    @staticmethod
    def decode_bwd(grad, latent, unit, lo_u, st_u, consts, rows, block, nmax, g_latent, g_lo,
                   g_st):
        dev = _lib.require_gpu(grad, latent, lo_u, st_u, consts, rows, g_latent, g_lo, g_st)
        k, n = _group_args(latent, unit, lo_u, st_u, consts, rows, block)
        for name, t in (("grad", grad), ("g_latent", g_latent), ("g_lo", g_lo), ("g_st", g_st)):
            _check(t, torch.float32, name)
        if grad.shape != latent.shape or g_latent.shape != latent.shape:
            raise RuntimeError("grad and g_latent must have the latent's shape")
        if g_lo.shape != lo_u.shape or g_st.shape != lo_u.shape:
            raise RuntimeError("g_lo / g_st must have the shape of lo_u")
        if n:
            _lib.call("hi2x_qad_decode_bwd", dev, _lib.ptr(grad), _lib.ptr(latent), _opt(unit),
                      _lib.ptr(lo_u), _lib.ptr(st_u), _lib.ptr(consts), _lib.ptr(rows), n,
                      latent.shape[0], k, int(block), float(nmax), _lib.ptr(g_latent),
                      _lib.ptr(g_lo), _lib.ptr(g_st))

    @staticmethod
    def wht_scale(x, flags, scale, pre_div, out):
        dev = _lib.require_gpu(x, flags, out)
        _check(x, torch.float32, "x")
        _check(out, torch.float32, "out")
        _check(flags, torch.uint8, "flags")
        n, k = x.shape
        if k % 16 or flags.numel() != k // 16:
            raise RuntimeError("K must be a multiple of 16 with one flag per 16 columns")
        if scale is not None and scale.numel():
            _check(scale, torch.float16, "scale")
            if scale.numel() != k:
                raise RuntimeError("scale must have K entries")
        if out.shape != x.shape:
            raise RuntimeError("out must have the shape of x")
        if n:
            _lib.call("hi2x_qad_wht_scale", dev, _lib.ptr(x), n, k, _lib.ptr(flags),
                      _opt(scale), int(bool(pre_div)), _lib.ptr(out))


_KERNELS = _Kernels()


def load():
    """The kernels (an object with ``decode_fwd``, ``decode_bwd``, ``wht_scale``), or None
    with :func:`failure` recorded."""
    if _lib.load() is None:
        if os.environ.get("HI2_QAD_BACKEND") == "kernel":
            raise RuntimeError(f"hi2x library unavailable: {_lib.failure()}")
        return None
    return _KERNELS


def available(dev: torch.device) -> bool:
    backend = os.environ.get("HI2_QAD_BACKEND", "auto")
    if backend == "torch":
        return False
    ok = supported(dev) and load() is not None
    if backend == "kernel" and not ok:
        raise RuntimeError(f"qad kernel unavailable on {dev}: {_lib.failure()}")
    return ok


def failure() -> str | None:
    return _lib.failure()


def _mod():
    mod = load()
    if mod is None:
        raise RuntimeError(f"hi2x library unavailable: {_lib.failure()}")
    return mod


def _decode(latent, unit, meta, flags, scale, params, out) -> None:
    """Every group's rows of ``out``: the stored values, or with ``flags`` the weights in the
    model's basis, in one call."""
    _mod()
    if not meta:
        return
    tab = _group_table(latent, unit, meta, params)
    fl, sc = _transform_args(flags, scale, latent.shape[1])
    _lib.call("hi2x_qad_weights_fwd", _lib.require_gpu(latent, out, flags, _full(scale)),
              _lib.ptr(latent), _opt(unit), ctypes.cast(tab, ctypes.c_void_p), len(meta),
              latent.shape[0], latent.shape[1], fl, sc, _lib.ptr(out))


def _decode_grads(ctx, grad, flags, scale):
    """The latent's gradient and every group's byte gradients."""
    latent, unit, *params = ctx.saved_tensors
    _mod()
    grad = grad.contiguous()
    g_latent = torch.empty_like(latent)
    grads = [torch.empty_like(p) for p in params]
    if ctx.meta:
        _check(grad, torch.float32, "grad")
        if grad.shape != latent.shape:
            raise RuntimeError("grad must have the latent's shape")
        tab = _group_table(latent, unit, ctx.meta, params, grads)
        fl, sc = _transform_args(flags, scale, latent.shape[1])
        _lib.call("hi2x_qad_weights_bwd", _lib.require_gpu(grad, latent, flags, _full(scale)),
                  _lib.ptr(grad), _lib.ptr(latent), _opt(unit), ctypes.cast(tab, ctypes.c_void_p),
                  len(ctx.meta), latent.shape[0], latent.shape[1], fl, sc, _lib.ptr(g_latent))
    return g_latent, grads


class _StoredDecode(torch.autograd.Function):
    """``stored = decode(latent, unit, ladder bytes)`` over all groups of one tensor."""

    @staticmethod
    def forward(ctx, latent, unit, meta, *params):
        out = torch.empty_like(latent)
        _decode(latent, unit, meta, None, None, params, out)
        ctx.meta = meta
        ctx.save_for_backward(latent, unit, *params)
        return out

    @staticmethod
    def backward(ctx, grad):
        g_latent, grads = _decode_grads(ctx, grad, None, None)
        return (g_latent, None, None, *grads)


class _Transform(torch.autograd.Function):
    """``H(x) / scale`` over the flagged 16-column groups; the backward is ``H(grad / scale)``.
    :func:`original` fuses it with the decode (``_Weights``); it is here for code written against
    the reference's module."""

    @staticmethod
    def forward(ctx, x, flags, scale):
        out = torch.empty_like(x)
        _mod().wht_scale(x.contiguous(), flags, scale, False, out)
        ctx.flags, ctx.scale = flags, scale
        return out

    @staticmethod
    def backward(ctx, grad):
        out = torch.empty_like(grad)
        _mod().wht_scale(grad.contiguous(), ctx.flags, ctx.scale, True, out)
        return out, None, None


class _Weights(torch.autograd.Function):
    """``_Transform`` of ``_StoredDecode`` in one pass per group and direction."""

    @staticmethod
    def forward(ctx, latent, unit, meta, flags, scale, *params):
        out = torch.empty_like(latent)
        _decode(latent, unit, meta, flags, scale, params, out)
        ctx.meta, ctx.flags, ctx.scale = meta, flags, scale
        ctx.save_for_backward(latent, unit, *params)
        return out

    @staticmethod
    def backward(ctx, grad):
        g_latent, grads = _decode_grads(ctx, grad, ctx.flags, ctx.scale)
        return (g_latent, None, None, None, None, *grads)


def _groups(fq):
    return ([(g.rows, g.consts, g.nbits, g.block) for g in fq.groups],
            [p for g in fq.groups for p in (g.lo_u, g.step_u)])


def _values(fq, meta, params, flags, scale) -> torch.Tensor:
    with torch.no_grad():
        out = torch.empty_like(fq.latent)
        _decode(fq.latent.detach(), fq.unit, meta, flags, scale, [p.detach() for p in params],
                out)
        return out


def original(fq) -> torch.Tensor:
    """The weights of a fake-quantised Linear in the model's own basis, with the STE graph:
    the stored values, then the rotation of the flagged groups and the division by the
    smoothing vector, fused with the decode."""
    if not fq.has_had and not fq.has_scale:
        return stored(fq, True)
    meta, params = _groups(fq)
    scale = fq.col_scale if fq.has_scale else fq.col_scale[:0]
    if torch.is_grad_enabled():
        return _Weights.apply(fq.latent, fq.unit, meta, fq.had, scale, *params)
    return _values(fq, meta, params, fq.had, scale)


def stored(fq, grad: bool) -> torch.Tensor:
    """The stored-basis weights of a fake-quantised Linear (rows in the tensor's own order),
    with the STE graph when ``grad``."""
    meta, params = _groups(fq)
    if grad and torch.is_grad_enabled():
        return _StoredDecode.apply(fq.latent, fq.unit, meta, *params)
    return _values(fq, meta, params, None, None)
