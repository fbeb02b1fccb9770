"""Shared launch path for the dense-embedding MaxSim entry points.

Every public scoring function (``maxsim``, ``maxsim_pairs``, ``maxsim_varlen``,
``maxsim_padded``, ``score_pairs_packed``, ``maxsim_inference_fp8``,
``retrieve``) normalises its inputs here and calls ``lik_maxsim`` /
``lik_maxsim_pairs`` from liblik_hip.so.
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib

_FP8 = getattr(torch, "float8_e4m3fn", None)


def unify_dtype(Q: torch.Tensor, D: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Pick one compute dtype for Q and D.

    bf16 if either side is bf16 (the reference's rule, ``_utils.py:137-148``),
    fp16 if both are fp16, otherwise fp32. fp32 is computed as a three-term
    bf16 split on the MFMA units (about 16 mantissa bits per product), where
    the reference truncates fp32 to fp16.
    """
    if Q.dtype == _FP8 or D.dtype == _FP8:
        raise TypeError("fp8 inputs go through late_interaction_kernels.fp8.maxsim_inference_fp8")
    if not (Q.is_floating_point() and D.is_floating_point()):
        raise TypeError(f"Q and D must be floating point; got {Q.dtype} and {D.dtype}")
    if torch.bfloat16 in (Q.dtype, D.dtype):
        t = torch.bfloat16
    elif Q.dtype == torch.float16 and D.dtype == torch.float16:
        t = torch.float16
    else:
        t = torch.float32
    return Q.to(t), D.to(t)


def _mask_i8(m: torch.Tensor | None, shape: tuple[int, int]) -> torch.Tensor | None:
    """Keep flags as int8 for the kernels, which read ``mask[i * sn + t * sl] != 0``
    with the tensor's own strides: a bool / 8-bit mask is reinterpreted in place
    (no copy, broadcast strides kept); other dtypes become ``m != 0``."""
    if m is None:
        return None
    if tuple(m.shape) != tuple(shape):
        m = m.expand(shape)
    if m.dtype == torch.int8:
        return m
    if m.dtype in (torch.bool, torch.uint8):
        return m.view(torch.int8)
    return (m != 0).view(torch.int8)


def _i32(t: torch.Tensor | None) -> torch.Tensor | None:
    return None if t is None else t.to(torch.int32).contiguous()


def dense_maxsim(
    Q: torch.Tensor,
    D: torch.Tensor,
    q_mask: torch.Tensor | None = None,
    d_mask: torch.Tensor | None = None,
    *,
    normalize: bool = False,
    norm: int | None = None,
    kd: bool = False,
    q_lengths: torch.Tensor | None = None,
    d_lengths: torch.Tensor | None = None,
    q_scale: torch.Tensor | None = None,
    d_scale: torch.Tensor | None = None,
    out_scale: float = 1.0,
) -> torch.Tensor:
    """``Q[Nq, Lq, d]`` x ``D[Nd, Ld, d]`` -> ``[Nq, Nd]`` fp32 (KD: ``D[Nq*K, Ld, d]`` -> ``[Nq, K]``).

    Masks are ``[N, L]`` keep-flags; lengths are valid prefix lengths per
    sequence; scales are fp8 per-token dequant scales ``[N, L]``.
    """
    _lib.require_gpu(Q, D, q_mask, d_mask, q_lengths, d_lengths, q_scale, d_scale)
    Nq, Lq, _ = Q.shape
    Nd, Ld, _ = D.shape
    Nd_eff = (Nd // Nq if Nq else 0) if kd else Nd
    out = torch.empty(Nq, Nd_eff, device=Q.device, dtype=torch.float32)
    if Nq == 0 or Nd_eff == 0:
        return out
    if Lq == 0 or Ld == 0:
        return out.zero_()
    Q = _lib.prepare_tokens(Q)
    D = _lib.prepare_tokens(D)
    qm = _mask_i8(q_mask, (Nq, Lq))
    dm = _mask_i8(d_mask, (Nd, Ld))
    ql = _i32(q_lengths)
    dl = _i32(d_lengths)
    # a 0-d scale is one per-tensor scale (strides 0: the kernel folds it
    # into the score scale); [N, L] scales are per token
    qsc = None if q_scale is None else (q_scale.to(torch.float32).reshape(1, 1) if q_scale.dim() == 0
                                        else q_scale.to(torch.float32).expand(Nq, Lq).contiguous())
    dsc = None if d_scale is None else (d_scale.to(torch.float32).reshape(1, 1) if d_scale.dim() == 0
                                        else d_scale.to(torch.float32).expand(Nd, Ld).contiguous())
    qs = _lib.seqs(
        Q, n=Nq, length=Lq, stride_n=Q.stride(0), stride_l=Q.stride(1), lengths=ql, mask=qm,
        mask_strides=(qm.stride(0), qm.stride(1)) if qm is not None else (0, 0),
        token_scale=qsc, scale_strides=(qsc.stride(0), qsc.stride(1)) if qsc is not None and qsc.numel() > 1 else (0, 0),
    )
    ds = _lib.seqs(
        D, n=Nd, length=Ld, stride_n=D.stride(0), stride_l=D.stride(1), lengths=dl, mask=dm,
        mask_strides=(dm.stride(0), dm.stride(1)) if dm is not None else (0, 0),
        token_scale=dsc, scale_strides=(dsc.stride(0), dsc.stride(1)) if dsc is not None and dsc.numel() > 1 else (0, 0),
    )
    if norm is None:
        norm = 3 if normalize else 0
    flags = _lib.norm_flags(norm) | (_lib.LIK_KD_LAYOUT if kd else 0)
    _launch(qs, ds, flags, out_scale, out, Q.device)
    return out


def dense_maxsim_train(
    Q: torch.Tensor,
    D: torch.Tensor,
    q_mask: torch.Tensor | None,
    d_mask: torch.Tensor | None,
    *,
    norm: int,
    kd: bool,
):
    """Training forward: scores plus the saved state the backward needs.
    ``norm`` is a bitmask: 1 normalises query tokens, 2 doc tokens.

    Returns ``(scores, argmax, Qp, Dp, qm)``: ``argmax`` is ``[Nq * docs, Lq]``
    int32 (winning doc-token index, -1 for rows without a valid doc token);
    ``Qp`` / ``Dp`` are the kernel-ready (16-byte-row) copies of Q and D and
    ``qm`` the int8 query mask.
    """
    _lib.require_gpu(Q, D, q_mask, d_mask)
    Nq, Lq, _ = Q.shape
    Nd, Ld, _ = D.shape
    docs = (Nd // Nq if Nq else 0) if kd else Nd
    out = torch.empty(Nq, docs, device=Q.device, dtype=torch.float32)
    argmax = torch.empty((Nq * docs, Lq), device=Q.device, dtype=torch.int32)  # every entry is written
    Qp = _lib.prepare_tokens(Q.detach())
    Dp = _lib.prepare_tokens(D.detach())
    qm = _mask_i8(q_mask, (Nq, Lq))
    if Nq == 0 or docs == 0 or Lq == 0 or Ld == 0:
        return out.zero_(), argmax.fill_(-1), Qp, Dp, qm
    dm = _mask_i8(d_mask, (Nd, Ld))
    qs = _lib.seqs(Qp, n=Nq, length=Lq, stride_n=Qp.stride(0), stride_l=Qp.stride(1), mask=qm,
                   mask_strides=(qm.stride(0), qm.stride(1)) if qm is not None else (0, 0))
    ds = _lib.seqs(Dp, n=Nd, length=Ld, stride_n=Dp.stride(0), stride_l=Dp.stride(1), mask=dm,
                   mask_strides=(dm.stride(0), dm.stride(1)) if dm is not None else (0, 0))
    flags = _lib.norm_flags(norm) | (_lib.LIK_KD_LAYOUT if kd else 0)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_workspace_size(ctypes.byref(qs), ctypes.byref(ds), flags)
    ws = _lib.workspace(nbytes, Q.device)
    with _lib.on_device(Q.device):
        rc = lib.lik_maxsim_argmax(ctypes.byref(qs), ctypes.byref(ds), flags, out.data_ptr(), out.stride(0),
                                   out.stride(1), argmax.data_ptr(), _lib.ptr(ws), nbytes, _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_argmax")
    return out, argmax, Qp, Dp, qm


def maxsim_backward(
    grad: torch.Tensor,
    Qp: torch.Tensor,
    Dp: torch.Tensor,
    argmax: torch.Tensor,
    qm: torch.Tensor | None,
    *,
    norm: int,
    kd: bool,
) -> tuple[torch.Tensor, torch.Tensor]:
    """``(grad_Q [Nq, Lq, dp], grad_D [Nd, Ld, dp])`` in the input dtype for upstream ``grad`` [Nq, docs]."""
    Nq, Lq, dp = Qp.shape
    Nd, Ld, _ = Dp.shape
    if Nq == 0 or Nd == 0 or Lq == 0 or Ld == 0:
        return torch.zeros_like(Qp), torch.zeros_like(Dp)
    gq = torch.empty(Nq, Lq, dp, device=Qp.device, dtype=Qp.dtype)  # every element is written
    gd = torch.empty(Nd, Ld, dp, device=Dp.device, dtype=Dp.dtype)
    g = grad.to(torch.float32).contiguous()
    qs = _lib.seqs(Qp, n=Nq, length=Lq, stride_n=Qp.stride(0), stride_l=Qp.stride(1), mask=qm,
                   mask_strides=(qm.stride(0), qm.stride(1)) if qm is not None else (0, 0))
    ds = _lib.seqs(Dp, n=Nd, length=Ld, stride_n=Dp.stride(0), stride_l=Dp.stride(1))
    flags = _lib.norm_flags(norm) | (_lib.LIK_KD_LAYOUT if kd else 0)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_backward_workspace_size(ctypes.byref(qs), ctypes.byref(ds), flags)
    ws = _lib.workspace(nbytes, Qp.device)
    with _lib.on_device(Qp.device):
        rc = lib.lik_maxsim_backward(g.data_ptr(), g.stride(0), ctypes.byref(qs), ctypes.byref(ds), argmax.data_ptr(),
                                     flags, gq.data_ptr(), gd.data_ptr(), _lib.ptr(ws), nbytes,
                                     _lib.stream_of(gq))
    _lib.check(rc, "lik_maxsim_backward")
    return gq, gd


def packed_maxsim(
    Q_packed: torch.Tensor,
    D_packed: torch.Tensor,
    cu_q: torch.Tensor,
    cu_d: torch.Tensor,
    max_q: int,
    max_d: int,
    *,
    normalize: bool = False,
) -> torch.Tensor:
    """Packed (cu_seqlens) Q and D -> ``[Nq, Nd]`` fp32."""
    _lib.require_gpu(Q_packed, D_packed, cu_q, cu_d)
    Nq = cu_q.numel() - 1
    Nd = cu_d.numel() - 1
    out = torch.empty(max(Nq, 0), max(Nd, 0), device=Q_packed.device, dtype=torch.float32)
    if Nq <= 0 or Nd <= 0:
        return out
    if max_q <= 0 or Q_packed.shape[0] == 0 or D_packed.shape[0] == 0:
        return out.zero_()
    Qp = _lib.prepare_tokens(Q_packed)
    Dp = _lib.prepare_tokens(D_packed)
    cq = _i32(cu_q)
    cd = _i32(cu_d)
    # max_d is not a kernel bound (each doc's tile loop ends at its own length)
    qs = _lib.seqs(Qp, n=Nq, length=max_q, stride_l=Qp.stride(0), cu=cq)
    ds = _lib.seqs(Dp, n=Nd, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cd)
    flags = _lib.LIK_NORMALIZE if normalize else 0
    _launch(qs, ds, flags, 1.0, out, Q_packed.device)
    return out


def packed_maxsim_train(Q_packed, D_packed, cu_q, cu_d, max_q: int, max_d: int):
    """Training forward on packed Q and D: ``(scores [Nq, Nd], argmax [Nq*Nd, max_q], Qp, Dp)``."""
    _lib.require_gpu(Q_packed, D_packed, cu_q, cu_d)
    Nq = cu_q.numel() - 1
    Nd = cu_d.numel() - 1
    out = torch.empty(max(Nq, 0), max(Nd, 0), device=Q_packed.device, dtype=torch.float32)
    argmax = torch.empty((max(Nq, 0) * max(Nd, 0), max(max_q, 0)), device=Q_packed.device, dtype=torch.int32)
    Qp = _lib.prepare_tokens(Q_packed.detach())
    Dp = _lib.prepare_tokens(D_packed.detach())
    if Nq <= 0 or Nd <= 0 or max_q <= 0 or Q_packed.shape[0] == 0 or D_packed.shape[0] == 0:
        return out.zero_(), argmax.fill_(-1), Qp, Dp
    qs = _lib.seqs(Qp, n=Nq, length=max_q, stride_l=Qp.stride(0), cu=cu_q)
    ds = _lib.seqs(Dp, n=Nd, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cu_d)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_workspace_size(ctypes.byref(qs), ctypes.byref(ds), 0)
    ws = _lib.workspace(nbytes, Q_packed.device)
    with _lib.on_device(Q_packed.device):
        rc = lib.lik_maxsim_argmax(ctypes.byref(qs), ctypes.byref(ds), 0, out.data_ptr(), out.stride(0),
                                   out.stride(1), argmax.data_ptr(), _lib.ptr(ws), nbytes, _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_argmax")
    return out, argmax, Qp, Dp


def packed_backward(grad, Qp, Dp, cu_q, cu_d, argmax, max_q: int, max_d: int, *, need_d: bool = True):
    """Gradients of packed MaxSim: ``(grad_Q [rows_q, dp], grad_D [rows_d, dp] or None)`` in the input dtype.
    Rows outside ``cu[0] .. cu[-1]`` are zero."""
    Nq = cu_q.numel() - 1
    Nd = cu_d.numel() - 1
    gq = torch.zeros_like(Qp)
    gd = torch.zeros_like(Dp) if need_d else None
    if Nq <= 0 or Nd <= 0 or max_q <= 0 or Qp.shape[0] == 0 or Dp.shape[0] == 0:
        return gq, gd
    g = grad.to(torch.float32).contiguous()
    qs = _lib.seqs(Qp, n=Nq, length=max_q, stride_l=Qp.stride(0), cu=cu_q)
    ds = _lib.seqs(Dp, n=Nd, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cu_d)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_backward_workspace_size(ctypes.byref(qs), ctypes.byref(ds), 0)
    ws = _lib.workspace(nbytes, Qp.device)
    with _lib.on_device(Qp.device):
        rc = lib.lik_maxsim_backward(g.data_ptr(), g.stride(0), ctypes.byref(qs), ctypes.byref(ds), argmax.data_ptr(),
                                     0, gq.data_ptr(), _lib.ptr(gd), _lib.ptr(ws), nbytes, _lib.stream_of(gq))
    _lib.check(rc, "lik_maxsim_backward")
    return gq, gd


def _launch(qs, ds, flags: int, out_scale: float, out: torch.Tensor, device: torch.device) -> None:
    lib = _lib.load()
    opts = _lib.call_opts()
    nbytes = lib.lik_maxsim_workspace_size_ex(ctypes.byref(qs), ctypes.byref(ds), flags, opts)
    ws = _lib.workspace(nbytes, device)
    with _lib.on_device(device):
        rc = lib.lik_maxsim_ex(
            ctypes.byref(qs), ctypes.byref(ds), flags, float(out_scale), out.data_ptr(), out.stride(0),
            out.stride(1), _lib.ptr(ws), nbytes, opts, _lib.stream_of(out),
        )
    _lib.check(rc, "lik_maxsim")


def pairs_maxsim(
    Q_packed: torch.Tensor,
    D_packed: torch.Tensor,
    cu_q: torch.Tensor,
    cu_d: torch.Tensor,
    pair_q: torch.Tensor,
    pair_d: torch.Tensor,
    max_q: int,
    max_d: int,
) -> torch.Tensor:
    """Pair-list MaxSim over packed Q and D -> ``[num_pairs]`` fp32."""
    _lib.require_gpu(Q_packed, D_packed, cu_q, cu_d, pair_q, pair_d)
    P = pair_q.numel()
    out = torch.empty(P, device=Q_packed.device, dtype=torch.float32)
    if P == 0:
        return out
    if max_q <= 0 or Q_packed.shape[0] == 0 or D_packed.shape[0] == 0:
        return out.zero_()
    Qp = _lib.prepare_tokens(Q_packed)
    Dp = _lib.prepare_tokens(D_packed)
    cq, cd, pq, pd = _i32(cu_q), _i32(cu_d), _i32(pair_q), _i32(pair_d)
    qs = _lib.seqs(Qp, n=cq.numel() - 1, length=max_q, stride_l=Qp.stride(0), cu=cq)
    ds = _lib.seqs(Dp, n=cd.numel() - 1, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cd)
    lib = _lib.load()
    with _lib.on_device(Q_packed.device):
        rc = lib.lik_maxsim_pairs(
            ctypes.byref(qs), ctypes.byref(ds), pq.data_ptr(), pd.data_ptr(), P, 0, out.data_ptr(),
            _lib.stream_of(out),
        )
    _lib.check(rc, "lik_maxsim_pairs")
    return out


def pairs_maxsim_train(Q_packed, D_packed, cu_q, cu_d, pair_q, pair_d, max_q: int, max_d: int):
    """Pair-list training forward: ``(scores [P], argmax [P, max_q], Qp, Dp)``."""
    _lib.require_gpu(Q_packed, D_packed, cu_q, cu_d, pair_q, pair_d)
    P = pair_q.numel()
    out = torch.empty(P, device=Q_packed.device, dtype=torch.float32)
    argmax = torch.empty((P, max(max_q, 0)), device=Q_packed.device, dtype=torch.int32)
    Qp = _lib.prepare_tokens(Q_packed.detach())
    Dp = _lib.prepare_tokens(D_packed.detach())
    if P == 0 or max_q <= 0 or Q_packed.shape[0] == 0 or D_packed.shape[0] == 0:
        return out.zero_(), argmax.fill_(-1), Qp, Dp
    qs = _lib.seqs(Qp, n=cu_q.numel() - 1, length=max_q, stride_l=Qp.stride(0), cu=cu_q)
    ds = _lib.seqs(Dp, n=cu_d.numel() - 1, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cu_d)
    lib = _lib.load()
    with _lib.on_device(Q_packed.device):
        rc = lib.lik_maxsim_pairs_argmax(ctypes.byref(qs), ctypes.byref(ds), pair_q.data_ptr(), pair_d.data_ptr(), P,
                                         0, out.data_ptr(), argmax.data_ptr(), _lib.stream_of(out))
    _lib.check(rc, "lik_maxsim_pairs_argmax")
    return out, argmax, Qp, Dp


def pairs_backward(grad, Qp, Dp, cu_q, cu_d, pair_q, pair_d, argmax, max_q: int, max_d: int, *,
                   need_d: bool = True):
    """Gradients of pair-list MaxSim: ``(grad_Q [rows_q, dp], grad_D [rows_d, dp] or None)``."""
    P = pair_q.numel()
    gq = torch.zeros_like(Qp)
    gd = torch.zeros_like(Dp) if need_d else None
    if P == 0 or max_q <= 0 or Qp.shape[0] == 0 or Dp.shape[0] == 0:
        return gq, gd
    g = grad.to(torch.float32).contiguous()
    qs = _lib.seqs(Qp, n=cu_q.numel() - 1, length=max_q, stride_l=Qp.stride(0), cu=cu_q)
    ds = _lib.seqs(Dp, n=cu_d.numel() - 1, length=max(int(max_d), 0), stride_l=Dp.stride(0), cu=cu_d)
    lib = _lib.load()
    nbytes = lib.lik_maxsim_pairs_backward_workspace_size(ctypes.byref(qs), ctypes.byref(ds), P)
    ws = _lib.workspace(nbytes, Qp.device)
    with _lib.on_device(Qp.device):
        rc = lib.lik_maxsim_pairs_backward(g.data_ptr(), ctypes.byref(qs), ctypes.byref(ds), pair_q.data_ptr(),
                                           pair_d.data_ptr(), P, argmax.data_ptr(), 0, gq.data_ptr(), _lib.ptr(gd),
                                           _lib.ptr(ws), nbytes, _lib.stream_of(gq))
    _lib.check(rc, "lik_maxsim_pairs_backward")
    return gq, gd


def seqlen_max(cu: torch.Tensor) -> int:
    """Longest sequence in ``cu_seqlens`` (one device->host sync)."""
    if cu.numel() <= 1:
        return 0
    return int((cu[1:] - cu[:-1]).max().item())


_COVER_MAX = 1 << 15  # sequences the one-workgroup check reads (more: torch's reductions)


def assert_max_seqlens_cover(*checks: tuple[torch.Tensor, int | None, str]) -> None:
    """On-device check that caller-supplied bounds cover every sequence of one or
    two ``cu_seqlens`` (``_utils.py:32-50``): a bound sizes the query block, so a
    too-small value would drop tokens. One kernel reads both arrays
    (``lik_seqlens_cover_each``), and each bound has its own assert; the
    differences, maximum and comparison as torch operators are three launches
    for each."""
    todo = [(cu, m, name) for cu, m, name in checks if m is not None and cu.numel() > 1]
    if not todo:
        return
    passed = None
    if (len(todo) <= 2 and sum(cu.numel() for cu, _, _ in todo) <= _COVER_MAX
            and all(cu.device == todo[0][0].device and cu.dtype == torch.int32 and cu.is_contiguous()
                    and abs(m) < 1 << 62 for cu, m, _ in todo)
            and _lib.plain_op(*(cu for cu, _, _ in todo))):
        ok = torch.empty(2, device=todo[0][0].device, dtype=torch.bool)
        (a, ma, _), (b, mb, _) = todo[0], todo[-1]
        with _lib.on_device(ok.device):
            rc = _lib.load().lik_seqlens_cover_each(a.data_ptr(), a.numel() - 1, ma, b.data_ptr(), b.numel() - 1, mb,
                                                    ok.data_ptr(), ok.data_ptr() + 1, _lib.stream_of(ok))
        _lib.check(rc, "lik_seqlens_cover_each")
        passed = ok.unbind(0)
    for k, (cu, m, name) in enumerate(todo):
        torch._assert_async(
            (cu[1:] - cu[:-1]).max().le(m) if passed is None else passed[k],
            f"{name}={m} is smaller than the longest sequence in cu_seqlens; "
            "it is a hard bound and would silently truncate tokens.",
        )


def from_hidden_forward(Q, H, W, b, d_mask, *, normalize: bool, want_argmax: bool):
    """Projection head fused into MaxSim (``lik_maxsim_from_hidden``): scores of
    ``Q [Nq, Lq, d_out]`` against ``normalize(H @ W^T + b)`` for ``H [Nd, Ld, d_model]``
    without forming the projected docs. Returns ``(scores, argmax or None)``, or
    ``None`` when the library reports the shape or dtype unsupported (the
    caller then projects first)."""
    _lib.require_gpu(Q, H, W, b, d_mask)
    if not (Q.dtype == H.dtype == W.dtype and Q.dtype in (torch.bfloat16, torch.float16)):
        return None
    Nq, Lq, d_out = Q.shape
    Nd, Ld, _ = H.shape
    # head_finish_kernel writes every score (and every argmax entry)
    out = torch.empty(Nq, Nd, device=Q.device, dtype=torch.float32)
    argmax = torch.empty((Nq * Nd, Lq), device=Q.device, dtype=torch.int32) if want_argmax else None
    Qc = Q.detach().contiguous()
    Hc = H.detach()
    if Hc.stride(-1) != 1 or Hc.data_ptr() % 16 or any(s % 8 for s in Hc.stride()[:-1]):
        Hc = Hc.contiguous()
    Wc = W.detach().contiguous()
    # a bias in the inputs' 16-bit dtype is read and widened by the kernel
    bias16 = b is not None and b.dtype == Q.dtype
    bias = None if b is None else (b.detach().contiguous() if bias16 else b.detach().to(torch.float32).contiguous())
    dm = _mask_i8(d_mask, (Nd, Ld))
    qs = _lib.seqs(Qc, n=Nq, length=Lq, stride_n=Qc.stride(0), stride_l=Qc.stride(1))
    hs = _lib.seqs(Hc, n=Nd, length=Ld, stride_n=Hc.stride(0), stride_l=Hc.stride(1), mask=dm,
                   mask_strides=(dm.stride(0), dm.stride(1)) if dm is not None else (0, 0))
    lib = _lib.load()
    nbytes = lib.lik_maxsim_from_hidden_workspace_size(ctypes.byref(qs), ctypes.byref(hs))
    ws = _lib.workspace(nbytes, Q.device)
    flags = (_lib.LIK_NORMALIZE_D if normalize else 0) | (_lib.LIK_BIAS_16 if bias16 else 0)
    with _lib.on_device(Q.device):
        rc = lib.lik_maxsim_from_hidden(ctypes.byref(qs), ctypes.byref(hs), Wc.data_ptr(), Wc.stride(0),
                                        _lib.ptr(bias), flags, out.data_ptr(), out.stride(0), out.stride(1),
                                        _lib.ptr(argmax), _lib.ptr(ws), nbytes, _lib.stream_of(out))
    if rc == _lib.LIK_ERR_UNSUPPORTED:
        return None
    _lib.check(rc, "lik_maxsim_from_hidden")
    return out, argmax



def head_backward(argmax, Nq: int, Lq: int, gd, H, W, *, need_h: bool, need_w: bool, need_b: bool):
    """Projection-head gradients (``lik_head_backward``): ``(grad_H, grad_W, grad_b fp32)``
    with ``None`` where not needed, or ``None`` for calls the kernels do not take
    (fp32, mixed dtypes, d_out > 128, d_model % 8, docs of more than 65536 tokens)."""
    Nd, Ld, d_model = H.shape
    dp, d_out = gd.shape[-1], W.shape[0]
    if not (H.dtype == W.dtype == gd.dtype and H.dtype in (torch.bfloat16, torch.float16)) or not _lib.plain_op(gd, H, W):
        return None
    lib = _lib.load()
    nbytes = lib.lik_head_backward_workspace_size(_lib.DTYPE_CODE[H.dtype], Nq, Lq, Nd, Ld, dp, d_out, d_model)
    if nbytes == 0 or gd.data_ptr() % 16:
        return None
    if H.stride(-1) != 1 or H.data_ptr() % 4 or any(s % 2 for s in H.stride()[:-1]):
        H = H.contiguous()
    if W.stride(-1) != 1 or W.data_ptr() % 16 or W.stride(0) % 8:
        W = W.contiguous()
    gh = torch.empty(H.shape, dtype=H.dtype, device=H.device) if need_h else None
    gw = torch.empty(W.shape, dtype=W.dtype, device=W.device) if need_w else None
    gb = torch.empty(d_out, dtype=torch.float32, device=W.device) if need_b else None
    hs = _lib.seqs(H, n=Nd, length=Ld, stride_n=H.stride(0), stride_l=H.stride(1))
    ws = _lib.workspace(nbytes, H.device)
    with _lib.on_device(H.device):
        rc = lib.lik_head_backward(argmax.data_ptr(), Nq, Lq, gd.data_ptr(), dp, ctypes.byref(hs), W.data_ptr(),
                                   W.stride(0), d_out, _lib.ptr(gh), _lib.ptr(gw), _lib.ptr(gb), _lib.ptr(ws), nbytes,
                                   _lib.stream_of(gd))
    if rc == _lib.LIK_ERR_UNSUPPORTED:
        return None
    _lib.check(rc, "lik_head_backward")
    return gh, gw, gb
