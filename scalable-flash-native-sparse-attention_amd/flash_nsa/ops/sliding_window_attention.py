"""Causal sliding-window attention over packed sequences (upstream
flash_nsa/ops/sliding_window_attention.py:26-157, which delegates to FlashAttention with window=(W,-1))."""
import torch

from .. import _lib
from ..utils import NSAHelper
from . import bwd_ds
from ._common import check_bf16, check_thd, default_scale, delta_of, dq_target


def swa_fwd(q, k, v, sm_scale=None, helper=NSAHelper):
    """-> o [T,QH,VD], lse [T,QH] fp32 in log2 units.  Query t attends keys max(0,t-W) .. t of its sequence."""
    check_thd(q, "q"), check_thd(k, "k"), check_thd(v, "v")
    T, QH, D = q.shape
    _, KH, VD = v.shape
    sm_scale = default_scale(q, sm_scale)
    o = torch.empty(T, QH, VD, device=q.device, dtype=q.dtype)
    lse = torch.empty(T, QH, device=q.device, dtype=torch.float32)
    _lib.call("nsa_swa_fwd", q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1),
              v.data_ptr(), v.stride(0), v.stride(1), o.data_ptr(), o.stride(0), o.stride(1), lse.data_ptr(),
              lse.stride(0), lse.stride(1), helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH, D,
              VD, helper.window_size, sm_scale, _lib.stream_ptr())
    return o, lse


def swa_fwd_tail(q, k, v, slc_o, slc_lse, all_below, cmp_o=None, w=None, store=True, sm_scale=None,
                 helper=NSAHelper):
    """swa_fwd, finishing the selected branch of the queries at positions below all_below (they select every block they
    can see: the window branch continued over the keys before it) into slc_o / slc_lse and, with cmp_o and the gates w,
    forming the gated sum of the three branches.  -> (o, lse, out or None); with store=False only `out` is defined."""
    for t, n in ((q, "q"), (k, "k"), (v, "v"), (slc_o, "slc_o")):
        check_thd(t, n)
    T, QH, D = q.shape
    _, KH, VD = v.shape
    sm_scale = default_scale(q, sm_scale)
    o = torch.empty(T, QH, VD, device=q.device, dtype=q.dtype)
    lse = torch.empty(T, QH, device=q.device, dtype=torch.float32) if store else None
    out = None
    if cmp_o is not None:
        check_thd(cmp_o, "cmp_o"), check_bf16(w)
        assert cmp_o.shape == o.shape and w.shape == (T, QH, 3)
        out = torch.empty_like(o)
    st = lambda t: (None, 0, 0) if t is None else (t.data_ptr(), t.stride(0), t.stride(1))
    _lib.call("nsa_swa_fwd_tail", *st(q), *st(k), *st(v), *st(o), *st(lse), *st(slc_o), *st(slc_lse), all_below,
              *st(cmp_o), *st(w), *st(out), int(store), helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen,
              QH, KH, D, VD, helper.window_size, sm_scale, _lib.stream_ptr())
    return o, lse, out


def short_fwd(q, k, v, cmp_k, cmp_v, w, all_below, store=True, sm_scale=None, helper=NSAHelper):
    """cmp_attn_fwd and swa_fwd_tail in one launch, for batches of sequences of at most all_below tokens (their queries select every
    block they can see) -> (cmp_o, cmp_lse), (slc_o, slc_lse), (swa_o, swa_lse), out; with store=False only out is defined."""
    for t, n in ((q, "q"), (k, "k"), (v, "v"), (cmp_k, "k"), (cmp_v, "v")):
        check_thd(t, n)
    check_bf16(w)
    T, QH, D = q.shape
    _, KH, VD = v.shape
    assert cmp_k.shape == (helper.y_len, KH, D) and cmp_v.shape == (helper.y_len, KH, VD) and QH % KH == 0
    assert w.shape == (T, QH, 3)
    new = lambda *shape: torch.empty(*shape, T, QH, VD, device=q.device, dtype=q.dtype)
    out = new()
    cmp_o, slc_o, swa_o = (new(), new(), new()) if store else new(3).unbind()
    cmp_lse = slc_lse = swa_lse = None
    if store:
        cmp_lse = torch.empty(QH, T, device=q.device, dtype=torch.float32)
        slc_lse, swa_lse = (torch.empty(T, QH, device=q.device, dtype=torch.float32) for _ in range(2))
    st = lambda t: (None, 0, 0) if t is None else (t.data_ptr(), t.stride(0), t.stride(1))
    lse_c = (None, 0, 0) if cmp_lse is None else (cmp_lse.data_ptr(), cmp_lse.stride(1), cmp_lse.stride(0))
    _lib.call("nsa_fwd_short", *st(q), *st(k), *st(v), *st(cmp_k), *st(cmp_v), *st(cmp_o), *lse_c, *st(swa_o), *st(swa_lse), *st(slc_o),
              *st(slc_lse), all_below, *st(w), *st(out), int(store), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(),
              helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.kernel_size, helper.stride, helper.window_size,
              default_scale(q, sm_scale), _lib.stream_ptr())
    return (cmp_o, cmp_lse), (slc_o, slc_lse), (swa_o, swa_lse), out


def slc_fwd_first_queries(q, k, v, slc_o, slc_lse, all_below, sm_scale=None, helper=NSAHelper):
    """What swa_fwd_tail does for the selected branch alone: slc_o / slc_lse of the queries at positions below all_below."""
    T, QH, D = q.shape
    _, KH, VD = v.shape
    st = lambda t: (t.data_ptr(), t.stride(0), t.stride(1))
    none = (None, 0, 0)
    _lib.call("nsa_swa_fwd_tail", *st(q), *st(k), *st(v), *none, *none, *st(slc_o), *st(slc_lse), all_below, *none, *none,
              *none, 1, helper.x_cu_seqlens.data_ptr(), helper.batch, min(helper.x_maxlen, all_below), QH, KH, D, VD,
              helper.window_size, default_scale(q, sm_scale), _lib.stream_ptr())


def swa_bwd_dq_tail(q, k, v, lse, do, delta, slc_lse, slc_do, slc_delta, all_below, dq, sm_scale=None,
                    helper=NSAHelper, store=False):
    """dq of the window branch added into (store: written to) the fp32 buffer dq.  lse, delta and slc_lse, slc_delta are
    combine_bwd_gates' (lse[1], delta[2] and lse[0], delta[1], with the gates in them), with the same all_below: the queries
    at positions below it also take the selected branch's keys before their window, and their dq is stored."""
    T, QH, D = q.shape
    _, KH, VD = v.shape
    st = lambda t: (t.data_ptr(), t.stride(0), t.stride(1))
    _lib.call("nsa_swa_bwd_dq_tail_store" if store else "nsa_swa_bwd_dq_tail", *st(q), *st(k), *st(v), *st(do), *st(lse),
              *st(delta), *st(slc_do), *st(slc_lse), *st(slc_delta), all_below, *st(dq), helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH,
              KH, D, VD, helper.window_size, default_scale(q, sm_scale), _lib.stream_ptr())


def dense_bwd_dq(q, k, v, lse, do, delta, slc_lse, slc_do, slc_delta, all_below, cmp_k, cmp_v, cmp_lse, cmp_do, cmp_delta, dq, dq32=None,
                 sm_scale=None, helper=NSAHelper):
    """dq of the compressed branch and of swa_bwd_dq_tail's in one launch: the queries at positions below all_below into dq (q's dtype),
    the others into the fp32 dq32 (None: there are none)."""
    T, QH, D = q.shape
    _, KH, VD = v.shape
    st = lambda t: (None, 0, 0) if t is None else (t.data_ptr(), t.stride(0), t.stride(1))
    _lib.call("nsa_bwd_dq_dense", *st(q), *st(k), *st(v), *st(do), *st(lse), *st(delta), *st(slc_do), *st(slc_lse), *st(slc_delta),
              all_below, *st(cmp_k), *st(cmp_v), *st(cmp_do), cmp_lse.data_ptr(), cmp_lse.stride(1), cmp_lse.stride(0), *st(cmp_delta),
              *st(dq), *st(dq32), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH,
              D, VD, helper.kernel_size, helper.stride, helper.window_size, default_scale(q, sm_scale), _lib.stream_ptr())
    return dq


def swa_bwd(q, k, v, o, lse, do, sm_scale=None, helper=NSAHelper, delta=None, dq=None, dkv_fp32=False, parts="both"):
    """Backward of the window branch.  Returns (dq, dk, dv); dq is a fresh bf16 tensor or the caller's fp32
    buffer (added into); dk/dv are fresh (bf16, or fp32 when dkv_fp32): one writer per element, or, for batches that do
    not fill the GPU, partial results added in a fixed order (up to 64 MB of scratch) -- bit-identical across runs.
    parts = "dq" / "dkdv" launches only that kernel (the other results are None), so that a caller can put the
    two on different streams; "both" forms dq from the dS that the dk / dv kernel leaves behind where the shapes have that
    path (bwd_ds: up to 4 GB of scratch for the dS and 512 MB for partial results)."""
    check_thd(do, "do")
    T, QH, D = q.shape
    _, KH, VD = v.shape
    sm_scale = default_scale(q, sm_scale)
    if delta is None:
        delta = delta_of(o, do)
    if parts == "both" and bwd_ds.takes(q, k, v, do, sm_scale, helper):
        ds = bwd_ds.DenseDs(q, k, helper, with_cmp=False)
        if ds.fits:
            dq_buf, mode = dq_target(q, dq)
            kv_dtype = torch.float32 if dkv_fp32 else k.dtype
            dk = torch.empty(T, KH, D, device=q.device, dtype=kv_dtype)
            dv = torch.empty(T, KH, VD, device=q.device, dtype=kv_dtype)
            for r in ds.ranges:
                ds.dkdv_swa(r, q, k, v, lse, do, delta, sm_scale, dk, dv)
                ds.dq(r, None, k, VD, sm_scale, dq_buf, mode)
            return dq_buf, dk, dv
    common = (q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(),
              v.stride(0), v.stride(1), do.data_ptr(), do.stride(0), do.stride(1), lse.data_ptr(), lse.stride(0),
              lse.stride(1), delta.data_ptr(), delta.stride(0), delta.stride(1))
    dq_buf = dk = dv = None
    if parts in ("both", "dq"):
        dq_buf, mode = dq_target(q, dq)
        _lib.call("nsa_swa_bwd_dq", *common, dq_buf.data_ptr(), dq_buf.stride(0), dq_buf.stride(1), mode,
                  helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.window_size,
                  sm_scale, _lib.stream_ptr())
    if parts in ("both", "dkdv"):
        kv_dtype = torch.float32 if dkv_fp32 else k.dtype
        dk = torch.empty(T, KH, D, device=q.device, dtype=kv_dtype)
        dv = torch.empty(T, KH, VD, device=q.device, dtype=kv_dtype)
        need = _lib.value("nsa_swa_bwd_dkdv_ws_bytes", helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.window_size)
        ws = torch.empty(need, device=q.device, dtype=torch.uint8) if need else None
        _lib.call("nsa_swa_bwd_dkdv_ws", *common, dk.data_ptr(), dk.stride(0), dk.stride(1), dv.data_ptr(),
                  dv.stride(0), dv.stride(1), int(dkv_fp32), helper.x_cu_seqlens.data_ptr(), helper.batch,
                  helper.x_maxlen, QH, KH, D, VD, helper.window_size, sm_scale, _lib.ptr(ws), need, _lib.stream_ptr())
    return dq_buf, dk, dv


class _SWA(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, sm_scale):
        o, lse = swa_fwd(q, k, v, sm_scale)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.sm_scale = sm_scale
        ctx.helper = NSAHelper.get_bwd_helper()
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse = ctx.saved_tensors
        do = do if do.stride(-1) == 1 else do.contiguous()
        dq, dk, dv = swa_bwd(q, k, v, o, lse, do, sm_scale=ctx.sm_scale, helper=ctx.helper)
        return dq, dk, dv, None


def swa_varlen_func(q, k, v, sm_scale=None):
    """Differentiable causal sliding-window attention over the registered packed batch."""
    return _SWA.apply(q, k, v, sm_scale)
