"""Compressed attention (upstream flash_nsa/ops/compress_attn.py:531-776)."""
import torch

from .. import _lib
from ..utils import NSAHelper
from . import bwd_ds
from ._common import check_thd, default_scale, delta_of, dq_target, zeros_pair


def cmp_attn_fwd(q, k, v, sm_scale=None, helper=NSAHelper):
    """q [T,QH,D], k [y_len,KH,D], v [y_len,KH,VD] (compressed rows) -> o [T,QH,VD], lse [QH,T] fp32 (log2 units).
    Query t sees compressed row i iff t >= stride*i + kernel-1; rows that see nothing give o = 0, lse = 0."""
    check_thd(q, "q"), check_thd(k, "k"), check_thd(v, "v")
    T, QH, D = q.shape
    Y, KH, VD = v.shape
    assert k.shape == (Y, KH, D) and QH % KH == 0 and Y == helper.y_len
    sm_scale = default_scale(q, sm_scale)
    o = torch.empty(T, QH, VD, device=q.device, dtype=q.dtype)
    lse = torch.empty(QH, T, device=q.device, dtype=torch.float32)
    _lib.call("nsa_cmp_attn_fwd", q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1),
              v.data_ptr(), v.stride(0), v.stride(1), o.data_ptr(), o.stride(0), o.stride(1), lse.data_ptr(),
              lse.stride(1), lse.stride(0), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(),
              helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.kernel_size, helper.stride, sm_scale,
              _lib.stream_ptr())
    return o, lse


# most scratch for the partial dk / dv of the compressed branch.  Its size grows with the square of the sequence length,
# and slots and their sum are faster than atomic additions only where it is small (d = 128, MB, us with slots / atomics:
# 64 q / 4 kv heads, 2K tokens 16 MB 57 / 62, 4K 48 MB 110 / 120, 8K 80 MB 275 / 277, 16K 144 MB 815 / 813, 8 x 4K-8K 160 MB
# 1592 / 1592; 16 q / 1 kv heads, 8K 40 MB 100 / 120, 16K 72 MB 255 / 276, 32K 136 MB 781 / 792).
DKDV_SLOTS_LIMIT = 80 << 20


def cmp_attn_bwd(q, k, v, o, lse, do, dq=None, dkdv_repeat=False, sm_scale=None, helper=NSAHelper, delta=None,
                 q_chunk_tokens=0, finalize_dq=False, parts="both", finalize_below=None):
    """Backward of compressed attention.  Returns (dq, dk, dv).
    dq: fresh bf16 tensor, or the caller's fp32 buffer, which is added into; with finalize_dq the fp32 buffer is
    only read and the returned dq is a fresh tensor in q's dtype holding buffer + this branch.  finalize_below (with
    finalize_dq): a tensor of q's dtype and n; that sum is for the queries at positions below n stored there, for the others
    kept in the buffer.
    parts = "dq" / "dkdv" launches only that kernel (the other results are None); "both" forms dq from the dS that the dk / dv
    kernel leaves behind where the shapes have that path (bwd_ds: up to 4 GB of scratch).
    dk, dv: fp32 [y_len,KH,*].  Every work item (query chunk of a key tile) stores its partial result into its own slot
    of a scratch buffer and a second launch sums the slots in a fixed order -- bit-identical results across runs.
    Where the slots would take more than DKDV_SLOTS_LIMIT bytes and neither dkdv_repeat nor
    NSAHelper.set_deterministic(True) asks for that order, the work items add with fp32 atomics instead.
    delta may be passed when already known (delta[T,QH] fp32 = rowsum(o*do)).
    q_chunk_tokens: queries per work item of the dk/dv kernel (0: chosen by the library from the sizes)."""
    check_thd(do, "do")
    T, QH, D = q.shape
    Y, KH, VD = v.shape
    sm_scale = default_scale(q, sm_scale)
    if delta is None:
        delta = delta_of(o, do)
    if parts == "both" and not (finalize_dq or dkdv_repeat or q_chunk_tokens) and bwd_ds.takes(q, k, v, do, sm_scale, helper):
        ds, sums = bwd_ds.DenseDs(q, k, helper, with_swa=False), ()
        if ds.fits:
            dq_buf, mode = dq_target(q, dq)
            for r in ds.ranges:
                sums = ds.dkdv_cmp(r, q, k, v, lse, do, delta, sm_scale, *sums)
                ds.dq(r, k, None, VD, sm_scale, dq_buf, mode)
            return (dq_buf, *sums)
    common = (q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(),
              v.stride(0), v.stride(1), do.data_ptr(), do.stride(0), do.stride(1), lse.data_ptr(), lse.stride(1),
              lse.stride(0), delta.data_ptr(), delta.stride(0), delta.stride(1))
    tail = (helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH,
            D, VD, helper.kernel_size, helper.stride, sm_scale, _lib.stream_ptr())
    dq_buf = dk = dv = None
    if parts in ("both", "dq"):
        if finalize_dq:
            # last branch of a fused backward: dq (fp32 sum of the other branches) + this branch -> fresh tensor in
            # q's dtype
            assert dq is not None and dq.dtype == torch.float32 and dq.shape == q.shape and dq.stride(-1) == 1
            bufs = lambda out: (dq.data_ptr(), dq.stride(0), dq.stride(1), out.data_ptr(), out.stride(0), out.stride(1))
            if finalize_below is not None:
                dq_buf, below = finalize_below
                _lib.call("nsa_cmp_attn_bwd_dq_final_below", *common, *bufs(dq_buf), below, *tail)
            else:
                dq_buf = torch.empty_like(q)
                _lib.call("nsa_cmp_attn_bwd_dq_final", *common, *bufs(dq_buf), *tail)
        else:
            dq_buf, mode = dq_target(q, dq)
            _lib.call("nsa_cmp_attn_bwd_dq", *common, dq_buf.data_ptr(), dq_buf.stride(0), dq_buf.stride(1), mode,
                      *tail)
    if parts in ("both", "dkdv"):
        sizes = (helper.batch, helper.x_maxlen, helper.y_maxlen, QH, KH, D, VD, helper.kernel_size, helper.stride,
                 q_chunk_tokens)
        need = _lib.value("nsa_cmp_attn_bwd_dkdv_det_bytes", *sizes)
        slots = dkdv_repeat or getattr(helper, "deterministic", False) or need <= DKDV_SLOTS_LIMIT
        if slots:
            dk = torch.empty(Y, KH, D, device=q.device, dtype=torch.float32)
            dv = torch.empty(Y, KH, VD, device=q.device, dtype=torch.float32)
        else:
            dk, dv = zeros_pair((Y, KH, D), (Y, KH, VD), q.device)
        args = (*common, dk.data_ptr(), dk.stride(0), dk.stride(1), dv.data_ptr(), dv.stride(0), dv.stride(1),
                helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), *sizes, sm_scale)
        if slots:
            ws = torch.empty(max(need, 1), dtype=torch.uint8, device=q.device)
            _lib.call("nsa_cmp_attn_bwd_dkdv_det", *args, ws.data_ptr(), ws.numel(), _lib.stream_ptr())
        else:
            _lib.call("nsa_cmp_attn_bwd_dkdv", *args, _lib.stream_ptr())
    return dq_buf, dk, dv


class _CompressAttn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, sm_scale):
        o, lse = cmp_attn_fwd(q, k, v, sm_scale)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.sm_scale = sm_scale
        ctx.helper = NSAHelper.get_bwd_helper()
        ctx.mark_non_differentiable(lse)
        return o, lse

    @staticmethod
    def backward(ctx, do, _dlse):
        q, k, v, o, lse = ctx.saved_tensors
        do = do if do.stride(-1) == 1 else do.contiguous()
        dq, dk, dv = cmp_attn_bwd(q, k, v, o, lse, do, sm_scale=ctx.sm_scale, helper=ctx.helper)
        return dq, dk.to(k.dtype), dv.to(v.dtype), None


def compress_attn(q, k, v, sm_scale=None):
    """Differentiable compressed attention -> (o, lse)."""
    return _CompressAttn.apply(q, k, v, sm_scale)
