"""Sigmoid-gated sum of the three branch outputs (upstream flash_nsa/ops/combine.py:114-216)."""
import torch

from .. import _lib
from ._common import check_thd, check_bf16


def combine_fwd(a, b, c, w):
    """o = a*sigmoid(w[...,0]) + b*sigmoid(w[...,1]) + c*sigmoid(w[...,2]);  a,b,c [T,H,D], w [T,H,3]."""
    for t, n in ((a, "a"), (b, "b"), (c, "c")):
        check_thd(t, n)
    assert a.shape == b.shape == c.shape and a.stride() == b.stride() == c.stride()
    check_bf16(w)
    assert w.shape == (a.size(0), a.size(1), 3)
    T, H, D = a.shape
    o = torch.empty(T, H, D, device=a.device, dtype=a.dtype)
    _lib.call("nsa_combine_fwd", a.data_ptr(), b.data_ptr(), c.data_ptr(), a.stride(0), a.stride(1), w.data_ptr(),
              w.stride(0), w.stride(1), o.data_ptr(), o.stride(0), o.stride(1), T, H, D, _lib.stream_ptr())
    return o


def combine_bwd(a, b, c, w, do, return_delta=False):
    """Returns da, db, dc (contiguous [T,H,D]), dw [T,H,3] and optionally delta [3,T,H] fp32 with
    delta[k] = rowsum(branch_k * d branch_k), which the attention backward kernels consume."""
    T, H, D = a.shape
    assert a.stride() == b.stride() == c.stride()
    do = do if do.stride(-1) == 1 else do.contiguous()
    da = torch.empty(T, H, D, device=a.device, dtype=a.dtype)
    db = torch.empty_like(da)
    dc = torch.empty_like(da)
    dw = torch.empty(T, H, 3, device=a.device, dtype=w.dtype)
    delta = torch.empty(3, T, H, device=a.device, dtype=torch.float32) if return_delta else None
    _lib.call("nsa_combine_bwd", a.data_ptr(), b.data_ptr(), c.data_ptr(), a.stride(0), a.stride(1), w.data_ptr(),
              w.stride(0), w.stride(1), do.data_ptr(), do.stride(0), do.stride(1), da.data_ptr(), db.data_ptr(),
              dc.data_ptr(), dw.data_ptr(), _lib.ptr(delta), T, H, D, _lib.stream_ptr())
    if return_delta:
        return da, db, dc, dw, delta
    return da, db, dc, dw


def combine_bwd_gates(a, b, c, w, do, lse_b, lse_c, all_below, helper):
    """Backward of the gated sum for kernels of the selected branch b and the window branch c that read do itself: the
    gate of a branch goes into its log-sum-exp (lse_b, lse_c [T,H]).
    Returns da (the compressed branch's gradient), dw [T,H,3], delta [3,T,H] and lse [2,T,H] (fp32), which the branches'
    backward kernels take with do.
    For the tokens at positions below all_below, which select every block they can see, delta[2] and lse[1] also carry
    the selected branch's gradient over the window's keys (swa_bwd_dq_tail, slc_attn_bwd_dkdv_before_window take the
    rest)."""
    T, H, D = a.shape
    assert a.stride() == b.stride() == c.stride() and do.stride(-1) == 1
    da = torch.empty(T, H, D, device=a.device, dtype=a.dtype)
    dw = torch.empty(T, H, 3, device=a.device, dtype=w.dtype)
    delta, lse = torch.empty(5, T, H, device=a.device, dtype=torch.float32).split((3, 2))
    _lib.call("nsa_combine_bwd_gates", a.data_ptr(), b.data_ptr(), c.data_ptr(), a.stride(0), a.stride(1), w.data_ptr(),
              w.stride(0), w.stride(1), do.data_ptr(), do.stride(0), do.stride(1), lse_b.data_ptr(), lse_b.stride(0),
              lse_b.stride(1), lse_c.data_ptr(), lse_c.stride(0), lse_c.stride(1), da.data_ptr(), dw.data_ptr(),
              delta.data_ptr(), lse.data_ptr(), helper.x_cu_seqlens.data_ptr(), helper.batch, all_below, T, H, D,
              _lib.stream_ptr())
    return da, dw, delta, lse


class _Combine(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b, c, w):
        ctx.save_for_backward(a, b, c, w)
        return combine_fwd(a, b, c, w)

    @staticmethod
    def backward(ctx, do):
        a, b, c, w = ctx.saved_tensors
        return combine_bwd(a, b, c, w, do)


def fused_sigmoid_combine(a, b, c, w):
    return _Combine.apply(a, b, c, w)
