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


def combine_bwd(a, b, c, w, do, return_delta=False, all_below=0, slc_lse=None, swa_lse=None, helper=None):
    """Returns da, db, dc (contiguous [T,H,D]), dw [T,H,3] and optionally delta [3,T,H] fp32 with
    delta[k] = rowsum(branch_k * d branch_k), which the attention backward kernels consume.
    all_below > 0 (b = selected, c = window branch, with their log-sum-exps [T,H] and the batch's helper; needs
    return_delta): for the tokens at positions below it, which select every block they can see, dc and delta[2] also
    carry the selected branch's gradient over the window's keys (swa_bwd_dq_tail, slc_attn_bwd_dkdv_before_window take
    the rest)."""
    T, H, D = a.shape
    assert a.stride() == b.stride() == c.stride()
    do = do if do.stride(-1) == 1 else do.contiguous()
    da = torch.empty(T, H, D, device=a.device, dtype=a.dtype)
    db = torch.empty_like(da)
    dc = torch.empty_like(da)
    dw = torch.empty(T, H, 3, device=a.device, dtype=w.dtype)
    delta = torch.empty(3, T, H, device=a.device, dtype=torch.float32) if return_delta else None
    tail = ()
    name = "nsa_combine_bwd"
    if all_below > 0:
        assert slc_lse.stride() == swa_lse.stride() and return_delta
        name = "nsa_combine_bwd_tail"
        tail = (slc_lse.data_ptr(), swa_lse.data_ptr(), slc_lse.stride(0), slc_lse.stride(1),
                helper.x_cu_seqlens.data_ptr(), helper.batch, all_below)
    _lib.call(name, a.data_ptr(), b.data_ptr(), c.data_ptr(), a.stride(0), a.stride(1), w.data_ptr(),
              w.stride(0), w.stride(1), do.data_ptr(), do.stride(0), do.stride(1), da.data_ptr(), db.data_ptr(),
              dc.data_ptr(), dw.data_ptr(), _lib.ptr(delta), *tail, T, H, D, _lib.stream_ptr())
    if return_delta:
        return da, db, dc, dw, delta
    return da, db, dc, dw


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
