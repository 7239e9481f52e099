"""Megatron-level NSA core: the whole sparse attention as ONE autograd node with fp32 dq/dk/dv accumulation
across the three branches and optional recomputation of saved activations
(mirrors the interface of upstream flash_nsa/modules/megatron_level_nsa.py:46-159, 386-545; the
context-parallel function of that file is outside this single-GPU build)."""
import contextlib
import math

import torch

from ..config import NSAConfig, check_supported
from ..utils import NSAHelper
from ..ops._common import thd_rows
from ..ops.compress_kv import (compress_linear_fwd, compress_linear_bwd, construct_block_fwd, construct_block_bwd, mean_pooling_fwd,
                               mean_pooling_bwd, mean_pooling_bwd_sum, takes_weight)
from ..ops import bwd_ds
from ..ops.compress_attn import cmp_attn_fwd, cmp_attn_bwd
from ..ops.select_attn import (slc_attn_fwd, slc_attn_bwd, slc_attn_bwd_dkdv_before_window,
                               slc_bwd_ds_tokens, wait_for)
from ..ops.topk import slc_topk_indices
from ..ops.act import swiglu_fwd, swiglu_bwd, sigmoid_mul_fwd, sigmoid_mul_bwd
from ..ops.combine import combine_bwd_gates
from ..ops.sliding_window_attention import (short_fwd, slc_fwd_first_queries, swa_fwd, swa_fwd_tail, swa_bwd,
                                            swa_bwd_dq_tail, dense_bwd_dq)


# The backward runs on two streams, the dense dq kernels next to the dk/dv passes: batches that do not fill the GPU gain
# (eight samples of up to 2.8K tokens, 16 heads of 128: 1705 -> 1488 us; 64 heads, 4K tokens 1825 -> 1744), full ones neither
# gain nor lose (64K tokens 55.0 ms either way); the same split of the forward gained nothing.
# Setting this module attribute to False puts everything back on the caller's stream.
OVERLAP_STREAMS = True
# A second stream costs a small step 60 to 100 us of events, waits and first launches, of the host and of the GPU.  The second stream of
# small batches is therefore the caller's: of those whose tokens x q-heads x longest sequence (at most 2048: the window and the selected
# blocks end there) x channels (128 on top, for what does not grow with them) stay below this.  Whole steps on two streams / on one, us
# (this number, 1e9): 64 / 4 heads of 128, 1024 tokens 448 / 352 (26), 1500 586 / 538 (55), 2000 689 / 728 (98), 8 x 700 848 / 853 (96); 16
# / 1, 3000 571 / 472 (38), 4096 575 / 530 (52), 4 x 1500 498 to 580 / 541 (55), 6000 721 / 773 (75); 32 / 2 of 192, 1500 568 / 514 (32), 2000 618
# / 671 (57), 12 x 400 531 / 508 (28); 16 / 2 of 64, 4096 511 / 431 (34), 6000 541 / 566 (50), 9000 779 / 836 (75); 8 / 1 of 128, 6000 677 /
# 570 (38), 9000 766 / 798 (57).
# Shapes without a dk / dv pass that stores dS have longer kernels, and a lower line.  More than 128 channels, a fifth: 16 / 4 heads of
# 256, 4 x 500 429 / 422 (10), 12 x 400 787 / 828 (20); 20 / 4 of 192, 1024 403 / 341 (9.4), 12 x 400 412 / 423 (17), 1500 570 / 610 (20).
# Batches that select everything, two fifths above 64 channels: 24 / 8 of 128, 4 x 500 285 / 221 (9.2), 8 x 700 546 / 586 (36); 32 / 8, 12
# x 400 441 / 439 (24); the whole up to 64: 16 / 16 of 64, 8 x 700 395 / 331 (16); 8 / 8 of 32, 4 x 3000 with top_n 64 382 to 397 / 286 to
# 331 (38). Others, counted in whole groups of 16 q-heads, of which the kernels of the selected blocks are made, 1.78 times: 12 / 4 of 128
# (64 heads), 2000 596 / 558 (98), 3000 777 / 827 (151), 6000 1519 / 1629 (302); 8 / 8 of 32 (128 heads), 2000 528 / 445 (98), 3000 654 /
# 679 (151), 6000 1216 / 1257 (302); 12 / 2 of 64, 4096 549 / 508 (69), 6000 626 / 675 (101).
# Ordered sums, two ninths whatever the shape: 16 / 1 of 128, 12 x 400 383 / 334 (12), 1500 664 / 724 (14), 4096 857 / 915 (52); 8 / 1,
# 2000 527 / 526 (12), 3000 545 / 591 (19); 32 / 2 of 192, 1024 570 / 578 (15).
OVERLAP_FROM = 5.6e10
_side_streams = {}


def _gains_from_overlap(q, v, helper):
    T, QH, D = q.shape
    KH, VD = v.shape[1:]
    heads, line = QH, OVERLAP_FROM
    if getattr(helper, "deterministic", False):
        line /= 4.5
    elif QH // KH not in (8, 16, 32, 64) or (D, VD) not in ((64, 64), (128, 128), (192, 128)):
        if max(D, VD) > 128:
            line /= 5
        elif helper.x_maxlen <= helper.all_below():
            line *= 0.4 if max(D, VD) > 64 else 1
        else:
            heads, line = KH * 16 * -(-QH // KH // 16), line * 1.78
    return T * heads * min(helper.x_maxlen, 2048) * (D + VD + 128) >= line


def _side_stream(main, q, v, helper):
    """The second stream of this batch's backward beside the caller's, main."""
    if not _gains_from_overlap(q, v, helper):
        return main
    device = q.device
    key = device.index if device.index is not None else torch.cuda.current_device()
    s = _side_streams.get(key)
    if s is None:
        s = _side_streams[key] = torch.cuda.Stream(device=device)
    return s


def _on(side, main):
    return torch.cuda.stream(side) if side is not main else contextlib.nullcontext()


def weight_grad(inp, grad_out, weight):
    """dW = grad_out^T @ inp; accumulated into weight.main_grad (fp32) when the optimizer keeps one."""
    inp = inp.reshape(-1, inp.size(-1))
    grad_out = grad_out.reshape(-1, grad_out.size(-1))
    main_grad = getattr(weight, "main_grad", None)
    if main_grad is None:
        return torch.matmul(grad_out.t(), inp)
    # bf16 operands, fp32 accumulator added to the fp32 buffer in the GEMM's epilogue: no rounding of dW to bf16
    # (upstream's wgrad GEMM adds its fp32 accumulator tiles the same way, flash_nsa/ops/gemm.py:131-133)
    torch.addmm(main_grad, grad_out.t(), inp, out_dtype=torch.float32, out=main_grad)
    return _added_to_main_grad(weight, inp)


def _kernels_add_to(main_grad, weight):
    """Whether the kernels add dW to this buffer: they read and write four fp32 values at a time, and a view into the flat buffer of an
    optimizer may begin anywhere."""
    return (type(main_grad) in (torch.Tensor, torch.nn.Parameter) and main_grad.dtype == torch.float32 and
            main_grad.shape == weight.shape and main_grad.device == weight.device and main_grad.is_contiguous() and
            main_grad.data_ptr() % 16 == 0 and main_grad.data_ptr() != 0)


def _added_to_main_grad(weight, like):
    if hasattr(weight, "grad_added_to_main_grad"):
        weight.grad_added_to_main_grad = True
        return torch.empty(weight.main_grad.shape, dtype=like.dtype, device=like.device)
    return None


def _compress_fwd(x, weight, version, helper=NSAHelper, keep=True):
    """compress_kv_fwd without the windows where the kernels do not need them; keep=False: only the rows are asked for"""
    if version == "mean":
        return None, None, mean_pooling_fwd(x, helper=helper)
    if takes_weight(x, weight, version, helper):
        return (None, *compress_linear_fwd(x, weight, version, helper, keep))
    windows = construct_block_fwd(x, helper=helper)
    hidden = torch.matmul(windows.flatten(-2, -1), weight.t())
    if version == "linear":
        out = hidden
    elif version == "sigmoid-mul":
        out = sigmoid_mul_fwd(hidden)
    elif version == "swiglu":
        out = swiglu_fwd(hidden)
    else:
        raise ValueError(version)
    return windows, hidden, out


def compress_kv_fwd(x, weight, version, helper=NSAHelper):
    """-> (windows or None, pre-activation or None, compressed rows)"""
    windows, hidden, out = _compress_fwd(x, weight, version, helper)
    if windows is None and hidden is not None:
        windows = construct_block_fwd(x, helper=helper)
    return windows, hidden, out


def _compress_bwd(x, weight, windows, hidden, dout, dx, version, helper=NSAHelper):
    """For what _compress_fwd returned -> (bf16 sum of the compression gradient and the fp32 buffer dx, which may be overwritten, dW);
    dout: fp32."""
    if version == "mean":
        return mean_pooling_bwd_sum(x, dout, dx, helper), None
    if windows is None:
        main_grad = getattr(weight, "main_grad", None)
        if main_grad is not None and not _kernels_add_to(main_grad, weight):
            windows = construct_block_fwd(x, helper=helper)
        else:
            dx, dw = compress_linear_bwd(x, weight, hidden, dout, dx, version, main_grad, helper)
            return dx, dw if main_grad is None else _added_to_main_grad(weight, x)
    dx, dw = compress_kv_bwd(x, weight, windows, hidden, dout, dx, version, helper)
    return dx.to(x.dtype), dw


def compress_kv_bwd(x, weight, windows, hidden, dout, dx, version, helper=NSAHelper, async_dw=False):
    """Adds the compression gradient into the fp32 buffer dx and returns (dx, dW or a thunk computing it)."""
    dout = dout.to(x.dtype)
    if version == "mean":
        mean_pooling_bwd(x, dout, dx, helper=helper)
        return dx, None
    if version == "linear":
        dhidden = dout
    elif version == "sigmoid-mul":
        dhidden = sigmoid_mul_bwd(hidden, dout, inplace=False)
    else:
        dhidden = swiglu_bwd(hidden, dout, inplace=False)
    dwindows = torch.matmul(dhidden, weight).view(*windows.shape)
    construct_block_bwd(x, dwindows, dx, helper=helper)

    def dw_fn():
        return weight_grad(windows.flatten(-2, -1), dhidden, weight)

    return dx, (dw_fn if async_dw else dw_fn())


def slc_swa_fwd(q, k, v, topk, sm_scale, helper, cmp_o=None, w=None, store=True):
    """Selected and window branch, and, with the compressed branch's output and the gates, the gated sum: the gather of
    the queries that have blocks to choose from, then the window kernel, which finishes the rest.
    -> (slc_o, slc_lse), (swa_o, swa_lse), out; with store=False only out is defined."""
    all_below = helper.all_below()
    slc_o, slc_lse = slc_attn_fwd(q, k, v, topk, sm_scale=sm_scale, helper=helper, t_begin=all_below)
    swa_o, swa_lse, out = swa_fwd_tail(q, k, v, slc_o, slc_lse, all_below, cmp_o, w, store, sm_scale, helper)
    return (slc_o, slc_lse), (swa_o, swa_lse), out


def bwd_from_ds(ds, q, k, v, topk, cmp_k, cmp_v, do, dcmp_o, cmp_lse, lse_slc, lse_swa, delta, ds_tokens, sm_scale, helper):
    """The backward of the three branches where all of them leave their dS behind -> dq, dk, dv, dcmp_k, dcmp_v.
    ds: the scratch of the dense branches; ds_tokens: slc_bwd_ds_tokens; 0: every query selects all blocks it sees."""
    all_below = helper.all_below()
    dq = torch.empty_like(q)
    dq32 = torch.empty(q.shape, device=q.device, dtype=torch.float32) if ds_tokens else None
    # the window branch writes every element of dk / dv, the selected branch then adds to them
    dk = torch.empty(k.shape, device=q.device, dtype=torch.float32)
    dv = torch.empty(v.shape, device=q.device, dtype=torch.float32)

    def dkdv_cmp(r, *sums):
        return ds.dkdv_cmp(r, q, cmp_k, cmp_v, cmp_lse, dcmp_o, delta[0], sm_scale, *sums)

    def dkdv_raw(r):
        ds.dkdv_swa(r, q, k, v, lse_swa, do, delta[2], sm_scale, dk, dv)
        ds.dkdv_far(r, q, k, v, lse_slc, do, delta[1], sm_scale, dk, dv)

    def dense_dq(r):
        # (the selected dq comes last and adds this one; the queries that the gather leaves out are done)
        ds.dq(r, cmp_k, k, v.size(2), sm_scale, dq, 3 if ds_tokens else 0, dq32)

    def selected(dq_after=None):
        if ds_tokens:
            slc_attn_bwd(q, k, v, topk, None, lse_slc, do, dq=dq32, dk=dk, dv=dv, delta=delta[1], t_begin=all_below,
                         finalize_dq=dq, dq_after=dq_after, ds_tokens=ds_tokens, sm_scale=sm_scale, helper=helper)
        else:
            wait_for(dq_after)

    if OVERLAP_STREAMS and len(ds.ranges) == 1:
        # the compressed dk / dv next to the window's, the dense dq next to the selected dk / dv
        main, r = torch.cuda.current_stream(), ds.ranges[0]
        side = _side_stream(main, q, v, helper)
        side.wait_stream(main)
        with _on(side, main):
            dcmp_k, dcmp_v = dkdv_cmp(r)
        dkdv_raw(r)
        window_done = main.record_event() if side is not main else None
        with _on(side, main):
            wait_for(window_done)
            dense_dq(r)
        dcmp_k.record_stream(main)
        dcmp_v.record_stream(main)
        selected(side)
    else:  # ranges follow each other on one scratch, and each of them fills the GPU
        sums = ()
        for r in ds.ranges:
            sums = dkdv_cmp(r, *sums)
            dkdv_raw(r)
            dense_dq(r)
        dcmp_k, dcmp_v = sums
        ds.release()  # (in stream order, before the selected branch takes its own)
        selected()
    return dq, dk, dv, dcmp_k, dcmp_v


class NSAFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, combine_weight, cmp_k_weight, cmp_v_weight, sm_scale=None, for_backward=True):
        if sm_scale is None:
            sm_scale = q.size(-1) ** -0.5
        H = NSAHelper
        win_k, hid_k, cmp_k = _compress_fwd(k, cmp_k_weight, H.cmp_k_method, keep=for_backward)
        win_v, hid_v, cmp_v = _compress_fwd(v, cmp_v_weight, H.cmp_v_method, keep=for_backward)
        if 0 < H.x_maxlen <= H.all_below():  # nothing to choose from: no block is selected
            topk = torch.empty(k.size(1), q.size(0), H.top_n, device=q.device, dtype=torch.int32)
            (cmp_o, cmp_lse), (slc_o, slc_lse), (swa_o, swa_lse), out = short_fwd(q, k, v, cmp_k, cmp_v, combine_weight, H.all_below(),
                                                                                 for_backward, sm_scale, H)
        else:
            cmp_o, cmp_lse = cmp_attn_fwd(q, cmp_k, cmp_v, sm_scale=sm_scale)
            topk, _ = slc_topk_indices(q, cmp_k, cmp_lse, sm_scale=sm_scale, all_below=H.all_below())
            (slc_o, slc_lse), (swa_o, swa_lse), out = slc_swa_fwd(q, k, v, topk, sm_scale, H, cmp_o, combine_weight,
                                                                  store=for_backward)
        if not for_backward:
            return out

        keep = lambda flag, *ts: [None if flag else t for t in ts]
        saved = [q, k, v, combine_weight, cmp_k_weight, cmp_v_weight, topk]
        saved += keep(H.recompute_cmp_kv, win_k, hid_k, cmp_k, win_v, hid_v, cmp_v)
        saved += keep(H.recompute_cmp_o, cmp_o, cmp_lse)
        saved += keep(H.recompute_slc_o, slc_o, slc_lse)
        saved += keep(H.recompute_swa_o, swa_o, swa_lse)
        ctx.save_for_backward(*saved)
        ctx.sm_scale = sm_scale
        ctx.helper = H.get_bwd_helper()
        ctx.methods = (H.cmp_k_method, H.cmp_v_method)
        return out

    @staticmethod
    def backward(ctx, do):
        (q, k, v, combine_weight, cmp_k_weight, cmp_v_weight, topk, win_k, hid_k, cmp_k, win_v, hid_v, cmp_v, cmp_o,
         cmp_lse, slc_o, slc_lse, swa_o, swa_lse) = ctx.saved_tensors
        sm_scale, helper = ctx.sm_scale, ctx.helper
        k_method, v_method = ctx.methods
        do = thd_rows(do)

        if cmp_k is None:
            win_k, hid_k, cmp_k = _compress_fwd(k, cmp_k_weight, k_method, helper)
            win_v, hid_v, cmp_v = _compress_fwd(v, cmp_v_weight, v_method, helper)
        if cmp_o is None:
            cmp_o, cmp_lse = cmp_attn_fwd(q, cmp_k, cmp_v, sm_scale=sm_scale, helper=helper)
        if slc_o is None and swa_o is None:
            (slc_o, slc_lse), (swa_o, swa_lse), _ = slc_swa_fwd(q, k, v, topk, sm_scale, helper)
        elif slc_o is None:
            slc_o, slc_lse = slc_attn_fwd(q, k, v, topk, sm_scale=sm_scale, helper=helper, t_begin=helper.all_below())
            slc_fwd_first_queries(q, k, v, slc_o, slc_lse, helper.all_below(), sm_scale, helper)
        elif swa_o is None:
            swa_o, swa_lse = swa_fwd(q, k, v, sm_scale=sm_scale, helper=helper)

        # the kernels of the selected and the window branch read do itself, with the gates in their log-sum-exps; what the
        # selected branch of the first all_below tokens of a sequence has in common with the window branch is folded into
        # the latter
        all_below = helper.all_below()
        dcmp_o, dw, delta, (lse_slc, lse_swa) = combine_bwd_gates(cmp_o, slc_o, swa_o, combine_weight, do, slc_lse, swa_lse,
                                                                  all_below, helper)
        kw = dict(sm_scale=sm_scale, helper=helper)

        ds_tokens = slc_bwd_ds_tokens(q, k, v, do, topk, **kw) if helper.x_maxlen > all_below else 0
        stored_ds = ds_tokens > 0
        if (stored_ds or helper.x_maxlen <= all_below) and bwd_ds.takes(q, k, v, do, sm_scale, helper) and \
                bwd_ds.takes(q, cmp_k, cmp_v, dcmp_o, sm_scale, helper):
            ds = bwd_ds.DenseDs(q, k, helper, all_below=all_below)
            if ds.fits:
                dq, dk, dv, dcmp_k, dcmp_v = bwd_from_ds(ds, q, k, v, topk, cmp_k, cmp_v, do, dcmp_o, cmp_lse, lse_slc, lse_swa,
                                                         delta, ds_tokens, sm_scale, helper)
                dk, dwk = _compress_bwd(k, cmp_k_weight, win_k, hid_k, dcmp_k, dk, k_method, helper)
                dv, dwv = _compress_bwd(v, cmp_v_weight, win_v, hid_v, dcmp_v, dv, v_method, helper)
                return dq, dk, dv, dw, dwk, dwv, None, None

        # Where the selected branch's dk / dv pass can leave its dS behind, the selected dq comes last: it adds the other
        # branches', which one launch forms, and writes q's dtype (that launch does for the queries that the gather leaves out, and
        # for short batches there are no others).  Else it stores first, the window branch (matrix bound, with bandwidth to spare
        # for the read-modify-write) adds, or stores where the selected branch left rows out, and the compressed branch adds and
        # writes q's dtype.
        short = helper.x_maxlen <= all_below
        dq32 = None if short else torch.empty(q.shape, device=q.device, dtype=torch.float32)
        dq_last = torch.empty_like(q) if stored_ds or short else None

        def dq_chain():
            if dq_last is not None:
                return dense_bwd_dq(q, k, v, lse_swa, do, delta[2], lse_slc, do, delta[1], all_below, cmp_k, cmp_v, cmp_lse, dcmp_o,
                                    delta[0], dq_last, dq32, **kw)
            slc_attn_bwd(q, k, v, topk, slc_o, lse_slc, do, _store_into(dq32), delta=delta[1], parts="dq",
                         t_begin=all_below, **kw)
            swa_bwd_dq_tail(q, k, v, lse_swa, do, delta[2], lse_slc, do, delta[1], all_below, dq32, **kw)
            return cmp_attn_bwd(q, cmp_k, cmp_v, cmp_o, cmp_lse, dcmp_o, dq32, delta=delta[0], finalize_dq=True,
                                parts="dq", **kw)[0]

        def dkdv_raw(dq_after=None):
            # the window branch writes every element of dk / dv, the selected branch then adds to them
            _, dk, dv = swa_bwd(q, k, v, swa_o, lse_swa, do, delta=delta[2], dkv_fp32=True, parts="dkdv", **kw)
            slc_attn_bwd_dkdv_before_window(q, k, v, lse_slc, do, delta[1], dk, dv, all_below, **kw)
            last = dict(dq=dq32, finalize_dq=dq_last, dq_after=dq_after, ds_tokens=ds_tokens) if stored_ds else dict(parts="dkdv")
            slc_attn_bwd(q, k, v, topk, slc_o, lse_slc, do, dk=dk, dv=dv, delta=delta[1], t_begin=all_below, **last, **kw)
            return dk, dv

        def dkdv_cmp():
            return cmp_attn_bwd(q, cmp_k, cmp_v, cmp_o, cmp_lse, dcmp_o, delta=delta[0], parts="dkdv", **kw)[1:]

        main = torch.cuda.current_stream()
        if OVERLAP_STREAMS and stored_ds:
            # the dense dq kernels next to the dk / dv passes whose dS the selected dq waits for, the compressed dk / dv
            # next to the selected dq
            side = _side_stream(main, q, v, helper)
            side.wait_stream(main)
            with _on(side, main):
                dq = dq_chain()
                dense_dq = side.record_event() if side is not main else None
                dcmp_k, dcmp_v = dkdv_cmp()
                dcmp_k.record_stream(main)
                dcmp_v.record_stream(main)
            dk, dv = dkdv_raw(dense_dq)
            main.wait_stream(side)
        elif OVERLAP_STREAMS:
            side = _side_stream(main, q, v, helper)
            side.wait_stream(main)
            with _on(side, main):
                dq = dq_chain()
                dq.record_stream(main)
            # dk/dv kernels on the caller's stream.  The compressed branch (matrix bound) goes first, next to the selected
            # dq kernel (bound by the gather path) on the other stream: 0.7-1.7 ms per step less at T = 64K (67.7 -> 67.0
            # and 67.2 -> 65.5 ms on two GPUs) than the order window, selected, compressed, which ran the two selected
            # kernels side by side.
            dcmp_k, dcmp_v = dkdv_cmp()
            dk, dv = dkdv_raw()
        else:
            dq = dq_chain()
            dk, dv = dkdv_raw()
            dcmp_k, dcmp_v = dkdv_cmp()
        dk, dwk = _compress_bwd(k, cmp_k_weight, win_k, hid_k, dcmp_k, dk, k_method, helper)
        dv, dwv = _compress_bwd(v, cmp_v_weight, win_v, hid_v, dcmp_v, dv, v_method, helper)
        if OVERLAP_STREAMS and not stored_ds:
            main.wait_stream(side)
        return dq, dk, dv, dw, dwk, dwv, None, None


class _StoreTarget:
    """Marks an fp32 dq buffer that the first branch overwrites instead of adding into."""

    def __init__(self, buf):
        self.buf = buf


def _store_into(buf):
    return _StoreTarget(buf)


def flash_nsa_varlen_func(q, k, v, combine_weight, cmp_k_weight=None, cmp_v_weight=None, sm_scale=None):
    # without gradients nothing is kept for a backward: the branch outputs need not be stored
    return NSAFunction.apply(q, k, v, combine_weight, cmp_k_weight, cmp_v_weight, sm_scale, torch.is_grad_enabled())


def cp_flash_nsa_varlen_func(*args, **kwargs):
    raise NotImplementedError("context parallelism is outside this single-GPU build")


class NSACore(torch.nn.Module):
    def __init__(self, config: NSAConfig, process_group=None, pp_size=1):
        super().__init__()
        assert process_group is None, "context parallelism is outside this single-GPU build"
        self.config = config
        self.qk_head_dim = config.qk_head_dim if config.qk_head_dim is not None else config.head_dim
        self.v_head_dim = config.v_head_dim if config.v_head_dim is not None else config.head_dim
        g = lambda name, default: getattr(config, name, default)
        self.kernel_size, self.stride, self.block_size = g("kernel_size", 32), g("stride", 16), g("block_size", 64)
        self.top_n, self.window_size = g("top_n", 16), g("window_size", 512)
        self.num_init_blocks, self.num_local_blocks = g("num_init_blocks", 1), g("num_local_blocks", 2)
        self.cmp_k_method, self.cmp_v_method = g("cmp_k_method", "mean"), g("cmp_v_method", "mean")
        self.recompute = dict(recompute_cmp_kv=g("recompute_cmp_kv", False), recompute_cmp_o=g("recompute_cmp_o", False),
                              recompute_slc_o=g("recompute_slc_o", False), recompute_swa_o=g("recompute_swa_o", False))
        self.pp_size = pp_size
        self.sm_scale = self.qk_head_dim ** -0.5
        # the core also accepts config objects other than NSAConfig (any object with these attributes): validate here too
        check_supported(self.qk_head_dim, self.v_head_dim, self.kernel_size, self.stride, self.block_size)
        self._set_helper()

        def make_weight(method, dim):
            if method == "mean":
                return None
            out_features = dim if method == "linear" else 2 * dim
            w = torch.empty(out_features, self.kernel_size * dim)
            torch.nn.init.kaiming_uniform_(w, a=math.sqrt(5))
            return torch.nn.Parameter(w)

        self.cmp_k_weight = make_weight(self.cmp_k_method, self.qk_head_dim)
        self.cmp_v_weight = make_weight(self.cmp_v_method, self.v_head_dim)

    def _set_helper(self):
        NSAHelper.set_hyperparameters(kernel_size=self.kernel_size, stride=self.stride, block_size=self.block_size,
                                      window_size=self.window_size, top_n=self.top_n,
                                      num_init_blocks=self.num_init_blocks, num_local_blocks=self.num_local_blocks)
        NSAHelper.set_recompute(**self.recompute)
        NSAHelper.set_cmp_kv_method(cmp_k_method=self.cmp_k_method, cmp_v_method=self.cmp_v_method)
        NSAHelper.set_pipeline_parallel_world_size(pp_size=self.pp_size)

    def forward(self, q, k, v, combine_weight, cu_seqlens, cu_seqlens_np=None, cp_mode=None):
        """q [T,QH,Dqk], k [T,KH,Dqk], v [T,KH,Dv], combine_weight [T,QH,3], cu_seqlens int32 [B+1] -> [T,QH,Dv]"""
        assert cu_seqlens is not None
        self._set_helper()
        NSAHelper.init_cu_seqlens(cu_seqlens)
        return flash_nsa_varlen_func(q, k, v, combine_weight, self.cmp_k_weight, self.cmp_v_weight, self.sm_scale)
