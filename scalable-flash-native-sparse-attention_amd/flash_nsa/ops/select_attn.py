"""Selected-block attention (upstream flash_nsa/ops/select_attn.py:439-748)."""
import torch

from .. import _lib
from ..utils import NSAHelper
from ._common import check_thd, default_scale, delta_of, dq_target, zeros_pair


def slc_attn_fwd(q, k, v, topk, sm_scale=None, helper=NSAHelper, t_begin=0):
    """q [T,QH,D], k [T,KH,D], v [T,KH,VD], topk [KH,T,top_n] int32 -> o [T,QH,VD], lse [T,QH] fp32 (log2).
    Query t of a sequence attends the keys <= t of the blocks in its first min(top_n, t//block+1) slots.
    t_begin: only the queries at positions from here on (the other rows of o and lse stay unwritten: swa_fwd_tail)."""
    check_thd(q, "q"), check_thd(k, "k"), check_thd(v, "v")
    T, QH, D = q.shape
    _, KH, VD = v.shape
    assert topk.dtype == torch.int32 and topk.shape[:2] == (KH, T) and topk.stride(-1) == 1
    sm_scale = default_scale(q, sm_scale)
    o = torch.empty(T, QH, VD, device=q.device, dtype=q.dtype)
    lse = torch.empty(T, QH, device=q.device, dtype=torch.float32)
    if 0 < helper.x_maxlen <= t_begin:
        return o, lse
    _lib.call("nsa_slc_attn_fwd_from", q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1),
              v.data_ptr(), v.stride(0), v.stride(1), topk.data_ptr(), topk.stride(0), topk.stride(1), o.data_ptr(),
              o.stride(0), o.stride(1), lse.data_ptr(), lse.stride(0), lse.stride(1),
              helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.block_size,
              topk.size(-1), t_begin, sm_scale, _lib.stream_ptr())
    return o, lse


def slc_bwd_ds_tokens(q, k, v, do, topk, sm_scale=None, helper=NSAHelper):
    """Tokens per call of the backward that computes dq from the dS of the dk / dv pass, 0 where dq and dk / dv are computed
    apart.  The scratch holds the dS of so many tokens (32 KB per token and kv head for 16 q-heads, 16 blocks of 64 keys), 2 GB
    at most; shapes of which that does not hold 512 tokens are computed apart."""
    T, QH, D = q.shape
    _, KH, VD = v.shape
    if getattr(helper, "deterministic", False):
        return 0
    return _lib.value("nsa_slc_bwd_ds_tokens", T, q.stride(1), do.stride(1), k.stride(0), QH, KH, D, VD, helper.block_size,
                      topk.size(-1), default_scale(q, sm_scale))


def wait_for(done):
    """The current stream waits for an event, or for what has been launched on another stream (None: for nothing)."""
    if isinstance(done, torch.cuda.Stream):
        torch.cuda.current_stream().wait_stream(done)
    elif done is not None:
        torch.cuda.current_stream().wait_event(done)


def _slc_attn_bwd_ds(common, topk, dq, dq_mode, partial, dk, dv, shape, tokens, t_begin, sm_scale, helper, dq_after):
    T, QH, KH, D, VD = shape
    N, nblk, dev = topk.size(-1), helper.k_len, topk.device
    chunk = _lib.value("nsa_slc_bwd_chunk_tokens", tokens, KH, N)
    ds_bytes = _lib.value("nsa_slc_bwd_ds_bytes", tokens, QH, KH, helper.block_size, N)
    # (the last range, the only shorter one, may need more: short ranges are counted in shorter chunks)
    ws_elems = max(_lib.value("nsa_inverse_index_workspace_elems", n, KH, nblk) for n in {tokens, (T - 1) % tokens + 1})
    # one buffer: dS, token list, the list builder's scratch, list and item offsets, slot of every list entry
    entries, n_off, index_at = KH * tokens * N, KH * (nblk + 1), (ds_bytes + 255) // 256 * 256
    buf = torch.empty(index_at + 4 * (entries + ws_elems + 2 * n_off) + entries, dtype=torch.uint8, device=dev)
    ds = buf.data_ptr()
    index = ds + index_at
    scratch = index + 4 * entries
    csr_off = scratch + 4 * ws_elems
    item_off = csr_off + 4 * n_off
    slot = item_off + 4 * n_off
    stream = _lib.stream_ptr()
    x_cu, k_cu = helper.x_cu_seqlens.data_ptr(), helper.k_cu_seqlens.data_ptr()
    tk = (topk.data_ptr(), topk.stride(0), topk.stride(1))
    heads = (helper.batch, QH, KH, D, VD, helper.block_size, N)
    dqs = (dq.data_ptr(), dq.stride(0), dq.stride(1), dq_mode)
    dqs += (None, 0, 0) if partial is None else (partial.data_ptr(), partial.stride(0), partial.stride(1))
    for tok0 in range(0, T, tokens):
        n = min(tokens, T - tok0)
        _lib.call("nsa_build_inverse_index_slots", *tk, N, x_cu, k_cu, helper.batch, tok0, n, KH, nblk, helper.block_size,
                  chunk, t_begin, csr_off, index, slot, item_off, scratch, ws_elems, stream)
        _lib.call("nsa_slc_attn_bwd_dkdv_ds", *common, dk.data_ptr(), dk.stride(0), dk.stride(1), dv.data_ptr(), dv.stride(0),
                  dv.stride(1), x_cu, k_cu, helper.blk_seq.data_ptr(), csr_off, index, slot, item_off, nblk, chunk,
                  (n * N + chunk - 1) // chunk + nblk, *heads, tok0, n, sm_scale, ds, ds_bytes, stream)
        if tok0 == 0:
            wait_for(dq_after)
        _lib.call("nsa_slc_attn_bwd_dq_ds", *common[3:6], *tk, *dqs, x_cu, *heads, t_begin, tok0, n, sm_scale, ds, ds_bytes,
                  stream)


def slc_attn_bwd(q, k, v, topk, o, lse, do, dq=None, dk=None, dv=None, sm_scale=None, helper=NSAHelper, delta=None,
                 bind=None, parts="both", dkdv_repeat=False, t_begin=0, finalize_dq=None, dq_after=None,
                 ds_tokens=None):
    """Backward of selected attention.  Returns (dq, dk, dv).
    dq: fresh bf16 tensor, or the caller's fp32 buffer (added into).  dk/dv: fp32 [T,KH,*]; the caller's buffers
    are added into, otherwise zero-filled ones are created.  dkdv_repeat=False (default): with fp32 atomics, so the
    summation order changes from run to run (as upstream's dkdv_repeat=False); dkdv_repeat=True (or
    NSAHelper.set_deterministic(True)): the work items store into slots of a scratch buffer that a second launch adds
    in a fixed order -- bit-identical results across runs.
    `bind` is the inverse index from get_bind_from_find (built here when absent).
    parts = "dq" / "dkdv" launches only that kernel (the other results are None).
    t_begin: only the queries at positions from here on (a given `bind` then has to leave the others out).
    ds_tokens: what slc_bwd_ds_tokens has returned for these tensors, if the caller has asked.
    finalize_dq (where slc_bwd_ds_tokens > 0): a tensor of q's dtype that takes the sum of this branch's dq and dq, the fp32
    sum of the others, which is ready when the event dq_after is, or what has been launched on the stream dq_after."""
    from .topk import get_bind_from_find
    check_thd(do, "do")
    T, QH, D = q.shape
    _, KH, VD = v.shape
    sm_scale = default_scale(q, sm_scale)
    if delta is None:
        delta = delta_of(o, do)
    common = (q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(),
              v.stride(0), v.stride(1), do.data_ptr(), do.stride(0), do.stride(1), lse.data_ptr(), lse.stride(0),
              lse.stride(1), delta.data_ptr(), delta.stride(0), delta.stride(1))
    dq_buf = None
    ordered = dkdv_repeat or getattr(helper, "deterministic", False)
    if parts != "both" or ordered or bind is not None or 0 < helper.x_maxlen <= t_begin:
        ds_tokens = 0
    elif ds_tokens is None:
        ds_tokens = slc_bwd_ds_tokens(q, k, v, do, topk, sm_scale, helper)
    if finalize_dq is not None:
        assert ds_tokens and dq.dtype == torch.float32 and dq.shape == q.shape and dq.stride(-1) == 1
        dq_buf, mode, partial = finalize_dq, 3, dq
    elif parts in ("both", "dq"):
        (dq_buf, mode), partial = dq_target(q, dq), None
    if parts in ("both", "dq") and not ds_tokens:
        _lib.call("nsa_slc_attn_bwd_dq_from", *common, topk.data_ptr(), topk.stride(0), topk.stride(1), dq_buf.data_ptr(),
                  dq_buf.stride(0), dq_buf.stride(1), mode, helper.x_cu_seqlens.data_ptr(), helper.batch,
                  helper.x_maxlen, QH, KH, D, VD, helper.block_size, topk.size(-1), t_begin, sm_scale,
                  _lib.stream_ptr())
    if parts == "dq":
        return dq_buf, None, None
    if dk is None and dv is None:
        dk, dv = zeros_pair((T, KH, D), (T, KH, VD), q.device)
    elif dk is None:
        dk = torch.zeros(T, KH, D, device=q.device, dtype=torch.float32)
    elif dv is None:
        dv = torch.zeros(T, KH, VD, device=q.device, dtype=torch.float32)
    assert dk.dtype == torch.float32 and dv.dtype == torch.float32
    if 0 < helper.x_maxlen <= t_begin:
        return dq_buf, dk, dv
    if ds_tokens:
        _slc_attn_bwd_ds(common, topk, dq_buf, mode, partial, dk, dv, (T, QH, KH, D, VD), ds_tokens, t_begin, sm_scale,
                         helper, dq_after)
        return dq_buf, dk, dv
    if bind is None:
        bind = get_bind_from_find(topk, helper, t_begin=t_begin, deterministic=ordered)
    args = (*common, dk.data_ptr(), dk.stride(0), dk.stride(1), dv.data_ptr(), dv.stride(0), dv.stride(1),
            helper.x_cu_seqlens.data_ptr(), helper.k_cu_seqlens.data_ptr(), helper.blk_seq.data_ptr(),
            bind["csr_off"].data_ptr(), bind["csr_tok"].data_ptr(), bind["item_off"].data_ptr(), bind["nblk"],
            bind["chunk_tokens"], bind["n_items_bound"], helper.batch, QH, KH, D, VD, helper.block_size, sm_scale)
    if ordered:
        nbytes = _lib.value("nsa_slc_attn_bwd_dkdv_det_bytes", bind["n_items_bound"], KH, D, VD, helper.block_size)
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=q.device)
        _lib.call("nsa_slc_attn_bwd_dkdv_det", *args, ws.data_ptr(), ws.numel(), _lib.stream_ptr())
    else:
        _lib.call("nsa_slc_attn_bwd_dkdv", *args, _lib.stream_ptr())
    return dq_buf, dk, dv


def slc_attn_bwd_dkdv_before_window(q, k, v, lse, do, delta, dk, dv, all_below, sm_scale=None, helper=NSAHelper):
    """Adds to dk / dv (fp32) what the queries at positions below all_below, which select every block they can see, give
    the keys before their window.  lse and delta are combine_bwd_gates' (lse[0] and delta[1], with the gates in them), with
    the same all_below: the keys inside the window are in what it gives the window branch."""
    T, QH, D = q.shape
    _, KH, VD = v.shape
    _lib.call("nsa_slc_attn_bwd_dkdv_before_window", q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0),
              k.stride(1), v.data_ptr(), v.stride(0), v.stride(1), do.data_ptr(), do.stride(0), do.stride(1),
              lse.data_ptr(), lse.stride(0), lse.stride(1), delta.data_ptr(), delta.stride(0), delta.stride(1),
              dk.data_ptr(), dk.stride(0), dk.stride(1), dv.data_ptr(), dv.stride(0), dv.stride(1),
              helper.x_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, QH, KH, D, VD, helper.window_size,
              all_below, int(helper.deterministic), default_scale(q, sm_scale), _lib.stream_ptr())


class _SelectAttn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, topk, sm_scale):
        o, lse = slc_attn_fwd(q, k, v, topk, sm_scale)
        ctx.save_for_backward(q, k, v, topk, o, lse)
        ctx.sm_scale = sm_scale
        ctx.helper = NSAHelper.get_bwd_helper()
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, topk, o, lse = ctx.saved_tensors
        do = do if do.stride(-1) == 1 else do.contiguous()
        dq, dk, dv = slc_attn_bwd(q, k, v, topk, o, lse, do, sm_scale=ctx.sm_scale, helper=ctx.helper)
        return dq, dk.to(k.dtype), dv.to(v.dtype), None, None


def select_attn(q, k, v, topk, sm_scale=None):
    """Differentiable selected-block attention (no gradient flows into topk)."""
    return _SelectAttn.apply(q, k, v, topk, sm_scale)
