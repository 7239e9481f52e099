"""dq of the compressed and the window branch from the dS that their dk / dv passes leave behind (upstream computes S and dP
once more for dq, flash_nsa/ops/compress_attn.py:385-528)."""
import torch

from .. import _lib
from ..utils import NSAHelper
from . import compress_attn
from ._common import zeros_pair


def takes(q, k, v, do, sm_scale, helper=NSAHelper):
    """Whether these shapes and strides have a dk / dv pass that stores dS."""
    if q.size(0) == 0 or helper.x_maxlen == 0 or getattr(helper, "deterministic", False):
        return False
    return bool(_lib.value("nsa_bwd_ds_takes", q.stride(1), do.stride(1), k.stride(0), q.size(1), k.size(1), q.size(2),
                           v.size(2), sm_scale))


def _st(t, row=0):
    """Address of row `row` of t, strides."""
    at = t.data_ptr()
    if row:
        at += row * t.stride(0) * t.element_size()
    return at, t.stride(0), t.stride(1)


class _Part:
    """Sequences b0 .. b1 - 1 of a batch as a batch of their own: its first token x0 and compressed row y0, lengths, offsets from
    there on, and the ranges of its T tokens (one range: (0, 0)), `ring` tokens the longest of them (one range: 0)."""

    def __init__(self, helper, T, b0=0, b1=None):
        b1 = helper.batch if b1 is None else b1
        self.batch, self.T = b1 - b0, T
        if self.batch == helper.batch:
            self.x0 = self.y0 = 0
            self.x_maxlen, self.y_maxlen = helper.x_maxlen, helper.y_maxlen
            self.x_cu, self.y_cu = helper.x_cu_seqlens, helper.y_cu_seqlens
            return
        lens = [e - s for s, e in zip(helper._host_cu, helper._host_cu[1:])]
        y = [max((n - helper.kernel_size) // helper.stride + 1, 0) for n in lens[:b1]]
        self.x0, self.y0 = sum(lens[:b0]), sum(y[:b0])
        self.x_maxlen, self.y_maxlen = max(lens[b0:b1]), max(y[b0:b1])
        self.x_cu = helper.x_cu_seqlens[b0:b1 + 1] - self.x0
        self.y_cu = helper.y_cu_seqlens[b0:b1 + 1] - self.y0

    def plan(self, end_of):
        end = end_of(0, self.T, self.batch, self.x_maxlen)
        if end == self.T:
            self.ranges, self.ring = ((0, 0),), 0
            return True
        self.ranges, at = [], 0
        while 0 < end:
            self.ranges.append((at, end))
            if end == self.T:
                self.ring = max(e - s for s, e in self.ranges)
                return True
            at, end = end, end_of(end, self.T, self.batch, self.x_maxlen)
        return False


def _cut(cu, b0, b1, end_of):
    """The sequences b0 .. b1 - 1 (offsets cu) in consecutive groups that one range holds, or of one sequence: halved, by tokens,
    while they do not.  A tile's dS is as wide as the longest sequence beside it, so a range over a long and many short ones is
    short: one of 60K tokens before 400 of 350, 64 / 4 heads of 128, 105 ms in 29 ranges of the whole batch, 85 with dq
    recomputed, 77 so."""
    n = cu[b1] - cu[b0]
    if n == 0:
        return []
    if b1 - b0 == 1 or end_of(0, n, b1 - b0, max(e - s for s, e in zip(cu[b0:b1], cu[b0 + 1:b1 + 1]))) == n:
        return [(b0, b1)]
    at = min(range(b0 + 1, b1), key=lambda b: abs(2 * (cu[b] - cu[b0]) - n))
    return _cut(cu, b0, at, end_of) + _cut(cu, at, b1, end_of)


class DenseDs:
    """The scratch of one backward of the compressed branch (with_cmp), the window (with_swa) and, with all_below > 0, the keys
    before the window of the queries below it, up to 4 GB each; `ranges` are the (part of the batch, tok0, tok1) that dkdv_cmp,
    dkdv_swa and dq are called for, in this order.  `fits`: whether there are such ranges (else dq and dk / dv are to be computed
    apart)."""

    def __init__(self, q, k, helper=NSAHelper, with_cmp=True, with_swa=True, all_below=0):
        T, QH, D = q.shape
        self.h, self.QH, self.KH, self.D = helper, QH, k.size(1), D
        self.all_below = all_below
        cmp_sizes = (helper.kernel_size, helper.stride)
        branches = (*(cmp_sizes if with_cmp else (0, 0)), helper.window_size if with_swa else -1, all_below)

        def end_of(at, T, batch, longest):
            return _lib.value("nsa_bwd_ds_range_end", at, T, batch, longest, QH, self.KH, *branches)

        parts = [_Part(helper, T)]
        self.fits = parts[0].plan(end_of)
        host = getattr(helper, "_host_cu", None)
        if host is not None and helper.batch > 1 and not (self.fits and parts[0].ring == 0):
            parts = [_Part(helper, host[e] - host[b], b, e) for b, e in _cut(host, 0, helper.batch, end_of)]
            self.fits = all([p.plan(end_of) for p in parts])
        self.ranges = [(p, *r) for p in parts for r in p.ranges] if self.fits else []
        if not self.fits:
            return
        n_cmp = n_swa = n_far = 0
        for p in parts:
            sizes = (p.T, p.batch, p.x_maxlen, QH, self.KH)
            if with_cmp:
                n_cmp = max([n_cmp] + [_lib.value("nsa_cmp_attn_bwd_ds_bytes", *sizes, *cmp_sizes, *r) for r in p.ranges])
            if with_swa:
                n_swa = max(n_swa, _lib.value("nsa_swa_bwd_ds_bytes", *sizes, helper.window_size, p.ring))
            if with_swa and all_below:
                n_far = max(n_far, _lib.value("nsa_slc_bwd_before_window_ds_bytes", *sizes, helper.window_size, all_below, p.ring))
        n_cmp, n_swa, n_far = ((n + 255) // 256 * 256 for n in (n_cmp, n_swa, n_far))
        self.buf = torch.empty(n_cmp + n_swa + n_far, dtype=torch.uint8, device=q.device)
        base = self.buf.data_ptr()
        self.cmp = (base if n_cmp else None, n_cmp)
        self.swa = (base + n_cmp if n_swa else None, n_swa)
        self.far = (base + n_cmp + n_swa if n_far else None, n_far)

    def release(self):
        """Gives the scratch back (to the current stream's pool)."""
        self.buf = None

    def dkdv_cmp(self, r, q, k, v, lse, do, delta, sm_scale, dk=None, dv=None):
        """dk, dv of the compressed rows from the queries of range r, added to those of the ranges before (dk, dv)."""
        p, tok0, tok1 = r
        h = self.h
        shape = (self.QH, self.KH, self.D, v.size(2), h.kernel_size, h.stride)
        if dk is None:
            self.cmp_slots = max([_lib.value("nsa_cmp_attn_bwd_dkdv_ds_slot_bytes", x.batch, x.x_maxlen, x.y_maxlen, *shape, *t)
                                  for x, *t in self.ranges])
            shapes = (k.shape, v.shape)
            if self.cmp_slots <= compress_attn.DKDV_SLOTS_LIMIT:
                dk, dv = (torch.empty(s, device=q.device, dtype=torch.float32) for s in shapes)
            else:
                dk, dv = zeros_pair(*shapes, q.device)
        n = self.cmp_slots if self.cmp_slots <= compress_attn.DKDV_SLOTS_LIMIT else 0
        ws = torch.empty(n, dtype=torch.uint8, device=q.device) if n else None
        _lib.call("nsa_cmp_attn_bwd_dkdv_ds", *_st(q, p.x0), *_st(k, p.y0), *_st(v, p.y0), *_st(do, p.x0),
                  lse.data_ptr() + 4 * p.x0 * lse.stride(1), lse.stride(1), lse.stride(0), *_st(delta, p.x0), *_st(dk, p.y0),
                  *_st(dv, p.y0), p.x_cu.data_ptr(), p.y_cu.data_ptr(), p.batch, p.x_maxlen, p.y_maxlen, *shape, sm_scale, p.T,
                  tok0, tok1, *self.cmp, _lib.ptr(ws), n, int(tok0 > 0), _lib.stream_ptr())
        return dk, dv

    def dkdv_swa(self, r, q, k, v, lse, do, delta, sm_scale, dk, dv):
        """dk, dv (bf16 or fp32) of the keys of range r."""
        p, tok0, tok1 = r
        h, x = self.h, p.x0
        sizes = (p.batch, p.x_maxlen, self.QH, self.KH, self.D, v.size(2), h.window_size)
        n = _lib.value("nsa_swa_bwd_dkdv_ds_ws_bytes", p.T, *sizes, tok0, tok1)
        ws = torch.empty(n, dtype=torch.uint8, device=q.device) if n else None
        _lib.call("nsa_swa_bwd_dkdv_ds", *_st(q, x), *_st(k, x), *_st(v, x), *_st(do, x), *_st(lse, x), *_st(delta, x), *_st(dk, x),
                  *_st(dv, x), int(dk.dtype == torch.float32), p.x_cu.data_ptr(), *sizes, sm_scale, p.T, p.ring, tok0, tok1,
                  *self.swa, _lib.ptr(ws), n, _lib.stream_ptr())

    def dkdv_far(self, r, q, k, v, lse, do, delta, sm_scale, dk, dv):
        """slc_attn_bwd_dkdv_before_window for the keys of range r."""
        if not self.far[1]:
            return
        p, tok0, tok1 = r
        h, x = self.h, p.x0
        _lib.call("nsa_slc_attn_bwd_dkdv_before_window_ds", *_st(q, x), *_st(k, x), *_st(v, x), *_st(do, x), *_st(lse, x),
                  *_st(delta, x), *_st(dk, x), *_st(dv, x), p.x_cu.data_ptr(), p.batch, p.x_maxlen, self.QH, self.KH, self.D,
                  v.size(2), h.window_size, self.all_below, sm_scale, p.T, p.ring, tok0, tok1, *self.far, _lib.stream_ptr())

    def dq(self, r, ck, k, VD, sm_scale, dq, mode, partial=None):
        """dq of the tokens of range r from the compressed rows ck and / or the keys k: mode as nsa_attn_bwd_dq_ds."""
        p, tok0, tok1 = r
        h = self.h
        none = (None, 0, 0)
        _lib.call("nsa_attn_bwd_dq_ds", *(none if ck is None else _st(ck, p.y0)), *self.cmp,
                  *(none if k is None else _st(k, p.x0)), *self.swa, *self.far, *_st(dq, p.x0), mode,
                  *(none if partial is None else _st(partial, p.x0)), p.x_cu.data_ptr(), p.y_cu.data_ptr(), p.batch, p.x_maxlen,
                  self.QH, self.KH, self.D, VD, h.kernel_size, h.stride, h.window_size, self.all_below, sm_scale, p.T, p.ring, tok0, tok1,
                  _lib.stream_ptr())
