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


def _st(t):
    return t.data_ptr(), t.stride(0), t.stride(1)


class DenseDs:
    """The scratch of one backward of the compressed branch (with_cmp), the window (with_swa) and, with all_below > 0, the keys
    before the window of the queries below it, up to 4 GB each; `ranges` are the (tok0, tok1) that dkdv_cmp, dkdv_swa and dq are
    called for, in this order.  `fits`: whether there are such ranges (else dq and dk / dv are to be computed apart)."""

    def __init__(self, q, k, helper=NSAHelper, with_cmp=True, with_swa=True, all_below=0):
        T, QH, D = q.shape
        self.h, self.T, self.QH, self.KH, self.D = helper, T, QH, k.size(1), D
        self.all_below = all_below
        sizes = (T, helper.batch, helper.x_maxlen, QH, self.KH)
        cmp_sizes = (helper.kernel_size, helper.stride)
        branches = (*(cmp_sizes if with_cmp else (0, 0)), helper.window_size if with_swa else -1, all_below)
        cuts, at, self.fits = [], 0, True
        while at < T:
            end = _lib.value("nsa_bwd_ds_range_end", at, *sizes, *branches)
            if end < 0:
                self.fits, self.ranges = False, []
                return
            cuts.append((at, end))
            at = end
        if len(cuts) == 1:
            cuts = [(0, 0)]
        self.ranges = cuts
        self.ring = max(e - s for s, e in cuts)
        n_cmp = max(_lib.value("nsa_cmp_attn_bwd_ds_bytes", *sizes, *cmp_sizes, *r) for r in cuts) if with_cmp else 0
        n_swa = _lib.value("nsa_swa_bwd_ds_bytes", *sizes, helper.window_size, self.ring) if with_swa else 0
        n_far = (_lib.value("nsa_slc_bwd_before_window_ds_bytes", *sizes, helper.window_size, all_below, self.ring)
                 if with_swa and all_below else 0)
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
        h, VD = self.h, v.size(2)
        sizes = (h.batch, h.x_maxlen, h.y_maxlen, self.QH, self.KH, self.D, VD, h.kernel_size, h.stride)
        first = dk is None
        if first:
            self.cmp_slots = max(_lib.value("nsa_cmp_attn_bwd_dkdv_ds_slot_bytes", *sizes, *x) for x in self.ranges)
            shapes = (k.shape, v.shape)
            if self.cmp_slots <= compress_attn.DKDV_SLOTS_LIMIT:
                dk, dv = (torch.empty(s, device=q.device, dtype=torch.float32) for s in shapes)
            else:
                dk, dv = zeros_pair(*shapes, q.device)
        n = self.cmp_slots if self.cmp_slots <= compress_attn.DKDV_SLOTS_LIMIT else 0
        ws = torch.empty(n, dtype=torch.uint8, device=q.device) if n else None
        _lib.call("nsa_cmp_attn_bwd_dkdv_ds", *_st(q), *_st(k), *_st(v), *_st(do), lse.data_ptr(), lse.stride(1),
                  lse.stride(0), *_st(delta), *_st(dk), *_st(dv), h.x_cu_seqlens.data_ptr(), h.y_cu_seqlens.data_ptr(),
                  *sizes, sm_scale, self.T, *r, *self.cmp, _lib.ptr(ws), n, int(not first), _lib.stream_ptr())
        return dk, dv

    def dkdv_swa(self, r, q, k, v, lse, do, delta, sm_scale, dk, dv):
        """dk, dv (bf16 or fp32) of the keys of range r."""
        h, VD = self.h, v.size(2)
        sizes = (h.batch, h.x_maxlen, self.QH, self.KH, self.D, VD, h.window_size)
        n = _lib.value("nsa_swa_bwd_dkdv_ds_ws_bytes", self.T, *sizes, *r)
        ws = torch.empty(n, dtype=torch.uint8, device=q.device) if n else None
        _lib.call("nsa_swa_bwd_dkdv_ds", *_st(q), *_st(k), *_st(v), *_st(do), *_st(lse), *_st(delta), *_st(dk), *_st(dv),
                  int(dk.dtype == torch.float32), h.x_cu_seqlens.data_ptr(), *sizes, sm_scale, self.T, self.ring, *r,
                  *self.swa, _lib.ptr(ws), n, _lib.stream_ptr())

    def dkdv_far(self, r, q, k, v, lse, do, delta, sm_scale, dk, dv):
        """slc_attn_bwd_dkdv_before_window for the keys of range r."""
        if not self.far[1]:
            return
        h, VD = self.h, v.size(2)
        _lib.call("nsa_slc_attn_bwd_dkdv_before_window_ds", *_st(q), *_st(k), *_st(v), *_st(do), *_st(lse), *_st(delta),
                  *_st(dk), *_st(dv), h.x_cu_seqlens.data_ptr(), h.batch, h.x_maxlen, self.QH, self.KH, self.D, VD,
                  h.window_size, self.all_below, sm_scale, self.T, self.ring, *r, *self.far, _lib.stream_ptr())

    def dq(self, r, ck, k, VD, sm_scale, dq, mode, partial=None):
        """dq of the tokens of range r from the compressed rows ck and / or the keys k: mode as nsa_attn_bwd_dq_ds."""
        h = self.h
        none = (None, 0, 0)
        _lib.call("nsa_attn_bwd_dq_ds", *(none if ck is None else _st(ck)), *self.cmp, *(none if k is None else _st(k)),
                  *self.swa, *self.far, *_st(dq), mode, *(none if partial is None else _st(partial)),
                  h.x_cu_seqlens.data_ptr(), h.y_cu_seqlens.data_ptr(), h.batch, h.x_maxlen, self.QH, self.KH, self.D, VD,
                  h.kernel_size, h.stride, h.window_size, self.all_below, sm_scale, self.T, self.ring, *r,
                  _lib.stream_ptr())
