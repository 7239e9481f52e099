"""KV compression operators: mean pooling and im2col of the compression windows
(upstream flash_nsa/ops/compress_kv.py:126-426)."""
import torch

from .. import _lib
from ..utils import NSAHelper
from ._common import check_thd, thd_rows
from .act import _glu_bwd


def mean_pooling_fwd(x, helper=NSAHelper):
    """x [T,H,D] -> y [y_len,H,D]: mean over windows [stride*i, stride*i+kernel) of every sequence."""
    check_thd(x, "x")
    T, H, D = x.shape
    y = torch.empty(helper.y_len, H, D, device=x.device, dtype=x.dtype)
    _lib.call("nsa_mean_pool_fwd", x.data_ptr(), x.stride(0), x.stride(1), y.data_ptr(), y.stride(0), y.stride(1),
              helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.y_maxlen, H, D,
              helper.kernel_size, helper.stride, _lib.stream_ptr())
    return y


def mean_pooling_bwd(x, dy, dx=None, helper=NSAHelper):
    """Gradient of mean pooling.  With dx=None a new tensor of x's dtype is returned; an fp32 dx is
    accumulated into (each element has a single writer, so the result is deterministic)."""
    check_thd(dy, "dy")
    T, H, D = x.shape
    accumulate = dx is not None
    if dx is None:
        dx = torch.empty(T, H, D, device=x.device, dtype=x.dtype)
    else:
        assert dx.dtype == torch.float32 and dx.shape == x.shape and dx.stride(-1) == 1
    _lib.call("nsa_mean_pool_bwd", dy.data_ptr(), dy.stride(0), dy.stride(1), dx.data_ptr(), dx.stride(0),
              dx.stride(1), int(dx.dtype == torch.float32), int(accumulate), helper.x_cu_seqlens.data_ptr(),
              helper.y_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, H, D, helper.kernel_size, helper.stride,
              _lib.stream_ptr())
    return dx


def construct_block_fwd(x, helper=NSAHelper):
    """x [T,H,D] -> [y_len,H,kernel,D] (im2col of the compression windows)."""
    check_thd(x, "x")
    T, H, D = x.shape
    y = torch.empty(helper.y_len, H, helper.kernel_size, D, device=x.device, dtype=x.dtype)
    _lib.call("nsa_construct_block_fwd", x.data_ptr(), x.stride(0), x.stride(1), y.data_ptr(),
              helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.y_maxlen, H, D,
              helper.kernel_size, helper.stride, _lib.stream_ptr())
    return y


def construct_block_bwd(x, dy, dx=None, helper=NSAHelper):
    T, H, D = x.shape
    dy = dy.contiguous()
    accumulate = dx is not None
    if dx is None:
        dx = torch.empty(T, H, D, device=x.device, dtype=x.dtype)
    else:
        assert dx.dtype == torch.float32 and dx.shape == x.shape and dx.stride(-1) == 1
    _lib.call("nsa_construct_block_bwd", dy.data_ptr(), dx.data_ptr(), dx.stride(0), dx.stride(1),
              int(dx.dtype == torch.float32), int(accumulate), helper.x_cu_seqlens.data_ptr(),
              helper.y_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, H, D, helper.kernel_size, helper.stride,
              _lib.stream_ptr())
    return dx


_ACT = {"linear": -1, "sigmoid-mul": 0, "swiglu": 1}


def takes_weight(x, weight, version, helper=NSAHelper):
    """Whether the kernels below take this weight (others go through the windows and the library's products).  Subclasses that wrap
    other tensors (quantised, distributed) have the shape and the type of a weight, but no memory of their own."""
    D, N = x.size(-1), (1 if version == "linear" else 2) * x.size(-1)
    return (type(weight) in (torch.nn.Parameter, torch.Tensor) and D % 32 == 0 and x.is_cuda and weight.device == x.device
            and x.dtype == weight.dtype == torch.bfloat16 and weight.shape == (N, helper.kernel_size * D) and weight.stride(1) == 1
            and weight.stride(0) % 8 == 0 and weight.data_ptr() % 16 == 0 and weight.data_ptr() != 0
            and not (weight.numel() > MIB and _faster_by_products(helper.y_len * x.size(1), weight.numel(), D)))


MIB = 1 << 20


def _faster_by_products(rows, weight, D):
    """Whether the library's products of so many rows are faster than the kernels'.  These read a weight of more than 4 MB (2 M numbers)
    from behind an XCD's L2 again for every tile of rows, and the sums of dW's parts grow with it.  Forward and backward, us, kernels /
    windows and library, by rows: 256 channels, gated: 250 85 / 55, 1000 109 / 96, 3000 222 / 181, 8200 585 / 481, 65500 4175 / 2977; linear:
    250 60 / 44, 500 64 / 60, 1000 72 / 82, 32800 1251 / 1410, 48000 1823 / 1862 (forward 595 / 481), 131000 4990 / 4676 (short batches save 80 us
    of the host with the kernels, and attention of 256 channels waits for it up to 100 rows: staged steps of 16 / 4 heads, 300 tokens, 68
    rows, 630 / 840, 700 tokens, 172 rows, 968 / 935).  192, gated: 2000 104 / 119, 3000 162 / 146, 6000 263 / 255, 16400 656 / 690, 65500 2440 /
    2253 (the forward alone: 6000 91 / 70, 16400 187 / 175); linear: 32800 962 / 1073, 48000 1405 / 1466, 65500 1948 / 1861, 262000 7996 / 6842.
    Smaller weights: 128, gated: 2000 68 / 110, 65500 1146 / 1428, 262000 4632 / 5125."""
    if D > 192:
        return rows > 100 and (weight > 2 * MIB or not 700 < rows <= 40000)
    return rows > (2500 if weight > 2 * MIB else 40000)


def weight_rows(weight):
    """weight, or a copy of it where its layout is not one that takes_weight accepts."""
    if weight.stride(1) == 1 and weight.stride(0) % 8 == 0 and weight.data_ptr() % 16 == 0:
        return weight
    return weight.clone(memory_format=torch.contiguous_format)


def compress_linear_fwd(x, weight, version, helper=NSAHelper, keep=True):
    """x [T,H,D], weight [N, kernel*D] -> hidden [y_len,H,N], the product of the windows and the weight, and the compressed rows
    [y_len,H,D], its activation ("linear": itself).  keep=False: nobody asks for hidden."""
    check_thd(x, "x")
    H, D = x.shape[1:]
    N, act = weight.size(0), _ACT[version]
    hidden = torch.empty(helper.y_len, H, N, device=x.device, dtype=x.dtype) if keep or act < 0 else None
    out = hidden if act < 0 else torch.empty(helper.y_len, H, D, device=x.device, dtype=x.dtype)
    _lib.call("nsa_compress_linear_fwd", x.data_ptr(), x.stride(0), x.stride(1), weight.data_ptr(), weight.stride(0),
              _lib.ptr(hidden), out.data_ptr(), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch,
              helper.y_maxlen, H, D, helper.kernel_size, helper.stride, N, act, _lib.stream_ptr())
    return hidden, out


def compress_linear_bwd_x(x, weight, dhidden, dx=None, helper=NSAHelper):
    """The gradient with respect to x, added to the fp32 dx, if given, in bf16."""
    T, H, D = x.shape
    dst = torch.empty(T, H, D, device=x.device, dtype=x.dtype)
    dxs = (None, 0, 0) if dx is None else (dx.data_ptr(), dx.stride(0), dx.stride(1))
    _lib.call("nsa_compress_linear_bwd_dx", dhidden.data_ptr(), weight.data_ptr(), weight.stride(0), *dxs, dst.data_ptr(),
              dst.stride(0), dst.stride(1), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch,
              helper.x_maxlen, H, D, helper.kernel_size, helper.stride, weight.size(0), _lib.stream_ptr())
    return dst


def compress_linear_bwd_weight(x, weight, dhidden, dw=None, helper=NSAHelper):
    """dW in a new bf16 tensor, or added to the fp32 dw."""
    H, D = x.shape[1:]
    N, f32 = weight.size(0), dw is not None
    if not helper.y_len:
        return dw if f32 else torch.zeros(weight.shape, device=x.device, dtype=x.dtype)
    if not f32:
        dw = torch.empty(weight.shape, device=x.device, dtype=x.dtype)
    n = _lib.value("nsa_compress_linear_bwd_dw_ws_bytes", helper.y_len, H, D, helper.kernel_size, N)
    ws = torch.empty(n, dtype=torch.uint8, device=x.device)
    _lib.call("nsa_compress_linear_bwd_dw", dhidden.data_ptr(), x.data_ptr(), x.stride(0), x.stride(1), dw.data_ptr(), int(f32),
              helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.y_len, H, D,
              helper.kernel_size, helper.stride, N, ws.data_ptr(), n, _lib.stream_ptr())
    return dw


def compress_linear_bwd(x, weight, hidden, dout, dx, version, dw=None, helper=NSAHelper):
    """From the fp32 gradient dout of the compressed rows: (the bf16 sum of the fp32 dx and the gradient with respect to x, dw).
    dw: None for a new bf16 tensor, else an fp32 one that is added to."""
    H, D = x.shape[1:]
    weight, hidden = weight_rows(weight), thd_rows(hidden.contiguous())  # (saved-tensor hooks may give them back in any layout)
    assert dout.dtype == dx.dtype == torch.float32 and dout.is_contiguous() and dx.stride(-1) == 1
    dhidden = torch.empty(helper.y_len, H, weight.size(0), device=x.device, dtype=x.dtype)
    _lib.call("nsa_compress_act_bwd", hidden.data_ptr(), dout.data_ptr(), dhidden.data_ptr(), helper.y_len * H, D, _ACT[version],
              _lib.stream_ptr())
    return (compress_linear_bwd_x(x, weight, dhidden, dx, helper), compress_linear_bwd_weight(x, weight, dhidden, dw, helper))


def mean_pooling_bwd_sum(x, dout, dx, helper=NSAHelper):
    """The bf16 sum of the fp32 dx and the gradient of mean pooling, from the fp32 gradient dout of its rows."""
    T, H, D = x.shape
    assert dout.dtype == dx.dtype == torch.float32 and dout.is_contiguous() and dx.stride(-1) == 1
    dst = torch.empty(T, H, D, device=x.device, dtype=x.dtype)
    _lib.call("nsa_mean_pool_bwd_sum", dout.data_ptr(), dx.data_ptr(), dx.stride(0), dx.stride(1), dst.data_ptr(), dst.stride(0),
              dst.stride(1), helper.x_cu_seqlens.data_ptr(), helper.y_cu_seqlens.data_ptr(), helper.batch, helper.x_maxlen, H, D,
              helper.kernel_size, helper.stride, _lib.stream_ptr())
    return dst


class _MeanPooling(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.helper = NSAHelper.get_bwd_helper()
        ctx.x_meta = x
        return mean_pooling_fwd(x)

    @staticmethod
    def backward(ctx, dy):
        return mean_pooling_bwd(ctx.x_meta, dy.contiguous(), helper=ctx.helper)


class _ConstructBlock(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, helper):
        ctx.helper = NSAHelper.get_bwd_helper() if helper is None else helper
        ctx.x_meta = x
        return construct_block_fwd(x, ctx.helper)

    @staticmethod
    def backward(ctx, dy):
        return construct_block_bwd(ctx.x_meta, dy, helper=ctx.helper), None


class _CompressLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, version):
        ctx.helper, ctx.version = NSAHelper.get_bwd_helper(), version
        needed = any(ctx.needs_input_grad[:2])
        hidden, out = compress_linear_fwd(x, weight, version, keep=needed)
        ctx.save_for_backward(x, weight, None if version == "linear" else hidden)
        return out

    @staticmethod
    def backward(ctx, dout):
        x, weight, hidden = ctx.saved_tensors
        # (the products read whole 16 bytes; a contiguous gradient may still be a view that begins between them, and so may what
        # saved-tensor hooks give back)
        x, weight = thd_rows(x), weight_rows(weight)
        dhidden = thd_rows(dout.contiguous()) if hidden is None else _glu_bwd(hidden, dout, ctx.version, inplace=False)
        dx = compress_linear_bwd_x(x, weight, dhidden, helper=ctx.helper) if ctx.needs_input_grad[0] else None
        if not ctx.needs_input_grad[1]:
            dw = None
        elif torch.is_grad_enabled():  # create_graph: dW is differentiated again, as a product of the gradient and the windows
            dw = torch.matmul(dhidden.flatten(0, 1).t(), _ConstructBlock.apply(x, ctx.helper).flatten(0, 1).flatten(1))
        else:
            dw = compress_linear_bwd_weight(x, weight, dhidden, helper=ctx.helper)
        return dx, dw, None


def compress_linear(x, weight, version):
    """Windows, product with the weight and activation in one autograd node (weights of takes_weight)."""
    return _CompressLinear.apply(x, weight, version)


def mean_pooling(x):
    return _MeanPooling.apply(x)


def construct_block(x):
    return _ConstructBlock.apply(x, None)
