"""Learned compression without its windows in memory, against float64 (upstream flash_nsa/modules/megatron_level_nsa.py:46-86)."""
import pytest
import torch

from gpu_util import Wrapper, make_cu, make_qkvw, randn_bf16

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -9  # relative rounding error of bf16


def rel(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


def reference(x, w, version, lens, K, S, dout, dx):
    """hidden, out, dx + gradient and dw in float64; windows in the order (position, channel)."""
    x, w = x.double().requires_grad_(), w.double().requires_grad_()
    D, a, rows = x.shape[2], 0, []
    for n in lens:
        rows += [x[a + S * i:a + S * i + K].transpose(0, 1).reshape(x.shape[1], -1) for i in range(max((n - K) // S + 1, 0))]
        a += n
    hidden = torch.stack(rows) @ w.t()
    out = hidden
    if version != "linear":
        g = hidden[..., :D]
        out = torch.sigmoid(g) * (g if version == "swiglu" else 1) * hidden[..., D:]
    out.backward(dout.double())
    return hidden.detach(), out.detach(), x.grad + dx.double(), w.grad


@pytest.mark.parametrize("version", ["linear", "sigmoid-mul", "swiglu"])
@pytest.mark.parametrize("H,D,K,S,lens", [
    (4, 128, 32, 16, [700, 31, 32, 0, 47, 1000]),   # sequences without a window, with one, with tokens behind the last
    (1, 64, 32, 16, [300]),
    (3, 32, 32, 16, [200, 90, 17]),                 # one block of channels; rows of 128 hold heads of several windows
    (2, 192, 32, 16, [513, 64]),                    # three pairs of blocks; columns of a chunk not a multiple of 128 * 2
    (1, 256, 32, 16, [130]),
    (2, 64, 64, 16, [500, 100]),                    # four windows over a token
    (2, 128, 16, 16, [100, 15]),                    # windows that do not overlap
    (5, 64, 16, 4, [77, 33]),
    (1, 32, 8, 2, [40, 9]),                         # contraction shorter than the waves' parts; chunks of 64 columns
])
def test_learned_compression_against_float64(device, version, H, D, K, S, lens):
    from flash_nsa import NSAHelper
    from flash_nsa.ops import compress_kv as C
    T = sum(lens)
    try:
        NSAHelper.set_hyperparameters(kernel_size=K, stride=S)
        NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
        x = randn_bf16(T, 2, H, D, seed=1)[:, 1]    # a strided view
        N = D if version == "linear" else 2 * D
        w = (randn_bf16(N, K * D, seed=2).float() * (K * D) ** -0.5).to(torch.bfloat16)
        dx = randn_bf16(T, H, D, seed=3).float()
        xd, wd = x.to(device), torch.cat([w, w], 1).to(device)[:, :K * D]
        assert C.takes_weight(xd, wd, version)
        hidden, out = C.compress_linear_fwd(xd, wd, version)
        dout = randn_bf16(*out.shape, seed=4).float() + 1e-3
        base = torch.full((N, K * D), 0.25, device=device)
        dst, dw = C.compress_linear_bwd(xd, wd, hidden, dout.to(device), dx.to(device), version)
        dst2, added = C.compress_linear_bwd(xd, wd, hidden, dout.to(device), dx.to(device), version, base)
        want = reference(x, w, version, lens, K, S, dout, dx)
    finally:
        NSAHelper.set_hyperparameters()
    assert torch.equal(dst, dst2) and added is base
    # hidden: one rounding.  Its activation: that of gate and value, the gate's amplified by |g f'(g) / f(g)| <= 1 + |g| < 6, and
    # its own; the gradients: that of dout, of hidden through the activation's derivative, of dhidden, and their own.
    assert rel(hidden, want[0]) <= 1.02 * EPS
    assert rel(out, want[1]) <= (1.02 if version == "linear" else 8) * EPS
    assert rel(dst, want[2]) <= (3 if version == "linear" else 9) * EPS
    assert rel(dw, want[3]) <= (3 if version == "linear" else 9) * EPS
    assert rel(added - 0.25, want[3]) <= (2 if version == "linear" else 8) * EPS


@pytest.mark.parametrize("H,D,version,T", [(4, 128, "sigmoid-mul", 26000), (2, 192, "linear", 34000), (1, 32, "swiglu", 600)])
def test_compressed_rows_do_not_depend_on_the_batch(device, H, D, version, T):
    """Every form of the forward kernel sums a product in the same order: prefixes of 300 and 9000 tokens give the same bits."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops import compress_kv as C
    N = D if version == "linear" else 2 * D
    x, w = randn_bf16(T, H, D, seed=5).to(device), (randn_bf16(N, 32 * D, seed=6) / 64).to(device)
    NSAHelper.set_hyperparameters()
    rows = []
    for n in (T, min(9000, T), 300):
        NSAHelper.init_cu_seqlens(torch.tensor([0, n], dtype=torch.int32, device=device))
        rows.append(C.compress_linear_fwd(x[:n], w, version))
    for got in rows[1:]:
        for a, b in zip(got, rows[0]):
            assert torch.equal(a, b[:a.size(0)])


@pytest.mark.parametrize("H,D,K,S,lens", [(2, 64, 32, 16, [300, 5, 33]), (3, 128, 16, 4, [50, 0, 16]), (1, 32, 8, 8, [23])])
def test_mean_pooling_gradient_and_sum_in_one(device, H, D, K, S, lens):
    """The same bits as the gradient of the rounded rows added to the fp32 buffer, then rounded."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops import compress_kv as C
    T = sum(lens)
    try:
        NSAHelper.set_hyperparameters(kernel_size=K, stride=S)
        NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
        x = randn_bf16(T, H, D, seed=7).to(device)
        dout = torch.randn(NSAHelper.y_len, H, D, generator=torch.Generator().manual_seed(8)).to(device)
        dx = torch.randn(T, H, D, generator=torch.Generator().manual_seed(9)).to(device)
        got = C.mean_pooling_bwd_sum(x, dout, dx)
        want = C.mean_pooling_bwd(x, dout.to(torch.bfloat16), dx.clone()).to(torch.bfloat16)
    finally:
        NSAHelper.set_hyperparameters()
    assert torch.equal(got, want)


def test_weights_that_the_kernels_do_not_take_go_through_the_windows(device):
    """A weight whose rows are not 16-byte aligned: windows and library products, the same gradients to rounding."""
    from flash_nsa import NSAConfig, NSACore
    lens, D = [200, 77], 64
    q, k, v, w = [t.to(device) for t in make_qkvw(sum(lens), 8, 1, D, seed=10)]
    do = randn_bf16(sum(lens), 8, D, seed=11).to(device)
    cores = []
    for odd in (False, True):
        torch.manual_seed(0)
        core = NSACore(NSAConfig(head_dim=D, num_heads=8, num_kv_heads=1, cmp_k_method="linear", cmp_v_method="swiglu"))
        core = core.to(device=device, dtype=torch.bfloat16)
        if odd:
            for name in ("cmp_k_weight", "cmp_v_weight"):
                p = getattr(core, name).detach()
                wide = torch.empty(p.size(0), p.size(1) + 1, device=device, dtype=p.dtype)
                wide[:, :-1] = p
                setattr(core, name, torch.nn.Parameter(wide[:, :-1]))
        ts = [t.clone().requires_grad_() for t in (q, k, v, w)]
        out = core(*ts, make_cu(lens).to(device))
        out.backward(do)
        cores.append([out.detach()] + [t.grad for t in ts] + [core.cmp_k_weight.grad, core.cmp_v_weight.grad])
    for i, (a, b) in enumerate(zip(*cores)):
        assert a.dtype == b.dtype and rel(a, b.double().cpu()) < 2e-2, i  # (selections of near-tied blocks aside: all are selected)


@pytest.mark.parametrize("version", ["linear", "sigmoid-mul", "swiglu"])
@pytest.mark.parametrize("H,D,lens", [(2, 64, [300, 0, 31, 77]), (1, 128, [600])])
def test_module_with_and_without_its_windows(device, version, H, D, lens):
    """CompressKV computes a plain fc where the windows lie and calls one with a hook on them: the same to rounding, with the same
    gradient types, also with only one of the two gradients asked for and without any."""
    from flash_nsa import NSAConfig, NSAHelper
    from flash_nsa.modules.hf_level_nsa import CompressKV
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
    torch.manual_seed(0)
    mod = CompressKV(NSAConfig(head_dim=D), head_dim=D, version=version).to(device=device, dtype=torch.bfloat16)
    x = randn_bf16(sum(lens), H, D, seed=12).to(device)
    do = randn_bf16(NSAHelper.y_len, H, D, seed=13).to(device)

    def run():
        xs = x.clone().requires_grad_()
        mod.fc.weight.grad = None
        out = mod(xs)
        out.backward(do)
        return out.detach(), xs.grad, mod.fc.weight.grad

    plain, calls = run(), []
    hook = mod.fc.register_forward_hook(lambda *a: calls.append(1))
    through = run()
    hook.remove()
    assert calls
    for a, b in zip(plain, through):
        assert a.dtype == b.dtype and a.shape == b.shape and rel(a, b.double().cpu()) <= 8 * EPS
    with torch.no_grad():
        assert torch.equal(mod(x), plain[0])
    mod.fc.weight.requires_grad_(False)
    xs = x.clone().requires_grad_()
    mod(xs).backward(do)
    assert torch.equal(xs.grad, plain[1])
    mod.fc.weight.requires_grad_(True)
    mod.fc.weight.grad = None
    mod(x).backward(do)
    assert torch.equal(mod.fc.weight.grad, plain[2])


@pytest.mark.parametrize("methods", [("linear", "swiglu"), ("sigmoid-mul", "linear")])
@pytest.mark.parametrize("lens", [[20, 5, 0, 31], [1]])
def test_batches_without_a_window(device, methods, lens):
    """Every sequence is shorter than a window: no compressed row, so learned compression is mean pooling bit for bit and the weights'
    gradients are zero, in the fused and the staged core."""
    from flash_nsa import HFNSACore, NSAConfig, NSACore
    T, D = sum(lens), 64
    ins = [t.to(device) for t in make_qkvw(T, 8, 2, D, seed=14)]
    do, cu = randn_bf16(T, 8, D, seed=15).to(device), make_cu(lens).to(device)
    for Core in (NSACore, HFNSACore):
        runs = []
        for k_method, v_method in (methods, ("mean", "mean")):
            core = Core(NSAConfig(head_dim=D, num_heads=8, num_kv_heads=2, cmp_k_method=k_method, cmp_v_method=v_method))
            core = core.to(device=device, dtype=torch.bfloat16)
            ts = [t.clone().requires_grad_() for t in ins]
            out = core(*ts, cu)
            out.backward(do)
            with torch.no_grad():
                assert torch.equal(core(*ins, cu), out)
            runs.append([out.detach()] + [t.grad for t in ts])
            for p in core.parameters():
                assert p.grad.dtype == p.dtype and int(p.grad.count_nonzero()) == 0
        for a, b in zip(*runs):
            assert torch.equal(a, b)


@pytest.mark.parametrize("version", ["linear", "swiglu"])
def test_weights_that_wrap_another_tensor_go_through_the_library(device, version):
    """They have no memory of their own to hand to a kernel; their products are those of the tensor inside, to rounding."""
    from flash_nsa import NSAConfig, NSAHelper
    from flash_nsa.modules.hf_level_nsa import CompressKV
    from flash_nsa.modules.megatron_level_nsa import compress_kv_fwd
    lens, D = [200, 77], 64
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
    torch.manual_seed(0)
    mod = CompressKV(NSAConfig(head_dim=D), head_dim=D, version=version).to(device=device, dtype=torch.bfloat16)
    x = randn_bf16(sum(lens), 2, D, seed=16).to(device)
    with torch.no_grad():
        plain = mod(x)
        mod.fc.weight = torch.nn.Parameter(Wrapper(mod.fc.weight.detach()), requires_grad=False)
        for got in (mod(x), compress_kv_fwd(x, mod.fc.weight, version)[2]):
            assert rel(got, plain.double().cpu()) <= 8 * EPS


def test_hooks_on_all_modules_see_the_linear_layer(device):
    """A hook registered for every module (as FLOP counters do) fires for CompressKV's fc, forward and backward."""
    from flash_nsa import NSAConfig, NSAHelper
    from flash_nsa.modules.hf_level_nsa import CompressKV
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu([100]).to(device))
    mod = CompressKV(NSAConfig(head_dim=64), head_dim=64, version="linear").to(device=device, dtype=torch.bfloat16)
    x, seen = randn_bf16(100, 1, 64, seed=17).to(device).requires_grad_(), []
    m = torch.nn.modules.module
    handles = [m.register_module_forward_hook(lambda mod, *a: seen.append(("forward", mod))),
               m.register_module_full_backward_hook(lambda mod, *a: seen.append(("backward", mod)))]
    try:
        mod(x).float().sum().backward()
    finally:
        for h in handles:
            h.remove()
    assert ("forward", mod.fc) in seen and ("backward", mod.fc) in seen


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_autocast_decides_the_type_of_linear_compression(device, dtype):
    """CompressKV("linear") under autocast returns what its layer returns there."""
    from flash_nsa import NSAConfig, NSAHelper, construct_block
    from flash_nsa.modules.hf_level_nsa import CompressKV
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu([100]).to(device))
    mod = CompressKV(NSAConfig(head_dim=64), head_dim=64, version="linear").to(device=device, dtype=torch.bfloat16)
    x = randn_bf16(100, 1, 64, seed=18).to(device)
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
        got, want = mod(x), mod.fc(construct_block(x).flatten(-2, -1))
    assert got.dtype == want.dtype == dtype and rel(got, want.double().cpu()) <= 2 * EPS


@pytest.mark.parametrize("dout_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("version", ["mean", "linear", "sigmoid-mul", "swiglu"])
def test_compress_kv_functions_keep_their_contract(device, version, dout_dtype):
    """compress_kv_fwd returns the windows, compress_kv_bwd adds into the caller's fp32 buffer and returns it with dW, or with a function
    that computes it, from gradients of either type."""
    from flash_nsa import NSAHelper
    from flash_nsa.modules.megatron_level_nsa import compress_kv_bwd, compress_kv_fwd
    from flash_nsa.ops import compress_kv as C
    lens, H, D = [200, 20, 90], 2, 64
    T, N = sum(lens), D if version == "linear" else 2 * D
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
    x = randn_bf16(T, H, D, seed=19)
    w = None if version == "mean" else (randn_bf16(N, 32 * D, seed=20).float() * (32 * D) ** -0.5).to(torch.bfloat16)
    xd, wd = x.to(device), w if w is None else w.to(device)
    windows, hidden, out = compress_kv_fwd(xd, wd, version)
    dout = randn_bf16(*out.shape, seed=21).to(device, dout_dtype)
    runs = []
    for kw in ({}, {"async_dw": True}):
        dx = torch.ones(T, H, D, device=device)
        got, dw = compress_kv_bwd(xd, wd, windows, hidden, dout, dx, version, NSAHelper, **kw)
        assert got is dx
        runs.append((dx, dw() if callable(dw) else dw))
        assert callable(dw) == (version != "mean" and bool(kw))
    assert torch.equal(runs[0][0], runs[1][0])
    if version == "mean":
        assert windows is None and hidden is None and runs[0][1] is None
        assert torch.equal(dx, C.mean_pooling_bwd(xd, dout.to(torch.bfloat16), torch.ones_like(dx)))
        return
    assert torch.equal(windows, C.construct_block_fwd(xd)) and torch.equal(runs[0][1], runs[1][1])
    want = reference(x, w, version, lens, 32, 16, dout.cpu(), torch.ones(T, H, D))
    # as in test_learned_compression_against_float64; dx also has the rounding of the windows' gradient
    for a, b, n in ((hidden, want[0], 1.02), (out, want[1], 8), (dx, want[2], 10), (runs[0][1], want[3], 9)):
        assert rel(a, b) <= n * EPS


def test_gradients_that_begin_between_16_bytes(device, monkeypatch):
    """A gradient of the linear method that is contiguous at an odd offset: the kernels get an aligned copy, the results are those of
    an aligned gradient bit for bit."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops import compress_kv as C
    lens, H, D = [150, 60], 2, 64
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
    x, w = randn_bf16(sum(lens), H, D, seed=22).to(device), (randn_bf16(D, 32 * D, seed=23) / 32).to(device)
    do = randn_bf16(NSAHelper.y_len, H, D, seed=24).to(device)
    flat = torch.empty(do.numel() + 1, device=device, dtype=do.dtype)
    flat[1:] = do.flatten()
    seen, product = [], C.compress_linear_bwd_x
    monkeypatch.setattr(C, "compress_linear_bwd_x", lambda x, w, g, *a, **kw: seen.append(g.data_ptr() % 16) or product(x, w, g, *a, **kw))
    grads = []
    for g in (do, flat[1:].view(do.shape)):
        xs, ws = x.clone().requires_grad_(), w.clone().requires_grad_()
        C.compress_linear(xs, ws, "linear").backward(g)
        grads.append((xs.grad, ws.grad))
    assert seen == [0, 0]
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("version", ["linear", "swiglu"])
def test_weight_gradients_can_be_differentiated_again(device, version):
    """create_graph=True through CompressKV: a penalty on dW has the gradients that it has where the layer is called."""
    from flash_nsa import NSAConfig, NSAHelper
    from flash_nsa.modules.hf_level_nsa import CompressKV
    lens, H, D = [200, 20, 90], 2, 64
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
    torch.manual_seed(0)
    mod = CompressKV(NSAConfig(head_dim=D), head_dim=D, version=version).to(device=device, dtype=torch.bfloat16)
    x, do = randn_bf16(sum(lens), H, D, seed=25).to(device), randn_bf16(NSAHelper.y_len, H, D, seed=26).to(device)

    def penalty():
        xs, ds, mod.fc.weight.grad = x.clone().requires_grad_(), do.clone().requires_grad_(), None
        dw, = torch.autograd.grad((mod(xs) * ds).sum(), mod.fc.weight, create_graph=True)
        assert dw.requires_grad
        dw.float().pow(2).sum().backward()
        return [dw.detach(), xs.grad] + ([ds.grad] if version == "linear" else [])  # (nothing goes through the gate's gradient twice)

    plain = penalty()
    hook = mod.fc.register_forward_hook(lambda *a: None)
    called = penalty()
    hook.remove()
    # "linear": products of the same operands, dW rounded once on either side; its gradients have dW's rounding, that of a product and
    # their own on either side.  The gate: the 8 of test_module_with_and_without_its_windows in dW, and twice that and 4 behind it.
    for i, (a, b) in enumerate(zip(plain, called)):
        bound = {"linear": (2, 6), "swiglu": (8, 20)}[version][i > 0]
        assert rel(a, b.double().cpu()) <= bound * EPS


def test_a_tangent_of_the_weight_goes_through_the_linear_layer(device):
    """Forward-mode differentiation of CompressKV("linear") with respect to its weight: the product of the windows and the tangent."""
    from flash_nsa import NSAConfig, NSAHelper, construct_block
    from flash_nsa.modules.hf_level_nsa import CompressKV
    from torch.autograd import forward_ad
    NSAHelper.set_hyperparameters()
    NSAHelper.init_cu_seqlens(make_cu([100, 40]).to(device))
    mod = CompressKV(NSAConfig(head_dim=64), head_dim=64, version="linear").to(device=device, dtype=torch.bfloat16)
    x, dw = randn_bf16(140, 1, 64, seed=27).to(device), randn_bf16(64, 32 * 64, seed=28).to(device)
    plain = mod(x).detach()
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(mod.fc.weight.detach(), dw)
        out, tangent = forward_ad.unpack_dual(torch.func.functional_call(mod, {"fc.weight": dual}, (x,)))
        assert torch.equal(mod(x), plain)  # (a weight without a tangent beside it)
    windows = construct_block(x).flatten(-2, -1).double().cpu()
    assert rel(tangent, windows @ dw.double().cpu().t()) <= 1.02 * EPS
    assert rel(out, plain.double().cpu()) <= 2 * EPS


@pytest.mark.parametrize("core_name", ["NSACore", "HFNSACore"])
@pytest.mark.parametrize("k_method,v_method", [("linear", "swiglu"), ("sigmoid-mul", "linear")])
def test_saved_tensors_that_come_back_in_another_layout(device, core_name, k_method, v_method):
    """Saved-tensor hooks that keep weights at odd offsets and pre-activations in another order of their axes: the same gradients."""
    import flash_nsa
    lens, D, moved = [200, 77], 64, []
    T = sum(lens)
    core = getattr(flash_nsa, core_name)(flash_nsa.NSAConfig(head_dim=D, num_heads=8, num_kv_heads=2, cmp_k_method=k_method,
                                                             cmp_v_method=v_method)).to(device=device, dtype=torch.bfloat16)
    ins = [t.to(device) for t in make_qkvw(T, 8, 2, D, seed=29)]
    do, cu = randn_bf16(T, 8, D, seed=30).to(device), make_cu(lens).to(device)

    def pack(t):
        if t.dtype == torch.bfloat16 and t.dim() == 2:
            flat = torch.empty(t.numel() + 1, device=device, dtype=t.dtype)
            flat[1:] = t.detach().flatten()
            t = flat[1:].view(t.shape)
        elif t.dtype == torch.bfloat16 and t.size(-1) == 2 * D:
            t = t.detach().transpose(0, 1).contiguous().transpose(0, 1)
        else:
            return t
        moved.append(t)
        return t

    def grads():
        core.zero_grad()
        ts = [t.clone().requires_grad_() for t in ins]
        core(*ts, cu).backward(do)
        return [t.grad for t in ts] + [p.grad for p in core.parameters()]

    plain = grads()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        hooked = grads()
    assert len(moved) == 3 and sum(t.data_ptr() % 16 != 0 for t in moved) == 2 and sum(not t.is_contiguous() for t in moved) == 1
    for a, b in zip(hooked, plain):  # (dk, dv and what follows from them: sums of fp32 atomics)
        assert a.dtype == b.dtype and rel(a, b.double().cpu()) <= EPS
