"""CPU-side checks: the built library exports every symbol the C header declares (no compute calls), the host
metadata logic, and the config validation."""
import ctypes
import os

import pytest
import torch


def test_library_exports_every_declared_symbol():
    from flash_nsa import _lib
    protos = _lib.parse_header()
    assert len(protos) >= 25
    assert os.path.exists(_lib.LIB_PATH), "libnsa_hip.so is not built (run __graft_entry__.build())"
    dll = ctypes.CDLL(_lib.LIB_PATH)
    for name in protos:
        assert hasattr(dll, name), f"{name} is declared in include/nsa_hip.h but not exported"
    dll.nsa_abi_version.restype = ctypes.c_int
    assert dll.nsa_abi_version() >= 1


def test_entry_points_reject_bad_arguments_without_a_gpu():
    from flash_nsa import _lib
    with pytest.raises(RuntimeError, match="multiple of 8"):
        _lib.call("nsa_mean_pool_fwd", None, 0, 0, None, 0, 0, None, None, 1, 1, 1, 12, 32, 16, None)
    with pytest.raises(RuntimeError, match="power of 2"):
        _lib.call("nsa_cmp_attn_fwd", None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, None, 1, 8, 16,
                  1, 128, 128, 32, 12, 1.0, None)
    with pytest.raises(RuntimeError, match="kv heads"):
        _lib.call("nsa_swa_fwd", None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, 1, 8, 16, 3, 128,
                  128, 512, 1.0, None)
    with pytest.raises(RuntimeError, match="unsupported head dims"):
        _lib.call("nsa_swa_fwd", None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, 0, 0, None, 1, 8, 16, 1, 96,
                  96, 512, 1.0, None)
    with pytest.raises(RuntimeError, match="csr_slot"):  # the list of nsa_build_inverse_index_from, without the places of dS
        _lib.call("nsa_slc_attn_bwd_dkdv_ds", *(None, 128, 128) * 6, None, 128, 128, None, 128, 128, None, None, None, None, None,
                  None, None, 1, 64, 1, 1, 16, 1, 128, 128, 64, 4, 0, 8, 0.1, 1 << 20, 1 << 30, None)


@pytest.mark.parametrize("N,act", [(64, -1), (128, 0), (128, 1)])
def test_learned_compression_of_no_windows_has_nothing_to_do(N, act):
    """Sequences that are all shorter than a window: the compressed rows are empty tensors, whose addresses are null."""
    from flash_nsa import _lib
    _lib.call("nsa_compress_linear_fwd", None, 64, 64, None, 2048, None, None, None, None, 2, 0, 1, 64, 32, 16, N, act, None)
    with pytest.raises(RuntimeError, match="no output"):
        _lib.call("nsa_compress_linear_fwd", None, 64, 64, None, 2048, None, None, None, None, 2, 1, 1, 64, 32, 16, N, act, None)


def test_learned_compression_takes_only_weights_with_memory_of_their_own():
    """A weight that wraps another tensor looks like one that the kernels take, but has no address: it stays with the library."""
    from types import SimpleNamespace
    from flash_nsa import NSAHelper
    from flash_nsa.ops.compress_kv import takes_weight
    from gpu_util import Wrapper
    NSAHelper.set_hyperparameters()
    x = SimpleNamespace(size=lambda i: 64, is_cuda=True, device=torch.device("cpu"), dtype=torch.bfloat16)
    w = torch.randn(64, 32 * 64).bfloat16()
    wrapped = Wrapper(w)
    assert wrapped.dtype == w.dtype and wrapped.shape == w.shape and wrapped.stride() == w.stride()
    assert takes_weight(x, w, "linear") and takes_weight(x, torch.nn.Parameter(w), "linear")
    assert not takes_weight(x, wrapped, "linear") and not takes_weight(x, torch.nn.Parameter(wrapped), "linear")


@pytest.mark.parametrize("D,version,heads,tokens,taken", [
    (256, "swiglu", 1, 1616, True), (256, "swiglu", 1, 1632, False),             # 100 and 101 rows
    (256, "linear", 4, 416, True), (256, "linear", 1, 1632, False), (256, "linear", 1, 11216, False), (256, "linear", 1, 11232, True),
    (192, "swiglu", 1, 40016, True), (192, "swiglu", 1, 40032, False),           # 2500 and 2501
    (256, "linear", 4, 160016, True), (256, "linear", 4, 160032, False),         # 40000 and 40004
    (192, "sigmoid-mul", 4, 160016, False), (192, "linear", 4, 160032, False),
    (128, "swiglu", 4, 1 << 20, True), (64, "linear", 8, 1 << 20, True)])
def test_long_products_with_wide_weights_stay_with_the_library(D, version, heads, tokens, taken):
    """The line lies at a number of rows that depends on the weight's size."""
    from types import SimpleNamespace
    from flash_nsa.ops.compress_kv import takes_weight
    helper = SimpleNamespace(kernel_size=32, y_len=(tokens - 32) // 16 + 1)
    x = SimpleNamespace(size=lambda i: (tokens, heads, D)[i], is_cuda=True, device=torch.device("cpu"), dtype=torch.bfloat16)
    w = torch.empty(D if version == "linear" else 2 * D, 32 * D, dtype=torch.bfloat16)
    assert takes_weight(x, w, version, helper) == taken


@pytest.mark.parametrize("shape,tokens,longest,deterministic,two", [
    ((16, 1, 128, 128), 4096, 4096, False, False), ((16, 1, 128, 128), 6000, 6000, False, True),      # dS is stored
    ((32, 2, 192, 128), 2000, 2000, False, True), ((64, 4, 128, 128), 1024, 1024, False, False),
    ((16, 1, 128, 128), 1500, 1500, True, True), ((16, 1, 128, 128), 4800, 400, True, False),         # ordered sums
    ((12, 4, 128, 128), 2000, 2000, False, False), ((12, 4, 128, 128), 3000, 3000, False, True),      # groups of other sizes
    ((8, 8, 32, 32), 2000, 2000, False, False), ((8, 8, 32, 32), 3000, 3000, False, True),
    ((12, 4, 128, 128), 5600, 700, False, False), ((24, 8, 128, 128), 5600, 700, False, True),        # every block selected
    ((16, 16, 64, 64), 5600, 700, False, False), ((16, 16, 64, 64), 24000, 1000, False, True),
    ((16, 4, 256, 256), 1000, 1000, False, False), ((16, 4, 256, 256), 4800, 400, False, True),       # wide channels
    ((16, 1, 128, 128), 0, 0, False, False)])
def test_batches_that_gain_from_a_second_stream(shape, tokens, longest, deterministic, two):
    """The fused backward forks for these batches and not for those, by the kernels that their shapes have."""
    from types import SimpleNamespace
    from flash_nsa.modules.megatron_level_nsa import _gains_from_overlap
    QH, KH, D, VD = shape
    q, v = torch.empty(tokens, QH, D, device="meta"), torch.empty(tokens, KH, VD, device="meta")
    helper = SimpleNamespace(x_maxlen=longest, all_below=lambda: 1024, deterministic=deterministic)
    assert _gains_from_overlap(q, v, helper) == two


def test_weights_of_any_layout_are_copied_for_the_kernels():
    """What saved-tensor hooks give back may begin anywhere and lie in any order: the kernels get whole, aligned rows."""
    from flash_nsa.ops.compress_kv import weight_rows
    flat = torch.randn(8 * 64 + 16).bfloat16()
    at = -flat.data_ptr() // 2 % 8  # the first 16-byte boundary
    view = lambda offset: flat[at + offset:at + offset + 512].view(8, 64)
    wide = torch.randn(8, 72).bfloat16()
    for same in (view(0), view(8), wide[:, :64]):
        assert weight_rows(same) is same
    for other in (view(1), view(4), view(0).view(64, 8).t(), torch.randn(8, 65).bfloat16()[:, :64]):
        got = weight_rows(other)
        assert torch.equal(got, other) and got.is_contiguous() and got.data_ptr() % 16 == 0


def test_weight_gradients_are_added_to_aligned_buffers_by_the_kernels():
    """Other places of a main_grad are left to the library's product, which takes any."""
    from flash_nsa.modules.megatron_level_nsa import _kernels_add_to
    from gpu_util import Wrapper
    w = torch.empty(8, 64, dtype=torch.bfloat16)
    flat = torch.zeros(2 * w.numel() + 64)
    at = -flat.data_ptr() // 4 % 4  # the first 16-byte boundary
    view = lambda offset: flat[at + offset:at + offset + w.numel()].view(w.shape)
    assert _kernels_add_to(view(0), w) and _kernels_add_to(view(4), w)
    assert not any(_kernels_add_to(view(n), w) for n in (1, 2, 3))
    wide = torch.zeros(8, 128)
    for other in (wide[:, :64], view(0).t(), view(0).bfloat16(), view(0).view(-1), Wrapper(view(0))):
        assert not _kernels_add_to(other, w)


def test_learned_compression_refuses_null_operands():
    """The entry points of learned compression name a missing operand instead of launching on it."""
    from flash_nsa import _lib
    some, sizes = 1 << 20, (1, 8, 1, 64, 32, 16)  # never dereferenced: every call below is refused
    for x, w in ((None, some), (some, None)):
        with pytest.raises(RuntimeError, match="null"):
            _lib.call("nsa_compress_linear_fwd", x, 64, 64, w, 2048, some, some, some, some, *sizes, 64, -1, None)
    for dhidden, w, n in ((None, some, 40), (some, None, 40), (None, None, 20)):
        with pytest.raises(RuntimeError, match="null"):
            _lib.call("nsa_compress_linear_bwd_dx", dhidden, w, 2048, None, 0, 0, some, 64, 64, some, some, 1, n, 1, 64, 32, 16, 64, None)
    for dhidden, x, dw, ws in ((None, *(some,) * 3), (some, None, some, some), (some, some, None, some), (*(some,) * 3, None)):
        with pytest.raises(RuntimeError, match="null"):
            _lib.call("nsa_compress_linear_bwd_dw", dhidden, x, 64, 64, dw, 0, some, some, *sizes, 64, ws, 1 << 30, None)
    for hidden, dy, dhidden in ((None, some, some), (some, None, some), (some, some, None)):
        with pytest.raises(RuntimeError, match="null"):
            _lib.call("nsa_compress_act_bwd", hidden, dy, dhidden, 8, 64, 0, None)
    for dy, dx, dst in ((None, some, some), (some, None, some), (some, some, None)):
        with pytest.raises(RuntimeError, match="null"):
            _lib.call("nsa_mean_pool_bwd_sum", dy, dx, 64, 64, dst, 64, 64, some, some, 1, 40, 1, 64, 32, 16, None)


@pytest.mark.parametrize("kind", ["forward_hook", "forward_pre_hook", "full_backward_hook", "full_backward_pre_hook"])
def test_hooks_of_a_linear_layer_are_seen(kind):
    """Hooks on the layer and hooks on all modules: learned compression calls a layer that anything waits for."""
    from flash_nsa.modules.hf_level_nsa import _hooked
    fc, fn = torch.nn.Linear(4, 4), lambda *a: None
    assert not _hooked(fc)
    for register in (getattr(fc, "register_" + kind), getattr(torch.nn.modules.module, "register_module_" + kind)):
        handle = register(fn)
        try:
            assert _hooked(fc)
        finally:
            handle.remove()
        assert not _hooked(fc)


def test_tangents_of_a_weight_are_seen():
    """Inside forward-mode differentiation, the tensors that carry a tangent and no others."""
    from flash_nsa.modules.hf_level_nsa import _has_tangent
    from torch.autograd import forward_ad
    w = torch.nn.Parameter(torch.randn(4, 4))
    assert not _has_tangent(w)
    with forward_ad.dual_level():
        assert not _has_tangent(w)
        assert _has_tangent(forward_ad.make_dual(w.detach(), torch.ones(4, 4)))
    assert not _has_tangent(w)


def test_nsa_helper_metadata():
    from flash_nsa import NSAHelper
    NSAHelper.set_hyperparameters()
    cu = torch.tensor([0, 31, 63, 163, 163, 4259], dtype=torch.int32)
    NSAHelper.init_cu_seqlens(cu)
    assert NSAHelper.batch == 5
    assert NSAHelper.x_maxlen == 4096
    assert NSAHelper.y_seqlens.tolist() == [0, 1, 5, 0, 255]
    assert NSAHelper.y_cu_seqlens.tolist() == [0, 0, 1, 6, 6, 261]
    assert NSAHelper.k_seqlens.tolist() == [1, 1, 2, 0, 64]
    assert NSAHelper.k_len == 68 and NSAHelper.y_len == 261 and NSAHelper.y_maxlen == 255
    assert NSAHelper.blk_seq.tolist() == [0, 1, 2, 2] + [4] * 64
    # changing the hyper-parameters invalidates the cached batch
    NSAHelper.set_hyperparameters(kernel_size=64, stride=32, block_size=128)
    NSAHelper.init_cu_seqlens(cu)
    assert NSAHelper.y_seqlens.tolist() == [0, 0, 2, 0, 127]
    NSAHelper.set_hyperparameters()


def test_config_validation(tmp_path):
    from flash_nsa import NSAConfig
    c = NSAConfig(head_dim=64)
    assert c.qk_head_dim == 64 and c.v_head_dim == 64
    with pytest.raises(AssertionError):
        NSAConfig(stride=12)
    with pytest.raises(AssertionError):
        NSAConfig(kernel_size=40)
    with pytest.raises(AssertionError):
        NSAConfig(block_size=16)
    p = tmp_path / "c.json"
    p.write_text('{"num_heads": 32, "top_n": 8, "slc_block_size": 64}')
    c = NSAConfig.from_json(str(p))
    assert c.num_heads == 32 and c.top_n == 8 and c.slc_block_size == 64


def test_bench_flop_model_matches_closed_form():
    import bench
    nc, ns, nw = bench.branch_counts([65536])
    assert (nc, ns, nw) == (134123535, 66617344, 33488640)
    f = bench.stage_flops([65536], 64, 128, 128)
    assert abs(f["fwd_total"] / 1e12 - 9.87) < 0.01
    assert abs(f["bwd_total"] / 1e12 - 19.19) < 0.01


@pytest.mark.parametrize("name", ["random", "clustered"])
def test_bench_selection_patterns_name_every_block_once(name):
    """The list builder counts on a query's blocks being different and none behind its own."""
    import bench
    T = 9000
    topk = bench.selection_pattern(name, T, 2, "cpu")
    cur = torch.arange(T) // 64
    slot = torch.arange(16)
    used = slot < (cur[:, None] + 1).clamp(max=16)
    ids = torch.where(used, topk, -1 - slot.int())
    assert (ids.sort(-1).values.diff(dim=-1) > 0).all()
    assert ((topk >= 0) & (topk <= cur[:, None]))[used.expand_as(topk)].all()


def test_helper_does_not_confuse_a_new_tensor_with_the_registered_one():
    """A second cu_seqlens tensor with other lengths must be re-registered even when it is as long as the first one
    (an allocator may even hand it the same address); the same unmodified object is recognised without a read."""
    import torch
    from flash_nsa import NSAHelper
    NSAHelper.set_hyperparameters()
    a = torch.tensor([0, 700, 960], dtype=torch.int32)
    NSAHelper.init_cu_seqlens(a)
    assert (NSAHelper.x_maxlen, NSAHelper.y_len) == (700, 42 + 15)
    del a
    b = torch.tensor([0, 400, 730], dtype=torch.int32)
    NSAHelper.init_cu_seqlens(b)
    assert (NSAHelper.x_maxlen, NSAHelper.y_len) == (400, 24 + 19)
    NSAHelper.init_cu_seqlens(b)
    assert NSAHelper.x_maxlen == 400
    b[1] = 330                      # in-place edit of the registered tensor bumps its version
    NSAHelper.init_cu_seqlens(b)
    assert (NSAHelper.x_maxlen, NSAHelper.y_len) == (400, 19 + 24)
    assert NSAHelper._host_cu == [0, 330, 730]


def test_split_decode_lds_budget_counts_static_arrays():
    """nsa_decode_split_fits must imply dynamic + statically declared LDS <= 160 KB for the second launch: a
    capacity whose dynamic part alone fits but whose total does not has to be reported as not fitting, so that
    nsa_decode falls back instead of failing at launch.  Host arithmetic only."""
    from flash_nsa import _lib
    limit = 160 * 1024
    seen_near_limit = 0
    for D in (128, 64):
        for y in (512, 2048, 8192, 16384, 20000, 20480, 24576, 32768):
            for nb in (64, 512, 2048, 4096, 8192):
                prev_fit = True
                for tw in list(range(8, 6000, 97)):
                    fits = _lib.value("nsa_decode_split_fits", D, D, y, nb, tw)
                    total = _lib.value("nsa_decode_split_lds_total", D, D, y, nb, tw)
                    assert (total > 0) == bool(fits)
                    if fits:
                        assert 4288 < total <= limit, (D, y, nb, tw, total)
                        assert prev_fit, "a wider table cannot fit where a narrower one did not"
                        seen_near_limit += total > limit - 4288
                    prev_fit = bool(fits)
    assert seen_near_limit > 0, "the sweep must reach totals within the static part of the limit"


def test_two_launch_decode_lds_budget():
    """nsa_decode_two_launch_lds follows the kernels' layouts: staging slots of eight waves (32 rows of D + 24 bf16, or 16
    rows of VD + 4 fp32 where that is more), merge words, scores, tables.  What does not fit 160 KB is reported as 0, so
    that nsa_decode takes another route instead of failing at launch.  Host arithmetic only."""
    from flash_nsa import _lib
    limit, seen = 160 * 1024, set()
    up4 = lambda x: (x + 3) // 4 * 4
    for D, VD in ((128, 128), (64, 64), (192, 128)):
        slots = 8 * max(32 * (D + 24) * 2, 16 * (VD + 4) * 4)
        for y in (1, 512, 8192, 12800, 16384, 32768, 65536):
            for nb in (1, 64, 2048, 4096, 16384):
                for tw in (1, 512, 9000, 14000, 40000):
                    for page in (64, 256):
                        ntab = -(-y // page)
                        topk = slots + 4 * (2 * 8 * 16 + 16 + nb + up4(ntab) + y)
                        attend = slots + 4 * (2 * 8 * 16 + 192 + up4(tw)) + 4 * (3 * 16 + 64 * 16)
                        partial = slots // 2 + 4 * (2 * 4 * 16 + ntab)
                        for parts, n in ((0, max(topk, attend)), (1, max(partial, attend + 4 * up4(nb)))):
                            got = _lib.value("nsa_decode_two_launch_lds", D, VD, y, nb, tw, page, parts)
                            assert got == (n if n <= limit else 0), (D, y, nb, tw, page, parts)
                            seen.add((D, parts, got > 0))
    assert len(seen) == 12, "the sweep must have sizes on both sides of the limit for every kernel"
    # 192 channels, 16384 compressed rows and 4096 blocks: neither the one-launch nor the two-launch form holds them
    assert _lib.value("nsa_decode_fused_fits", 192, 128, 16384, 4096, 64, 256) == 0
    assert _lib.value("nsa_decode_two_launch_lds", 192, 128, 16384, 4096, 64, 256, 0) == 0


def test_inverse_index_refuses_more_blocks_than_its_histogram_holds():
    """The inverse index counts per selection block in an LDS histogram of 16384 entries: a batch with more blocks
    (more than 1048576 tokens at 64 per block) is refused with a message instead of launched."""
    from flash_nsa import _lib
    with pytest.raises(RuntimeError, match="exceed the LDS histogram"):
        _lib.call("nsa_build_inverse_index", None, 0, 0, 16, None, None, 1, 1 << 21, 4, 16385, 64, 1024, None, None,
                  None, None, 0, None)


@pytest.mark.parametrize("T", [700, 131072, 131073, 262144, 262145, 300001])
@pytest.mark.parametrize("QH,KH,top_n", [(16, 1, 6), (8, 1, 8), (64, 4, 16)])
def test_selected_backward_scratch_holds_every_range(monkeypatch, T, QH, KH, top_n):
    """Every range of tokens gets the dS, list and builder's scratch that the library asks for, all inside the one buffer."""
    import types
    from flash_nsa import _lib
    from flash_nsa.ops import select_attn
    nblk = -(-T // 64)
    one = torch.zeros(1, dtype=torch.int32)
    helper = types.SimpleNamespace(block_size=64, k_len=nblk, batch=1, x_cu_seqlens=one, k_cu_seqlens=one, blk_seq=one)
    tokens = _lib.value("nsa_slc_bwd_ds_tokens", T, 128, 128, KH * 128, QH, KH, 128, 128, 64, top_n, 128 ** -0.5)
    assert 0 < tokens <= T
    calls, buffers = [], []
    monkeypatch.setattr(select_attn._lib, "call", lambda *a: calls.append(a))
    monkeypatch.setattr(select_attn._lib, "stream_ptr", lambda: 0)
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: buffers.append(empty(*a, **kw)) or buffers[-1])
    meta = empty(KH, T, top_n, dtype=torch.int32)  # (never touched)
    grad = torch.zeros(1, 1, 1)
    select_attn._slc_attn_bwd_ds((0,) * 18, meta, grad, 2, None, grad, grad, (T, QH, KH, 128, 128), tokens, 0, 0.1, helper, None)
    (buf,) = buffers
    lo, hi = buf.data_ptr(), buf.data_ptr() + buf.numel()
    built = [a[1:] for a in calls if a[0] == "nsa_build_inverse_index_slots"]
    assert sum(a[8] for a in built) == T and [a[7] for a in built] == [sum(b[8] for b in built[:i]) for i in range(len(built))]
    for a in built:
        n, (csr_off, csr_tok, csr_slot, item_off, ws, ws_elems) = a[8], a[14:20]
        assert ws_elems >= _lib.value("nsa_inverse_index_workspace_elems", n, KH, nblk)
        parts = [(csr_off, 4 * KH * (nblk + 1)), (csr_tok, 4 * KH * n * top_n), (csr_slot, KH * n * top_n),
                 (item_off, 4 * KH * (nblk + 1)), (ws, 4 * ws_elems),
                 (lo, _lib.value("nsa_slc_bwd_ds_bytes", n, QH, KH, 64, top_n))]
        ends = [(at, at + size) for at, size in sorted(parts)]
        assert ends[0][0] >= lo and ends[-1][1] <= hi and all(x[1] <= y[0] for x, y in zip(ends, ends[1:]))
    del buf
    buffers.clear()


@pytest.mark.parametrize("QH,KH", [(16, 1), (8, 1), (64, 1), (64, 4), (128, 8)])
@pytest.mark.parametrize("block_size,top_n", [(32, 1), (64, 16), (64, 64), (512, 64), (2048, 64)])
@pytest.mark.parametrize("limit_mb", [None, 64])
def test_selected_backward_scratch_has_a_limit(QH, KH, block_size, top_n, limit_mb):
    """The stored dS keeps to its limit (beside one spare entry per kv head) at every length, or the shape takes the other
    kernels: also at every length, since a query's dq does not depend on the batch around it."""
    from flash_nsa import _lib
    if limit_mb is not None:
        _lib.call("nsa_set_tuning", b"slc_ds_mb", limit_mb)
    limit = (2048 if limit_mb is None else limit_mb) << 20
    size = lambda n: _lib.value("nsa_slc_bwd_ds_bytes", n, QH, KH, block_size, top_n)
    per_token = size(2) - size(1)
    taken = set()
    for T in (1, 100, 511, 513, 5000, 65536, 1000003):
        n = _lib.value("nsa_slc_bwd_ds_tokens", T, 128, 128, KH * 128, QH, KH, 128, 128, block_size, top_n, 128 ** -0.5)
        assert 0 <= n <= T and n * per_token <= limit
        taken.add(n > 0)
    assert taken == {512 * per_token <= limit}


def test_tuning_values_are_set_by_name_not_by_environment():
    from flash_nsa import _lib
    _lib.call("nsa_set_tuning", b"topk_seg_blocks", 64)
    _lib.call("nsa_reset_tuning")
    with pytest.raises(RuntimeError, match="unknown name"):
        _lib.call("nsa_set_tuning", b"no_such_value", 1)


@pytest.mark.parametrize("D", [32, 64, 128, 192, 256])
def test_slots_of_the_compressed_dkdv_follow_the_kernel_that_runs(D):
    """Two 32-key blocks per wave exist for 64 to 192 channels only; elsewhere the tuning value leaves the key tile at 128
    keys.  The slots (one key tile of fp32 rows per work item) and the launch that adds them up have to follow that, or the
    sums are taken from the wrong rows."""
    from flash_nsa import _lib
    VD = min(D, 128) if D < 256 else 256
    T, y, chunk, KH = 4096, 255, 256, 2
    need = {}
    for blocks in (1, 2):
        _lib.call("nsa_set_tuning", b"dkdv_key_blocks", blocks)
        need[blocks] = _lib.value("nsa_cmp_attn_bwd_dkdv_det_bytes", 1, T, y, 16, KH, D, VD, 32, 16, chunk)
        keys = 256 if blocks == 2 and 64 <= D <= 192 else 128
        items = sum(T // chunk - (16 * keys * kt + 31) // chunk for kt in range(-(-y // keys)))
        assert need[blocks] == items * KH * keys * (D + VD) * 4, (D, blocks)
    _lib.call("nsa_reset_tuning")


def test_unsupported_shapes_are_rejected_where_the_model_is_configured():
    """Block sizes that are not multiples of 32 and head dims that are not built fail in NSAConfig and in both
    cores' constructors (also for a plain attribute object), not at the first launch in the middle of a forward."""
    from types import SimpleNamespace
    from flash_nsa import NSAConfig, NSACore, HFNSACore
    NSAConfig(block_size=32)
    NSAConfig(block_size=256, kernel_size=64)
    NSAConfig(qk_head_dim=192, v_head_dim=128)
    with pytest.raises(AssertionError, match="multiples of 32"):
        NSAConfig(block_size=48)
    NSAConfig(head_dim=256)
    NSAConfig(head_dim=32)
    with pytest.raises(AssertionError, match="not built"):
        NSAConfig(head_dim=512)
    with pytest.raises(AssertionError, match="not built"):
        NSAConfig(qk_head_dim=256, v_head_dim=128)
    loose = SimpleNamespace(head_dim=128, qk_head_dim=None, v_head_dim=None, num_heads=16, num_kv_heads=1,
                            kernel_size=32, stride=16, block_size=80, cmp_k_method="mean", cmp_v_method="mean")
    for core in (NSACore, HFNSACore):
        with pytest.raises(AssertionError, match="multiples of 32"):
            core(loose)
    loose.block_size, loose.head_dim = 64, 96
    for core in (NSACore, HFNSACore):
        with pytest.raises(AssertionError, match="not built"):
            core(loose)


def test_ranges_of_stored_ds_cover_the_batch():
    """Ranges of whole 128-token groups, none shorter than the rows that fill the GPU, up to the last token."""
    from flash_nsa import _lib
    for T, B, longest, QH, KH in ((65536, 1, 65536, 64, 4), (48362, 8, 8192, 64, 4), (1 << 20, 1, 1 << 20, 64, 4),
                                  (70001, 3, 60000, 16, 1), (100, 2, 60, 8, 1)):
        at, ranges = 0, []
        while at < T:
            end = _lib.value("nsa_bwd_ds_next", at, T, B, longest, QH, KH, 32, 16, 512)
            ranges.append((at, end))
            at = end
        assert at == T and all(s % 128 == 0 for s, _ in ranges)
        assert len(ranges) == 1 or min(e - s for s, e in ranges) * QH >= 131072
        ring = max(e - s for s, e in ranges)
        for s, e in ranges:  # a range's tiles fit what the whole batch would take
            whole = _lib.value("nsa_cmp_attn_bwd_ds_bytes", T, B, longest, QH, KH, 32, 16, 0, 0)
            assert 0 < _lib.value("nsa_cmp_attn_bwd_ds_bytes", T, B, longest, QH, KH, 32, 16, s, e) <= whole
        assert 0 < _lib.value("nsa_swa_bwd_ds_bytes", T, B, longest, QH, KH, 512, ring) <= \
            _lib.value("nsa_swa_bwd_ds_bytes", T, B, longest, QH, KH, 512, 0)
    # no scratch where no query has keys before its window
    assert _lib.value("nsa_slc_bwd_before_window_ds_bytes", 5000, 1, 5000, 64, 4, 2000, 1024, 0) == 0


def test_grid_of_the_storing_dkdv_covers_every_share_of_a_range():
    """The compressed dk / dv launch that stores dS has one grid for all sequences of a range, in which each of them numbers
    its work items (key tile of 128, chunk of queries that sees it) from its own first row on."""
    import random
    from flash_nsa import _lib
    QH, KH, D, VD, W = 64, 4, 128, 128, 512
    rng = random.Random(5)
    batches = [([20480] * 2, 32, 16), ([45056] * 2, 32, 16), ([12288] * 10, 32, 16), ([65000], 32, 16), ([700] * 3, 32, 16)]
    for _ in range(60):
        longest = int(2 ** rng.uniform(9, 16))
        batches.append(([rng.randint(1, longest) for _ in range(rng.randint(1, 12))], *rng.choice(((32, 16), (64, 32), (16, 8)))))
    tight = 0
    for lens, kernel_size, stride in batches:
        T, B, longest = sum(lens), len(lens), max(lens)
        y = [max((n - kernel_size) // stride + 1, 0) for n in lens]
        cuts, at = [], 0
        while at < T:
            end = _lib.value("nsa_bwd_ds_next", at, T, B, longest, QH, KH, kernel_size, stride, W)
            cuts.append((at, end))
            at = end
        for a in range(0, T, max(T // 3 // 128, 1) * 128):  # and others than the library's
            cuts.append((a, min(a + rng.randint(1, 200) * 128, T)))
        for tok0, tok1 in ([(0, 0)] if len(cuts) == 1 else cuts):
            for chunk in (32, 64, 128, 256, 512, 1024, 2048):
                have = _lib.value("nsa_cmp_attn_bwd_dkdv_ds_items", B, longest, max(y), QH, KH, D, VD, kernel_size, stride,
                                  chunk, tok0, tok1)
                x0 = 0
                for n, keys in zip(lens, y):
                    lo, hi = 0, n
                    if tok1:
                        lo, hi = max(-(-(tok0 - x0) // 128) * 128, 0), min(-(-(tok1 - x0) // 128) * 128, n)
                    chunks, need = -(-max(hi - lo, 0) // chunk), 0
                    for first in range(kernel_size - 1, min(hi, kernel_size - 1 + stride * keys), stride * 128):
                        need += chunks - min(chunks, max(first - lo, 0) // chunk)
                    assert need <= have, (lens, (tok0, tok1), chunk, need, have)
                    tight += need == have > 0
                    x0 += n
    assert tight > 100


@pytest.mark.parametrize("lens,shape,settings", [
    ([65536], (64, 4), {}), ([8192] * 6, (64, 4), {}), ([20480] * 2, (64, 4), {}), ([1000] * 100, (64, 4), {}),
    ([4096] * 16, (64, 4), dict(top_n=64)),
    ([4096] * 64, (64, 4), dict(top_n=64, window_size=64)),
    ([8192] * 16, (64, 4), dict(block_size=128, top_n=64, window_size=64)),
    ([70001, 300, 2500], (16, 1), dict(top_n=40, window_size=0)),
    ([250000], (64, 4), {}), ([1 << 20], (64, 4), {}), ([1 << 20], (8, 1), {}), ([300000, 500], (32, 2), {}),
])
def test_scratch_of_stored_ds_is_bounded(lens, shape, settings):
    """No branch's dS takes more than its limit of 4 GB, whatever the settings, or there are no ranges; up to a million tokens
    there are.  A lower limit holds as well."""
    from flash_nsa import NSAHelper, _lib
    from flash_nsa.ops import bwd_ds
    from flash_nsa.utils import BwdNSAHelper

    def batch_of(lens):
        NSAHelper.init_cu_seqlens(torch.tensor([0, *lens]).cumsum(0).to(torch.int32))
        return BwdNSAHelper()

    T, (QH, KH) = sum(lens), shape
    q, k = torch.empty(T, QH, 128, device="meta"), torch.empty(T, KH, 128, device="meta")
    NSAHelper.set_hyperparameters(**settings)
    helper = batch_of(lens)
    fitted = 0
    for mb in (4096, 700, 0):
        _lib.call("nsa_set_tuning", b"dense_ds_mb", mb)
        for with_cmp, with_swa in ((True, True), (True, False), (False, True)):
            ds = bwd_ds.DenseDs(q, k, helper, with_cmp=with_cmp, with_swa=with_swa,
                                all_below=NSAHelper.all_below() if with_cmp and with_swa else 0)
            if not ds.fits:
                assert not ds.ranges and (mb < 4096 or settings.get("block_size") == 128)
                continue
            fitted += 1
            assert max(n for _, n in (ds.cmp, ds.swa, ds.far)) <= mb << 20
            assert (ds.cmp[1] > 0) == with_cmp and (ds.swa[1] > 0) == with_swa
    assert fitted > 0
    _lib.call("nsa_reset_tuning")
    # the same for a short batch: a query's dq is to be the same bits whatever follows it
    assert _lib.value("nsa_bwd_ds_range_end", 0, 500, 1, 500, QH, KH, 32, 16, 512, 2 ** 31 - 64) == -1
    assert _lib.value("nsa_bwd_ds_range_end", 0, 500, 1, 500, QH, KH, 32, 16, 2 ** 31 - 1, 2 ** 31 - 64) == 500
    short = bwd_ds.DenseDs(q[:500], k[:500], batch_of([500]), all_below=NSAHelper.all_below())
    assert short.fits == (settings.get("block_size") != 128)
    NSAHelper.set_hyperparameters()


@pytest.mark.parametrize("lens,behind,most", [
    ([60000] + [350] * 400, 0, 8), ([350] * 200 + [60000] + [350] * 200, 7, 9), ([16384] + [512] * 96, 0, 3), ([20480] * 2, 0, 2),
    ([12288] * 10, 0, 4), ([1000] * 100, 0, 2), ([0, 60000, 0, 0, 31, 500, 0], 0, 7), ([65536], 0, 6), ([300] * 20, 0, 1),
    ([1000] * 50, 50000, 1),  # rows of q behind the last sequence
])
def test_parts_of_a_batch_whose_stored_ds_takes_several_ranges(lens, behind, most):
    """A batch that one range does not hold is cut between its sequences, so that short ones do not get the width of the longest:
    every token in one part, in order; several ranges in parts of one sequence alone."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops import bwd_ds
    T, QH, KH = sum(lens), 64, 4
    NSAHelper.set_hyperparameters()
    cu = torch.tensor([0, *lens]).cumsum(0).to(torch.int32)
    NSAHelper.init_cu_seqlens(cu)
    ds = bwd_ds.DenseDs(torch.empty(T + behind, QH, 128, device="meta"), torch.empty(T + behind, KH, 128, device="meta"),
                        all_below=NSAHelper.all_below())
    assert ds.fits and len(ds.ranges) <= most
    parts = list(dict.fromkeys(p for p, *_ in ds.ranges))
    x, y = cu.tolist(), NSAHelper.y_cu_seqlens.tolist()
    seqs, at = [], 0
    for p in parts:
        b0 = max(b for b in range(len(lens)) if x[b] == p.x0 and lens[b:b + p.batch] and
                 [c + p.x0 for c in p.x_cu.tolist()] == x[b:b + p.batch + 1])
        assert p.x0 == at and p.T == p.x_cu.tolist()[-1] and p.y0 == y[b0]
        assert [c + p.y0 for c in p.y_cu.tolist()] == y[b0:b0 + p.batch + 1]
        assert p.x_maxlen == max(lens[b0:b0 + p.batch])
        assert p.y_maxlen == max(d - c for c, d in zip(p.y_cu.tolist(), p.y_cu.tolist()[1:]))
        assert len(p.ranges) == 1 or p.batch == 1
        seqs += range(b0, b0 + p.batch)
        at += p.T
        ends = [r[2] for r in ds.ranges if r[0] is p]
        starts = [r[1] for r in ds.ranges if r[0] is p]
        assert (starts, ends) == ([0], [0]) or (starts == [0] + ends[:-1] and ends[-1] == p.T and p.ring > 0)
    assert at == T and set(range(len(lens))) - set(seqs) <= {b for b, n in enumerate(lens) if n == 0}
    NSAHelper.set_hyperparameters()


def test_backward_of_the_selected_branch_takes_the_event_of_the_other_dq():
    import inspect
    from flash_nsa.ops.select_attn import slc_attn_bwd
    names = list(inspect.signature(slc_attn_bwd).parameters)
    assert names[-3:] == ["finalize_dq", "dq_after", "ds_tokens"]
