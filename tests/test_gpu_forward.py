"""GPU parity of the forward operators against the CPU oracle (same seeded bf16 inputs).
Mirrors upstream test.py --func mean/construct/cmp/topk/slc/combine (test.py:74-318), with asserted tolerances."""
import math
import pytest
import torch

from oracle import nsa_oracle as O
from gpu_util import make_cu, make_qkvw, randn_bf16, assert_close

pytestmark = pytest.mark.gpu

LENS_CASES = [
    [1000],
    [5, 31, 32, 47, 48, 100, 333, 700],
    [64, 0, 129, 513],
]
HEAD_CASES = [(16, 1, 128), (8, 2, 128), (4, 4, 64)]


def setup_helper(cu_dev, **kw):
    from flash_nsa import NSAHelper
    NSAHelper.set_hyperparameters(**kw)
    NSAHelper.init_cu_seqlens(cu_dev)
    return NSAHelper


@pytest.mark.parametrize("lens", LENS_CASES)
def test_mean_pooling_and_construct_block(device, lens):
    from flash_nsa.ops.compress_kv import mean_pooling_fwd, construct_block_fwd
    cu = make_cu(lens)
    T = int(cu[-1])
    x = randn_bf16(T, 4, 128, seed=1)
    setup_helper(cu.to(device))
    y = mean_pooling_fwd(x.to(device))
    ref = O.mean_pooling(x.float(), cu)
    assert y.shape == ref.shape
    # fp32 mean rounded to bf16: allow one bf16 ulp of slack for summation order
    assert_close(y, ref, "mean_pooling", atol=2e-3, rtol=8e-3)
    blk = construct_block_fwd(x.to(device))
    refb = O.construct_block(x.float(), cu)
    assert torch.equal(blk.float().cpu(), refb)


@pytest.mark.parametrize("lens", LENS_CASES)
@pytest.mark.parametrize("QH,KH,D", HEAD_CASES)
def test_cmp_attn_fwd(device, lens, QH, KH, D):
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    cu = make_cu(lens)
    T = int(cu[-1])
    q, k, v, _ = make_qkvw(T, QH, KH, D, seed=10)
    setup_helper(cu.to(device))
    ck = mean_pooling_fwd(k.to(device))
    cv = mean_pooling_fwd(v.to(device))
    o, lse = cmp_attn_fwd(q.to(device), ck, cv)
    ro, rl = O.cmp_attn(q.float(), ck.float().cpu(), cv.float().cpu(), cu)
    assert_close(o, ro, "cmp_o")
    assert_close(lse, rl, "cmp_lse", atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("lens", LENS_CASES)
@pytest.mark.parametrize("QH,KH,D", HEAD_CASES)
def test_swa_fwd(device, lens, QH, KH, D):
    from flash_nsa.ops.sliding_window_attention import swa_fwd
    cu = make_cu(lens)
    T = int(cu[-1])
    q, k, v, _ = make_qkvw(T, QH, KH, D, seed=20)
    setup_helper(cu.to(device), window_size=200)
    o, lse = swa_fwd(q.to(device), k.to(device), v.to(device))
    ro, rl = O.swa(q.float(), k.float(), v.float(), cu, 200)
    assert_close(o, ro, "swa_o")
    assert_close(lse, rl, "swa_lse", atol=1e-3, rtol=1e-4)
    setup_helper(cu.to(device))


GROUP_CASES = [(32, 1, 128), (64, 1, 64), (16, 2, 128), (6, 3, 64), (12, 4, 64)]  # groups of 32, 64, 8, 2, 3


@pytest.mark.parametrize("lens,QH,KH,D", [(l, *h) for l in LENS_CASES for h in HEAD_CASES] +
                         [(LENS_CASES[1], *h) for h in GROUP_CASES])
def test_topk_and_slc_fwd(device, lens, QH, KH, D):
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.topk import slc_topk_indices
    from flash_nsa.ops.select_attn import slc_attn_fwd
    cu = make_cu(lens)
    T = int(cu[-1])
    q, k, v, _ = make_qkvw(T, QH, KH, D, seed=30)
    top_n = 6
    setup_helper(cu.to(device), top_n=top_n)
    cfg = O.OracleConfig(top_n=top_n)
    qd, kd, vd = q.to(device), k.to(device), v.to(device)
    ck = mean_pooling_fwd(kd)
    cv = mean_pooling_fwd(vd)
    _, lse = cmp_attn_fwd(qd, ck, cv)
    topk, probs = slc_topk_indices(qd, ck, lse, return_slc_prob=True)
    rt, imps = O.slc_topk(q.float(), ck.float().cpu(), None, cu, cfg, return_importance=True)
    assert topk.dtype == torch.int32 and topk.shape == (KH, T, top_n)
    n_rows, n_diff, n_bad = O.topk_mismatch_report(topk.cpu(), rt, imps, cu, 64, top_n, tie_tol=1e-3)
    assert n_bad == 0, f"{n_bad} rows differ beyond score ties ({n_diff} differing of {n_rows})"
    assert n_diff <= max(1, n_rows // 200)
    # slot order and ignore value: rows identical to the oracle wherever the sets agree
    same = (topk.cpu() == rt).all(-1)
    assert same.float().mean() > 0.99
    # block scores returned on request match the oracle's
    for b in range(len(lens)):
        a, e = int(cu[b]), int(cu[b + 1])
        nb = imps[b].shape[-1]
        if e > a:
            assert_close(probs[:, a:e, :nb], imps[b], "block scores", atol=2e-3, rtol=2e-3)
    # selected attention with the device's own indices fed to the oracle
    o, l2 = slc_attn_fwd(qd, kd, vd, topk)
    ro, rl = O.slc_attn(q.float(), k.float(), v.float(), topk.cpu(), cu, 64)
    assert_close(o, ro, "slc_o")
    assert_close(l2, rl, "slc_lse", atol=1e-3, rtol=1e-4)
    setup_helper(cu.to(device))


@pytest.mark.parametrize("lens,QH,KH,D", [([9000, 2500, 700], 32, 2, 128), ([6000, 100], 4, 4, 64),
                                          ([5000, 3000], 4, 2, 128), ([4500], 64, 1, 64)])
def test_topk_segmented_selection_equals_one_pass(device, lens, QH, KH, D):
    """Three forms of the block selector must return bit-identical indices and scores: the one-launch kernel with the
    scores of all blocks in LDS, the same kernel working segment by segment (long contexts; the segment length is a
    tuning value), and the two-launch form with the scores in a workspace -- in one pass over all tokens and in chunks
    of as many tokens as a small workspace holds.  All of them match the oracle."""
    from flash_nsa import _lib
    from flash_nsa.ops import topk as topk_mod
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.topk import slc_topk_indices
    cu = make_cu(lens)
    T = int(cu[-1])
    q, k, _, _ = make_qkvw(T, QH, KH, D, seed=33)
    setup_helper(cu.to(device))
    qd, kd = q.to(device), k.to(device)
    ck = mean_pooling_fwd(kd)
    _, lse = cmp_attn_fwd(qd, ck, ck)
    G = QH // KH
    results = {}
    try:
        _lib.call("nsa_set_tuning", b"topk_two_pass", 0)
        for seg in (0, 32, 64, 96):
            if seg == 0 and G <= 2:
                continue  # the score rows of 64 / 32 tokens per workgroup do not fit in one pass at this length
            _lib.call("nsa_set_tuning", b"topk_seg_blocks", seg)
            results[seg] = slc_topk_indices(qd, ck, lse, return_slc_prob=True)
    finally:
        _lib.call("nsa_reset_tuning")
    results["auto"] = slc_topk_indices(qd, ck, lse, return_slc_prob=True)
    limit = topk_mod.TOPK_WORKSPACE_LIMIT
    try:
        for small in (1 << 20, 300 << 10):   # a few hundred tokens per chunk, chunk edges inside sequences
            topk_mod.TOPK_WORKSPACE_LIMIT = small
            results[f"workspace {small}"] = slc_topk_indices(qd, ck, lse, return_slc_prob=True)
    finally:
        topk_mod.TOPK_WORKSPACE_LIMIT = limit
    keys = list(results)
    for key in keys[1:]:
        assert torch.equal(results[key][0], results[keys[0]][0]), f"indices differ: segment {key} vs {keys[0]}"
        assert torch.equal(results[key][1], results[keys[0]][1]), f"scores differ: segment {key} vs {keys[0]}"
    topk, probs = results["auto"]
    cfg = O.OracleConfig()
    rt, imps = O.slc_topk(q.float(), ck.float().cpu(), None, cu, cfg, return_importance=True)
    n_rows, n_diff, n_bad = O.topk_mismatch_report(topk.cpu(), rt, imps, cu, 64, 16, tie_tol=1e-3)
    assert n_bad == 0, f"{n_bad} rows differ beyond score ties ({n_diff} differing of {n_rows})"
    assert n_diff <= max(1, n_rows // 200)
    for b in range(len(lens)):
        a, e = int(cu[b]), int(cu[b + 1])
        assert_close(probs[:, a:e, :imps[b].shape[-1]], imps[b], "block scores", atol=2e-3, rtol=2e-3)


def test_combine_fwd(device):
    from flash_nsa.ops.combine import combine_fwd
    a, b, c = [randn_bf16(300, 8, 128, seed=s) for s in (1, 2, 3)]
    w = randn_bf16(300, 8, 3, seed=4)
    o = combine_fwd(a.to(device), b.to(device), c.to(device), w.to(device))
    assert_close(o, O.combine(a.float(), b.float(), c.float(), w.float()), "combine")


def _attend64(q, k, v, visible, scale):
    """softmax attention in float64: q [T,QH,D], k / v [N,KH,*], visible [KH,T,N] -> [T,QH,VD]; rows without keys are 0"""
    G = q.size(1) // k.size(1)
    out = []
    for h in range(q.size(1)):
        kk, vv = k[:, h // G].double(), v[:, h // G].double()
        s = (q[:, h].double() @ kk.t() * scale).masked_fill(~visible[h // G], float("-inf"))
        out.append(torch.nan_to_num(torch.softmax(s, -1), nan=0.0) @ vv)
    return torch.stack(out, 1)


@pytest.mark.parametrize("QH,KH,D,VD", [(16, 1, 128, 128), (8, 2, 64, 64), (3, 1, 32, 32), (4, 1, 192, 128),
                                        (2, 1, 256, 256)])
@pytest.mark.parametrize("T,window", [(33, 512), (700, 512), (1100, 100), (1400, 512)])
def test_gated_sum_of_the_window_launch_is_no_less_exact(device, QH, KH, D, VD, T, window):
    """The window launch continues its softmax into the selected branch of the queries that select everything, so the two
    branches' roundings of P no longer average out; it makes up for that by not rounding the rows it holds.  Its gated
    sum has to be no further from 64 bits than that of separately launched branches, with and without stored branches,
    and in the paged launch.  (A CPU model of the roundings puts it at 0.86 to 0.92 of the separate launches' error, and
    at 1.09 to 1.11 with rounded rows.)"""
    from flash_nsa.ops.combine import combine_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.select_attn import slc_attn_fwd
    from flash_nsa.ops.sliding_window_attention import swa_fwd, swa_fwd_tail
    from flash_nsa.ops.topk import slc_topk_indices
    from flash_nsa.inference.stages import swa_combine_prefill
    cu = make_cu([T])
    q, k, v, w = [x.to(device) for x in make_qkvw(T, QH, KH, D, VD, seed=170)]
    H = setup_helper(cu.to(device), window_size=window)
    n = H.all_below()
    ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
    cmp_o, lse = cmp_attn_fwd(q, ck, cv)
    topk, _ = slc_topk_indices(q, ck, lse)
    t = torch.arange(T, device=device)
    rows = torch.arange(ck.size(0), device=device)
    dist = t[:, None] - t[None]
    picked = torch.zeros(KH, T, (T + 63) // 64 + 1, dtype=torch.bool, device=device)
    slots = torch.arange(topk.size(-1), device=device) < (t // 64 + 1)[:, None]
    picked.scatter_(2, torch.where(slots, topk, picked.size(-1) - 1).long(), True)
    picked = picked[..., :-1].repeat_interleave(64, -1)[..., :T] & (dist >= 0)
    s = torch.sigmoid(w.double())
    sc = D ** -0.5
    seen = (t[:, None] >= 16 * rows + 31).expand(KH, -1, -1)
    exact = (_attend64(q, ck, cv, seen, sc) * s[..., :1] + _attend64(q, k, v, picked, sc) * s[..., 1:2] +
             _attend64(q, k, v, ((dist >= 0) & (dist <= window)).expand(KH, -1, -1), sc) * s[..., 2:])
    off = lambda o: float((o.double() - exact).norm() / exact.norm())
    separate = off(combine_fwd(cmp_o, slc_attn_fwd(q, k, v, topk)[0], swa_fwd(q, k, v)[0], w))
    for store in (True, False):
        so, sl = slc_attn_fwd(q, k, v, topk, t_begin=n)
        assert off(swa_fwd_tail(q, k, v, so, sl, n, cmp_o, w, store)[2]) <= separate, (store, separate)
    page = 64
    pages = -(-T // page)
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(1)).to(torch.int32)
    where = (table[torch.arange(T) // page].long() * page + torch.arange(T) % page).to(device)
    pools = []
    for x in (k, v):
        pool = torch.zeros(pages * page, KH, x.size(-1), device=device, dtype=x.dtype)
        pool[where] = x
        pools.append(pool.view(pages, page, KH, -1))
    so, _ = slc_attn_fwd(q, k, v, topk, t_begin=n)
    out = swa_combine_prefill(q, *pools, cmp_o, so, w, cu.to(device), T, table[None].to(device), cu[1:].to(device),
                              window_size=window, all_below=n)
    assert off(out) <= separate
    setup_helper(cu.to(device))


@pytest.mark.parametrize("QH,KH,D,VD", [(16, 1, 128, 128), (8, 2, 64, 64), (4, 1, 32, 32), (16, 1, 192, 128),
                                        (2, 1, 256, 256)])
def test_selected_and_window_branch_round_their_probabilities_apart(device, QH, KH, D, VD):
    """The selected branch attends the window's keys as well.  If it rounded P to the same bf16 values, the two branches'
    errors would add up in their gated sum: against float64 they have to be uncorrelated, 0.03 being far outside what 1000
    rows of two heads leave of independent roundings (below 0.01) and far inside what shared ones give (0.08 to 0.2).  Rows
    behind the window, where the branches differ by more than the rounding of the same output."""
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.select_attn import slc_attn_fwd
    from flash_nsa.ops.sliding_window_attention import swa_fwd
    from flash_nsa.ops.topk import slc_topk_indices
    T, W = 1513, 512
    cu = make_cu([T])
    q, k, v, _ = [x.to(device) for x in make_qkvw(T, QH, KH, D, VD, seed=230)]
    setup_helper(cu.to(device), window_size=W)
    ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
    topk, _ = slc_topk_indices(q, ck, cmp_attn_fwd(q, ck, cv)[1])
    t = torch.arange(T, device=device)
    dist = t[:, None] - t[None]
    picked = torch.zeros(KH, T, (T + 63) // 64 + 1, dtype=torch.bool, device=device)
    slots = torch.arange(topk.size(-1), device=device) < (t // 64 + 1)[:, None]
    picked.scatter_(2, torch.where(slots, topk, picked.size(-1) - 1).long(), True)
    picked = picked[..., :-1].repeat_interleave(64, -1)[..., :T] & (dist >= 0)
    near = ((dist >= 0) & (dist <= W)).expand(KH, -1, -1)
    a = (slc_attn_fwd(q, k, v, topk)[0].double() - _attend64(q, k, v, picked, D ** -0.5))[W + 1:]
    b = (swa_fwd(q, k, v)[0].double() - _attend64(q, k, v, near, D ** -0.5))[W + 1:]
    assert float((a * b).sum() / a.norm() / b.norm()) < 0.03
    setup_helper(cu.to(device))


@pytest.mark.parametrize("QH,KH,lens", [(8, 1, [1, 31, 63, 64, 65, 129]), (32, 2, [700, 1100]), (12, 2, [513, 40])])
def test_192_channels_staged_straight_into_lds(device, QH, KH, lens):
    """192 q/k channels: both staging variants of the dense kernels do the same arithmetic in the same order, so the branches,
    the window branch continued over earlier keys and the gated sum are the same bits."""
    from flash_nsa import HFNSACore, NSAConfig, NSACore, _lib
    cu = make_cu(lens).to(device)
    args = [t.to(device) for t in make_qkvw(sum(lens), QH, KH, 192, 128, seed=71)]
    cfg = NSAConfig(qk_head_dim=192, v_head_dim=128, num_heads=QH, num_kv_heads=KH, window_size=300)
    for core in (NSACore(cfg), HFNSACore(cfg)):
        with torch.no_grad():
            got = core(*args, cu)
            _lib.call("nsa_set_tuning", b"fwd_variant", 1)
            try:
                want = core(*args, cu)
            finally:
                _lib.call("nsa_reset_tuning")
        assert torch.equal(got, want)


@pytest.mark.parametrize("QH,KH,D,VD,lens", [
    (16, 1, 128, 128, [511, 512, 513, 1, 700]),       # top_n * block_size = 512: the window kernel finishes rows below it
    (12, 4, 64, 64, [40, 0, 640]),
    (8, 2, 192, 128, [300, 33]),                      # no query has blocks to choose from
])
def test_staged_core_without_gradients_is_the_staged_core(device, QH, KH, D, VD, lens):
    """Evaluation gives the training forward's output, bit for bit (a reentrant activation checkpoint runs its first pass
    without gradients and its second with them).  Sizes that the selector refuses are refused either way."""
    from flash_nsa import HFNSACore, NSAConfig
    cu = make_cu(lens).to(device)
    q, k, v, w = [t.to(device) for t in make_qkvw(sum(lens), QH, KH, D, VD, seed=72)]
    kw = dict(qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH, top_n=8, window_size=128)
    core = HFNSACore(NSAConfig(**kw))
    want = core(q.clone().requires_grad_(), k, v, w, cu)
    with torch.no_grad():
        got = core(q, k, v, w, cu)
        assert want.requires_grad and not got.requires_grad and torch.equal(got, want)
        core.num_local_blocks = 8  # with the initial block more than top_n
        with pytest.raises(RuntimeError):
            core(q, k, v, w, cu)


@pytest.mark.parametrize("G,D,edge", [(16, 128, 12288), (5, 128, 12288), (16, 192, 16384)])
def test_selected_branch_either_side_of_the_length_that_v_stays_in_registers_for(device, G, D, edge):
    """128 v channels: queries below `edge` transpose V in registers, later ones through LDS.  Both are the selected attention
    of their blocks, with a boundary unit of every size among them."""
    from flash_nsa.ops.select_attn import slc_attn_fwd
    T, first, top_n = edge + 70, edge - 70, 16
    cu = make_cu([T]).to(device)
    setup_helper(cu, top_n=top_n)
    q, k, v, _ = [x.to(device) for x in make_qkvw(T, G, 1, D, 128, seed=83)]
    g = torch.Generator().manual_seed(84)
    topk = torch.stack([torch.randperm(t // 64, generator=g)[:top_n] for t in range(first, T)]).to(torch.int32)
    topk[:, 5] = torch.arange(first, T) // 64  # the query's own block
    full = torch.zeros(1, T, top_n, dtype=torch.int32)
    full[0, first:] = topk
    o, lse = slc_attn_fwd(q, k, v, full.to(device), t_begin=first)
    keys = (topk.long()[:, :, None] * 64 + torch.arange(64)).reshape(T - first, -1).to(device)
    t = torch.arange(first, T, device=device)
    kk, vv = k[:, 0].float()[keys.clamp(max=T - 1)], v[:, 0].float()[keys.clamp(max=T - 1)]
    s = torch.matmul(q[first:].float(), kk.transpose(1, 2).contiguous()) * D ** -0.5
    s = s.masked_fill((keys > t[:, None])[:, None], float("-inf"))
    want = torch.matmul(s.softmax(-1), vv)
    assert_close(o[first:], want, "slc_o")
    assert_close(lse[first:], s.logsumexp(-1) / math.log(2.0), "slc_lse", atol=1e-3, rtol=1e-4)
    setup_helper(make_cu([64]).to(device))


@pytest.mark.parametrize("D", [128, 192])
def test_row_strides_that_a_32_bit_offset_does_not_hold(device, D):
    """K and V rows 302 MB apart (15 of them are more than 4 GB), full tiles of 64 and a partial one: the same bits as
    contiguous rows."""
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.sliding_window_attention import swa_fwd
    sr, n, G = (1 << 27) + (1 << 24), 74, 8
    for fwd, T in ((swa_fwd, n), (cmp_attn_fwd, 16 * (n - 1) + 32)):
        setup_helper(make_cu([T]).to(device))
        q = randn_bf16(T, G, D, seed=90).to(device)
        k, v = randn_bf16(n, 1, D, seed=91).to(device), randn_bf16(n, 1, 128, seed=92).to(device)
        want = fwd(q, k, v)
        wide = []
        for t in (k, v):
            wide.append(torch.empty((n - 1) * sr + 192, dtype=torch.bfloat16, device=device).as_strided(t.shape, (sr, 192, 1)))
            wide[-1].copy_(t)
        got = fwd(q, *wide)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        del wide
    torch.cuda.empty_cache()
    setup_helper(make_cu([64]).to(device))


@pytest.mark.parametrize("QH,KH,D,VD,lens", [
    (8, 2, 64, 64, [1100, 1, 0, 17, 700, 1040, 513]),
    (12, 3, 128, 128, [129, 640, 31]),                 # a row tile of 128 holds parts of tokens; odd number of kv heads
    (16, 1, 192, 128, [300, 33]),
])
def test_window_launch_of_few_workgroups_takes_last_rows_first(device, QH, KH, D, VD, lens):
    """The order of the workgroups changes no bit: sequences among so many others that the launch goes by rows equal the same
    sequences in a launch that starts with the last rows of all of them, and each alone."""
    from flash_nsa import NSAConfig, NSACore
    many = lens + [max(lens)] + [3] * (8192 * 128 // (max(lens) * QH) + 1)  # more than 8192 workgroups, most of them empty
    q, k, v, w = [t.to(device) for t in make_qkvw(sum(many), QH, KH, D, VD, seed=73)]
    core = NSACore(NSAConfig(qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH))
    with torch.no_grad():
        want = core(q, k, v, w, make_cu(many).to(device))
        n = sum(lens)
        got = core(q[:n], k[:n], v[:n], w[:n], make_cu(lens).to(device))
        assert torch.equal(got, want[:n])
        first = lens[0]
        assert torch.equal(core(q[:first], k[:first], v[:first], w[:first], make_cu([first]).to(device)), want[:first])


@pytest.mark.parametrize("QH,KH,D,VD,lens,kw", [
    (8, 2, 64, 64, [1, 31, 32, 700, 0, 1024], {}),                       # no compressed key, one, 63 in one tile
    (12, 3, 128, 128, [513, 640, 33], {}),
    (4, 1, 192, 128, [300, 47], dict(window_size=100)),                  # direct-to-LDS tiles, sources of other strides
    (3, 1, 32, 32, [200], dict(top_n=8, window_size=64)),
    (2, 1, 256, 256, [150], {}),
    (8, 1, 64, 64, [500], dict(kernel_size=16, stride=2, window_size=40)),  # several tiles of compressed keys
])
def test_short_batches_in_one_launch_equal_two(device, QH, KH, D, VD, lens, kw):
    """Sequences whose queries all select everything: the compressed branch, the window, the selected branch and the gated sum of one
    launch are the bits of two, with and without what the backward asks for."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.sliding_window_attention import short_fwd, swa_fwd_tail
    T = sum(lens)
    try:
        setup_helper(make_cu(lens).to(device), **kw)
        q, k, v, w = [t.to(device) for t in make_qkvw(T, QH, KH, D, VD, seed=74)]
        kk = torch.cat([k, k], 1)[:, :KH]  # the keys' strides are not those of the compressed rows
        ck, cv, below = mean_pooling_fwd(k), mean_pooling_fwd(v), NSAHelper.all_below()
        cmp_o, cmp_lse = cmp_attn_fwd(q, ck, cv)
        slc_o, slc_lse = torch.empty_like(cmp_o), torch.empty(T, QH, device=device)
        swa_o, swa_lse, out = swa_fwd_tail(q, kk, v, slc_o, slc_lse, below, cmp_o, w)
        one = short_fwd(q, kk, v, ck, cv, w, below)
        bare = short_fwd(q, kk, v, ck, cv, w, below, store=False)[3]
    finally:
        NSAHelper.set_hyperparameters()
    want = ((cmp_o, cmp_lse), (slc_o, slc_lse), (swa_o, swa_lse))
    for got, ref in zip(one[:3], want):
        assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])
    assert torch.equal(one[3], out) and torch.equal(bare, out)


@pytest.mark.parametrize("lens,kind,kw", [
    ([66100], "random", {}),                                    # every list length, registers per lane changing on the way
    ([9000], "random", dict(top_n=48)),                         # more picks than half a wave holds
    ([8200, 17000], "pairs", {}),                               # equal scores in pairs
    ([8200], "few", {}),                                        # seven different scores
    ([5000], "zero", {}), ([5000], "large", {}),
    ([70] * 100 + [0, 2100, 1, 0], "random", dict(top_n=8)),    # sequences counted in two steps
])
def test_block_selection_is_that_of_its_scores(device, lens, kind, kw):
    """Picks of the two-launch selector against a stable descending sort of the scores that it returns: exact."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops.topk import slc_topk_indices
    T, QH, KH, D = sum(lens), 4, 2, 64
    g = torch.Generator().manual_seed(31)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(device)
    try:
        NSAHelper.set_hyperparameters(**kw)
        NSAHelper.init_cu_seqlens(cu)
        h = NSAHelper
        Y = int(h.y_cu_seqlens[-1])
        q = torch.randn(T, QH, D, generator=g).bfloat16().to(device)
        rows = torch.randn(Y, KH, D, generator=g).bfloat16().to(device)
        period = dict(pairs=Y // 2 // 4 * 4, few=28).get(kind, Y)  # (4 compressed rows per selection block)
        ck = rows[torch.arange(Y, device=device) % period].contiguous()
        lse = torch.full((QH, T), dict(zero=1e4, large=-60.0).get(kind, 4.0), device=device)
        topk, probs = slc_topk_indices(q, ck, lse, return_slc_prob=True)
        top_n, init, local, bs = h.top_n, h.num_init_blocks, h.num_local_blocks, h.block_size
        ignore = -(-max(lens) // bs)
        t = torch.cat([torch.arange(n) for n in lens]).to(device)
        for r0 in range(0, T, 16384):
            nk = t[r0:r0 + 16384, None] // bs
            p, got = probs[:, r0:r0 + 16384], topk[:, r0:r0 + 16384]
            j = torch.arange(p.size(-1), device=device)
            free = (j >= init) & (j <= nk - local)
            order = torch.where(free, p, -1.0).sort(dim=-1, descending=True, stable=True).indices
            slot = torch.arange(top_n, device=device)
            want = order[..., (slot - init - local).clamp(min=0)]
            want = torch.where(slot < init, slot, torch.where(slot < init + local, nk - (slot - init), want))
            want = torch.where(slot <= nk, want, ignore)
            assert torch.equal(got, want.int()), (got != want).nonzero()[:4]
    finally:
        NSAHelper.set_hyperparameters()


@pytest.mark.parametrize("QH,KH,D,VD,n,counts", [(16, 1, 64, 64, 1500, (1, 3, 60)), (16, 2, 128, 128, 1000, (1, 20, 40)),
                                                 (16, 1, 192, 128, 1100, (1, 8, 40)), (8, 2, 256, 256, 700, (1, 5, 50))])
def test_a_sequence_does_not_depend_on_the_batch_around_it(device, QH, KH, D, VD, n, counts):
    """Forwards whose launches take the rows in their order and those that start the last rows first (by sequence length and number of
    workgroups): every copy of a sequence has the same bits."""
    from flash_nsa import NSAConfig, NSACore
    core = NSACore(NSAConfig(qk_head_dim=D, v_head_dim=VD, num_heads=QH, num_kv_heads=KH))
    ins, want = [t.to(device) for t in make_qkvw(n, QH, KH, D, VD, seed=70)], None
    for count in counts:
        with torch.no_grad():
            out = core(*(t.repeat(count, 1, 1) for t in ins), make_cu([n] * count).to(device)).view(count, n, QH, VD)
        want = out[0].clone() if want is None else want
        assert bool((out == want).all())
