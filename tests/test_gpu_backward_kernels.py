"""The dk/dv kernel for 8, 16, 32 or 64 q-heads per kv head at the sizes where it can go wrong, against the oracle with the
rounding points of a bf16 pipeline (the bar of test_gpu_backward.py); the selected forward's lists of key units."""
import pytest
import torch

from oracle import nsa_oracle as O
from gpu_util import make_cu, make_qkvw, randn_bf16, assert_close
from test_gpu_backward import setup_helper

pytestmark = pytest.mark.gpu

# tiles of 64 rows = 64 / (heads per kv head) tokens, key tiles of 64 / 128: one token, just below / at / above either
EDGES = [1, 7, 8, 9, 63, 64, 65, 127, 129, 0, 300]


@pytest.mark.parametrize("QH,KH,D,VD", [(8, 1, 64, 64), (16, 2, 128, 128), (32, 2, 192, 128), (32, 1, 128, 128),
                                        (64, 1, 64, 64)])
@pytest.mark.parametrize("block_size", [32, 64, 96, 256])
def test_dkdv_of_every_branch(device, QH, KH, D, VD, block_size):
    """All three branches, strided q and do, selection blocks narrower and wider than a workgroup's keys."""
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd, cmp_attn_bwd
    from flash_nsa.ops.select_attn import slc_attn_fwd, slc_attn_bwd
    from flash_nsa.ops.sliding_window_attention import swa_fwd, swa_bwd
    from flash_nsa.ops.topk import slc_topk_indices
    cu = make_cu(EDGES)
    T = int(cu[-1])
    q, k, v, _ = make_qkvw(T, QH, KH, D, VD, seed=300)
    do = randn_bf16(T, QH, VD, seed=304)
    setup_helper(cu.to(device), block_size=block_size, top_n=3, window_size=70)
    cfg = O.OracleConfig(block_size=block_size, top_n=3, window_size=70)
    wide = torch.zeros(T, QH + 1, D, dtype=torch.bfloat16, device=device)  # rows of q inside rows of something wider
    wide[:, 1:] = q.to(device)
    qd, kd, vd, dod = wide[:, 1:], k.to(device), v.to(device), do.to(device)
    ck, cv = mean_pooling_fwd(kd), mean_pooling_fwd(vd)
    rounded = dict(round_dtype=torch.bfloat16, round_mma=True)

    def check(name, got, ref):
        for g, n in zip(got, ("dq", "dk", "dv")):
            if g is not None:
                assert_close(g, ref[n], f"{name} {n}", row_scale=n != "dq")

    co, cl = cmp_attn_fwd(qd, ck, cv)
    ref = O.branch_forward_backward("cmp", q.float(), ck.float().cpu(), cv.float().cpu(), do.float(), cu, cfg, **rounded)
    for chunk in (32, 256):
        check(f"cmp, chunks of {chunk}", cmp_attn_bwd(qd, ck, cv, co, cl, dod, q_chunk_tokens=chunk), ref)
    wo, wl = swa_fwd(qd, kd, vd)
    check("swa", swa_bwd(qd, kd, vd, wo, wl, dod, dkv_fp32=True),
          O.branch_forward_backward("swa", q.float(), k.float(), v.float(), do.float(), cu, cfg, **rounded))
    topk, _ = slc_topk_indices(qd, ck, cl)
    so, sl = slc_attn_fwd(qd, kd, vd, topk)
    ref = O.branch_forward_backward("slc", q.float(), k.float(), v.float(), do.float(), cu, cfg, topk=topk.cpu(), **rounded)
    check("slc", slc_attn_bwd(qd, kd, vd, topk, so, sl, dod), ref)
    check("slc, dq recomputed", (slc_attn_bwd(qd, kd, vd, topk, so, sl, dod, parts="dq")[0], None, None), ref)


@pytest.mark.parametrize("QH,KH,D,VD", [(16, 2, 64, 64), (16, 1, 128, 128), (32, 2, 192, 128)])
def test_selected_forward_with_long_unit_lists(device, QH, KH, D, VD):
    """More than 64 units of 32 keys, the blocks in any order and negative ids between them, against masked attention."""
    from flash_nsa.ops.select_attn import slc_attn_fwd
    T, bs = 2310, 256
    n = -(-T // bs)
    q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, D, VD, seed=330)]
    setup_helper(make_cu([T]).to(device), block_size=bs, top_n=n + 1)
    own = (torch.arange(T, device=device) // bs)[None, :, None]
    rank = torch.rand(KH, T, n, generator=torch.Generator().manual_seed(331)).to(device)
    topk = torch.where(torch.arange(n, device=device) <= own, rank, 2.0).argsort(-1).int()
    topk = torch.where((rank[..., :1] < 0.3) & (topk != own) & (topk == 1), -1, topk)
    topk = torch.cat([topk, torch.zeros_like(topk[..., :1])], -1).contiguous()
    o, lse = slc_attn_fwd(q, k, v, topk)
    taken = torch.zeros(KH, T, n + 1, dtype=torch.bool, device=device).scatter_(2, topk[..., :n].long() % (n + 1), True)
    keys = torch.arange(T, device=device)
    seen = taken[:, :, :n].repeat_interleave(bs, 2)[:, :, :T] & (keys <= keys[:, None])
    for h in range(QH):
        kh = h // (QH // KH)
        s = (q[:, h].float() @ k[:, kh].float().t() * D ** -0.5).masked_fill(~seen[kh], float("-inf"))
        # P and o are rounded to bf16 once each: 2 * 2^-9 of the largest value
        assert (o[:, h].float() - s.softmax(-1) @ v[:, kh].float()).abs().max() <= 2 ** -8 * v.float().abs().max()
        assert (lse[:, h] - s.logsumexp(-1) * 1.4426950408889634).abs().max() < 1e-4


@pytest.mark.parametrize("QH,KH,D,VD", [(16, 1, 128, 128), (32, 1, 192, 128)])
def test_selected_gradients_over_ranges_of_tokens(device, QH, KH, D, VD):
    """dq from stored dS with a scratch that holds 2048 tokens: ranges that cut sequences, queries below t_begin left out,
    added into fp32 -- against dq recomputed and dk / dv without ranges.  dS is the same bf16 value either way up to its last
    place, so dq may differ by 2^-8 of a term's size; dk / dv only by the order of their fp32 sums."""
    from flash_nsa import _lib
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.select_attn import slc_attn_fwd, slc_attn_bwd, slc_bwd_ds_tokens
    from flash_nsa.ops.topk import slc_topk_indices
    cu = make_cu([1, 1500, 0, 3001, 77])
    T, t_begin = int(cu[-1]), 300
    q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, D, VD, seed=350)]
    do = randn_bf16(T, QH, VD, seed=354).to(device)
    setup_helper(cu.to(device), top_n=5)
    ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
    _, cl = cmp_attn_fwd(q, ck, cv)
    topk, _ = slc_topk_indices(q, ck, cl)
    o, lse = slc_attn_fwd(q, k, v, topk)
    base = torch.randn(T, QH, D, generator=torch.Generator().manual_seed(355)).to(device)
    entry_kb = QH // KH * 5 * 64 * 2 / 1024
    results = []
    for mb in (-(-2048 * entry_kb // 1024), 0):
        _lib.call("nsa_set_tuning", b"slc_ds_mb", int(mb))
        try:
            assert (0 < slc_bwd_ds_tokens(q, k, v, do, topk) < T) == (mb > 0)
            results.append(slc_attn_bwd(q, k, v, topk, o, lse, do, base.clone(), t_begin=t_begin))
        finally:
            _lib.call("nsa_reset_tuning")
    (dq, dk, dv), (dq_ref, dk_ref, dv_ref) = results
    early = torch.cat([torch.arange(a, min(a + t_begin, b)) for a, b in zip(cu[:-1].tolist(), cu[1:].tolist())])
    assert torch.equal(dq[early], base[early])
    scale = (dq_ref - base).pow(2).mean().sqrt()
    assert (dq - dq_ref).abs().max() <= 2 ** -6 * scale + 2 ** -8 * (dq_ref - base).abs().max()
    for a, b in ((dk, dk_ref), (dv, dv_ref)):
        assert (a - b).norm() <= 1e-4 * b.norm()


@pytest.mark.parametrize("QH,KH,D,VD,T", [(16, 1, 128, 128, 8292), (16, 2, 64, 64, 16484), (16, 1, 192, 128, 6653)])
def test_selected_forward_around_the_length_from_which_blocks_are_rotated(device, QH, KH, D, VD, T):
    """The last 200 queries, some on either side of the line, blocks in any order and negative ids, against masked attention."""
    from flash_nsa.ops.select_attn import slc_attn_fwd
    bs, top_n, first = 64, 16, T - 200
    n = -(-T // bs)
    assert first < (4 << 20) // ((D + VD) * 2) < T - 1
    q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, D, VD, seed=360)]
    setup_helper(make_cu([T]).to(device), block_size=bs, top_n=top_n)
    own = (torch.arange(first, T, device=device) // bs)[None, :, None]
    rank = torch.rand(KH, T - first, n, generator=torch.Generator().manual_seed(361)).to(device)
    rank = torch.where(torch.arange(n, device=device) == own, -1.0, rank)  # the own block is among the selected
    picked = torch.where(torch.arange(n, device=device) <= own, rank, 2.0).argsort(-1)[..., :top_n].int()
    picked = torch.where((picked % 7 == 3) & (picked != own), -1, picked).roll(5, -1)
    topk = torch.zeros(KH, T, top_n, dtype=torch.int32, device=device)
    topk[:, first:] = picked
    o, lse = slc_attn_fwd(q, k, v, topk, t_begin=first)
    taken = torch.zeros(KH, T - first, n + 1, dtype=torch.bool, device=device).scatter_(2, picked.long() % (n + 1), True)
    keys = torch.arange(T, device=device)
    seen = taken[:, :, :n].repeat_interleave(bs, 2)[:, :, :T] & (keys <= keys[first:, None])
    for h in range(QH):
        kh = h // (QH // KH)
        s = (q[first:, h].float() @ k[:, kh].float().t() * D ** -0.5).masked_fill(~seen[kh], float("-inf"))
        # P and o are rounded to bf16 once each: 2 * 2^-9 of the largest value
        assert (o[first:, h].float() - s.softmax(-1) @ v[:, kh].float()).abs().max() <= 2 ** -8 * v.float().abs().max()
        assert (lse[first:, h] - s.logsumexp(-1) * 1.4426950408889634).abs().max() < 1e-4


@pytest.mark.parametrize("block_size", [64, 256])
def test_selected_gradients_with_rows_behind_the_last_sequence(device, block_size):
    """Rows of q behind cu_seqlens[-1] belong to no sequence: whatever topk holds there, their dq is left alone and dk / dv are
    those of the batch without them, up to the order of their fp32 sums.  Ids of blocks that do not exist count as none."""
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.compress_attn import cmp_attn_fwd
    from flash_nsa.ops.select_attn import slc_attn_fwd, slc_attn_bwd
    from flash_nsa.ops.topk import slc_topk_indices
    cu = make_cu([100, 0, 1400, 333])
    T, more, QH, KH, D = int(cu[-1]), 70, 16, 1, 128
    q, k, v, _ = [t.to(device) for t in make_qkvw(T + more, QH, KH, D, seed=370)]
    do = randn_bf16(T + more, QH, D, seed=374).to(device)
    setup_helper(cu.to(device), top_n=5, block_size=block_size)
    ck, cv = mean_pooling_fwd(k[:T]), mean_pooling_fwd(v[:T])
    _, cl = cmp_attn_fwd(q[:T], ck, cv)
    topk, _ = slc_topk_indices(q[:T], ck, cl)
    o, lse = slc_attn_fwd(q[:T], k[:T], v[:T], topk)
    base = torch.randn(T + more, QH, D, generator=torch.Generator().manual_seed(375)).to(device)
    ref = slc_attn_bwd(q[:T], k[:T], v[:T], topk, o, lse, do[:T], base[:T].clone())
    behind = torch.randint(0, 3, (KH, more, 5), generator=torch.Generator().manual_seed(376)).int().to(device)
    behind[:, 1::4], behind[:, 2::4, 1], behind[:, 3::4, 0] = 2 ** 31 - 1, 2 ** 25 + 1, 2 ** 23 + 1
    pad = lambda t, value: torch.cat([t, torch.full((more, *t.shape[1:]), value, dtype=t.dtype, device=device)])
    wide = torch.cat([topk, behind], 1)
    got = slc_attn_bwd(q, k, v, wide, pad(o, 0.5), pad(lse, 1.0), do, base.clone())
    assert torch.equal(got[0][T:], base[T:]) and torch.equal(got[0][:T], ref[0])
    for a, b in zip(got[1:], ref[1:]):
        assert (a[:T] - b).norm() <= 1e-4 * b.norm() and not a[T:].any()
    # an id no key up to the query belongs to, in the place of the last block: as if the place were empty
    last = (torch.arange(1400, device=device) // block_size).clamp(max=4)
    results = []
    for value in (-1, 2 ** 31 - 1, 2 ** 25 + 1):
        t = topk.clone()
        rows = t[0, 100:1500]
        rows.scatter_(1, last[:, None], torch.where(last > 2, value, rows.gather(1, last[:, None])[:, 0])[:, None].int())
        results.append(slc_attn_bwd(q[:T], k[:T], v[:T], t, o, lse, do[:T], base[:T].clone())[0])
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])


@pytest.mark.parametrize("KH,D,VD,chunk,same", [(1, 128, 128, 4096, True), (1, 128, 128, 130, False), (2, 192, 128, 4096, False)])
def test_paged_selected_attention_rotates_blocks_in_long_chunks_only(device, KH, D, VD, chunk, same):
    """A chunk at the end of 9000 tokens: the bits of the unpaged launch where both rotate, else its values up to the order."""
    from flash_nsa.inference.stages import slc_attn_prefill
    from flash_nsa.ops.select_attn import slc_attn_fwd
    from paged_util import build_pool
    bs, top_n, T, QH = 64, 16, 9000, 16 * KH
    case = build_pool([T], KH, D, VD, page=128, seed=380)
    k, v = [O.gather_rows(case[n], case["bt"][0], T).to(device) for n in ("k", "v")]
    q = randn_bf16(T, QH, D, seed=381).to(device)
    n = torch.arange(T, device=device) // bs + 1  # blocks up to the own one
    step = torch.arange(top_n, device=device) * 5 + torch.arange(KH, device=device)[:, None, None]
    topk = torch.where(n[:, None] > 80, (n[:, None] - 1 - step) % n[:, None], torch.arange(top_n, device=device)).int()
    setup_helper(make_cu([T]).to(device), block_size=bs, top_n=top_n)
    first = T - chunk
    ref, ref_lse = [x[first:] for x in slc_attn_fwd(q, k, v, topk)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)
    o, lse = slc_attn_prefill(q[first:], case["k"].to(device), case["v"].to(device), topk[:, first:], i32([0, chunk]), chunk,
                              case["bt"].to(device), i32([T]), block_size=bs, top_n=top_n)
    assert torch.equal(o, ref) == same
    # P and o are rounded to bf16 once each in either: 4 * 2^-9 of the largest value
    assert (o.float() - ref.float()).abs().max() <= 2 ** -7 * v.float().abs().max()
    assert (lse - ref_lse).abs().max() < 1e-4


@pytest.mark.parametrize("QH,KH,D,VD,lens,kw", [
    (16, 2, 64, 64, [1200, 31, 0, 33, 700], {}),
    (8, 2, 64, 64, [1024, 1, 129], {}),                                    # nobody is at or above all_below
    (6, 2, 32, 32, [300, 17], dict(top_n=4, window_size=50)),              # groups of 3; keys before the window
    (12, 3, 128, 128, [90, 400], dict(top_n=2, num_init_blocks=1, num_local_blocks=1, window_size=200)),
    (4, 1, 192, 128, [500], dict(top_n=4)),
    (2, 1, 256, 256, [260], dict(top_n=2, window_size=64)),
    (8, 1, 64, 64, [300], dict(kernel_size=16, stride=2, top_n=3)),        # several tiles of compressed keys
])
def test_dense_dq_in_one_launch_equals_two(device, QH, KH, D, VD, lens, kw):
    """Window, keys before it and compressed branch in one launch against the window's launch and the compressed branch's that adds
    to it: the same products summed in fp32 in another order, so the fp32 rows to 1e-5 and the bf16 ones to a rounding."""
    from flash_nsa import NSAHelper
    from flash_nsa.ops.compress_attn import cmp_attn_bwd, cmp_attn_fwd
    from flash_nsa.ops.compress_kv import mean_pooling_fwd
    from flash_nsa.ops.sliding_window_attention import dense_bwd_dq, swa_bwd_dq_tail, swa_fwd
    T = sum(lens)
    try:
        NSAHelper.set_hyperparameters(**kw)
        NSAHelper.init_cu_seqlens(make_cu(lens).to(device))
        below, short = NSAHelper.all_below(), max(lens) <= NSAHelper.all_below()
        q, k, v, _ = [t.to(device) for t in make_qkvw(T, QH, KH, D, VD, seed=120)]
        ck, cv = mean_pooling_fwd(k), mean_pooling_fwd(v)
        _, cmp_lse = cmp_attn_fwd(q, ck, cv)
        _, lse = swa_fwd(q, k, v)
        do, cmp_do = [randn_bf16(T, QH, VD, seed=s).to(device) for s in (125, 126)]
        delta = torch.randn(3, T, QH, generator=torch.Generator().manual_seed(127)).to(device)
        slc_lse = lse + 1
        nan = lambda dtype: torch.full((T, QH, D), float("nan"), device=device, dtype=dtype)
        want32, want = nan(torch.float32), nan(torch.bfloat16)
        swa_bwd_dq_tail(q, k, v, lse, do, delta[2], slc_lse, do, delta[1], below, want32, store=True)
        cmp_attn_bwd(q, ck, cv, None, cmp_lse, cmp_do, want32, delta=delta[0], finalize_dq=True, parts="dq",
                     finalize_below=(want, below))
        got32, got = None if short else nan(torch.float32), nan(torch.bfloat16)
        dense_bwd_dq(q, k, v, lse, do, delta[2], slc_lse, do, delta[1], below, ck, cv, cmp_lse, cmp_do, delta[0], got, got32)
    finally:
        NSAHelper.set_hyperparameters()
    low = torch.cat([torch.arange(n) < below for n in lens]).to(device)
    a, b = got[low].float(), want[low].float()
    # (a step between neighbours of bf16 is up to 2^-7 of the value; sums that cancel: fp32 of the row's largest value)
    over = (a - b).abs() - 2.0 ** -7 * b.abs() - 1e-5 * b.abs().amax(-1, keepdim=True)
    assert float(over.max()) <= 0, (float(over.max()), float((a != b).float().mean()))
    if not short:
        a, b = got32[~low], want32[~low]
        assert float((a - b).norm() / b.norm()) < 1e-5, float((a - b).norm() / b.norm())
        assert bool(got[~low].isnan().all()) and bool(got32[low].isnan().all())  # written by nobody
